// Grouped expert launches of larger batches on the int8 matrix unit (included by moe.hip).
//
// A workgroup takes up to 16 MT (token, slot) pairs of one expert and some 16-row tiles of one of its matrices.  Lane
// (c, l) = (lane & 15, lane / 16) decodes what quad lane l decodes of row c: two whole blocks of a super-block, so a
// wavefront decodes 16 rows of a super-block at a time and every weight once for all pairs of the tile (the quad-lane
// kernel below once for four pairs).  v_mfma_i32_16x16x32_i8 wants lane (c, l) to hold elements 8 l .. of one block of
// row c: the four lanes of a row exchange quarters of their blocks with four lane swaps per pair of registers.  Operand
// one is the pairs' activations, [block][pair][32] in LDS, so the exact block sums of pairs 4 l .. 4 l + 3 lie with row c.
// The scales need no exchange: the matrix unit multiplies a lane's own by those of the pairs and leaves the products where the
// block sums lie.  Minima (Q4_K) are exchanged with the same swaps.
//
// Bound by the decoders (vector instructions and, for IQ3_S, table gathers: the LDS is busy four fifths of the time), the
// weights' bytes, and a workgroup's start (a chain of five loads; half as many row tiles a workgroup take 15 % longer, for all that
// their last round is fuller); the products and the rescale of 16 pairs are a seventh of the instructions.  256 experts of 2048 x 512
// and one for all tokens, IQ3_S, 333 tokens of 9 slots: gate and up 279 -> 138 us, down 134 -> 70 us against one decode for
// four pairs (the weights alone are 45 and 23 us of reads).  Scales multiplied on the matrix unit, sums without a conversion
// and carries by branches are 258 instead of 352 vector instructions a super-block; whole feed-forwards, IQ3_S: 440 tokens, 128 experts of
// 2048 x 1024 (32 pairs a tile) 327 -> 292 us, the 333 tokens above 1 to 2 % (the tables); Q4_K 217 -> 208, 440 tokens, 64 of 4096 x 768 519 -> 470.
#pragma once

#include <type_traits>

namespace llamql
{
    constexpr int MOE_MFMA_WAVES = 8;
    constexpr int MOE_MFMA_MAX_SB = 16; // super-blocks of a row
    typedef float v16f_moe __attribute__((ext_vector_type(16)));
    constexpr float MOE_MFMA_BIAS = 12582912.0f; // 1.5 * 2^23
    constexpr size_t MOE_MFMA_LDS = 150 * 1024; // of the 160 KB, beside the decoders' tables

    // bytes of a block's activations in LDS: a pad, so that neighbouring blocks of a pair start in different banks
    __host__ __device__ constexpr int moe_mfma_block_bytes(int mt) { return mt * 16 * 32 + 16; }
    template <bool HAS_MIN>
    __host__ __device__ constexpr size_t moe_mfma_lds(int mt, int nsb)
    {
        return (size_t)nsb * 8 * (moe_mfma_block_bytes(mt) + mt * 16 * 4 * (HAS_MIN ? 2 : 1));
    }

    // Dwords u[k] = (unit k of this lane's 32 bytes) of the lanes (c, 0..3) of a row become y[m] = unit (own l) of lane
    // (c, m).  permlane32_swap exchanges the upper half of one register with the lower of another, permlane16_swap the
    // odd rows of 16 lanes with the even ones.
    __device__ __forceinline__ void quarter_exchange(uint32_t (&u)[4])
    {
        typedef uint32_t v2u __attribute__((ext_vector_type(2)));
        const v2u a = __builtin_bit_cast(v2u, __builtin_amdgcn_permlane32_swap(u[0], u[2], false, false));
        const v2u b = __builtin_bit_cast(v2u, __builtin_amdgcn_permlane32_swap(u[1], u[3], false, false));
        const v2u c = __builtin_bit_cast(v2u, __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false));
        const v2u d = __builtin_bit_cast(v2u, __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false));
        u[0] = c[0], u[1] = c[1], u[2] = d[0], u[3] = d[1];
    }

    // grid: (workgroups per matrix, tiles of pairs (upper bound), DOWN ? 1 : 2 = gate|up)
    // m.rows_per_wave: 16-row tiles of a wavefront
    template <class F, int MT, bool DOWN>
    __global__ void __launch_bounds__(MOE_MFMA_WAVES *WAVE) __attribute__((amdgpu_waves_per_eu(F::TABLE_BYTES > 0 ? 4 : 1)))
        moe_grouped_mfma_kernel(const MoEArgs m, void *ws, int P)
    {
        typedef typename F::Quad Q;
        constexpr int KBS = moe_mfma_block_bytes(MT);
        extern __shared__ __attribute__((aligned(16))) uint8_t moe_mfma_smem[];
        __shared__ int s_pairs[MT * 16];
        const MoEGroupView g = moe_group_view(ws, P);
        const int lane = threadIdx.x & (WAVE - 1);
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));

        // the tile's expert: the segments' tiles one after the other
        const int want = blockIdx.y, segments = g.head[0];
        int seg = -1, tile = 0, seen = 0;
        for (int s0 = 0; s0 < segments && seg < 0; s0 += WAVE)
        {
            const int s = s0 + lane < segments ? s0 + lane : segments - 1;
            const int n = s0 + lane < segments ? g.seg_begin[s + 1] - g.seg_begin[s] : 0;
            const int tiles = (n + MT * 16 - 1) / (MT * 16);
            int upto = tiles;
#pragma unroll
            for (int off = 1; off < WAVE; off <<= 1)
            {
                const int o = __shfl_up(upto, off);
                upto += lane >= off ? o : 0;
            }
            const unsigned long long past = __ballot(seen + upto > want);
            if (past)
            {
                const int who = __builtin_ctzll(past);
                seg = s0 + who;
                tile = want - (seen + __shfl(upto - tiles, who));
            }
            seen += __shfl(upto, WAVE - 1);
        }
        if (seg < 0)
            return; // uniform
        seg = __builtin_amdgcn_readfirstlane(seg);
        const int begin = __builtin_amdgcn_readfirstlane(g.seg_begin[seg] + tile * MT * 16);
        const int left = __builtin_amdgcn_readfirstlane(g.seg_begin[seg + 1]) - begin;
        const int n = left < MT * 16 ? left : MT * 16;
        const int e = g.seg_expert[seg];
        const void *w = DOWN ? m.experts[e].d_down : (blockIdx.z == 0 ? m.experts[e].d_gate : m.experts[e].d_up);
        if (!w)
            return; // an expert whose matrices live elsewhere (uniform)
        const int K = DOWN ? m.inter : m.hidden, N = DOWN ? m.hidden : m.inter;
        const int nsb = K / 256, nkb = nsb * 8, row_tiles = N / 16;
        GemvArgs a; // weight addressing only
        a.w = uniform_base(w);
        a.N = N;
        a.SB = nsb;

        const int c = lane & 15, l = lane >> 4;
        const typename Q::Lane lc = Q::lane_consts(l);
        const int tile0 = ((int)blockIdx.x * MOE_MFMA_WAVES + wave) * m.rows_per_wave;
        const int own = row_tiles - tile0 < m.rows_per_wave ? row_tiles - tile0 : m.rows_per_wave;
        const int nsteps = own > 0 ? own * nsb : 0;
        // loads are never predicated: past the end a lane reads its first super-block again
        const typename Q::Cursor wc = Q::cursor(a, (size_t)((own > 0 ? tile0 : 0) * 16 + c) * nsb, 0, lc);
        int ld_step = 0, ld_tile = 0, ld_sb = 0;
        auto issue = [&](typename Q::Raw &buf) {
            Q::load_at(buf, wc, lc, ld_step < nsteps ? ld_tile * 16 * nsb + ld_sb : 0);
            ++ld_step;
            if (++ld_sb == nsb)
            {
                ld_sb = 0;
                ++ld_tile;
            }
        };
        typename Q::Raw bufA, bufB;
        issue(bufA);
        issue(bufB);

        // the pairs' activations, a thread per Q8_1 block (pairs past the last repeat it)
        float *ad = reinterpret_cast<float *>(moe_mfma_smem + (size_t)nkb * KBS), *asd = ad + nkb * MT * 16;
        const int32_t *pairs = g.pair_sorted + begin;
        for (int idx = threadIdx.x; idx < MT * 16 * nkb; idx += MOE_MFMA_WAVES * WAVE)
        {
            const int q = idx / nkb, kb = idx - q * nkb;
            if ((q & ~15) >= n)
                break; // (whole groups of 16 pairs that are not there)
            const int pair = pairs[q < n ? q : n - 1];
            if (kb == 0)
                s_pairs[q] = pair;
            const uint32_t *src = m.q8 + ((size_t)(DOWN ? pair : pair / m.top_k) * nkb + kb) * 9;
            uint32_t v[9];
#pragma unroll
            for (int i = 0; i < 9; ++i)
                v[i] = src[i];
            const float d = h2f((uint16_t)(v[0] & 0xFFFFu));
            uint4 *dst = reinterpret_cast<uint4 *>(moe_mfma_smem + (size_t)kb * KBS + q * 32);
            dst[0] = make_uint4(v[1], v[2], v[3], v[4]);
            dst[1] = make_uint4(v[5], v[6], v[7], v[8]);
            ad[kb * MT * 16 + q] = d;
            if (F::HAS_MIN)
                asd[kb * MT * 16 + q] = (float)(int16_t)(v[0] >> 16) * d;
        }
        Q::stage();
        __syncthreads();
        Q::keep(bufA);
        Q::keep(bufB);

        float *out = DOWN ? m.out1 : (blockIdx.z == 0 ? m.out0 : m.out1);
        // A row's blocks are summed as the quad-lane kernels' lanes sum them, as a binary tree over lanes and super-blocks
        // (the same bits where a row is a power of two of them): level[k] holds the sum of 2^k super-blocks, a carry
        // walks up it like in a counter.  (A single chain over 64 blocks is also off by twice as much.)
        constexpr int LEVELS = 5;
        static_assert(MOE_MFMA_MAX_SB < 1 << LEVELS, "levels of the tree");
        float level[MT][LEVELS][4];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int k = 0; k < LEVELS; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    level[t][k][r] = 0.0f;
        int step = 0, sb = 0, row = tile0 * 16 + c;
        // (branches, which are uniform, and not choices between registers: those were 32 of 350 instructions a super-block)
        auto carry = [&](auto &self, int t, float (&sum)[4], auto depth) __attribute__((always_inline)) {
            constexpr int k = decltype(depth)::value;
            if constexpr (k + 1 < LEVELS)
            {
                if ((sb >> k) & 1)
                {
                    asm volatile("");
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        sum[r] = level[t][k][r] + sum[r];
                    self(self, t, sum, std::integral_constant<int, k + 1>());
                    return;
                }
                asm volatile("");
            }
#pragma unroll
            for (int r = 0; r < 4; ++r)
                level[t][k][r] = sum[r];
        };
        v4i bias;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            bias[r] = __float_as_int(MOE_MFMA_BIAS);
        asm volatile("" : "+v"(bias));
        const uint8_t *a_lane = moe_mfma_smem + c * 32 + l * 8;
        auto compute = [&](const typename Q::Raw &buf) {
            v4i wq[4];
            typename Q::Scale S;
            Q::decode(buf, lc, wq, S);
            uint32_t lo[2][4], hi[2][4], low[2][4];
#pragma unroll
            for (int i = 0; i < 2; ++i)
            {
                const uint32_t mn = __float_as_uint(Q::min_f32(S, i));
#pragma unroll
                for (int k = 0; k < 4; ++k)
                {
                    lo[i][k] = (uint32_t)wq[2 * i + (k >> 1)][2 * (k & 1)];
                    hi[i][k] = (uint32_t)wq[2 * i + (k >> 1)][2 * (k & 1) + 1];
                    low[i][k] = mn;
                }
                quarter_exchange(lo[i]);
                quarter_exchange(hi[i]);
                if (F::HAS_MIN)
                    quarter_exchange(low[i]);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t)
            {
                if (t > 0 && t * 16 >= n)
                    break; // uniform
                float sum[4][4];
#pragma unroll
                for (int i = 0; i < 2; ++i)
                {
                    // A lane's own scale times the pairs' of its block: rank-1 matrices of four blocks, in the layout of the block sums
                    // (exact: both factors are fp16 values)
                    const v16f_moe none = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
                    const v16f_moe scale = __builtin_amdgcn_mfma_f32_16x16x1f32(ad[(sb * 8 + Q::block_of(l, i)) * MT * 16 + t * 16 + c], Q::scale_f32(S, i), none, 0, 0, 0);
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                    {
                        const int kb = sb * 8 + Q::block_of(k, i);
                        const long b = (long)(((uint64_t)hi[i][k] << 32) | lo[i][k]);
                        const float bm = __uint_as_float(low[i][k]);
                        const long x = *reinterpret_cast<const long *>(a_lane + (size_t)kb * KBS + t * 512);
                        // started from the bits of 1.5 * 2^23, the integer result has those of 1.5 * 2^23 + sum: no conversion
                        const v4i d = __builtin_amdgcn_mfma_i32_16x16x32_i8(x, b, bias, 0, 0, 0);
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                        {
                            const float f = __int_as_float(d[r]) - MOE_MFMA_BIAS;
                            sum[k][r] = i == 0 ? f * scale[4 * k + r] : fmaf(f, scale[4 * k + r], sum[k][r]);
                        }
                        if (F::HAS_MIN)
                        {
                            const float4 sa = *reinterpret_cast<const float4 *>(asd + kb * MT * 16 + t * 16 + 4 * l);
                            const float ss[4] = {sa.x, sa.y, sa.z, sa.w};
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                sum[k][r] = fmaf(ss[r], bm, sum[k][r]);
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    sum[0][r] = (sum[0][r] + sum[1][r]) + (sum[2][r] + sum[3][r]);
                carry(carry, t, sum[0], std::integral_constant<int, 0>());
            }
            ++step;
            if (++sb == nsb)
            {
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                    {
                        const int q = t * 16 + 4 * l + r;
                        float y = 0.0f;
                        bool first = true;
#pragma unroll
                        for (int k = LEVELS - 1; k >= 0; --k)
                            if ((nsb >> k) & 1) // uniform
                            {
                                y = first ? level[t][k][r] : y + level[t][k][r];
                                first = false;
                            }
                        if (q < n)
                            out[(size_t)s_pairs[q] * N + row] = y;
                    }
                sb = 0;
                row += 16;
            }
        };
        for (int s0 = 0; s0 < nsteps; s0 += 2)
        {
            Q::template wait<Q::LOADS>(bufA);
            compute(bufA);
            __builtin_amdgcn_sched_barrier(0);
            issue(bufA);
            Q::template wait<Q::LOADS>(bufB);
            if (step < nsteps) // uniform
                compute(bufB);
            __builtin_amdgcn_sched_barrier(0);
            issue(bufB);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // loads issued past the end
        Q::keep(bufA);
        Q::keep(bufB);
    }
} // namespace llamql
