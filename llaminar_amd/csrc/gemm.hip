// Prefill GEMM for gfx950: GGUF block-quantized weights x Q8_1 activations on
// int8 MFMA with int32 accumulation per 32-column block and fp32 rescale.
//
//   C[m,n] = sum_kb float(idot[m,n,kb]) * (f32(a.d[m,kb]) * b_scale[n,kb])
//          + sum_kb (float(a.sum[m,kb]) * f32(a.d[m,kb])) * b_min[n,kb]
//
// idot is formed by ONE v_mfma_i32_32x32x32_i8 per 32x32 output tile and K-block
// (K depth 32 = exactly one Q8_1 block, zero accumulator input), so it is the
// same exact integer the reference forms with vpdpbusd
// (CPUNativeVNNIGemv.h:1046-1231); the per-block rescale is fp32 work: the scale
// products a_d[m] * b_scale[n] of a block, a rank-1 matrix, come from the matrix unit too
// (v_mfma_f32_32x32x1_2b_f32: two blocks per instruction, exact), convert and multiply-add per
// output element stay on
// the vector unit (two operations against 64 int8 MFMA operations: this, not the int8
// rate of the matrix unit, bounds the kernel), and the rank-1 min term goes through
// another v_mfma_f32_32x32x2f32 straight into the accumulator.
//
// Workgroup: 512 threads = 8 wavefronts, tile 128 tokens x 64 weight rows, 64 KiB
// of LDS, so two workgroups share a compute unit and one's staging overlaps the
// other's multiply.  K advances one 256-column super-block at a time.  The global
// data of a step (raw weight blocks, 72 bytes of Q8_1 per thread) is fetched into
// registers while the previous step is multiplied; then the weights are decoded
// (nibble unpack / requantise, shared with the GEMV decoders) into LDS as int8
// [row][k], the activations copied beside them, both with a 272-byte row stride
// (conflict-free ds_read_b128 for MFMA operands).  Wavefront w owns weight rows
// 32*(w%2).. and tokens 32*(w/2)..: one 32x32 MFMA tile.  The MFMA's A operand is
// the activation tile, B the weight tile, so a lane holds one weight row n and 16
// tokens: stores of C are 128-byte coalesced and b_scale is one register per block.
#include "gemv_traits_all.h"

#include "llaminar_amd/ql_api.h"

#include <type_traits>

namespace llamql
{
    typedef float v16f __attribute__((ext_vector_type(16)));
    typedef float v32f __attribute__((ext_vector_type(32)));

    constexpr int GEMM_BM = 128;        // tokens per workgroup
    // (launches of up to 32 and up to 64 tokens run tiles of 32 and 64 tokens: gemm_kernel's BM)
    constexpr int GEMM_BN = 64;         // weight rows per workgroup
    constexpr int GEMM_THREADS = 512;
    constexpr int GEMM_STRIDE = 256 + 16; // bytes per LDS row (one super-block + pad)
    // per-block scale tables [8][rows + 8]: the pad spreads the four threads that write one
    // row's scales of different blocks over different banks
    constexpr int GEMM_SN = GEMM_BN + 8;

    struct GemmArgs
    {
        GemvArgs w;         // only w.w, w.N, w.SB are used (weight addressing)
        const uint32_t *q8; // [M][K/32] blocks as dwords
        float *y;
        int M, ldy;
        // DUMP kernels only: the exact per-block int32 sums of weight rows [row0, row0+nrows) go to
        // sums[(m * nrows + n - row0) * (K/32) + block]
        int32_t *sums;
        int row0, nrows;
        int tile0; // first 64-row tile of the launch
    };

    template <class F, int BM>
    constexpr size_t gemm_lds_bytes()
    {
        return (size_t)(BM + GEMM_BN) * GEMM_STRIDE + (size_t)2 * 8 * (BM + 8 + GEMM_SN) * sizeof(float);
    }

    // Two adjacent Q8_1 blocks (72 bytes, 4-byte aligned) of one token, fetched with loads
    // the kernel waits for itself: written as ordinary loads the compiler moves them down
    // to their first use, behind the multiply they are meant to overlap.
    typedef int v2i __attribute__((ext_vector_type(2)));
    struct GemmActRaw
    {
        v4i q0, q1, q2, q3;
        v2i q4;
        __device__ __forceinline__ void load(const uint32_t *p)
        {
            asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(q0) : "v"(p));
            asm volatile("global_load_dwordx4 %0, %1, off offset:16" : "=&v"(q1) : "v"(p));
            asm volatile("global_load_dwordx4 %0, %1, off offset:32" : "=&v"(q2) : "v"(p));
            asm volatile("global_load_dwordx4 %0, %1, off offset:48" : "=&v"(q3) : "v"(p));
            asm volatile("global_load_dwordx2 %0, %1, off offset:64" : "=&v"(q4) : "v"(p));
        }
        // every load issued so far has arrived
        __device__ __forceinline__ void wait()
        {
            asm volatile("s_waitcnt vmcnt(0)" : "+v"(q0), "+v"(q1), "+v"(q2), "+v"(q3), "+v"(q4));
        }
        __device__ __forceinline__ uint32_t dword(int i) const
        {
            // i is a compile-time constant after unrolling
            return (uint32_t)(i < 4 ? q0[i] : i < 8 ? q1[i - 4] : i < 12 ? q2[i - 8] : i < 16 ? q3[i - 12] : q4[i - 16]);
        }
    };

    // Weight data of one K step held in registers while the previous step is multiplied.
    template <class F, bool QUAD = F::USE_QUAD>
    struct GemmPrefetch;

    // Formats with a quad-lane decoder: thread = (weight row, quad lane), 64 weights.
    template <class F>
    struct GemmPrefetch<F, true>
    {
        typedef typename F::Quad Q;
        typename Q::Raw raw;
        typename Q::Lane lc;
        typename Q::Cursor wc;
        int row, l;
        bool active; // wavefront-uniform: BN rows x 4 quad lanes = the first 4*BN threads

        // first: the first of the 4 BN decoding threads (a multiple of 4 BN)
        __device__ __forceinline__ void init(const GemmArgs &g, long n0, int tid, int first)
        {
            const int t0 = __builtin_amdgcn_readfirstlane(tid);
            active = t0 >= first && t0 < first + GEMM_BN * 4;
            row = (tid >> 2) & (GEMM_BN - 1);
            l = tid & 3;
            lc = Q::lane_consts(l);
            long n = n0 + row;
            if (n >= g.w.N)
                n = g.w.N - 1; // tail rows: decode a valid row, never stored
            wc = Q::cursor(g.w, (size_t)n * g.w.SB, (size_t)n * g.w.SB, lc);
        }
        __device__ __forceinline__ void issue(const GemmArgs &, int sb)
        {
            // the other wavefronts load the same bytes again (cache hits) and drop them: a
            // load under a condition would need a register copy that waits for it at once
            // (asking for the rows of a later step instead, to warm the L2 cache, changed nothing)
            Q::load_at(raw, wc, lc, sb);
        }
        __device__ __forceinline__ void store(uint8_t *Wl, float *bs, float *bm, const void *)
        {
            Q::template wait<0>(raw);
            if (!active)
                return;
            v4i w[4];
            typename Q::Scale S;
            Q::decode(raw, lc, w, S);
#pragma unroll
            for (int i = 0; i < 2; ++i)
            {
                const int j = Q::block_of(l, i);
                v4i *dst = reinterpret_cast<v4i *>(Wl + row * GEMM_STRIDE + 32 * j);
                dst[0] = w[2 * i];
                dst[1] = w[2 * i + 1];
                bs[j * GEMM_SN + row] = Q::scale_f32(S, i);
                bm[j * GEMM_SN + row] = Q::min_f32(S, i);
            }
        }
        __device__ __forceinline__ void finish() { Q::template wait<0>(raw); }
    };

    // Other formats: the 8-lane decode of the GEMV skeleton, one task per thread.
    template <class F>
    struct GemmPrefetch<F, false>
    {
        static_assert(GEMM_BN * 8 == GEMM_THREADS, "one (row, lane) task per thread");
        typename F::Raw raw;
        long n;
        int row, c;

        __device__ __forceinline__ void init(const GemmArgs &g, long n0, int tid, int)
        {
            row = tid >> 3;
            c = tid & 7;
            n = n0 + row;
            if (n >= g.w.N)
                n = g.w.N - 1;
        }
        __device__ __forceinline__ void issue(const GemmArgs &g, int sb) { raw = F::load(g.w, n, sb, c); }
        __device__ __forceinline__ void store(uint8_t *Wl, float *bs, float *bm, const void *tab)
        {
            v4i w0, w1;
            int j;
            float bscale, bmin;
            F::decode(raw, c, w0, w1, j, bscale, bmin, tab);
            int j0, e0, j1, e1;
            F::where(c, j0, e0, j1, e1);
            *reinterpret_cast<v4i *>(Wl + row * GEMM_STRIDE + 32 * j0 + e0) = w0;
            *reinterpret_cast<v4i *>(Wl + row * GEMM_STRIDE + 32 * j1 + e1) = w1;
            bs[j * GEMM_SN + row] = bscale;
            bm[j * GEMM_SN + row] = bmin;
        }
        __device__ __forceinline__ void finish() {}
    };

    // DUMP: also store the matrix unit's results, the exact int32 block sums (the parity hook of
    // the C-ABI), for a window of weight rows; otherwise the same code.
    // BM = 128: wavefront w owns one 32x32 tile (tokens 32 (w / 2).., weight rows 32 (w % 2)..) and all eight
    // blocks of a K step.  BM = 64 and 32 (few tokens): the workgroup has four or two tiles only, so two or
    // four wavefronts share a tile and take four or two of a step's eight blocks each -- the rescale work per
    // wavefront falls with the tokens -- and their partial accumulators are added in wavefront order at the
    // end.
    template <class F, bool DUMP = false, int BM = GEMM_BM>
    // (the block-sum variant of the small tile also carries the addresses of the sums: it may take the
    // registers of three wavefronts per SIMD unit; it is the parity hook, not a timed path)
    __global__ void __launch_bounds__(GEMM_THREADS)
        __attribute__((amdgpu_waves_per_eu(DUMP && BM != GEMM_BM ? 3 : 4, 4)))
        gemm_kernel(const GemmArgs g)
    {
        static_assert(BM == 128 || BM == 64 || BM == 32, "tiles of 128, 64 or 32 tokens");
        constexpr int GEMM_SM = BM + 8; // per-block scale table [8][tokens + 8]
        constexpr int MTILES = BM / 32;             // 32-token tiles of the workgroup
        constexpr int KPARTS = 4 / MTILES;          // wavefronts that share a tile's K step
        constexpr int KB_PER = 8 / KPARTS;          // blocks of a K step per wavefront
        extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
        uint8_t *Al = smem;                             // [BM][STRIDE] activations int8
        uint8_t *Wl = Al + BM * GEMM_STRIDE;            // [BN][STRIDE] weights int8
        float *ad = reinterpret_cast<float *>(Wl + GEMM_BN * GEMM_STRIDE); // [8][SM] a_d
        float *asd = ad + 8 * GEMM_SM;                  // [8][SM]
        float *bs = asd + 8 * GEMM_SM;                  // [8][SN]
        float *bm = bs + 8 * GEMM_SN;                   // [8][SN]
        void *tab = format_tables_lds<F>(); // static LDS beside the dynamic tiles

        if (F::TABLE_BYTES > 0)
            F::stage_tables(tab);

        const int tid = threadIdx.x;
        const int lane = tid & 63;
        // (small tiles: in a scalar register, like all it leads to -- they have no vector register to spare)
        const int wave = BM == GEMM_BM ? tid >> 6 : __builtin_amdgcn_readfirstlane(tid >> 6);
        const int ntile = wave & 1;
        const int mtile = KPARTS == 1 ? wave >> 1 : (wave >> 1) % MTILES;
        const int kpart = KPARTS == 1 ? 0 : (wave >> 1) / MTILES; // this wavefront's blocks of a step: kpart * KB_PER ..
        const int l32 = lane & 31;
        const int lh = lane >> 5;

        const long n0 = ((long)blockIdx.x + g.tile0) * GEMM_BN;
        const long m0 = (long)blockIdx.y * BM;
        const int KB = g.w.SB * 8;

        // activations: thread = (token, pair of adjacent Q8_1 blocks) -> 72 contiguous bytes; the first
        // 4 BM threads (whole wavefronts) have a token, the others load and store nothing
        const bool a_thread = BM * 4 >= GEMM_THREADS || __builtin_amdgcn_readfirstlane(tid) < BM * 4; // per wavefront
        const int am = (tid >> 2) & (BM - 1);
        const int ap = tid & 3;
        long am_src = m0 + am;
        if (am_src >= g.M)
            am_src = g.M - 1; // tail tokens: a valid row, never stored
        const uint32_t *asrc = g.q8 + ((size_t)am_src * KB + 2 * ap) * 9;
        GemmActRaw areg;

        GemmPrefetch<F> pf;
        // small tiles: the wavefronts that stage no activations decode the weights (the second half of
        // the workgroup), so that the two kinds of staging run side by side
        pf.init(g, n0, tid, BM == GEMM_BM ? 0 : GEMM_THREADS - GEMM_BN * 4);

        auto issue = [&](int sb) {
            pf.issue(g, sb);
            if (a_thread)
                areg.load(asrc + (size_t)sb * 72);
        };

        // One K step's staging: registers -> LDS (weights as int8 [row][k] + scales, activations
        // beside them), then the next step's global data is asked for, to travel while this one
        // is multiplied (the last step re-reads itself: every issued load is consumed, none is
        // conditional).
        auto stage = [&](int sb) {
            __syncthreads(); // previous step's LDS reads (and the table staging) are done
            pf.store(Wl, bs, bm, tab);
            areg.wait();
            if (a_thread)
            {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                {
                    const uint32_t h = areg.dword(9 * i);
                    const float d = h2f((uint16_t)(h & 0xFFFFu));
                    const int kb = 2 * ap + i;
                    ad[kb * GEMM_SM + am] = d;
                    asd[kb * GEMM_SM + am] = (float)(int16_t)(h >> 16) * d;
                    v4i *dst = reinterpret_cast<v4i *>(Al + am * GEMM_STRIDE + kb * 32);
                    dst[0] = (v4i){(int)areg.dword(9 * i + 1), (int)areg.dword(9 * i + 2), (int)areg.dword(9 * i + 3),
                                   (int)areg.dword(9 * i + 4)};
                    dst[1] = (v4i){(int)areg.dword(9 * i + 5), (int)areg.dword(9 * i + 6), (int)areg.dword(9 * i + 7),
                                   (int)areg.dword(9 * i + 8)};
                }
            }
            __syncthreads();
            issue(sb + 1 < g.w.SB ? sb + 1 : sb);
        };

        v16f acc;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            acc[r] = 0.0f;

        issue(0);
        for (int sb = 0; sb < g.w.SB; ++sb)
        {
            stage(sb);

            // ---- multiply ------------------------------------------------------------------
            // 8 block products per step; the other wavefronts of the SIMD unit keep the vector
            // unit busy while this one waits for the matrix unit.
            const uint8_t *wrow = Wl + (ntile * 32 + l32) * GEMM_STRIDE + lh * 16;
            const uint8_t *arow = Al + (mtile * 32 + l32) * GEMM_STRIDE + lh * 16;
            v16i zero;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                zero[r] = 0;
            v32f zero2f;
#pragma unroll
            for (int r = 0; r < 32; ++r)
                zero2f[r] = 0.0f;
            v16f zero1f;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                zero1f[r] = 0.0f;
            auto product = [&](int kb) {
                const v4i bw = *reinterpret_cast<const v4i *>(wrow + kb * 32);
                const v4i aa = *reinterpret_cast<const v4i *>(arow + kb * 32);
                return __builtin_amdgcn_mfma_i32_32x32x32_i8(aa, bw, zero, 0, 0, 0);
            };
            // The scale products a_d[m] * b_scale[n] of a block are a rank-1 matrix: the matrix
            // unit forms them in the layout of the block sums instead of 16 multiplies per lane,
            // two blocks per instruction (v_mfma_f32_32x32x1_2b_f32: lane half lh supplies block
            // kb + lh, results 0-15 belong to block kb, 16-31 to block kb + 1).  Exact: both
            // factors are fp16 values.
            auto scales = [&](int kb) {
                const float av = ad[(kb + lh) * GEMM_SM + mtile * 32 + l32];
                const float bv = bs[(kb + lh) * GEMM_SN + ntile * 32 + l32];
                return __builtin_amdgcn_mfma_f32_32x32x1f32(av, bv, zero2f, 0, 0, 0);
            };
            // Formats whose prefetch registers leave no room for two blocks' scale products form
            // them one block at a time (v_mfma_f32_32x32x2_f32 adds (a_d/2) * b_scale twice: exact).
            auto scales1 = [&](int kb) {
                const float av = 0.5f * ad[kb * GEMM_SM + mtile * 32 + l32];
                const float bv = bs[kb * GEMM_SN + ntile * 32 + l32];
                return __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, zero1f, 0, 0, 0);
            };
            v32f cs;
            v16f cs1;
            const int kb0 = kpart * KB_PER; // (KB_PER is even: the pairs of the scale and min-term products stay whole)
            if constexpr (F::GEMM_PAIR_SCALES)
                cs = scales(kb0);
            else
                cs1 = scales1(kb0);
#pragma unroll
            for (int kk8 = 0; kk8 < KB_PER; ++kk8)
            {
                const int kb = kb0 + kk8;
                // (one set of result registers: with the scale products held as well, a second
                // set would not fit the 128 registers that four wavefronts per SIMD unit leave;
                // the other wavefronts cover the product's latency)
                const v16i d = product(kb);
                if constexpr (DUMP)
                {
                    const long n = n0 + ntile * 32 + l32;
                    const long nn = n - g.row0;
                    if (n < g.w.N && nn >= 0 && nn < g.nrows)
                    {
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                        {
                            const long m = m0 + mtile * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
                            if (m < g.M)
                                g.sums[((size_t)m * g.nrows + (size_t)nn) * (size_t)KB + (size_t)sb * 8 + kb] = d[r];
                        }
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[r] = fmaf((float)d[r], F::GEMM_PAIR_SCALES ? cs[16 * (kk8 & 1) + r] : cs1[r], acc[r]);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (F::GEMM_PAIR_SCALES)
                {
                    if ((kk8 & 1) && kk8 + 1 < KB_PER)
                        cs = scales(kb + 1); // the other wavefronts of the unit cover its latency
                }
                else
                {
                    if (kk8 + 1 < KB_PER)
                        cs1 = scales1(kb + 1);
                }
                __builtin_amdgcn_sched_barrier(0);
                if (F::HAS_MIN && (kk8 & 1))
                {
                    // rank-2 update over blocks kb-1, kb, straight into the accumulator: lane
                    // half lh supplies block kb-1+lh
                    const int kk = kb - 1 + lh;
                    const float bmin = bm[kk * GEMM_SN + ntile * 32 + l32];
                    const float av = asd[kk * GEMM_SM + mtile * 32 + l32];
                    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bmin, acc, 0, 0, 0);
                }
            }
        }
        pf.finish();
        areg.wait();

        if constexpr (KPARTS > 1 && !DUMP)
        {
            // the tile's wavefronts add their partial accumulators in wavefront order (kpart 0 + 1 + ..)
            __syncthreads(); // every wavefront is done with the step's LDS
            float *red = reinterpret_cast<float *>(smem); // [wavefront][16][64]
#pragma unroll
            for (int r = 0; r < 16; ++r)
                red[(wave * 16 + r) * 64 + lane] = acc[r];
            __syncthreads();
            if (kpart != 0)
                return;
#pragma unroll
            for (int p = 1; p < KPARTS; ++p)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[r] += red[((wave + 2 * MTILES * p) * 16 + r) * 64 + lane];
        }

        // ---- store: lane holds weight row n, 16 tokens -------------------------------------
        const long n = n0 + ntile * 32 + l32;
        if (!DUMP && n < g.w.N)
        {
#pragma unroll
            for (int r = 0; r < 16; ++r)
            {
                const long m = m0 + mtile * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
                if (m < g.M)
                    g.y[(size_t)m * g.ldy + n] = acc[r];
            }
        }
    }

    // ---- activations as they lie, a tile's K steps dealt to the wavefronts ------------------------
    // Tile of 32 MT tokens x 32 RN weight rows, a step of KS super-blocks, 2 KS RN = 8 wavefronts: wavefront (rn, kw) multiplies
    // half a super-block, the blocks of quad lanes 2 (kw % 2) and 2 (kw % 2) + 1, of rows 32 rn .. by all tokens of the tile, and
    // the 2 KS partial sums are added through LDS, always by the same twos.  Lane (r, h) decodes what quad lane h of the half decodes, two
    // whole blocks, and a swap of half registers between the lanes (r, 0) and (r, 1) makes both lanes' blocks into matrix operands.
    // The wavefront's raw weights come by way of LDS where it has room (HalfRows).  The Q8_1 blocks of the tokens go from memory
    // into LDS a step ahead, two buffers, one barrier a step: the quants as 16-byte pieces, [super-block][token][16], piece p of
    // token m at p ^ (m & 15) (so that reads of 16 tokens' pieces meet no bank twice), the heads {d, sum} as
    // [super-block][token][8], block k of token m at k ^ (m / 8 & 7).
    // The weights are the products' first operand, so a lane holds 16 rows' sums of one token: its scale is one register, the rows'
    // scales, copied into that layout by the matrix unit once for all tokens of the tile, are 16.  A block sum then costs two
    // multiply-adds (rescale below), where a subtraction, a multiply-add and a 32-bit matrix product for the pairs of scales took 352
    // cycles for two products, two wavefronts a SIMD unit: now 221 to 239 (products with 32-bit operands hold the vector unit up).
    // What bounds it: a step's time is the sum of what its two wavefronts a SIMD unit decode and rescale, as far as loads, swaps
    // and the first products do not add to it (step of 128 x 128, Q6_K: 6350 cycles; decoding 1000 and 16 products 1750 of each of the
    // two).  The older wavefront of the two is served first and waited at the barrier for a third of the step, so decoding goes
    // ahead of rescaling, and the younger's rescaling ahead of the older's.  One workgroup of eight wavefronts fits a compute unit.
    // Against a subtraction, a multiply-add and scales on the 32-bit matrix unit, weights straight into registers: 199 x 5120 x 25600
    // Q6_K 206 -> 136 to 146 us by card (tiles of 96 x 64; of 128 x 64 that walk is 194), 40 x 8192 x 5120 IQ3_S 20.0 -> 17.3, 512 x 25600 x 5120
    // Q4_K 270 -> 229 to 236 (gemm_kernel before; two launches now), 256 x 25600 x 5120 Q4_K 139 -> 132, 130 x 5000 x 5120 Q4_K 24.9 -> 22.5,
    // 63 x 5034 x 18944 Q6_K 71 -> 62 to 67.  Counters of 512 x 25600 x 5120: 242 cycles of a SIMD unit a product, the vector unit issues in 0.9
    // of them and the matrix unit works in 0.23.
    // Errors against 64 bits: 0.4 to 1.0 times those before (199 x 5120 x 25600 Q6_K 2.57e-7 -> 2.04e-7, 512 x 25600 x 5120 Q4_K 3.20e-7 ->
    // 1.55e-7, 40 x 8192 x 5120 IQ3_S 9.9e-8 -> 9.8e-8); 1.05 to 1.09 for the one size in 2000 that eight sums of block after block were
    // before and 96 x 64 is now (326 x 2709 x 24832 IQ3_S 1.86e-7 -> 2.03e-7, 145 -> 124 us).
    template <int MT, int RN, int KS>
    struct GemmSplit
    {
        static constexpr int BM = MT * 32, KW = 2 * KS, WAVES = RN * KW; // wavefronts along K, and of a workgroup
        static constexpr int QUANTS = KS * BM * 256, HEADS = KS * BM * 32; // bytes of a step
        static constexpr int QLOADS = QUANTS / 1024 / WAVES, HLOADS = HEADS / 256 / WAVES; // per wavefront
        static constexpr int QROWS = 4 * WAVES;                  // tokens x super-blocks that one load of every wavefront covers
        static constexpr int QM = BM > QROWS ? BM / QROWS : 1;   // tokens a lane loads pieces of
        static constexpr int HM = 8 * WAVES % BM == 0 ? 1 : BM % (8 * WAVES) == 0 ? BM / (8 * WAVES) : HLOADS; // tokens a lane loads heads of
        static_assert(QLOADS * WAVES * 1024 == QUANTS && HLOADS * WAVES * 256 == HEADS, "whole loads");
        static_assert(QROWS % 16 == 0 && (BM % QROWS == 0 || QROWS % BM == 0), "a lane's piece and tokens stay the same");
        static constexpr size_t STAGE = QUANTS + HEADS;
        static constexpr size_t SUMS = (size_t)KW * RN * MT * 16 * WAVE * sizeof(float);
        // with `half` bytes of raw weights a wavefront beside the activations, where there is room for them
        static constexpr bool raw_lds(size_t half) { return 2 * STAGE + WAVES * half + 6 * 1024 <= 160 * 1024; }
        static constexpr size_t lds(size_t half)
        {
            const size_t walk = 2 * STAGE + (raw_lds(half) ? WAVES * half : 0), end = SUMS + 4 * WAVES;
            return walk > end ? walk : end;
        }
    };

    // Block sums as floats without a conversion: the products start from the bits of 1.5 * 2^23 instead of zero, so that the bits of
    // their integer result are those of the float 1.5 * 2^23 + sum (sums stay within 32 * 128 * 128 = 2^19, a unit of the last
    // place is 1), and one subtraction leaves the sum, exactly.  Conversions and matrix instructions hold each other up: two
    // products with their rescaling take 308 cycles instead of 409, two wavefronts a SIMD unit.
    constexpr float BIAS = 12582912.0f;
    __device__ __forceinline__ v16i integer_bias()
    {
        v16i b;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            b[r] = __builtin_bit_cast(int, BIAS);
        asm volatile("" : "+v"(b)); // kept in registers: made anew for every product it would cost what it saves
        return b;
    }
    __device__ __forceinline__ float biased_to_float(int sum) { return __builtin_bit_cast(float, sum) - BIAS; }

    // BY_LDS: the raw weights come by way of LDS where there is room
    template <class F, int MT, int RN, int KS, bool DUMP, bool BY_LDS>
    __global__ void __launch_bounds__(RN * 2 * KS * WAVE) gemm_split_kernel(const GemmArgs g)
    {
        typedef typename F::Quad Q;
        typedef GemmSplit<MT, RN, KS> G;
        typedef int v2i_dword __attribute__((ext_vector_type(2), aligned(4)));
        constexpr int BM = G::BM, KW = G::KW;
        extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
        void *tab = format_tables_lds<F>();
        if (F::TABLE_BYTES > 0)
            F::stage_tables(tab);

        const int tid = threadIdx.x, lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int rn = wave % RN, kw = wave / RN;
        const int own_sb = kw >> 1, half = kw & 1; // of a step; of the super-block
        const int l32 = lane & 31, lh = lane >> 5;
        const long n0 = ((long)blockIdx.x * RN + rn) * 32 + (long)g.tile0 * GEMM_BN, m0 = (long)blockIdx.y * BM;
        const int SB = g.w.SB, KB = SB * 8;

        long n = n0 + l32;
        if (n >= g.w.N)
            n = g.w.N - 1; // tail rows: decode a valid row, never stored
        const typename Q::Lane lc = Q::lane_consts(lh + 2 * half);
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;
        // the weights, by way of LDS or, where the activations leave no room, straight into registers
        constexpr bool RAW_LDS = BY_LDS && G::raw_lds(Q::Half::BYTES);
        const typename Q::Cursor wc = Q::cursor(g.w, (size_t)n * SB, (size_t)n * SB, lc);
        typename Q::Half rows_half;
        if constexpr (RAW_LDS)
            rows_half.init(g.w, n0, half, lane);
        const uint32_t raw_at = (uint32_t)(2 * G::STAGE) + (uint32_t)(wave * Q::Half::BYTES);
        typename Q::Raw raw;
        auto issue_weights = [&](int sb) __attribute__((always_inline)) {
            const int at = sb < SB ? sb : SB - 1; // (past the end: the last super-block again)
            if constexpr (RAW_LDS)
                rows_half.load(lds0 + raw_at, at);
            else
                Q::load_at(raw, wc, lc, at);
        };
        auto wait_weights = [&]() __attribute__((always_inline)) {
            if constexpr (RAW_LDS)
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            else
                Q::template wait<0>(raw);
        };
        // bytes from the tile's first token to what this lane loads of super-block 0 (past the last token: the last one)
        const uint8_t *abase = reinterpret_cast<const uint8_t *>(g.q8 + (size_t)m0 * KB * 9);
        auto token = [&](int m) { return (uint32_t)(m0 + m < g.M ? m : g.M - 1 - m0) * (uint32_t)(KB * 36); };
        uint32_t qfrom[G::QM], hfrom[G::HM];
        {
            const int row = wave * 4 + (lane >> 4), p = (lane & 15) ^ (row & 15);
#pragma unroll
            for (int i = 0; i < G::QM; ++i)
                qfrom[i] = token((row + i * G::QROWS) % BM) + (uint32_t)((p >> 1) * 36 + 4 + (p & 1) * 16);
#pragma unroll
            for (int i = 0; i < G::HM; ++i)
            {
                const int group = (wave + i * G::WAVES) % (BM / 8);
                hfrom[i] = token(group * 8 + (lane >> 3)) + (uint32_t)((lane & 7) ^ (group & 7)) * 36;
            }
        }
        // Load i of the step of super-block sb0 (past the end: the last super-block); `lanes` are none where there is no such step (a
        // branch among the products would have the compiler copy their registers at its ends).
        constexpr int LOADS = G::QLOADS + G::HLOADS;
        auto issue_act = [&](int i, int sb0, int buf, uint64_t lanes) {
            const bool quants = i < G::QLOADS;
            const int h = i - G::QLOADS, part = KS == 1 ? 0 : quants ? (wave * 4 + i * G::QROWS) / BM : (wave + h * G::WAVES) / (BM / 8);
            const uint8_t *from = abase + (size_t)(sb0 + part < SB ? sb0 + part : SB - 1) * 288;
            const uint32_t to = lds0 + (uint32_t)(buf * (int)G::STAGE + (quants ? wave * 1024 + i * G::WAVES * 1024 : G::QUANTS + wave * 256 + h * G::WAVES * 256));
            if (quants)
                asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                             :: "s"(to), "v"(qfrom[i % G::QM]), "s"(from), "s"(lanes) : "memory");
            else
                asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dword %1, %2\n\ts_mov_b64 exec, -1"
                             :: "s"(to), "v"(hfrom[h % G::HM]), "s"(from), "s"(lanes) : "memory");
        };
        const v16i bias = integer_bias();
        v16f acc[MT], zero1f;
        v32f zero2f;
#pragma unroll
        for (int r = 0; r < 32; ++r)
            zero2f[r] = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            zero1f[r] = 0.0f;

        // The walk along K.  WHOLE: the sums as such, for tiles that hold something infinite or not a number.
        auto walk = [&](auto whole) __attribute__((always_inline)) {
        constexpr bool WHOLE = decltype(whole)::value;
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                acc[t][r] = 0.0f;
        int first = 0;
        asm volatile("" : "+s"(first)); // (addresses of both walks known ahead would fill the scalar registers)
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            issue_act(i, first, 0, ~0ull);
        issue_weights(own_sb);
        int buf = 0;
        for (int sb0 = 0; sb0 < SB; sb0 += KS, buf ^= 1)
        {
            const int sb = sb0 + own_sb;
            uint64_t more;
            asm("s_cmp_lt_i32 %1, %2\n\ts_cselect_b64 %0, -1, 0" : "=s"(more) : "s"(sb0 + KS), "s"(SB) : "scc");
            // this step's weights and activations have arrived, everybody is done with the other buffer
            wait_weights();
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_s_setprio(2);
            v4i w[4];
            typename Q::Scale S;
            if constexpr (RAW_LDS)
            {
                Q::Half::read(raw, smem + raw_at, l32, lh);
                Q::keep(raw);
                // (read, before they are asked for again; ahead of the decoding, to leave while it goes on)
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                issue_weights(sb + KS);
            }
            Q::decode(raw, lc, w, S);
            // decoded here, before the registers are asked for again: sunk below, the decoding would have the compiler copy
            // the raw words, and copies made ahead of the wait hold what the loads have not brought yet
            v2i_dword two = __builtin_bit_cast(v2i_dword, S);
            asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(two));
            S = __builtin_bit_cast(typename Q::Scale, two);
            __builtin_amdgcn_sched_barrier(0);
            // (the weights at once: they come from memory, and dealt out behind the products they were waited for)
            if constexpr (!RAW_LDS)
                issue_weights(sb + KS);
            __builtin_amdgcn_sched_barrier(0);
            if (sb < SB) // uniform in the wavefront
            {
                const uint8_t *rows = smem + buf * G::STAGE + (size_t)(own_sb * BM + l32) * 256;
                const uint32_t *heads = reinterpret_cast<const uint32_t *>(smem + buf * G::STAGE + G::QUANTS) + own_sb * 8 * BM + l32 * 8;
                // block x of the half's first quad lane, block y of its second: elements 0 .. 15 with lanes (r, 0), 16 .. 31 with (r, 1)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                    {
                        typedef uint32_t v2u __attribute__((ext_vector_type(2)));
                        const v2u s = __builtin_bit_cast(v2u, __builtin_amdgcn_permlane32_swap((uint32_t)w[2 * i][d], (uint32_t)w[2 * i + 1][d], false, false));
                        w[2 * i][d] = (int)s[0], w[2 * i + 1][d] = (int)s[1];
                    }
                // Product j: pair of blocks i_of(j) by tokens 32 t_of(j) ...  The matrix unit works on a product while the vector
                // unit rescales the one before it, and the LDS brings the operands of the next.
                constexpr int JOBS = 2 * MT, EACH = (LOADS + JOBS - 1) / JOBS;
                // (tokens by tokens, where the rows' scales of all four blocks fit the registers; else there and back, so that one tile of
                // tokens has its four blocks in a row)
                constexpr bool APART = KW < 8 && (MT > 1 || !F::HAS_MIN) && (MT < 4 || RAW_LDS), FOURS = APART && (MT == 1 || (MT == 2 && RAW_LDS));
                auto t_of = [](int j) { return FOURS ? j >> 1 : j < MT ? j : 2 * MT - 1 - j; };
                auto i_of = [](int j) { return FOURS ? j & 1 : j / MT; };
                // Sums of a job's two blocks that are added up by themselves (see rescale): with those of the job before, of the job after
                auto with_before = [](int j) { return APART && (FOURS ? j & 1 : j == MT); };
                auto with_after = [](int j) { return APART && (FOURS ? !(j & 1) : j == MT - 1); };
                // (of 128 x 128 as many as keep two sums as exact as four of block after block; of 96 x 64, which has four, those that cost
                // no addition more: with one more pair 199 x 5120 x 25600 Q6_K is 1.91e-7 instead of 2.04e-7 away, and 2 % slower)
                constexpr int APARTS = FOURS ? JOBS : KW == 2 ? (F::HAS_MIN ? MT + 2 : JOBS) : MT + 1;
                auto is_apart = [](int j) { return APART ? j < APARTS : MT == 4 && j >= MT; };
                auto fence = []() __attribute__((always_inline)) {
                    if (MT > 1) // (two products of a step are not enough for it: the compiler's order is 10 % faster)
                        __builtin_amdgcn_sched_barrier(0);
                };
                auto block = [&](int j, int which) { return Q::block_of(2 * half + which, i_of(j)); };
                auto quants = [&](int j, int which) {
                    return *reinterpret_cast<const v4i *>(rows + t_of(j) * 32 * 256 + (((2 * block(j, which) + lh) ^ (l32 & 15)) << 4));
                };
                auto head_of = [&](int j, int which) { return heads[(block(j, which) ^ ((t_of(j) & 1) * 4 + (l32 >> 3))) + t_of(j) * 256]; };
                // a block's scales of the rows that a lane's sums belong to: the matrix unit copies them there (times one: exact)
                auto scales = [&](int i, int which) {
                    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
                    const _Float16 none = (_Float16)0.0f;
                    const v4h own = {lh == which ? (_Float16)Q::scale_f32(S, i) : none, none, none, none};
                    const v4h one = {(_Float16)1.0f, none, none, none};
                    return __builtin_amdgcn_mfma_f32_32x32x8f16(own, one, zero1f, 0, 0, 0);
                };
                auto scales_of_both = [&](int i) {
                    typedef _Float16 v4h __attribute__((ext_vector_type(4)));
                    const _Float16 none = (_Float16)0.0f;
                    const v4h own = {(_Float16)Q::scale_f32(S, i), none, none, none}, one = {(_Float16)1.0f, none, none, none};
                    return __builtin_amdgcn_mfma_f32_32x32x4f16(own, one, zero2f, 0, 0, 0);
                };
                auto product = [&](int j, int which, v4i a) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(w[2 * i_of(j) + which], a, bias, 0, 0, 0); };
                auto dump = [&](int j, int which, const v16i &d) {
                    // (less than 2 GiB of sums: offsets of 32 bits, made anew for each, or they would fill the registers)
                    const int m = (int)m0 + t_of(j) * 32 + l32, nn = (int)(n0 - g.row0) + 4 * lh;
                    uint32_t at = ((uint32_t)m * (uint32_t)g.nrows + (uint32_t)nn) * (uint32_t)KB + (uint32_t)(sb * 8 + block(j, which));
                    if (m < g.M)
                    {
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                        {
                            const int row = 8 * (r >> 2) + (r & 3);
                            asm volatile("" : "+v"(at));
                            if (n0 + 4 * lh + row < g.w.N && nn + row >= 0 && nn + row < g.nrows)
                                g.sums[at + (uint32_t)row * (uint32_t)KB] = (int32_t)biased_to_float(d[r]);
                        }
                    }
                };
                // Two multiply-adds a sum: biased sum times the token's scale less bias times scale is the sum times the scale, rounded
                // once, and that times the row's scale.  Four blocks of a token, or two, are added up by themselves, their minima
                // among them, before they meet the sum of those before: 1 or 2 roundings at the size of the whole sum instead of 4, or 6
                // with minima.  Two partial sums are then no coarser than four of block after block: 232 x 16587 x 13312 Q6_K
                // 1.83e-7 from 64 bits (1.88e-7 by four such sums, 2.28e-7 with two blocks of four apart), Q4_K 2.42e-7 (2.58e-7, 3.38e-7),
                // at an addition to four or eight multiply-adds (1 to 3 % of 128 x 128).  Eight partial sums need it not,
                // 128 x 64 has registers for the second pairs only, and one token tile's with minima stay as they were (17 x 8370 x
                // 18944 Q4_K 51.1 us and 2.95e-7, or 53.7 and 1.26e-7).
                v16f apart;
                auto rescale = [&](int j, int which, const v16i &d, uint32_t head, const v16f &cs) __attribute__((always_inline)) {
                    typedef float v2f __attribute__((ext_vector_type(2)));
                    typedef float v8f __attribute__((ext_vector_type(8)));
                    const int t = t_of(j);
                    const bool start = which == 0 && !with_before(j), last = which == 1 && !with_after(j);
                    v2f da; // {scale, offset}
                    da[0] = h2f((uint16_t)(head & 0xFFFFu));
                    da[1] = -BIAS * da[0];
                    if (!WHOLE)
                        asm("" : "+v"(da)); // (floats from here on: v_fma_mix_f32, which would read the half, takes twice as long)
#pragma unroll
                    for (int r = 0; r < 16; r += 8)
                    {
                        v8f s; // (that of row r + i in place i ^ 1: an instruction waits for three operands of even, or three of odd registers)
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                            s[i ^ 1] = WHOLE ? biased_to_float(d[r + i]) : fmaf(__int_as_float(d[r + i]), da[0], da[1]);
                        if (!WHOLE)
                            asm("" : "+v"(s));
#pragma unroll
                        for (int i = 0; i < 8; ++i)
                        {
                            const float c = WHOLE ? da[0] * cs[r + i] : cs[r + i];
                            if (!is_apart(j))
                                acc[t][r + i] = fmaf(s[i ^ 1], c, acc[t][r + i]);
                            else if (start)
                                apart[r + i] = s[i ^ 1] * c;
                            else if (!last)
                                apart[r + i] = fmaf(s[i ^ 1], c, apart[r + i]);
                            else
                                acc[t][r + i] += fmaf(s[i ^ 1], c, apart[r + i]);
                        }
                    }
                };
                // Minima times the tokens' scaled sums.  The matrix unit's 32-bit products hold the vector unit up for all of their 64
                // cycles; of bf16 it does 16 in 32, so three pieces of a sum that add up to it (24 bits) times the two of a minimum (11).
                constexpr bool PIECES = !WHOLE && (MT > 1 || KW == 8); // (in walks of one token tile and four or fewer sums their making would take longer)
                v4i low[2];
                if constexpr (F::HAS_MIN && PIECES)
#pragma unroll
                    for (int i = 0; i < 2; ++i)
                    {
                        const float m = Q::min_f32(S, i), m1 = __uint_as_float(and_k<0xFFFF0000u>(__float_as_uint(m))), m2 = m - m1;
                        const uint32_t u1 = __float_as_uint(m1), u2 = __float_as_uint(m2);
                        low[i] = (v4i){(int)(u1 | u1 >> 16), (int)(u2 | u2 >> 16), (int)u1, (int)u2};
                    }
                const uint32_t upper = vector_constant(lh ? ~0u : 0u);
                auto add_minima = [&](int j, uint32_t x, uint32_t y) __attribute__((always_inline)) {
                    const uint32_t h = bit_select(y, x, upper);
                    const float sum = (float)(int16_t)(h >> 16) * h2f((uint16_t)(h & 0xFFFFu));
                    if constexpr (!PIECES)
                        acc[t_of(j)] = __builtin_amdgcn_mfma_f32_32x32x2f32(Q::min_f32(S, i_of(j)), sum, acc[t_of(j)], 0, 0, 0);
                    else
                    {
                        typedef __bf16 v8b __attribute__((ext_vector_type(8)));
                        const float p1 = __uint_as_float(and_k<0xFFFF0000u>(__float_as_uint(sum))), rest = sum - p1;
                        const float p2 = __uint_as_float(and_k<0xFFFF0000u>(__float_as_uint(rest))), p3 = rest - p2;
                        const int both = (int)__builtin_amdgcn_perm(__float_as_uint(p2), __float_as_uint(p1), 0x07060302u);
                        // slots p1 p2 p1 p2 0 p3 0 p3 of the block of either half of the lanes, times m1 m1 m2 m2 0 m1 0 m2
                        v16f &to = is_apart(j) ? apart : acc[t_of(j)];
                        const v4i pieces = {both, both, __float_as_int(p3), __float_as_int(p3)};
                        to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8b, low[i_of(j)]), __builtin_bit_cast(v8b, pieces), to, 0, 0, 0);
                    }
                };
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    if (!DUMP)
                        asm("" : "+v"(acc[t]));
                v16f cs[4];
                auto scales_of_pair = [&](int i) {
                    const v32f both = scales_of_both(i);
                    cs[2 * i] = __builtin_shufflevector(both, both, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15);
                    cs[2 * i + 1] = __builtin_shufflevector(both, both, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31);
                };
                constexpr bool LATER = MT == 1 && KW < 8; // (the second pair's scales beside the first pair's products: 388 x 1157 x 18688 Q4_K 51.8 -> 49.9 us)
                if constexpr (MT <= 2)
                {
                    scales_of_pair(0);
                    if (!LATER)
                        scales_of_pair(1);
                }
                else
                    cs[0] = scales(0, 0), cs[1] = scales(0, 1);
                uint32_t hx = head_of(0, 0), hy = head_of(0, 1);
                v16i dx = product(0, 0, quants(0, 0)), dy = product(0, 1, quants(0, 1));
                // (of one and two token tiles, too: 12 x 1483 x 20992 Q6_K 40.4 -> 35.8 us)
                if (wave >= G::WAVES / 2)
                    __builtin_amdgcn_s_setprio(1);
                else
                    __builtin_amdgcn_s_setprio(0);
#pragma unroll
                for (int j = 0; j < JOBS; ++j)
                {
                    v4i a, b;
                    uint32_t nx = 0, ny = 0;
                    fence();
                    if (j + 1 < JOBS)
                    {
                        nx = head_of(j + 1, 0), ny = head_of(j + 1, 1);
                        a = quants(j + 1, 0), b = quants(j + 1, 1);
                    }
                    fence();
#pragma unroll
                    for (int i = j * EACH; i < (j + 1) * EACH; ++i)
                        if (i < LOADS)
                            issue_act(i, sb0 + KS, buf ^ 1, more);
                    fence();
                    if (DUMP)
                        dump(j, 0, dx);
                    else
                        rescale(j, 0, dx, hx, cs[2 * i_of(j)]);
                    fence();
                    if (j + 1 < JOBS)
                        dx = product(j + 1, 0, a);
                    if (LATER && j == 0)
                        scales_of_pair(1);
                    if (MT > 2 && j + 1 == MT)
                        cs[2] = scales(1, 0);
                    if (F::HAS_MIN && !DUMP && is_apart(j))
                        add_minima(j, hx, hy);
                    fence();
                    if (DUMP)
                        dump(j, 1, dy);
                    else
                        rescale(j, 1, dy, hy, cs[2 * i_of(j) + 1]);
                    fence();
                    if (j + 1 < JOBS)
                        dy = product(j + 1, 1, b);
                    if (MT > 2 && j + 1 == MT)
                        cs[3] = scales(1, 1);
                    if (F::HAS_MIN && !DUMP && !is_apart(j))
                        add_minima(j, hx, hy);
                    hx = nx, hy = ny;
                }
            }
        }
        wait_weights();
        };
        walk(std::integral_constant<bool, DUMP>());
        if (DUMP)
            return;

        // The KW partial sums of a place are added by twos, by all wavefronts: wavefront kw adds and stores the kw-th part of
        // its tile's registers.
        constexpr int SHARE = MT * 16 / KW, AT_ONCE = SHARE < 4 ? SHARE : 4;
        float *red = reinterpret_cast<float *>(smem) + rn * MT * 16 * WAVE + lane;
        int *odd = reinterpret_cast<int *>(smem + G::SUMS);
        auto gather = [&]() __attribute__((always_inline)) {
            float finite = 0.0f;
            __syncthreads(); // everybody is done with the activations
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                {
                    finite = fmaf(acc[t][r], 0.0f, finite);
                    red[(kw * RN * MT * 16 + t * 16 + r) * WAVE] = acc[t][r];
                }
            const bool own = __any(!(finite == 0.0f));
            if (lane == 0)
                odd[wave] = own;
            __syncthreads();
            int any = 0;
            for (int i = 0; i < G::WAVES; ++i)
                any |= odd[i];
            return __builtin_amdgcn_readfirstlane(any) != 0;
        };
        // a lane holds a token's sums of rows 8 k + 4 lh .. + 3
        typedef float vf_dword __attribute__((ext_vector_type(AT_ONCE), aligned(4)));
        // again: after the second walk, whose sums are rounded otherwise.  What was finite stays (nothing else of its token or row was
        // infinite then), so that no element depends on another one's infinity.
        auto store = [&](auto again) __attribute__((always_inline)) {
            int row_base = (int)n0, l = lane;
            asm volatile("" : "+s"(row_base), "+v"(l)); // (addresses made anew: kept over the second walk they would fill the registers)
            const float *sums = reinterpret_cast<const float *>(smem) + rn * MT * 16 * WAVE + l;
#pragma unroll
            for (int q = 0; q < SHARE; q += AT_ONCE)
            {
                const int reg = kw * SHARE + q, r = reg & 15; // uniform
                const long m = m0 + (reg >> 4) * 32 + (l & 31);
                vf_dword sum;
#pragma unroll
                for (int i = 0; i < AT_ONCE; ++i)
                {
                    float part[KW];
#pragma unroll
                    for (int k = 0; k < KW; ++k)
                        part[k] = sums[(k * RN * MT * 16 + reg + i) * WAVE];
#pragma unroll
                    for (int k = 1; k < KW; k *= 2)
#pragma unroll
                        for (int l = 0; l < KW; l += 2 * k)
                            part[l] += part[l + k];
                    sum[i] = part[0];
                }
                const long at = row_base + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3), left = g.w.N - at;
                if (m < g.M && left > 0)
                {
                    float *y = g.y + (size_t)m * g.ldy + at;
                    if (decltype(again)::value)
#pragma unroll
                        for (int i = 0; i < AT_ONCE; ++i)
                            if (i < left && __builtin_isfinite(y[i]))
                                sum[i] = y[i];
                    if (left >= AT_ONCE)
                        *reinterpret_cast<vf_dword *>(y) = sum;
                    else
#pragma unroll
                        for (int i = 0; i < AT_ONCE - 1; ++i)
                            if (i < left)
                                y[i] = sum[i];
                }
            }
        };
        const bool any_odd = gather();
        store(std::false_type());
        if (__builtin_expect(any_odd, 0))
        {
            __syncthreads();
            walk(std::true_type());
            gather();
            store(std::true_type());
        }
    }

    __global__ void __launch_bounds__(256)
        epilogue_kernel(float *__restrict__ c, const float *__restrict__ t, const float *__restrict__ bias,
                        long M, int N, int ldc, float alpha, float beta)
    {
        const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
        if (i >= M * N)
            return;
        const long m = i / N;
        const int n = (int)(i - m * N);
        float *dst = c + m * ldc + n;
        float v = (beta == 0.0f) ? 0.0f : beta * *dst;
        v += alpha * t[i];
        if (bias)
            v += bias[n];
        *dst = v;
    }

    template <class F, bool DUMP, int BM>
    bool gemm_launch_bm(const char *fn, const GemmArgs &g, int tiles_n, int M, hipStream_t st)
    {
        constexpr size_t lds = gemm_lds_bytes<F, BM>();
        static_assert(lds >= (size_t)8 * 16 * 64 * sizeof(float), "room for the partial accumulators");
        static LdsGrant grant;
        const hipError_t e = allow_lds(grant, reinterpret_cast<const void *>(&gemm_kernel<F, DUMP, BM>), lds);
        if (e != hipSuccess)
            return fail(fn, "cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        const dim3 grid((unsigned)tiles_n, (unsigned)((M + BM - 1) / BM));
        hipLaunchKernelGGL((gemm_kernel<F, DUMP, BM>), grid, dim3(GEMM_THREADS), lds, st, g);
        return launched(fn);
    }

    template <class F, bool DUMP, int MT, int RN, int KS, bool BY_LDS = true>
    bool gemm_split_launch(const char *fn, const GemmArgs &g, int rows, int M, hipStream_t st)
    {
        constexpr size_t lds = GemmSplit<MT, RN, KS>::lds(F::Quad::Half::BYTES);
        static_assert(lds + 6 * 1024 <= 160 * 1024, "LDS, with the decoders' tables");
        static LdsGrant grant;
        const auto kernel = &gemm_split_kernel<F, MT, RN, KS, DUMP, BY_LDS>;
        const hipError_t e = allow_lds(grant, reinterpret_cast<const void *>(kernel), lds);
        if (e != hipSuccess)
            return fail(fn, "cannot reserve %zu bytes of LDS: %s", lds, hipGetErrorString(e));
        hipLaunchKernelGGL(kernel, dim3((unsigned)((rows + 32 * RN - 1) / (32 * RN)), (unsigned)((M + 32 * MT - 1) / (32 * MT))),
                           dim3(RN * 2 * KS * WAVE), lds, st, g);
        return launched(fn);
    }

    // Which kernel a shape takes: -1 for gemm_kernel, or an entry of SPLIT.  gemm_kernel's workgroup walks the whole of K
    // alone, two of them on a compute unit; gemm_split_kernel has one there and gives the walk to 2, 4 or 8 wavefronts.
    // The expected times in microseconds are fitted to measurements, weights from memory (us, gemm_kernel and the entries):
    //   tokens x rows x K             gemm_kernel  0: 1,1,4  1: 1,2,2  2: 2,1,4  3: 2,2,2  4: 2,4,1  5: 3,2,2  6: 4,4,1  7: 4,2,2
    //   10 x 4096 x 4096, Q4_K           19.0      8.8     12.8     12.5     17.9     30.1     24.0     50.2     28.5
    //   64 x 4096 x 4096, IQ3_S          33.1     11.3     16.5     15.5     20.1     34.4     25.1     50.0     31.5
    //   20 x 12000 x 4096, IQ3_S         24.9     19.5     16.8     27.2     20.4     34.3     25.6     49.4     31.9
    //   40 x 8192 x 5120, IQ3_S          41.1     23.8     20.8     18.0     24.2     42.2     30.8     61.7     39.2
    //   63 x 5034 x 18944, Q6_K           165     77.8     74.9     67.0     92.2      155      109      219      146
    //   130 x 5000 x 5120, Q4_K          52.0     38.9     32.4     30.0     23.6     37.3     29.8     61.7     35.6
    //   64 x 25600 x 5120, Q4_K          53.7     72.0     64.1     61.6     45.7     40.4     59.6     64.4     73.0
    //   80 x 9762 x 3072, Q6_K           39.9     34.3     28.9     36.6     31.9     30.2     22.9     41.5     30.0
    //   199 x 5120 x 25600, Q6_K          295      238      249      229      204      209      139      296      194
    //   256 x 8192 x 8192, Q4_K          87.0      122     96.7     94.9     67.9     62.9     89.9     96.7     62.9
    //   1000 x 4096 x 4096, Q4_K         66.5      129     99.5     97.6     71.7     64.4     74.3     58.8     64.2
    //   256 x 25600 x 5120, Q4_K          152      246      203      193      152      153      149      136      146
    //   16 x 25600 x 5120, Q6_K          49.9     51.2     46.5     73.5     55.1     51.9     66.2     69.4     86.0
    //   384 x 25600 x 5120, Q4_K          198      374      296      279      216      191      213      200      184
    //   512 x 25600 x 5120, Q4_K          264      491      389      368      282      267      295      268      254
    //   2048 x 6400 x 5120, IQ3_S         265      508      465      359      296      293      270      263      259
    // Tiles that fill their last round exactly, one round or several (us, gemm_kernel and the entry that is taken; Q4_K, Q6_K, IQ3_S):
    //   1024 x 4096 x 4096     66.8, 75.9, 66.8 -> 58.8, 58.9, 57.0 (6)
    //   512 x 16384 x 4096     128.2, 147.5, 130.3 -> 114.3, 115.4, 112.0 (6)
    //   512 x 8192 x 12800     197.4, 229.9, 199.7 -> 166.2, 167.5, 161.7 (6)
    //   40 x 32768 x 1024      14.8, 18.1, 16.0 -> 13.1, 15.5, 13.9 (4)
    //   2048 x 4096 x 2048     67.5, 75.0, 67.5 -> 63.6, 62.7, 62.1 (6)
    //   1024 x 8192 x 2048     66.4, 75.2, 66.9 -> 63.2, 63.4, 61.6 (6)
    //   64 x 32768 x 2048      26.0, 32.5, 28.1 -> 21.2, 26.3, 23.3 (4)
    // and gemm_kernel's (us, gemm_kernel and the entry that would come next):
    //   1000 x 4096 x 512      12.6, 13.4, 12.5 : 14.2, 13.9, 14.0 (6)
    struct SplitTile
    {
        int mt, rn, ks;
        double step[3]; // microseconds: a step (KS super-blocks) of Q4_K, Q6_K and IQ3_S
    };
    constexpr SplitTile SPLIT[] = {
        {1, 1, 4, {1.7, 1.85, 1.75}}, {1, 2, 2, {1.45, 1.8, 1.68}}, {2, 1, 4, {2.25, 2.9, 2.9}}, {2, 2, 2, {1.85, 2.2, 2.07}},
        {2, 4, 1, {1.65, 2.15, 1.95}}, {3, 2, 2, {2.5, 2.6, 2.7}}, {4, 4, 1, {3.2, 3.3, 2.9}},
        {4, 2, 2, {3.75, 4.15, 3.6}}}; // (the last one's activations leave the weights no room in LDS)
    constexpr int SPLITS = (int)(sizeof(SPLIT) / sizeof(SPLIT[0]));
    constexpr double SPLIT_START = 3.5, WHOLE_START = 2.0; // a workgroup's start and end
    inline double split_expected(const SplitTile &t, int format, int M, int N, int K, int cus)
    {
        const auto over = [](long a, long b) { return (a + b - 1) / b; };
        const long groups = over(N, 32 * t.rn) * over(M, 32 * t.mt), left = groups % cus;
        const double round = (double)over(K / 256, t.ks) * t.step[format] + SPLIT_START;
        // A last round of few workgroups is faster, for they have the memory and the clock to themselves: of a tenth of the chip by 8 % in
        // rounds of up to 10 us, by a quarter from 40 us on.  (Second rounds of 26 and of 128 workgroups, as shares of whole ones: entry 0, Q4_K,
        // 5 us 0.91 and 0.86, 18 us 0.90, 0.87; entry 1, Q6_K, 8 us 0.90, 0.87, 19 us 0.78, 0.75; entry 3, Q4_K, 12 us 0.93, 0.92, 35 us 0.86,
        // 0.90; entry 6, Q4_K, 22 us 0.76, 0.76, 60 us 0.78, 0.83; Q6_K, 35 us 0.68, 0.73; entry 7, Q4_K, 14 us 0.87, 0.85, 50 us 0.81, 0.82.)
        const double lighter = 0.08 + 0.17 * (round < 10 ? 0.0 : round > 40 ? 1.0 : (round - 10) / 30);
        const double last = left == 0 ? 0.0 : 1.0 - lighter * (1.0 - (double)left / cus);
        return (groups <= cus ? 1.0 : (double)(groups / cus) + last) * round;
    }
    // gemm_kernel: microseconds a super-block of a tile of 32, 64 or 128 tokens takes in a round of two workgroups a compute unit
    // that others follow, in the last round, and in a last round of one
    struct WholeTile
    {
        int tokens;
        double full[3], last[3], alone[3];
    };
    constexpr WholeTile WHOLE[] = {{32, {1.4, 2.2, 1.9}, {1.6, 2.5, 2.2}, {1.2, 1.5, 1.4}},
                                   {64, {2.4, 3.1, 2.65}, {2.7, 3.6, 3.05}, {1.65, 2.2, 1.9}},
                                   {GEMM_BM, {3.55, 3.95, 3.55}, {4.2, 4.8, 4.35}, {2.6, 3.0, 2.8}}};

    inline int gemm_split_choice(int format, int M, int N, int K, int cus, double *expected = nullptr)
    {
        if (expected)
            *expected = 1e30;
        if (K > 1 << 24) // 32-bit offsets from a tile's first token
            return -1;
        const auto over = [](long a, long b) { return (a + b - 1) / b; };
        const int SB = K / 256;
        const WholeTile &whole = WHOLE[M <= 32 ? 0 : M <= 64 ? 1 : 2];
        const long tiles = over(N, GEMM_BN) * over(M, whole.tokens), rounds_before = (tiles - 1) / (2 * cus), rest = tiles - rounds_before * 2 * cus;
        // (a last round that is exactly full is a last round all the same; but tiles of 32 tokens fare better in it, and the entry of
        // the largest tiles, which alone rivals full rounds of 128 tokens, starts too slowly for walks of four super-blocks and less)
        const bool light = rest == 2 * cus && (M <= 32 || (M > 64 && SB <= 4));
        const double *last = rest <= cus ? whole.alone : light ? whole.full : whole.last;
        const double undivided = WHOLE_START + SB * ((double)rounds_before * whole.full[format] + last[format]);
        double best = 0.97 * undivided;
        int choice = -1;
        for (int i = 0; i < SPLITS; ++i)
        {
            const SplitTile &t = SPLIT[i];
            if (over(M, 32 * t.mt) > 65535) // (the grid's second extent)
                continue;
            const double us = split_expected(t, format, M, N, K, cus);
            if (us < best)
                best = us, choice = i;
        }
        if (expected)
            *expected = choice < 0 ? undivided : best;
        return choice;
    }

    // A launch whose last round of tiles is sparse does better as two: the rows whose tiles fill whole rounds by themselves (a
    // multiple of 64), and the rest, as tiles that fit it.  The second waits for the first to end and starts anew: GEMM_SECOND
    // microseconds, and only where a twentieth is gained.
    // Measured, one launch and two: 512 x 25600 x 5120 Q4_K 260 -> 227 us, Q6_K 263 -> 229, 2048 x 6400 x 5120 Q4_K 262 -> 222, 82 x 19449 x 19968
    // Q4_K 210 -> 164, 384 x 25600 x 5120 IQ3_S 193 -> 169, 37 x 17420 x 7680 Q6_K 78.3 -> 60.3, 101 x 17640 x 3328 Q4_K 43.8 -> 36.9.
    constexpr double GEMM_SECOND = 3.0;
    struct GemmPlan
    {
        int choice, first, rest; // weight rows [0, first) by `choice`, the others by `rest`; first = 0: all by `choice`
    };
    inline GemmPlan gemm_plan(int format, int M, int N, int K, int cus)
    {
        const auto over = [](long a, long b) { return (a + b - 1) / b; };
        const int SB = K / 256;
        double whole;
        GemmPlan plan = {gemm_split_choice(format, M, N, K, cus, &whole), 0, -1};
        if (K > 1 << 24)
            return plan;
        double best = 0.95 * whole;
        for (int i = 0; i < SPLITS; ++i)
        {
            const SplitTile &t = SPLIT[i];
            const long across = over(M, 32 * t.mt), rounds = over(N, 32 * t.rn) * across / cus;
            const int first = (int)(rounds * cus / across * 32 * t.rn) & ~63;
            if (first < 64 || first >= N || across > 65535)
                continue;
            double after;
            const int rest = gemm_split_choice(format, M, N - first, K, cus, &after);
            const double us = (double)rounds * ((double)over(SB, t.ks) * t.step[format] + SPLIT_START) + GEMM_SECOND + after;
            if (us < best)
                best = us, plan = {i, first, rest};
        }
        return plan;
    }

    // weight rows from 64 g.tile0 up to rows_end, by the kernel of gemm_plan's answer
    template <class F, bool DUMP>
    bool gemm_launch_rows(const char *fn, const GemmArgs &g, int choice, int rows_end, int M, hipStream_t st)
    {
        const int rows = rows_end - g.tile0 * GEMM_BN, tiles = (rows + GEMM_BN - 1) / GEMM_BN;
        switch (choice)
        {
        case 0: return gemm_split_launch<F, DUMP, 1, 1, 4>(fn, g, rows, M, st);
        case 1:
            // Q4_K weights of several token tiles come from the cache but for the first time, and straight into registers is the shorter
            // way (us, by LDS and straight: 388 x 1157 x 18688 51.7 and 49.9, 138 x 3037 x 11264 32.5 and 32.1; 14 x 12406 x 18432 51.4 and
            // 59.9, 16 x 16000 x 8192 27.0 and 29.3)
            if (F::HAS_MIN && M > 32)
                return gemm_split_launch<F, DUMP, 1, 2, 2, !F::HAS_MIN>(fn, g, rows, M, st);
            return gemm_split_launch<F, DUMP, 1, 2, 2>(fn, g, rows, M, st);
        case 2: return gemm_split_launch<F, DUMP, 2, 1, 4>(fn, g, rows, M, st);
        case 3: return gemm_split_launch<F, DUMP, 2, 2, 2>(fn, g, rows, M, st);
        case 4: return gemm_split_launch<F, DUMP, 2, 4, 1>(fn, g, rows, M, st);
        case 5: return gemm_split_launch<F, DUMP, 3, 2, 2>(fn, g, rows, M, st);
        case 6: return gemm_split_launch<F, DUMP, 4, 4, 1>(fn, g, rows, M, st);
        case 7: return gemm_split_launch<F, DUMP, 4, 2, 2>(fn, g, rows, M, st);
        default: break;
        }
        // few tokens: one smaller tile of tokens (a 128-token tile would rescale 128 rows for them)
        if (M <= 32)
            return gemm_launch_bm<F, DUMP, 32>(fn, g, tiles, M, st);
        if (M <= 64)
            return gemm_launch_bm<F, DUMP, 64>(fn, g, tiles, M, st);
        return gemm_launch_bm<F, DUMP, GEMM_BM>(fn, g, tiles, M, st);
    }

    // d_sums: the block-sum variant of the same launches over weight rows [row0, row0+nrows); only the workgroups
    // whose rows meet the window are launched.
    template <class F, bool DUMP = false>
    bool gemm_launch(const char *fn, const void *d_w, const void *d_q8, float *d_y, int M, int N, int K, int ldy,
                     int device_id, hipStream_t st, int32_t *d_sums = nullptr, int row0 = 0, int nrows = 0)
    {
        GemmArgs g;
        g.w = GemvArgs{};
        g.w.w = d_w;
        g.w.N = N;
        g.w.SB = K / 256;
        g.q8 = static_cast<const uint32_t *>(d_q8);
        g.y = d_y;
        g.M = M;
        g.ldy = ldy;
        g.sums = d_sums;
        g.row0 = row0;
        g.nrows = nrows;
        // (the quad-lane decoders address a matrix through 32-bit offsets)
        if constexpr (F::USE_QUAD)
        {
            if (!F::Quad::addressable(N, K / 256))
                return fail(fn, "matrix too large for the kernel's 32-bit offsets (N=%d K=%d)", N, K);
        }
        constexpr int format = F::HAS_MIN ? 0 : F::TABLE_BYTES > 0 ? 2 : 1; // Q4_K, Q6_K, IQ3_S
        const GemmPlan plan = gemm_plan(format, M, N, K, cu_count(device_id));
        // weight rows from `from` to `to`, as far as they are wanted
        const auto part = [&](int choice, int from, int to) {
            const int low = DUMP && row0 > from ? row0 : from, high = DUMP && row0 + nrows < to ? row0 + nrows : to;
            if (low >= high)
                return true;
            const int tile = choice < 0 || SPLIT[choice].rn < 2 ? GEMM_BN : 32 * SPLIT[choice].rn;
            g.tile0 = (from + (low - from) / tile * tile) / GEMM_BN;
            return gemm_launch_rows<F, DUMP>(fn, g, choice, high, M, st);
        };
        return part(plan.choice, 0, plan.first > 0 ? plan.first : N) && (plan.first == 0 || part(plan.rest, plan.first, N));
    }
} // namespace llamql

extern "C" bool llam_ql_gemm(uint8_t fmt, const void *d_w, const void *d_q8, float *d_y,
                             int M, int N, int K, int ldy, int device_id, void *stream)
{
    using namespace llamql;
    static const char *fn = "llam_ql_gemm";
    if (fmt != LLAM_FMT_Q4_K && fmt != LLAM_FMT_Q6_K && fmt != LLAM_FMT_IQ3_S)
        return fail(fn, "unsupported weight format id %d", (int)fmt);
    if (M < 0)
        return fail(fn, "negative M");
    if (M == 0)
        return true;
    if (N < 1 || K < 1 || (K % 256) != 0)
        return fail(fn, "need N >= 1 and K a positive multiple of 256 (N=%d K=%d)", N, K);
    if (!d_w || !d_q8 || !d_y)
        return fail(fn, "null pointer");
    if (!aligned16(d_w) || !aligned4(d_q8))
        return fail(fn, "d_w must be 16-byte and d_q8 4-byte aligned");
    if (ldy < N)
        return fail(fn, "ldy=%d smaller than N=%d", ldy, N);
    if ((M + GEMM_BM - 1) / GEMM_BM > 65535)
        return fail(fn, "M=%d too large for one launch", M);
    if (!set_device(fn, device_id))
        return false;
    hipStream_t st = as_stream(stream);
    switch (fmt)
    {
    case LLAM_FMT_Q4_K: return gemm_launch<Q4KTraits>(fn, d_w, d_q8, d_y, M, N, K, ldy, device_id, st);
    case LLAM_FMT_Q6_K: return gemm_launch<Q6KTraits>(fn, d_w, d_q8, d_y, M, N, K, ldy, device_id, st);
    default: return gemm_launch<IQ3STraits>(fn, d_w, d_q8, d_y, M, N, K, ldy, device_id, st);
    }
}

extern "C" bool llam_ql_gemm_block_sums(uint8_t fmt, const void *d_w, const void *d_q8, int32_t *d_sums,
                                        int M, int N, int K, int row0, int nrows, int device_id, void *stream)
{
    using namespace llamql;
    static const char *fn = "llam_ql_gemm_block_sums";
    if (fmt != LLAM_FMT_Q4_K && fmt != LLAM_FMT_Q6_K && fmt != LLAM_FMT_IQ3_S)
        return fail(fn, "unsupported weight format id %d", (int)fmt);
    if (M < 1 || N < 1 || K < 1 || (K % 256) != 0)
        return fail(fn, "need M, N >= 1 and K a positive multiple of 256 (M=%d N=%d K=%d)", M, N, K);
    if (!d_w || !d_q8 || !d_sums)
        return fail(fn, "null pointer");
    if (!aligned16(d_w) || !aligned4(d_q8) || !aligned4(d_sums))
        return fail(fn, "d_w must be 16-byte, d_q8 and d_sums 4-byte aligned");
    if (row0 < 0 || nrows < 1 || (long)row0 + nrows > N)
        return fail(fn, "row window [%d,%d) outside [0,%d)", row0, row0 + nrows, N);
    if ((M + GEMM_BM - 1) / GEMM_BM > 65535)
        return fail(fn, "M=%d too large for one launch", M);
    if ((size_t)M * (size_t)nrows * (size_t)(K / 32) * sizeof(int32_t) >= ((size_t)1 << 31))
        return fail(fn, "M=%d x %d rows x %d blocks of sums exceed 2 GiB", M, nrows, K / 32);
    if (!set_device(fn, device_id))
        return false;
    hipStream_t st = as_stream(stream);
    switch (fmt)
    {
    case LLAM_FMT_Q4_K: return gemm_launch<Q4KTraits, true>(fn, d_w, d_q8, nullptr, M, N, K, 0, device_id, st, d_sums, row0, nrows);
    case LLAM_FMT_Q6_K: return gemm_launch<Q6KTraits, true>(fn, d_w, d_q8, nullptr, M, N, K, 0, device_id, st, d_sums, row0, nrows);
    default: return gemm_launch<IQ3STraits, true>(fn, d_w, d_q8, nullptr, M, N, K, 0, device_id, st, d_sums, row0, nrows);
    }
}

extern "C" bool llam_ql_epilogue(float *d_c, const float *d_t, const float *d_bias, int M,
                                 int N, int ldc, float alpha, float beta, int device_id,
                                 void *stream)
{
    using namespace llamql;
    static const char *fn = "llam_ql_epilogue";
    if (M < 0 || N < 0)
        return fail(fn, "negative size");
    if (M == 0 || N == 0)
        return true;
    if (!d_c || !d_t)
        return fail(fn, "null pointer");
    if (ldc < N)
        return fail(fn, "ldc=%d smaller than N=%d", ldc, N);
    if (!set_device(fn, device_id))
        return false;
    const long total = (long)M * N;
    const long grid = (total + 255) / 256;
    if (grid > 0x7FFFFFFFL)
        return fail(fn, "problem too large");
    hipLaunchKernelGGL(epilogue_kernel, dim3((unsigned)grid), dim3(256), 0, as_stream(stream), d_c, d_t, d_bias,
                       (long)M, N, ldc, alpha, beta);
    return launched(fn);
}
