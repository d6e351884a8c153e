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
        int tile0; // first 64-row tile of the launch (0 unless DUMP)
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
    // the 2 KS partial sums are added through LDS in their order.  The weights never pass through LDS: lane (r, h) decodes
    // what quad lane h of the half decodes, two whole blocks, and a swap of half registers between the lanes (r, 0) and (r, 1)
    // makes both lanes' blocks into matrix operands.  The Q8_1 blocks of the tokens go from memory into LDS a step ahead, two
    // buffers, one barrier a step: the quants as 16-byte pieces, [super-block][token][16], piece p of token m at p ^ (m & 15)
    // (so that reads of 16 tokens' pieces meet no bank twice), the heads {d, sum} as [super-block][8 tokens][block][8], block k
    // of the group of tokens g at k ^ (g & 7): a load of 64 heads reads 8 tokens' whole super-blocks, 24 cache lines, where a
    // block of 64 tokens would read 64.
    // What bounds it: the address unit of the loads (5000 of 11000 cycles a step when every lane's head was a line of its own and
    // all loads were issued together, the wavefronts standing still meanwhile), then the vector unit: rescaling and decoding.  So
    // the loads are dealt out among the products, a wavefront takes half a super-block of twice the tokens (half the decoding and
    // half the loads of weights a product), and the matrix unit works on a product while the vector unit rescales the one before.
    // One workgroup of eight wavefronts fits a compute unit (up to 250 registers a lane).
    // Against whole super-blocks a wavefront and loads together: 199 x 5120 x 25600 Q6_K 272 -> 207 us, 40 x 8192 x 5120 IQ3_S
    // 23.3 -> 19.0, 256 x 8192 x 8192 Q4_K 79 -> 65, 63 x 5034 x 18944 Q6_K 93 -> 70.5, 130 x 5000 x 5120 Q4_K 29.2 -> 26.7.
    // The sums are kept in 2 to 8 parts: their error against 64 bits is 0.5 to 0.9 times gemm_kernel's.
    template <int MT, int RN, int KS>
    struct GemmSplit
    {
        static constexpr int BM = MT * 32, KW = 2 * KS, WAVES = RN * KW; // wavefronts along K, and of a workgroup
        static constexpr int QUANTS = KS * BM * 256, HEADS = KS * BM * 32; // bytes of a step
        static constexpr int QLOADS = QUANTS / 1024 / WAVES, HLOADS = HEADS / 256 / WAVES; // per wavefront
        static constexpr int QROWS = 4 * WAVES;                  // tokens x super-blocks that one load of every wavefront covers
        static constexpr int QM = BM > QROWS ? BM / QROWS : 1;   // tokens a lane loads pieces of
        static constexpr int HM = BM > 8 * WAVES ? BM / (8 * WAVES) : 1; // tokens a lane loads heads of
        static_assert(QLOADS * WAVES * 1024 == QUANTS && HLOADS * WAVES * 256 == HEADS, "whole loads");
        static_assert(QROWS % 16 == 0 && (BM % QROWS == 0 || QROWS % BM == 0), "a lane's piece and tokens stay the same");
        static_assert(BM % (8 * WAVES) == 0 || 8 * WAVES % BM == 0, "a lane's tokens stay the same");
        static constexpr size_t STAGE = QUANTS + HEADS;
        static constexpr size_t SUMS = (size_t)(KW - 1) * RN * MT * 16 * WAVE * sizeof(float);
        static constexpr size_t LDS = 2 * STAGE > SUMS ? 2 * STAGE : SUMS;
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

    template <class F, int MT, int RN, int KS, bool DUMP>
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
        const typename Q::Cursor wc = Q::cursor(g.w, (size_t)n * SB, (size_t)n * SB, lc);
        typename Q::Raw raw;
        auto issue_weights = [&](int sb) { Q::load_at(raw, wc, lc, sb < SB ? sb : SB - 1); }; // (past the end: the last super-block again)
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
                hfrom[i] = token(group * 8 + (lane & 7)) + (uint32_t)((lane >> 3) ^ (group & 7)) * 36;
            }
        }
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem;
        auto super_block = [&](int sb) { return abase + (size_t)(sb < SB ? sb : SB - 1) * 288; }; // (past the end: the last one)
        // Load i of the step of super-block sb0, where there is one: else no lane takes part (a branch among the products would
        // have the compiler copy their registers at its ends).
        constexpr int LOADS = G::QLOADS + G::HLOADS;
        auto issue_act = [&](int i, int sb0, int buf) {
            uint64_t all;
            if (i < G::QLOADS)
                asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, exec\n\ts_cmp_lt_i32 %4, %5\n\ts_cselect_b64 exec, -1, 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b64 exec, %0"
                             : "=&s"(all)
                             : "s"(lds0 + (uint32_t)(buf * (int)G::STAGE + wave * 1024 + i * G::WAVES * 1024)), "v"(qfrom[i % G::QM]),
                               "s"(super_block(sb0 + (wave * 4 + i * G::QROWS) / BM)), "s"(sb0), "s"(SB)
                             : "memory", "scc");
            else
            {
                const int h = i - G::QLOADS;
                asm volatile("s_mov_b32 m0, %1\n\ts_mov_b64 %0, exec\n\ts_cmp_lt_i32 %4, %5\n\ts_cselect_b64 exec, -1, 0\n\tglobal_load_lds_dword %2, %3\n\ts_mov_b64 exec, %0"
                             : "=&s"(all)
                             : "s"(lds0 + (uint32_t)(buf * (int)G::STAGE + G::QUANTS + wave * 256 + h * G::WAVES * 256)), "v"(hfrom[h % G::HM]),
                               "s"(super_block(sb0 + (wave + h * G::WAVES) / (BM / 8))), "s"(sb0), "s"(SB)
                             : "memory", "scc");
            }
        };
        const v16i bias = integer_bias();
        v16f acc[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                acc[t][r] = 0.0f;
        v32f zero2f;
#pragma unroll
        for (int r = 0; r < 32; ++r)
            zero2f[r] = 0.0f;

#pragma unroll
        for (int i = 0; i < LOADS; ++i)
            issue_act(i, 0, 0);
        issue_weights(own_sb);
        int buf = 0;
        for (int sb0 = 0; sb0 < SB; sb0 += KS, buf ^= 1)
        {
            const int sb = sb0 + own_sb;
            // this step's weights and activations have arrived, everybody is done with the other buffer
            Q::template wait<0>(raw);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            v4i w[4];
            typename Q::Scale S;
            Q::decode(raw, lc, w, S);
            // decoded here, before the registers are asked for again: sunk below, the decoding would have the compiler copy
            // the raw words, and copies made ahead of the wait hold what the loads have not brought yet
            v2i_dword two = __builtin_bit_cast(v2i_dword, S);
            asm volatile("" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(two));
            S = __builtin_bit_cast(typename Q::Scale, two);
            __builtin_amdgcn_sched_barrier(0);
            // (the weights at once: they come from memory, and dealt out behind the products they were waited for)
            issue_weights(sb + KS);
            __builtin_amdgcn_sched_barrier(0);
            if (sb < SB) // uniform in the wavefront
            {
                const uint8_t *rows = smem + buf * G::STAGE + (size_t)(own_sb * BM + l32) * 256;
                const uint32_t *heads = reinterpret_cast<const uint32_t *>(smem + buf * G::STAGE + G::QUANTS) + own_sb * 8 * BM + (l32 >> 3) * 64 + (l32 & 7);
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
                // Product j: pair of blocks j / MT by tokens 32 (j % MT) ...  The matrix unit works on a product while the vector
                // unit rescales the one before it, and the LDS brings the operands of the next.
                constexpr int JOBS = 2 * MT, EACH = (LOADS + JOBS - 1) / JOBS;
                auto fence = []() __attribute__((always_inline)) {
                    if (MT > 1) // (two products of a step are not enough for it: the compiler's order is 10 % faster)
                        __builtin_amdgcn_sched_barrier(0);
                };
                auto block = [&](int j, int which) { return Q::block_of(2 * half + which, j / MT); };
                auto quants = [&](int j, int which) {
                    return *reinterpret_cast<const v4i *>(rows + (j % MT) * 32 * 256 + (((2 * block(j, which) + lh) ^ (l32 & 15)) << 4));
                };
                auto head_of = [&](int j) { return heads[(((lh ? block(j, 1) : block(j, 0)) ^ ((j % MT & 1) * 4 + (l32 >> 3))) * 8) + (j % MT) * 256]; };
                auto scale_of = [](uint32_t head) { return h2f((uint16_t)(head & 0xFFFFu)); };
                // the scale products of both blocks, a rank-1 matrix each (exact: both factors are fp16 values)
                auto scales = [&](int j, uint32_t head) { return __builtin_amdgcn_mfma_f32_32x32x1f32(scale_of(head), Q::scale_f32(S, j / MT), zero2f, 0, 0, 0); };
                auto product = [&](int j, int which, v4i a) { return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, w[2 * (j / MT) + which], bias, 0, 0, 0); };
                auto dump = [&](int j, int which, const v16i &d) {
                    const long nn = n0 + l32 - g.row0;
                    if (n0 + l32 < g.w.N && nn >= 0 && nn < g.nrows)
                    {
                        // (less than 2 GiB of sums: offsets of 32 bits, made anew for each, or they would fill the registers)
                        const uint32_t token = (uint32_t)g.nrows * (uint32_t)KB;
                        uint32_t at = ((uint32_t)m0 + 4 * lh) * token + (uint32_t)nn * (uint32_t)KB + (uint32_t)(sb * 8 + block(j, which));
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                        {
                            const int m = j % MT * 32 + 8 * (r >> 2) + (r & 3);
                            asm volatile("" : "+v"(at));
                            if (m0 + 4 * lh + m < g.M)
                                g.sums[at + (uint32_t)m * token] = (int32_t)biased_to_float(d[r]);
                        }
                    }
                };
                uint32_t head[2] = {head_of(0), 0};
                v32f cs[2];
                cs[0] = scales(0, head[0]);
                v16i dx = product(0, 0, quants(0, 0)), dy = product(0, 1, quants(0, 1));
#pragma unroll
                for (int j = 0; j < JOBS; ++j)
                {
                    const int t = j % MT, now = j & 1, next = now ^ 1;
                    v4i a;
                    fence();
#pragma unroll
                    for (int i = j * EACH; i < (j + 1) * EACH; ++i)
                        if (i < LOADS)
                            issue_act(i, sb0 + KS, buf ^ 1);
                    fence();
                    if (j + 1 < JOBS)
                    {
                        head[next] = head_of(j + 1);
                        a = quants(j + 1, 0);
                    }
                    if (DUMP)
                        dump(j, 0, dx);
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        acc[t][r] = fmaf(biased_to_float(dx[r]), cs[now][r], acc[t][r]);
                    fence();
                    if (j + 1 < JOBS)
                    {
                        cs[next] = scales(j + 1, head[next]);
                        dx = product(j + 1, 0, a);
                        a = quants(j + 1, 1);
                    }
                    fence();
                    if (DUMP)
                        dump(j, 1, dy);
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        acc[t][r] = fmaf(biased_to_float(dy[r]), cs[now][16 + r], acc[t][r]);
                    fence();
                    if (j + 1 < JOBS)
                        dy = product(j + 1, 1, a);
                    if (F::HAS_MIN)
                        acc[t] = __builtin_amdgcn_mfma_f32_32x32x2f32((float)(int16_t)(head[now] >> 16) * scale_of(head[now]), Q::min_f32(S, j / MT), acc[t], 0, 0, 0);
                }
            }
        }
        Q::template wait<0>(raw);
        if (DUMP)
            return;

        __syncthreads(); // everybody is done with the activations
        float *red = reinterpret_cast<float *>(smem) + rn * MT * 16 * WAVE + lane;
        if (kw > 0)
        {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    red[((kw - 1) * RN * MT * 16 + t * 16 + r) * WAVE] = acc[t][r];
        }
        __syncthreads();
        if (kw > 0)
            return;
        // (not unrolled: all sums asked for at once would not fit the registers)
#pragma unroll 1
        for (int k = 0; k < KW - 1; ++k)
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[t][r] += red[(k * RN * MT * 16 + t * 16 + r) * WAVE];
        if (n0 + l32 < g.w.N)
        {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                {
                    const long m = m0 + t * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
                    if (m < g.M)
                        g.y[(size_t)m * g.ldy + n0 + l32] = acc[t][r];
                }
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

    template <class F, bool DUMP, int MT, int RN, int KS>
    bool gemm_split_launch(const char *fn, const GemmArgs &g, int rows, int M, hipStream_t st)
    {
        constexpr size_t lds = GemmSplit<MT, RN, KS>::LDS;
        static_assert(lds + 6 * 1024 <= 160 * 1024, "LDS, with the decoders' tables");
        static LdsGrant grant;
        const auto kernel = &gemm_split_kernel<F, MT, RN, KS, DUMP>;
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
    //   tokens x rows x K             gemm_kernel  0: 1,1,4  1: 1,2,2  2: 2,1,4  3: 2,2,2  4: 2,4,1  5: 4,2,2  6: 4,4,1
    //   10 x 4096 x 4096, Q4_K           16.5         9.8     13.5      13.5      20.5      32.9      32.5      52.6
    //   64 x 4096 x 4096, IQ3_S          31.3        12.6     18.3      16.7      23.6      38.2      33.7      55.0
    //   20 x 12000 x 4096, IQ3_S         23.1        21.6     18.5      28.9      24.1      38.2      34.5      55.2
    //   40 x 8192 x 5120, IQ3_S          38.4        25.2     21.9      19.0      28.7      46.8      40.7      67.7
    //   63 x 5034 x 18944, Q6_K          162         103      96.0      70.5      114       201       153       279
    //   130 x 5000 x 5120, Q4_K          52.2        36.7     30.0      33.2      26.7      40.7      40.9      65.6
    //   64 x 25600 x 5120, Q4_K          53.8        68.1     60.0      68.4      51.9      45.1      82.0      70.5
    //   80 x 9762 x 3072, Q6_K           37.3        38.1     31.7      39.8      37.8      31.9      29.1      45.3
    //   199 x 5120 x 25600, Q6_K         298         298      314       230       260       241       207       369
    //   256 x 8192 x 8192, Q4_K          86.2        122      92.2      97.1      75.8      65.7      64.8      106
    //   1000 x 4096 x 4096, Q4_K         65.8        122      94.1      110       79.4      66.5      68.1      57.8
    //   256 x 25600 x 5120, Q4_K         154         228      184       211       167       160       161       140
    // and gemm_kernel's shapes, tiles of 32 tokens in one round, or three and more rounds of tiles of 128:
    //   16 x 25600 x 5120, Q6_K          49.9        65.1     57.7      77.0      67.4      59.0      93.0      83.2
    //   384 x 25600 x 5120, Q4_K         194         339      267       303       236       201       201       208
    //   512 x 25600 x 5120, Q4_K         266         445      351       401       309       280       282       275
    //   2048 x 6400 x 5120, IQ3_S        263         518      473       410       350       322       279       272
    // Tiles that fill their last round exactly, one round or several (us, gemm_kernel and the entry that is taken; Q4_K, Q6_K, IQ3_S):
    //   1024 x 4096 x 4096    67.2, 75.3, 66.8 -> 59.5, 62.6, 59.0 (6)     512 x 16384 x 4096    130, 147, 130 -> 118, 124, 120 (6)
    //   512 x 8192 x 12800    200, 228, 199 -> 172, 183, 174 (6)           40 x 32768 x 1024     15.4, 18.4, 16.7 -> 14.2, 17.0, 15.8 (4)
    // and gemm_kernel's (us, gemm_kernel and the entry that would come next):
    //   512 x 8192 x 768      17.2, 18.4, 17.4 : 18.2, 18.7, 18.4 (6)      16 x 32768 x 8192     49.3, 75.2, 67.7 : 55.5, 75.8, 69.2 (1)
    //   1000 x 4096 x 512     13.1, 13.9, 13.0 : 13.3, 15.4, 13.2 (6)      256 x 16384 x 1024    21.3, 24.2, 21.4 : 21.7, 24.1, 22.0 (6)
    struct SplitTile
    {
        int mt, rn, ks;
        double step[3]; // microseconds: a step (KS super-blocks) of Q4_K, Q6_K and IQ3_S
    };
    constexpr SplitTile SPLIT[] = {
        {1, 1, 4, {1.6, 2.8, 2.4}}, {1, 2, 2, {1.35, 2.45, 1.9}}, {2, 1, 4, {2.65, 3.5, 3.2}}, {2, 2, 2, {2.35, 3.05, 2.6}},
        {2, 4, 1, {2.05, 2.9, 2.4}}, {4, 2, 2, {3.83, 4.1, 4.0}}, {4, 4, 1, {3.45, 3.85, 3.6}}};
    constexpr double SPLIT_START = 3.5, WHOLE_START = 2.0; // a workgroup's start and end
    // gemm_kernel: microseconds a super-block of a tile of 32, 64 or 128 tokens takes in a round of two workgroups a compute unit
    // that others follow, in the last round, and in a last round of one
    struct WholeTile
    {
        int tokens;
        double full[3], last[3], alone[3];
    };
    constexpr WholeTile WHOLE[] = {{32, {1.4, 2.2, 1.9}, {1.6, 2.5, 2.2}, {0.9, 1.5, 1.4}},
                                   {64, {2.4, 3.1, 2.65}, {2.7, 3.6, 3.05}, {1.65, 2.2, 1.9}},
                                   {GEMM_BM, {3.55, 3.95, 3.55}, {4.2, 4.8, 4.35}, {2.6, 3.0, 2.8}}};

    inline int gemm_split_choice(int format, int M, int N, int K, int cus)
    {
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
        for (int i = 0; i < (int)(sizeof(SPLIT) / sizeof(SPLIT[0])); ++i)
        {
            const SplitTile &t = SPLIT[i];
            if (over(M, 32 * t.mt) > 65535) // (the grid's second extent)
                continue;
            // (a last round of few workgroups is faster: they have the memory and the clock to themselves)
            const long groups = over(N, 32 * t.rn) * over(M, 32 * t.mt), left = groups % cus;
            const double rounds = groups <= cus ? 1.0 : (double)(groups / cus) + (left ? 0.6 + 0.4 * (double)left / cus : 0.0);
            const double us = rounds * ((double)over(SB, t.ks) * t.step[format] + SPLIT_START);
            if (us < best)
                best = us, choice = i;
        }
        return choice;
    }

    // d_sums: the block-sum variant over weight rows [row0, row0+nrows); only the workgroups
    // whose 64-row tile meets the window are launched.
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
        g.tile0 = DUMP ? row0 / GEMM_BN : 0;
        // (the quad-lane decoders address a matrix through 32-bit offsets)
        if constexpr (F::USE_QUAD)
        {
            if (!F::Quad::addressable(N, K / 256))
                return fail(fn, "matrix too large for the kernel's 32-bit offsets (N=%d K=%d)", N, K);
        }
        const int tile_end = DUMP ? (row0 + nrows + GEMM_BN - 1) / GEMM_BN : (N + GEMM_BN - 1) / GEMM_BN;
        const int rows_end = DUMP ? row0 + nrows : N, rows = rows_end - g.tile0 * GEMM_BN;
        constexpr int format = F::HAS_MIN ? 0 : F::TABLE_BYTES > 0 ? 2 : 1; // Q4_K, Q6_K, IQ3_S
        switch (gemm_split_choice(format, M, N, K, cu_count(device_id)))
        {
        case 0: return gemm_split_launch<F, DUMP, 1, 1, 4>(fn, g, rows, M, st);
        case 1: return gemm_split_launch<F, DUMP, 1, 2, 2>(fn, g, rows, M, st);
        case 2: return gemm_split_launch<F, DUMP, 2, 1, 4>(fn, g, rows, M, st);
        case 3: return gemm_split_launch<F, DUMP, 2, 2, 2>(fn, g, rows, M, st);
        case 4: return gemm_split_launch<F, DUMP, 2, 4, 1>(fn, g, rows, M, st);
        case 5: return gemm_split_launch<F, DUMP, 4, 2, 2>(fn, g, rows, M, st);
        case 6: return gemm_split_launch<F, DUMP, 4, 4, 1>(fn, g, rows, M, st);
        default: break;
        }
        // few tokens: one smaller tile of tokens (a 128-token tile would rescale 128 rows for them)
        if (M <= 32)
            return gemm_launch_bm<F, DUMP, 32>(fn, g, tile_end - g.tile0, M, st);
        if (M <= 64)
            return gemm_launch_bm<F, DUMP, 64>(fn, g, tile_end - g.tile0, M, st);
        return gemm_launch_bm<F, DUMP, GEMM_BM>(fn, g, tile_end - g.tile0, M, st);
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
