// Linear layers with bf16 weights in matrix-unit tiles, for gfx950.
//
// Up to 16 rows (decoding): one workgroup per 16-row tile of W (or half of one), its wavefronts dealing the
// k-steps among themselves and summing through LDS; each weight byte is read once, a contiguous
// kilobyte per load instruction, several in flight per wavefront.  The rows of A are the second
// matrix operand (16 columns, those past M ignored).  HBM-bound.
// More rows (prompts): linear_tiled.hip.
#include "linear.h"

#include <type_traits>

namespace llamql
{
    // ---- up to 16 rows ------------------------------------------------------------------------
    constexpr int NORM_PAD = 8; // between normed rows in LDS: they start in different banks

    template <typename T>
    size_t norm_lds(const LinearArgs &a)
    {
        return (size_t)(sizeof(T) == 4 ? 3 : 1) * a.M * (a.K + NORM_PAD) * sizeof(bf16);
    }

    template <int NW>
    __device__ __forceinline__ float inverse_norm(const float *sums, int k_real, float eps)
    {
        float total = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w)
            total += sums[w];
        return 1.0f / sqrtf(total / (float)k_real + eps);
    }

    // fp32 rows normed, into h_out as T (from the first workgroup) and into LDS: as bf16, or, for T fp32, in three bf16
    // pieces that add up to the value (8 + 8 + 8 significant bits, cut off), the pieces
    // p.M * ldh apart.  Three products of bf16 take 48 cycles of the matrix unit a k-step, one of fp32 256 (3 x 32768 x
    // 2048: 43.4 -> 34.5 us; the error against 64 bits falls from 3.0e-7 to 2.0e-7).  R rows at a time are asked for and summed,
    // and all rows share one barrier: a row at a time, eight rows of 768 values took 6 us of a 9 us launch.
    template <typename T, int NW, int R>
    __device__ __forceinline__ void norm_rows(const LinearArgs &p, bf16 *h, int ldh, bool record, float (&s_sum)[SMALL_M][NW])
    {
        typedef T t4 __attribute__((ext_vector_type(4)));
        static_assert(SMALL_M % R == 0, "sums of whole groups");
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const auto row = [&](int m) { return reinterpret_cast<const f32x4 *>(static_cast<const float *>(p.a) + (size_t)(m < p.M ? m : p.M - 1) * p.lda); };
        for (int m0 = 0; m0 < p.M; m0 += R)
        {
            float sum[R] = {};
            for (int i = threadIdx.x; i < p.K / 4; i += NW * 64)
            {
                f32x4 v[R];
#pragma unroll
                for (int k = 0; k < R; ++k)
                    v[k] = row(m0 + k)[i];
#pragma unroll
                for (int k = 0; k < R; ++k)
                    sum[k] += v[k][0] * v[k][0] + v[k][1] * v[k][1] + v[k][2] * v[k][2] + v[k][3] * v[k][3];
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1)
#pragma unroll
                for (int k = 0; k < R; ++k)
                    sum[k] += __shfl_xor(sum[k], off, 64);
            if (lane == 0)
            {
#pragma unroll
                for (int k = 0; k < R; ++k)
                    s_sum[m0 + k][wave] = sum[k];
            }
        }
        __syncthreads();
        for (int m0 = 0; m0 < p.M; m0 += R)
        {
            float inv[R];
#pragma unroll
            for (int k = 0; k < R; ++k)
                inv[k] = inverse_norm<NW>(s_sum[m0 + k], p.k_real, p.eps);
            for (int i = threadIdx.x; i < p.K / 4; i += NW * 64)
            {
                f32x4 v[R];
                const f32x4 scale = reinterpret_cast<const f32x4 *>(p.norm)[i];
#pragma unroll
                for (int k = 0; k < R; ++k)
                    v[k] = row(m0 + k)[i];
#pragma unroll
                for (int k = 0; k < R; ++k)
                    if (m0 + k < p.M)
                    {
                        const t4 o = __builtin_convertvector(v[k] * inv[k] * scale, t4);
                        bf16 *to = h + (size_t)(m0 + k) * ldh + 4 * i;
                        if constexpr (sizeof(T) == 2)
                            *reinterpret_cast<t4 *>(to) = o;
                        else
                        {
                            f32x4 rest = o;
#pragma unroll
                            for (int piece = 0; piece < 3; ++piece, to += p.M * ldh)
                            {
                                u32x4 cut = __builtin_bit_cast(u32x4, rest);
                                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                                *reinterpret_cast<u32x2 *>(to) = u32x2{__builtin_amdgcn_perm(cut[1], cut[0], 0x07060302u),
                                                                       __builtin_amdgcn_perm(cut[3], cut[2], 0x07060302u)}; // upper halves
                                cut &= 0xffff0000u;
                                rest -= __builtin_bit_cast(f32x4, cut);
                            }
                        }
                        if (record)
                            *reinterpret_cast<t4 *>(static_cast<T *>(p.h_out) + (size_t)(m0 + k) * p.K + 4 * i) = o;
                    }
            }
        }
        __syncthreads();
    }

    // RT tiles of W per workgroup (2 for a gate tile beside its up tile, or to share the rows), NW wavefronts, U steps
    // in flight per wavefront.  NORM: A is fp32, normed by the workgroup into LDS (as T) while the
    // first weights are on their way.
    // HALF: up to 8 rows of A, and a workgroup for 8 rows of W, half a tile: a step is two k-steps, W's rows of the second
    // beside those of the first as the matrix unit's other 8 rows, A's likewise as its other 8 columns, and of the product
    // the two blocks that match are kept.  Twice the workgroups, for layers of fewer tiles than the chip has compute units.
    template <typename T, int NW, int RT, bool NORM, bool HALF = false>
    __device__ __forceinline__ void linear_small_tile(const LinearArgs &p, int block)
    {
        using O = Operand<T>;
        using V = typename O::V;
        static_assert(!HALF || RT == 1, "half a tile");
        constexpr int U = RT == 1 && (NORM || sizeof(T) == 2) ? 8 : 4;
        constexpr int STEP = HALF ? 2 : 1;   // k-steps (their number is even)
        constexpr bool CUT = NORM && sizeof(T) == 4; // rows in three bf16 pieces
        extern __shared__ __attribute__((aligned(16))) char smem[];
        __shared__ __attribute__((aligned(16))) float s_red[NW][RT][64][4];
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int n = lane & 15, g = lane >> 4;
        const int z = blockIdx.y;
        const int ksteps = p.K >> 5, steps = ksteps / STEP;
        const int second = HALF ? n >> 3 : 0;                                 // which k-step of a step is this lane's
        const int piece = HALF ? g * 16 + (block & 1) * 8 + (n & 7) : lane;   // of a k-step of W
        const int tile = HALF ? block >> 1 : block * RT;
        const int row = HALF ? n & 7 : n;                                     // of A

        const u32x4 *w[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t)
            w[t] = weight_tile(static_cast<const bf16 *>(p.w) + (size_t)z * p.w_stride - (t && (tile + t) * 16 >= p.N ? (size_t)ksteps * 512 : 0), (size_t)tile + t, ksteps, piece) + second * 64;
        u32x4 next[RT][U];
        auto fetch = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                const int s = s0 + u * NW;
#pragma unroll
                for (int t = 0; t < RT; ++t)
                    next[t][u] = w[t][(size_t)(s < steps ? s : wave < steps ? wave : 0) * (64 * STEP)];
            }
        };
        fetch(wave);

        using A = std::conditional_t<NORM, bf16, T>;
        const int ldh = p.K + NORM_PAD;
        const A *arow;
        __shared__ float s_sum[NORM ? SMALL_M : 1][NW];
        if constexpr (NORM)
        {
            bf16 *h = reinterpret_cast<bf16 *>(smem);
            const bool record = p.h_out && block == 0;
            // (two rows not as four, two of them in vain: 2 x 5120 x 2048 in bf16 6.4 -> 5.3 us; the way of many rows first in the
            // code: behind the others it took 1.3 us more where compute units have several workgroups, 4 x 12288 x 512 10.8 and 9.5)
            if (__builtin_expect(p.M > 2, 1))
                norm_rows<T, NW, 4>(p, h, ldh, record, s_sum);
            else if (p.M == 2)
                norm_rows<T, NW, 2>(p, h, ldh, record, s_sum);
            else
                norm_rows<T, NW, 1>(p, h, ldh, record, s_sum);
            arow = h + (size_t)(row < p.M ? row : 0) * ldh + 8 * g;
        }
        else
            arow = static_cast<const T *>(p.a) + (size_t)z * p.a_stride + (size_t)(row < p.M ? row : 0) * p.lda + 8 * g;
        arow += second * 32;

        f32x4 acc[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t)
            acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int s0 = wave; s0 < steps; s0 += NW * U)
        {
            u32x4 cur[RT][U];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int t = 0; t < RT; ++t)
                    cur[t][u] = next[t][u];
            // Rows that come from memory are asked for ahead of the next weights: loads arrive in order, so a product that
            // waits for a row asked for behind them would wait for all of them (3 x 2048 x 10240 bf16 11.8 -> 10.3 us, fp32
            // 18.7 -> 12.8; 8 x 5120 x 25600 bf16 72 -> 67 us, fp32 108 -> 85).  Not in a last round with fewer than U steps:
            // there are no next weights, and rows asked for in vain took as long as the others (16 x 5120 x 1024 in
            // bf16 6.3 -> 4.6).
            constexpr bool AHEAD = !NORM && (sizeof(T) == 2 || RT == 1); // (two tiles of fp32 rows: registers of a second workgroup)
            if (AHEAD && __builtin_amdgcn_readfirstlane(s0 + (U - 1) * NW < steps))
            {
                V b[AHEAD ? U : 1];
#pragma unroll
                for (int u = 0; u < (AHEAD ? U : 1); ++u)
                    b[u] = O::load(reinterpret_cast<const T *>(arow) + (s0 + u * NW) * (32 * STEP));
                __builtin_amdgcn_sched_barrier(0);
                if (s0 + NW * U < steps)
                    fetch(s0 + NW * U);
#pragma unroll
                for (int u = 0; u < (AHEAD ? U : 1); ++u)
#pragma unroll
                    for (int t = 0; t < RT; ++t)
                        acc[t] = O::mma(O::from_weights(cur[t][u]), b[u], acc[t]);
                continue;
            }
            // Such a round's rows are all asked for before the first product waits: 1 x 512 x 512 in bf16 2.65 -> 2.35 us, 4 x 2048 x
            // 11008 12.1 -> 11.3, 8 x 12288 x 2048 in fp32 17.4 -> 15.3.  Whole tiles of bf16 rows and eight wavefronts have no
            // registers for it (8 x 32768 x 2048 25.7 -> 31.2), half tiles of fp32 rows no need (8 x 1024 x 1024 3.9 -> 4.2): their
            // products wait one by one.
            if constexpr (AHEAD && (sizeof(T) == 4 ? !HALF : HALF || NW == 4))
            {
                V b[U];
                const int left = __builtin_amdgcn_readfirstlane((steps - s0 + NW - 1) / NW);
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (u < left)
                        b[u] = O::load(arow + (s0 + u * NW) * (32 * STEP));
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (u < left)
                    {
#pragma unroll
                        for (int t = 0; t < RT; ++t)
                            acc[t] = O::mma(O::from_weights(cur[t][u]), b[u], acc[t]);
                    }
                break;
            }
            if (s0 + NW * U < steps)
                fetch(s0 + NW * U);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (s0 + u * NW < steps)
                {
                    if constexpr (CUT)
                    {
#pragma unroll
                        for (int piece = 2; piece >= 0; --piece)
                        {
                            const bf16x8 part = Operand<bf16>::load(arow + piece * p.M * ldh + (s0 + u * NW) * (32 * STEP));
#pragma unroll
                            for (int t = 0; t < RT; ++t)
                                acc[t] = Operand<bf16>::mma(Operand<bf16>::from_weights(cur[t][u]), part, acc[t]);
                        }
                    }
                    else
                    {
                        const V b = O::load(arow + (s0 + u * NW) * (32 * STEP));
#pragma unroll
                        for (int t = 0; t < RT; ++t)
                            acc[t] = O::mma(O::from_weights(cur[t][u]), b, acc[t]);
                    }
                }
        }
#pragma unroll
        for (int t = 0; t < RT; ++t)
            *reinterpret_cast<f32x4 *>(s_red[wave][t][lane]) = acc[t];
        __syncthreads();
        if (threadIdx.x < 64 && n < p.M && (!HALF || (n < 8 && g < 2)))
        {
            f32x4 sum[RT];
#pragma unroll
            for (int t = 0; t < RT; ++t)
            {
                sum[t] = *reinterpret_cast<const f32x4 *>(s_red[0][t][lane]);
#pragma unroll
                for (int v = 1; v < NW; ++v)
                    sum[t] = sum[t] + *reinterpret_cast<const f32x4 *>(s_red[v][t][lane]);
                if (HALF)
                {
#pragma unroll
                    for (int v = 0; v < NW; ++v) // rows and columns 8 ..
                        sum[t] = sum[t] + *reinterpret_cast<const f32x4 *>(s_red[v][t][lane + 40]);
                }
            }
            if constexpr (CUT)
            {
                // sums that the pieces do not carry (see pieces_fail), once more as products of the whole values
                bool fail = false;
#pragma unroll
                for (int t = 0; t < RT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        fail |= pieces_fail(sum[t][r]);
                if (__builtin_expect(__ballot(fail) != 0, 0))
                {
                    const float inv = inverse_norm<NW>(s_sum[n], p.k_real, p.eps);
                    const float *x = static_cast<const float *>(p.a) + (size_t)n * p.lda, *scale = p.norm;
                    const int first = (HALF ? (block & 1) * 8 : 0) + 4 * g; // of the tile's rows
                    f32x4 whole[RT];
#pragma unroll
                    for (int t = 0; t < RT; ++t)
                        whole[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
                    for (int k = 0; k < 32 * ksteps; k += 8)
                    {
                        const f32x8 v = Operand<float>::load(x + k) * inv * Operand<float>::load(scale + k);
#pragma unroll
                        for (int t = 0; t < RT; ++t)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                            {
                                const f32x8 q = Operand<float>::from_weights(w[t][(k >> 5) * 64 + ((k >> 3) & 3) * 16 + first + r - piece - second * 64]);
#pragma unroll
                                for (int e = 0; e < 8; ++e)
                                    whole[t][r] = fmaf(v[e], q[e], whole[t][r]);
                            }
                    }
#pragma unroll
                    for (int t = 0; t < RT; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            sum[t][r] = pieces_fail(sum[t][r]) ? whole[t][r] : sum[t][r];
                }
            }
            const size_t elem = p.out == LLAM_SEQ_OUT_F32 || p.out == LLAM_SEQ_OUT_ADD ? 4 : sizeof(T);
            char *y = static_cast<char *>(p.y) + (size_t)z * p.y_stride * elem;
            if (RT == 2 && is_gated(p.out))
                store4<T>(p, y, n, block * 16 + 4 * g, gated4(p, sum[0], sum[RT - 1]));
            else if (HALF)
                store4<T>(p, y, n, block * 8 + 4 * g, sum[0]);
            else
            {
                // (the last tile of an odd number of them is a copy)
#pragma unroll
                for (int t = 0; t < RT; ++t)
                    if ((block * RT + t) * 16 < p.N)
                        store4<T>(p, y, n, (block * RT + t) * 16 + 4 * g, sum[t]);
            }
        }
    }

    template <typename T, int NW, int RT, bool NORM, bool HALF>
    __global__ void __launch_bounds__(NW * 64)
        linear_small_kernel(LinearArgs p)
    {
        linear_small_tile<T, NW, RT, NORM, HALF>(p, blockIdx.x);
    }

    // Two layers over the same rows: the first `blocks` workgroups belong to p.
    template <typename T, int NW, bool NORM>
    __global__ void __launch_bounds__(NW * 64)
        linear_small_pair_kernel(LinearArgs p, LinearArgs second, int blocks)
    {
        // (either way its own code: of arguments chosen at run time the compiler keeps a copy in scratch memory)
        if ((int)blockIdx.x < blocks)
            linear_small_tile<T, NW, 2, NORM>(p, blockIdx.x);
        else
            linear_small_tile<T, NW, 2, NORM>(second, (int)blockIdx.x - blocks);
    }

    namespace
    {
        template <typename T, int NW, int RT, bool NORM, bool HALF = false>
        bool small_launch(const char *fn, const LinearArgs &a, int batch, hipStream_t st)
        {
            static LdsGrant grant;
            const size_t lds = NORM ? norm_lds<T>(a) : 0;
            const auto kernel = &linear_small_kernel<T, NW, RT, NORM, HALF>;
            if (lds > 32 * 1024 && allow_lds(grant, reinterpret_cast<const void *>(kernel), 64 * 1024) != hipSuccess)
                return fail(fn, "cannot reserve %zu bytes of LDS", lds);
            hipLaunchKernelGGL(kernel, dim3(a.N / (HALF ? 8 : 16 * RT), batch), dim3(NW * 64), lds, st, a);
            return launched(fn);
        }
        template <typename T, int NW, bool NORM>
        bool small_tiles(const char *fn, const LinearArgs &a, int batch, int cus, hipStream_t st)
        {
            // Half tiles where they too find a compute unit each and whole ones need more than a round of eight steps for K (fp32
            // rows from memory: always, their products take as long as the weights).  M x N x K, us, whole and half tiles, weights
            // from memory as in a decode step, whose layers do not fit the caches:
            //   8 x 1024 x 3072  bf16  6.3,  5.3  fp32  8.2,  7.0      1 x 2048 x 5120   bf16  7.8,  7.1  normed  8.4,  8.0
            //   8 x 2048 x 10240 bf16 14.9, 13.1  fp32 20.7, 16.2      8 x 2304 x 10240  bf16 15.1, 20.4  fp32   20.9, 27.2
            //   8 x 2048 x 2048  bf16  5.0,  5.0  fp32  7.3,  6.1      8 x 512 x 512     bf16  2.9,  2.8  fp32    3.7,  3.0
            //   1 x 2048 x 8192  bf16  9.9,  8.3  normed 11.4, 10.9    1 x 4080 x 4096   bf16  8.0,  7.9  normed  9.5,  9.6
            // (Of weights that the caches hold, as in a loop over one matrix, rows of W 8 or 16 KB apart meet in the same channels, and
            // 1 x 2048 x 8192 normed takes 7.8 and 9.8, unnormed 6.2 and 6.8.)
            const long tiles = (long)a.N / 16 * batch;
            const bool half = a.M <= 8 && tiles <= cus / 2 && ((sizeof(T) == 4 && !NORM) || a.K > 2048);
            return half ? small_launch<T, NW, 1, NORM, true>(fn, a, batch, st) : small_launch<T, NW, 1, NORM>(fn, a, batch, st);
        }
        template <typename T>
        bool small_dispatch(const char *fn, const LinearArgs &a, int batch, int cus, hipStream_t st)
        {
            const bool gated = is_gated(a.out);
            const bool wide = a.K >= 1024;
            if (a.norm)
                return gated ? small_launch<T, 8, 2, true>(fn, a, batch, st) : small_tiles<T, 8, true>(fn, a, batch, cus, st);
            if (gated)
                return small_launch<T, 8, 2, false>(fn, a, batch, st);
            return wide ? small_tiles<T, 8, false>(fn, a, batch, cus, st) : small_tiles<T, 4, false>(fn, a, batch, cus, st);
        }
    } // namespace

    namespace
    {
        template <typename T, bool NORM>
        bool small_pair_launch(const char *fn, const LinearArgs &a, const LinearArgs &b, hipStream_t st)
        {
            static LdsGrant grant;
            const size_t lds = NORM ? norm_lds<T>(a) : 0;
            if (lds > 32 * 1024 && allow_lds(grant, reinterpret_cast<const void *>(&linear_small_pair_kernel<T, 8, NORM>), 64 * 1024) != hipSuccess)
                return fail(fn, "cannot reserve %zu bytes of LDS", lds);
            const int blocks = ceil_div(a.N, 32);
            hipLaunchKernelGGL((linear_small_pair_kernel<T, 8, NORM>), dim3(blocks + ceil_div(b.N, 32)), dim3(512), lds, st, a, b, blocks);
            return launched(fn);
        }
        template <typename T>
        bool small_pair_dispatch(const char *fn, const LinearArgs &a, const LinearArgs &b, hipStream_t st)
        {
            return a.norm ? small_pair_launch<T, true>(fn, a, b, st) : small_pair_launch<T, false>(fn, a, b, st);
        }
    } // namespace

    bool linear_small(const char *fn, const LinearArgs &a, int batch, int dtype, int device_id, hipStream_t st)
    {
        const int cus = cu_count(device_id);
        return dtype == LLAM_SEQ_F32 ? small_dispatch<float>(fn, a, batch, cus, st) : small_dispatch<bf16>(fn, a, batch, cus, st);
    }
} // namespace llamql

using namespace llamql;

namespace
{
    bool linear_args(const char *fn, const llam_seq_linear_args *a, int dtype, LinearArgs &p)
    {
        if (!a || !a->d_a || !a->d_w || !a->d_y)
            return fail(fn, "null pointer");
        if (a->M < 0 || a->N < 1 || a->K < 1 || a->batch < 1 || a->batch > 65535)
            return fail(fn, "bad size (M=%d N=%d K=%d batch=%d)", a->M, a->N, a->K, a->batch);
        if (dtype != LLAM_SEQ_BF16 && dtype != LLAM_SEQ_F32)
            return fail(fn, "dtype %d", dtype);
        const int elem = dtype == LLAM_SEQ_F32 ? 4 : 2;
        const bool gated = is_gated(a->out);
        if ((a->N % (gated ? 32 : 16)) != 0 || (a->K % PAD) != 0)
            return fail(fn, "N=%d must be a multiple of %d and K=%d of %d", a->N, gated ? 32 : 16, a->K, PAD);
        if (a->out < LLAM_SEQ_OUT_F32 || a->out > LLAM_SEQ_OUT_GATED_CLAMP)
            return fail(fn, "output kind %d", a->out);
        if (a->lda < a->K || a->ldy < (gated ? a->N / 2 : a->N))
            return fail(fn, "row strides smaller than the rows");
        if (!aligned16(a->d_a) || !aligned16(a->d_w) || !aligned16(a->d_y) || ((a->lda * (a->d_norm ? 4 : elem)) % 16) != 0 ||
            (a->ldy % 4) != 0 || ((a->a_stride * elem) % 16) != 0 || ((a->w_stride * 2) % 16) != 0 || (a->y_stride % 4) != 0)
            return fail(fn, "misaligned rows");
        if (a->d_norm && (a->M > SMALL_M || a->batch != 1 || (long)a->M * a->K > NORM_FUSE_MAX || a->k_real < 1 || !aligned16(a->d_norm)))
            return fail(fn, "a fused norm takes up to %d rows and %d values, unbatched", SMALL_M, NORM_FUSE_MAX);
        p = LinearArgs{};
        p.a = a->d_a, p.w = a->d_w, p.y = a->d_y, p.bias = a->d_bias, p.norm = a->d_norm, p.h_out = a->d_h_out;
        p.eps = a->eps, p.k_real = a->k_real, p.M = a->M, p.N = a->N, p.K = a->K, p.lda = a->lda, p.ldy = a->ldy;
        p.out = a->out, p.limit = a->limit, p.a_stride = a->a_stride, p.w_stride = a->w_stride, p.y_stride = a->y_stride;
        p.source_div = 1;
        return true;
    }
} // namespace

extern "C" size_t llam_seq_linear_scratch_bytes(int max_rows, int N, int K, int dtype, int device_id)
{
    if (max_rows <= SMALL_M || N < 1 || K < 1 || K % PAD != 0 || (dtype != LLAM_SEQ_BF16 && dtype != LLAM_SEQ_F32))
        return 0;
    return linear_split_bytes(max_rows, N, K, dtype, device_id);
}

extern "C" bool llam_seq_linear_within(const llam_seq_linear_args *a, void *d_scratch, size_t scratch_bytes, int dtype, int device_id, void *stream)
{
    static const char *fn = "llam_seq_linear";
    LinearArgs p;
    if (!linear_args(fn, a, dtype, p))
        return false;
    if (d_scratch && !aligned16(d_scratch))
        return fail(fn, "misaligned scratch");
    if (a->M == 0)
        return true;
    if (!set_device(fn, device_id))
        return false;
    return a->M <= SMALL_M ? linear_small(fn, p, a->batch, dtype, device_id, as_stream(stream))
                           : linear_tiled(fn, p, a->batch, dtype, device_id, as_stream(stream), d_scratch, scratch_bytes);
}

extern "C" bool llam_seq_linear(const llam_seq_linear_args *a, int dtype, int device_id, void *stream)
{
    return llam_seq_linear_within(a, nullptr, 0, dtype, device_id, stream);
}

extern "C" bool llam_seq_linear_rows(const llam_seq_linear_args *a, int n, const int *first, const int *rows, int dtype, int device_id, void *stream)
{
    static const char *fn = "llam_seq_linear_rows";
    LinearSomeArgs p{};
    if (!linear_args(fn, a, dtype, p))
        return false;
    if (a->M <= SMALL_M || n < 0 || (n > 0 && (!first || !rows)))
        return fail(fn, "bad size (M=%d, of more than %d; n=%d)", a->M, SMALL_M, n);
    for (int i = 0, at = 0; i < n; at = first[i] + rows[i], ++i)
        if (rows[i] < 1 || first[i] < at || first[i] > a->M - rows[i])
            return fail(fn, "stretch %d: %d rows from row %d of %d", i, rows[i], first[i], a->M);
    if (n > 0 && !set_device(fn, device_id))
        return false;
    for (int i = 0; i < n; i += p.stretches)
    {
        p.stretches = n - i < LINEAR_STRETCHES ? n - i : LINEAR_STRETCHES;
        for (int k = 0; k < p.stretches; ++k)
            p.first[k] = first[i + k], p.rows[k] = rows[i + k];
        if (!linear_tiled_rows(fn, p, a->batch, dtype, device_id, as_stream(stream)))
            return false;
    }
    return true;
}

extern "C" bool llam_seq_linear_pair(const llam_seq_linear_args *a, const llam_seq_linear_args *b, int dtype, int device_id, void *stream)
{
    static const char *fn = "llam_seq_linear_pair";
    LinearArgs p, q;
    if (!linear_args(fn, a, dtype, p) || !linear_args(fn, b, dtype, q))
        return false;
    if (p.M != q.M || p.K != q.K || a->batch != 1 || b->batch != 1 || !p.norm != !q.norm)
        return fail(fn, "the layers of a pair have the same rows and columns (M=%d, %d K=%d, %d)", p.M, q.M, p.K, q.K);
    if (p.M == 0)
        return true;
    if (!set_device(fn, device_id))
        return false;
    hipStream_t st = as_stream(stream);
    if (p.M <= SMALL_M)
        return dtype == LLAM_SEQ_F32 ? small_pair_dispatch<float>(fn, p, q, st) : small_pair_dispatch<bf16>(fn, p, q, st);
    return linear_tiled(fn, p, 1, dtype, device_id, st) && linear_tiled(fn, q, 1, dtype, device_id, st);
}

namespace
{
    // Eight values of an inner row of the turned matrix a thread
    __global__ void __launch_bounds__(256)
        transpose_tiles_kernel(const bf16 *__restrict__ w, bf16 *__restrict__ out, int N, int K)
    {
        const int piece = blockIdx.x * 256 + threadIdx.x;
        if (piece >= N * K / 8)
            return;
        const int lane = piece & 63, tile = piece >> 6, steps = N >> 5; // of the turned matrix, [K/16][N/32][64]
        const int k = tile / steps * 16 + (lane & 15), n0 = tile % steps * 32 + 8 * (lane >> 4);
        const bf16 *from = w + (size_t)blockIdx.y * N * K + ((size_t)(n0 >> 4) * (K >> 5) + (k >> 5)) * 512 + ((k & 31) >> 3) * 128 + (n0 & 15) * 8 + (k & 7);
        bf16x8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] = from[e * 8];
        *reinterpret_cast<bf16x8 *>(out + (size_t)blockIdx.y * N * K + (size_t)piece * 8) = v;
    }
} // namespace

extern "C" bool llam_seq_transpose_tiles(const void *d_w, void *d_out, int N, int K, int batch, int device_id, void *stream)
{
    static const char *fn = "llam_seq_transpose_tiles";
    if (N < 1 || K < 1 || N % 32 != 0 || K % 32 != 0 || batch < 1 || batch > 65535 || (long)N * K > 0x7fffffff)
        return fail(fn, "bad size (N=%d K=%d batch=%d)", N, K, batch);
    if (!d_w || !d_out || !aligned16(d_w) || !aligned16(d_out))
        return fail(fn, "null or misaligned pointer");
    if (!set_device(fn, device_id))
        return false;
    hipLaunchKernelGGL(transpose_tiles_kernel, dim3(ceil_div(N * (K / 8), 256), batch), dim3(256), 0, as_stream(stream), static_cast<const bf16 *>(d_w),
                       static_cast<bf16 *>(d_out), N, K);
    return launched(fn);
}
