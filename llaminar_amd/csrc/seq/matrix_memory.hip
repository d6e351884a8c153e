// Matrix-memory recurrence (per head: memory S [dim x vdim], normaliser n [dim], running maximum m),
// for gfx950.
//
// The normaliser is carried as one more column of S: a column whose value is 1 for every token.
// S and the outputs have vdim + 16 columns, column vdim being n (the other 15 stay zero).
//
// Decoding streams S once through the chip (read, update, write: HBM-bound).  Prompts run in chunks of
// LC tokens.  With F_t the sum of the log forget gates from the chunk's start to t, m0 the running
// maximum before it and a_j = i_j - F_j, the recurrence unrolls to
//   m_t = F_t + max(m0, max_{j<=t} a_j)
//   S_t' q = e^(F_t + m0 - m_t) S_0' q + sum_{j<=t} e^(F_t + a_j - m_t) (k_j . q) v_j
//   S_end = e^(F_end + m0 - m_end) S_0 + sum_j e^(F_end + a_j - m_end) k_j v_j'
// in three launches: the gates (one wavefront per head walks the portion; F, a and F - m in double, so
// that differences of long sums keep 32-bit accuracy), the token-by-token products of every chunk
// (independent of each other), and the walk over the chunks, where a wavefront owns 16 columns of
// S in its accumulators from the first chunk to the last.  An accumulator tile is also a second
// operand of the next product as it lies: lane (c, g) holds rows 4 g .. 4 g + 3, and the first operand
// is read in the same order.  In bf16, S and the gated values enter the products in three pieces,
// i.e. as 32-bit values; q, k and v are bf16 (the output format of a projection).
#include "seq_common.h"

#include <algorithm>

#include "llaminar_amd/seq_api.h"

namespace llamql
{
    struct MemoryArgs
    {
        const float *proj;
        int ldp;
        const float *gate_bias, *norm;
        float *state, *m;
        void *y;
        int ldy;
        int heads, dim, vdim, vdim_real;
        float q_scale, gate_cap, eps;
        const int32_t *row0, *ntok, *slot, *pos;
        int entry;      // first entry of the call
        bool many;      // several portions: a portion's chunks are kept from chunk row0 / LC + (its place among them) on
        double *ga, *a; // [rows][heads]: F_t - m_t, a_t
        float *mt;      // [rows][heads]: m_t
        float *m0;      // [portions][heads]: m before the portion
        float *prod;    // [chunks][heads][LC][LC]
        float *num;     // [rows][heads][vdim + 16]; decoding: [entries][heads][splits][vdim + 16]
        int splits;     // decoding: workgroups along dim
        void *qk;       // T [2][heads][rows of the portion][dim]: scaled q, then k
        int qk_rows;
        // long portions: stretches (a portion's at most, the most of any of the call's), what each adds to the memory and keeps of it
        int most, parts;
        float *starts; // [portions][stretches][heads][dim][vdim + 16]: the memory before the portion, then what stretch 0 .. adds
        float *kept;   // [portions][stretches][heads]: what is left of the memory after stretch 0 ..
    };

    constexpr int STRETCH_MIN = 3; // chunks of a stretch at least
    // Stretches of a portion that are walked side by side (1: the walk is one): a portion's own length decides, so that its
    // sums are the same whatever portions lie beside it, and a long one keeps its stretches beside short ones (a step of 2048, 60
    // and 60 tokens, Kogilix, width 2048: 2.99 -> 2.94 ms).  Portions that are cut and would fill the chip uncut pay for it:
    // five of 400 tokens take two launches of each kernel and 118 us a layer instead of 61.
    __host__ __device__ __forceinline__ int memory_stretches(int chunks, int most)
    {
        const int n = chunks / STRETCH_MIN;
        return n < 2 || most < 2 ? 1 : n < most ? n : most;
    }

    __device__ __forceinline__ void memory_gates(const MemoryArgs &p, const float *row, int h, float &i, float &f)
    {
        const float *raw = row + (size_t)p.heads * 2 * (p.dim + p.vdim);
        const float zi = raw[h] + p.gate_bias[h], zf = raw[p.heads + h] + p.gate_bias[p.heads + h];
        i = p.gate_cap * tanhf(zi / p.gate_cap);
        const float c = p.gate_cap * tanhf(zf / p.gate_cap);
        f = fminf(c, 0.0f) - log1pf(expf(-fabsf(c)));
    }

    // ---- decoding -------------------------------------------------------------------------------
    // Workgroup = 64 columns of one head's memory of one sequence, and a stretch of its rows.
    constexpr int STEP_ROWS = 64; // rows of a stretch when there are several
    template <typename T>
    __global__ void __launch_bounds__(256)
        memory_step_kernel(MemoryArgs p)
    {
        __shared__ float s_q[512], s_k[512];
        __shared__ __attribute__((aligned(16))) float s_o[16][64];
        const int h = blockIdx.y, ei = blockIdx.z, e = p.entry + ei;
        const int ldv = p.vdim + 16, blocks = (ldv + 63) >> 6;
        const int split = blockIdx.x / blocks, block = blockIdx.x - split * blocks;
        const int rows = p.splits > 1 ? STEP_ROWS : p.dim, first = split * rows;
        const int r = p.row0[e], slot = p.slot[e];
        const float *row = p.proj + (size_t)r * p.ldp;
        const int col = block * 64 + (threadIdx.x & 15) * 4, d0 = threadIdx.x >> 4;
        const bool fresh = p.pos[e] == 0;
        float *S = p.state + (((size_t)slot * p.heads + h) * p.dim + first) * ldv + col;
        const bool live = col < ldv;

        f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
        if (col < p.vdim)
        {
            v = *reinterpret_cast<const f32x4 *>(row + (size_t)p.heads * 2 * p.dim + h * p.vdim + col);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                v[j] = rounded<T>(v[j]);
        }
        else if (col == p.vdim)
            v[0] = 1.0f;
        for (int d = threadIdx.x; d < rows; d += 256)
        {
            s_q[d] = rounded<T>(row[h * p.dim + first + d] * p.q_scale);
            s_k[d] = rounded<T>(row[(p.heads + h) * p.dim + first + d]);
        }
        constexpr int U = STEP_ROWS / 16; // the first rows are requested before the gates are worked out
        f32x4 s[U];
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            s[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (live && !fresh)
                s[u] = *reinterpret_cast<const f32x4 *>(S + (size_t)(d0 + 16 * u) * ldv);
        }
        float gi, gf;
        memory_gates(p, row, h, gi, gf);
        const float m_old = fresh ? 0.0f : p.m[slot * p.heads + h];
        const float m_new = fmaxf(gf + m_old, gi);
        const float keep = expf(gf + m_old - m_new), take = expf(gi - m_new);
        v = v * take;
        __syncthreads();
        f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
        if (live)
            for (int d = d0; d < rows; d += STEP_ROWS)
            {
                if (d != d0)
                {
#pragma unroll
                    for (int u = 0; u < U; ++u)
                        s[u] = fresh ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : *reinterpret_cast<const f32x4 *>(S + (size_t)(d + 16 * u) * ldv);
                }
#pragma unroll
                for (int u = 0; u < U; ++u)
                {
                    s[u] = s[u] * keep + v * s_k[d + 16 * u];
                    *reinterpret_cast<f32x4 *>(S + (size_t)(d + 16 * u) * ldv) = s[u];
                    o = o + s[u] * s_q[d + 16 * u];
                }
            }
        *reinterpret_cast<f32x4 *>(&s_o[d0][(threadIdx.x & 15) * 4]) = o;
        __syncthreads();
        if (threadIdx.x < 64 && block * 64 + threadIdx.x < ldv)
        {
            float sum = 0.0f;
#pragma unroll
            for (int k = 0; k < 16; ++k)
                sum += s_o[k][threadIdx.x];
            p.num[(((size_t)ei * p.heads + h) * p.splits + split) * ldv + block * 64 + threadIdx.x] = sum;
        }
    }

    // where the chunks of the call's portion ei are kept
    template <int LC>
    __device__ __forceinline__ int first_chunk(const MemoryArgs &p, int ei)
    {
        return p.many ? p.row0[p.entry + ei] / LC + ei : 0;
    }

    // ---- prompts: gates -------------------------------------------------------------------------
    // A wavefront scans a chunk by itself; the running maximum passes from chunk to chunk by the chunks' totals.
    constexpr int GATE_WAVES = 16;
    template <int LC>
    __global__ void __launch_bounds__(GATE_WAVES * 64)
        memory_gates_kernel(MemoryArgs p)
    {
        __shared__ double s_total[GATE_WAVES], s_top[GATE_WAVES];
        const int h = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, e = p.entry + blockIdx.y;
        const int r0 = p.row0[e], n = p.ntok[e], slot = p.slot[e];
        float m = p.pos[e] == 0 ? 0.0f : p.m[slot * p.heads + h];
        if (threadIdx.x == 0)
            p.m0[blockIdx.y * p.heads + h] = m;
        for (int t0 = 0; t0 < n; t0 += GATE_WAVES * LC)
        {
            const int t = t0 + wave * LC + lane;
            const bool in = lane < LC && t < n;
            float gi = -INFINITY, gf = 0.0f;
            if (in)
                memory_gates(p, p.proj + (size_t)(r0 + t) * p.ldp, h, gi, gf);
            double F = gf;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1)
            {
                const double o = __shfl_up(F, off, 64);
                if (lane >= off)
                    F += o;
            }
            const double a = (double)gi - F;
            double top = in ? a : -INFINITY;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1)
            {
                const double o = __shfl_up(top, off, 64);
                if (lane >= off)
                    top = fmax(top, o);
            }
            __syncthreads();
            if (lane == 63)
            {
                s_total[wave] = F;
                s_top[wave] = top;
            }
            __syncthreads();
            // the running maximum is a 32-bit number of the recurrence
            float mine = m;
            for (int w = 0; w < GATE_WAVES; ++w)
            {
                if (w == wave)
                    mine = m;
                if (t0 + w * LC < n)
                    m = (float)(s_total[w] + fmax((double)m, s_top[w]));
            }
            if (in)
            {
                const float mt = (float)(F + fmax((double)mine, top));
                const size_t at = (size_t)(r0 + t) * p.heads + h;
                p.ga[at] = F - (double)mt;
                p.a[at] = a;
                p.mt[at] = mt;
            }
        }
        if (threadIdx.x == 0)
            p.m[slot * p.heads + h] = m;
    }

    // ---- prompts: products within a chunk ----------------------------------------------------------
    // prod[t][j] = e^(F_t + a_j - m_t) (q_t . k_j) for j <= t, else 0.  Wavefront w: rows 16 w ...  It also leaves
    // its rows of q (scaled) and k as T for the walk over the chunks, and the others their rows of k by way of LDS.  There is
    // a workgroup for every second compute unit at best, so it is as fast as its loads are few in a row: PRODUCT_COLS columns of
    // all rows are asked for at once (2048 tokens, 4 heads of 256: 20.0 -> 11.7 us against a step of 32 at a time, every wavefront
    // with the rows of k that it needs).
    constexpr int PRODUCT_COLS = 256;
    template <typename T, int LC>
    __global__ void __launch_bounds__(LC * 4)
        memory_product_kernel(MemoryArgs p)
    {
        using O = Operand<T>;
        using V = typename O::V;
        constexpr int LD = PRODUCT_COLS + 16 / (int)sizeof(T), STEPS = PRODUCT_COLS / 32;
        __shared__ __attribute__((aligned(16))) T s_k[LC][LD];
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
        const int h = blockIdx.y, chunk = blockIdx.x, e = p.entry + blockIdx.z;
        const int n = p.ntok[e] - chunk * LC < LC ? p.ntok[e] - chunk * LC : LC;
        if (n <= 0)
            return;
        const int r0 = p.row0[e] + chunk * LC, own = wave * 16 + c;
        const float *q = p.proj + (size_t)(r0 + (own < n ? own : n - 1)) * p.ldp + h * p.dim + 8 * g, *k = q + p.heads * p.dim;
        const int kept = chunk + first_chunk<LC>(p, blockIdx.z);
        T *qk = static_cast<T *>(p.qk) + ((size_t)h * p.qk_rows + kept * LC + own) * p.dim + 8 * g;
        const size_t k_after = (size_t)p.heads * p.qk_rows * p.dim;
        f32x4 acc[LC / 16];
#pragma unroll
        for (int j = 0; j < LC / 16; ++j)
            acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        double aj[LC / 16], ga[4];
        for (int s0 = 0; s0 < p.dim; s0 += PRODUCT_COLS)
        {
            f32x8 x[STEPS][2];
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                if (s0 + 32 * s < p.dim)
                {
                    x[s][0] = Operand<float>::load(q + s0 + 32 * s);
                    x[s][1] = Operand<float>::load(k + s0 + 32 * s);
                }
            if (s0 == 0)
            {
                const auto at = [&](int t) __attribute__((always_inline)) { return (size_t)(r0 + (t < n ? t : n - 1)) * p.heads + h; };
#pragma unroll
                for (int j = 0; j < LC / 16; ++j)
                    aj[j] = p.a[at(j * 16 + c)];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    ga[r] = p.ga[at(wave * 16 + 4 * g + r)];
            }
            V a[STEPS];
            __syncthreads();
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                if (s0 + 32 * s < p.dim)
                {
                    V one[1];
                    split_pieces<T, 1>(x[s][0] * p.q_scale, one);
                    a[s] = one[0];
                    *reinterpret_cast<V *>(qk + s0 + 32 * s) = a[s];
                    split_pieces<T, 1>(x[s][1], one);
                    *reinterpret_cast<V *>(qk + k_after + s0 + 32 * s) = one[0];
                    *reinterpret_cast<V *>(&s_k[own][32 * s + 8 * g]) = one[0];
                }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                if (s0 + 32 * s < p.dim)
                {
#pragma unroll
                    for (int j = 0; j < LC / 16; ++j)
                        if (j <= wave)
                            acc[j] = O::mma(a[s], *reinterpret_cast<const V *>(&s_k[j * 16 + c][32 * s + 8 * g]), acc[j]);
                }
        }
        float *out = p.prod + ((size_t)kept * p.heads + h) * LC * LC;
#pragma unroll
        for (int j = 0; j < LC / 16; ++j)
        {
            const int tj = j * 16 + c;
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const int t = wave * 16 + 4 * g + r;
                float y = 0.0f;
                if (tj <= t && t < n)
                    y = acc[j][r] * expf((float)(ga[r] + aj[j]));
                out[t * LC + tj] = y;
            }
        }
    }

    // ---- prompts: the walk over the chunks ----------------------------------------------------------
    // Workgroup = up to four wavefronts of 16 columns each, of one head.  DT: 16-row tiles of S (dim <= 16 DT); FULL:
    // dim is 16 DT exactly, so that no product hangs on a condition.
    // What the next chunk needs from memory (q and k for the LDS, this column's values, the products) is
    // requested before the matrix work of the current one.
    // The walk is a chain, 6 to 7 us a chunk of 64 tokens, and 36 workgroups (4 heads of 256 x 512) leave most of the chip idle.
    // A long portion is therefore cut into stretches that run side by side (blockIdx.z): the recurrence is linear in S, so a first
    // launch (SUM) walks each stretch from an empty memory without outputs and leaves what the stretch adds, and the walk
    // proper starts each stretch from the sum of what those before it added, each scaled by what the ones between keep.
    // 2048 tokens, 4 heads of 256 x 512: 232 -> 80 us for both launches, seven stretches of five chunks.  Stretches of fewer than
    // three chunks gain nothing: a chunk without outputs takes half the time of one with them, and is walked twice.
    // (CUT: portions may be cut.  Of more than 256 rows of S it would take more registers than there are.)
    template <typename T, int LC, int DT, bool FULL, bool CUT, bool SUM>
    __global__ void __launch_bounds__(256)
        memory_chunk_kernel(MemoryArgs p)
    {
        using O = Operand<T>;
        using V = typename O::V;
        typedef T t4 __attribute__((ext_vector_type(4)));
        constexpr int NP = O::PIECES;
        constexpr int LPAD = 16 / sizeof(T);
        constexpr int TPR = 256 / LC;                            // threads of a row when q and k are staged
        constexpr int LOADS = DT * 16 * (int)sizeof(T) / 16 / TPR; // 16-byte pieces of a row per thread
        constexpr bool AHEAD = LOADS <= 8;                       // staged rows of the next chunk fit the registers
        extern __shared__ __attribute__((aligned(16))) char smem[];
        __shared__ float s_carry[LC], s_gate[LC]; // e^(F_t + m0 - m_t), e^(F_end + a_j - m_end)
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
        const int h = blockIdx.y, ei = CUT ? (int)blockIdx.z / p.parts : (int)blockIdx.z, e = p.entry + ei;
        const int chunk0 = first_chunk<LC>(p, ei);
        const int ntok = p.ntok[e], slot = p.slot[e], row0 = p.row0[e];
        const int dim = FULL ? 16 * DT : p.dim;
        const int ldv = p.vdim + 16, ld = dim + LPAD;
        const int col = (blockIdx.x * 4 + wave) * 16 + c;
        const bool live = (blockIdx.x * 4 + wave) * 16 < ldv; // of the wavefront
        const bool ones = (blockIdx.x * 4 + wave) * 16 == p.vdim;
        T *sq = reinterpret_cast<T *>(smem), *sk = sq + LC * ld;
        const int dtiles = FULL ? DT : dim >> 4;

        f32x4 S[DT];
        float *state = p.state + ((size_t)slot * p.heads + h) * dim * ldv + (live ? col : 0);
        const bool fresh = p.pos[e] == 0;
        auto load_state = [&](const float *from) {
#pragma unroll
            for (int t = 0; t < DT; ++t)
                if (t < dtiles)
                {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        S[t][r] = from[(size_t)(16 * t + 4 * g + r) * ldv];
                }
        };
        auto store_state = [&](float *to) {
#pragma unroll
            for (int t = 0; t < DT; ++t)
                if (t < dtiles)
                {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        to[(size_t)(16 * t + 4 * g + r) * ldv] = S[t][r];
                }
        };
        const int chunks = (ntok + LC - 1) / LC, parts = CUT ? memory_stretches(chunks, p.most) : 1;
        const int part = CUT ? (int)blockIdx.z - ei * p.parts : 0;
        if (part >= parts || (SUM && parts == 1))
            return;
        const int stretch = (chunks + parts - 1) / parts * LC, first = part * stretch; // tokens of a stretch, the first of this one
        const bool last = part + 1 == parts;
        const int stop = last || first + stretch > ntok ? ntok : first + stretch;
        const size_t part_floats = (size_t)p.heads * dim * ldv;
        float *starts = p.starts + (size_t)ei * p.parts * part_floats + (size_t)h * dim * ldv + (live ? col : 0);
        float *part_kept = p.kept + (size_t)ei * p.parts * p.heads + h;
#pragma unroll
        for (int t = 0; t < DT; ++t)
            S[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (SUM)
        {
            if (last)
            {
                // the last stretch adds to nobody's start: here the memory before the portion is put aside
                if (!fresh && live)
                {
                    load_state(state);
                    store_state(starts);
                }
                return;
            }
        }
        else if (live)
        {
            if (!fresh)
                load_state(parts > 1 ? starts : state);
            for (int i = 1; CUT && i <= part; ++i)
            {
                const float kept = part_kept[(i - 1) * p.heads];
                const float *add = starts + i * part_floats;
#pragma unroll
                for (int t = 0; t < DT; ++t)
                    if (t < dtiles)
                    {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            S[t][r] = fmaf(S[t][r], kept, add[(size_t)(16 * t + 4 * g + r) * ldv]);
                    }
            }
        }

        const int srow = threadIdx.x / TPR, sseg = threadIdx.x % TPR, pieces = dim * (int)sizeof(T) / 16;
        const T *qrows = static_cast<const T *>(p.qk) + ((size_t)h * p.qk_rows + (size_t)chunk0 * LC) * dim;
        const T *krows = qrows + (size_t)p.heads * p.qk_rows * dim;
        u32x4 hq[AHEAD ? LOADS : 1], hk[AHEAD ? LOADS : 1];
        f32x8 hv[LC / 32];
        double h_ga = 0.0, h_a = 0.0, h_end = 0.0;
        float h_mt = 0.0f;
        auto request = [&](int t0) __attribute__((always_inline)) {
            const int n = ntok - t0 < LC ? ntok - t0 : LC;
            const int r0 = row0 + t0;
            if constexpr (AHEAD)
            {
                // (the product kernel wrote whole chunks: rows past the portion repeat its last one)
                const u32x4 *q = reinterpret_cast<const u32x4 *>(qrows + (size_t)(t0 + srow) * dim) + sseg;
                const u32x4 *k = reinterpret_cast<const u32x4 *>(krows + (size_t)(t0 + srow) * dim) + sseg;
#pragma unroll
                for (int i = 0; i < LOADS; ++i)
                {
                    const int at = sseg + i * TPR < pieces ? i * TPR : 0;
                    if (!SUM)
                        hq[i] = q[at];
                    hk[i] = k[at];
                }
            }
            const size_t end = (size_t)(r0 + n - 1) * p.heads + h;
            const int t = threadIdx.x & (LC - 1);
            const size_t at = (size_t)(r0 + (t < n ? t : n - 1)) * p.heads + h;
            h_ga = p.ga[at];
            h_a = p.a[at];
            h_end = p.ga[end];
            h_mt = p.mt[end];
#pragma unroll
            for (int s = 0; s < LC / 32; ++s)
#pragma unroll
                for (int j = 0; j < 8; ++j)
                {
                    const int tt = 32 * s + 8 * g + j;
                    hv[s][j] = ones || !live ? 0.0f
                                             : p.proj[(size_t)(r0 + (tt < n ? tt : n - 1)) * p.ldp + (size_t)p.heads * 2 * dim + h * p.vdim + col];
                }
        };
        if (first < ntok)
            request(first);
        float m0 = first == 0 ? p.m0[ei * p.heads + h] : first < ntok ? p.mt[(size_t)(row0 + first - 1) * p.heads + h] : 0.0f;
        float kept = 1.0f;
        for (int t0 = first; t0 < stop; t0 += LC)
        {
            const int n = ntok - t0 < LC ? ntok - t0 : LC;
            const int r0 = row0 + t0;
            const float decay = expf((float)(h_end + (double)m0));
            const float m_end = h_mt;
            kept *= decay;
            __syncthreads();
            if (threadIdx.x < LC)
            {
                const int t = threadIdx.x;
                s_carry[t] = t < n ? expf((float)(h_ga + (double)m0)) : 0.0f;
                s_gate[t] = t < n ? expf((float)(h_end + h_a)) : 0.0f;
            }
            {
                u32x4 *dq = reinterpret_cast<u32x4 *>(sq + srow * ld) + sseg, *dk = reinterpret_cast<u32x4 *>(sk + srow * ld) + sseg;
                if constexpr (AHEAD)
                {
#pragma unroll
                    for (int i = 0; i < LOADS; ++i)
                        if (sseg + i * TPR < pieces)
                        {
                            if (!SUM)
                                dq[i * TPR] = hq[i];
                            dk[i * TPR] = hk[i];
                        }
                }
                else
                {
                    const u32x4 *q = reinterpret_cast<const u32x4 *>(qrows + (size_t)(t0 + srow) * dim) + sseg;
                    const u32x4 *k = reinterpret_cast<const u32x4 *>(krows + (size_t)(t0 + srow) * dim) + sseg;
#pragma unroll 4
                    for (int i = 0; sseg + i < pieces; i += TPR)
                    {
                        if (!SUM)
                            dq[i] = q[i];
                        dk[i] = k[i];
                    }
                }
            }
            f32x8 x[LC / 32];
#pragma unroll
            for (int s = 0; s < LC / 32; ++s)
                x[s] = hv[s];
            __syncthreads();
            // the chunk's products, 16 rows at a time (a row block needs columns up to its own)
            const float *prod = p.prod + ((size_t)(chunk0 + t0 / LC) * p.heads + h) * LC * LC;
            f32x8 w[LC / 16][LC / 32];
#pragma unroll
            for (int i = 0; i < LC / 16; ++i)
#pragma unroll
                for (int s = 0; s < LC / 32; ++s)
                    if (!SUM && 32 * s <= 16 * i + 15)
                        w[i][s] = Operand<float>::load(prod + (16 * i + c) * LC + 32 * s + 8 * g);
            if (t0 + LC < stop)
                request(t0 + LC);
            if (live)
            {
                // values of this column, as they are and gated
                V v[LC / 32], gv[LC / 32][NP];
#pragma unroll
                for (int s = 0; s < LC / 32; ++s)
                {
                    if (ones)
                    {
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            x[s][j] = c == 0 && 32 * s + 8 * g + j < n ? 1.0f : 0.0f;
                    }
                    V one[1];
                    split_pieces<T, 1>(x[s], one);
                    v[s] = one[0];
                    f32x8 y;
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        y[j] = (float)one[0][j] * s_gate[32 * s + 8 * g + j];
                    split_pieces<T, NP>(y, gv[s]);
                }
                if constexpr (!SUM)
                {
                    // carried part: q . S
                    f32x4 out[LC / 16];
#pragma unroll
                    for (int i = 0; i < LC / 16; ++i)
                        out[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int t = 0; t < DT; t += 2)
                        if (t < dtiles)
                        {
                            V b[NP], a[LC / 16];
                            split_pieces<T, NP>(__builtin_shufflevector(S[t], S[t + 1], 0, 1, 2, 3, 4, 5, 6, 7), b);
#pragma unroll
                            for (int i = 0; i < LC / 16; ++i)
                            {
                                const T *qr = sq + (16 * i + c) * ld + 16 * t + 4 * g;
                                const t4 lo = *reinterpret_cast<const t4 *>(qr), hi = *reinterpret_cast<const t4 *>(qr + 16);
                                a[i] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                            }
#pragma unroll
                            for (int k = 0; k < NP; ++k)
#pragma unroll
                                for (int i = 0; i < LC / 16; ++i)
                                    out[i] = O::mma(a[i], b[k], out[i]);
                        }
                    // plus the chunk's own tokens
#pragma unroll
                    for (int i = 0; i < LC / 16; ++i)
                    {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            out[i][r] *= s_carry[16 * i + 4 * g + r];
                    }
#pragma unroll
                    for (int s = 0; s < LC / 32; ++s)
#pragma unroll
                        for (int i = 0; i < LC / 16; ++i)
                            if (32 * s <= 16 * i + 15)
                            {
                                V q[NP];
                                split_pieces<T, NP>(w[i][s], q);
#pragma unroll
                                for (int k = 0; k < NP; ++k)
                                    out[i] = O::mma(q[k], v[s], out[i]);
                            }
#pragma unroll
                    for (int i = 0; i < LC / 16; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                        {
                            const int t = 16 * i + 4 * g + r;
                            if (t < n)
                                p.num[((size_t)(r0 + t) * p.heads + h) * ldv + col] = out[i][r];
                        }
                }
                // S of the next chunk
#pragma unroll
                for (int t = 0; t < DT; ++t)
                    if (t < dtiles)
                    {
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            S[t][r] *= decay;
                    }
#pragma unroll
                for (int t = 0; t < DT; t += 4)
                    if (t < dtiles)
                    {
#pragma unroll
                        for (int s = 0; s < LC / 32; ++s)
                        {
                            V k[4];
#pragma unroll
                            for (int u = 0; u < 4; ++u)
                                k[u] = load_columns(sk + 32 * s * ld + 16 * (t + u), ld, lane);
#pragma unroll
                            for (int i = 0; i < NP; ++i)
#pragma unroll
                                for (int u = 0; u < 4; ++u)
                                    S[t + u] = O::mma(k[u], gv[s][i], S[t + u]);
                        }
                    }
            }
            m0 = m_end;
        }
        if (SUM)
        {
            if (live)
                store_state(starts + (part + 1) * part_floats);
            if (blockIdx.x == 0 && threadIdx.x == 0)
                part_kept[part * p.heads] = kept;
        }
        else if (live && last)
            store_state(state);
    }

    // ---- output: normaliser, head norm, gate ------------------------------------------------------------
    // Workgroup = one head of one row.  DECODE: also the new running maximum of the sequence.
    template <typename T, bool DECODE>
    __global__ void __launch_bounds__(128)
        memory_output_kernel(MemoryArgs p)
    {
        __shared__ float s_sum[2];
        const int h = blockIdx.x;
        const int e = p.entry + (DECODE ? blockIdx.y : blockIdx.z);
        if (!DECODE && (int)blockIdx.y >= p.ntok[e])
            return;
        const int r = DECODE ? p.row0[e] : p.row0[e] + blockIdx.y;
        const float *row = p.proj + (size_t)r * p.ldp;
        const int ldv = p.vdim + 16;
        const int splits = DECODE ? p.splits : 1;
        const float *num = p.num + ((size_t)(DECODE ? blockIdx.y : r) * p.heads + h) * splits * ldv;
        float m;
        if (DECODE)
        {
            float gi, gf;
            memory_gates(p, row, h, gi, gf);
            float *keep = p.m + p.slot[e] * p.heads + h;
            m = fmaxf(gf + (p.pos[e] == 0 ? 0.0f : *keep), gi);
            __syncthreads();
            if (threadIdx.x == 0)
                *keep = m;
        }
        else
            m = p.mt[(size_t)r * p.heads + h];
        // columns 4 threadIdx.x .. + 3, and 512 further on (the first are kept for the second pass)
        auto total = [&](int d) {
            f32x4 o = *reinterpret_cast<const f32x4 *>(num + d);
            for (int k = 1; k < splits; ++k)
                o = o + *reinterpret_cast<const f32x4 *>(num + (size_t)k * ldv + d);
            return o;
        };
        const float inv = 1.0f / (fmaxf(fabsf(total(p.vdim)[0]), expf(-m)) + 1e-6f);
        const int d0 = threadIdx.x * 4;
        f32x4 kept = {0.0f, 0.0f, 0.0f, 0.0f};
        float sum = 0.0f;
        for (int d = d0; d < p.vdim; d += 512)
        {
            const f32x4 o = total(d) * inv;
            if (d == d0)
                kept = o;
            sum += o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
        }
        sum = block_sum<128>(sum, s_sum);
        const float scale = 1.0f / sqrtf(sum / (float)p.vdim_real + p.eps);
        const float *gate = row + (size_t)p.heads * (2 * p.dim + p.vdim) + h * p.vdim;
        typedef T t4 __attribute__((ext_vector_type(4)));
        T *y = static_cast<T *>(p.y) + (size_t)r * p.ldy + h * p.vdim;
        for (int d = d0; d < p.vdim; d += 512)
        {
            f32x4 o = (d == d0 ? kept : total(d) * inv) * scale * *reinterpret_cast<const f32x4 *>(p.norm + h * p.vdim + d);
            const f32x4 z = *reinterpret_cast<const f32x4 *>(gate + d);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                o[k] *= sigmoidf(z[k]);
            *reinterpret_cast<t4 *>(y + d) = __builtin_convertvector(o, t4);
        }
    }

    namespace
    {
        constexpr int LC16 = 64, LC32 = 32; // chunk lengths of the two number formats
        constexpr int CUT_TILES = 16;                    // 16-row tiles of S up to which a portion is cut into stretches
        constexpr int MANY = 16;                         // portions of a launch at most
        constexpr int STRETCHES = 8;                     // stretches of a portion at most, and that there is room for
        constexpr int STEP_SPLIT_ENTRIES = 32; // sequences up to which a decoding step splits the rows of S (in at most 8)

        struct MemoryScratch
        {
            size_t ga, a, mt, m0, prod, num, qk, starts, kept, total;
        };
        // Stretches that the scratch of `rows` has room for (the shorter chunks: the most that any portion has).
        int stretch_room(int rows, int dim) { return dim > 16 * CUT_TILES ? 1 : memory_stretches(ceil_div(rows, LC32), STRETCHES); }
        // rows of whole chunks; of several portions each has some of its own
        int kept_rows(int rows, int portions) { return round_up(rows, LC16) + (portions > 1 ? portions * LC16 : 0); }
        MemoryScratch memory_scratch(int rows, int portions, int heads, int dim, int vdim)
        {
            MemoryScratch s{};
            size_t at = 0;
            auto take = [&at](size_t bytes) {
                const size_t here = at;
                at += (bytes + 255) & ~(size_t)255;
                return here;
            };
            s.ga = take((size_t)rows * heads * 8);
            s.a = take((size_t)rows * heads * 8);
            s.mt = take((size_t)rows * heads * 4);
            s.m0 = take((size_t)portions * heads * 4);
            const size_t kept = kept_rows(rows, portions);
            s.prod = take(kept * heads * LC16 * 4);
            const size_t outs = (size_t)(rows > STEP_SPLIT_ENTRIES * 8 ? rows : STEP_SPLIT_ENTRIES * 8);
            s.num = take(outs * heads * (vdim + 16) * 4);
            s.qk = take((size_t)2 * heads * kept * dim * 4);
            const int stretches = stretch_room(rows, dim);
            s.starts = take(stretches > 1 ? (size_t)stretches * heads * dim * (vdim + 16) * 4 : 0);
            s.kept = take((size_t)stretches * heads * 4);
            s.total = at;
            return s;
        }

        bool memory_args(const char *fn, const llam_seq_memory_args *a, const llam_seq_entries *e, void *d_scratch,
                         int dtype, MemoryArgs &p)
        {
            if (!a || !e || !a->d_proj || !a->d_gate_bias || !a->d_norm || !a->d_state || !a->d_m || !a->d_y || !d_scratch ||
                !e->d_row0 || !e->d_ntok || !e->d_slot || !e->d_pos)
                return fail(fn, "null pointer");
            if (dtype != LLAM_SEQ_BF16 && dtype != LLAM_SEQ_F32)
                return fail(fn, "dtype %d", dtype);
            if (a->heads < 1 || a->heads > 65535 || a->dim < 1 || a->dim > 512 || (a->dim % PAD) != 0 || a->vdim < 1 || (a->vdim % PAD) != 0 ||
                a->vdim_real < 1 || a->vdim_real > a->vdim)
                return fail(fn, "heads=%d dim=%d vdim=%d: dim up to 512, both multiples of %d", a->heads, a->dim, a->vdim, PAD);
            if (a->ldp < a->heads * (2 * a->dim + 2 * a->vdim + 2) || (a->ldp % 4) != 0 || !aligned16(a->d_proj))
                return fail(fn, "ldp=%d too small or rows misaligned", a->ldp);
            if (a->ldy < a->heads * a->vdim || (a->ldy % 8) != 0)
                return fail(fn, "ldy=%d too small or rows misaligned", a->ldy);
            if (!(a->gate_cap > 0.0f))
                return fail(fn, "gate_cap must be positive");
            p = MemoryArgs{};
            p.proj = a->d_proj, p.ldp = a->ldp, p.gate_bias = a->d_gate_bias, p.norm = a->d_norm, p.state = a->d_state;
            p.m = a->d_m, p.y = a->d_y, p.ldy = a->ldy, p.heads = a->heads, p.dim = a->dim, p.vdim = a->vdim, p.vdim_real = a->vdim_real;
            p.q_scale = a->q_scale, p.gate_cap = a->gate_cap, p.eps = a->eps;
            p.row0 = e->d_row0, p.ntok = e->d_ntok, p.slot = e->d_slot, p.pos = e->d_pos;
            return true;
        }
        void place_scratch(MemoryArgs &p, void *d_scratch, size_t scratch_bytes, int portions)
        {
            // rows of the step are absolute, so the offsets are those of the whole buffer: the largest
            // row count whose scratch fits
            int rows = 64;
            while (memory_scratch(rows + 64, portions, p.heads, p.dim, p.vdim).total <= scratch_bytes)
                rows += 64;
            const MemoryScratch at = memory_scratch(rows, portions, p.heads, p.dim, p.vdim);
            char *s = static_cast<char *>(d_scratch);
            p.ga = reinterpret_cast<double *>(s + at.ga), p.a = reinterpret_cast<double *>(s + at.a);
            p.mt = reinterpret_cast<float *>(s + at.mt), p.m0 = reinterpret_cast<float *>(s + at.m0);
            p.prod = reinterpret_cast<float *>(s + at.prod), p.num = reinterpret_cast<float *>(s + at.num);
            p.qk = s + at.qk, p.qk_rows = kept_rows(rows, portions);
            p.parts = stretch_room(rows, p.dim); // (as many as there is room for)
            p.starts = reinterpret_cast<float *>(s + at.starts), p.kept = reinterpret_cast<float *>(s + at.kept);
        }

        template <typename T, int LC, int DT, bool FULL, bool CUT, bool SUM>
        bool chunk_launch_one(const char *fn, const MemoryArgs &p, int n, hipStream_t st)
        {
            static LdsGrant grant;
            const size_t lds = (size_t)2 * LC * (p.dim + 16 / sizeof(T)) * sizeof(T);
            const auto kernel = &memory_chunk_kernel<T, LC, DT, FULL, CUT, SUM>;
            if (lds > 48 * 1024 && allow_lds(grant, reinterpret_cast<const void *>(kernel), 140 * 1024) != hipSuccess)
                return fail(fn, "cannot reserve %zu bytes of LDS", lds);
            hipLaunchKernelGGL(kernel, dim3(ceil_div(p.vdim + 16, 64), p.heads, p.parts * n), dim3(256), lds, st, p);
            return launched(fn);
        }
        template <typename T, int LC, int DT, bool FULL>
        bool chunk_launch_as(const char *fn, const MemoryArgs &p, int n, hipStream_t st)
        {
            if constexpr (DT <= CUT_TILES)
                return (p.parts == 1 || chunk_launch_one<T, LC, DT, FULL, true, true>(fn, p, n, st)) &&
                       chunk_launch_one<T, LC, DT, FULL, true, false>(fn, p, n, st);
            else
                return chunk_launch_one<T, LC, DT, FULL, false, false>(fn, p, n, st);
        }
        template <typename T, int LC, int DT>
        bool chunk_launch(const char *fn, const MemoryArgs &p, int n, hipStream_t st)
        {
            if constexpr (sizeof(T) == 2)
            {
                if (p.dim == 16 * DT)
                    return chunk_launch_as<T, LC, DT, true>(fn, p, n, st);
            }
            return chunk_launch_as<T, LC, DT, false>(fn, p, n, st);
        }
        template <typename T, int LC>
        bool prefill_run(const char *fn, MemoryArgs p, int n, int ntok, int cus, hipStream_t st)
        {
            // (a workgroup fills a compute unit: no second round of a portion's)
            const int room = p.parts;
            p.most = p.dim > 16 * CUT_TILES ? 1 : std::min(STRETCHES, cus / (ceil_div(p.vdim + 16, 64) * p.heads));
            p.parts = memory_stretches(ceil_div(ntok, LC), p.most);
            if (p.parts > 1 && n > room / p.parts) // as many portions at a time as there is room for the stretches of
            {
                const int few = room / p.parts, entry = p.entry;
                p.parts = room;
                for (int k = 0; k < n; k += few)
                {
                    p.entry = entry + k;
                    if (!prefill_run<T, LC>(fn, p, std::min(few, n - k), ntok, cus, st))
                        return false;
                }
                return true;
            }
            hipLaunchKernelGGL(memory_gates_kernel<LC>, dim3(p.heads, n), dim3(GATE_WAVES * 64), 0, st, p);
            if (!launched(fn))
                return false;
            hipLaunchKernelGGL((memory_product_kernel<T, LC>), dim3(ceil_div(ntok, LC), p.heads, n), dim3(LC * 4), 0, st, p);
            if (!launched(fn))
                return false;
            const bool ok = p.dim <= 64 ? chunk_launch<T, LC, 4>(fn, p, n, st) : p.dim <= 128 ? chunk_launch<T, LC, 8>(fn, p, n, st)
                            : p.dim <= 256 ? chunk_launch<T, LC, 16>(fn, p, n, st) : chunk_launch<T, LC, 32>(fn, p, n, st);
            if (!ok)
                return false;
            hipLaunchKernelGGL((memory_output_kernel<T, false>), dim3(p.heads, ntok, n), dim3(128), 0, st, p);
            return launched(fn);
        }
        template <typename T>
        bool decode_run(const char *fn, MemoryArgs p, int n, hipStream_t st)
        {
            p.splits = n <= STEP_SPLIT_ENTRIES ? p.dim / STEP_ROWS : 1;
            hipLaunchKernelGGL(memory_step_kernel<T>, dim3(ceil_div(p.vdim + 16, 64) * p.splits, p.heads, n), dim3(256), 0, st, p);
            if (!launched(fn))
                return false;
            hipLaunchKernelGGL((memory_output_kernel<T, true>), dim3(p.heads, n), dim3(128), 0, st, p);
            return launched(fn);
        }
    } // namespace
} // namespace llamql

using namespace llamql;

extern "C" size_t llam_seq_memory_scratch_bytes(int max_rows, int heads, int dim, int vdim)
{
    return llam_seq_memory_portions_scratch_bytes(max_rows, MANY, heads, dim, vdim);
}

extern "C" size_t llam_seq_memory_portions_scratch_bytes(int max_rows, int portions, int heads, int dim, int vdim)
{
    if (max_rows < 1 || portions < 1 || heads < 1 || dim < 1 || vdim < 1)
        return 0;
    return memory_scratch(round_up(max_rows, LC16), portions < MANY ? portions : MANY, heads, dim, vdim).total;
}

extern "C" bool llam_seq_memory_decode(const llam_seq_memory_args *a, const llam_seq_entries *e, int first, int n,
                                       void *d_scratch, size_t scratch_bytes, int dtype, int device_id, void *stream)
{
    static const char *fn = "llam_seq_memory_decode";
    MemoryArgs p;
    if (n < 0 || first < 0 || n > 65535)
        return fail(fn, "bad size (first=%d n=%d)", first, n);
    if (n == 0)
        return true;
    if (!memory_args(fn, a, e, d_scratch, dtype, p))
        return false;
    if (llam_seq_memory_portions_scratch_bytes(first + n, 1, p.heads, p.dim, p.vdim) > scratch_bytes)
        return fail(fn, "scratch too small");
    p.entry = first;
    place_scratch(p, d_scratch, scratch_bytes, 1);
    if (!set_device(fn, device_id))
        return false;
    return dtype == LLAM_SEQ_F32 ? decode_run<float>(fn, p, n, as_stream(stream)) : decode_run<bf16>(fn, p, n, as_stream(stream));
}

extern "C" bool llam_seq_memory_prefill(const llam_seq_memory_args *a, const llam_seq_entries *e, int entry, int ntok,
                                        void *d_scratch, size_t scratch_bytes, int dtype, int device_id, void *stream)
{
    return llam_seq_memory_prefill_many(a, e, entry, 1, ntok, ntok, d_scratch, scratch_bytes, dtype, device_id, stream);
}

extern "C" bool llam_seq_memory_prefill_many(const llam_seq_memory_args *a, const llam_seq_entries *e, int first, int n, int max_ntok,
                                             int rows, void *d_scratch, size_t scratch_bytes, int dtype, int device_id, void *stream)
{
    static const char *fn = "llam_seq_memory_prefill";
    MemoryArgs p;
    if (n < 0 || max_ntok < 0 || first < 0 || max_ntok > 65535 || rows < max_ntok)
        return fail(fn, "bad size (first=%d n=%d ntok=%d rows=%d)", first, n, max_ntok, rows);
    if (n == 0 || max_ntok == 0)
        return true;
    if (!memory_args(fn, a, e, d_scratch, dtype, p))
        return false;
    const int portions = n < MANY ? n : MANY;
    if (llam_seq_memory_portions_scratch_bytes(rows, portions, p.heads, p.dim, p.vdim) > scratch_bytes)
        return fail(fn, "scratch too small");
    place_scratch(p, d_scratch, scratch_bytes, portions);
    if (!set_device(fn, device_id))
        return false;
    p.many = n > 1;
    for (int k = 0; k < n; k += MANY)
    {
        const int some = n - k < MANY ? n - k : MANY;
        p.entry = first + k;
        if (!(dtype == LLAM_SEQ_F32 ? prefill_run<float, LC32>(fn, p, some, max_ntok, cu_count(device_id), as_stream(stream))
                                    : prefill_run<bf16, LC16>(fn, p, some, max_ntok, cu_count(device_id), as_stream(stream))))
            return false;
    }
    return true;
}
