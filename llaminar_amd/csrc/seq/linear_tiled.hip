// Linear layers of many rows (prompts) for gfx950: y = A W^T, W in matrix-unit tiles.
//
// Both operands go from global memory straight into LDS, some turns of 64 columns ahead, and from there into registers
// one sixteen-column step ahead of the products, across the one barrier of a turn.  W is the first operand, so a lane
// ends with four neighbouring output columns of one row; results go through LDS so that they leave by whole lines.  32-bit rows are multiplied in three bf16 pieces that add up to
// them (weights are bf16 anyway): the products stay exact, the sums 32-bit, on a unit that is 16 times as fast.
//
// What bounds it, 2048 x 15440 x 5120 in bf16: the matrix unit is busy in 57 % of the cycles, at the 1.9 GHz that the chip
// holds under this load; without any loads of A and W the same loop takes 260 instead of 285 us, LDS conflicts are none.
// Time before (128 x 128 tiles staged through registers) and now: 390 -> 285 us (830 -> 1140 TFLOP/s), 2048 x 51200 x
// 5120 1200 -> 940 us, 300 x 2048 x 8192 63 -> 28 us; 32-bit rows (v_mfma_f32_16x16x4 before) 2048 x 51200 x 5120 9490 ->
// 2480 us, 522 x 2048 x 10240 380 -> 126 us.
#include "linear.h"

#include <type_traits>

namespace llamql
{
    typedef float f32x16 __attribute__((ext_vector_type(16)));

    constexpr int TILE_K = 64; // columns of K per turn and group of wavefronts

    // 16 bytes a lane from global memory into LDS, at lds + lane * 16: no registers, no LDS store instructions.
    // vmcnt counts these loads in order.
    __device__ __forceinline__ void load_to_lds(const void *from, uint32_t lds)
    {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(from) : "memory");
    }
    // This wavefront's loads have arrived but for the newest N, what it asked the LDS for is in registers, and all
    // wavefronts are as far.
    template <int N>
    __device__ __forceinline__ void arrive()
    {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"(N) : "memory");
    }

    // A 32-bit value as three bf16 values that add up to it: 8 + 8 + 8 significant bits, cut off and not rounded, so that
    // none is larger than the value.  Of an infinity the second piece is not a number, nor are the sums then: those are made
    // again without pieces (see pieces_fail).
    __device__ __forceinline__ void three_pieces(f32x8 x, bf16x8 (&out)[3])
    {
        f32x8 r;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            r[e] = x[e] - __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, (float)x[e]) & 0xffff0000u);
        u32x4 p[3];
#pragma unroll
        for (int k = 0; k < 4; ++k)
        {
            uint32_t t[2][3];
#pragma unroll
            for (int e = 0; e < 2; ++e)
            {
                t[e][0] = __builtin_bit_cast(uint32_t, (float)x[2 * k + e]);
                t[e][1] = __builtin_bit_cast(uint32_t, (float)r[2 * k + e]);
                t[e][2] = __builtin_bit_cast(uint32_t, r[2 * k + e] - __builtin_bit_cast(float, t[e][1] & 0xffff0000u));
            }
#pragma unroll
            for (int i = 0; i < 3; ++i)
                p[i][k] = __builtin_amdgcn_perm(t[1][i], t[0][i], 0x07060302u); // the upper halves of both
        }
#pragma unroll
        for (int i = 0; i < 3; ++i)
            out[i] = __builtin_bit_cast(bf16x8, p[i]);
    }

    constexpr int OUT_BYTES = 4096; // 32 x 32 results
    // 16 bytes of results into a row of y (whole: rows of 16-bit values start at 16 bytes, else at 8)
    __device__ __forceinline__ void store_piece(const LinearArgs &p, char *y, bool, int row, int col, f32x4 v)
    {
        f32x4 *at = reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(y) + (size_t)row * p.ldy + col);
        if (p.out == LLAM_SEQ_OUT_F32 && p.bias)
        {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                v[r] += p.bias[col + r];
        }
        if (p.out == LLAM_SEQ_OUT_ADD)
            v = *at + v;
        *at = v;
    }
    __device__ __forceinline__ void store_piece(const LinearArgs &p, char *y, bool whole, int row, int col, bf16x8 v)
    {
        bf16 *at = reinterpret_cast<bf16 *>(y) + (size_t)row * p.ldy + col;
        if (whole)
            *reinterpret_cast<bf16x8 *>(at) = v;
        else
        {
            reinterpret_cast<bf16x4 *>(at)[0] = __builtin_shufflevector(v, v, 0, 1, 2, 3);
            reinterpret_cast<bf16x4 *>(at)[1] = __builtin_shufflevector(v, v, 4, 5, 6, 7);
        }
    }

    template <typename T>
    struct TiledOperand;
    template <>
    struct TiledOperand<bf16>
    {
        using Raw = bf16x8;
        static constexpr int PIECES = 1;
        static __device__ __forceinline__ void pieces(Raw x, bf16x8 (&out)[1]) { out[0] = x; }
    };
    template <>
    struct TiledOperand<float>
    {
        using Raw = f32x8;
        static constexpr int PIECES = 3;
        static __device__ __forceinline__ void pieces(Raw x, bf16x8 (&out)[3]) { three_pieces(x, out); }
    };

    // Workgroup tile BM rows of A x BN rows of W; KG groups of WM x WN wavefronts, each with every KG-th turn of 64
    // columns, STAGES turns of LDS.
    template <typename T, int BM, int BN, int WM, int WN, int KG, int STAGES>
    __global__ void __launch_bounds__(WM *WN *KG * 64)
        linear_wide_kernel(LinearArgs p, int m_tiles, int n_tiles)
    {
        using O = TiledOperand<T>;
        constexpr int NW = WM * WN;                         // wavefronts of a group
        constexpr int TM = BM / WM / 32, TN = BN / WN / 32; // 32x32 products of a wavefront
        constexpr int AROW = TILE_K * sizeof(T), AROWS = 1024 / AROW, APIECES = AROW / 16; // bytes; rows of a load; 16-byte pieces
        constexpr int ALOADS = BM / AROWS / NW, WLOADS = BN / 8 / NW, LOADS = ALOADS + WLOADS; // of a turn, per wavefront
        constexpr int ABYTES = BM * AROW, STAGE = ABYTES + BN * TILE_K * 2;
        static_assert(BM % (AROWS * NW) == 0 && BN % (8 * NW) == 0 && TM >= 1 && TN >= 1, "whole loads and products");
        static_assert(STAGES >= 2 && (STAGES - 1) * LOADS < 64, "counted by six bits");
        extern __shared__ __attribute__((aligned(16))) char smem[];
        const int lane = threadIdx.x & 63, all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int kg = KG == 1 ? 0 : all / NW, wave = KG == 1 ? all : all % NW;
        const int c = lane & 31, h = lane >> 5;
        const int wm = wave % WM, wn = wave / WM;

        // groups g0 .. g0 + 63, one a lane: its first row, rows and tiles; returns the tiles up to the lane's
        int lo = 0, n = 0, tiles = 0;
        auto look = [&](int g0) __attribute__((always_inline)) {
            const int e = g0 + lane < p.groups ? g0 + lane : p.groups - 1;
            lo = p.group_offset[e], n = g0 + lane < p.groups ? p.group_offset[e + 1] - lo : 0;
            tiles = (n + BM - 1) / BM;
            int upto = tiles;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1)
            {
                const int o = __shfl_up(upto, off, 64);
                upto += lane >= off ? o : 0;
            }
            return upto;
        };
        int upto = 0;
        if (p.group_offset)
        {
            // the tiles of rows that there are: dealt out by the most there can be, the first dies would get them all (300 rows,
            // 8 of 128 experts of 768 x 2048 each, mostly of the first 40: 182 -> 123 us, of all of them: 210 -> 193)
            int live = 0;
            for (int g0 = (p.groups - 1) / 64 * 64; g0 >= 0; g0 -= 64)
            {
                upto = look(g0);
                live += __shfl(upto, 63, 64);
            }
            m_tiles = __builtin_amdgcn_readfirstlane(live);
        }
        // neighbouring tiles go to one die (blocks are dealt round robin over the eight dies), eight tiles of rows side
        // by side, then the next tile of W: what a die works on at a time is about square
        const int total = m_tiles * n_tiles;
        int id = blockIdx.x;
        if (id >= total)
            return;
        const int per = total / 8;
        if (id < per * 8)
            id = (id & 7) * per + (id >> 3);
        const int band = id / (8 * n_tiles), in = id - band * 8 * n_tiles;
        const int high = m_tiles - band * 8 < 8 ? m_tiles - band * 8 : 8;
        const int nt = in / high;
        int mt = band * 8 + in - nt * high;
        int z = blockIdx.y, row0 = 0, rows = p.M;
        if (p.group_offset)
        {
            // the mt-th tile of rows among those of all groups
            const int want = mt;
            int seen = 0;
            z = -1;
            for (int g0 = 0; g0 < p.groups; g0 += 64)
            {
                if (g0 > 0) // (the first ones were looked at last)
                    upto = look(g0);
                const unsigned long long past = __ballot(seen + upto > want);
                if (past)
                {
                    const int who = __builtin_ctzll(past);
                    z = g0 + who;
                    row0 = __shfl(lo, who, 64);
                    rows = __shfl(n, who, 64);
                    mt = want - (seen + __shfl(upto - tiles, who, 64));
                    break;
                }
                seen += __shfl(upto, 63, 64);
            }
            if (z < 0)
                return;
            z = __builtin_amdgcn_readfirstlane(z), row0 = __builtin_amdgcn_readfirstlane(row0);
            rows = __builtin_amdgcn_readfirstlane(rows), mt = __builtin_amdgcn_readfirstlane(mt);
        }
        const T *abase = static_cast<const T *>(p.a) + (size_t)z * p.a_stride;
        const char *wbase = reinterpret_cast<const char *>(static_cast<const bf16 *>(p.w) + (size_t)z * p.w_stride);
        const int ksteps = p.K >> 5, w_tiles = p.N >> 4, turns = p.K / TILE_K;
        const int rounds = (turns + KG - 1) / KG; // the group's turn k is columns 64 (k KG + kg) .. of K
        const int first = kg < turns ? kg : turns - 1;

        // Where the wavefront's loads come from: load i of A fills rows AROWS (wave + i NW) .. of the stage, a lane
        // one 16-byte piece.  Pieces of a row are permuted so that one piece of 16 rows lies in 16 different banks:
        // place q of row r holds piece q ^ spread(r).
        auto swizzle = [](int r) __attribute__((always_inline)) { return sizeof(T) == 2 ? (r >> 1) & 7 : r & 15; };
        const char *src[LOADS];
#pragma unroll
        for (int i = 0; i < ALOADS; ++i)
        {
            const int r = (wave + i * NW) * AROWS + lane / APIECES, q = lane % APIECES;
            int m = mt * BM + r;
            m = row0 + (m < rows ? m : rows - 1);
            if (p.row_source)
                m = p.row_source[m] / p.source_div;
            src[i] = reinterpret_cast<const char *>(abase + (size_t)m * p.lda + first * TILE_K) + (q ^ swizzle(r)) * 16;
        }
#pragma unroll
        for (int i = 0; i < WLOADS; ++i)
        {
            const int k = wave + i * NW; // kilobyte k of the stage: k-step k & 1 of its tile k / 2
            int tile = nt * (BN / 16) + (k >> 1);
            tile = tile < w_tiles ? tile : w_tiles - 1;
            src[ALOADS + i] = wbase + ((size_t)tile * ksteps + 2 * first + (k & 1)) * 1024 + lane * 16;
        }
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)smem;
        // load i of turn t into its buffer; a group without a turn t reads its last one again, which nothing uses
        auto issue = [&](int i, int buf, int t) __attribute__((always_inline)) {
            const uint32_t at = lds0 + (buf * KG + kg) * STAGE + wave * 1024;
            load_to_lds(src[i], at + (i < ALOADS ? i * NW * 1024 : ABYTES + (i - ALOADS) * NW * 1024));
            if (KG == 1 || (t + 1) * KG + kg < turns)
                src[i] += KG * (i < ALOADS ? AROW : 2048);
        };

        f32x16 acc[TN][TM];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    acc[j][i][r] = 0.0f;

#pragma unroll
        for (int t = 0; t < STAGES; ++t)
            if (t < rounds)
            {
#pragma unroll
                for (int i = 0; i < LOADS; ++i)
                    issue(i, t, t);
            }
        const int arow = (wm * TM * 32 + c) * AROW, wrow = ABYTES + (wn * TN * 2 + (c >> 4)) * 2048 + (h * 16 + (c & 15)) * 16;
        typename O::Raw a[2][TM];
        bf16x8 w[2][TN];
        // operand n of the 16 columns s of a stage (k-step s / 2 of W, its pieces 2 (s & 1) + h): A's first, W's, A's others
        auto read = [&](int buf, int s, int b, int n) __attribute__((always_inline)) {
            const char *at = smem + (buf * KG + kg) * STAGE;
            if (n >= 1 && n <= TN)
                w[b][n - 1] = *reinterpret_cast<const bf16x8 *>(at + wrow + (n - 1) * 4096 + (s >> 1) * 1024 + (s & 1) * 512);
            else
            {
                const int i = n == 0 ? 0 : n - TN;
                const char *row = at + arow + i * 32 * AROW;
                if constexpr (sizeof(T) == 2)
                    a[b][i] = *reinterpret_cast<const bf16x8 *>(row + ((2 * s + h) ^ swizzle(c)) * 16);
                else
                    a[b][i] = __builtin_shufflevector(*reinterpret_cast<const f32x4 *>(row + ((4 * s + 2 * h) ^ swizzle(c)) * 16),
                                                      *reinterpret_cast<const f32x4 *>(row + ((4 * s + 2 * h + 1) ^ swizzle(c)) * 16), 0, 1, 2, 3, 4, 5, 6, 7);
            }
        };
        // the products of the operands b, in this order, with what `between` asks for after each: left to itself the
        // compiler asks for operands just before it needs them
        auto multiply = [&](int b, auto between) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
            {
                bf16x8 piece[O::PIECES];
                O::pieces(a[b][i], piece);
#pragma unroll
                for (int j = 0; j < TN; ++j)
                {
#pragma unroll
                    for (int k = O::PIECES - 1; k >= 0; --k)
                        acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[b][j], piece[k], acc[j][i], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                    between(i * TN + j);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        // f(0) .. f(count - 1), dealt to the products
        auto deal = [&](int n, auto f, int count) __attribute__((always_inline)) {
            const int each = (count + TN * TM - 1) / (TN * TM);
#pragma unroll
            for (int k = 0; k < 16; ++k)
                if (k < each && n * each + k < count)
                    f(n * each + k);
        };
        if (rounds >= STAGES)
            arrive<(STAGES - 1) * LOADS>();
        else
            arrive<0>();
#pragma unroll
        for (int n = 0; n < TM + TN; ++n)
            read(0, 0, 0, n);
        int buf = 0;
        for (int t = 0; t < rounds - 1; ++t)
        {
            const int next = buf + 1 < STAGES ? buf + 1 : 0;
#pragma unroll
            for (int s = 0; s < 3; ++s)
                multiply(s & 1, [&](int n) { deal(n, [&](int k) { read(buf, s + 1, (s + 1) & 1, k); }, TM + TN); });
            // this stage is in registers; the next one has arrived, later ones may be on their way
            if (t + STAGES <= rounds)
                arrive<(STAGES - 2) * LOADS>();
            else
                arrive<0>();
            const bool more = t + STAGES < rounds;
            multiply(1, [&](int n) {
                deal(n, [&](int k) { read(next, 0, 0, k); }, TM + TN);
                if (more)
                    deal(n, [&](int k) { issue(k, buf, t + STAGES); }, LOADS);
            });
            buf = next;
        }
        if (KG == 1 || (rounds - 1) * KG + kg < turns)
        {
#pragma unroll
            for (int s = 0; s < 3; ++s)
                multiply(s & 1, [&](int n) { deal(n, [&](int k) { read(buf, s + 1, (s + 1) & 1, k); }, TM + TN); });
            multiply(1, [](int) {});
        }

        if constexpr (KG > 1)
        {
            // the groups' sums, added in their order
            arrive<0>();
            f32x4 *sums = reinterpret_cast<f32x4 *>(smem) + wave * (TN * TM * 256) + lane;
            if (kg > 0)
            {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            sums[(kg - 1) * NW * TN * TM * 256 + ((j * TM + i) * 4 + q) * 64] =
                                f32x4{acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
            }
            __syncthreads();
            if (kg > 0)
                return;
#pragma unroll
            for (int k = 0; k < KG - 1; ++k)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                        {
                            const f32x4 v = sums[k * NW * TN * TM * 256 + ((j * TM + i) * 4 + q) * 64];
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                acc[j][i][4 * q + r] += v[r];
                        }
        }

        if constexpr (sizeof(T) == 4)
        {
            // sums that the pieces do not carry (see pieces_fail), once more as products of the whole values, straight from memory
            bool fail = false;
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        fail |= pieces_fail(acc[j][i][r]);
            if (__builtin_expect(__ballot(fail) != 0, 0))
            {
                const float *rows_of_a[TM];
                const bf16x8 *rows_of_w[TN];
#pragma unroll
                for (int i = 0; i < TM; ++i)
                {
                    int m = mt * BM + (wm * TM + i) * 32 + c;
                    m = row0 + (m < rows ? m : rows - 1);
                    if (p.row_source)
                        m = p.row_source[m] / p.source_div;
                    rows_of_a[i] = abase + (size_t)m * p.lda + 8 * h;
                }
#pragma unroll
                for (int j = 0; j < TN; ++j)
                {
                    int tile = nt * (BN / 16) + (wn * TN + j) * 2 + (c >> 4);
                    tile = tile < w_tiles ? tile : w_tiles - 1;
                    rows_of_w[j] = reinterpret_cast<const bf16x8 *>(wbase) + (size_t)tile * ksteps * 64 + h * 16 + (c & 15);
                }
                f32x16 whole[TN][TM];
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            whole[j][i][r] = 0.0f;
                for (int s = 0; s < 2 * ksteps; ++s) // sixteen columns
                {
                    f32x8 x[TM], v[TN];
#pragma unroll
                    for (int i = 0; i < TM; ++i)
                        x[i] = Operand<float>::load(rows_of_a[i] + s * 16);
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        v[j] = __builtin_convertvector(rows_of_w[j][(s >> 1) * 64 + (s & 1) * 32], f32x8);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
#pragma unroll
                        for (int j = 0; j < TN; ++j)
#pragma unroll
                            for (int i = 0; i < TM; ++i)
                                whole[j][i] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[j][e], x[i][e], whole[j][i], 0, 0, 0);
                }
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            acc[j][i][r] = pieces_fail(acc[j][i][r]) ? whole[j][i][r] : acc[j][i][r];
            }
        }

        // Results by way of LDS, where a wavefront lays 32 rows of its own columns and takes them up again by whole rows: straight
        // from the accumulators a store instruction of 64 lanes touches 32 rows, 8 or 16 bytes a lane, and loads of other workgroups
        // wait behind that (bf16, straight and by way of LDS: 2048 x 16384 x 2048 165 -> 112 us, 2048 x 16384 x 8192 503 -> 426).
        const size_t elem = p.out == LLAM_SEQ_OUT_F32 || p.out == LLAM_SEQ_OUT_ADD ? 4 : sizeof(T);
        char *y = static_cast<char *>(p.y) + (p.group_offset ? 0 : (size_t)z * p.y_stride * elem);
        if constexpr (KG == 1)
            arrive<0>(); // all wavefronts are done with the stages (of several groups, the place of the wavefront's own sums)
        char *own = smem + wave * (KG == 1 ? TN * OUT_BYTES : TN * TM * 4096);
        auto out = [&](auto gated, auto value) __attribute__((always_inline)) {
            typedef decltype(value) V;
            constexpr bool GATED = decltype(gated)::value;
            constexpr int COLS = GATED ? TN * 16 : TN * 32, PITCH = COLS * sizeof(V);
            constexpr int EACH = 16 / sizeof(V), PIECES = COLS / EACH; // values of a 16-byte piece, pieces of a row
            typedef V four_t __attribute__((ext_vector_type(4)));
            typedef V piece_t __attribute__((ext_vector_type(EACH)));
            // piece x of row r lies at x ^ spread(r)
            auto spread = [](int r) __attribute__((always_inline)) { return r / (PIECES < 8 ? 8 / PIECES : 1) & (PIECES - 1); };
            const int n0 = (nt * BN + wn * TN * 32) / (GATED ? 2 : 1), columns = GATED ? p.N / 2 : p.N;
            const bool whole = ((p.ldy | p.y_stride) & (EACH - 1)) == 0; // (rows of 16-bit values may start at 8 bytes)
#pragma unroll
            for (int i = 0; i < TM; ++i)
            {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int q = 0; q < (GATED ? 2 : 4); ++q)
                    {
                        auto four = [&](int q) __attribute__((always_inline)) {
                            return f32x4{acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
                        };
                        f32x4 v = four(q);
                        if constexpr (GATED) // rows 0 .. 15 of the product are gates, 16 .. 31 the same of up
                            v = gated4(p, v, four(q + 2));
                        else if (sizeof(V) == sizeof(T) && p.out == LLAM_SEQ_OUT_RELU2)
                            v = relu2(v);
                        const int col = j * (GATED ? 16 : 32) + 8 * q + 4 * h;
                        *reinterpret_cast<four_t *>(own + c * PITCH + (col / EACH ^ spread(c)) * 16 + col % EACH * sizeof(V)) = __builtin_convertvector(v, four_t);
                    }
                asm volatile("" ::: "memory"); // (a wavefront's LDS instructions run in order)
#pragma unroll
                for (int k = 0; k < PIECES / 2; ++k)
                {
                    const int r = (k * 64 + lane) / PIECES, x = (k * 64 + lane) % PIECES, col = n0 + x * EACH;
                    const int m = mt * BM + (wm * TM + i) * 32 + r;
                    piece_t v = *reinterpret_cast<const piece_t *>(own + r * PITCH + (x ^ spread(r)) * 16);
                    if (m < rows && col < columns)
                        store_piece(p, y, whole, row0 + m, col, v);
                }
                asm volatile("" ::: "memory");
            }
        };
        if (is_gated(p.out))
            out(std::true_type(), T());
        else if (elem == sizeof(T))
            out(std::false_type(), T());
        else
            out(std::false_type(), float());
    }

    namespace
    {
        template <typename T, int BM, int BN, int WM, int WN, int KG, int STAGES>
        bool wide_launch(const char *fn, const LinearArgs &a, int batch, hipStream_t st)
        {
            static LdsGrant grant;
            constexpr size_t stages = (size_t)STAGES * KG * (BM * sizeof(T) + BN * 2) * TILE_K, sums = (size_t)(KG - 1) * BM * BN * 4;
            static_assert(KG > 1 || stages >= (size_t)WM * BN * OUT_BYTES / 32, "the results' place");
            constexpr size_t lds = stages > sums ? stages : sums;
            static_assert(lds <= 160 * 1024, "stages must fit the LDS");
            const auto kernel = &linear_wide_kernel<T, BM, BN, WM, WN, KG, STAGES>;
            if (lds > 64 * 1024 && allow_lds(grant, reinterpret_cast<const void *>(kernel), lds) != hipSuccess)
                return fail(fn, "cannot reserve %zu bytes of LDS", lds);
            const int nt = ceil_div(a.N, BN);
            // groups: no more tiles than if every group had one that is not full
            const long mt = a.group_offset ? a.group_rows / BM + (batch < a.group_rows ? batch : a.group_rows) : ceil_div(a.M, BM);
            if (mt * nt > 0x7fffffff)
                return fail(fn, "M=%d rows of N=%d columns are too many", a.M, a.N);
            hipLaunchKernelGGL(kernel, dim3((unsigned)(mt * nt), a.group_offset ? 1 : batch), dim3(WM * WN * KG * 64), lds, st, a, (int)mt, nt);
            return launched(fn);
        }

        // A tile, and what a turn of it takes in microseconds where few compute units are busy and where all are (with
        // `resident` workgroups each), and a workgroup's start and end.
        struct Tile
        {
            int rows, columns, groups, resident;
            float alone, full, start;
            bool (*launch)(const char *, const LinearArgs &, int, hipStream_t);
        };
        // Measured as time over turns for widths of 2048 to 51200, 40 to 2048 rows and K of 2048 to 30720.  Large tiles
        // read the LDS least per product (256 x 256: 1130 TFLOP/s at 2048 x 51200 x 5120, 128 x 128: 1010), small ones
        // and groups of wavefronts that share K fill the chip where there are few tiles (522 x 2048 x 10240: 50 us with
        // 128 x 64 and two groups, 120 with 256 x 128).  The same figures hold for the rows of routed experts: over 7 models' experts
        // (8 to 256 of 64 to 1536, both ways) and 17 to 2000 rows, evenly chosen and not, the tile chosen is 0.9 % slower than
        // the best in the mean, 15 % at most (1000 rows, 2 of 16 experts of 1536 x 5120, up: 210 and 182 us); fp32 0.6 %, 15 %.
        // 187 rows, 6 of 64 experts of 1408 x 2048 and a shared one: bf16 209 -> 190 us against two tiles by the mean
        // rows of a group, fp32 369 -> 267 against tiles as if every group had all rows.
        const Tile TILES_BF16[] = {
            {256, 256, 1, 1, 1.30f, 1.70f, 4.0f, wide_launch<bf16, 256, 256, 2, 4, 1, 2>},
            {256, 128, 1, 1, 0.75f, 1.00f, 4.0f, wide_launch<bf16, 256, 128, 4, 2, 1, 3>},
            {128, 128, 1, 2, 0.65f, 1.05f, 4.0f, wide_launch<bf16, 128, 128, 2, 2, 1, 2>},
            {128, 128, 1, 1, 0.57f, 0.60f, 3.0f, wide_launch<bf16, 128, 128, 4, 2, 1, 3>},
            {128, 64, 2, 1, 0.60f, 0.70f, 3.0f, wide_launch<bf16, 128, 64, 2, 2, 2, 3>},
            {64, 64, 2, 1, 0.40f, 0.50f, 3.0f, wide_launch<bf16, 64, 64, 2, 2, 2, 4>},
            {64, 64, 1, 2, 0.26f, 0.43f, 3.0f, wide_launch<bf16, 64, 64, 2, 2, 1, 4>},
        };
        // (in three pieces: the cutting up of A costs as much as the products where a wavefront has few columns)
        const Tile TILES_F32[] = {
            {128, 256, 1, 1, 2.00f, 2.60f, 4.0f, wide_launch<float, 128, 256, 4, 2, 1, 2>},
            {128, 128, 1, 1, 1.34f, 1.65f, 3.0f, wide_launch<float, 128, 128, 4, 2, 1, 3>},
            {64, 128, 2, 1, 1.45f, 1.75f, 3.0f, wide_launch<float, 64, 128, 2, 2, 2, 2>},
            {64, 64, 2, 1, 1.15f, 1.30f, 3.0f, wide_launch<float, 64, 64, 2, 2, 2, 3>},
        };

        float expected(const Tile &t, const LinearArgs &a, int batch, int cus)
        {
            float rows = (float)ceil_div(a.M, t.rows) * batch;
            if (a.group_offset)
            {
                // rows in groups: a tile of every group at least, else half a tile a group more than full ones
                const float groups = (float)(batch < a.group_rows ? batch : a.group_rows);
                rows = fmaxf(groups, (float)a.group_rows / t.rows + 0.5f * groups);
            }
            const float tiles = rows * ceil_div(a.N, t.columns), slots = (float)cus * t.resident;
            const float fill = tiles < slots ? tiles / slots : 1.0f;
            const float turn = t.alone + (t.full - t.alone) * fill;
            return ceilf(tiles / slots) * (ceil_div(a.K / TILE_K, t.groups) * turn + t.start);
        }
    } // namespace

    bool linear_tiled(const char *fn, const LinearArgs &a, int batch, int dtype, int device_id, hipStream_t st)
    {
        const int cus = cu_count(device_id);
        const Tile *tiles = dtype == LLAM_SEQ_F32 ? TILES_F32 : TILES_BF16, *best = tiles;
        const size_t n = dtype == LLAM_SEQ_F32 ? sizeof TILES_F32 / sizeof(Tile) : sizeof TILES_BF16 / sizeof(Tile);
        for (size_t i = 1; i < n; ++i)
            if (expected(tiles[i], a, batch, cus) < expected(*best, a, batch, cus))
                best = &tiles[i];
        return best->launch(fn, a, batch, st);
    }
} // namespace llamql
