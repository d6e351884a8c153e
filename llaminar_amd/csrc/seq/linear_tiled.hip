// Linear layers of many rows (prompts) for gfx950: y = A W^T, W in matrix-unit tiles.
//
// Both operands go from global memory straight into LDS, some turns of 64 columns ahead, and from there into registers
// one sixteen-column step ahead of the products, across the one barrier of a turn.  W is the first operand, so a lane
// ends with four neighbouring output columns of one row; results go through LDS so that they leave by whole lines.  32-bit rows are multiplied in three bf16 pieces that add up to
// them (weights are bf16 anyway): the products stay exact, the sums 32-bit, on a unit that is 16 times as fast.
//
// What bounds it, 2048 x 15440 x 5120 in bf16: the matrix unit is busy in 63 % of the cycles (2048 x 51200 x 5120 68 %, 32-bit rows, 522 x 51200 x
// 5120, 65 %), the LDS with reads in 25 %, and the two wavefronts of a SIMD unit meet at the barrier of every turn; where such products
// follow each other the clock falls, from 1.85 to 1.3 GHz (266 to 380 us).
// Time before (128 x 128 tiles staged through registers) and now, with the clock up: 390 -> 266 us (830 -> 1220 TFLOP/s), 2048 x 51200 x
// 5120 1200 -> 875 us, 333 x 2048 x 8192 63 -> 28 us; 32-bit rows (v_mfma_f32_16x16x4 before) 522 x 2048 x 10240 380 -> 82 us (in slices).
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

    // 32 rows from m0 on of TN x 32 products, a lane's as the matrix unit leaves them, to rows row0 + m of y.  By way of LDS, where the
    // wavefront lays them (own) and takes them up again by whole rows: straight from the accumulators a store instruction of 64 lanes
    // touches 32 rows, 8 or 16 bytes a lane, and loads of other workgroups wait behind that (bf16, straight and by way of LDS:
    // 2048 x 16384 x 2048 165 -> 112 us, 2048 x 16384 x 8192 503 -> 426).
    template <typename T, int TN>
    __device__ __forceinline__ void results(const LinearArgs &p, int z, const f32x16 (&strip)[TN], char *own, int lane, int m0, int rows, int row0, int n0)
    {
        const int c = lane & 31, h = lane >> 5;
        const size_t elem = p.out == LLAM_SEQ_OUT_F32 || p.out == LLAM_SEQ_OUT_ADD ? 4 : sizeof(T);
        char *y = static_cast<char *>(p.y) + (size_t)z * p.y_stride * elem;
        auto out = [&](auto gated, auto value) __attribute__((always_inline)) {
            typedef decltype(value) V;
            constexpr bool GATED = decltype(gated)::value;
            constexpr int COLS = GATED ? TN * 16 : TN * 32, PITCH = COLS * sizeof(V);
            constexpr int EACH = 16 / sizeof(V), PIECES = COLS / EACH; // values of a 16-byte piece, pieces of a row
            typedef V four_t __attribute__((ext_vector_type(4)));
            typedef V piece_t __attribute__((ext_vector_type(EACH)));
            // piece x of row r lies at x ^ spread(r)
            auto spread = [](int r) __attribute__((always_inline)) { return r / (PIECES < 8 ? 8 / PIECES : 1) & (PIECES - 1); };
            const int first = GATED ? n0 / 2 : n0, columns = GATED ? p.N / 2 : p.N;
            const bool whole = ((p.ldy | p.y_stride) & (EACH - 1)) == 0; // (rows of 16-bit values may start at 8 bytes)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int q = 0; q < (GATED ? 2 : 4); ++q)
                {
                    auto four = [&](int q) __attribute__((always_inline)) {
                        return f32x4{strip[j][4 * q], strip[j][4 * q + 1], strip[j][4 * q + 2], strip[j][4 * q + 3]};
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
                const int r = (k * 64 + lane) / PIECES, x = (k * 64 + lane) % PIECES, col = first + x * EACH;
                const piece_t v = *reinterpret_cast<const piece_t *>(own + r * PITCH + (x ^ spread(r)) * 16);
                if (m0 + r < rows && col < columns)
                    store_piece(p, y, whole, row0 + m0 + r, col, v);
            }
            asm volatile("" ::: "memory");
        };
        if (is_gated(p.out))
            out(std::true_type(), T());
        else if (elem == sizeof(T))
            out(std::false_type(), T());
        else
            out(std::false_type(), float());
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

    // Neighbouring tiles go to one die (blocks are dealt round robin over the eight dies), eight tiles of rows side
    // by side, then the next tile of W: what a die works on at a time is about square.
    __device__ __forceinline__ int die_order(int id, int count)
    {
        const int per = count / 8;
        return id < per * 8 ? (id & 7) * per + (id >> 3) : id;
    }
    __device__ __forceinline__ void tile_place(int id, int m_tiles, int n_tiles, int &mt, int &nt)
    {
        const int band = id / (8 * n_tiles), in = id - band * 8 * n_tiles;
        const int high = m_tiles - band * 8 < 8 ? m_tiles - band * 8 : 8;
        nt = in / high;
        mt = band * 8 + in - nt * high;
    }

    // Workgroup tile BM rows of A x BN rows of W; KG groups of WM x WN wavefronts, each with every KG-th turn of 64
    // columns, STAGES turns of A in LDS and WSTAGES of W.  SPLIT: the tiles from p.full on have p.slices workgroups each, every one with a slice of K,
    // which leave their accumulators in p.parts for linear_join_kernel.  Args: LinearSomeArgs for some of the rows alone.
    template <typename T, int BM, int BN, int WM, int WN, int KG, int STAGES, int WSTAGES, bool SPLIT, typename Args = LinearArgs>
    __global__ void __launch_bounds__(WM *WN *KG * 64)
        linear_wide_kernel(Args p, int m_tiles, int n_tiles)
    {
        using O = TiledOperand<T>;
        constexpr int NW = WM * WN;                         // wavefronts of a group
        constexpr int TM = BM / WM / 32, TN = BN / WN / 32; // 32x32 products of a wavefront
        constexpr int AROW = TILE_K * sizeof(T), AROWS = 1024 / AROW, APIECES = AROW / 16; // bytes; rows of a load; 16-byte pieces
        constexpr int ALOADS = BM / AROWS / NW, WLOADS = BN / 8 / NW, LOADS = ALOADS + WLOADS; // of a turn, per wavefront
        constexpr int ABYTES = BM * AROW, WBYTES = BN * TILE_K * 2, WBASE = STAGES * KG * ABYTES; // a turn's, where W's turns begin
        static_assert(BM % (AROWS * NW) == 0 && BN % (8 * NW) == 0 && TM >= 1 && TN >= 1, "whole loads and products");
        static_assert(STAGES >= 2 && (WSTAGES == STAGES || WSTAGES == STAGES + 1) && (WSTAGES - 1) * LOADS < 64, "counted by six bits");
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
        int row0 = 0, rows = p.M;
        if constexpr (std::is_same_v<Args, LinearSomeArgs>)
        {
            row0 = p.first[blockIdx.z], rows = p.rows[blockIdx.z];
            m_tiles = (rows + BM - 1) / BM;
        }
        const int total = m_tiles * n_tiles;
        if ((int)blockIdx.x >= (SPLIT ? p.full + (total - p.full) * p.slices : total))
            return;
        // (split: behind the whole tiles the first slices of the others, then their second ones, ..: what is at work at a time
        // reads the same columns)
        const bool whole = !SPLIT || (int)blockIdx.x < p.full;
        const int slice = whole ? 0 : ((int)blockIdx.x - p.full) / (total - p.full);
        const int part = whole ? blockIdx.x : blockIdx.x - p.full - slice * (total - p.full); // of the whole tiles or of the others
        int mt, nt;
        tile_place(whole ? die_order(part, SPLIT ? p.full : total) : p.full + die_order(part, total - p.full), m_tiles, n_tiles, mt, nt);
        int z = blockIdx.y;
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
        const int turn0 = whole ? 0 : slice * turns / p.slices, count = (whole ? turns : (slice + 1) * turns / p.slices) - turn0; // of K
        const int rounds = (count + KG - 1) / KG; // the group's turn k is columns 64 (turn0 + k KG + kg) .. of K
        const int first = turn0 + (kg < count ? kg : count - 1);

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
            load_to_lds(src[i], lds0 + wave * 1024 + (i < ALOADS ? (buf * KG + kg) * ABYTES + i * NW * 1024 : WBASE + (buf * KG + kg) * WBYTES + (i - ALOADS) * NW * 1024));
            if (KG == 1 || (t + 1) * KG + kg < count)
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
        for (int t = 0; t < WSTAGES; ++t)
            if (t < rounds)
            {
#pragma unroll
                for (int i = t < STAGES ? 0 : ALOADS; i < LOADS; ++i)
                    issue(i, t, t);
            }
        const int arow = (wm * 32 + c) * AROW, wrow = WBASE + (wn * TN * 2 + (c >> 4)) * 2048 + (h * 16 + (c & 15)) * 16;
        typename O::Raw a[2][TM];
        bf16x8 w[2][TN];
        // operand n of the 16 columns s of a stage (k-step s / 2 of W, its pieces 2 (s & 1) + h): A's first, W's, A's others
        auto read = [&](int buf, int wbuf, int s, int b, int n) __attribute__((always_inline)) {
            if (n >= 1 && n <= TN)
                w[b][n - 1] = *reinterpret_cast<const bf16x8 *>(smem + (wbuf * KG + kg) * WBYTES + wrow + (n - 1) * 4096 + (s >> 1) * 1024 + (s & 1) * 512);
            else
            {
                const int i = n == 0 ? 0 : n - TN;
                const char *row = smem + (buf * KG + kg) * ABYTES + arow + i * WM * 32 * AROW;
                if constexpr (sizeof(T) == 2)
                    a[b][i] = *reinterpret_cast<const bf16x8 *>(row + ((2 * s + h) ^ swizzle(c)) * 16);
                else
                    a[b][i] = __builtin_shufflevector(*reinterpret_cast<const f32x4 *>(row + ((4 * s + 2 * h) ^ swizzle(c)) * 16),
                                                      *reinterpret_cast<const f32x4 *>(row + ((4 * s + 2 * h + 1) ^ swizzle(c)) * 16), 0, 1, 2, 3, 4, 5, 6, 7);
            }
        };
        // all turns, with the first `strips` of the wavefront's TM strips of 32 rows
        auto walk = [&](auto strips) __attribute__((always_inline)) {
            constexpr int L = decltype(strips)::value;
            // the products of the operands b, in this order, with what `between` asks for after each: left to itself the
            // compiler asks for operands just before it needs them
            auto multiply = [&](int b, auto between) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < L; ++i)
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
                const int each = (count + TN * L - 1) / (TN * L);
#pragma unroll
                for (int k = 0; k < 16; ++k)
                    if (k < each && n * each + k < count)
                        f(n * each + k);
            };
            if (rounds >= WSTAGES)
                arrive<(STAGES - 1) * LOADS + (WSTAGES - STAGES) * WLOADS>();
            else
                arrive<0>();
#pragma unroll
            for (int n = 0; n < L + TN; ++n)
                read(0, 0, 0, 0, n);
            int buf = 0, wbuf = 0;
            for (int t = 0; t < rounds - 1; ++t)
            {
                const int next = buf + 1 < STAGES ? buf + 1 : 0, wnext = wbuf + 1 < WSTAGES ? wbuf + 1 : 0;
#pragma unroll
                for (int s = 0; s < 3; ++s)
                    multiply(s & 1, [&](int n) { deal(n, [&](int k) { read(buf, wbuf, s + 1, (s + 1) & 1, k); }, L + TN); });
                // this stage is in registers; the next one has arrived, later ones may be on their way
                constexpr int LATER = (STAGES - 2) * LOADS + (WSTAGES - STAGES) * WLOADS;
                // (with none later, no branch: the cutting up of A and the first products go before the wait, fp32, 251 x 5120 x 25600
                // 287 and 268 us)
                if (LATER > 0 && t + WSTAGES <= rounds)
                    arrive<LATER>();
                else
                    arrive<0>();
                const bool more = t + STAGES < rounds, wmore = t + WSTAGES < rounds;
                multiply(1, [&](int n) {
                    deal(n, [&](int k) { read(next, wnext, 0, 0, k); }, L + TN);
                    deal(n, [&](int k) {
                        if (k < ALOADS ? more : wmore)
                            issue(k, k < ALOADS ? buf : wbuf, t + (k < ALOADS ? STAGES : WSTAGES));
                    }, LOADS);
                });
                buf = next, wbuf = wnext;
            }
            if (KG == 1 || (rounds - 1) * KG + kg < count)
            {
#pragma unroll
                for (int s = 0; s < 3; ++s)
                    multiply(s & 1, [&](int n) { deal(n, [&](int k) { read(buf, wbuf, s + 1, (s + 1) & 1, k); }, L + TN); });
                multiply(1, [](int) {});
            }
        };
        // strips past the last row are left out: a wavefront's strips lie WM apart, so all wavefronts have about as many.  (64 experts
        // of 52 to 87 rows, tiles of 256 x 128: 1408 x 2048 103 -> 83 us; the matrix unit is also what the clock goes down for.)
        const int strips = __builtin_amdgcn_readfirstlane((rows - mt * BM + (WM - 1 - wm) * 32 + 31) / (WM * 32));
        if (TM > 3 && strips == 3)
            walk(std::integral_constant<int, (TM > 3 ? 3 : TM)>());
        else if (TM > 2 && strips == 2)
            walk(std::integral_constant<int, (TM > 2 ? 2 : TM)>());
        else if (TM > 1 && strips < 2)
            walk(std::integral_constant<int, 1>());
        else
            walk(std::integral_constant<int, TM>());

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
                    int m = mt * BM + (wm + i * WM) * 32 + c;
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
                for (int s = 4 * turn0; s < 4 * (turn0 + count); ++s) // sixteen columns
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

        if constexpr (SPLIT)
        {
            if (!whole)
            {
                // as the lanes hold them
                f32x4 *part_sums = p.parts + ((size_t)slice * (total - p.full) + die_order(part, total - p.full)) * (BM * BN / 4) +
                                   wave * (TN * TM * 256) + lane;
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            part_sums[((i * TN + j) * 4 + q) * 64] =
                                f32x4{acc[j][i][4 * q], acc[j][i][4 * q + 1], acc[j][i][4 * q + 2], acc[j][i][4 * q + 3]};
                return;
            }
        }
        if constexpr (KG == 1)
            arrive<0>(); // all wavefronts are done with the stages (of several groups, the place of the wavefront's own sums)
        char *own = smem + wave * (KG == 1 ? TN * OUT_BYTES : TN * TM * OUT_BYTES);
#pragma unroll
        for (int i = 0; i < TM; ++i)
        {
            f32x16 strip[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j)
                strip[j] = acc[j][i];
            results<T>(p, p.group_offset ? 0 : z, strip, own, lane, mt * BM + (wm + i * WM) * 32, rows, row0, nt * BN + wn * TN * 32);
        }
    }

    // A wavefront joins the slices of 32 rows of what a wavefront of linear_wide_kernel had, in the order of K.
    template <typename T, int BM, int BN, int WM, int WN>
    __global__ void __launch_bounds__(256)
        linear_join_kernel(LinearArgs p, int m_tiles, int n_tiles)
    {
        constexpr int NW = WM * WN, TM = BM / WM / 32, TN = BN / WN / 32;
        __shared__ __attribute__((aligned(16))) char smem[4 * TN * OUT_BYTES];
        const int lane = threadIdx.x & 63, here = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int unit = blockIdx.x * 4 + here, split = m_tiles * n_tiles - p.full;
        static_assert(NW * TM % 4 == 0, "whole workgroups");
        const int id = unit / (NW * TM), wave = unit / TM % NW, i = unit % TM;
        int mt, nt;
        tile_place(p.full + id, m_tiles, n_tiles, mt, nt);
        const f32x4 *from = p.parts + (size_t)id * (BM * BN / 4) + (wave * TM + i) * (TN * 256) + lane;
        f32x16 strip[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                strip[j][r] = 0.0f;
        // `count` slices from k on, asked for together
        auto add = [&](auto count, int k) __attribute__((always_inline)) {
            f32x4 v[count.value][TN * 4];
#pragma unroll
            for (int u = 0; u < count.value; ++u)
#pragma unroll
                for (int x = 0; x < TN * 4; ++x)
                    v[u][x] = from[(size_t)(k + u) * split * (BM * BN / 4) + x * 64];
#pragma unroll
            for (int u = 0; u < count.value; ++u)
#pragma unroll
                for (int x = 0; x < TN * 4; ++x)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        strip[x / 4][x % 4 * 4 + r] += v[u][x][r];
        };
        constexpr int GROUP = TN > 2 ? 2 : 4;
        int k = 0;
        for (; k + GROUP <= p.slices; k += GROUP)
            add(std::integral_constant<int, GROUP>(), k);
        if (GROUP == 4 && k + 2 <= p.slices)
            add(std::integral_constant<int, 2>(), k), k += 2;
        if (k < p.slices)
            add(std::integral_constant<int, 1>(), k);
        results<T>(p, 0, strip, smem + here * (TN * OUT_BYTES), lane, mt * BM + (wave % WM + i * WM) * 32, p.M, 0, nt * BN + wave / WM * TN * 32);
    }

    namespace
    {
        template <typename T, int BM, int BN, int WM, int WN, int KG, int STAGES, int WSTAGES = STAGES>
        bool wide_launch(const char *fn, const LinearArgs &a, int batch, hipStream_t st, const LinearSomeArgs *some)
        {
            static LdsGrant grant, grant_some;
            constexpr size_t stages = (size_t)KG * (STAGES * BM * sizeof(T) + WSTAGES * BN * 2) * TILE_K, sums = (size_t)(KG - 1) * BM * BN * 4;
            static_assert(KG > 1 || stages >= (size_t)WM * BN * OUT_BYTES / 32, "the results' place");
            constexpr size_t lds = stages > sums ? stages : sums;
            static_assert(lds <= 160 * 1024, "stages must fit the LDS");
            const auto kernel = &linear_wide_kernel<T, BM, BN, WM, WN, KG, STAGES, WSTAGES, false>;
            if (lds > 64 * 1024 && allow_lds(grant, reinterpret_cast<const void *>(kernel), lds) != hipSuccess)
                return fail(fn, "cannot reserve %zu bytes of LDS", lds);
            const int nt = ceil_div(a.N, BN);
            // groups: no more tiles than if every group had one that is not full
            const long mt = a.group_offset ? a.group_rows / BM + (batch < a.group_rows ? batch : a.group_rows) : ceil_div(a.M, BM);
            if (mt * nt > 0x7fffffff)
                return fail(fn, "M=%d rows of N=%d columns are too many", a.M, a.N);
            if (some)
            {
                const auto rows = &linear_wide_kernel<T, BM, BN, WM, WN, KG, STAGES, WSTAGES, false, LinearSomeArgs>;
                if (lds > 64 * 1024 && allow_lds(grant_some, reinterpret_cast<const void *>(rows), lds) != hipSuccess)
                    return fail(fn, "cannot reserve %zu bytes of LDS", lds);
                hipLaunchKernelGGL(rows, dim3((unsigned)(mt * nt), batch, some->stretches), dim3(WM * WN * KG * 64), lds, st, *some, 0, nt);
                return launched(fn);
            }
            hipLaunchKernelGGL(kernel, dim3((unsigned)(mt * nt), a.group_offset ? 1 : batch), dim3(WM * WN * KG * 64), lds, st, a, (int)mt, nt);
            return launched(fn);
        }

        // The same with the tiles from a.full on in a.slices slices of K each, which a second launch joins.
        template <typename T, int BM, int BN, int WM, int WN, int KG, int STAGES, int WSTAGES = STAGES>
        bool split_launch(const char *fn, const LinearArgs &a, hipStream_t st)
        {
            static LdsGrant grant;
            constexpr size_t stages = (size_t)KG * (STAGES * BM * sizeof(T) + WSTAGES * BN * 2) * TILE_K, sums = (size_t)(KG - 1) * BM * BN * 4;
            constexpr size_t lds = stages > sums ? stages : sums;
            const auto kernel = &linear_wide_kernel<T, BM, BN, WM, WN, KG, STAGES, WSTAGES, true>;
            if (lds > 64 * 1024 && allow_lds(grant, reinterpret_cast<const void *>(kernel), lds) != hipSuccess)
                return fail(fn, "cannot reserve %zu bytes of LDS", lds);
            const int nt = ceil_div(a.N, BN), mt = ceil_div(a.M, BM), split = mt * nt - a.full;
            hipLaunchKernelGGL(kernel, dim3((unsigned)(a.full + split * a.slices)), dim3(WM * WN * KG * 64), lds, st, a, mt, nt);
            if (!launched(fn))
                return false;
            hipLaunchKernelGGL((linear_join_kernel<T, BM, BN, WM, WN>), dim3((unsigned)(split * (BM / 32) * WN / 4)), dim3(256), 0, st, a, mt, nt);
            return launched(fn);
        }

        // A tile, and what a turn of it takes in microseconds where few compute units are busy and where all are (with
        // `resident` workgroups each), and a workgroup's start and end.
        struct Tile
        {
            int rows, columns, groups, resident;
            float alone, full, start;
            bool (*launch)(const char *, const LinearArgs &, int, hipStream_t, const LinearSomeArgs *);
            bool (*split)(const char *, const LinearArgs &, hipStream_t); // (none where two workgroups share a compute unit)
        };
        // Measured as time over turns for widths of 2048 to 51200, 40 to 2048 rows and K of 2048 to 30720.  Large tiles
        // read the LDS least per product (256 x 256: 1220 TFLOP/s at 2048 x 51200 x 5120, 128 x 128: 1010), small ones
        // and groups of wavefronts that share K fill the chip where there are few tiles (522 x 2048 x 10240: 50 us with
        // 128 x 64 and two groups, 120 with 256 x 128).  Over 16 layers of 1280 to 51200 x 1024 to 30720 with 12 numbers of rows in bf16 the tile
        // chosen is 1.1 % above the best in the mean, 27 % at most (1000 rows of 5120 columns, 256 x 128 would be better: x 25600 399 and 315 us); of
        // 10 with 8 in fp32 it is the best.  The same figures hold for the rows of routed experts: over 7 models' experts
        // (8 to 256 of 512 to 4096, both ways) and 17 to 2000 rows, evenly chosen and not, a layer is 4.5 % above that of the best two tiles,
        // 26 % at most (512 rows, 4 of 32 experts of 1024 x 2048, unevenly: 102 and 81 us); fp32 3.1 %, 30 %.
        // 187 rows, 6 of 64 experts of 1408 x 2048 and a shared one: bf16 209 -> 190 us against two tiles by the mean
        // rows of a group, fp32 369 -> 267 against tiles as if every group had all rows.
        // 256 x 256 has a third turn of W in its LDS, for that is what comes from memory, where A mostly comes from the cache: 64 experts of 155 to
        // 217 rows, 2048 x 1408 108 -> 105 us, 1536 x 5120 287 -> 263, 2048 x 5120 x 30720 662 -> 645; the tile that such experts had, 128 x 128
        // by four wavefronts, takes 129 and 297.  (A third turn of W for the others, of 256 x 128 a fourth: no faster.)
        const Tile TILES_BF16[] = {
            {256, 256, 1, 1, 1.15f, 1.45f, 4.0f, wide_launch<bf16, 256, 256, 2, 4, 1, 2, 3>, split_launch<bf16, 256, 256, 2, 4, 1, 2, 3>},
            {256, 128, 1, 1, 0.75f, 1.00f, 4.0f, wide_launch<bf16, 256, 128, 4, 2, 1, 3>, split_launch<bf16, 256, 128, 4, 2, 1, 3>},
            {128, 128, 1, 2, 0.65f, 1.05f, 4.0f, wide_launch<bf16, 128, 128, 2, 2, 1, 2>, nullptr},
            {128, 128, 1, 1, 0.57f, 0.60f, 3.0f, wide_launch<bf16, 128, 128, 4, 2, 1, 3>, split_launch<bf16, 128, 128, 4, 2, 1, 3>},
            {128, 64, 2, 1, 0.60f, 0.70f, 3.0f, wide_launch<bf16, 128, 64, 2, 2, 2, 3>, split_launch<bf16, 128, 64, 2, 2, 2, 3>},
            {64, 64, 2, 1, 0.40f, 0.50f, 3.0f, wide_launch<bf16, 64, 64, 2, 2, 2, 4>, split_launch<bf16, 64, 64, 2, 2, 2, 4>},
            {64, 64, 1, 2, 0.26f, 0.43f, 3.0f, wide_launch<bf16, 64, 64, 2, 2, 1, 4>, nullptr},
        };
        // (in three pieces: the cutting up of A costs as much as the products where a wavefront has few columns)
        const Tile TILES_F32[] = {
            {128, 256, 1, 1, 2.00f, 2.60f, 4.0f, wide_launch<float, 128, 256, 4, 2, 1, 2>, split_launch<float, 128, 256, 4, 2, 1, 2>},
            {128, 128, 1, 1, 1.34f, 1.65f, 3.0f, wide_launch<float, 128, 128, 4, 2, 1, 3>, split_launch<float, 128, 128, 4, 2, 1, 3>},
            {64, 128, 2, 1, 1.45f, 1.75f, 3.0f, wide_launch<float, 64, 128, 2, 2, 2, 2>, split_launch<float, 64, 128, 2, 2, 2, 2>},
            {64, 64, 2, 1, 1.15f, 1.30f, 3.0f, wide_launch<float, 64, 64, 2, 2, 2, 3>, split_launch<float, 64, 64, 2, 2, 2, 3>},
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

    namespace
    {
        // Tiles that fill no round of workgroups by themselves, cut into slices of K that do: in the time of a slice instead of that of a
        // tile, for the sums that leave and come back and a launch that joins them.  (us, whole and in slices: bf16, 2048 x 5120 x 30720 637 -> 558,
        // 512 x 5120 x 30720 251 -> 158, 64 x 2048 x 10240 32 -> 17, 1000 x 51200 x 5120 487 -> 449; fp32, 522 x 2048 x 10240 106 -> 80,
        // 64 x 2048 x 16384 130 -> 30.)  Over 16 layers of 1280 to 51200 x 1024 to 30720 with 12 numbers of rows in bf16, 10 with 8 in fp32, 71 of 192
        // and 57 of 80 are cut, to 0.76 and 0.69 times their time in the mean; none is slower by more than 3 % (0.3 us); the choice is 1.9 and 1.6 % above
        // the best of all, 25 and 30 % at most (187 x 5120 x 10240 48 and 38 us; 20 x 2816 x 2048 16.7 and 12.9).
        constexpr int SLICES = 8;                        // at most
        constexpr size_t SPLIT_BYTES = (size_t)192 << 20; // sums of a launch, at most
        constexpr float JOIN_START = 4.0f, JOIN_BYTE = 0.45e-6f; // microseconds: a launch; a byte there and back

        struct Split
        {
            float us; // expected
            int full, slices;
            size_t bytes;
        };
        Split best_split(const Tile &t, const LinearArgs &a, size_t bytes, int cus)
        {
            Split best = {1e30f, 0, 0, 0};
            const long tiles = (long)ceil_div(a.M, t.rows) * ceil_div(a.N, t.columns), full = tiles / cus * cus, rest = tiles - full;
            const int turns = a.K / TILE_K;
            if (!t.split || rest == 0 || full + rest * SLICES > 0x7fffffff)
                return best;
            for (int slices = 2; slices <= SLICES && slices * 2 * t.groups <= turns; ++slices)
            {
                const long pieces = rest * slices, rounds = (pieces + cus - 1) / cus;
                const size_t need = (size_t)pieces * t.rows * t.columns * 4;
                if (need > bytes)
                    break;
                const float turn = t.alone + (t.full - t.alone) * (pieces < cus ? (float)pieces / cus : 1.0f);
                const float us = (float)(full / cus) * (ceil_div(turns, t.groups) * t.full + t.start) +
                                 rounds * (ceil_div(ceil_div(turns, slices), t.groups) * turn + t.start) + JOIN_START + JOIN_BYTE * need;
                if (us < best.us)
                    best = {us, (int)full, slices, need};
            }
            return best;
        }

        struct Plan
        {
            const Tile *tile;
            Split split; // slices = 0: every tile whole
        };
        struct Tiles
        {
            const Tile *tiles;
            size_t n;
        };
        Tiles tiles_of(int dtype)
        {
            return dtype == LLAM_SEQ_F32 ? Tiles{TILES_F32, sizeof TILES_F32 / sizeof(Tile)} : Tiles{TILES_BF16, sizeof TILES_BF16 / sizeof(Tile)};
        }
        Plan linear_plan(const LinearArgs &a, int batch, int dtype, size_t bytes, int cus)
        {
            const auto [tiles, n] = tiles_of(dtype);
            Plan plan = {tiles, {expected(*tiles, a, batch, cus), 0, 0, 0}};
            for (size_t i = 1; i < n; ++i)
                if (const float us = expected(tiles[i], a, batch, cus); us < plan.split.us)
                    plan = {&tiles[i], {us, 0, 0, 0}};
            if (batch == 1 && !a.group_offset && bytes)
                for (size_t i = 0; i < n; ++i)
                    if (const Split s = best_split(tiles[i], a, bytes < SPLIT_BYTES ? bytes : SPLIT_BYTES, cus); s.us < plan.split.us)
                        plan = {&tiles[i], s};
            return plan;
        }
    } // namespace

    size_t linear_split_bytes(int max_rows, int N, int K, int dtype, int device_id)
    {
        const int cus = cu_count(device_id);
        size_t most = 0;
        LinearArgs a{};
        a.N = N, a.K = K;
        for (int rows = 64; rows - 64 < max_rows; rows += 64) // (a plan depends on the tiles of rows alone)
        {
            a.M = rows < max_rows ? rows : max_rows;
            const size_t need = a.M > SMALL_M ? linear_plan(a, 1, dtype, SPLIT_BYTES, cus).split.bytes : 0;
            most = need > most ? need : most;
        }
        return most;
    }

    // A sum is of the turns of its group of wavefronts, one after the other, so tiles of as many groups have the same bits
    // (all with one are rows of 32x32 products of 16 columns each).  Among these, the best for the rows that there are.
    bool linear_tiled_rows(const char *fn, const LinearSomeArgs &a, int batch, int dtype, int device_id, hipStream_t st)
    {
        const int cus = cu_count(device_id);
        const Tile *all = linear_plan(a, batch, dtype, 0, cus).tile, *tile = all;
        LinearSomeArgs some = a;
        some.M = 0;
        for (int k = 0; k < a.stretches; ++k)
            some.M = some.M > a.rows[k] ? some.M : a.rows[k]; // (the grid is of the longest)
        const auto [tiles, n] = tiles_of(dtype);
        for (size_t i = 0; i < n; ++i)
            if (tiles[i].groups == all->groups && expected(tiles[i], some, batch * a.stretches, cus) < expected(*tile, some, batch * a.stretches, cus))
                tile = &tiles[i];
        return tile->launch(fn, some, batch, st, &some);
    }

    bool linear_tiled(const char *fn, const LinearArgs &a, int batch, int dtype, int device_id, hipStream_t st, void *scratch, size_t bytes)
    {
        const Plan plan = linear_plan(a, batch, dtype, scratch ? bytes : 0, cu_count(device_id));
        if (plan.split.slices == 0)
            return plan.tile->launch(fn, a, batch, st, nullptr);
        LinearArgs cut = a;
        cut.parts = static_cast<f32x4 *>(scratch), cut.full = plan.split.full, cut.slices = plan.split.slices;
        return plan.tile->split(fn, cut, st);
    }
} // namespace llamql
