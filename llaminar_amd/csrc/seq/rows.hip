// Row operators of sequence models: token embedding, RMS norm, and the routed expert
// feed-forward (choice of experts, grouping of tokens by expert, weighted sum).
#include "linear.h"
#include <algorithm>
#include <climits>
#include <type_traits>

namespace llamql
{
    constexpr int ROW_THREADS = 256;

    constexpr int EMBED_WIDE_ROWS = 256; // rows from which a workgroup takes a whole row
    __global__ void __launch_bounds__(ROW_THREADS)
        seq_embed_kernel(llam_seq_embed_args p, const int32_t *__restrict__ ids, float *__restrict__ x, int ldx)
    {
        const int m = blockIdx.y, id = ids[m], last = m > 0 ? ids[m - 1] : 0;
        const bool ok = id >= 0 && id < p.vocab;
        const bf16 *table = static_cast<const bf16 *>(p.d_table), *pairs = static_cast<const bf16 *>(p.d_pairs);
        long pair = -1;
        if (pairs)
        {
            const int slot = p.d_row_slot[m], pos = p.d_row_pos[m];
            int32_t *history = p.d_history + (size_t)slot * p.cap;
            if (pos == 0)
                pair = p.buckets;
            else if (pos > 0 && pos < p.cap)
            {
                const int before = m > 0 && p.d_row_slot[m - 1] == slot ? last : history[pos - 1];
                const long sum = (long)before * p.mul_prev + (long)id * p.mul_cur;
                pair = (sum >> 32) == 0 ? (long)((uint32_t)sum % (uint32_t)p.buckets) : sum % p.buckets;
            }
            if (blockIdx.x == 0 && threadIdx.x == 0 && pos >= 0 && pos < p.cap)
                history[pos] = id;
        }
        if ((p.width & 3) == 0 && (ldx & 3) == 0)
        {
            // four columns at a time
#pragma unroll 2
            for (int c = (blockIdx.x * ROW_THREADS + threadIdx.x) * 4; c < ldx; c += gridDim.x * ROW_THREADS * 4)
            {
                f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                if (ok && c < p.width)
                {
                    v = __builtin_convertvector(*reinterpret_cast<const bf16x4 *>(table + (size_t)id * p.width + c), f32x4) * p.scale;
                    if (pair >= 0)
                        v = v + __builtin_convertvector(*reinterpret_cast<const bf16x4 *>(pairs + (size_t)pair * p.width + c), f32x4);
                }
                *reinterpret_cast<f32x4 *>(x + (size_t)m * ldx + c) = v;
            }
            return;
        }
        for (int c = blockIdx.x * ROW_THREADS + threadIdx.x; c < ldx; c += gridDim.x * ROW_THREADS)
        {
            float v = 0.0f;
            if (ok && c < p.width)
            {
                v = (float)table[(size_t)id * p.width + c] * p.scale;
                if (pair >= 0)
                    v += (float)pairs[(size_t)pair * p.width + c];
            }
            x[(size_t)m * ldx + c] = v;
        }
    }

    // Workgroup = a row.  A few rows are bound by the chain of waits, so a thread asks for its HOLD pieces of the row and of the
    // norms at once and keeps them, where it used to read the row again and the norm only after the sum (0: longer rows still do).
    // The norm of 8 rows of 2048: a step of 33 passes with nine norms each 19.03 -> 18.80 ms; 2048 rows of 2048 columns
    // 6.3 -> 5.7 us, of 5120 21.9 -> 19.0.
    template <typename T, int HOLD>
    __global__ void __launch_bounds__(ROW_THREADS)
        seq_rmsnorm_kernel(const float *__restrict__ x, int ldx, const int32_t *__restrict__ rows,
                           const float *__restrict__ norm, float eps, int k_real, T *__restrict__ y, int K,
                           const float *__restrict__ norm2, T *__restrict__ y2)
    {
        typedef T t4 __attribute__((ext_vector_type(4)));
        __shared__ float s_sum[ROW_THREADS / 64];
        const int m = blockIdx.x;
        const f32x4 *row = reinterpret_cast<const f32x4 *>(x + (size_t)(rows ? rows[m] : m) * ldx);
        const f32x4 *scale = reinterpret_cast<const f32x4 *>(norm), *scale2 = reinterpret_cast<const f32x4 *>(norm2);
        t4 *out = reinterpret_cast<t4 *>(y + (size_t)m * K), *out2 = reinterpret_cast<t4 *>(y2 + (norm2 ? (size_t)m * K : 0));
        f32x4 v[HOLD + 1], a[HOLD + 1], b[HOLD + 1];
        float sum = 0.0f;
        auto add = [&sum](f32x4 u) { sum += u[0] * u[0] + u[1] * u[1] + u[2] * u[2] + u[3] * u[3]; };
#pragma unroll
        for (int j = 0; j < HOLD; ++j)
        {
            const int i = threadIdx.x + j * ROW_THREADS, at = i < K / 4 ? i : 0;
            v[j] = row[at], a[j] = scale[at];
            if (norm2)
                b[j] = scale2[at];
        }
        if (HOLD)
        {
#pragma unroll
            for (int j = 0; j < HOLD; ++j)
                if ((int)threadIdx.x + j * ROW_THREADS < K / 4)
                    add(v[j]);
        }
        else
            for (int i = threadIdx.x; i < K / 4; i += ROW_THREADS)
                add(row[i]);
        sum = block_sum<ROW_THREADS>(sum, s_sum);
        const float inv = 1.0f / sqrtf(sum / (float)k_real + eps);
        if (HOLD)
        {
#pragma unroll
            for (int j = 0; j < HOLD; ++j)
            {
                const int i = threadIdx.x + j * ROW_THREADS;
                if (i >= K / 4)
                    break;
                const f32x4 u = v[j] * inv;
                out[i] = __builtin_convertvector(u * a[j], t4);
                if (norm2)
                    out2[i] = __builtin_convertvector(u * b[j], t4);
            }
        }
        else
            for (int i = threadIdx.x; i < K / 4; i += ROW_THREADS)
            {
                const f32x4 u = row[i] * inv;
                out[i] = __builtin_convertvector(u * scale[i], t4);
                if (norm2)
                    out2[i] = __builtin_convertvector(u * scale2[i], t4);
            }
    }

    // ---- routed experts -------------------------------------------------------------------------
    struct ExpertArgs
    {
        const float *logits;
        int ldz;
        const bf16 *up, *down, *shared_up, *shared_down;
        long up_stride, down_stride;
        int experts, top, ff, shared_ff, K, N;
        const void *h; // T [M][K]
        float *x;
        int ldx;
        int *ids;       // [M][top]
        float *weights; // [M][top + 1]: of the chosen experts, then of the shared one
        bool routed;    // few rows: ids and weights are there already
        void *act;      // T: few rows [M][top * ff + shared_ff], many rows [M * top][ff] then [M][shared_ff]
        int *lists;     // few rows (see ExpertUse)
    };

    // Few rows: what their choices come to.  A list for every EXPERT_ROWS rows or half as many: the count of the experts that any of them
    // chose, in a piece of 16 bytes, [most][rows] uses of an expert by a row, in the order of the experts' numbers, and the numbers.
    constexpr int EXPERT_ROWS = 16;
    struct ExpertUse
    {
        float weight;
        int act; // where the row's activations begin, and the top bit; without that the row did not choose the expert (and they are another row's)
    };
    struct ExpertLists
    {
        int rows, most; // rows of a list, experts at most
        __host__ __device__ size_t ints() const { return 4 + (size_t)most * (rows * 2 + 1) + 3 & ~(size_t)3; }
        __device__ __forceinline__ int *at(int *lists, int i) const { return lists + i * ints(); }
        __device__ __forceinline__ ExpertUse *uses(int *list) const { return reinterpret_cast<ExpertUse *>(list + 4); }
        __device__ __forceinline__ int *numbers(int *list) const { return list + 4 + most * rows * 2; }
    };
    ExpertLists expert_lists(int M, int rows, int experts, int top)
    {
        const int of = M < rows ? M : rows;
        return {rows, of * top < experts ? of * top : experts};
    }
    __device__ __forceinline__ ExpertUse expert_use(float weight, int act, bool chosen) { return {weight, chosen ? act | (int)0x80000000 : act}; }

    // A wavefront per token chooses its experts.
    __global__ void __launch_bounds__(ROW_THREADS)
        expert_route_kernel(ExpertArgs p, int M)
    {
        const int lane = threadIdx.x & 63, m = blockIdx.x * (ROW_THREADS / 64) + (threadIdx.x >> 6);
        if (m >= M)
            return;
        const float *z = p.logits + (size_t)m * p.ldz;
        int id;
        float weight;
        route_wave(z, p.experts, p.top, lane, id, weight);
        if (lane < p.top)
        {
            p.ids[m * p.top + lane] = id;
            p.weights[m * (p.top + 1) + lane] = weight;
        }
        if (lane == 0 && p.shared_ff)
            p.weights[m * (p.top + 1) + p.top] = sigmoidf(z[p.experts]);
    }

    constexpr int EXPERT_WAVES = 8;
    // The lists of few rows, by one workgroup beside those of the up projections, which need none (by the launch that chooses: 1.8 us more).
    __device__ __forceinline__ void expert_list(const ExpertArgs &p, int M, ExpertLists lists, int from, int step)
    {
        constexpr int THREADS = EXPERT_WAVES * 64, BLOCKS = 64 * ROUTE_MAX / 64; // of experts, 64 in each
        struct Choice
        {
            int id;
            float weight;
        };
        __shared__ Choice s_choice[EXPERT_ROWS * 64];
        __shared__ int s_count[BLOCKS], s_number[64 * ROUTE_MAX];
        __shared__ uint8_t s_used[64 * ROUTE_MAX];
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        for (int i = threadIdx.x; i < M * p.top; i += THREADS)
            s_choice[i] = {p.ids[i], p.weights[i + i / p.top]};
        for (int first = from * lists.rows; first < M; first += step * lists.rows)
        {
            int *list = lists.at(p.lists, first / lists.rows);
            for (int i = threadIdx.x; i < 64 * ROUTE_MAX; i += THREADS)
                s_used[i] = 0;
            __syncthreads();
            const int rows = lists.rows < M - first ? lists.rows : M - first;
            for (int i = threadIdx.x; i < rows * p.top; i += THREADS)
                s_used[s_choice[first * p.top + i].id] = 1;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < BLOCKS / EXPERT_WAVES; ++i)
            {
                const unsigned long long used = __ballot(s_used[(i * EXPERT_WAVES + wave) * 64 + lane]);
                if (lane == 0)
                    s_count[i * EXPERT_WAVES + wave] = __builtin_popcountll(used);
            }
            __syncthreads();
            int count = 0;
            for (int i = 0; i < BLOCKS; ++i)
            {
                if (i % EXPERT_WAVES == wave)
                {
                    const bool is = s_used[i * 64 + lane];
                    const int place = count + __builtin_popcountll(__ballot(is) & ((1ull << lane) - 1));
                    if (is)
                        s_number[place] = lists.numbers(list)[place] = i * 64 + lane;
                }
                count += s_count[i];
            }
            if (threadIdx.x == 0)
                list[0] = count;
            __syncthreads();
            // a thread for every expert of the list and row, sixteen lanes for one
            const int n = threadIdx.x & (EXPERT_ROWS - 1), pitch = p.top * p.ff + p.shared_ff;
            for (int i = threadIdx.x / EXPERT_ROWS; i < ((count + 3) & ~3); i += THREADS / EXPERT_ROWS)
            {
                const int id = s_number[i < count ? i : 0];
                float weight = 0.0f;
                int at = -1;
                for (int j = 0; j < p.top; ++j)
                {
                    const Choice c = s_choice[(n < rows ? first + n : 0) * p.top + j];
                    const bool is = n < rows && c.id == id;
                    weight += is ? c.weight : 0.0f; // (several: logits that are not numbers)
                    at = is && at < 0 ? j : at;
                }
                const unsigned chosen = (unsigned)(__ballot(at >= 0) >> (lane & 48)) & 0xffff;
                const int lead = (lane & 48) | (__builtin_ctz(chosen | 0x10000) & 15);
                const int act = (first + n) * pitch + at * p.ff, others = __shfl(act, lead, 64);
                if (i < count && n < lists.rows)
                    lists.uses(list)[i * lists.rows + n] = expert_use(weight, at >= 0 ? act : others, at >= 0);
            }
            __syncthreads();
        }
    }
    // the list of a single row, by the wavefront that has chosen
    __device__ __forceinline__ void expert_list_one(const ExpertArgs &p, ExpertLists lists, int lane, int id, float weight)
    {
        int place = 0, first = lane;
        float sum = 0.0f;
        for (int j = p.top - 1; j >= 0; --j)
            first = __builtin_amdgcn_readlane(id, j) == id ? j : first;
        const unsigned long long leads = __ballot(lane < p.top && first == lane);
        for (int j = 0; j < p.top; ++j)
        {
            const int other = __builtin_amdgcn_readlane(id, j);
            sum += other == id ? __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, weight), j)) : 0.0f;
            place += (leads >> j & 1) != 0 && other < id ? 1 : 0;
        }
        if ((leads >> lane & 1) != 0)
        {
            for (int n = 0; n < lists.rows; ++n)
                lists.uses(p.lists)[place * lists.rows + n] = expert_use(sum, lane * p.ff, n == 0);
            lists.numbers(p.lists)[place] = id;
        }
        if (lane == 0)
            p.lists[0] = __builtin_popcountll(leads);
    }

    // Few rows.  Workgroup = 16 outputs of one expert, for every token that chose it: the tokens are the columns of the
    // matrix unit's second operand, so an expert's weights are read once however many chose it (the shared one: all).  Of
    // the workgroups of a (token, choice) pair those of the first token to choose the expert work, the others end.
    // With a single row all workgroups choose the token's experts for themselves from the logits, and the first records
    // the choice for the down projections; with more, a launch before has chosen.
    // Bound by the weights: 8 tokens, 6 of 64 experts of 1408 x 2048 each and a shared one of 2816, 56 us when each token
    // read its own and 44 now (about 200 MB of distinct weights).  The bits are the same: columns do not meet.
    template <typename T>
    __global__ void __launch_bounds__(EXPERT_WAVES * 64)
        expert_up_small_kernel(ExpertArgs p, int M, ExpertLists lists)
    {
        using O = Operand<T>;
        typedef T t4 __attribute__((ext_vector_type(4)));
        __shared__ __attribute__((aligned(16))) float s_red[EXPERT_WAVES][64][4];
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
        const int job = blockIdx.y, m = blockIdx.z; // jobs 0 .. top - 1: chosen experts; top: the shared one
        const bool shared = job == p.top;
        const int tile = blockIdx.x;
        const float *z = p.logits + (size_t)m * p.ldz;
        int expert = 0;
        unsigned long long mine = n < M ? 1 : 0; // which of token n's choices the expert is (several: logits that are not numbers)
        if (shared)
        {
            if (m >= 1 && tile == 0)
                expert_list(p, M, lists, m - 1, M - 1);
            if (m > 0 || tile * 16 >= p.shared_ff)
                return;
        }
        else if (tile * 16 >= p.ff)
            return;
        else if (p.routed)
        {
            expert = p.ids[m * p.top + job];
            mine = 0;
            for (int j = g; j < p.top; j += 4)
                if (n < M && p.ids[n * p.top + j] == expert)
                    mine |= 1ull << j;
            mine |= __shfl_xor(mine, 16, 64);
            mine |= __shfl_xor(mine, 32, 64);
            if ((__ballot(mine != 0) & ((1ull << m) - 1)) != 0)
                return; // an earlier token's workgroup
        }
        else
        {
            int id;
            float weight;
            route_wave(z, p.experts, p.top, lane, id, weight);
            if (tile == 0 && job == 0 && wave == 0)
            {
                expert_list_one(p, lists, lane, id, weight);
                if (lane == 0 && p.shared_ff)
                    p.weights[m * (p.top + 1) + p.top] = sigmoidf(z[p.experts]);
            }
            expert = __shfl(id, job, 64);
            mine <<= job;
        }
        const int ksteps = p.K >> 5;
        const u32x4 *w = weight_tile(shared ? p.shared_up : p.up + (size_t)expert * p.up_stride, tile, ksteps, lane);
        const T *h = static_cast<const T *>(p.h) + (size_t)(mine != 0 ? n : m) * p.K + 8 * g; // (other columns: m's, unused)
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        constexpr int U = 8;
        for (int s0 = wave; s0 < ksteps; s0 += EXPERT_WAVES * U)
        {
            u32x4 raw[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                const int s = s0 + u * EXPERT_WAVES;
                raw[u] = w[(size_t)(s < ksteps ? s : s0) * 64];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                const int s = s0 + u * EXPERT_WAVES;
                if (s < ksteps)
                    acc = O::mma(O::from_weights(raw[u]), O::load(h + s * 32), acc);
            }
        }
        *reinterpret_cast<f32x4 *>(s_red[wave][lane]) = acc;
        __syncthreads();
        if (threadIdx.x < 64 && mine != 0)
        {
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int i = 0; i < EXPERT_WAVES; ++i)
                v = v + *reinterpret_cast<const f32x4 *>(s_red[i][lane]);
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const float y = fmaxf(v[r], 0.0f);
                v[r] = y * y;
            }
            T *act = static_cast<T *>(p.act) + (size_t)n * (p.top * p.ff + p.shared_ff) + tile * 16 + 4 * g;
            do
            {
                const int at = shared ? p.top : __builtin_ctzll(mine);
                *reinterpret_cast<t4 *>(act + (size_t)at * p.ff) = __builtin_convertvector(v, t4);
                mine &= mine - 1;
            } while (mine != 0);
        }
    }

    // Few rows.  Workgroup = 8 columns of the output, or 16, of up to as many rows and over all experts that any of these chose: the shared
    // one, then those of the list, so that an expert's weights are read once however many rows chose it.  The k-steps of an expert
    // are taken in twos and dealt to the wavefronts, beginning with another one for every expert; a row's sums are of its own
    // experts, in the order of their numbers, so its bits are the same whatever other rows there are, also none.
    // HALF: rows 8 .. of the matrix unit's first operand are the same columns' second k-step of the two, and columns 8 .. of the
    // second operand the rows' (see linear_small_tile): twice the workgroups, and one product where there were two.
    // U: steps asked for at once, two turns of them on their way.
    // Bound by the weights, and for one or two rows by the chain of list, first weights and sums.  The weights were waited for where they were asked
    // for (the turn that is used was a copy of the one that came), and with small experts the walk from one to the next, by what LDS says, took as
    // long as they did.  us of this launch, 6 of 64 experts of 1408 x 2048 and a shared one of 2816 (in brackets: a workgroup for every row that
    // reads its own experts): 8 rows bf16 (47) 37.7 -> 37.8, fp32 (76) 57 -> 53; 16 rows 63.4 -> 57, 94 -> 88; 1 row (12) 10.7 -> 10.3,
    // (24) 15.9 -> 15.2.  8 of 128 of 768 x 2048, evenly chosen, 4 rows (17.2) 19.7 -> 17.7, fp32 (23) 29.5 -> 25.6; 8 rows (30.4) 32 -> 29, (43) 50 -> 42.
    // 4 of 128 of 256 x 1024, 8 rows (5.8) 12 -> 7.7.  16 rows at 1536 x 5120 177 -> 174, fp32 238 -> 223.
    // Slower than a workgroup for every row only where experts are hardly shared: a layer of 4 rows, 8 of 128 of 768 x 2048 45.6 and 47.0, fp32
    // 58.1 and 61.1, and by the list's 1 to 2 us at widths of 1024 and less.
    // Halves with U = 3 or 4: 8 rows 40.8, 41.2; U = 1, bf16, 8 rows 41, 9 rows 45.7 against 42.8, 12 rows 53.2 and 53.6, 16 rows 57 and 65.5.
    constexpr int DOWN_MANY = 10; // rows from beyond which on a step at a time is better
    template <typename T, bool HALF, int U>
    __global__ void __launch_bounds__(EXPERT_WAVES * 64, 4)
        expert_down_small_kernel(ExpertArgs p, int M, ExpertLists lists)
    {
        using O = Operand<T>;
        using V = typename O::V;
        constexpr int P = HALF ? 1 : 2; // products of a step
        __shared__ __attribute__((aligned(16))) float s_red[EXPERT_WAVES][P][64][4];
        extern __shared__ __attribute__((aligned(16))) char smem[]; // the list's uses
        const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
        const int tile = HALF ? blockIdx.x >> 1 : blockIdx.x;
        const int second = HALF ? n >> 3 : 0, row = HALF ? n & 7 : n, first = blockIdx.y * lists.rows;
        const int rows = lists.rows < M - first ? lists.rows : M - first, mine = row < rows ? row : 0;
        const int piece = (HALF ? g * 16 + (blockIdx.x & 1) * 8 + (n & 7) : lane) + second * 64;
        const int pitch = p.top * p.ff + p.shared_ff, esteps = p.ff >> 6, ssteps = p.shared_ff >> 6;
        // (the shared expert is the first of the list here, of a number that turns nothing)
        const int own = p.shared_ff ? 1 : 0;
        int *list = lists.at(p.lists, blockIdx.y);
        const auto number = [&](int job) __attribute__((always_inline)) {
            const int at = job - own < lists.most ? job - own : lists.most - 1;
            return at < 0 ? -EXPERT_WAVES : lists.numbers(list)[at];
        };
        int coming = number(lane);
        const int count = own + __builtin_amdgcn_readfirstlane(list[0]);
        ExpertUse *uses = reinterpret_cast<ExpertUse *>(smem);
        for (int i = threadIdx.x; i < lists.most * lists.rows; i += EXPERT_WAVES * 64)
            uses[own * lists.rows + i] = lists.uses(list)[i];
        if (own && (int)threadIdx.x < rows)
            uses[threadIdx.x] = expert_use(p.weights[(first + threadIdx.x) * (p.top + 1) + p.top], (first + threadIdx.x) * pitch + p.top * p.ff, true);

        f32x4 acc[P];
#pragma unroll
        for (int i = 0; i < P; ++i)
            acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int w0 = 0; w0 < count; w0 += 64)
        {
            // Lane j: the (w0 + j)-th of the list, the first of its steps among the wavefront's and their end.  An expert has as many as the
            // others or one more, so they are counted by one ballot and a step is found by another.
            const int job = w0 + lane, id = job < count ? coming : 0, start = (wave + id) & (EXPERT_WAVES - 1);
            coming = number(job + 64);
            const bool shared = own && job == 0;
            const int each = esteps / EXPERT_WAVES, some = (shared ? ssteps : esteps) & (EXPERT_WAVES - 1);
            const unsigned long long more = __ballot(job >= own && job < count && start < some);
            const int before = w0 > 0 || own == 0 || lane == 0 ? lane * each
                               : (lane - 1) * each + ssteps / EXPERT_WAVES + (wave < (ssteps & (EXPERT_WAVES - 1)) ? 1 : 0);
            const int from = before + __builtin_popcountll(more & ((1ull << lane) - 1));
            const int end = job < count ? from + (shared ? ssteps : esteps) / EXPERT_WAVES + (start < some ? 1 : 0) : INT_MAX;
            const int total = __builtin_amdgcn_readlane(end, (count - w0 < 64 ? count - w0 : 64) - 1);
            // the wavefront's steps s0 .. : their weights, their place in the expert, its uses (past the end the last step again, for no row)
            const u32x4 *w[U];
            int at[U], use_at[U];
            ExpertUse use[U];
            const auto find = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < U; ++u)
                {
                    const int s = s0 + u < total ? s0 + u : total - 1;
                    const int j = __builtin_popcountll(__ballot(end <= s));
                    const int e = __builtin_amdgcn_readlane(id, j), steps = e < 0 ? ssteps : esteps;
                    at[u] = ((wave + e) & (EXPERT_WAVES - 1)) + (s - __builtin_amdgcn_readlane(from, j)) * EXPERT_WAVES;
                    w[u] = reinterpret_cast<const u32x4 *>(e < 0 ? p.shared_down : p.down + (size_t)e * p.down_stride) + ((size_t)tile * steps + at[u]) * 128;
                    use_at[u] = (w0 + j) * lists.rows + mine;
                }
            };
            const auto look = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < U; ++u)
                    use[u] = uses[use_at[u]];
            };
            // Two turns of steps, one after the other: handed over (cur = next), the weights were waited for where they were asked for.
            u32x4 raw[2][U][P];
            V b[2][U][P];
            float scale[2][U];
            int act[2][U];
            const auto ask = [&](auto half) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < P; ++i)
                        raw[half.value][u][i] = w[u][i * 64 + piece];
            };
            const auto meet = [&](auto half, int s0) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < U; ++u)
                {
                    const T *from = static_cast<const T *>(p.act) + (size_t)(use[u].act & 0x7fffffff) + at[u] * 64 + 8 * g + second * 32;
#pragma unroll
                    for (int i = 0; i < P; ++i)
                        b[half.value][u][i] = O::load(from + i * 32);
                    scale[half.value][u] = use[u].weight;
                    act[half.value][u] = s0 + u < total ? use[u].act : 0;
                }
                find(s0 + U); // (a turn ahead of the weights)
                look();
            };
            const auto add = [&](auto half) __attribute__((always_inline)) {
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int i = 0; i < P; ++i)
                    {
                        const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
                        const f32x4 sum = acc[i] + O::mma(O::from_weights(raw[half.value][u][i]), b[half.value][u][i], zero) * scale[half.value][u];
                        acc[i] = act[half.value][u] < 0 ? sum : acc[i];
                    }
            };
            const std::integral_constant<int, 0> one;
            const std::integral_constant<int, 1> two;
            if (total > 0)
            {
                find(0);
                ask(one);
            }
            if (w0 == 0)
                __syncthreads(); // the uses are in LDS
            if (total == 0)
                continue;
            look();
            meet(one, 0);
            for (int s = 0; s < total; s += 2 * U)
            {
                ask(two);
                meet(two, s + U);
                add(one);
                ask(one);
                meet(one, s + 2 * U);
                add(two);
            }
        }
#pragma unroll
        for (int i = 0; i < P; ++i)
            *reinterpret_cast<f32x4 *>(s_red[wave][i][lane]) = acc[i];
        __syncthreads();
        if (threadIdx.x < 64 && n < rows && (!HALF || g < 2))
        {
            f32x4 *x = reinterpret_cast<f32x4 *>(p.x + (size_t)(first + n) * p.ldx + blockIdx.x * (HALF ? 8 : 16) + 4 * g);
            f32x4 v = *x;
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
                for (int i = 0; i < EXPERT_WAVES; ++i)
                    v = v + *reinterpret_cast<const f32x4 *>(s_red[i][HALF ? 0 : half][HALF ? lane + half * 40 : lane]);
            *x = v;
        }
    }

    // Many rows: after the choice of experts
    // the (token, choice) pairs are put in order of their expert, each expert's in the order of
    // the tokens: one workgroup per expert counts the pairs of lower experts and places its own.
    // Bound by waits: sixteen ids a thread are asked for at once and kept, and the wavefronts' shares of all sixteen rounds meet
    // in LDS behind one barrier, where every round used to read the ids twice and wait at two.  12288 pairs, 64 experts: 12.6 -> 5.6 us.
    constexpr int GROUP_THREADS = 1024, GROUP_WAVES = GROUP_THREADS / 64, GROUP_HOLD = 16;
    __global__ void __launch_bounds__(GROUP_THREADS)
        expert_group_kernel(const int *__restrict__ ids, int pairs, int experts, int *__restrict__ offset,
                            int *__restrict__ order, int *__restrict__ place)
    {
        __shared__ int s_low[GROUP_WAVES], s_own[GROUP_HOLD][GROUP_WAVES];
        const int e = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int rounds = (pairs + GROUP_THREADS - 1) / GROUP_THREADS; // of an id a thread
        int held[GROUP_HOLD];
        auto fetch = [&](int r0) {
#pragma unroll
            for (int j = 0; j < GROUP_HOLD; ++j)
            {
                const int i = (r0 + j) * GROUP_THREADS + threadIdx.x;
                held[j] = r0 + j < rounds && i < pairs ? ids[i] : INT_MAX; // (no expert, and none below)
            }
        };
        int low = 0;
        for (int r0 = 0; r0 < rounds; r0 += GROUP_HOLD)
        {
            fetch(r0);
#pragma unroll
            for (int j = 0; j < GROUP_HOLD; ++j)
                low += held[j] < e;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
            low += __shfl_xor(low, off, 64);
        if (lane == 0)
            s_low[wave] = low;
        int base = 0;
        for (int r0 = 0; r0 < rounds; r0 += GROUP_HOLD)
        {
            if (rounds > GROUP_HOLD)
                fetch(r0);
            if (r0 > 0)
                __syncthreads(); // the shares before have been read
#pragma unroll
            for (int j = 0; j < GROUP_HOLD; ++j)
            {
                const unsigned long long mask = __ballot(held[j] == e);
                if (lane == 0)
                    s_own[j][wave] = __popcll(mask);
            }
            __syncthreads();
            if (r0 == 0)
            {
#pragma unroll
                for (int w = 0; w < GROUP_WAVES; ++w)
                    base += s_low[w];
                if (threadIdx.x == 0)
                {
                    offset[e] = base;
                    if (e == experts - 1)
                        offset[experts] = pairs;
                }
            }
            // every wavefront adds the 256 shares up, four a lane: lane 4 j + w / 4 then knows what goes before wavefront w's of round j
            static_assert(GROUP_HOLD * GROUP_WAVES == 256 && GROUP_WAVES == 16, "four shares a lane");
            const int *share = &s_own[0][0] + 4 * lane;
            const int s0 = share[0], s1 = s0 + share[1], s2 = s1 + share[2], s3 = s2 + share[3];
            int upto = s3;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1)
            {
                const int below = __shfl_up(upto, off, 64);
                upto += lane >= off ? below : 0;
            }
            const int before = base + upto - s3 + ((wave & 3) == 0 ? 0 : (wave & 3) == 1 ? s0 : (wave & 3) == 2 ? s1 : s2);
            base += __builtin_amdgcn_readlane(upto, 63);
#pragma unroll
            for (int j = 0; j < GROUP_HOLD; ++j)
            {
                const unsigned long long mask = __ballot(held[j] == e);
                if (mask == 0)
                    continue;
                const int first = __builtin_amdgcn_readlane(before, 4 * j + (wave >> 2));
                if (held[j] == e)
                {
                    const int at = first + __popcll(mask & ((1ull << lane) - 1)), i = (r0 + j) * GROUP_THREADS + threadIdx.x;
                    order[at] = i;
                    place[i] = at;
                }
            }
        }
    }

    // and the experts' outputs are summed in the order of the choice
    __global__ void __launch_bounds__(ROW_THREADS)
        expert_combine_kernel(ExpertArgs p, const float *__restrict__ pair_out, const float *__restrict__ shared_out,
                              const int *__restrict__ place)
    {
        const int m = blockIdx.x;
        const float *weights = p.weights + m * (p.top + 1);
        for (int i = threadIdx.x; i < p.N / 4; i += ROW_THREADS)
        {
            f32x4 *x = reinterpret_cast<f32x4 *>(p.x + (size_t)m * p.ldx) + i;
            f32x4 y = {0.0f, 0.0f, 0.0f, 0.0f};
            for (int t = 0; t < p.top; ++t)
                y = y + reinterpret_cast<const f32x4 *>(pair_out + (size_t)place[m * p.top + t] * p.N)[i] * weights[t];
            if (p.shared_ff)
                y = y + reinterpret_cast<const f32x4 *>(shared_out + (size_t)m * p.N)[i] * weights[p.top];
            *x = *x + y;
        }
    }

    namespace
    {
        // scratch of the experts, from one buffer
        struct ExpertScratch
        {
            size_t ids, weights, act, lists, offset, order, place, pair_out, shared_out, total;
        };
        ExpertScratch expert_scratch(int M, int experts, int top, int ff, int shared_ff, int N)
        {
            ExpertScratch s{};
            size_t at = 0;
            auto take = [&at](size_t bytes) {
                const size_t here = at;
                at += (bytes + 255) & ~(size_t)255;
                return here;
            };
            const size_t pairs = (size_t)M * top;
            s.ids = take(pairs * 4);
            s.weights = take((size_t)M * (top + 1) * 4);
            s.act = take((pairs * ff + (size_t)M * shared_ff) * 4);
            size_t lists = 0;
            for (int rows = EXPERT_ROWS; rows > 0; rows /= 2)
                lists = std::max(lists, ceil_div(std::min(M, EXPERT_ROWS), rows) * expert_lists(M, rows, experts, top).ints());
            s.lists = take(lists * 4);
            s.offset = take((size_t)(experts + 1) * 4);
            s.order = take(pairs * 4);
            s.place = take(pairs * 4);
            s.pair_out = take(pairs * N * 4);
            s.shared_out = take(shared_ff ? (size_t)M * N * 4 : 0);
            s.total = at;
            return s;
        }

        template <typename T, bool HALF, int U>
        bool expert_down_launch(const char *fn, const ExpertArgs &p, int M, ExpertLists lists, hipStream_t st)
        {
            auto *kernel = expert_down_small_kernel<T, HALF, U>;
            static LdsGrant grant;
            const size_t use = lists.rows * sizeof(ExpertUse), lds = (lists.most + (p.shared_ff ? 1 : 0)) * use;
            if (lds > 48 * 1024 && allow_lds(grant, reinterpret_cast<const void *>(kernel), (64 * ROUTE_MAX + 1) * EXPERT_ROWS / (HALF ? 2 : 1) * sizeof(ExpertUse)) != hipSuccess)
                return fail(fn, "cannot reserve %zu bytes of LDS", lds);
            hipLaunchKernelGGL(kernel, dim3(p.N / (HALF ? 8 : 16), ceil_div(M, lists.rows)), dim3(EXPERT_WAVES * 64), lds, st, p, M, lists);
            return launched(fn);
        }

        template <typename T>
        bool experts_run(const char *fn, ExpertArgs p, int M, char *scratch, int dtype, int device_id, hipStream_t st)
        {
            const ExpertScratch at = expert_scratch(M, p.experts, p.top, p.ff, p.shared_ff, p.N);
            p.ids = reinterpret_cast<int *>(scratch + at.ids);
            p.weights = reinterpret_cast<float *>(scratch + at.weights);
            p.act = scratch + at.act;
            if (M > 1)
            {
                hipLaunchKernelGGL(expert_route_kernel, dim3(ceil_div(M, ROW_THREADS / 64)), dim3(ROW_THREADS), 0, st, p, M);
                if (!launched(fn))
                    return false;
                p.routed = true;
            }
            if (M <= SMALL_M)
            {
                static_assert(SMALL_M == EXPERT_ROWS, "a list has a column for each of few rows");
                // Halves of tiles, for eight rows at a time, but for more rows whole ones where these alone occupy the chip (bf16, us, halves
                // and whole tiles: 16 rows, 64 experts of 1536 x 5120 351, 332; 16 of 4096 x 4096 207, 170; 64 of 1408 x 2048 135, 141;
                // 8 rows, 1536 x 5120 226, 238; the down projections alone, 12 rows of 1408 x 2048 54, 62).
                const bool half = M <= EXPERT_ROWS / 2 || p.N / 16 < cu_count(device_id);
                // Fewer rows at a time where these would leave compute units without a workgroup (us, 8 rows, 4 of 128 of 256 x 1024, lists
                // of 8 and 4 rows 19.1, 17.9, fp32 25.3, 22.5).
                int rows = half ? EXPERT_ROWS / 2 : EXPERT_ROWS;
                while (half && rows > 1 && p.N / 8 * ceil_div(M, rows) < cu_count(device_id))
                    rows /= 2;
                const ExpertLists lists = expert_lists(M, rows, p.experts, p.top);
                p.lists = reinterpret_cast<int *>(scratch + at.lists);
                const int widest = p.shared_ff > p.ff ? p.shared_ff : p.ff;
                hipLaunchKernelGGL(expert_up_small_kernel<T>, dim3(widest / 16, p.top + (p.shared_ff || M > 1 ? 1 : 0), M),
                                   dim3(EXPERT_WAVES * 64), 0, st, p, M, lists);
                if (!launched(fn))
                    return false;
                if (!half)
                    return expert_down_launch<T, false, sizeof(T) == 2 ? 2 : 1>(fn, p, M, lists, st);
                return M > DOWN_MANY ? expert_down_launch<T, true, 1>(fn, p, M, lists, st) : expert_down_launch<T, true, 2>(fn, p, M, lists, st);
            }
            int *offset = reinterpret_cast<int *>(scratch + at.offset), *order = reinterpret_cast<int *>(scratch + at.order);
            int *place = reinterpret_cast<int *>(scratch + at.place);
            float *pair_out = reinterpret_cast<float *>(scratch + at.pair_out);
            float *shared_out = reinterpret_cast<float *>(scratch + at.shared_out);
            hipLaunchKernelGGL(expert_group_kernel, dim3(p.experts), dim3(GROUP_THREADS), 0, st, p.ids, M * p.top, p.experts,
                               offset, order, place);
            if (!launched(fn))
                return false;
            LinearArgs l{};
            l.source_div = 1;
            T *act = static_cast<T *>(p.act), *shared_act = act + (size_t)M * p.top * p.ff;
            // the gated tokens of each expert: every expert may get all M
            l.a = p.h, l.lda = p.K, l.w = p.up, l.w_stride = p.up_stride, l.y = act, l.ldy = p.ff;
            l.M = M, l.N = p.ff, l.K = p.K, l.out = LLAM_SEQ_OUT_RELU2;
            l.group_offset = offset, l.row_source = order, l.source_div = p.top, l.groups = p.experts, l.group_rows = M * p.top;
            if (!linear_tiled(fn, l, p.experts, dtype, device_id, st))
                return false;
            l.a = act, l.lda = p.ff, l.w = p.down, l.w_stride = p.down_stride, l.y = pair_out, l.ldy = p.N;
            l.N = p.N, l.K = p.ff, l.out = LLAM_SEQ_OUT_F32, l.row_source = nullptr, l.source_div = 1;
            if (!linear_tiled(fn, l, p.experts, dtype, device_id, st))
                return false;
            if (p.shared_ff)
            {
                LinearArgs s{};
                s.source_div = 1;
                s.a = p.h, s.lda = p.K, s.w = p.shared_up, s.y = shared_act, s.ldy = p.shared_ff;
                s.M = M, s.N = p.shared_ff, s.K = p.K, s.out = LLAM_SEQ_OUT_RELU2;
                if (!linear_tiled(fn, s, 1, dtype, device_id, st))
                    return false;
                s.a = shared_act, s.lda = p.shared_ff, s.w = p.shared_down, s.y = shared_out, s.ldy = p.N;
                s.N = p.N, s.K = p.shared_ff, s.out = LLAM_SEQ_OUT_F32;
                if (!linear_tiled(fn, s, 1, dtype, device_id, st))
                    return false;
            }
            hipLaunchKernelGGL(expert_combine_kernel, dim3(M), dim3(ROW_THREADS), 0, st, p, pair_out, shared_out, place);
            return launched(fn);
        }
    } // namespace
} // namespace llamql

using namespace llamql;

extern "C" bool llam_seq_embed(const llam_seq_embed_args *a, const int32_t *d_ids, float *d_x, int M, int ldx, int device_id,
                               void *stream)
{
    static const char *fn = "llam_seq_embed";
    if (!a || !a->d_table || !d_ids || !d_x)
        return fail(fn, "null pointer");
    if (M < 0 || M > 65535 || a->vocab < 1 || a->width < 1 || ldx < a->width)
        return fail(fn, "bad size (M=%d vocab=%d width=%d ldx=%d)", M, a->vocab, a->width, ldx);
    if (a->d_pairs && (!a->d_row_slot || !a->d_row_pos || !a->d_history || a->buckets < 1 || a->cap < 1))
        return fail(fn, "pairs of tokens need rows, a history and buckets=%d cap=%d of at least 1", a->buckets, a->cap);
    if (!aligned16(a->d_table) || !aligned16(a->d_pairs) || !aligned16(d_x))
        return fail(fn, "misaligned rows");
    if (M == 0)
        return true;
    if (!set_device(fn, device_id))
        return false;
    hipLaunchKernelGGL(seq_embed_kernel, dim3(M >= EMBED_WIDE_ROWS ? 1 : ceil_div(ldx, 4 * ROW_THREADS), M), dim3(ROW_THREADS), 0, as_stream(stream), *a, d_ids, d_x, ldx);
    return launched(fn);
}

namespace
{
    // two or six pieces of four columns a thread, or any number
    template <typename T>
    void rmsnorm_launch(int M, hipStream_t st, const float *x, int ldx, const int32_t *rows, const float *norm, float eps, int k_real, T *y, int K,
                        const float *norm2, T *y2)
    {
        auto *kernel = K <= 2 * 4 * ROW_THREADS   ? seq_rmsnorm_kernel<T, 2>
                       : K <= 6 * 4 * ROW_THREADS ? seq_rmsnorm_kernel<T, 6>
                                                  : seq_rmsnorm_kernel<T, 0>;
        hipLaunchKernelGGL(kernel, dim3(M), dim3(ROW_THREADS), 0, st, x, ldx, rows, norm, eps, k_real, y, K, norm2, y2);
    }

    bool rmsnorm(const char *fn, const float *d_x, int ldx, const int32_t *d_rows, const float *d_norm, const float *d_norm2, float eps,
                 int k_real, void *d_y, void *d_y2, int M, int K, int dtype, int device_id, void *stream)
    {
        if (M < 0 || K < 1 || k_real < 1 || k_real > K || ldx < K)
            return fail(fn, "bad size (M=%d K=%d k_real=%d ldx=%d)", M, K, k_real, ldx);
        if (M == 0)
            return true;
        if (!d_x || !d_norm || !d_y)
            return fail(fn, "null pointer");
        if ((K % 8) != 0 || (ldx % 4) != 0 || !aligned16(d_x) || !aligned16(d_norm) || !aligned16(d_y) || !aligned16(d_norm2) || !aligned16(d_y2))
            return fail(fn, "misaligned rows");
        if (!set_device(fn, device_id))
            return false;
        if (dtype == LLAM_SEQ_F32)
            rmsnorm_launch(M, as_stream(stream), d_x, ldx, d_rows, d_norm, eps, k_real, static_cast<float *>(d_y), K, d_norm2, static_cast<float *>(d_y2));
        else
            rmsnorm_launch(M, as_stream(stream), d_x, ldx, d_rows, d_norm, eps, k_real, static_cast<bf16 *>(d_y), K, d_norm2, static_cast<bf16 *>(d_y2));
        return launched(fn);
    }
} // namespace

extern "C" bool llam_seq_rmsnorm(const float *d_x, int ldx, const int32_t *d_rows, const float *d_norm, float eps,
                                 int k_real, void *d_y, int M, int K, int dtype, int device_id, void *stream)
{
    return rmsnorm("llam_seq_rmsnorm", d_x, ldx, d_rows, d_norm, nullptr, eps, k_real, d_y, nullptr, M, K, dtype, device_id, stream);
}

extern "C" bool llam_seq_rmsnorm_pair(const float *d_x, int ldx, const float *d_norm_a, const float *d_norm_b, float eps, int k_real,
                                      void *d_ya, void *d_yb, int M, int K, int dtype, int device_id, void *stream)
{
    static const char *fn = "llam_seq_rmsnorm_pair";
    if (!d_norm_b || !d_yb)
        return fail(fn, "null pointer");
    return rmsnorm(fn, d_x, ldx, nullptr, d_norm_a, d_norm_b, eps, k_real, d_ya, d_yb, M, K, dtype, device_id, stream);
}

extern "C" size_t llam_seq_experts_scratch_bytes(int max_rows, int experts, int top, int ff, int shared_ff, int N)
{
    if (max_rows < 1 || experts < 1 || top < 1 || ff < 1 || shared_ff < 0 || N < 1)
        return 0;
    return expert_scratch(max_rows, experts, top, ff, shared_ff, N).total;
}

extern "C" bool llam_seq_experts(const llam_seq_experts_args *a, int M, void *d_scratch, size_t scratch_bytes, int dtype,
                                 int device_id, void *stream)
{
    static const char *fn = "llam_seq_experts";
    if (!a || !a->d_logits || !a->d_up || !a->d_down || !a->d_h || !a->d_x || !d_scratch)
        return fail(fn, "null pointer");
    if (M < 0 || a->experts < 1 || a->top < 1 || a->top > a->experts || a->top > 64 || a->experts > 64 * ROUTE_MAX)
        return fail(fn, "bad size (M=%d experts=%d top=%d)", M, a->experts, a->top);
    if (M == 0)
        return true;
    if ((a->ff % PAD) != 0 || a->ff < PAD || (a->shared_ff % PAD) != 0 || (a->K % PAD) != 0 || (a->N % 16) != 0 || (a->ldx % 4) != 0 || a->ldx < a->N)
        return fail(fn, "ff=%d, shared_ff=%d and K=%d must be multiples of %d, N=%d of 16", a->ff, a->shared_ff, a->K, PAD, a->N);
    if (a->shared_ff && (!a->d_shared_up || !a->d_shared_down))
        return fail(fn, "null pointer (shared expert)");
    if (a->ldz < a->experts + (a->shared_ff ? 1 : 0))
        return fail(fn, "ldz=%d too small", a->ldz);
    if (llam_seq_experts_scratch_bytes(M, a->experts, a->top, a->ff, a->shared_ff, a->N) > scratch_bytes)
        return fail(fn, "scratch too small");
    if (M > 65535)
        return fail(fn, "M=%d rows", M);
    if (!set_device(fn, device_id))
        return false;
    ExpertArgs p{};
    p.logits = a->d_logits, p.ldz = a->ldz;
    p.up = static_cast<const bf16 *>(a->d_up), p.down = static_cast<const bf16 *>(a->d_down);
    p.shared_up = static_cast<const bf16 *>(a->d_shared_up), p.shared_down = static_cast<const bf16 *>(a->d_shared_down);
    p.up_stride = a->up_stride, p.down_stride = a->down_stride;
    p.experts = a->experts, p.top = a->top, p.ff = a->ff, p.shared_ff = a->shared_ff, p.K = a->K, p.N = a->N;
    p.h = a->d_h, p.x = a->d_x, p.ldx = a->ldx;
    return dtype == LLAM_SEQ_F32 ? experts_run<float>(fn, p, M, static_cast<char *>(d_scratch), dtype, device_id, as_stream(stream))
                                 : experts_run<bf16>(fn, p, M, static_cast<char *>(d_scratch), dtype, device_id, as_stream(stream));
}
