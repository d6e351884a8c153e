// Quad-lane decode GEMV (gfx950): four lanes own one 256-element super-block.
//
// Lane l of a quad decodes 64 weights -- the two complete 32-element blocks 2l and
// 2l+1 of its super-block -- so it forms both exact int32 block sums by itself (no
// exchange between lanes) and decodes the super-block header once for two blocks.
// A wavefront step covers 16 consecutive super-blocks.
//
// A wavefront owns a contiguous range of weight rows and walks it as ONE run of
// super-blocks, 16 per step, whatever the row length: a step may contain the end of
// one row and the start of the next.  Two running sums per lane (`cur`: the row being
// finished, `nxt`: the row after it) take the step's contribution according to the
// lane's position; when a row ends inside a step its 64 partial sums are reduced in a
// fixed order and stored, and `nxt` becomes `cur`.  Rows must have at least 16
// super-blocks (K >= 4096) so that a step touches at most two rows.
//
// Loads run U steps ahead in two alternating register buffers.  Activations (Q8_1)
// are staged once per workgroup in LDS, 320 bytes per super-block and activation row:
//   [m][sb]{ part 0..3: [l][16 B of quants]   part = 2*(first|second block of the lane) + half
//            [l]{f32 d, f32 sum*d of the lane's first block ; same of its second} }
// so a lane reads its five 16-byte pieces at fixed offsets from ONE address (the super-block
// of a lane changes by 16 modulo the row length from step to step) and the 16 lanes served
// together fall into different banks.  The Q8_1 blocks are asked for BEFORE the first weight
// chunks: a wavefront's loads return in issue order, and activations queued behind 14 KB of
// weights would hold up the staging, the barrier and with them the first product.
//
// Per block: idot exact; acc = fma(float(idot), f32(a.d)*b_scale, acc);
// acc = fma(float(a.sum)*f32(a.d), b_min, acc) -- the reference's arithmetic
// (CPUNativeVNNIGemv.h:417-487); only the order in which blocks are added differs.
#pragma once

#include "gemv_core.h"

namespace llamql
{
    constexpr int QUAD_STEP_SB = 16; // super-blocks per wavefront step
    constexpr size_t QUAD_MAX_LDS = 160 * 1024; // LDS of one gfx950 compute unit
    constexpr int QUAD_MAX_PROJ = 4;            // weight matrices one launch can walk

    // Where the activations come from.  The fp32 kinds quantise to Q8_1 inside the kernel,
    // every workgroup for itself while its first weight loads are in flight, with the
    // arithmetic of the stand-alone quantisers: the launch of a quantiser kernel and the
    // round trip of its output through memory are saved, the results are the same bits.
    constexpr int QUAD_SRC_Q8 = 0;     // Q8_1 blocks
    constexpr int QUAD_SRC_F32 = 1;    // fp32 rows
    constexpr int QUAD_SRC_SWIGLU = 2; // silu(gate) * up of two fp32 inputs
    constexpr int QUAD_SRC_RMSNORM = 3; // RMSNorm of fp32 residual rows (+ delta), batches of 1..QUAD_NORM_MAX_M
    // (every workgroup normalises and quantises all rows again: measured against a norm launch of
    // its own, 3.4 us, that pays for a single row of 5120 and no longer for four)
    constexpr int QUAD_NORM_MAX_M = 1;
    constexpr int QUAD_NORM_LDS = 8 * 8 * QUAD_NORM_MAX_M; // LDS bytes of the norm's partial sums

    // One launch: up to QUAD_MAX_PROJ weight matrices of one row length against the same
    // activations (projections that share an input: Q, K and V; gate and up).  The
    // wavefronts of the launch are dealt to the matrices in order: matrix p owns the
    // wavefronts from wave_begin[p] on (those beyond its last row idle).  Matrices from
    // first_b on are in the second format of a two-format launch and start at a workgroup
    // boundary, because a workgroup stages the activations in its format's order.
    struct QuadArgs
    {
        const uint32_t *q8; // Q8_1 activations as dwords (9 per block), M rows (QUAD_SRC_Q8)
        const float *x;     // fp32 activations, M rows of ldx floats (QUAD_SRC_F32); the gate
        const float *x2;    // rows for QUAD_SRC_SWIGLU, whose up rows are x2
        int ldx;
        // QUAD_SRC_RMSNORM: x are the residual rows, x2 the delta rows added first (or null), gamma the
        // norm's weights; workgroup 0 stores x + delta to x_out (when there is a delta).  The
        // partial sums of squares live in QUAD_NORM_LDS bytes of LDS at byte offset norm_lds.
        const float *gamma;
        float *x_out;
        float eps;
        int norm_lds;
        int SB;             // super-blocks per weight row
        int nproj;
        const void *w[QUAD_MAX_PROJ];
        float *y[QUAD_MAX_PROJ];
        int N[QUAD_MAX_PROJ];
        int ldy[QUAD_MAX_PROJ];
        int R[QUAD_MAX_PROJ]; // rows per wavefront (the most any wavefront of the matrix walks)
        // The rows of a matrix are dealt round robin: wavefront j of its TW walks rows j, j + TW, ..
        // (rows_min of them, one more for the first N - rows_min * TW wavefronts).  At any moment
        // the wavefronts of the launch then read rows that lie close together in memory.
        int TW[QUAD_MAX_PROJ];
        int rows_min[QUAD_MAX_PROJ];
        int wave_begin[QUAD_MAX_PROJ];
        int first_b; // nproj in a launch of one format
        // DUMP kernels only (one matrix): the exact per-block int32 sums of rows [row0, row0+nrows)
        // go to sums[(m * nrows + row - row0) * (SB * 8) + block]
        int32_t *sums;
        int row0, nrows;
        // up to QUAD_RING_MAX_M activation rows: the launch reserves QUAD_RING_BYTES of LDS per
        // wavefront and row behind the activations and the kernel runs in QUAD_MODE_RING
        int ring;
        // QUAD_MODE_RING only, wavefronts of at most QUAD_RING_ROWS rows: the row sums are ADDED to what
        // y holds (y += W a: the residual add of the next norm done by the projection that feeds it)
        int accumulate;
    };

    // LDS bytes for M activation rows of nsb super-blocks.
    constexpr int QUAD_SB_LDS = 320; // LDS bytes per super-block and activation row
    // Single activation row (QUAD_MODE_RING): finished rows park their 64 per-lane partial sums in a
    // per-wavefront LDS ring and are reduced 16 rows at a time (lane = (row, quarter): 16 values each,
    // then two exchanges inside the quad), so the loop carries no reduction chain and the row
    // sums leave as 64-byte stores.  The additions are associated exactly as wave_sum() does it
    // (pairs, quads, eights, sixteens, then (r0+r1)+(r2+r3)): the same bits either way.
    constexpr int QUAD_RING_ROWS = 16;
    constexpr int QUAD_RING_STRIDE = 68; // floats per parked row: 64 + 4 so neighbouring rows start 4 banks apart
    constexpr size_t QUAD_RING_BYTES = (size_t)QUAD_RING_ROWS * QUAD_RING_STRIDE * 4; // per wavefront and activation row
    constexpr int QUAD_RING_MAX_M = 4; // batches that may run in QUAD_MODE_RING (where the LDS has the room)
    inline size_t quad_lds_bytes(int M, int nsb)
    {
        return (size_t)M * (size_t)nsb * QUAD_SB_LDS;
    }

    // One thread per Q8_1 block.  Block j of a super-block goes to the quad lane that
    // decodes it (Q::owner) as that lane's first or second block.
    template <class Q, int M>
    __device__ __forceinline__ void quad_stage_q8(const uint32_t *__restrict__ q8, int nsb, uint8_t *aq, uint8_t *ads,
                                                  int aq_stride, int ads_stride)
    {
        const int nkb = nsb * 8;
#pragma unroll
        for (int m = 0; m < M; ++m)
        {
            for (int kb = threadIdx.x; kb < nkb; kb += blockDim.x)
            {
                const uint32_t *src = q8 + ((size_t)m * nkb + kb) * 9;
                uint32_t v[9];
#pragma unroll
                for (int i = 0; i < 9; ++i)
                    v[i] = src[i];
                const float d = h2f((uint16_t)(v[0] & 0xFFFFu));
                const int sb = kb >> 3, j = kb & 7;
                int l, odd;
                Q::owner(j, l, odd);
                uint8_t *base = aq + m * aq_stride + sb * QUAD_SB_LDS + l * 16;
                *reinterpret_cast<float2 *>(base + 256 + odd * 8) = make_float2(d, (float)(int16_t)(v[0] >> 16) * d);
                *reinterpret_cast<uint4 *>(base + (odd * 2) * 64) = make_uint4(v[1], v[2], v[3], v[4]);
                *reinterpret_cast<uint4 *>(base + (odd * 2 + 1) * 64) = make_uint4(v[5], v[6], v[7], v[8]);
            }
        }
    }

    // Q8_1 blocks fetched ahead of the weights.  A wavefront's loads return in the order they
    // were issued: activations asked for after the first weight chunks would arrive behind
    // them, and the staging (and the barrier after it) would wait for 18 KB of weights per
    // wavefront first.  Here every thread asks for up to QUAD_ACT_PASSES blocks before the
    // weight loads go out and waits for exactly those (the weights stay in flight).  The loads
    // are assembly so that the kernel decides where they are waited for; they are never
    // predicated (threads without a block re-read the last one).
    constexpr int QUAD_ACT_PASSES = 2;
    struct QuadActRaw
    {
        v4i lo, hi;
        int tail;
    };
    // thread `tid` of `nthreads` that share the `total` blocks (a workgroup, or one wavefront of it)
    template <int PASSES>
    __device__ __forceinline__ void quad_act_issue(QuadActRaw (&r)[PASSES], const uint32_t *q8, int total, int tid,
                                                   int nthreads)
    {
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
        {
            int idx = tid + p * nthreads;
            idx = idx < total ? idx : total - 1;
            const uint32_t *src = q8 + (size_t)idx * 9;
            asm volatile("global_load_dwordx4 %0, %1, off" : "=&v"(r[p].lo) : "v"(src));
            asm volatile("global_load_dwordx4 %0, %1, off offset:16" : "=&v"(r[p].hi) : "v"(src));
            asm volatile("global_load_dword %0, %1, off offset:32" : "=&v"(r[p].tail) : "v"(src));
        }
    }
    template <int PASSES>
    __device__ __forceinline__ void quad_act_issue(QuadActRaw (&r)[PASSES], const uint32_t *q8, int total)
    {
        quad_act_issue(r, q8, total, (int)threadIdx.x, (int)blockDim.x);
    }
    // until at most NEWER vector memory operations issued after the activation loads are pending
    template <int NEWER, int PASSES>
    __device__ __forceinline__ void quad_act_wait(QuadActRaw (&r)[PASSES])
    {
        static_assert(NEWER <= 63, "vmcnt is a 6-bit counter");
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
            asm volatile("s_waitcnt vmcnt(%3)" : "+v"(r[p].lo), "+v"(r[p].hi), "+v"(r[p].tail) : "n"(NEWER));
    }
    template <class Q, int PASSES>
    __device__ __forceinline__ void quad_act_store(const QuadActRaw (&r)[PASSES], int nsb, int total,
                                                   uint8_t *aq, int aq_stride, int tid, int nthreads)
    {
        const int nkb = nsb * 8;
#pragma unroll
        for (int p = 0; p < PASSES; ++p)
        {
            const int idx = tid + p * nthreads;
            if (idx < total)
            {
                const int m = idx / nkb, kb = idx - m * nkb;
                const uint32_t head = (uint32_t)r[p].lo.x;
                const float d = h2f((uint16_t)(head & 0xFFFFu));
                const int sb = kb >> 3, j = kb & 7;
                int l, odd;
                Q::owner(j, l, odd);
                uint8_t *base = aq + m * aq_stride + sb * QUAD_SB_LDS + l * 16;
                *reinterpret_cast<float2 *>(base + 256 + odd * 8) = make_float2(d, (float)(int16_t)(head >> 16) * d);
                *reinterpret_cast<v4i *>(base + (odd * 2) * 64) = (v4i){r[p].lo.y, r[p].lo.z, r[p].lo.w, r[p].hi.x};
                *reinterpret_cast<v4i *>(base + (odd * 2 + 1) * 64) = (v4i){r[p].hi.y, r[p].hi.z, r[p].hi.w, r[p].tail};
            }
        }
    }

    template <class Q, int PASSES>
    __device__ __forceinline__ void quad_act_store(const QuadActRaw (&r)[PASSES], int nsb, int total,
                                                   uint8_t *aq, int aq_stride)
    {
        quad_act_store<Q, PASSES>(r, nsb, total, aq, aq_stride, (int)threadIdx.x, (int)blockDim.x);
    }

    // One lane's share (float4 number i of the row) of a quantised 32-element block into the
    // activation row at aq_row, in the layout the decoder Q reads.
    template <class Q>
    __device__ __forceinline__ void quad_store_q8_lane(const Q8Lane q, int i, uint8_t *aq_row)
    {
        const int kb = i >> 3, sub = i & 7;
        const int sb = kb >> 3, j = kb & 7;
        int l, odd;
        Q::owner(j, l, odd);
        uint8_t *base = aq_row + sb * QUAD_SB_LDS + l * 16;
        if (sub == 0)
        {
            const float d = h2f((uint16_t)(q.head & 0xFFFFu));
            *reinterpret_cast<float2 *>(base + 256 + odd * 8) = make_float2(d, (float)(int16_t)(q.head >> 16) * d);
        }
        *reinterpret_cast<uint32_t *>(base + (odd * 2 + (sub >> 2)) * 64 + (sub & 3) * 4) = q.packed;
    }

    // The same from fp32 rows (SRC = QUAD_SRC_F32) or from silu(x) * x2 (QUAD_SRC_SWIGLU):
    // eight neighbouring threads quantise one 32-element block.
    template <class Q, int M, int SRC>
    __device__ __forceinline__ void quad_stage_f32(const float *__restrict__ x, const float *__restrict__ x2, int ldx,
                                                   int nsb, uint8_t *aq, uint8_t *ads, int aq_stride, int ads_stride)
    {
        const int nvec = nsb * 64; // float4 per row; workgroup sizes are multiples of 64
#pragma unroll
        for (int m = 0; m < M; ++m)
        {
            const float4 *row = reinterpret_cast<const float4 *>(x + (size_t)m * ldx);
            const float4 *row2 = reinterpret_cast<const float4 *>(x2 + (size_t)m * ldx);
            // four loads in flight per thread: the latency of a round trip is paid per batch
            constexpr int UN = SRC == QUAD_SRC_SWIGLU ? 2 : 4;
            for (int i0 = threadIdx.x; i0 < nvec; i0 += UN * (int)blockDim.x)
            {
                float4 v[UN], v2[UN];
#pragma unroll
                for (int u = 0; u < UN; ++u)
                {
                    const int i = min(i0 + u * (int)blockDim.x, nvec - 1);
                    v[u] = row[i];
                    if constexpr (SRC == QUAD_SRC_SWIGLU)
                        v2[u] = row2[i];
                }
#pragma unroll
                for (int u = 0; u < UN; ++u)
                {
                    const int i = i0 + u * (int)blockDim.x;
                    if (i >= nvec) // whole 8-thread groups leave together
                        break;
                    if constexpr (SRC == QUAD_SRC_SWIGLU)
                        v[u] = swiglu4(v[u], v2[u]);
                    quad_store_q8_lane<Q>(q8_1_quantize_lane(v[u]), i, aq + m * aq_stride);
                }
            }
        }
    }

    // RMSNorm of the residual rows in front of the quantiser (QUAD_SRC_RMSNORM), with the bits of the
    // stand-alone operator (rmsnorm_q8_1_kernel: 512 threads, thread t sums the squares of float4
    // t, t + 512, .. in double, the 64 lanes of a wavefront are added as a butterfly, the eight
    // wavefronts in order).  Here the threads of the workgroup play those 512 "virtual threads",
    // every workgroup of the launch for itself.  Workgroups of 512 threads and more on rows of up to
    // 8192 values keep a virtual thread's values and weights in registers between the sum and the
    // scaling (all loads are issued before the sum, nothing is read twice); the others play the
    // virtual threads in turn, whole wavefronts at a time, and read the row again from the caches.
    // Contains a workgroup barrier.
    template <class Q, int M>
    __device__ __forceinline__ void quad_stage_rmsnorm(const QuadArgs &qa, int nsb, uint8_t *aq, int aq_stride,
                                                       uint8_t *quad_lds)
    {
        constexpr int VT = 512; // threads of the stand-alone kernel
        constexpr int KEEP = 4; // float4 of a virtual thread kept in registers
        const int H = nsb * 256, nvec = nsb * 64;
        double *s_part = reinterpret_cast<double *>(quad_lds + qa.norm_lds); // [M][8]
        // (the workgroup that stores x + delta: a variant that added a workgroup without rows for it
        // measured the same)
        const bool writer = blockIdx.x == 0 && qa.x2 != nullptr && qa.x_out != nullptr;
        const float4 *g4 = reinterpret_cast<const float4 *>(qa.gamma);
        auto add4 = [](float4 v, const float4 d) {
            v.x += d.x;
            v.y += d.y;
            v.z += d.z;
            v.w += d.w;
            return v;
        };
        auto row_value = [&](int m, int i) {
            const float4 v = reinterpret_cast<const float4 *>(qa.x + (size_t)m * qa.ldx)[i];
            return qa.x2 ? add4(v, reinterpret_cast<const float4 *>(qa.x2 + (size_t)m * qa.ldx)[i]) : v;
        };
        auto square = [](double &acc, const float4 v) {
            acc += (double)v.x * (double)v.x;
            acc += (double)v.y * (double)v.y;
            acc += (double)v.z * (double)v.z;
            acc += (double)v.w * (double)v.w;
        };
        auto butterfly = [](double acc) { return wave_sum(acc); }; // the stand-alone norm's reduction
        auto inverse_rms = [&](int m) {
            double sum_sq = 0.0;
#pragma unroll
            for (int w = 0; w < VT / WAVE; ++w)
                sum_sq += s_part[m * 8 + w];
            const float rms = __fsqrt_rn(__fadd_rn((float)(sum_sq / (double)H), qa.eps));
            return __fdiv_rn(1.0f, rms);
        };
        auto emit = [&](int m, int i, const float4 v, const float4 g, float inv) {
            float4 o;
            o.x = __fmul_rn(__fmul_rn(v.x, inv), g.x);
            o.y = __fmul_rn(__fmul_rn(v.y, inv), g.y);
            o.z = __fmul_rn(__fmul_rn(v.z, inv), g.z);
            o.w = __fmul_rn(__fmul_rn(v.w, inv), g.w);
            quad_store_q8_lane<Q>(q8_1_quantize_lane(o), i, aq + m * aq_stride);
        };

        if ((int)blockDim.x >= VT && nvec <= KEEP * VT) // uniform
        {
            const int vt = threadIdx.x;
            float4 keep[M][KEEP], gk[KEEP];
            if (vt < VT) // whole wavefronts
            {
                // every load first (one branch around all loads of the delta), then the additions
                float4 dk[M][KEEP];
#pragma unroll
                for (int k = 0; k < KEEP; ++k)
                {
                    const int i = min(vt + k * VT, nvec - 1);
                    gk[k] = g4[i];
#pragma unroll
                    for (int m = 0; m < M; ++m)
                        keep[m][k] = reinterpret_cast<const float4 *>(qa.x + (size_t)m * qa.ldx)[i];
                }
                if (qa.x2) // uniform
                {
#pragma unroll
                    for (int k = 0; k < KEEP; ++k)
#pragma unroll
                        for (int m = 0; m < M; ++m)
                            dk[m][k] = reinterpret_cast<const float4 *>(qa.x2 + (size_t)m * qa.ldx)[min(vt + k * VT, nvec - 1)];
#pragma unroll
                    for (int k = 0; k < KEEP; ++k)
#pragma unroll
                        for (int m = 0; m < M; ++m)
                            keep[m][k] = add4(keep[m][k], dk[m][k]);
                }
#pragma unroll
                for (int m = 0; m < M; ++m)
                {
                    double acc = 0.0;
#pragma unroll
                    for (int k = 0; k < KEEP; ++k)
                        if (vt + k * VT < nvec)
                        {
                            if (writer)
                                reinterpret_cast<float4 *>(qa.x_out + (size_t)m * qa.ldx)[vt + k * VT] = keep[m][k];
                            square(acc, keep[m][k]);
                        }
                    acc = butterfly(acc);
                    if ((vt & (WAVE - 1)) == 0)
                        s_part[m * 8 + (vt >> 6)] = acc;
                }
            }
            __syncthreads();
            if (vt < VT)
            {
#pragma unroll
                for (int m = 0; m < M; ++m)
                {
                    const float inv = inverse_rms(m);
#pragma unroll
                    for (int k = 0; k < KEEP; ++k)
                        if (vt + k * VT < nvec) // whole 8-thread groups stay together (nvec is a multiple of 64)
                            emit(m, vt + k * VT, keep[m][k], gk[k], inv);
                }
            }
            return;
        }

#pragma unroll
        for (int m = 0; m < M; ++m)
            for (int vt = threadIdx.x; vt < VT; vt += (int)blockDim.x) // uniform per wavefront
            {
                double acc = 0.0;
                for (int i = vt; i < nvec; i += VT)
                {
                    const float4 v = row_value(m, i);
                    if (writer)
                        reinterpret_cast<float4 *>(qa.x_out + (size_t)m * qa.ldx)[i] = v;
                    square(acc, v);
                }
                acc = butterfly(acc);
                if ((vt & (WAVE - 1)) == 0)
                    s_part[m * 8 + (vt >> 6)] = acc;
            }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < M; ++m)
        {
            const float inv = inverse_rms(m);
            for (int i = threadIdx.x; i < nvec; i += (int)blockDim.x) // whole 8-thread groups stay together
                emit(m, i, row_value(m, i), g4[i], inv);
        }
    }

    // 32 rows of one half of a super-block, raw, by way of LDS: what the quad lanes 2 half and 2 half + 1 of every row decode.
    // A load of 16 bytes a lane reads a row's piece of a plane with neighbouring lanes (four cover 64 bytes), where a lane that
    // loads for itself meets a cache line of its own: 16 or 32 instead of 64 cycles of the address unit.  A piece lies in LDS where
    // eight lanes that read eight neighbouring rows meet no bank twice.
    // PIECES: 16-byte pieces of a row
    template <int PIECES>
    struct HalfRows
    {
        static constexpr int ROWS = 64 / PIECES < 32 ? 64 / PIECES : 32; // of a load
        static constexpr int LOADS = 32 / ROWS, BYTES = 32 * PIECES * 16;
        static constexpr uint64_t LANES = ROWS * PIECES == 64 ? ~0ull : (1ull << (ROWS * PIECES)) - 1;
        __device__ __forceinline__ static int place(int row, int piece)
        {
            return PIECES == 4 ? piece ^ ((row >> 1) & 3) : PIECES == 2 ? piece ^ ((row >> 2) & 1) : piece;
        }
        // row_of(r): where row r's pieces start, in bytes from the base that the load is given
        template <class R>
        __device__ __forceinline__ static void offsets(uint32_t (&from)[LOADS], int lane, R row_of)
        {
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
            {
                const int row = (i * ROWS + lane / PIECES) & 31;
                from[i] = row_of(row) + 16u * (uint32_t)place(row, lane % PIECES);
            }
        }
        // to: LDS address (uniform).  (m0 is written a wait state before the load that reads it: the compiler inserts none here)
        __device__ __forceinline__ static void load(uint32_t to, const uint32_t (&from)[LOADS], const uint8_t *base)
        {
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                if (LANES == ~0ull)
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to + (uint32_t)(i * 1024)), "v"(from[i]), "s"(base) : "memory");
                else
                    asm volatile("s_mov_b32 m0, %0\n\ts_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b64 exec, -1"
                                 ::"s"(to + (uint32_t)(i * 1024)), "v"(from[i]), "s"(base), "s"(LANES) : "memory");
        }
        template <class V>
        __device__ __forceinline__ static V read(const uint8_t *at, int row, int piece, int byte = 0)
        {
            return *reinterpret_cast<const V *>(at + (row * PIECES + place(row, piece)) * 16 + byte);
        }
    };

    // ---- Q4_K ------------------------------------------------------------------------
    // Super-block = 144 bytes: header piece {d, dmin, scales[12]} and four 32-byte groups;
    // group l holds blocks 2l (low nibbles) and 2l+1 (high nibbles), element e in byte e
    // (Q4_KTensor.cpp:768-792).  Effective scale f16(d*sc), min f16(-dmin*m) with the
    // packer's fp16 rounding (Q4_KTensor.cpp:794-799, FP16Utils.h:75-118).
    struct Q4KQuad
    {
        static constexpr int SB_BYTES = 144;
        static constexpr int STATIC_LDS = 0;     // bytes of static LDS (decode tables) beside the activations
        // wavefronts per compute unit the launch shape may use in one round; with 16 the shape
        // search also avoids a lone wavefront per SIMD unit (measured on 5120 x 8192: 7.5 us with
        // seven wavefronts per compute unit against 8.2 us with four)
        static constexpr int RESIDENT_WAVES = 16;
        __device__ __forceinline__ static void stage() {}
        // decode tables fetched ahead of dependent loads (formats that have tables): none here
        struct TablesRaw
        {
        };
        static constexpr int TABLE_THREADS = 0;
        __device__ __forceinline__ static void tables_issue(TablesRaw &) {}
        template <int NEWER>
        __device__ __forceinline__ static void tables_wait(TablesRaw &) {}
        __device__ __forceinline__ static void tables_store(const TablesRaw &) {}
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        // workgroup size bound: one activation row leaves room for 16 wavefronts of 128 registers
        static constexpr int max_threads(int M) { return M == 1 ? 1024 : 512; }
        // whether this matrix can be addressed by the kernel at all: super-block indices are 24-bit
        // multiplicands, byte offsets from the matrix's base 32-bit
        static bool addressable(long N, int SB) { return (double)N * SB < 16777216.0; }
        // lane l decodes blocks 2l (first) and 2l+1 (second)
        __device__ __forceinline__ static void owner(int j, int &l, int &which)
        {
            l = j >> 1;
            which = j & 1;
        }
        __device__ __forceinline__ static int block_of(int l, int which) { return 2 * l + which; }

        struct Raw
        {
            v4i head, qa, qb;
        };
        static constexpr int LOADS = 3; // vector memory loads per Raw
        struct Lane
        {
            uint32_t sel, m1, m2, m3;
            int byte_off; // of this lane's group inside the super-block
        };
        struct Scale
        {
            h2 s; // {b_scale of block 2l, of block 2l+1}
            h2 m; // {|b_min| ...}
        };

        __device__ __forceinline__ static Lane lane_consts(int l)
        {
            Lane c;
            const uint32_t h = (uint32_t)(l & 1);
            // bytes {2h, zero, 2h+1, zero} of a dword
            c.sel = (2u * h) | (0x0Cu << 8) | ((2u * h + 1u) << 16) | (0x0Cu << 24);
            c.m1 = (l < 2) ? 0x003F003Fu : 0u;
            c.m2 = (l < 2) ? 0u : 0x00300030u;
            c.m3 = (l < 2) ? 0u : 0x000F000Fu;
            c.byte_off = 16 + 32 * l;
            return c;
        }

        // Where a lane reads: its current super-block, and the one it reads instead once it
        // is past the end of its run (its last valid one, still in the caches): loads are
        // never predicated, a load under a lane mask would be waited for at once.
        // The cursor is a super-block index; addresses are the matrix's base (uniform, in scalar
        // registers) plus a 32-bit byte offset per lane: one multiply-add per load address where
        // 64-bit pointers per lane took six vector instructions a step to move and select.
        struct Cursor
        {
            const uint8_t *base; // uniform
            uint32_t t, first;
        };
        __device__ __forceinline__ static Cursor cursor(const GemvArgs &a, size_t t, size_t t_safe, const Lane &)
        {
            Cursor c;
            c.base = static_cast<const uint8_t *>(a.w);
            c.t = (uint32_t)t;
            c.first = (uint32_t)t_safe;
            return c;
        }
        // What a lane's position moves by from one step to the next (uniform), in super-blocks: the
        // step's, and `jump` more when the lane's next super-block lies in the next row.
        struct Stride
        {
            uint32_t plain, cross;
        };
        __device__ __forceinline__ static Stride stride(uint32_t jump)
        {
            Stride st;
            st.plain = (uint32_t)QUAD_STEP_SB;
            st.cross = (uint32_t)QUAD_STEP_SB + jump;
            return st;
        }
        __device__ __forceinline__ static void next(Cursor &c, bool cross, const Stride &st)
        {
            c.t += cross ? st.cross : st.plain;
        }
        __device__ __forceinline__ static void load(Raw &r, const Cursor &c, const Lane &lc, bool valid)
        {
            load_index(r, c, lc, valid ? c.t : c.first);
        }
        // super-block sb_off after the cursor's
        __device__ __forceinline__ static void load_at(Raw &r, const Cursor &c, const Lane &lc, int sb_off)
        {
            load_index(r, c, lc, c.t + (uint32_t)sb_off);
        }
        // The loads are issued as assembly so that the kernel, not the compiler, decides where
        // they are waited for (wait() below); the compiler would wait right after issue.
        __device__ __forceinline__ static void load_index(Raw &r, const Cursor &c, const Lane &lc, uint32_t t)
        {
            const uint32_t osb = __umul24(t, (uint32_t)SB_BYTES);
            const uint32_t ogrp = __umul24(t, (uint32_t)SB_BYTES) + (uint32_t)lc.byte_off;
            asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(r.head) : "v"(osb), "s"(c.base));
            asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(r.qa) : "v"(ogrp), "s"(c.base));
            asm volatile("global_load_dwordx4 %0, %1, %2 offset:16" : "=&v"(r.qb) : "v"(ogrp), "s"(c.base));
        }
        // (HalfRows: a row's header, and the 64 bytes of two groups)
        struct Half
        {
            typedef HalfRows<1> Head;
            typedef HalfRows<4> Group;
            static constexpr int BYTES = Head::BYTES + Group::BYTES;
            uint32_t head[Head::LOADS], group[Group::LOADS];
            const uint8_t *base;
            __device__ __forceinline__ void init(const GemvArgs &a, long n0, int half, int lane)
            {
                base = uniform_base(static_cast<const uint8_t *>(a.w));
                const auto row = [&](int r) { return (uint32_t)(n0 + r < a.N ? n0 + r : a.N - 1) * (uint32_t)(a.SB * SB_BYTES); };
                Head::offsets(head, lane, row);
                Group::offsets(group, lane, [&](int r) { return row(r) + 16u + 64u * (uint32_t)half; });
            }
            __device__ __forceinline__ void load(uint32_t to, int sb) const
            {
                Head::load(to, head, base + (size_t)sb * SB_BYTES);
                Group::load(to + Head::BYTES, group, base + (size_t)sb * SB_BYTES);
            }
            // what lane (row, l & 1) of them decodes
            __device__ __forceinline__ static void read(Raw &r, const uint8_t *at, int row, int odd)
            {
                r.head = Head::read<v4i>(at, row, 0);
                r.qa = Group::read<v4i>(at + Head::BYTES, row, 2 * odd);
                r.qb = Group::read<v4i>(at + Head::BYTES, row, 2 * odd + 1);
            }
        };
        // Marks r's registers as in use up to this point (emits nothing).
        __device__ __forceinline__ static void keep(Raw &r)
        {
            asm volatile("" : "+v"(r.head), "+v"(r.qa), "+v"(r.qb));
        }
        // Until at most `newer` vector memory operations issued after r's loads are pending.
        template <int NEWER>
        __device__ __forceinline__ static void wait(Raw &r)
        {
            asm volatile("s_waitcnt vmcnt(%3)" : "+v"(r.head), "+v"(r.qa), "+v"(r.qb) : "n"(NEWER));
        }

        __device__ __forceinline__ static uint16_t f16_trunc_bits(float x)
        {
            const uint32_t mag = (uint32_t)truncf(fabsf(x) * 16777216.0f);
            return (uint16_t)(mag | ((__float_as_uint(x) >> 16) & 0x8000u));
        }

        // w[0], w[1]: elements 0-15, 16-31 of block 2l; w[2], w[3]: of block 2l+1.
        __device__ __forceinline__ static void decode(const Raw &r, const Lane &c, v4i (&w)[4], Scale &S)
        {
            const uint32_t k = 0x0F0F0F0Fu;
            w[0] = (v4i){(int)((uint32_t)r.qa.x & k), (int)((uint32_t)r.qa.y & k), (int)((uint32_t)r.qa.z & k), (int)((uint32_t)r.qa.w & k)};
            w[1] = (v4i){(int)((uint32_t)r.qb.x & k), (int)((uint32_t)r.qb.y & k), (int)((uint32_t)r.qb.z & k), (int)((uint32_t)r.qb.w & k)};
            w[2] = (v4i){(int)(((uint32_t)r.qa.x >> 4) & k), (int)(((uint32_t)r.qa.y >> 4) & k),
                         (int)(((uint32_t)r.qa.z >> 4) & k), (int)(((uint32_t)r.qa.w >> 4) & k)};
            w[3] = (v4i){(int)(((uint32_t)r.qb.x >> 4) & k), (int)(((uint32_t)r.qb.y >> 4) & k),
                         (int)(((uint32_t)r.qb.z >> 4) & k), (int)(((uint32_t)r.qb.w >> 4) & k)};
            decode_scales(r.head, c, S);
        }

        // Effective scales and mins of blocks 2l, 2l+1 from the header piece: the 6-bit
        // scales / mins as two 16-bit integers each
        // (get_scale_min_k4: j<4: q[j]&63, q[j+4]&63; else (q[j+4]&15)|((q[j-4]>>6)<<4),
        // (q[j+4]>>4)|((q[j]>>6)<<4) -- SIMDHelpers.h:10791-10803)
        __device__ __forceinline__ static void decode_scales(const v4i &head, const Lane &c, Scale &S)
        {
            const uint32_t A = __builtin_amdgcn_perm(0u, (uint32_t)head.y, c.sel);
            const uint32_t B = __builtin_amdgcn_perm(0u, (uint32_t)head.z, c.sel);
            const uint32_t P = __builtin_amdgcn_perm(0u, (uint32_t)head.w, c.sel);
            const uint32_t bias = 0x64006400u; // fp16 1024.0: 0x6400|n is 1024+n
            const uint32_t sc = (P & c.m3) | (((A >> 2) & c.m2) | ((A & c.m1) | bias));
            const uint32_t mn = ((P >> 4) & c.m3) | (((B >> 2) & c.m2) | ((B & c.m1) | bias));
            const h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
            const h2 scf = __builtin_bit_cast(h2, sc) - k1024;
            const h2 mnf = __builtin_bit_cast(h2, mn) - k1024;
            const uint32_t hx = (uint32_t)head.x;
            const h2 dd = __builtin_bit_cast(h2, hx); // {d, dmin}
            // d (11-bit significand) times a 6-bit integer is exact before rounding, so the
            // fp16 multiply equals f16(fp32 product) wherever the result is normal
            S.s = (h2){dd.x, dd.x} * scf;
            S.m = (h2){dd.y, dd.y} * mnf;
            const uint32_t e = hx & 0x7C007C00u;
            if (__builtin_expect(((e - 0x08000800u) & 0x80008000u) != 0u, 0))
            {
                // d or dmin below 2^-13: results may be fp16-subnormal, which the packer truncates
                const float d = (float)dd.x, dmin = (float)dd.y;
                uint32_t sb = __builtin_bit_cast(uint32_t, S.s), mb = __builtin_bit_cast(uint32_t, S.m);
                const float s0 = d * (float)(sc & 0x3Fu), s1 = d * (float)((sc >> 16) & 0x3Fu);
                const float m0 = dmin * (float)(mn & 0x3Fu), m1 = dmin * (float)((mn >> 16) & 0x3Fu);
                if (fabsf(s0) < 6.103515625e-05f)
                    sb = (sb & 0xFFFF0000u) | f16_trunc_bits(s0);
                if (fabsf(s1) < 6.103515625e-05f)
                    sb = (sb & 0x0000FFFFu) | ((uint32_t)f16_trunc_bits(s1) << 16);
                if (fabsf(m0) < 6.103515625e-05f)
                    mb = (mb & 0xFFFF0000u) | f16_trunc_bits(m0);
                if (fabsf(m1) < 6.103515625e-05f)
                    mb = (mb & 0x0000FFFFu) | ((uint32_t)f16_trunc_bits(m1) << 16);
                S.s = __builtin_bit_cast(h2, sb);
                S.m = __builtin_bit_cast(h2, mb);
            }
        }

        // effective scale / min (fp32 value of the fp16 the packer stores) of block 2l+i
        __device__ __forceinline__ static float scale_f32(const Scale &S, int i) { return i ? (float)S.s.y : (float)S.s.x; }
        __device__ __forceinline__ static float min_f32(const Scale &S, int i) { return i ? -(float)S.m.y : -(float)S.m.x; }

        // contribution of the lane's two blocks, added onto acc
        __device__ __forceinline__ static float apply(const Scale &S, int idot0, int idot1, const float4 sd, float acc)
        {
            // sd = {d0, sum0*d0, d1, sum1*d1}
            const float cs0 = fmaf(sd.x, (float)S.s.x, 0.0f);
            const float cs1 = fmaf(sd.z, (float)S.s.y, 0.0f);
            acc = fmaf((float)idot0, cs0, acc);
            acc = fmaf(sd.y, -(float)S.m.x, acc);
            acc = fmaf((float)idot1, cs1, acc);
            acc = fmaf(sd.w, -(float)S.m.y, acc);
            return acc;
        }
    };

    // ---- Q6_K ------------------------------------------------------------------------
    // Device layout: planes ql [T][128], qh [T][64], scales [T][16], d [T] over T = N*K/256
    // super-blocks.  Quad lane l = 2n + h works on half n of the super-block: its 32 ql
    // bytes 64n+32h.. hold block 4n+h in the low and block 4n+2+h in the high nibbles, the
    // 32 qh bytes 32n.. their upper two bits at bit offsets 2h and 2h+4.  Each block is
    // requantised to int8 as the reference's packer does (SIMDHelpers.h:12023-12204):
    //   msc = max(|sc0|,|sc1|) ; f_i = rne(sc_i*127*256 / (msc*32)) ; w = ((q-32)*f_i + 128) >> 8
    //   b_scale = f16(d*msc*32/127)
    // The half whose |sc| equals msc has f = +-1016 exactly, so one division per block
    // suffices.  Weight addresses are 32-bit offsets from the plane bases.
    struct Q6KQuad
    {
        typedef unsigned short v2s __attribute__((ext_vector_type(2)));
        typedef int v2i_ __attribute__((ext_vector_type(2)));
        static constexpr int LOADS = 5;
        static constexpr int STATIC_LDS = 0;
        // arithmetic keeps a lone wavefront per SIMD unit busy here (5120 x 25600: 24.3 us with four
        // wavefronts per compute unit, 25.7 with seven)
        static constexpr int RESIDENT_WAVES = 8;
        __device__ __forceinline__ static void stage() {}
        // decode tables fetched ahead of dependent loads (formats that have tables): none here
        struct TablesRaw
        {
        };
        static constexpr int TABLE_THREADS = 0;
        __device__ __forceinline__ static void tables_issue(TablesRaw &) {}
        template <int NEWER>
        __device__ __forceinline__ static void tables_wait(TablesRaw &) {}
        __device__ __forceinline__ static void tables_store(const TablesRaw &) {}
        static constexpr int max_threads(int M) { return M == 1 ? 1024 : 512; }
        static bool addressable(long N, int SB) { return (double)N * SB * 128.0 < 4.0e9; }

        struct Raw
        {
            v4i qla, qlb, qha, qhb;
            v2i_ fc; // the factor records of the lane's two blocks (q6k_block_code)
        };
        struct Lane
        {
            uint32_t ql_off, qh_off, fc_off; // byte offsets of this lane inside a super-block's planes
            uint32_t hshift;                 // 2h: bit offset of the low-nibble block's upper bits
        };
        struct Scale
        {
            float bs0, bs1;
        };
        struct Cursor
        {
            const uint8_t *ql, *qh, *fc; // plane bases (uniform)
            uint32_t t, first;               // this lane's super-block index: current, and the one
                                             // read instead past the end of the run
        };

        __device__ __forceinline__ static Lane lane_consts(int l)
        {
            Lane c;
            const uint32_t n = (uint32_t)l >> 1, h = (uint32_t)l & 1u;
            c.ql_off = 64u * n + 32u * h;
            c.qh_off = 32u * n;
            c.fc_off = 8u * (uint32_t)l; // records of blocks 4n+h and 4n+2+h are neighbours
            c.hshift = 2u * h;
            return c;
        }
        // block j = 4n + sub: lane 2n + (sub & 1), its first (sub < 2) or second block
        __device__ __forceinline__ static void owner(int j, int &l, int &which)
        {
            l = 2 * (j >> 2) + (j & 1);
            which = (j >> 1) & 1;
        }
        __device__ __forceinline__ static Cursor cursor(const GemvArgs &a, size_t t, size_t t_safe, const Lane &)
        {
            const size_t T = (size_t)a.N * a.SB;
            Cursor c;
            c.ql = static_cast<const uint8_t *>(a.w);
            c.qh = c.ql + T * 128;
            c.fc = c.ql + q6k_factors_offset(T);
            c.t = (uint32_t)t;
            c.first = (uint32_t)t_safe;
            return c;
        }
        // super-blocks a lane moves by per step, without and with a row crossing (Q4KQuad::Stride)
        struct Stride
        {
            uint32_t plain, cross;
        };
        __device__ __forceinline__ static Stride stride(uint32_t jump)
        {
            Stride st;
            st.plain = (uint32_t)QUAD_STEP_SB;
            st.cross = (uint32_t)QUAD_STEP_SB + jump;
            return st;
        }
        __device__ __forceinline__ static void next(Cursor &c, bool cross, const Stride &st)
        {
            c.t += cross ? st.cross : st.plain;
        }
        __device__ __forceinline__ static int block_of(int l, int which) { return 4 * (l >> 1) + (l & 1) + 2 * which; }

        __device__ __forceinline__ static void load(Raw &r, const Cursor &c, const Lane &lc, bool valid)
        {
            load_index(r, c, lc, valid ? c.t : c.first);
        }
        __device__ __forceinline__ static void load_at(Raw &r, const Cursor &c, const Lane &lc, int sb_off)
        {
            load_index(r, c, lc, c.t + (uint32_t)sb_off);
        }
        // Loads issued as assembly so that the kernel decides where they are waited for.
        __device__ __forceinline__ static void load_index(Raw &r, const Cursor &c, const Lane &lc, uint32_t t)
        {
            const uint32_t oql = t * 128u + lc.ql_off, oqh = t * 64u + lc.qh_off, ofc = t * 32u + lc.fc_off;
            asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(r.qla) : "v"(oql), "s"(c.ql));
            asm volatile("global_load_dwordx4 %0, %1, %2 offset:16" : "=&v"(r.qlb) : "v"(oql), "s"(c.ql));
            asm volatile("global_load_dwordx4 %0, %1, %2" : "=&v"(r.qha) : "v"(oqh), "s"(c.qh));
            asm volatile("global_load_dwordx4 %0, %1, %2 offset:16" : "=&v"(r.qhb) : "v"(oqh), "s"(c.qh));
            asm volatile("global_load_dwordx2 %0, %1, %2" : "=&v"(r.fc) : "v"(ofc), "s"(c.fc));
        }
        // (HalfRows: 64 bytes of low bits, 32 of upper bits, four factor records)
        struct Half
        {
            typedef HalfRows<4> Low;
            typedef HalfRows<2> Upper;
            typedef HalfRows<1> Factors;
            static constexpr int BYTES = Low::BYTES + Upper::BYTES + Factors::BYTES;
            uint32_t low[Low::LOADS], upper[Upper::LOADS], factors[Factors::LOADS];
            const uint8_t *ql, *qh, *fc;
            __device__ __forceinline__ void init(const GemvArgs &a, long n0, int half, int lane)
            {
                const size_t T = (size_t)a.N * a.SB;
                ql = uniform_base(static_cast<const uint8_t *>(a.w));
                qh = ql + T * 128;
                fc = ql + q6k_factors_offset(T);
                const auto row = [&](int r) { return (uint32_t)(n0 + r < a.N ? n0 + r : a.N - 1) * (uint32_t)a.SB; };
                Low::offsets(low, lane, [&](int r) { return row(r) * 128u + 64u * (uint32_t)half; });
                Upper::offsets(upper, lane, [&](int r) { return row(r) * 64u + 32u * (uint32_t)half; });
                Factors::offsets(factors, lane, [&](int r) { return row(r) * 32u + 16u * (uint32_t)half; });
            }
            __device__ __forceinline__ void load(uint32_t to, int sb) const
            {
                Low::load(to, low, ql + (size_t)sb * 128);
                Upper::load(to + Low::BYTES, upper, qh + (size_t)sb * 64);
                Factors::load(to + Low::BYTES + Upper::BYTES, factors, fc + (size_t)sb * 32);
            }
            __device__ __forceinline__ static void read(Raw &r, const uint8_t *at, int row, int odd)
            {
                r.qla = Low::read<v4i>(at, row, 2 * odd);
                r.qlb = Low::read<v4i>(at, row, 2 * odd + 1);
                r.qha = Upper::read<v4i>(at + Low::BYTES, row, 0);
                r.qhb = Upper::read<v4i>(at + Low::BYTES, row, 1);
                r.fc = Factors::read<v2i_>(at + Low::BYTES + Upper::BYTES, row, 0, 8 * odd);
            }
        };
        __device__ __forceinline__ static void keep(Raw &r)
        {
            asm volatile("" : "+v"(r.qla), "+v"(r.qlb), "+v"(r.qha), "+v"(r.qhb), "+v"(r.fc));
        }
        template <int NEWER>
        __device__ __forceinline__ static void wait(Raw &r)
        {
            asm volatile("s_waitcnt vmcnt(%5)"
                         : "+v"(r.qla), "+v"(r.qlb), "+v"(r.qha), "+v"(r.qhb), "+v"(r.fc)
                         : "n"(NEWER));
        }

        // ((q-32)*f + 128) >> 8 on four 6-bit values packed in the bytes of q: in wrapping
        // 16-bit arithmetic q*f + (128 - 32 f) is exact (|value| < 2^15 for |f| <= 1016) and
        // ">> 8, keep the low byte" is "take the high byte".
        __device__ __forceinline__ static int requant4(uint32_t q, v2s ff, v2s cc)
        {
            // bytes 0, 2 and bytes 1, 3 of q, each widened to 16 bits: one byte permute apiece
            const uint32_t e = __builtin_amdgcn_perm(0u, q, 0x0C020C00u);
            const uint32_t o = __builtin_amdgcn_perm(0u, q, 0x0C030C01u);
            const v2s re = __builtin_bit_cast(v2s, e) * ff + cc;
            const v2s ro = __builtin_bit_cast(v2s, o) * ff + cc;
            return (int)__builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, ro), __builtin_bit_cast(uint32_t, re),
                                              0x07030501u);
        }

        // The two 8.8 factors (with their constants 128 - 32 f, each doubled into a packed pair)
        // and the scale of one block from its record.
        __device__ __forceinline__ static void block_factors(uint32_t code, v2s &f0, v2s &c0, v2s &f1, v2s &c1,
                                                             float &bscale)
        {
            int fi0, fi1;
            q6k_block_decode(code, fi0, fi1, bscale);
            const unsigned short u0 = (unsigned short)fi0, u1 = (unsigned short)fi1;
            const unsigned short k0 = (unsigned short)(128 - 32 * fi0), k1 = (unsigned short)(128 - 32 * fi1);
            f0 = (v2s){u0, u0};
            c0 = (v2s){k0, k0};
            f1 = (v2s){u1, u1};
            c1 = (v2s){k1, k1};
        }

        // w[0], w[1]: elements 0-15, 16-31 of block 4n+h; w[2], w[3]: of block 4n+2+h.
        __device__ __forceinline__ static void decode(const Raw &r, const Lane &lc, v4i (&w)[4], Scale &S)
        {
            v2s fA0, cA0, fA1, cA1, fB0, cB0, fB1, cB1;
            block_factors((uint32_t)r.fc.x, fA0, cA0, fA1, cA1, S.bs0);
            block_factors((uint32_t)r.fc.y, fB0, cB0, fB1, cB1, S.bs1);

            const uint32_t k4 = 0x0F0F0F0Fu, k2 = 0x03030303u;
            auto pair = [&](uint32_t ql, uint32_t qh, v2s fa, v2s ca, v2s fb, v2s cb, int &wa, int &wb) {
                const uint32_t hs = qh >> lc.hshift;
                const uint32_t qa = (ql & k4) | ((hs & k2) << 4);
                const uint32_t qb = ((ql >> 4) & k4) | (((hs >> 4) & k2) << 4);
                wa = requant4(qa, fa, ca); // f == 0 (msc == 0) yields 0 bytes
                wb = requant4(qb, fb, cb);
            };
            // dwords 0-3 are elements 0-15 (first sub-scale), dwords 4-7 elements 16-31
            int a0[4], b0[4], a1[4], b1[4];
            pair((uint32_t)r.qla.x, (uint32_t)r.qha.x, fA0, cA0, fB0, cB0, a0[0], b0[0]);
            pair((uint32_t)r.qla.y, (uint32_t)r.qha.y, fA0, cA0, fB0, cB0, a0[1], b0[1]);
            pair((uint32_t)r.qla.z, (uint32_t)r.qha.z, fA0, cA0, fB0, cB0, a0[2], b0[2]);
            pair((uint32_t)r.qla.w, (uint32_t)r.qha.w, fA0, cA0, fB0, cB0, a0[3], b0[3]);
            pair((uint32_t)r.qlb.x, (uint32_t)r.qhb.x, fA1, cA1, fB1, cB1, a1[0], b1[0]);
            pair((uint32_t)r.qlb.y, (uint32_t)r.qhb.y, fA1, cA1, fB1, cB1, a1[1], b1[1]);
            pair((uint32_t)r.qlb.z, (uint32_t)r.qhb.z, fA1, cA1, fB1, cB1, a1[2], b1[2]);
            pair((uint32_t)r.qlb.w, (uint32_t)r.qhb.w, fA1, cA1, fB1, cB1, a1[3], b1[3]);
            w[0] = (v4i){a0[0], a0[1], a0[2], a0[3]};
            w[1] = (v4i){a1[0], a1[1], a1[2], a1[3]};
            w[2] = (v4i){b0[0], b0[1], b0[2], b0[3]};
            w[3] = (v4i){b1[0], b1[1], b1[2], b1[3]};
        }

        __device__ __forceinline__ static float scale_f32(const Scale &S, int i) { return i ? S.bs1 : S.bs0; }
        __device__ __forceinline__ static float min_f32(const Scale &, int) { return 0.0f; }

        // the reference's mins plane is all zero for Q6_K
        __device__ __forceinline__ static float apply(const Scale &S, int idot0, int idot1, const float4 sd, float acc)
        {
            acc = fmaf((float)idot0, sd.x * S.bs0, acc);
            acc = fmaf((float)idot1, sd.z * S.bs1, acc);
            return acc;
        }
    };

    // ---- kernel ----------------------------------------------------------------------

    template <class Q, int M, int U>
    __device__ __forceinline__ void quad_compute_step(const typename Q::Raw &r, const typename Q::Lane &lc,
                                                      const uint8_t *aq_lane, const uint8_t *ads_lane, int aq_stride,
                                                      int ads_stride, float (&t)[M], int (&idot)[M][2])
    {
        v4i w[4];
        typename Q::Scale S;
        Q::decode(r, lc, w, S);
#pragma unroll
        for (int m = 0; m < M; ++m)
        {
            const uint8_t *ap = aq_lane + m * aq_stride;
            const v4i a0 = *reinterpret_cast<const v4i *>(ap);
            const v4i a1 = *reinterpret_cast<const v4i *>(ap + 64);
            const v4i a2 = *reinterpret_cast<const v4i *>(ap + 128);
            const v4i a3 = *reinterpret_cast<const v4i *>(ap + 192);
            const float4 sd = *reinterpret_cast<const float4 *>(ap + 256);
            idot[m][0] = dot16(a1, w[1], dot16z(a0, w[0]));
            idot[m][1] = dot16(a3, w[3], dot16z(a2, w[2]));
            t[m] = Q::apply(S, idot[m][0], idot[m][1], sd, 0.0f);
        }
    }

    // Wait for step u of a chunk whose successor chunk has been issued after it.
    template <class Q, int U>
    __device__ __forceinline__ void wait_for(typename Q::Raw &r, int u)
    {
        // The counts below are the loads issued after step u's: the rest of its chunk and the whole
        // next chunk.  They hold only while nothing else touches vmcnt in between, which the
        // build enforces by refusing kernels that spill (scratch traffic counts in vmcnt too,
        // and a spilled destination register of a load in flight is overwritten when it lands).
        static_assert(U >= 1 && U <= 4, "wait_for covers chunks of 1..4 steps");
        static_assert(Q::LOADS * (2 * U - 1) <= 63, "vmcnt is a 6-bit counter");
        // u is a compile-time constant after unrolling
        switch (u)
        {
        case 0: Q::template wait<Q::LOADS *(2 * U - 1)>(r); break;
        case 1: Q::template wait<Q::LOADS *(2 * U - 2)>(r); break;
        case 2: Q::template wait<Q::LOADS *(2 * U - 3 > 0 ? 2 * U - 3 : 0)>(r); break;
        case 3: Q::template wait<Q::LOADS *(2 * U - 4 > 0 ? 2 * U - 4 : 0)>(r); break;
        default: Q::template wait<0>(r); break;
        }
    }

    // which matrix the wavefront works on, and the first wavefront of that matrix
    // orders the LDS traffic of one wavefront as seen by the compiler; the hardware runs a
    // wavefront's LDS instructions in order, so no instruction is needed
    __device__ __forceinline__ void wave_lds_sync()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    __device__ __forceinline__ void quad_which(const QuadArgs &qa, int wid_all, int &p, int &w_first)
    {
        p = 0;
        w_first = 0;
#pragma unroll
        for (int i = 1; i < QUAD_MAX_PROJ; ++i)
            if (i < qa.nproj && wid_all >= qa.wave_begin[i])
            {
                p = i;
                w_first = qa.wave_begin[i];
            }
    }

    // MODE: QUAD_MODE_DUMP also stores the exact int32 block sums the lanes form (the parity hook of
    // the C-ABI) and no fp32 output; QUAD_MODE_RING reduces finished rows through the LDS ring;
    // everything else is the same code.
    constexpr int QUAD_MODE_PLAIN = 0, QUAD_MODE_DUMP = 1, QUAD_MODE_RING = 2;
    template <class Q, int M, int U, int SRC, int MODE = QUAD_MODE_PLAIN>
    __device__ __forceinline__ void quad_body(const QuadArgs &qa, uint8_t *quad_lds, int p, int w_first, int wid_all)
    {
        constexpr bool DUMP = MODE == QUAD_MODE_DUMP, DEFER = MODE == QUAD_MODE_RING;
        const int nsb = qa.SB;
        const int aq_stride = nsb * QUAD_SB_LDS;
        const int ads_stride = 0;
        uint8_t *aq = quad_lds;
        uint8_t *ads = quad_lds;

        const int lane = threadIdx.x & (WAVE - 1);
        const int l = lane & 3;
        const int grp = lane >> 2;
        const typename Q::Lane lc = Q::lane_consts(l);

        GemvArgs a; // the matrix, for the format's addressing
        a.w = qa.w[p];
        a.N = qa.N[p];
        a.SB = nsb;
        float *const y = qa.y[p];
        const int ldy = qa.ldy[p];
        const int R = qa.R[p];

        // Rows j, j + TW, .. of this wavefront, walked as ONE run of `total` super-blocks: position
        // s of the run is super-block s % nsb of the wavefront's row number s / nsb.
        const long TW = qa.TW[p];
        const long j = wid_all - w_first;
        const long with_more = (long)a.N - (long)qa.rows_min[p] * TW; // wavefronts that walk a row more
        const int nrows = j < TW ? qa.rows_min[p] + (j < with_more ? 1 : 0) : 0; // wavefronts past the last idle
        const int total = nrows * nsb;
        const int nsteps = (total + QUAD_STEP_SB - 1) / QUAD_STEP_SB;

        // this lane's first super-block; past the end of the run it re-reads its super-block of
        // the wavefront's last row (an idle wavefront: of row 0)
        const size_t t0 = (size_t)(nrows > 0 ? j : 0) * nsb + grp;
        const size_t t_safe = (size_t)(nrows > 0 ? j + (long)(nrows - 1) * TW : 0) * nsb + grp;
        typename Q::Cursor wc = Q::cursor(a, t0, t_safe, lc);
        const typename Q::Stride stride = Q::stride((uint32_t)((TW - 1) * nsb));
        int ld_step = 0;
        int ld_sbr = grp; // where in its row the lane's next load lies (grp < 16 <= nsb)
        auto load_chunk = [&](typename Q::Raw(&buf)[U]) {
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                Q::load(buf[u], wc, lc, (ld_step + u) * QUAD_STEP_SB + grp < total);
                ld_sbr += QUAD_STEP_SB;
                const bool cross = ld_sbr >= nsb; // the next step's super-block belongs to the next row
                ld_sbr -= cross ? nsb : 0;
                Q::next(wc, cross, stride);
            }
            ld_step += U;
        };

        typename Q::Raw bufA[U], bufB[U];
        if constexpr (SRC == QUAD_SRC_Q8)
        {
            // activations first (they return first), then two chunks of weights, which stay in
            // flight while the activations are staged
            const int total_blk = M * nsb * 8;
            QuadActRaw ar[QUAD_ACT_PASSES];
            quad_act_issue(ar, qa.q8, total_blk);
            load_chunk(bufA);
            load_chunk(bufB);
            quad_act_wait<2 * U * Q::LOADS>(ar);
            if (total_blk <= QUAD_ACT_PASSES * (int)blockDim.x) // uniform
                quad_act_store<Q>(ar, nsb, total_blk, aq, aq_stride);
            else
                quad_stage_q8<Q, M>(qa.q8, nsb, aq, ads, aq_stride, ads_stride); // more blocks than the prefetch holds
        }
        else
        {
            load_chunk(bufA); // two chunks in flight while the activations are quantised and staged
            load_chunk(bufB);
            if constexpr (SRC == QUAD_SRC_RMSNORM)
                quad_stage_rmsnorm<Q, M>(qa, nsb, aq, aq_stride, quad_lds);
            else
                quad_stage_f32<Q, M, SRC>(qa.x, qa.x2, qa.ldx, nsb, aq, ads, aq_stride, ads_stride);
        }
        Q::stage(); // the format's decode tables, if it has any
        __syncthreads();
        // the staging code above must not reuse the registers of the loads in flight
#pragma unroll
        for (int u = 0; u < U; ++u)
        {
            Q::keep(bufA[u]);
            Q::keep(bufB[u]);
        }

        float cur[M]; // this lane's share of the row being walked
#pragma unroll
        for (int m = 0; m < M; ++m)
            cur[m] = 0.0f;

        int first = 0;  // super-block (inside its row) that lane group 0 handles in this step
        int row = 0;    // row `cur` belongs to, counted along the run: row j + row * TW of the matrix
        int step = 0;

        float *ring = reinterpret_cast<float *>(quad_lds + (size_t)M * aq_stride) +
                      (size_t)(threadIdx.x >> 6) * (QUAD_RING_ROWS * QUAD_RING_STRIDE * M);
        int slot = 0; // parked rows: row - slot .. row - 1
        // accumulate: what y holds for this lane's row of the (only) flush, requested now and long
        // there by the time the run ends
        float held[M];
#pragma unroll
        for (int m = 0; m < M; ++m)
            held[m] = 0.0f;
        if constexpr (DEFER)
        {
            if (qa.accumulate && (lane >> 2) < nrows)
            {
#pragma unroll
                for (int m = 0; m < M; ++m)
                    held[m] = y[(size_t)m * ldy + (size_t)(j + (long)(lane >> 2) * TW)];
            }
        }
        auto flush_ring = [&]() {
            wave_lds_sync(); // the wavefront's writes are in the ring (its LDS instructions run in order)
            const int r = lane >> 2, q = lane & 3;
#pragma unroll
            for (int m = 0; m < M; ++m)
            {
                const float4 *src = reinterpret_cast<const float4 *>(ring + (r * M + m) * QUAD_RING_STRIDE + q * 16);
                const float4 v0 = src[0], v1 = src[1], v2 = src[2], v3 = src[3];
                float sum = ((v0.x + v0.y) + (v0.z + v0.w)) + ((v1.x + v1.y) + (v1.z + v1.w));
                sum += ((v2.x + v2.y) + (v2.z + v2.w)) + ((v3.x + v3.y) + (v3.z + v3.w));
                sum += dpp_f32<DPP_QUAD_XOR1>(sum);
                sum += dpp_f32<DPP_QUAD_XOR2>(sum);
                if (q == 0 && r < slot)
                    y[(size_t)m * ldy + (size_t)(j + (long)(row - slot + r) * TW)] = qa.accumulate ? held[m] + sum : sum;
            }
            wave_lds_sync(); // reads done before the ring is written again
            slot = 0;
        };

        auto compute_step = [&](const typename Q::Raw &r) {
            // super-block of this lane inside its row: (first + grp) mod nsb (first < nsb, grp < 16 <= nsb)
            const uint32_t x = (uint32_t)(first + grp);
            const uint32_t sbr = min(x, x - (uint32_t)nsb);
            const uint8_t *aq_lane = aq + sbr * QUAD_SB_LDS + (l << 4);
            float t[M];
            int idot[M][2]; // the lane's two exact block sums per activation row
            quad_compute_step<Q, M, U>(r, lc, aq_lane, aq_lane, aq_stride, ads_stride, t, idot);

            const int gb = nsb - first;                       // lane groups still in the current row
            const int ge = total - step * QUAD_STEP_SB;       // lane groups with data at all
            if constexpr (DUMP)
            {
                const long rr = j + (long)(grp < gb ? row : row + 1) * TW - qa.row0;
                if (grp < ge && rr >= 0 && rr < qa.nrows)
                {
#pragma unroll
                    for (int m = 0; m < M; ++m)
                    {
                        int32_t *dst = qa.sums + ((size_t)m * qa.nrows + (size_t)rr) * ((size_t)nsb * 8) + (size_t)sbr * 8;
                        dst[Q::block_of(l, 0)] = idot[m][0];
                        dst[Q::block_of(l, 1)] = idot[m][1];
                    }
                }
            }
            if (ge < QUAD_STEP_SB) // the last step of the run: lane groups past its end hold nothing
            {
#pragma unroll
                for (int m = 0; m < M; ++m)
                    t[m] = grp < ge ? t[m] : 0.0f;
            }
            if (gb <= QUAD_STEP_SB)
            {
                // the current row ends in this step: lane groups below gb finish it, the others
                // start the next one
                const bool fin = grp < gb;
                if constexpr (DEFER)
                {
#pragma unroll
                    for (int m = 0; m < M; ++m)
                    {
                        ring[(slot * M + m) * QUAD_RING_STRIDE + lane] = cur[m] + (fin ? t[m] : 0.0f);
                        cur[m] = fin ? 0.0f : t[m];
                    }
                    ++slot;
                    ++row;
                    if (slot == QUAD_RING_ROWS) // uniform
                        flush_ring();
                }
                else
                {
#pragma unroll
                    for (int m = 0; m < M; ++m)
                    {
                        const float tot = wave_sum(cur[m] + (fin ? t[m] : 0.0f));
                        if constexpr (!DUMP) // the block-sum variant has no fp32 output (y is null)
                        {
                            if (lane == 0)
                                y[(size_t)m * ldy + (size_t)(j + (long)row * TW)] = tot;
                        }
                        cur[m] = fin ? 0.0f : t[m];
                    }
                    ++row;
                }
                first = QUAD_STEP_SB - gb;
            }
            else
            {
#pragma unroll
                for (int m = 0; m < M; ++m)
                    cur[m] += t[m];
                first += QUAD_STEP_SB;
            }
            ++step;
        };

        // buf was loaded one chunk ago; the loads of the chunk after it (U steps) are in flight.
        // Every buffer is waited for, also when its step lies past the end of the run: a
        // register whose load is still in flight must not look free to the compiler.
        auto compute_chunk = [&](typename Q::Raw(&buf)[U]) {
#pragma unroll
            for (int u = 0; u < U; ++u)
            {
                wait_for<Q, U>(buf[u], u);
                if (step < nsteps) // uniform
                    compute_step(buf[u]);
            }
        };

        // Each buffer is reloaded (with the chunk two ahead) as soon as it has been consumed.
        // Loads are unconditional -- past the end of the run the lanes re-read their first
        // super-block: a load under a condition would need register copies that wait for
        // it straight away.
        for (int c0 = 0; c0 < nsteps; c0 += 2 * U)
        {
            compute_chunk(bufA);
            __builtin_amdgcn_sched_barrier(0); // keep the loads below the last use of their registers
            load_chunk(bufA);
            compute_chunk(bufB);
            __builtin_amdgcn_sched_barrier(0);
            load_chunk(bufB);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // loads issued past the end of the run
        if constexpr (DEFER)
        {
            if (slot > 0) // uniform
                flush_ring();
        }
    }

    template <class Q, int M, int U, int SRC, int MODE = QUAD_MODE_PLAIN>
    __global__ void __launch_bounds__(Q::max_threads(M)) gemv_quad_kernel(const QuadArgs qa)
    {
        extern __shared__ __attribute__((aligned(16))) uint8_t quad_lds[];
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const int wid_all = (int)blockIdx.x * (int)(blockDim.x >> 6) + wave;
        int p, w_first;
        quad_which(qa, wid_all, p, w_first);
        quad_body<Q, M, U, SRC, MODE>(qa, quad_lds, p, w_first, wid_all);
    }

    // Two formats in one launch (Q and K in Q4_K, V in Q6_K): whole workgroups belong to one
    // format, so the branch is uniform per workgroup.
    template <class QA, int UA, class QB, int UB, int M, int SRC, int MODE = QUAD_MODE_PLAIN>
    __global__ void __launch_bounds__(QA::max_threads(M) < QB::max_threads(M) ? QA::max_threads(M) : QB::max_threads(M))
        gemv_quad_dual_kernel(const QuadArgs qa)
    {
        extern __shared__ __attribute__((aligned(16))) uint8_t quad_lds[];
        const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const int wid_all = (int)blockIdx.x * (int)(blockDim.x >> 6) + wave;
        int p, w_first;
        quad_which(qa, wid_all, p, w_first);
        if (p < qa.first_b)
            quad_body<QA, M, UA, SRC, MODE>(qa, quad_lds, p, w_first, wid_all);
        else
            quad_body<QB, M, UB, SRC, MODE>(qa, quad_lds, p, w_first, wid_all);
    }

    template <class Q, int M, int U, int SRC, int MODE = QUAD_MODE_PLAIN>
    inline void gemv_quad_launch_mus(dim3 grid, dim3 block, size_t lds, hipStream_t st, const QuadArgs &a)
    {
        static LdsGrant grant;
        (void)allow_lds(grant, reinterpret_cast<const void *>(&gemv_quad_kernel<Q, M, U, SRC, MODE>),
                        QUAD_MAX_LDS - Q::STATIC_LDS);
        hipLaunchKernelGGL((gemv_quad_kernel<Q, M, U, SRC, MODE>), grid, block, lds, st, a);
    }

    // a.sums set: the block-sum variant of the same kernel (Q8_1 input only)
    template <class Q, int M, int U>
    inline void gemv_quad_launch_mu(int src, dim3 grid, dim3 block, size_t lds, hipStream_t st, const QuadArgs &a)
    {
        if (a.sums)
        {
            gemv_quad_launch_mus<Q, M, U, QUAD_SRC_Q8, QUAD_MODE_DUMP>(grid, block, lds, st, a);
            return;
        }
        // (the norm's staging holds a row's values and weights in registers across its barrier: with two
        // steps per load chunk as well a single row's kernel would spill, so gemv_quad_launch sends the
        // norm source to one step per chunk and the two-step instantiation does not exist)
        constexpr bool NORM = M <= QUAD_NORM_MAX_M && !(M == 1 && U == 2);
        if constexpr (M <= QUAD_RING_MAX_M)
        {
            if (a.ring)
            {
                if constexpr (NORM)
                    if (src == QUAD_SRC_RMSNORM)
                    {
                        gemv_quad_launch_mus<Q, M, U, QUAD_SRC_RMSNORM, QUAD_MODE_RING>(grid, block, lds, st, a);
                        return;
                    }
                switch (src)
                {
                case QUAD_SRC_F32: gemv_quad_launch_mus<Q, M, U, QUAD_SRC_F32, QUAD_MODE_RING>(grid, block, lds, st, a); break;
                case QUAD_SRC_SWIGLU: gemv_quad_launch_mus<Q, M, U, QUAD_SRC_SWIGLU, QUAD_MODE_RING>(grid, block, lds, st, a); break;
                default: gemv_quad_launch_mus<Q, M, U, QUAD_SRC_Q8, QUAD_MODE_RING>(grid, block, lds, st, a); break;
                }
                return;
            }
        }
        if constexpr (NORM)
            if (src == QUAD_SRC_RMSNORM)
            {
                gemv_quad_launch_mus<Q, M, U, QUAD_SRC_RMSNORM>(grid, block, lds, st, a);
                return;
            }
        switch (src)
        {
        case QUAD_SRC_F32: gemv_quad_launch_mus<Q, M, U, QUAD_SRC_F32>(grid, block, lds, st, a); break;
        case QUAD_SRC_SWIGLU: gemv_quad_launch_mus<Q, M, U, QUAD_SRC_SWIGLU>(grid, block, lds, st, a); break;
        default: gemv_quad_launch_mus<Q, M, U, QUAD_SRC_Q8>(grid, block, lds, st, a); break;
        }
    }

    // Steps per load chunk (two chunks are in flight).  Measured on 5120..25600-column matrices:
    // a single activation row is fastest with ONE step per chunk (4.6 KB in flight per wavefront;
    // deeper queues only lengthen the memory system's own queues) unless rows are long (64
    // super-blocks and more), where a wavefront holds few rows and two steps pay.
    constexpr int QUAD_LONG_ROW_SB = 64;

    template <class Q>
    inline void gemv_quad_launch(int M, int src, dim3 grid, dim3 block, size_t lds, hipStream_t st,
                                 const QuadArgs &a)
    {
        switch (M)
        {
        case 1:
            if (a.SB >= QUAD_LONG_ROW_SB && src != QUAD_SRC_RMSNORM)
                gemv_quad_launch_mu<Q, 1, 2>(src, grid, block, lds, st, a);
            else
                gemv_quad_launch_mu<Q, 1, 1>(src, grid, block, lds, st, a);
            break;
        case 2: gemv_quad_launch_mu<Q, 2, 2>(src, grid, block, lds, st, a); break;
        case 3: gemv_quad_launch_mu<Q, 3, 2>(src, grid, block, lds, st, a); break;
        case 4: gemv_quad_launch_mu<Q, 4, 2>(src, grid, block, lds, st, a); break;
        // (formats with many loads per step run out of registers at two steps per chunk)
        case 5: gemv_quad_launch_mu<Q, 5, Q::LOADS <= 3 ? 2 : 1>(src, grid, block, lds, st, a); break;
        case 6: gemv_quad_launch_mu<Q, 6, Q::LOADS <= 3 ? 2 : 1>(src, grid, block, lds, st, a); break;
        case 7: gemv_quad_launch_mu<Q, 7, Q::LOADS <= 3 ? 2 : 1>(src, grid, block, lds, st, a); break;
        default: gemv_quad_launch_mu<Q, 8, Q::LOADS <= 3 ? 2 : 1>(src, grid, block, lds, st, a); break;
        }
    }

    // steps per chunk the single-format launches use for a batch size
    template <class Q>
    constexpr int quad_unroll(int M)
    {
        return M == 1 ? 1 : M <= 4 ? 2 : (Q::LOADS <= 3 ? 2 : 1);
    }

    template <class QA, class QB, int M, int SRC>
    inline void gemv_quad_dual_launch_ms(dim3 grid, dim3 block, size_t lds, hipStream_t st, const QuadArgs &a)
    {
        if constexpr (M <= QUAD_RING_MAX_M)
        {
            if (a.ring)
            {
                auto kernel = &gemv_quad_dual_kernel<QA, quad_unroll<QA>(M), QB, quad_unroll<QB>(M), M, SRC, QUAD_MODE_RING>;
                static LdsGrant grant;
                (void)allow_lds(grant, reinterpret_cast<const void *>(kernel), QUAD_MAX_LDS);
                hipLaunchKernelGGL(kernel, grid, block, lds, st, a);
                return;
            }
        }
        auto kernel = &gemv_quad_dual_kernel<QA, quad_unroll<QA>(M), QB, quad_unroll<QB>(M), M, SRC>;
        static LdsGrant grant;
        (void)allow_lds(grant, reinterpret_cast<const void *>(kernel), QUAD_MAX_LDS);
        hipLaunchKernelGGL(kernel, grid, block, lds, st, a);
    }

    template <class QA, class QB, int M>
    inline void gemv_quad_dual_launch_m(int src, dim3 grid, dim3 block, size_t lds, hipStream_t st, const QuadArgs &a)
    {
        if constexpr (M <= QUAD_NORM_MAX_M)
            if (src == QUAD_SRC_RMSNORM)
            {
                gemv_quad_dual_launch_ms<QA, QB, M, QUAD_SRC_RMSNORM>(grid, block, lds, st, a);
                return;
            }
        if (src == QUAD_SRC_F32)
            gemv_quad_dual_launch_ms<QA, QB, M, QUAD_SRC_F32>(grid, block, lds, st, a);
        else
            gemv_quad_dual_launch_ms<QA, QB, M, QUAD_SRC_Q8>(grid, block, lds, st, a);
    }

    // M = 1..4, src Q8_1 or fp32
    template <class QA, class QB>
    inline void gemv_quad_dual_launch(int M, int src, dim3 grid, dim3 block, size_t lds, hipStream_t st,
                                      const QuadArgs &a)
    {
        switch (M)
        {
        case 1: gemv_quad_dual_launch_m<QA, QB, 1>(src, grid, block, lds, st, a); break;
        case 2: gemv_quad_dual_launch_m<QA, QB, 2>(src, grid, block, lds, st, a); break;
        case 3: gemv_quad_dual_launch_m<QA, QB, 3>(src, grid, block, lds, st, a); break;
        case 4: gemv_quad_dual_launch_m<QA, QB, 4>(src, grid, block, lds, st, a); break;
        case 5: gemv_quad_dual_launch_m<QA, QB, 5>(src, grid, block, lds, st, a); break;
        case 6: gemv_quad_dual_launch_m<QA, QB, 6>(src, grid, block, lds, st, a); break;
        case 7: gemv_quad_dual_launch_m<QA, QB, 7>(src, grid, block, lds, st, a); break;
        default: gemv_quad_dual_launch_m<QA, QB, 8>(src, grid, block, lds, st, a); break;
        }
    }

    // Launch shape.  R, the rows one wavefront walks, fixes which lane handles which
    // super-block of a row and with it the bits of the result, so it is chosen from N and
    // nsb alone: every batch size then shares the row partition and a batch row is
    // bit-identical to its single-row result.  The cost of a candidate is the number of
    // steps the busiest SIMD unit runs one after another (a compute unit has four; its
    // wavefronts are dealt round robin), which covers ragged last steps and uneven
    // wavefront counts; measured, that tracks the kernel time as long as a compute unit
    // has at least four wavefronts to keep loads in flight, two per SIMD unit being best.
    struct QuadShape
    {
        int waves, rows_per_wave;
        long grid;
    };
    // resident: wavefronts a compute unit should hold at once (8 for the memory-bound decoders:
    // two per SIMD unit; 16 for the arithmetic-bound one)
    inline QuadShape gemv_quad_shape(long N, int nsb, int cus, int max_waves, int resident = 8)
    {
        const int rpw_override = gemv_rows_per_wave_override();
        // the search below costs a microsecond or two: remember the last answers
        struct Memo
        {
            long N;
            int nsb, cus, max_waves, resident, rpw;
            QuadShape sh;
        };
        thread_local Memo memo[16] = {};
        thread_local int memo_next = 0;
        for (const Memo &e : memo)
            if (e.N == N && e.nsb == nsb && e.cus == cus && e.max_waves == max_waves && e.resident == resident &&
                e.rpw == rpw_override)
                return e.sh;
        int best_R = 1;
        long best_wpc = 1;
        double best_cost = 1e30;
        for (int R = 1; R <= 512; ++R)
        {
            if (rpw_override > 0 && R != rpw_override)
                continue;
            const long steps = ((long)R * nsb + QUAD_STEP_SB - 1) / QUAD_STEP_SB;
            const long waves = (N + R - 1) / R;
            const long wpc = (waves + cus - 1) / cus; // wavefronts on the busiest compute unit
            // at most `resident` wavefronts of the widest variant fit a compute unit at once
            const long rounds = (wpc + resident - 1) / resident;
            const long per_simd = rounds > 1 ? (resident / 4) * rounds : (wpc + 3) / 4;
            double cost = (double)(per_simd * steps) / ((double)N * nsb / cus / (4.0 * QUAD_STEP_SB));
            if (wpc < 4)
                cost *= 1.0 + 0.25 * (double)(4 - wpc); // too few loads in flight
            else if (resident <= 8 && wpc < 8)
                cost *= 1.10;                           // one wavefront cannot keep a SIMD unit busy
            if (resident > 8 && wpc <= 4)
                cost *= 1.28; // arithmetic-bound decoder: a lone wavefront leaves its SIMD unit idle
                              // while it waits (measured: 24.3 against 19.2 us at two per unit)
            if (steps < 4)
                cost *= 1.0 + 0.10 * (double)(4 - steps); // short runs do not amortise their start
            if (cost < best_cost - 1e-9)
            {
                best_cost = cost;
                best_R = R;
                best_wpc = wpc;
            }
            if (waves <= 1)
                break;
        }
        QuadShape sh;
        sh.rows_per_wave = best_R;
        const long waves = (N + best_R - 1) / best_R;
        const long wgs_per_cu = (best_wpc + max_waves - 1) / max_waves;
        long nw = (best_wpc + wgs_per_cu - 1) / wgs_per_cu;
        if (nw > waves)
            nw = waves;
        sh.waves = (int)(nw < 1 ? 1 : nw);
        sh.grid = (waves + sh.waves - 1) / sh.waves;
        memo[memo_next] = Memo{N, nsb, cus, max_waves, resident, rpw_override, sh};
        memo_next = (memo_next + 1) % 16;
        return sh;
    }
} // namespace llamql
