// Linear layers over tiled bf16 weights, as the launchers inside the library see them.
#pragma once

#include "seq_common.h"
#include "llaminar_amd/seq_api.h"

namespace llamql
{
    struct LinearArgs
    {
        const void *a; // T [M][lda], or fp32 [M][lda] when norm is set
        const void *w;
        void *y;
        const float *bias;
        const float *norm;
        void *h_out;
        float eps;
        int k_real;
        int M, N, K;
        int lda, ldy;
        int out; // LLAM_SEQ_OUT_*
        float limit;
        long a_stride, w_stride, y_stride;
        // rows in groups (routed experts): group z has the rows group_offset[z] .. group_offset[z + 1] - 1
        // of y; row r reads a[row_source ? row_source[r] / source_div : r]
        const int *group_offset;
        const int *row_source;
        int source_div;
        int groups, group_rows; // groups, and rows of all of them
        // many rows: tiles from `full` on are cut into slices of K, their sums in `parts` (linear_tiled)
        f32x4 *parts;
        int full, slices;
    };
    // Some of many rows: one stretch a layer of the grid.  (A type and a kernel of its own: read as part of the others' arguments it cost each of
    // their launches 0.5 to 1 us, bf16 24 x 15440 x 5120 28.9 -> 29.9.)
    constexpr int LINEAR_STRETCHES = 8; // in a launch, at most
    struct LinearSomeArgs : LinearArgs
    {
        int stretches;
        int first[LINEAR_STRETCHES], rows[LINEAR_STRETCHES];
    };

    constexpr int SMALL_M = 16;         // most rows of the row-at-a-time kernel: one operand of the matrix unit
    constexpr int NORM_FUSE_MAX = 8192; // most values (rows x columns) every workgroup norms for itself

    __host__ __device__ inline bool is_gated(int out) { return out == LLAM_SEQ_OUT_GATED || out == LLAM_SEQ_OUT_GATED_CLAMP; }
    bool linear_small(const char *fn, const LinearArgs &a, int batch, int dtype, int device_id, hipStream_t st);
    // scratch: for sums of tiles cut along K, as far as it reaches; what linear_split_bytes says serves layers of up to max_rows rows
    bool linear_tiled(const char *fn, const LinearArgs &a, int batch, int dtype, int device_id, hipStream_t st, void *scratch = nullptr,
                      size_t bytes = 0);
    // The same for some of its rows, with the bits that they have among all
    bool linear_tiled_rows(const char *fn, const LinearSomeArgs &a, int batch, int dtype, int device_id, hipStream_t st);
    size_t linear_split_bytes(int max_rows, int N, int K, int dtype, int device_id);

    // Whether a sum of products in three bf16 pieces of each 32-bit value may not be that of the whole values, which then
    // are multiplied once more without pieces: the second and third piece of most values are zero, and zero times an infinite
    // weight is not a number; and pieces end at 2^-133, the smallest bf16, so that something is lost of values below 2^-110.
    // That is less than 2^-133, so a sum of 2^-80 misses less than its own rounding as long as the magnitudes of its weights
    // add up to less than 2^29.  A sum of zero is taken at its word, so what lies below 2^-133 (9e-41) is missed where the
    // pieces add up to nothing.  (Looking out for it costs 8 to 10 % of a prompt's layer: 2048 x 51200 x 5120 2480 -> 2670 us.)
    __device__ __forceinline__ bool pieces_fail(float sum) { return !(fabsf(sum) >= 0x1p-80f) && sum != 0.0f; }

    __device__ __forceinline__ f32x4 relu2(f32x4 v)
    {
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const float z = fmaxf(v[r], 0.0f);
            v[r] = z * z;
        }
        return v;
    }

    // LLAM_SEQ_OUT_*: four neighbouring output columns of one row
    template <typename T>
    __device__ __forceinline__ void store4(const LinearArgs &p, char *ybase, int row, int col, f32x4 v)
    {
        typedef T t4 __attribute__((ext_vector_type(4)));
        const size_t at = (size_t)row * p.ldy + col;
        switch (p.out)
        {
        case LLAM_SEQ_OUT_F32:
            if (p.bias)
            {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    v[r] += p.bias[col + r];
            }
            *reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(ybase) + at) = v;
            break;
        case LLAM_SEQ_OUT_ADD:
        {
            f32x4 *dst = reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(ybase) + at);
            *dst = *dst + v;
            break;
        }
        case LLAM_SEQ_OUT_RELU2:
            *reinterpret_cast<t4 *>(reinterpret_cast<T *>(ybase) + at) = __builtin_convertvector(relu2(v), t4);
            break;
        default:
            *reinterpret_cast<t4 *>(reinterpret_cast<T *>(ybase) + at) = __builtin_convertvector(v, t4);
        }
    }

    __device__ __forceinline__ f32x4 gated4(const LinearArgs &p, f32x4 gate, f32x4 up)
    {
        f32x4 v;
        if (p.out == LLAM_SEQ_OUT_GATED_CLAMP)
        {
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const float a = fminf(gate[r], p.limit), u = fminf(fmaxf(up[r], -p.limit), p.limit);
                v[r] = a * sigmoidf(1.702f * a) * (u + 1.0f);
            }
            return v;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
            v[r] = gelu_tanh(gate[r]) * up[r];
        return v;
    }
} // namespace llamql
