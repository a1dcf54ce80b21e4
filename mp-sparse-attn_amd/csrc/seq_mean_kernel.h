// The mean over the sequence per (batch, head, channel): sums of chunks of rows, shared by quantize.hip (the stand-alone
// kernels) and prepare.hip (the preparation that takes the mean itself).  The order of the additions is the same everywhere.
#pragma once
#include "quantize_kernel.h"

namespace {

constexpr int MEAN_ROWS = 256;     // rows per partial sum

// partial sums x[0], x[stride], ... added in order; a batch of them is requested before its first is added (one at a time,
// 128 of them took 31 us)
__device__ __forceinline__ float seq_sum(const float* x, int count, int stride) {
    constexpr int BATCH = 32;
    float s = 0.0f;
    for (int k = 0; k < count; k += BATCH) {
        float v[BATCH];
#pragma unroll
        for (int i = 0; i < BATCH; ++i) v[i] = x[(int64_t)min(k + i, count - 1) * stride];
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            if (k + i < count) s += v[i];
    }
    return s;
}

// 256 threads, numbered t, sum MEAN_ROWS rows of one head: a thread owns 8 channels of every (256*8/D)-th row; the row
// groups are then added in a fixed order through LDS, so the result does not depend on timing.  A thread's rows are
// requested before the first is added: with one load in flight a short sequence took a memory round trip per row
// (2 x 16 heads, 333 rows: 8.3 us, this way 7.5).
template <int D> struct MeanChunk {
    static constexpr int CPR = D >> 3;                  // 8-channel groups per row (8 or 16)
    static constexpr int RTHREADS = 256 / CPR, EACH = MEAN_ROWS / RTHREADS;
    uint4 raw[EACH];
    // head: the head's first row; n rows, sn elements apart
    __device__ __forceinline__ void request(const char* head, int64_t sn, int row0, int n, uint32_t t = threadIdx.x) {
        const char* base = head + 16 * (t % CPR);
#pragma unroll
        for (int i = 0; i < EACH; ++i) {
            const int row = min(row0 + (int)(t / CPR) + i * RTHREADS, n - 1);
            raw[i] = *reinterpret_cast<const uint4*>(base + 2 * (int64_t)row * sn);
        }
    }
    // this thread's sums, into LDS
    template <int XDT>
    __device__ __forceinline__ void add(float (&part)[256][9], int row0, int n, uint32_t t = threadIdx.x) const {
        const int row1 = min(row0 + MEAN_ROWS, n);
        float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < EACH; ++i) {
            if (row0 + (int)(t / CPR) + i * RTHREADS >= row1) break;
            float x[8];
            unpack8<XDT>(raw[i], x);
#pragma unroll
            for (int q = 0; q < 8; ++q) acc[q] += x[q];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) part[t][i] = acc[i];
    }
    // channel c's sum
    __device__ static __forceinline__ float total(const float (&part)[256][9], int c) {
        float s = 0.0f;
#pragma unroll
        for (int t = 0; t < RTHREADS; ++t) s += part[t * CPR + (c >> 3)][c & 7];
        return s;
    }
};

// the mean in the inputs' 16-bit type
template <int XDT>
__device__ __forceinline__ uint16_t mean_bits(float m) {
    if constexpr (XDT == MPSA_BF16) {
        const uint32_t u = mpsa_f2u(m);
        return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
    } else {
        return __builtin_bit_cast(uint16_t, (_Float16)m);
    }
}

}  // namespace
