// Pieces shared by the block-scaled matmul kernels: the argument block and the output conversions.
#pragma once
#include "mpsa_common.h"

struct GemmArgs {
    const uint8_t *a, *sa, *b, *sb;
    void* c;
    int64_t ldc;
    int M, N, K;
    int packed;                // scales in the packed [rows/128, K/128, 32, 4, 4] form instead of [rows, K/32]
    int heads_a, heads_b;      // batched runs: blockIdx.y = batch * heads_a + head; B's head is head / (heads_a / heads_b)
};

// gemm_mx_split.hip: tiles of a few 16 x 16 blocks, K split between the waves; any M, N and pair of formats, K % 128 == 0
double gemm_split_cost(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int* tile);
void gemm_split_launch(const GemmArgs& g, int64_t batches, int tile, int fmt_a, int fmt_b, int c_dtype, hipStream_t st);
// gemm_mx_tile.hip: 128 x 128 tiles, any M, N and pair of formats, K % 128 == 0
void gemm_tile_launch(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int c_dtype, hipStream_t st);

// gemm_mx_edge.hip: 256 x 256 tiles with ragged edges; one format or 8-bit A against 4-bit B, K % 256 == 0 (4-bit A) / K % 128 == 0
void gemm_edge_launch(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int c_dtype, hipStream_t st);

namespace {

template <typename T> __device__ __forceinline__ T cvt_out(float v);
template <> __device__ __forceinline__ float cvt_out<float>(float v) { return v; }
template <> __device__ __forceinline__ __bf16 cvt_out<__bf16>(float v) { return (__bf16)v; }
template <> __device__ __forceinline__ _Float16 cvt_out<_Float16>(float v) { return (_Float16)v; }
// E5M2 output byte, round to nearest even, overflow to infinity (what a float32 -> float8_e5m2 cast does in torch;
// the reference's kernel casts with c.to(tl.float8e5), ours/block_scaled_matmul.py:185-190)
struct OutE5M2 { uint8_t b; };
template <> __device__ __forceinline__ OutE5M2 cvt_out<OutE5M2>(float v) {
    const uint32_t u = mpsa_f2u(v);
    const uint32_t a = u & 0x7FFFFFFFu;
    // 61440 = the largest finite E5M2 value plus half a step: from there on the cast gives infinity (or keeps NaN)
    if (a >= 0x47700000u) return OutE5M2{(uint8_t)(((u >> 24) & 0x80u) | (a > 0x7F800000u ? 0x7Fu : 0x7Cu))};
    // below that the conversion instruction rounds to nearest even, subnormals included
    return OutE5M2{(uint8_t)(__builtin_amdgcn_cvt_pk_bf8_f32(v, v, 0, false) & 0xFF)};
}

}  // namespace
