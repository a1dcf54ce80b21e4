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

// gemm_mx_edge.hip: 256 x 256 tiles with ragged edges, or with 4-bit codes, K % 256 == 128 and row-major scales; one format or 8-bit A
// against 4-bit B, K % 128 == 0
void gemm_edge_launch(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int c_dtype, hipStream_t st);
// gemm_mx_stage.hip: products with one stage of K and 16-bit results
bool gemm_stage_takes(const GemmArgs& g, int fmt_a, int fmt_b, int c_dtype);
void gemm_stage_launch(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int c_dtype, hipStream_t st);

namespace {

// lane L's BYTES bytes at base + off land at lds + L * BYTES.  As assembly, so that only the kernel's own partial waits apply
// (gemm_mx_kernel.h says why); base and lds are the same in every lane, whether the compiler sees it or not.
template <int BYTES>
__device__ __forceinline__ void load_to_lds_uniform(uint32_t off, const uint8_t* base, uint8_t* lds) {
    const uint32_t l = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)lds);
    const uint64_t b = uniform_bits(base);
    if constexpr (BYTES == 16) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(l), "v"(off), "s"(b) : "memory", "m0");
    else                       asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(l), "v"(off), "s"(b) : "memory", "m0");
}

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

// 128 rows of an operand for one stage of 128 elements of K, in LDS: the general kernel and the one for a single stage
template <int FMT> struct EdgeOp {
    static constexpr bool FP4 = FMT == MPSA_FMT_E2M1;
    static constexpr int ROW = FP4 ? 64 : 128;           // code bytes per row per stage
    static constexpr int CPR = ROW / 16;                 // 16-byte pieces per row
    static constexpr int BYTES = 128 * ROW;              // the operand's codes of one stage
    static constexpr int IPW = BYTES / 1024 / 4;         // direct-to-LDS instructions per wave and stage
    __device__ static __forceinline__ int swz(int row) { return FP4 ? (row >> 2) & 3 : (row >> 1) & 7; }
    // the fragment of matrix-instruction step k (0 / 1) of the stage, LDS row `row` of the operand's stage image
    __device__ static __forceinline__ v8i frag(const uint8_t* img, int row, int k, int h) {
        const uint8_t* p = img + row * ROW;
        const int f = swz(row);
        if constexpr (FP4) {
            const v4i x = *reinterpret_cast<const v4i*>(p + (((2 * k + h) ^ f) * 16));
            return (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
        } else {
            const v4i x0 = *reinterpret_cast<const v4i*>(p + (((4 * k + h) ^ f) * 16));
            const v4i x1 = *reinterpret_cast<const v4i*>(p + (((4 * k + h + 2) ^ f) * 16));
            return (v8i){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
        }
    }
};

// Whether 16-bit results may be stored in pieces of 16 bytes: every row starts on such a piece.
__device__ __forceinline__ bool rows16_aligned(const GemmArgs& g) { return ((reinterpret_cast<uintptr_t>(g.c) | (uintptr_t)(2 * g.ldc)) & 15) == 0; }

// LDS bytes a wave needs to store 32 rows of 32 * NJ 16-bit results
template <int NJ> constexpr int rows16_bytes() { return 32 * (NJ * 64 + 64); }

// A wave's NJ neighbouring 32 x 32 blocks (accumulator register e of lane (h, r) is element [8*(e/4) + 4*h + e%4][r]) as 16-bit
// results, through LDS of the wave's own, in pieces of 16 bytes.  Straight from the registers a store moves 2 bytes a lane, half
// of two rows' 128-byte lines, there are eight times as many, and ragged tiles check the edges for each element.  Measured
// (bf16 results): 16 score products of 2048 x 2048 x 128, 4-bit, 29.4 -> 25.1 us (5.3 TB/s of results; a fill of that size
// reaches 7.4), 8-bit 39.5 -> 31; 1000 x 14336 x 4096, 8-bit x 4-bit, 51.6 -> 47.5; 1000 x 4096 x 4096, 4-bit, 17.4 -> 16.4.
// Two rows of two neighbouring lanes trade places first, so that LDS is written a word at a time; the row pitch (16 words past a
// multiple of 32) puts the two rows of a write into different banks.
template <int NJ, typename OutT, bool EDGE>
__device__ __forceinline__ void store_rows16(const v16f (&acc)[NJ], uint8_t* lds, OutT* c, int64_t ldc, int row0, int col0, int M, int N, int lane) {
    typedef OutT v2o __attribute__((ext_vector_type(2)));
    constexpr int PITCH = NJ * 64 + 64, LPR = 4 * NJ;    // bytes from row to row; lanes per row on the way out
    const int h = lane >> 5, r = lane & 31;
    const uint32_t sel = (r & 1) ? 0x03020706u : 0x05040100u;
    uint8_t* const to = lds + (4 * h + (r & 1)) * PITCH + (r >> 1) * 4;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
            const uint32_t own = __builtin_bit_cast(uint32_t, (v2o){cvt_out<OutT>(acc[j][e]), cvt_out<OutT>(acc[j][e + 1])});
            const uint32_t other = (uint32_t)__builtin_amdgcn_mov_dpp((int)own, 0xB1, 0xf, 0xf, true);       // of lane ^ 1
            *reinterpret_cast<uint32_t*>(to + (8 * (e >> 2) + (e & 3)) * PITCH + j * 64) = __builtin_amdgcn_perm(other, own, sel);
        }
    const int lrow = lane / LPR, col = col0 + 8 * (lane % LPR);
    const uint8_t* const from = lds + lrow * PITCH + (lane % LPR) * 16;
    OutT* out = c + (int64_t)(row0 + lrow) * ldc + col;
#pragma unroll
    for (int x = 0; x < 32; x += 64 / LPR) {
        const v4i w = *reinterpret_cast<const v4i*>(from + x * PITCH);
        if (!EDGE || (row0 + lrow + x < M && col + 8 <= N)) {
            *reinterpret_cast<v4i*>(out + (int64_t)x * ldc) = w;
        } else if (row0 + lrow + x < M) {
#pragma unroll
            for (int y = 0; y < 8; ++y)
                if (col + y < N) out[(int64_t)x * ldc + y] = __builtin_bit_cast(OutT, (unsigned short)((uint32_t)w[y >> 1] >> (16 * (y & 1))));
        }
    }
}

}  // namespace
