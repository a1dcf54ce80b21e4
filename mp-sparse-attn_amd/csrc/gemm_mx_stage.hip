// Block-scaled NT matmul with one stage of K (K == 128, the score product of attention; gfx950): any M and N, one format or 8-bit A
// against 4-bit B, 16-bit results whose rows start on 16 bytes; the semantics of gemm_mx.hip.
//
// What bounds such a product is its results: 16 of 2048 x 2048 write 134 MB and read 4.  The general kernel makes a 128 x 128
// tile a workgroup -- wait for the operands, sixteen matrix instructions, store -- and stores half of the time.  Here a workgroup
// keeps its 128 rows of A and walks tiles of B: the next tile's operands are asked for before this one's results are stored, and
// waited for with the stores still on their way (they are younger, and requests are counted in order).  So the loads are never
// waited for behind a store, and a store is never waited for at all but where a tile is cut.
// Four tiles a workgroup, from 1024 tiles on (below that one each: workgroups run out).  Against the general kernel, bf16
// results: 16 x 2048 x 2048 25.0 -> 22.7 us 4-bit, 31.2 -> 25.5 8-bit; 32 x 3968 x 3968, 8-bit, 328 -> 202; 16 x 4096 x 4096, 4-bit,
// 122 -> 104; 4 x 2688 x 2688, 8-bit, 16.3 -> 13.0; 16 x 1024 x 1024, 4-bit, 9.6 -> 8.0; one a workgroup, 8 x 1000 x 1000, 8-bit x
// 4-bit, 6.8 -> 6.3.  Two and eight tiles are within 5 % of four on most of these and up to 30 % slower on one each.  5.9 TB/s of
// results at 2048; a fill reaches 7.4.  Fewer than 1024 blocks of 16 x 16 results are for tiles that split K (gemm_mx.hip).  Stores that pass the L2 by gain 5 to 15 % on some of these shapes and lose 20 to 30 %
// where rows are 4 KiB apart.
#include "gemm_mx_args.h"

namespace {

template <int FA, int FB> struct StageLds {
    static constexpr int A = 0, B = EdgeOp<FA>::BYTES, SA = B + 2 * EdgeOp<FB>::BYTES, SB = SA + 512, OUT = SB + 2 * 512, SMEM = OUT + 4 * rows16_bytes<2>();
};

struct StageArgs : GemmArgs {
    int tiles_m, tiles_n, span, runs;                    // tiles of B a workgroup walks; workgroups per row of tiles
};

template <int FA, int FB, typename OutT>
__global__ __launch_bounds__(256, 2) void gemm_mx_stage_kernel(StageArgs g) {
    typedef EdgeOp<FA> OA;
    typedef EdgeOp<FB> OB;
    typedef StageLds<FA, FB> L;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, h = lane >> 5, r = lane & 31;
    const int row = blockIdx.x / g.runs, m0 = row * 128;
    const int first = (blockIdx.x - row * g.runs) * g.span, last = min(first + g.span, g.tiles_n) - 1;
    const int bz = blockIdx.y, bb = bz / g.heads_a, ha = bz - bb * g.heads_a;
    const int64_t zb = (int64_t)bb * g.heads_b + ha / (g.heads_a / g.heads_b);
    const uint8_t* const a = g.a + ((int64_t)bz * g.M + m0) * OA::ROW;
    const uint8_t* const b = g.b + zb * g.N * OB::ROW;
    const uint8_t* const sa = g.sa + ((int64_t)bz * g.M + m0) * 4;
    const uint8_t* const sb = g.sb + zb * g.N * 4;

    // a tile's codes, rows XOR-swizzled, and its scale words: 512 bytes in a row in either layout.  Rows past the matrix are
    // its last row.
    auto fetch = [&](auto op, const uint8_t* codes, const uint8_t* scales, int rows, uint8_t* img, uint8_t* simg) __attribute__((always_inline)) {
        typedef decltype(op) O;
#pragma unroll
        for (int c = 0; c < O::IPW; ++c) {
            const int p = (wave * O::IPW + c) * 64 + lane, r_ = p / O::CPR;
            load_to_lds_uniform<16>((uint32_t)(min(r_, rows - 1) * O::ROW + ((p % O::CPR) ^ O::swz(r_)) * 16), codes, img + (wave * O::IPW + c) * 1024);
        }
        // (everybody asks, so that all waves count the same loads: waves 2 and 3 for what waves 0 and 1 do)
        load_to_lds_uniform<4>((uint32_t)(min((wave & 1) * 64 + lane, rows - 1) * 4), scales, simg + (wave & 1) * 256);
    };
    auto fetch_b = [&](int t) __attribute__((always_inline)) {
        fetch(OB{}, b + (int64_t)t * OB::BYTES, sb + (int64_t)t * 512, min(128, g.N - 128 * t), smem + L::B + (t & 1) * OB::BYTES, smem + L::SB + (t & 1) * 512);
    };
    // byte offset of a row's scale word
    auto word = [&](int x) { return g.packed ? (x & 31) * 16 + (x >> 5) * 4 : x * 4; };

    fetch(OA{}, a, sa, min(128, g.M - m0), smem + L::A, smem + L::SA);
    fetch_b(first);
    OutT* const c = static_cast<OutT*>(g.c) + (int64_t)bz * g.M * g.ldc;
    constexpr int STORES = 2 * 4;                        // of a whole tile, per wave: 2 x 32 rows, 8 rows a store
    bool stored = false;                                 // whether the loads waited for have exactly so many stores behind them
#pragma unroll 1
    for (int t = first; t <= last; ++t) {
        // this tile has landed, everybody's part of it, and everybody has read the one before
        __builtin_amdgcn_sched_barrier(0);
        if (stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(STORES) : "memory");
        else        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (t < last) fetch_b(t + 1);
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t* const img = smem + L::B + (t & 1) * OB::BYTES;
        const uint8_t* const simg = smem + L::SB + (t & 1) * 512;
        v16f acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
        int ca[2], cb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ca[i] = (int)(*reinterpret_cast<const uint32_t*>(smem + L::SA + word(wm * 64 + i * 32 + r)) >> (8 * h));
            cb[i] = (int)(*reinterpret_cast<const uint32_t*>(simg + word(wn * 64 + i * 32 + r)) >> (8 * h));
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            v8i fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[i] = OA::frag(smem + L::A, wm * 64 + i * 32 + r, k, h);
                fb[i] = OB::frag(img, wn * 64 + i * 32 + r, k, h);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (k == 0) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i], fb[j], acc[i][j], FA, FB, 0, ca[i], 0, cb[j]);
                    else        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i], fb[j], acc[i][j], FA, FB, 2, ca[i], 2, cb[j]);
                }
        }
        uint8_t* const out = smem + L::OUT + wave * rows16_bytes<2>();
        stored = m0 + 128 <= g.M && 128 * t + 128 <= g.N;
        if (stored) {
#pragma unroll
            for (int i = 0; i < 2; ++i) store_rows16<2, OutT, false>(acc[i], out, c, g.ldc, m0 + wm * 64 + i * 32, 128 * t + wn * 64, g.M, g.N, lane);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) store_rows16<2, OutT, true>(acc[i], out, c, g.ldc, m0 + wm * 64 + i * 32, 128 * t + wn * 64, g.M, g.N, lane);
        }
    }
}

template <int FA, int FB, typename OutT>
struct StageReg {
    static inline const bool registered = mpsa_register_lds_kernel(reinterpret_cast<const void*>(gemm_mx_stage_kernel<FA, FB, OutT>), StageLds<FA, FB>::SMEM);
};

template <int FA, int FB>
void launch_out(const StageArgs& s, int c_dtype, dim3 grid, hipStream_t st) {
    if (c_dtype == MPSA_BF16) {
        if (StageReg<FA, FB, __bf16>::registered) hipLaunchKernelGGL((gemm_mx_stage_kernel<FA, FB, __bf16>), grid, dim3(256), (StageLds<FA, FB>::SMEM), st, s);
    } else {
        if (StageReg<FA, FB, _Float16>::registered) hipLaunchKernelGGL((gemm_mx_stage_kernel<FA, FB, _Float16>), grid, dim3(256), (StageLds<FA, FB>::SMEM), st, s);
    }
}

}  // namespace

bool gemm_stage_takes(const GemmArgs& g, int fmt_a, int fmt_b, int c_dtype) {
    return g.K == 128 && (fmt_a == fmt_b || fmt_b == MPSA_FMT_E2M1) && (c_dtype == MPSA_BF16 || c_dtype == MPSA_F16) &&
           ((reinterpret_cast<uintptr_t>(g.c) | (uintptr_t)(2 * g.ldc)) & 15) == 0;
}

void gemm_stage_launch(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int c_dtype, hipStream_t st) {
    StageArgs s;
    static_cast<GemmArgs&>(s) = g;
    s.tiles_m = (g.M + 127) / 128;
    s.tiles_n = (g.N + 127) / 128;
    s.span = (int64_t)s.tiles_m * s.tiles_n * batches >= 1024 ? 4 : 1;
    s.runs = (s.tiles_n + s.span - 1) / s.span;
    const dim3 grid((unsigned)(s.tiles_m * s.runs), (unsigned)batches);
    if (fmt_a == MPSA_FMT_E2M1)                               launch_out<MPSA_FMT_E2M1, MPSA_FMT_E2M1>(s, c_dtype, grid, st);
    else if (fmt_a == MPSA_FMT_E4M3 && fmt_b == MPSA_FMT_E4M3) launch_out<MPSA_FMT_E4M3, MPSA_FMT_E4M3>(s, c_dtype, grid, st);
    else if (fmt_a == MPSA_FMT_E5M2 && fmt_b == MPSA_FMT_E5M2) launch_out<MPSA_FMT_E5M2, MPSA_FMT_E5M2>(s, c_dtype, grid, st);
    else if (fmt_a == MPSA_FMT_E4M3)                          launch_out<MPSA_FMT_E4M3, MPSA_FMT_E2M1>(s, c_dtype, grid, st);
    else                                                      launch_out<MPSA_FMT_E5M2, MPSA_FMT_E2M1>(s, c_dtype, grid, st);
}
