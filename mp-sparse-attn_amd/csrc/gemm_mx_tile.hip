// Block-scaled NT matmul on 128 x 128 tiles (gfx950): any M and N, any pair of element formats, K % 128 == 0; the
// semantics of gemm_mx.hip.  For matrices with too few or too ragged 256 x 256 tiles.
//
// What bounds a tile of this size is the way into LDS: 256 rows x 128 bytes a unit at 51 bytes a clock take 640 clocks,
// its matrix instructions 512 (4-bit) or 1024 (8-bit) -- if enough bytes are in flight.  So one workgroup has the CU to
// itself with a ring of four units (whole 128-byte lines per row: 256 elements of 4-bit codes, 128 of 8-bit ones), three
// in flight while one is multiplied, one barrier per unit; eight waves, two per quarter of the tile, share the unit: the
// two waves of a quarter take alternate matrix steps of it (K split inside the workgroup) and add their sums through LDS
// at the end, one half of the quarter each.
// Scale bytes: four words a row at a time (two units of 4-bit codes, four of 8-bit ones), 16 rows per load instruction;
// fetching a word per row and unit, one lane per line, took longer than the codes.
// Measured (bf16 output, which leaves through LDS in pieces of 16 bytes): 1000 x 4096 x 4096 16.1 us 4-bit, 20.8 8-bit x 4-bit, 22.9
// 8-bit (18.5 and 24 the first two when a lane stored its own elements); 2048^3 11.2, 13.1 and 13.9.  Reading the next unit's operands into
// a second set of registers while one is multiplied takes 1 to 11 % longer.  Clock stamps in a copy of this
// kernel, 1000 x 4096 x 4096: a unit takes 1390 clocks with 4-bit codes (512 of matrix work), 980 with 8-bit x 4-bit ones and
// 1060 with 8-bit ones (half a unit's K, 512); prologue and first unit 5000, adding up and storing 5700.
#include "gemm_mx_args.h"

namespace {

constexpr int RING = 4;
constexpr int TW = 8;                                    // waves

template <int FMT, int UNITK>
struct TileOp {
    static constexpr bool FP4 = FMT == MPSA_FMT_E2M1;
    static constexpr int ROW = FP4 ? UNITK / 2 : UNITK;  // code bytes per row and unit (64 | 128)
    static constexpr int CPR = ROW / 16;                 // 16-byte pieces per row
    static constexpr int BYTES = 128 * ROW;
    static constexpr int IPW = BYTES / 1024 / TW;        // load instructions per wave and unit
    __device__ static __forceinline__ int swz(int row) { return CPR == 4 ? (row >> 2) & 3 : (row >> 1) & 7; }
    // the fragment of matrix step k of the unit, row `row` of the operand's image
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

template <int FA, int FB>
struct TileGeom {
    static constexpr bool BOTH4 = FA == MPSA_FMT_E2M1 && FB == MPSA_FMT_E2M1;
    static constexpr int UNITK = BOTH4 ? 256 : 128;
    static constexpr int STEPS = UNITK / 64;             // matrix steps per unit (4 | 2)
    static constexpr int SGROUP = 512 / UNITK;           // units per scale group: four words (512 elements) a row
    typedef TileOp<FA, UNITK> OA;
    typedef TileOp<FB, UNITK> OB;
    static constexpr int UNIT = OA::BYTES + OB::BYTES;
    static constexpr int SCALES = 256 * 16;              // one group: 128 rows of A, then 128 of B
    static constexpr int LOADS = OA::IPW + OB::IPW;      // code instructions per wave and unit
    static constexpr int SMEM = RING * UNIT + 4 * SCALES;
    static_assert(4 * 16384 + TW * rows16_bytes<2>() <= SMEM, "the waves' sums, and behind them the results on their way out");
};

template <int FA, int FB, typename OutT>
__global__ __launch_bounds__(TW * 64, 1) void gemm_mx_tile_kernel(GemmArgs a) {
    typedef TileGeom<FA, FB> G;
    typedef typename G::OA OA;
    typedef typename G::OB OB;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    uint8_t* const scales = smem + RING * G::UNIT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;     // which steps of a unit; which quarter of the tile
    const int h = lane >> 5, r = lane & 31;

    // one contiguous range of tiles per XCD, walked in panels of eight tile rows: neighbours share both operands' slices in that L2
    const int tiles_m = (a.M + 127) / 128, tiles_n = (a.N + 127) / 128, total = tiles_m * tiles_n;
    int L = blockIdx.x;
    if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);
    const int panel = L / (8 * tiles_n), in = L - panel * 8 * tiles_n, rows = min(8, tiles_m - 8 * panel);
    const int m0 = (8 * panel + in % rows) * 128, n0 = (in / rows) * 128;
    const int bz = blockIdx.y;
    const int bb = bz / a.heads_a, ha = bz - bb * a.heads_a;
    const int64_t zb = (int64_t)bb * a.heads_b + ha / (a.heads_a / a.heads_b);
    const int rowb_a = OA::FP4 ? a.K / 2 : a.K, rowb_b = OB::FP4 ? a.K / 2 : a.K;
    const int kblocks = a.K / 32, words = a.K / 128;     // scale bytes / scale words per row
    const int units = (a.K + G::UNITK - 1) / G::UNITK;

    // ---- staging: rows past the matrix are its last row ----
    const int last_a = min(127, a.M - 1 - m0), last_b = min(127, a.N - 1 - n0);
    const uint8_t* const ta = a.a + ((int64_t)bz * a.M + m0) * rowb_a;
    const uint8_t* const tb = a.b + (zb * a.N + n0) * rowb_b;
    uint32_t ra[OA::IPW], pa[OA::IPW], rb[OB::IPW], pb[OB::IPW];         // row offset and 16-byte piece of this lane's loads
#pragma unroll
    for (int c = 0; c < OA::IPW; ++c) {
        const int p = (wave * OA::IPW + c) * 64 + lane, row = p / OA::CPR;
        ra[c] = (uint32_t)min(row, last_a) * (uint32_t)rowb_a;
        pa[c] = (uint32_t)((p % OA::CPR) ^ OA::swz(row)) * 16u;
    }
#pragma unroll
    for (int c = 0; c < OB::IPW; ++c) {
        const int p = (wave * OB::IPW + c) * 64 + lane, row = p / OB::CPR;
        rb[c] = (uint32_t)min(row, last_b) * (uint32_t)rowb_b;
        pb[c] = (uint32_t)((p % OB::CPR) ^ OB::swz(row)) * 16u;
    }
    // scale words: lane -> (row lane/4 of 16, word lane%4); waves 0-3 bring A's 128 rows, waves 4-7 B's, two instructions each
    const int sbase = a.packed ? 512 : 4;                // from one scale word of a row to the next
    const uint8_t* ts;
    uint32_t rs[2];
    {
        const bool isb = wave >= 4;
        const int first = isb ? n0 : m0, last = isb ? last_b : last_a;
        ts = isb ? a.sb + zb * a.N * kblocks : a.sa + (int64_t)bz * a.M * kblocks;
        ts += a.packed ? (int64_t)(first >> 7) * words * 512 : (int64_t)first * kblocks;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int row = min(((wave & 3) * 2 + q) * 16 + (lane >> 2), last);
            rs[q] = a.packed ? (uint32_t)((row & 31) * 16 + (row >> 5) * 4) : (uint32_t)(row * kblocks);
        }
    }
    // K % 256 == 128 under 4-bit codes: the last unit is half a unit, pieces and words past a row's end are its last ones
    auto issue_part = [&](int u, int part) __attribute__((always_inline)) {
        uint8_t* d = smem + (u & (RING - 1)) * G::UNIT;
        if (part == 0) {
            if (u % G::SGROUP == 0) {
                uint8_t* sd = scales + ((u / G::SGROUP) & 3) * G::SCALES + wave * 512;
                const uint32_t w = (uint32_t)(min(4 * (u / G::SGROUP) + (lane & 3), words - 1) * sbase);
                load_to_lds_uniform<4>(rs[0] + w, ts, sd);
                load_to_lds_uniform<4>(rs[1] + w, ts, sd + 256);
            }
#pragma unroll
            for (int c = 0; c < OA::IPW; ++c)
                load_to_lds_uniform<16>(ra[c] + min((uint32_t)(u * OA::ROW) + pa[c], (uint32_t)(rowb_a - 16)), ta, d + (wave * OA::IPW + c) * 1024);
        } else {
#pragma unroll
            for (int c = 0; c < OB::IPW; ++c)
                load_to_lds_uniform<16>(rb[c] + min((uint32_t)(u * OB::ROW) + pb[c], (uint32_t)(rowb_b - 16)), tb, d + OA::BYTES + (wave * OB::IPW + c) * 1024);
        }
    };

    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    constexpr int SPW = G::STEPS / 2;                    // this wave's steps of a unit: a contiguous half of them
    // scale words of this wave's rows for a whole group: one conflict-free 128-bit read a row (single words at a 16-byte
    // pitch, read unit by unit, cost LDS as much as a third of the codes)
    v4i wa[2], wb[2];
    auto read_scales = [&](int group) __attribute__((always_inline)) {
        const uint8_t* sc = scales + (group & 3) * G::SCALES;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            wa[i] = *reinterpret_cast<const v4i*>(sc + (wm * 64 + i * 32 + r) * 16);
            wb[i] = *reinterpret_cast<const v4i*>(sc + 2048 + (wn * 64 + i * 32 + r) * 16);
        }
    };
    // unit u, the x-th of its group; the loads of unit u + RING - 1 go out between the rows of matrix instructions
    auto multiply = [&](int u, int x, bool live) __attribute__((always_inline)) {
        const uint8_t* ia = smem + (u & (RING - 1)) * G::UNIT;
        const uint8_t* ib = ia + OA::BYTES;
        v8i fa[SPW][2], fb[SPW][2];
        int ca[2], cb[2];
        // the word (128 elements) the steps lie in: 4-bit units have two, one per half of the waves; 8-bit units one
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            ca[i] = (int)((uint32_t)(SPW == 2 ? (half ? wa[i][2 * x + 1] : wa[i][2 * x]) : wa[i][x]) >> (8 * h));
            cb[i] = (int)((uint32_t)(SPW == 2 ? (half ? wb[i][2 * x + 1] : wb[i][2 * x]) : wb[i][x]) >> (8 * h));
            if (SPW == 1 && half) { ca[i] = (int)((uint32_t)ca[i] >> 16); cb[i] = (int)((uint32_t)cb[i] >> 16); }
        }
#pragma unroll
        for (int s = 0; s < SPW; ++s)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[s][i] = OA::frag(ia, wm * 64 + i * 32 + r, half * SPW + s, h);
                fb[s][i] = OB::frag(ib, wn * 64 + i * 32 + r, half * SPW + s, h);
            }
        const bool refill = u + RING - 1 < units;
#pragma unroll
        for (int s = 0; s < SPW; ++s)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (live) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        if (s == 0) acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[s][i], fb[s][j], acc[i][j], FA, FB, 0, ca[i], 0, cb[j]);
                        else        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[s][i], fb[s][j], acc[i][j], FA, FB, 2, ca[i], 2, cb[j]);
                    }
                }
                if (s == 0) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (refill) issue_part(u + RING - 1, i);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
    };

#pragma unroll
    for (int u = 0; u < RING - 1; ++u)
        if (u < units) { issue_part(u, 0); issue_part(u, 1); }
    const bool ragged = SPW == 2 && (a.K & 128) != 0;    // half a unit at the end: nothing in it for the second half of the waves
    for (int u0 = 0; u0 < units; u0 += G::SGROUP) {
#pragma unroll
        for (int x = 0; x < G::SGROUP; ++x) {
            const int u = u0 + x;
            if (u >= units) break;
            // unit u has landed: at most the two newer ones' code loads are still on their way (a scale load among them makes
            // the wait a little early, which is harmless); everybody's have after the barrier, and unit u - 1 has been read
            __builtin_amdgcn_sched_barrier(0);
            if (u + 2 < units)      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * G::LOADS) : "memory");
            else if (u + 1 < units) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(G::LOADS) : "memory");
            else                    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
            if (x == 0) read_scales(u0 / G::SGROUP);
            multiply(u, x, !(ragged && half && u == units - 1));
        }
    }

    // ---- the two waves of a quarter add up: half 0 finishes the upper 32 rows, half 1 the lower ones ----
    __syncthreads();
    float* const x = reinterpret_cast<float*>(smem) + (wave & 3) * 4096;             // [half][j][e][lane] of this quarter
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) x[((half * 2 + j) * 16 + e) * 64 + lane] = half ? acc[0][j][e] : acc[1][j][e];
    __syncthreads();
    OutT* c = static_cast<OutT*>(a.c) + (int64_t)bz * a.M * a.ldc;
    const int row0 = m0 + wm * 64 + half * 32;
    v16f sum[2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float other = x[(((1 - half) * 2 + j) * 16 + e) * 64 + lane];
            sum[j][e] = half ? other + acc[1][j][e] : acc[0][j][e] + other;          // first half of K first
        }
    if constexpr (sizeof(OutT) == 2) {
        if (rows16_aligned(a)) {
            store_rows16<2, OutT, true>(sum, smem + 4 * 16384 + wave * rows16_bytes<2>(), c, a.ldc, row0, n0 + wn * 64, a.M, a.N, lane);
            return;
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int col = n0 + wn * 64 + j * 32 + r;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = row0 + 8 * (e >> 2) + 4 * h + (e & 3);
            if (row < a.M && col < a.N) c[(int64_t)row * a.ldc + col] = cvt_out<OutT>(sum[j][e]);
        }
    }
}

template <int FA, int FB, typename OutT>
struct TileLds {
    static inline const bool registered =
        mpsa_register_lds_kernel(reinterpret_cast<const void*>(gemm_mx_tile_kernel<FA, FB, OutT>), TileGeom<FA, FB>::SMEM);
};

template <int FA, int FB, typename OutT>
void launch_one(const GemmArgs& g, int64_t batches, hipStream_t st) {
    if (!TileLds<FA, FB, OutT>::registered) return;
    const unsigned tiles = (unsigned)((g.M + 127) / 128) * (unsigned)((g.N + 127) / 128);
    hipLaunchKernelGGL((gemm_mx_tile_kernel<FA, FB, OutT>), dim3(tiles, (unsigned)batches), dim3(TW * 64), (TileGeom<FA, FB>::SMEM), st, g);
}

template <int FA, int FB>
void launch_fmt(const GemmArgs& g, int64_t batches, int c_dtype, hipStream_t st) {
    if (c_dtype == MPSA_BF16)        launch_one<FA, FB, __bf16>(g, batches, st);
    else if (c_dtype == MPSA_F8E5M2) launch_one<FA, FB, OutE5M2>(g, batches, st);
    else if (c_dtype == MPSA_F16)    launch_one<FA, FB, _Float16>(g, batches, st);
    else                             launch_one<FA, FB, float>(g, batches, st);
}

template <int FA>
void launch_b(const GemmArgs& g, int64_t batches, int fmt_b, int c_dtype, hipStream_t st) {
    if (fmt_b == MPSA_FMT_E2M1)      launch_fmt<FA, MPSA_FMT_E2M1>(g, batches, c_dtype, st);
    else if (fmt_b == MPSA_FMT_E4M3) launch_fmt<FA, MPSA_FMT_E4M3>(g, batches, c_dtype, st);
    else                             launch_fmt<FA, MPSA_FMT_E5M2>(g, batches, c_dtype, st);
}

}  // namespace

void gemm_tile_launch(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int c_dtype, hipStream_t st) {
    if (fmt_a == MPSA_FMT_E2M1)      launch_b<MPSA_FMT_E2M1>(g, batches, fmt_b, c_dtype, st);
    else if (fmt_a == MPSA_FMT_E4M3) launch_b<MPSA_FMT_E4M3>(g, batches, fmt_b, c_dtype, st);
    else                             launch_b<MPSA_FMT_E5M2>(g, batches, fmt_b, c_dtype, st);
}
