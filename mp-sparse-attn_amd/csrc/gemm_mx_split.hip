// Block-scaled NT matmul for products with too few output tiles to fill the chip (gfx950): the semantics of
// gemm_mx.hip for small M (a decode step, a short prompt) or a small matrix.
//
// What bounds such a product is latency and the vector memory path: 16 x 4096 x 4096 is 32 tiles of 128 x 128, each
// walking K through a two-stage pipeline at a memory round trip per stage (29 us for 9 MB of weights).  Here a workgroup
// owns a tile of a few 16 x 16 blocks and its waves SPLIT K between them.  A wave stages its own slices of K -- a ring of
// RING units of 256 elements, direct-to-LDS loads -- and nobody else reads them, so the loop has no barrier: a wave waits
// for its own oldest unit and goes on.  The waves' partial tiles are added through LDS at the end, in wave order, so
// results do not depend on timing.
//
// Loads go through LDS although every byte is used once: the vector memory path is several times faster when neighbouring
// lanes share 128-byte lines (8 rows x 128 B) than when they do not, which is what the matrix operand layout (neighbouring
// lanes = different rows) would ask for.  Straight into registers the same kernel took 6.0 us for 16 x 4096 x 4096, this way
// 3.3; 16 x 4096 x 14336 takes 5.8 us = 5.3 TB/s, what a copy reaches.  Clock stamps in a copy of this kernel: 2400 clocks to the
// last of the first requests, 520 a unit of 256 elements from then on (4 units a wave, and 14), 730 for adding up and storing.
//
// v_mfma_scale_f32_16x16x128_f8f6f4: lane (g = lane/16, r = lane%16) supplies 32 elements of row r of either operand and
// the E8M0 byte of MX block g of the 128-element step.  4-bit elements: the lane's four registers are block g.  8-bit
// elements: registers 0-3 hold bytes 16g.. of the step's first 64 and registers 4-7 the same of its second 64.  The
// result has row 4g + e of A and row r of B in register e.
#include "gemm_mx_args.h"
#include <cmath>
#include <type_traits>

namespace {

template <int FMT>
struct SplitOp {
    static constexpr bool FP4 = FMT == MPSA_FMT_E2M1;
    static constexpr int UNIT = FP4 ? 128 : 256;         // code bytes per row and unit of 256 elements
    static constexpr int LINES = UNIT / 128;             // images of 128 bytes a row
    static constexpr int BLOCK = 16 * UNIT;              // LDS bytes of 16 rows of a unit
    static constexpr int LOADS = 2 * LINES;              // direct-to-LDS instructions (8 rows x 128 B) for them
    // fragment of step k (0 / 1) of the unit: 16-byte piece c of row r sits at slot c ^ (r & 7) of its 128-byte row
    __device__ static __forceinline__ v8i frag(const uint8_t* img, int k, int g, int r) {
        if constexpr (FP4) {
            const v4i x = *reinterpret_cast<const v4i*>(img + r * 128 + (((4 * k + g) ^ (r & 7)) * 16));
            return (v8i){x[0], x[1], x[2], x[3], 0, 0, 0, 0};
        } else {
            const uint8_t* row = img + k * 2048 + r * 128;       // line k of the unit: the step's 128 bytes
            const v4i x = *reinterpret_cast<const v4i*>(row + ((g ^ (r & 7)) * 16));
            const v4i y = *reinterpret_cast<const v4i*>(row + (((4 + g) ^ (r & 7)) * 16));
            return (v8i){x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
        }
    }
};

template <int FA, int FB, int MB, int NB, int WAVES, int RING>
struct SplitGeom {
    static constexpr int UNIT = MB * SplitOp<FA>::BLOCK + NB * SplitOp<FB>::BLOCK;
    static constexpr int LOADS = MB * SplitOp<FA>::LOADS + NB * SplitOp<FB>::LOADS;      // a unit's code instructions
    static constexpr int SLOADS = MB + NB;                                               // a pair of units' scale instructions
    static constexpr int MINE = RING * UNIT + 2 * SLOADS * 256;                          // LDS of one wave: ring, scales of two pairs
    static constexpr int LD = 16 * NB + 4;                                               // floats per row of a partial tile
    static constexpr int PART = 16 * MB * LD * 4;
    static constexpr int SMEM = WAVES * (MINE > PART ? MINE : PART);
    static constexpr bool FITS = RING <= 3 && (RING - 1) * LOADS + SLOADS < 64 && SMEM <= 163840;
};

template <int N> __device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

template <int FA, int FB, typename OutT, int MB, int NB, int WAVES, int RING>
__global__ __launch_bounds__(WAVES * 64) void gemm_mx_split_kernel(GemmArgs a) {
    typedef SplitOp<FA> OA;
    typedef SplitOp<FB> OB;
    typedef SplitGeom<FA, FB, MB, NB, WAVES, RING> G;
    constexpr int TM = 16 * MB, TN = 16 * NB;
    static_assert(G::FITS, "ring too deep");
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r = lane & 15;
    // one contiguous range of tiles per XCD, all row tiles of a column tile next to each other: B is read by one L2 only
    const int tiles_m = (a.M + TM - 1) / TM, total = gridDim.x;
    int L = blockIdx.x;
    if ((total & 7) == 0) L = (L & 7) * (total >> 3) + (L >> 3);
    const int m0 = (L % tiles_m) * TM, n0 = (L / tiles_m) * TN;
    const int bz = blockIdx.y;
    const int bb = bz / a.heads_a, ha = bz - bb * a.heads_a;
    const int64_t zb = (int64_t)bb * a.heads_b + ha / (a.heads_a / a.heads_b);
    const int rowb_a = OA::FP4 ? a.K / 2 : a.K, rowb_b = OB::FP4 ? a.K / 2 : a.K;
    const int kblocks = a.K / 32, steps = a.K / 128;

    // tile bases (uniform); rows past the matrix are its last row
    const int last_a = a.M - 1 - m0, last_b = a.N - 1 - n0;
    const uint8_t* const ta = a.a + ((int64_t)bz * a.M + m0) * rowb_a;
    const uint8_t* const tb = a.b + (zb * a.N + n0) * rowb_b;
    const uint8_t *tsa = a.sa + (int64_t)bz * a.M * kblocks, *tsb = a.sb + zb * a.N * kblocks;
    // packed scales: chunks of 128 rows x 128 elements, a tile stays inside one row of chunks
    tsa += a.packed ? (int64_t)(m0 >> 7) * steps * 512 : (int64_t)m0 * kblocks;
    tsb += a.packed ? (int64_t)(n0 >> 7) * steps * 512 : (int64_t)n0 * kblocks;
    const int sstep = a.packed ? 512 : 4;                // from one step's scale word to the next
    auto scale_off = [&](int first, int row) {           // of row `row` of the tile that starts at row `first`
        const int x = (first & 127) + row;
        return a.packed ? (uint32_t)((x & 31) * 16 + (x >> 5) * 4) : (uint32_t)(row * kblocks);
    };
    // staging: lane offsets of rows 8q .. 8q+7 of a tile, 16-byte piece (lane & 7) ^ row & 7 of a 128-byte line
    const int lr = lane >> 3;
    const uint32_t piece = (uint32_t)(((lane & 7) ^ (lr & 7)) * 16);
    uint32_t ra[2 * MB], rb[2 * NB], rsa[MB], rsb[NB];
#pragma unroll
    for (int q = 0; q < 2 * MB; ++q) ra[q] = (uint32_t)min(8 * q + lr, last_a) * (uint32_t)rowb_a;
#pragma unroll
    for (int q = 0; q < 2 * NB; ++q) rb[q] = (uint32_t)min(8 * q + lr, last_b) * (uint32_t)rowb_b;
#pragma unroll
    for (int q = 0; q < MB; ++q) rsa[q] = scale_off(m0, min(16 * q + (lane >> 2), last_a));
#pragma unroll
    for (int q = 0; q < NB; ++q) rsb[q] = scale_off(n0, min(16 * q + (lane >> 2), last_b));

    // this wave's units: a contiguous share
    const int units = (steps + 1) / 2, share = (units + WAVES - 1) / WAVES;
    const int u0 = min(wave * share, units), n = min(u0 + share, units) - u0;

    uint8_t* const mine = smem + wave * G::MINE;
    uint8_t* const myscales = mine + RING * G::UNIT;
    // The t-th unit of the share -> ring slot.  Even units bring the scale words of their pair first: four words a row, four
    // neighbouring lanes on one line.  The last unit of
    // K % 256 == 128 is half a unit: pieces and words past a row's end are the row's last ones, and its second step is not
    // multiplied.
    auto issue = [&](int t, int slot, bool even) __attribute__((always_inline)) {
        if (even) {
            uint8_t* d = myscales + ((t >> 1) & 1) * G::SLOADS * 256;
            const uint32_t sk = (uint32_t)(min(2 * (u0 + t) + (lane & 3), steps - 1) * sstep);
#pragma unroll
            for (int q = 0; q < MB; ++q, d += 256) load_to_lds_uniform<4>(rsa[q] + sk, tsa, d);
#pragma unroll
            for (int q = 0; q < NB; ++q, d += 256) load_to_lds_uniform<4>(rsb[q] + sk, tsb, d);
        }
        uint8_t* d = mine + slot * G::UNIT;
        auto codes = [&](const uint8_t* base, const uint32_t* rows, int nq, int unit_bytes, int rowb) __attribute__((always_inline)) {
#pragma unroll
            for (int q = 0; q < nq / 2; ++q)
#pragma unroll
                for (int l = 0; l < unit_bytes / 128; ++l) {
                    const uint32_t k = (uint32_t)min((u0 + t) * unit_bytes + l * 128 + (int)piece, rowb - 16);
#pragma unroll
                    for (int x = 0; x < 2; ++x, d += 1024) load_to_lds_uniform<16>(rows[2 * q + x] + k, base, d);
                }
        };
        codes(ta, ra, 2 * MB, OA::UNIT, rowb_a);
        codes(tb, rb, 2 * NB, OB::UNIT, rowb_b);
    };

    v4f acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = (v4f){0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](int t, int slot) __attribute__((always_inline)) {
        const bool whole = 2 * (u0 + t) + 1 < steps;
        const uint8_t* ia = mine + slot * G::UNIT;
        const uint8_t* ib = ia + MB * OA::BLOCK;
        const uint8_t* is = myscales + ((t >> 1) & 1) * G::SLOADS * 256 + r * 16 + (t & 1) * 8;
        uint2 wa[MB], wb[NB];
#pragma unroll
        for (int i = 0; i < MB; ++i) wa[i] = *reinterpret_cast<const uint2*>(is + i * 256);
#pragma unroll
        for (int j = 0; j < NB; ++j) wb[j] = *reinterpret_cast<const uint2*>(is + (MB + j) * 256);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            if (k == 1 && !whole) break;
            v8i fa[MB], fb[NB];
#pragma unroll
            for (int i = 0; i < MB; ++i) fa[i] = OA::frag(ia + i * OA::BLOCK, k, g, r);
#pragma unroll
            for (int j = 0; j < NB; ++j) fb[j] = OB::frag(ib + j * OB::BLOCK, k, g, r);
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fa[i], fb[j], acc[i][j], FA, FB,
                                    0, (int)((k ? wa[i].y : wa[i].x) >> (8 * g)), 0, (int)((k ? wb[j].y : wb[j].x) >> (8 * g)));
        }
    };

#pragma unroll
    for (int x = 0; x < RING - 1; ++x)
        if (x < n) issue(x, x, (x & 1) == 0);
    int slot = 0;
    // one unit: the one RING - 1 later is requested, then everything up to this one is waited for -- what may still be on its
    // way are the code loads of the newer units and the scale loads of the even ones among them
    auto unit = [&](int t, auto odd_c) __attribute__((always_inline)) {
        constexpr int ODD = decltype(odd_c)::value;
        constexpr bool ahead_even = ((ODD + RING - 1) & 1) == 0;
        const int newer = n - 1 - t;
        if (newer >= RING - 1) {
            // the slot (and every other time the scale words) that is refilled now is the one that the unit before was read from:
            // those reads are back, and none is moved behind the loads, which no register orders after them
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            issue(t + RING - 1, slot == 0 ? RING - 1 : slot - 1, ahead_even);
            wait_loads<(RING - 1) * G::LOADS + ((RING - 1 + ODD) / 2) * G::SLOADS>();
        } else if (RING > 2 && newer == 1) {
            wait_loads<G::LOADS + ODD * G::SLOADS>();
        } else {
            wait_loads<0>();
        }
        multiply(t, slot);
        slot = slot == RING - 1 ? 0 : slot + 1;
    };
    for (int t = 0; t < n; t += 2) {
        unit(t, std::integral_constant<int, 0>{});
        if (t + 1 < n) unit(t + 1, std::integral_constant<int, 1>{});
    }

    // ---- add the partial tiles, in wave order ----
    __syncthreads();
    float* const part = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[wave * (G::PART / 4) + (16 * i + 4 * g + e) * G::LD + 16 * j + r] = acc[i][j][e];
    __syncthreads();
    OutT* c = static_cast<OutT*>(a.c) + (int64_t)bz * a.M * a.ldc;
    for (int x = tid; x < TM * TN; x += WAVES * 64) {
        const int row = x / TN, col = x % TN;
        float v = part[row * G::LD + col];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v += part[w * (G::PART / 4) + row * G::LD + col];
        if (row <= last_a && col <= last_b) c[(int64_t)(m0 + row) * a.ldc + n0 + col] = cvt_out<OutT>(v);
    }
}

template <int FA, int FB, typename OutT, int MB, int NB, int WAVES, int RING>
struct SplitLds {
    static constexpr int smem = SplitGeom<FA, FB, MB, NB, WAVES, RING>::SMEM;
    static inline const bool registered =
        mpsa_register_lds_kernel(reinterpret_cast<const void*>(gemm_mx_split_kernel<FA, FB, OutT, MB, NB, WAVES, RING>), smem);
};

template <int FA, int FB, typename OutT, int MB, int NB, int WAVES, int RING>
void launch_tile(const GemmArgs& g, int64_t batches, hipStream_t st) {
    typedef SplitLds<FA, FB, OutT, MB, NB, WAVES, RING> L;
    if (!L::registered) return;
    const int64_t tiles = (int64_t)((g.M + 16 * MB - 1) / (16 * MB)) * ((g.N + 16 * NB - 1) / (16 * NB));
    hipLaunchKernelGGL((gemm_mx_split_kernel<FA, FB, OutT, MB, NB, WAVES, RING>), dim3((unsigned)tiles, (unsigned)batches), dim3(WAVES * 64), L::smem, st, g);
}

// Waves per workgroup and ring depth of a tile: as many bytes on their way as two workgroups' LDS allows where the tile is
// small, one workgroup's where it is not.  Measured over 20 shapes from 1 x 1024 x 4096 to 1408^3: the best or within 6 % of
// it, of the combinations that fit.
constexpr int config(int mb, int nb, bool a4, bool b4) {
    const int blocks = 10 * mb + nb, fours = a4 + b4;
    if (blocks == 11) return 43;
    if (blocks == 12) return 42;
    if (blocks == 14) return fours ? 42 : 32;
    if (blocks == 22) return fours ? 42 : 22;
    if (blocks == 24) return b4 ? 42 : 32;
    return fours == 2 ? 42 : fours ? 32 : 22;
}

template <int FA, int FB, typename OutT>
void launch_out(const GemmArgs& g, int64_t batches, int tile, hipStream_t st) {
    constexpr bool A4 = FA == MPSA_FMT_E2M1, B4 = FB == MPSA_FMT_E2M1;
#define MPSA_SPLIT_TILE(mb, nb) \
    case 10 * mb + nb: launch_tile<FA, FB, OutT, mb, nb, config(mb, nb, A4, B4) / 10, config(mb, nb, A4, B4) % 10>(g, batches, st); break
    switch (tile) {
        MPSA_SPLIT_TILE(1, 1);
        MPSA_SPLIT_TILE(1, 2);
        MPSA_SPLIT_TILE(1, 4);
        MPSA_SPLIT_TILE(2, 2);
        MPSA_SPLIT_TILE(2, 4);
        MPSA_SPLIT_TILE(4, 4);
    }
#undef MPSA_SPLIT_TILE
}

template <int FA, int FB>
void launch_fmt(const GemmArgs& g, int64_t batches, int tile, int c_dtype, hipStream_t st) {
    if (c_dtype == MPSA_BF16)        launch_out<FA, FB, __bf16>(g, batches, tile, st);
    else if (c_dtype == MPSA_F8E5M2) launch_out<FA, FB, OutE5M2>(g, batches, tile, st);
    else if (c_dtype == MPSA_F16)    launch_out<FA, FB, _Float16>(g, batches, tile, st);
    else                             launch_out<FA, FB, float>(g, batches, tile, st);
}

template <int FA>
void launch_b(const GemmArgs& g, int64_t batches, int tile, int fmt_b, int c_dtype, hipStream_t st) {
    if (fmt_b == MPSA_FMT_E2M1)      launch_fmt<FA, MPSA_FMT_E2M1>(g, batches, tile, c_dtype, st);
    else if (fmt_b == MPSA_FMT_E4M3) launch_fmt<FA, MPSA_FMT_E4M3>(g, batches, tile, c_dtype, st);
    else                             launch_fmt<FA, MPSA_FMT_E5M2>(g, batches, tile, c_dtype, st);
}

}  // namespace

// Workgroups of a tile that share a CU: its LDS holds so many.
template <bool A4, bool B4, int MB, int NB>
constexpr int places_of() {
    constexpr int c = config(MB, NB, A4, B4);
    return 163840 / SplitGeom<A4 ? MPSA_FMT_E2M1 : MPSA_FMT_E4M3, B4 ? MPSA_FMT_E2M1 : MPSA_FMT_E4M3, MB, NB, c / 10, c % 10>::SMEM;
}
template <bool A4, bool B4>
int places_of(int tile) {
    switch (tile) {
        case 11: return places_of<A4, B4, 1, 1>();
        case 12: return places_of<A4, B4, 1, 2>();
        case 14: return places_of<A4, B4, 1, 4>();
        case 22: return places_of<A4, B4, 2, 2>();
        case 24: return places_of<A4, B4, 2, 4>();
        default: return places_of<A4, B4, 4, 4>();
    }
}

// Estimated microseconds of a product on this kernel with its best tile, fitted as choose() in gemm_mx.hip says.  A workgroup costs
// by its blocks (adding up the waves' sums) and rows, and by its rows times K (what it brings into LDS; `tile`: how much more than the
// others).  Workgroups that share a CU take longer for the traffic alone (with one power for both parts, 8 x 512 x 128 x 9344, 8-bit,
// took 2 x 2 blocks and 29.8 us, 2 x 4 blocks 21.8), and it is the CU with the most of them that counts (`whole`); where there are
// more than places, whole rounds.
double gemm_split_cost(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int* tile) {
    const bool a4 = fmt_a == MPSA_FMT_E2M1, b4 = fmt_b == MPSA_FMT_E2M1;
    static const int TILES[6] = {11, 12, 14, 22, 24, 44};
    struct Fit { double start, block, piece, row, rounds, whole, deep, tile[6]; };
    static const Fit FIT[3] = {{1.984, 0.001, 0.336, 0.714, 1.746, 1.151, 1.058, {-0.151, 0.021, 0.186, -0.228, -0.06, 0.036}},
                               {1.889, 0.044, 0.26, 0.558, 1.47, 2.106, 0.864, {-0.029, -0.006, 0.16, -0.285, -0.054, -0.024}},
                               {1.803, 0.124, 0.277, 0.304, 1.513, 1.228, 0.934, {0.072, 0.065, 0.059, -0.049, -0.025, 0.2}}};
    const Fit& f = FIT[a4 && b4 ? 0 : a4 || b4 ? 1 : 2];
    double best = 0.0;
    for (int i = 0; i < 6; ++i) {
        const int t = TILES[i], mb = t / 10, nb = t % 10;
        const int places = a4 ? (b4 ? places_of<true, true>(t) : places_of<true, false>(t)) : b4 ? places_of<false, true>(t) : places_of<false, false>(t);
        const double w = (double)((g.M + 16 * mb - 1) / (16 * mb)) * ((g.N + 16 * nb - 1) / (16 * nb)) * (double)batches / 256.0;      // workgroups per CU
        const double row = mb * (a4 ? 0.5 : 1.0) + nb * (b4 ? 0.5 : 1.0);
        auto shared = [&](double x) { return x > 1.0 ? pow(f.whole * ceil(x) + (1.0 - f.whole) * x, f.deep) : 1.0; };
        double fixed = 1.0, load = shared(w);
        if (w > places) {
            const double full = floor(w / places), rest = w - full * places;
            fixed += f.rounds * (ceil(w / places) - 1.0);
            load += f.rounds * (full * pow(places, f.deep) + (rest > 0.0 ? shared(rest) : 0.0) - load);
        }
        const double cost = f.start + (f.block * mb * nb + f.row * row) * fixed + f.piece * (1.0 + f.tile[i]) * row * g.K / 1024.0 * load;
        if (best == 0.0 || cost < best) {
            best = cost;
            *tile = t;
        }
    }
    return best;
}

void gemm_split_launch(const GemmArgs& g, int64_t batches, int tile, int fmt_a, int fmt_b, int c_dtype, hipStream_t st) {
    if (fmt_a == MPSA_FMT_E2M1)      launch_b<MPSA_FMT_E2M1>(g, batches, tile, fmt_b, c_dtype, st);
    else if (fmt_a == MPSA_FMT_E4M3) launch_b<MPSA_FMT_E4M3>(g, batches, tile, fmt_b, c_dtype, st);
    else                             launch_b<MPSA_FMT_E5M2>(g, batches, tile, fmt_b, c_dtype, st);
}
