// Block-scaled NT matmul for gfx950: the entry points and the choice between the kernels -- 256 x 256 tiles
// (gemm_mx_kernel.h, here and in gemm_mx_edge.hip), 128 x 128 tiles (gemm_mx_tile.hip), tiles of a few 16 x 16 blocks with
// K split between the waves (gemm_mx_split.hip) and the general kernel below, which takes K % 128 == 64 alone and is one of the
// choices elsewhere: a few tiles past a whole number of 256, and short K.  Score products of attention (K = 128) with 16-bit results
// have a kernel of their own (gemm_mx_stage.hip).
#include "gemm_mx_kernel.h"
#include <cmath>

namespace {

// ---- general kernel: any M and N (edge tiles masked), operands of different element formats ----
// The reference's kernel tiles 128 x 256 with masked edges (ours/block_scaled_matmul.py:154-267) and takes the two
// operands' element widths separately (ELEM_PER_BYTE_A / ELEM_PER_BYTE_B, "mixed" = 8-bit A x 4-bit B,
// ours/block_scaled_matmul.py:318-324).  This kernel takes every shape, also what the others do not (K % 128 == 64, whose scale rows are two-byte aligned only): a workgroup of
// four waves owns a 128 x 128 tile, a wave 64 x 64 (2 x 2 accumulators), up to three workgroups share a CU.  K advances
// 128 elements per stage (two matrix-instruction steps; 64 code bytes per row of a 4-bit operand, 128 of an 8-bit
// one): the stage's codes travel L2 -> LDS with direct-to-LDS loads into one of two buffers while the other is
// multiplied, rows XOR-swizzled as in the 256 x 256 kernel; rows past M or N are fetched from the last valid row and
// never stored.  The four scale bytes a row has per stage come straight from global memory as one word, a stage
// ahead (byte by byte when K is not a multiple of 128: the last stage is then half a stage).  Each operand's
// registers follow its own format's layout (4-bit: the lane half's registers are MX block h of the step; 8-bit:
// registers 0-3 of both halves are block 0, 4-7 block 1).
// (EdgeOp: gemm_mx_args.h)

// scale byte of row `row`, MX block kb: row-major [rows, K/32] or the packed [rows/128, K/128, 32, 4, 4] form
__device__ __forceinline__ int load_scale(const uint8_t* s, int row, int kb, int kblocks, bool packed) {
    if (!packed) return s[(int64_t)row * kblocks + kb];
    const int64_t chunk = (int64_t)(row >> 7) * (kblocks >> 2) + (kb >> 2);
    return s[chunk * 512 + (row & 31) * 16 + ((row >> 5) & 3) * 4 + (kb & 3)];
}

template <int FA, int FB>
constexpr int general_smem() { return 2 * (EdgeOp<FA>::BYTES + EdgeOp<FB>::BYTES); }
static_assert(4 * rows16_bytes<2>() <= general_smem<MPSA_FMT_E2M1, MPSA_FMT_E2M1>(), "room for the results on their way out");

// (Asked for three workgroups a CU the compiler takes no fewer registers -- 134 to 157 -- but keeps the loads of a stage and the
// reads of the one before further apart: 4000 x 4000 x 4096, 8-bit x 4-bit, 109 -> 94 us, 2100 x 2100 x 1024, 8-bit, 18.1 ->
// 16.9, 4-bit 15.3 -> 14.9, K = 128 the same.  Four need scratch memory with 4-bit codes and take 4 to 7 % longer.)
template <int FA, int FB, typename OutT>
__global__ __launch_bounds__(256, 3) void gemm_mx_general_kernel(GemmArgs g) {
    typedef EdgeOp<FA> OA;
    typedef EdgeOp<FB> OB;
    constexpr int STAGE = OA::BYTES + OB::BYTES;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int h = lane >> 5, r = lane & 31;
    const int rowb_a = OA::FP4 ? g.K / 2 : g.K;
    const int rowb_b = OB::FP4 ? g.K / 2 : g.K;
    const int kblocks = g.K / 32;
    const int tiles_n = (g.N + 127) / 128;
    const int tm0 = (blockIdx.x / tiles_n) * 128, tn0 = (blockIdx.x % tiles_n) * 128;   // the workgroup's tile
    const int m0 = tm0 + wm * 64, n0 = tn0 + wn * 64;                                   // the wave's
    const int bz = blockIdx.y;
    const int bb = bz / g.heads_a, ha = bz - bb * g.heads_a;
    const int64_t zb = (int64_t)bb * g.heads_b + ha / (g.heads_a / g.heads_b);
    const uint8_t* a = g.a + ((int64_t)bz * g.M + tm0) * rowb_a;         // the tile's first rows: lane offsets stay below 2^31
    const uint8_t* b = g.b + (zb * g.N + tn0) * rowb_b;
    const uint8_t* sa = g.sa + (int64_t)bz * g.M * kblocks;
    const uint8_t* sb = g.sb + zb * g.N * kblocks;
    const int steps = g.K / 64;                          // matrix-instruction steps
    const int nstages = (steps + 1) / 2;                 // the last stage is half a stage when `steps` is odd
    const bool words = (g.K % 128) == 0;                 // a row's four scale bytes of a stage are one aligned word

    // ---- staging: lane offsets of this wave's pieces (rows past the matrix clamp to its last row) ----
    uint32_t loa[OA::IPW], lob[OB::IPW];
    bool firsta[OA::IPW], firstb[OB::IPW];               // the piece lies in the stage's first half (first step)
#pragma unroll
    for (int c = 0; c < OA::IPW; ++c) {
        const int p = (wave * OA::IPW + c) * 64 + lane;
        const int row = p / OA::CPR, cb = (p % OA::CPR) ^ OA::swz(row);
        loa[c] = (uint32_t)min(row, g.M - 1 - tm0) * (uint32_t)rowb_a + cb * 16;
        firsta[c] = cb < OA::CPR / 2;
    }
#pragma unroll
    for (int c = 0; c < OB::IPW; ++c) {
        const int p = (wave * OB::IPW + c) * 64 + lane;
        const int row = p / OB::CPR, cb = (p % OB::CPR) ^ OB::swz(row);
        lob[c] = (uint32_t)min(row, g.N - 1 - tn0) * (uint32_t)rowb_b + cb * 16;
        firstb[c] = cb < OB::CPR / 2;
    }
    auto issue = [&](int s) __attribute__((always_inline)) {
        uint8_t* st = smem + (s & 1) * STAGE;
        const bool half = 2 * s + 1 >= steps;            // only the stage's first step exists
#pragma unroll
        for (int c = 0; c < OA::IPW; ++c)
            if (!half || firsta[c]) load_to_lds<16>(loa[c], a + (int64_t)s * OA::ROW, st + (wave * OA::IPW + c) * 1024);
#pragma unroll
        for (int c = 0; c < OB::IPW; ++c)
            if (!half || firstb[c]) load_to_lds<16>(lob[c], b + (int64_t)s * OB::ROW, st + OA::BYTES + (wave * OB::IPW + c) * 1024);
    };

    // ---- this lane's rows (for the scale bytes) and the scale words of a stage ----
    int ra[2], rb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        ra[i] = min(m0 + i * 32 + r, g.M - 1);
        rb[i] = min(n0 + i * 32 + r, g.N - 1);
    }
    auto scale_word = [&](const uint8_t* sc, int row, int s) __attribute__((always_inline)) -> uint32_t {
        if (words) {
            const int64_t off = g.packed ? ((int64_t)(row >> 7) * (kblocks >> 2) + s) * 512 + (row & 31) * 16 + ((row >> 5) & 3) * 4
                                         : (int64_t)row * kblocks + 4 * s;
            return *reinterpret_cast<const uint32_t*>(sc + off);
        }
        uint32_t w = 0;                                  // K % 128 == 64 (row-major scales only): byte by byte
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (4 * s + q < kblocks) w |= (uint32_t)load_scale(sc, row, 4 * s + q, kblocks, false) << (8 * q);
        return w;
    };
    uint32_t wa[2], wb[2], na[2] = {0, 0}, nb[2] = {0, 0};
    auto fetch_scales = [&](int s, uint32_t (&xa)[2], uint32_t (&xb)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            xa[i] = scale_word(sa, ra[i], s);
            xb[i] = scale_word(sb, rb[i], s);
        }
    };

    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    issue(0);
    fetch_scales(0, wa, wb);
    for (int s = 0; s < nstages; ++s) {
        // stage s has landed for every wave, and every wave is through with the buffer stage s + 1 goes to
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0070);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        if (s + 1 < nstages) {
            issue(s + 1);
            fetch_scales(s + 1, na, nb);
        }
        const uint8_t* ia = smem + (s & 1) * STAGE;
        const uint8_t* ib = ia + OA::BYTES;
        const int nk = min(2, steps - 2 * s);
        for (int k = 0; k < nk; ++k) {
            v8i fa[2], fb[2];
            int ca[2], cb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                fa[i] = OA::frag(ia, wm * 64 + i * 32 + r, k, h);
                fb[i] = OB::frag(ib, wn * 64 + i * 32 + r, k, h);
                ca[i] = (int)(wa[i] >> (8 * (2 * k + h)));       // the matrix instruction takes the low byte
                cb[i] = (int)(wb[i] >> (8 * (2 * k + h)));
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i], fb[j], acc[i][j], FA, FB, 0, ca[i], 0, cb[j]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) { wa[i] = na[i]; wb[i] = nb[i]; }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                  // no direct-to-LDS load may outlive the workgroup

    // accumulator register e of lane (h, r) is C[8*(e/4) + 4*h + e%4][r] of its 32 x 32 block
    OutT* c = static_cast<OutT*>(g.c) + (int64_t)bz * g.M * g.ldc;
    if constexpr (sizeof(OutT) == 2) {
        if (rows16_aligned(g)) {
            __syncthreads();                             // everybody has read the last stage
#pragma unroll
            for (int i = 0; i < 2; ++i)
                store_rows16<2, OutT, true>(acc[i], smem + wave * rows16_bytes<2>(), c, g.ldc, m0 + i * 32, n0, g.M, g.N, lane);
            return;
        }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int col = n0 + j * 32 + r;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int row = m0 + i * 32 + 8 * (e >> 2) + 4 * h + (e & 3);
                if (row < g.M && col < g.N) c[(int64_t)row * g.ldc + col] = cvt_out<OutT>(acc[i][j][e]);
            }
        }
}

template <int FA, int FB, typename OutT>
struct GeneralLds {
    static inline const bool registered =
        mpsa_register_lds_kernel(reinterpret_cast<const void*>(gemm_mx_general_kernel<FA, FB, OutT>), general_smem<FA, FB>());
};

template <int FA, int FB, typename OutT>
void launch_general_kernel(const GemmArgs& g, dim3 grid, hipStream_t st) {
    if (!GeneralLds<FA, FB, OutT>::registered) return;
    constexpr int lds = general_smem<FA, FB>();
    hipLaunchKernelGGL((gemm_mx_general_kernel<FA, FB, OutT>), grid, dim3(256), lds, st, g);
}

template <int FA, int FB>
void launch_general_out(const GemmArgs& g, int c_dtype, dim3 grid, hipStream_t st) {
    if (c_dtype == MPSA_BF16)        launch_general_kernel<FA, FB, __bf16>(g, grid, st);
    else if (c_dtype == MPSA_F8E5M2) launch_general_kernel<FA, FB, OutE5M2>(g, grid, st);
    else if (c_dtype == MPSA_F16)    launch_general_kernel<FA, FB, _Float16>(g, grid, st);
    else                             launch_general_kernel<FA, FB, float>(g, grid, st);
}

template <int FA>
void launch_general_b(const GemmArgs& g, int fmt_b, int c_dtype, dim3 grid, hipStream_t st) {
    if (fmt_b == MPSA_FMT_E2M1)      launch_general_out<FA, MPSA_FMT_E2M1>(g, c_dtype, grid, st);
    else if (fmt_b == MPSA_FMT_E4M3) launch_general_out<FA, MPSA_FMT_E4M3>(g, c_dtype, grid, st);
    else                             launch_general_out<FA, MPSA_FMT_E5M2>(g, c_dtype, grid, st);
}

void launch_general(const GemmArgs& g, int fmt_a, int fmt_b, int c_dtype, dim3 grid, hipStream_t st) {
    if (fmt_a == MPSA_FMT_E2M1)      launch_general_b<MPSA_FMT_E2M1>(g, fmt_b, c_dtype, grid, st);
    else if (fmt_a == MPSA_FMT_E4M3) launch_general_b<MPSA_FMT_E4M3>(g, fmt_b, c_dtype, grid, st);
    else                             launch_general_b<MPSA_FMT_E5M2>(g, fmt_b, c_dtype, grid, st);
}

// MPSA_GEMM_GENERAL=1 in the environment sends every shape to the general kernel (cross-checking)
bool force_general() {
    static const bool on = [] {
        const char* v = getenv("MPSA_GEMM_GENERAL");
        return v && v[0] == '1';
    }();
    return on;
}

template <int FMT, int FMTB, typename OutT>
void launch_one(const GemmArgs& g, dim3 grid, hipStream_t st) {
    if constexpr (FMT == MPSA_FMT_E2M1) {
        if (g.K % 256) return launch_kernel<FMT, FMTB, OutT, false, true, false, true>(g, grid, st);      // packed scales
    }
    if (g.packed)            launch_kernel<FMT, FMTB, OutT, false, true, false>(g, grid, st);
    else if (g.K % 512 == 0) launch_kernel<FMT, FMTB, OutT, false, false, false>(g, grid, st);
    else                     launch_kernel<FMT, FMTB, OutT, true, false, false>(g, grid, st);
}

template <int FMT, int FMTB>
void launch_fmt(const GemmArgs& g, int c_dtype, dim3 grid, hipStream_t st) {
    if (c_dtype == MPSA_BF16)      launch_one<FMT, FMTB, __bf16>(g, grid, st);
    else if (c_dtype == MPSA_F8E5M2) launch_one<FMT, FMTB, OutE5M2>(g, grid, st);
    else if (c_dtype == MPSA_F16)  launch_one<FMT, FMTB, _Float16>(g, grid, st);
    else                           launch_one<FMT, FMTB, float>(g, grid, st);
}

}  // namespace

static bool known_fmt(int f) { return f == MPSA_FMT_E2M1 || f == MPSA_FMT_E4M3 || f == MPSA_FMT_E5M2; }

// The kernel of a product: what the caller named (MPSA_GEMM_*), if it takes the shape, or the one with the least estimated time
// (microseconds, from measurements of every kernel at 18 000 shapes in three types, one product or up to 32, M from 1 to 8192, N from
// 16 to 16384, K from 128 to 14336, weights not all in the cache).  The constants are those with the least time lost by the choice,
// losses past 5 % and past what an earlier choice lost counted more; over 7500 others it costs 0.5 % over always taking the fastest, and
// more than 10 % at 1.4 % of them.  Constants with the least error of the estimates cost 0.8 % and 2.5 % (619 x 6784 x 3072, 4-bit,
// 25.7 -> 34.6 us; 821 x 11136 x 1024, 8-bit, 22.0 -> 28.1), from K = 256 on a fit to 820 single products 1.3 % and 4.5 %, one to 130
// shapes 5.5 % and 20 %.
// What is left is luck: with a few workgroups more than CUs, 8-bit tiles of 2 x 2 blocks take 1.8 or 2.4 us per 1024 of K.
// A ring tile costs a fixed part -- pipeline fill, epilogue -- and one per 1024 of K; a started round of 256 tiles counts whole, at a
// clock that falls as the chip fills.  The general kernel shares a CU between up to three tiles and has no rounds: it is the
// fastest a few tiles past a whole number of them, and where K is short; with long K it falls behind, as its tiles pass the L2 by
// (4140 x 12160 x 10240, 8-bit x 4-bit, 980 us, on 256 x 256 tiles 427).  The lines fall near M = 256 (4096-wide layer, K = 4096),
// where a 128-wide tile takes over from the 16-row blocks, and near 2000 rows, where 256-wide tiles fill the chip.
static int64_t blocks16(const GemmArgs& g, int64_t batches) { return (int64_t)((g.M + 15) / 16) * ((g.N + 15) / 16) * batches; }

static int choose(int kernel, const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b) {
    const double K = g.K;
    const bool mixed = fmt_a != MPSA_FMT_E2M1 && fmt_b == MPSA_FMT_E2M1;
    const int kind = fmt_a == MPSA_FMT_E2M1 && fmt_b == MPSA_FMT_E2M1 ? 0 : mixed ? 1 : 2;
    auto tiles = [&](int edge) { return (double)((g.M + edge - 1) / edge) * (double)((g.N + edge - 1) / edge) * (double)batches; };
    // ragged 4-bit products that end in half a unit: from a quarter of the chip on (the estimates choose it from 130 tiles on)
    const bool half = kind == 0 && g.K % 256 && (g.M % BM || g.N % BN);
    const bool staged = g.K % 128 == 0 && (fmt_a == fmt_b || mixed) && (!half || tiles(256) >= 64.0);
    int tile = 0;
    switch (kernel) {
        case MPSA_GEMM_AUTO: break;
        case MPSA_GEMM_GENERAL: return kernel;
        case MPSA_GEMM_SPLIT: case MPSA_GEMM_SPLIT_TILE(1, 1): case MPSA_GEMM_SPLIT_TILE(1, 2): case MPSA_GEMM_SPLIT_TILE(1, 4):
        case MPSA_GEMM_SPLIT_TILE(2, 2): case MPSA_GEMM_SPLIT_TILE(2, 4): case MPSA_GEMM_SPLIT_TILE(4, 4):
            if (g.K % 128) return mpsa_fail(MPSA_EUNSUPPORTED, "gemm: this kernel needs K %% 128 == 0 (got %d)", g.K);
            if (kernel == MPSA_GEMM_SPLIT) (void)gemm_split_cost(g, batches, fmt_a, fmt_b, &tile);
            return kernel == MPSA_GEMM_SPLIT ? MPSA_GEMM_SPLIT_TILE(tile / 10, tile % 10) : kernel;
        case MPSA_GEMM_TILE128:
            if (g.K % 128) return mpsa_fail(MPSA_EUNSUPPORTED, "gemm: this kernel needs K %% 128 == 0 (got %d)", g.K);
            return kernel;
        case MPSA_GEMM_TILE256:
            if (!staged) return mpsa_fail(MPSA_EUNSUPPORTED, "gemm: the 256 x 256 kernel needs one format or 8-bit A with 4-bit B, and K %% 128 == 0; ragged 4-bit products with K %% 256 == 128 also 64 tiles");
            return kernel;
        default: return mpsa_fail(MPSA_EINVAL, "gemm: unknown kernel %d", kernel);
    }
    if (g.K % 128 || force_general()) return MPSA_GEMM_GENERAL;
    if (g.K == 128) {
        // one stage: a ring gains nothing (the fastest at none of 560 shapes), and the tiles that split K, all of whose waves but one
        // idle, are the fastest while two workgroups a CU hold them (their time over the general kernel's, 1024 to 2048 blocks: 0.87,
        // 2048 to 4096: 1.23)
        if (blocks16(g, batches) > 2048) return MPSA_GEMM_GENERAL;
        (void)gemm_split_cost(g, batches, fmt_a, fmt_b, &tile);
        return MPSA_GEMM_SPLIT_TILE(tile / 10, tile % 10);
    }
    struct Ring { double start, round, per_1024, empty; };                   // empty: share of per_1024 at an empty chip
    static const Ring RING[2][3] = {{{0.0, 5.519, 2.87, 1.11}, {2.133, 3.158, 4.755, 0.635}, {0.0, 5.366, 5.753, 0.499}},
                                    {{2.653, 6.175, 7.599, 0.971}, {2.78, 3.679, 12.764, 0.854}, {0.0, 7.642, 12.526, 1.136}}};
    struct Shared { double start, tile, least, base, per_1024, deep; };      // tile, per_1024: for 256 tiles; deep: more of it at K = 8192
    static const Shared SHARED[3] = {{1.949, 0.002, 7.953, 4.391, 4.181, 0.539}, {2.678, 0.022, 10.204, 2.743, 3.158, 3.752}, {2.015, 1.046, 11.081, 0.008, 5.136, 2.689}};
    auto ring = [&](int which, int edge) {
        const Ring& r = RING[which][kind];
        const double rounds = ceil(tiles(edge) / 256.0), clock = r.empty + (1.0 - r.empty) * tiles(edge) / (256.0 * rounds);
        return r.start + rounds * (r.round + r.per_1024 * clock * K / 1024.0);
    };
    const Shared& sh = SHARED[kind];
    const double load = tiles(128) / 256.0, slope = sh.base + sh.per_1024 * load * (1.0 + sh.deep * (K < 8192.0 ? K / 8192.0 : 1.0));
    const double general = sh.start + sh.tile * load + K / 1024.0 * (slope > sh.least ? slope : sh.least);
    const double cost16 = gemm_split_cost(g, batches, fmt_a, fmt_b, &tile), cost128 = ring(0, 128), cost256 = staged ? ring(1, 256) : 1e300;
    const double least = fmin(fmin(cost16, cost128), cost256);
    if (general < least) return MPSA_GEMM_GENERAL;
    return cost16 == least ? MPSA_GEMM_SPLIT_TILE(tile / 10, tile % 10) : cost128 == least ? MPSA_GEMM_TILE128 : MPSA_GEMM_TILE256;
}

static int check_shape(int fmt_a, int fmt_b, int64_t batch, int64_t heads_a, int64_t heads_b, int64_t M, int64_t N, int64_t K, bool packed) {
    if (!known_fmt(fmt_a) || !known_fmt(fmt_b)) return mpsa_fail(MPSA_EINVAL, "gemm: unknown format %d / %d", fmt_a, fmt_b);
    if (M <= 0 || N <= 0 || K <= 0) return mpsa_fail(MPSA_EINVAL, "gemm: bad shape");
    if (batch <= 0 || heads_a <= 0 || heads_b <= 0 || heads_a % heads_b) return mpsa_fail(MPSA_EINVAL, "gemm: bad batch shape (batch=%lld heads_a=%lld heads_b=%lld)", (long long)batch, (long long)heads_a, (long long)heads_b);
    if (K % 64) return mpsa_fail(MPSA_EUNSUPPORTED, "gemm: K must be a multiple of 64 (got %lld)", (long long)K);
    if (packed && (M % 128 || N % 128 || K % 128)) return mpsa_fail(MPSA_EUNSUPPORTED, "gemm: packed scales need M, N and K in multiples of 128 (got %lld,%lld,%lld)", (long long)M, (long long)N, (long long)K);
    if (M > (1 << 30) || N > (1 << 30) || K > (1 << 24) || ((M + 127) / 128) * ((N + 127) / 128) > (int64_t(1) << 30) || batch * heads_a > 65535)
        return mpsa_fail(MPSA_EUNSUPPORTED, "gemm: shape too large");
    return MPSA_OK;
}

static int gemm_entry(int kernel, const uint8_t* a, const uint8_t* sa, int fmt_a, const uint8_t* b, const uint8_t* sb, int fmt_b, bool packed,
                      int64_t batch, int64_t heads_a, int64_t heads_b, int64_t M, int64_t N, int64_t K,
                      void* c, int c_dtype, int64_t ldc, mpsa_stream_t stream) {
    if (!a || !sa || !b || !sb || !c) return mpsa_fail(MPSA_EINVAL, "gemm: null pointer");
    if (c_dtype != MPSA_BF16 && c_dtype != MPSA_F16 && c_dtype != MPSA_F32 && c_dtype != MPSA_F8E5M2) return mpsa_fail(MPSA_EINVAL, "gemm: unsupported output dtype %d", c_dtype);
    int rc = check_shape(fmt_a, fmt_b, batch, heads_a, heads_b, M, N, K, packed);
    if (rc != MPSA_OK) return rc;
    if (ldc < N) return mpsa_fail(MPSA_EINVAL, "gemm: bad shape");
    if (!mpsa_aligned16(a) || !mpsa_aligned16(b) || (reinterpret_cast<uintptr_t>(sa) & 3) || (reinterpret_cast<uintptr_t>(sb) & 3))
        return mpsa_fail(MPSA_EALIGN, "gemm: codes must be 16-byte and scales 4-byte aligned");
    if (packed && (!mpsa_aligned16(sa) || !mpsa_aligned16(sb))) return mpsa_fail(MPSA_EALIGN, "gemm: packed scales must be 16-byte aligned");
    GemmArgs g;
    g.a = a; g.sa = sa; g.b = b; g.sb = sb; g.c = c; g.ldc = ldc;
    g.M = (int)M; g.N = (int)N; g.K = (int)K;
    g.heads_a = (int)heads_a; g.heads_b = (int)heads_b;
    g.packed = packed ? 1 : 0;
    hipStream_t st = (hipStream_t)stream;
    const int64_t batches = batch * heads_a;
    // From 1024 blocks of 16 x 16 on (the time of the tiles that split K over this kernel's, 768 to 1024 blocks: 0.99, 1024 to 1536:
    // 1.10; below 256 blocks 0.81: 16 x 4096, 8-bit x 4-bit, 3.2 and 3.9 us, 4096 x 16, 4-bit, 3.2 and 4.2).
    const bool stage = kernel == MPSA_GEMM_AUTO && !force_general() && gemm_stage_takes(g, fmt_a, fmt_b, c_dtype) && blocks16(g, batches) > 1024;
    kernel = stage ? MPSA_GEMM_GENERAL : choose(kernel, g, batches, fmt_a, fmt_b);
    if (kernel < 0) return kernel;
    rc = mpsa_ensure_init();
    if (rc != MPSA_OK) return rc;
    if (stage) {
        gemm_stage_launch(g, batches, fmt_a, fmt_b, c_dtype, st);
        MPSA_CHECK_LAUNCH("gemm");
        return MPSA_OK;
    }
    if (kernel == MPSA_GEMM_GENERAL) {
        dim3 grid((unsigned)(((M + 127) / 128) * ((N + 127) / 128)), (unsigned)batches);
        launch_general(g, fmt_a, fmt_b, c_dtype, grid, st);
    } else if (kernel == MPSA_GEMM_TILE128) {
        gemm_tile_launch(g, batches, fmt_a, fmt_b, c_dtype, st);
    } else if (kernel != MPSA_GEMM_TILE256) {
        gemm_split_launch(g, batches, kernel, fmt_a, fmt_b, c_dtype, st);
    } else if (M % BM || N % BN || (!packed && fmt_a == MPSA_FMT_E2M1 && K % 256)) {
        gemm_edge_launch(g, batches, fmt_a, fmt_b, c_dtype, st);
    } else {
        const bool mixed = fmt_a != fmt_b;
        dim3 grid((unsigned)((M / BM) * (N / BN)), (unsigned)batches);
        if (fmt_a == MPSA_FMT_E2M1)      launch_fmt<MPSA_FMT_E2M1, MPSA_FMT_E2M1>(g, c_dtype, grid, st);
        else if (fmt_a == MPSA_FMT_E4M3) mixed ? launch_fmt<MPSA_FMT_E4M3, MPSA_FMT_E2M1>(g, c_dtype, grid, st) : launch_fmt<MPSA_FMT_E4M3, MPSA_FMT_E4M3>(g, c_dtype, grid, st);
        else                             mixed ? launch_fmt<MPSA_FMT_E5M2, MPSA_FMT_E2M1>(g, c_dtype, grid, st) : launch_fmt<MPSA_FMT_E5M2, MPSA_FMT_E5M2>(g, c_dtype, grid, st);
    }
    MPSA_CHECK_LAUNCH("gemm");
    return MPSA_OK;
}

extern "C" int mpsa_gemm_mx_batched(const uint8_t* a, const uint8_t* sa, int fmt_a, const uint8_t* b, const uint8_t* sb, int fmt_b,
                                    int64_t batch, int64_t heads_a, int64_t heads_b, int64_t M, int64_t N, int64_t K,
                                    void* c, int c_dtype, int64_t ldc, mpsa_stream_t stream) {
    return gemm_entry(MPSA_GEMM_AUTO, a, sa, fmt_a, b, sb, fmt_b, false, batch, heads_a, heads_b, M, N, K, c, c_dtype, ldc, stream);
}

extern "C" int mpsa_gemm_mx(const uint8_t* a, const uint8_t* sa, int fmt_a, const uint8_t* b, const uint8_t* sb, int fmt_b,
                            int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, mpsa_stream_t stream) {
    return gemm_entry(MPSA_GEMM_AUTO, a, sa, fmt_a, b, sb, fmt_b, false, 1, 1, 1, M, N, K, c, c_dtype, ldc, stream);
}

extern "C" int mpsa_gemm_mx_packed(const uint8_t* a, const uint8_t* sa5, int fmt_a, const uint8_t* b, const uint8_t* sb5, int fmt_b,
                                   int64_t M, int64_t N, int64_t K, void* c, int c_dtype, int64_t ldc, mpsa_stream_t stream) {
    return gemm_entry(MPSA_GEMM_AUTO, a, sa5, fmt_a, b, sb5, fmt_b, true, 1, 1, 1, M, N, K, c, c_dtype, ldc, stream);
}

extern "C" int mpsa_gemm_mx_batched_packed(const uint8_t* a, const uint8_t* sa5, int fmt_a, const uint8_t* b, const uint8_t* sb5, int fmt_b,
                                           int64_t batch, int64_t heads_a, int64_t heads_b, int64_t M, int64_t N, int64_t K,
                                           void* c, int c_dtype, int64_t ldc, mpsa_stream_t stream) {
    return gemm_entry(MPSA_GEMM_AUTO, a, sa5, fmt_a, b, sb5, fmt_b, true, batch, heads_a, heads_b, M, N, K, c, c_dtype, ldc, stream);
}

extern "C" int mpsa_gemm_mx_on(int kernel, const uint8_t* a, const uint8_t* sa, int fmt_a, const uint8_t* b, const uint8_t* sb, int fmt_b, int packed,
                               int64_t batch, int64_t heads_a, int64_t heads_b, int64_t M, int64_t N, int64_t K,
                               void* c, int c_dtype, int64_t ldc, mpsa_stream_t stream) {
    return gemm_entry(kernel, a, sa, fmt_a, b, sb, fmt_b, packed != 0, batch, heads_a, heads_b, M, N, K, c, c_dtype, ldc, stream);
}

extern "C" int mpsa_gemm_kernel(int kernel, int fmt_a, int fmt_b, int64_t batch, int64_t heads_a, int64_t M, int64_t N, int64_t K) {
    const int rc = check_shape(fmt_a, fmt_b, batch, heads_a, 1, M, N, K, false);
    if (rc != MPSA_OK) return rc;
    GemmArgs g = {};
    g.M = (int)M; g.N = (int)N; g.K = (int)K;
    return choose(kernel, g, batch * heads_a, fmt_a, fmt_b);
}
