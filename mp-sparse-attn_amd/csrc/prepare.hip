// One-launch operand preparation for the fused attention kernel (gfx950): the MX quantization of Q (with
// sm_scale*log2(e) folded in) and of K (optionally minus its sequence mean) and the value-tile repack of V run as
// three groups of workgroups of ONE kernel instead of three launches - at the benchmark shape the three kernels take
// about 45 us together and the gaps between their launches another 20.  The quantizer's and the repack's own code
// (quantize_kernel.h, v_tiles_kernel.h); this file routes workgroup ids.
// Replaces the prologue of the reference's wrapper, ours/mxfp_attn_kernel.py:27-57 (dtype normalisation, quant_mxfp4 /
// quant_mxfp8e5 calls, operand packaging).
#include "seq_mean_kernel.h"
#include "reciprocal.h"
#include "v_tiles_kernel.h"

namespace {

struct PrepArgs {
    QuantArgs q, k;
    VTArgs v;
    Reciprocal by_bq, by_bk, by_bv, by_hq, by_hkv;
    uint32_t bq, bk, bv;          // workgroups per (batch, head) of each job
    uint32_t hq, hkv;
    uint32_t q_total, k_total;    // of the Q job, of the K job
    const float* sums;            // [B,Hkv,nchunk,D]: sums of chunks of K's rows (MEAN_SUMS)
    int nchunk;
    float inv_n;
};

// Threads of a workgroup, each with two chunks (and two words of V).  One that adds up its head's rows itself has twice as many: there
// are half as many to read the whole head, and its rows are asked for in half as many rounds.
__host__ __device__ constexpr int threads_of(int source) { return source == MEAN_ROWS_ITSELF ? 512 : 256; }

// The mean over the sequence of one head of K, in the inputs' type, into LDS: from the chunks' sums, or from the rows
// themselves (1024 at most, all asked for at once).  The additions of mpsa_seq_mean in their order, so its bits.
constexpr int MEAN_CHUNKS = 4;
template <int XDT, int SOURCE, int D>
__device__ __forceinline__ void head_mean(const PrepArgs& p, uint32_t hh, uint32_t bb, uint16_t* mean) {
    const int c = threadIdx.x;
    float s = 0.0f;
    if constexpr (SOURCE == MEAN_SUMS) {
        if (c < D) s = seq_sum(p.sums + ((int64_t)bb * p.hkv + hh) * p.nchunk * D + c, p.nchunk, D);
    } else {
        constexpr int GROUPS = threads_of(SOURCE) / 256, SLOTS = MEAN_CHUNKS / GROUPS;      // of 256 threads; chunks of 256 rows each
        static_assert(MEAN_CHUNKS * D <= threads_of(SOURCE), "a thread a sum");
        __shared__ float part[MEAN_CHUNKS][256][9], sums[MEAN_CHUNKS * D];
        const char* head = static_cast<const char*>(p.k.x) + 2 * ((int64_t)bb * p.k.sb + (int64_t)hh * p.k.sh);
        const int group = __builtin_amdgcn_readfirstlane(c >> 8);
        MeanChunk<D> chunk[SLOTS];
#pragma unroll
        for (int y = 0; y < SLOTS; ++y) {
            const int k = y * GROUPS + group;
            if (k < p.nchunk) chunk[y].request(head, p.k.sn, k * MEAN_ROWS, p.k.n, c & 255);
        }
#pragma unroll
        for (int y = 0; y < SLOTS; ++y) {
            const int k = y * GROUPS + group;
            if (k < p.nchunk) chunk[y].template add<XDT>(part[k], k * MEAN_ROWS, p.k.n, c & 255);
        }
        __syncthreads();
        if (c / D < p.nchunk) sums[c] = MeanChunk<D>::total(part[c / D], c % D);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < MEAN_CHUNKS; ++k)
            if (k < p.nchunk) s += sums[k * D + c % D];
    }
    if (c < D) mean[c] = mean_bits<XDT>(s * p.inv_n);
    __syncthreads();
}

// A workgroup takes 512 chunks of one head, two a thread, and asks for both before it does anything else (a padded head has a
// whole number of 512: 64 rows of 64).  What bounds it for short sequences is the wait for memory, and two blocks of 256 one after the
// other, as it was, waited twice.  With V's rows read four bytes a lane instead of two, whole calls, us: 32 heads over 8, D = 128, causal,
// diag: 160 tokens 9.44 -> 8.75, 1000 21.7 -> 20.4, 8192 327.8 -> 323.5; 8 heads of 1024 x 64 with the mean 15.45 -> 14.66; 40 heads of
// 300 x 128 19.3 -> 17.7.  Four chunks a thread, and four words of V, take 0.98 to 1.03 of that.
template <int XDT, bool DO4, bool DO8, int FMT8, int TILE, int D, int SOURCE>
__global__ __launch_bounds__(threads_of(SOURCE)) void prepare_kernel(PrepArgs p) {
    constexpr uint32_t THREADS = threads_of(SOURCE);
    uint32_t blk = blockIdx.x;
    if (blk < p.q_total) {
        const uint32_t head = divide_by(blk, p.by_bq), bb = divide_by(head, p.by_hq), hh = head - bb * p.hq, c = (blk - head * p.bq) * (2 * THREADS) + threadIdx.x;
        QuantChunk q[2] = {QuantChunk(p.q, c), QuantChunk(p.q, c + THREADS)};
        q[0].request(p.q, hh, bb);
        q[1].request(p.q, hh, bb);
        quantize_chunks<XDT, DO4, DO8, FMT8>(p.q, q, head, [](int64_t, uint32_t, float (&)[8]) __attribute__((always_inline)) {});
        return;
    }
    blk -= p.q_total;
    if (blk < p.k_total) {
        const uint32_t head = divide_by(blk, p.by_bk), bb = divide_by(head, p.by_hkv), hh = head - bb * p.hkv, c = (blk - head * p.bk) * (2 * THREADS) + threadIdx.x;
        QuantChunk q[2] = {QuantChunk(p.k, c), QuantChunk(p.k, c + THREADS)};
        q[0].request(p.k, hh, bb);
        q[1].request(p.k, hh, bb);
        if constexpr (SOURCE == MEAN_SUMS || SOURCE == MEAN_ROWS_ITSELF) {
            __shared__ __attribute__((aligned(16))) uint16_t mean[D];
            head_mean<XDT, SOURCE, D>(p, hh, bb, mean);
            quantize_chunks<XDT, DO4, DO8, FMT8>(p.k, q, head, [&](int64_t, uint32_t col8, float (&x)[8]) __attribute__((always_inline)) {
                less_mean<XDT>(x, *reinterpret_cast<const uint4*>(mean + 8 * col8));
            });
        } else {
            quantize_chunks<XDT, DO4, DO8, FMT8>(p.k, q, head, [&](int64_t hd, uint32_t col8, float (&x)[8]) __attribute__((always_inline)) { less_given<XDT>(p.k, hd, col8, x); });
        }
        return;
    }
    blk -= p.k_total;
    const uint32_t head = divide_by(blk, p.by_bv), bb = divide_by(head, p.by_hkv);
    v_tiles_block<TILE, D, THREADS>(p.v, blk - head * p.bv, head - bb * p.hkv, bb, p.hkv);
}

template <int XDT, bool DO4, bool DO8, int FMT8, int TILE, int D>
void launch_source(const PrepArgs& p, MeanSource source, unsigned grid, hipStream_t st) {
    if (source == MEAN_SUMS)             hipLaunchKernelGGL((prepare_kernel<XDT, DO4, DO8, FMT8, TILE, D, MEAN_SUMS>), dim3(grid), dim3(threads_of(MEAN_SUMS)), 0, st, p);
    else if (source == MEAN_ROWS_ITSELF) hipLaunchKernelGGL((prepare_kernel<XDT, DO4, DO8, FMT8, TILE, D, MEAN_ROWS_ITSELF>), dim3(grid), dim3(threads_of(MEAN_ROWS_ITSELF)), 0, st, p);
    else                                 hipLaunchKernelGGL((prepare_kernel<XDT, DO4, DO8, FMT8, TILE, D, MEAN_GIVEN>), dim3(grid), dim3(threads_of(MEAN_GIVEN)), 0, st, p);
}

template <int XDT, bool DO4, bool DO8, int FMT8>
void launch_td(const PrepArgs& p, int tile, int d, MeanSource source, unsigned grid, hipStream_t st) {
    if (tile == 128 && d == 128)      launch_source<XDT, DO4, DO8, FMT8, 128, 128>(p, source, grid, st);
    else if (tile == 128 && d == 64)  launch_source<XDT, DO4, DO8, FMT8, 128, 64>(p, source, grid, st);
    else if (tile == 64 && d == 128)  launch_source<XDT, DO4, DO8, FMT8, 64, 128>(p, source, grid, st);
    else                              launch_source<XDT, DO4, DO8, FMT8, 64, 64>(p, source, grid, st);
}

template <int XDT>
void launch_mode(const PrepArgs& p, bool do4, bool do8, int fmt8, int tile, int d, MeanSource source, unsigned grid, hipStream_t st) {
    if (!do8) launch_td<XDT, true, false, MPSA_FMT_E4M3>(p, tile, d, source, grid, st);
    else if (!do4) {
        if (fmt8 == MPSA_FMT_E5M2) launch_td<XDT, false, true, MPSA_FMT_E5M2>(p, tile, d, source, grid, st);
        else                       launch_td<XDT, false, true, MPSA_FMT_E4M3>(p, tile, d, source, grid, st);
    } else {
        if (fmt8 == MPSA_FMT_E5M2) launch_td<XDT, true, true, MPSA_FMT_E5M2>(p, tile, d, source, grid, st);
        else                       launch_td<XDT, true, true, MPSA_FMT_E4M3>(p, tile, d, source, grid, st);
    }
}

}  // namespace

// Where the mean over K's sequence comes from.  On its own it takes two launches (sums of chunks of 256 rows; their sum), each
// of which costs the host as much as the preparation does and the device a round trip to memory.  The preparation's workgroups
// can add up the chunks' sums themselves, or its rows: every workgroup reads the whole head, 1024 of whose 16-byte pieces it
// quantizes.  That pays while the rows are asked for at once and the workgroups are one or two a CU: of 130 shapes (2 to 64 heads, 80 to 2600
// keys, both widths) all 89 within these bounds are faster that way, by up to 5 us.  Microseconds of whole calls, from sums,
// from rows (workgroups): 16 heads of 1018 x 128 24.0 21.1 (256); 32 of 653 x 128 31.6 30.1 (352); 48 of 512 x 128 44.7 44.1 (384);
// 32 of 779 x 128 25.5 26.6 (416); 48 of 611 x 128 27.1 28.3 (480); 32 of 1018 x 64 19.3 17.7 (256); 64 of 1024 x 64 29.7 32.1 (512); past
// 1024 rows 8 of 1443 x 128 24.7 22.5, 16 of 1414 x 128 31.2 34.8, 4 of 1146 x 128 17.8 19.0, 8 of 1281 x 64 15.4 16.7.  Sums up to
// 64 chunks (32 heads, 4096 x 64, 86.4 -> 84.8) and where the workgroups together read 14 MB of them at most: every one of a head
// reads them all, which is quadratic in the keys.  A mean of its own against sums, whole calls of 128 queries, us (MB): 8 heads
// of 4096 x 128 36.6 35.2 (8.4), 6144 44.1 44.1 (19), 16384 88.9 94.9 (134); 40 of 2048 x 128 36.3 36.5 (10), 4096 55.3 57.7 (42),
// 8656 116 129 (187); 24 of 8192 x 64 53.5 53.6 (25), 16000 92 97 (96).
MeanSource mpsa_mean_source(int64_t B, int64_t Hkv, int64_t nk, int64_t D) {
    if (mpsa_quantize_sw_encoders()) return MEAN_GIVEN;      // stand-alone kernels
    const double workgroups = (double)(B * Hkv) * (double)((nk * D / 8 + 1023) / 1024);
    if (nk <= MEAN_CHUNKS * MEAN_ROWS && workgroups <= 384.0) return MEAN_ROWS_ITSELF;
    const double read = (double)(B * Hkv) * (double)nk * (double)nk * (double)(D * D) / 262144.0;      // bytes of sums, all workgroups
    return nk <= 64 * MEAN_ROWS && read <= 14e6 ? MEAN_SUMS : MEAN_GIVEN;
}

// Host side of the preparation: which of the operand sets are made is up to the caller (do4 / do8 of either side; the
// mixed mode multiplies 8-bit Q with 4-bit K and needs one set of each).
int mpsa_prepare_operands(const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides, const void* v, const int64_t* v_strides,
                          int dtype, int64_t B, int64_t Hq, int64_t Hkv, int64_t Nq, int64_t Nk, int64_t D, int tile, int fmt8, float pre_scale_q,
                          MeanSource mean, const void* k_sub, bool q_do4, bool q_do8, bool k_do4, bool k_do8, uint8_t* q4, uint8_t* qs4, uint8_t* q8, uint8_t* qs8,
                          uint8_t* k4, uint8_t* ks4, uint8_t* k8, uint8_t* ks8, void* v_tiles, hipStream_t st) {
    const int64_t nq_pad = (Nq + tile - 1) / tile * tile, nk_pad = (Nk + tile - 1) / tile * tile;
    constexpr int EMAX4 = 3, EMAX8 = 7;            // ours/quant_mxint8.py:303, :191
    if (mpsa_quantize_sw_encoders() && q) {
        // the cross-checking encoders exist only as stand-alone kernels
        auto one = [&](const void* x, int64_t H, int64_t N, const int64_t* xs, const void* sub, float pre, bool do4, bool do8,
                       uint8_t* c4, uint8_t* s4, uint8_t* c8, uint8_t* s8, int64_t rows) {
            if (do4 && do8) return mpsa_quantize_mx_dual(x, dtype, B, H, N, D, xs, sub, pre, EMAX4, fmt8, EMAX8, c4, s4, c8, s8, rows, st);
            return mpsa_quantize_mx(x, dtype, B, H, N, D, xs, sub, pre, do4 ? MPSA_FMT_E2M1 : fmt8, do4 ? EMAX4 : EMAX8, do4 ? c4 : c8, do4 ? s4 : s8, rows, st);
        };
        int rc = one(q, Hq, Nq, q_strides, nullptr, pre_scale_q, q_do4, q_do8, q4, qs4, q8, qs8, nq_pad);
        if (rc != MPSA_OK) return rc;
        rc = one(k, Hkv, Nk, k_strides, k_sub, 1.0f, k_do4, k_do8, k4, ks4, k8, ks8, nk_pad);
        if (rc != MPSA_OK) return rc;
        return mpsa_v_tiles(v, dtype, B, Hkv, Nk, D, v_strides, tile, v_tiles, st);
    }
    PrepArgs p;
    unsigned bq = 0, bk = 0, bv = 0;
    int rc = MPSA_OK;
    if (q) {
        rc = mpsa_quantize_setup(q, dtype, B, Hq, Nq, D, q_strides, nullptr, pre_scale_q, q_do4, EMAX4, q_do8, fmt8, EMAX8, q4, qs4, q8, qs8, nq_pad, &p.q, &bq);
        if (rc != MPSA_OK) return rc;
    } else {
        p.q = QuantArgs{};                       // no Q job: the attention kernel quantizes Q itself (mpsa_attn_fwd_q16)
        q_do4 = q_do8 = false;
    }
    rc = mpsa_quantize_setup(k, dtype, B, Hkv, Nk, D, k_strides, mean == MEAN_GIVEN ? k_sub : nullptr, 1.0f, k_do4, EMAX4, k_do8, fmt8, EMAX8, k4, ks4, k8, ks8, nk_pad, &p.k, &bk);
    if (rc != MPSA_OK) return rc;
    rc = mpsa_v_tiles_setup(v, dtype, B, Hkv, Nk, D, v_strides, tile, v_tiles, &p.v, &bv);
    if (rc != MPSA_OK) return rc;
    // the set-ups count blocks of 256 chunks and of 512 words
    const unsigned blocks = (unsigned)(threads_of(mean) / 256 * 2);
    bq = (bq + blocks - 1) / blocks;
    bk = (bk + blocks - 1) / blocks;
    bv = (bv + blocks / 2 - 1) / (blocks / 2);
    const int64_t total = (int64_t)bq * Hq * B + (int64_t)(bk + bv) * Hkv * B;
    if (total >= (int64_t(1) << 30)) return mpsa_fail(MPSA_EUNSUPPORTED, "prepare: problem too large for one launch");
    p.bq = bq; p.bk = bk; p.bv = bv; p.hq = (uint32_t)Hq; p.hkv = (uint32_t)Hkv;
    p.by_bq = reciprocal_of(bq ? bq : 1); p.by_bk = reciprocal_of(bk); p.by_bv = reciprocal_of(bv); p.by_hq = reciprocal_of(p.hq); p.by_hkv = reciprocal_of(p.hkv);
    p.q_total = (uint32_t)((int64_t)bq * Hq * B); p.k_total = (uint32_t)((int64_t)bk * Hkv * B);
    p.sums = mean == MEAN_SUMS ? static_cast<const float*>(k_sub) : nullptr;
    p.nchunk = (int)((Nk + MEAN_ROWS - 1) / MEAN_ROWS);
    p.inv_n = 1.0f / (float)Nk;
    const bool do4 = q_do4 || k_do4, do8 = q_do8 || k_do8;
    if (dtype == MPSA_BF16) launch_mode<MPSA_BF16>(p, do4, do8, fmt8, tile, (int)D, mean, (unsigned)total, st);
    else                    launch_mode<MPSA_F16>(p, do4, do8, fmt8, tile, (int)D, mean, (unsigned)total, st);
    MPSA_CHECK_LAUNCH("prepare");
    return MPSA_OK;
}

extern "C" int mpsa_attn_prepare(const void* q, const int64_t q_strides[4], const void* k, const int64_t k_strides[4],
                                 const void* v, const int64_t v_strides[4], int dtype,
                                 int64_t B, int64_t Hq, int64_t Hkv, int64_t Nq, int64_t Nk, int64_t D, int tile, int mode, int fmt8,
                                 float pre_scale_q, const void* k_sub,
                                 uint8_t* q4, uint8_t* qs4, uint8_t* q8, uint8_t* qs8,
                                 uint8_t* k4, uint8_t* ks4, uint8_t* k8, uint8_t* ks8, void* v_tiles, mpsa_stream_t stream) {
    if (mode == MPSA_MODE_ROUTED || mode == MPSA_MODE_MIXED) mode = MPSA_MODE_DIAG;   // both operand sets, like a diag run
    if (mode != MPSA_MODE_MXFP4 && mode != MPSA_MODE_MXFP8 && mode != MPSA_MODE_DIAG) return mpsa_fail(MPSA_EINVAL, "prepare: unknown mode %d", mode);
    if (tile != 64 && tile != 128) return mpsa_fail(MPSA_EUNSUPPORTED, "prepare: tile must be 64 or 128 (got %d)", tile);
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || Nq <= 0 || Nk <= 0 || Hq % Hkv) return mpsa_fail(MPSA_EINVAL, "prepare: bad shape (B=%lld Hq=%lld Hkv=%lld Nq=%lld Nk=%lld)", (long long)B, (long long)Hq, (long long)Hkv, (long long)Nq, (long long)Nk);
    const bool do4 = mode != MPSA_MODE_MXFP8, do8 = mode != MPSA_MODE_MXFP4;
    return mpsa_prepare_operands(q, q_strides, k, k_strides, v, v_strides, dtype, B, Hq, Hkv, Nq, Nk, D, tile, fmt8, pre_scale_q, k_sub ? MEAN_GIVEN : MEAN_NONE, k_sub,
                                 do4, do8, do4, do8, q4, qs4, q8, qs8, k4, ks4, k8, ks8, v_tiles, (hipStream_t)stream);
}
