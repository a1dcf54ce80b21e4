// Fused diagonal-tiled MXFP attention forward for gfx950.
//
// Per query tile i of one head: for every visited key tile j, S = Q_i K_j^T on the scaled matrix cores
// (8-bit operands when the tile's precision is 8-bit, 4-bit otherwise), base-2 online softmax with
// float32 running max / sum, P rounded to 16 bits, O += P V_j, and O / l at the end -- the loop of the
// reference's block_scaled_batched_attn_kernel (ours/mxfp_attn_kernel.py:216-359).  Causal runs visit
// tiles j <= i and mask only tile j == i (ours/online_routing.py:68-77, :113-118); query head hq reads
// key/value head hq / (Hq/Hkv) (ours/online_routing.py:160-171).  Q already carries sm_scale*log2(e)
// (folded in by the quantizer, ours/quant_mxint8.py:494), so scores are in log2 units.
//
// Mapping of the kernel in attn_fwd_kernel.h, which takes what D = 128 with tile = 128 (attn_fwd_tile.hip) leaves, and there skipping
// inside the kernel.  A workgroup owns one TILE-query tile; each of its TILE/32 waves owns 32 queries and walks all
// keys of every tile.  Both products are computed transposed so that a lane always owns ONE query:
//   S^T = K Q^T   on v_mfma_scale_f32_32x32x64_f8f6f4: lane (h = lane/32, r = lane%32) of the K operand
//                 supplies 32 elements of key row r and the E8M0 byte of MX block h of the 64-wide step
//                 (4-bit: the lane's registers are block h; 8-bit: registers 0-3 of both lane halves are
//                 block 0, registers 4-7 block 1), the Q operand the same for query r; the result leaves query r's scores for 16 keys per 32-key block in
//                 that lane's registers, so the row maximum is a register reduction plus one exchange
//                 with lane^32, and running max / sum / rescale factors are plain per-lane scalars.
//   O^T += V^T P^T on v_mfma_f32_32x32x16_{bf16,f16}: the P^T operand of lane (h, r) is exactly the eight
//                 scores that lane already holds (keys are contracted in the order the score MFMA left
//                 them); V is pre-arranged by mpsa_v_tiles to match, one 16-byte LDS read per operand.
// Staging.  4-bit K codes and the V tile travel HBM/L2 -> LDS with direct-to-LDS loads (global_load_lds_dwordx4:
// each lane names a 16-byte global source, the wave's 64 pieces land contiguously in LDS), so they cost neither
// registers nor LDS-write instructions.  The V tile is already in operand order (a flat copy); K rows keep their
// row-major order but the 16-byte chunks of a row are XOR-swizzled with the row index, which makes the 128-bit
// operand reads of 16 consecutive rows hit 16 distinct 4-bank groups.  Both are double-buffered and the loop
// needs ONE barrier per tile: after the barrier of step t a wave issues the loads of V(t+1) and K(t+2), pulls the
// K(t+1) fragments from LDS into registers and runs P.V of step t; the next step's score MFMAs then start from
// registers.  The single 8-bit K tile of a "diag" run bypasses LDS (each lane reads its fragments from global memory);
// runs with many 8-bit tiles ("mxfp8", routed) stage them through the same LDS area, one buffer plus the fragment
// registers (see attn_fwd_kernel.h).  K scales are read from global memory one step ahead.  80 KiB of LDS and at most 256 registers per workgroup let two workgroups share a CU, so one's matrix
// instructions overlap the other's softmax VALU work.
#include "attn_fwd_kernel.h"
#include <cstdlib>

namespace {

template <int D, int TILE, int PVT>
int launch_mode(const AttnArgs& a, hipStream_t st) {
    if (a.mode == MPSA_MODE_MXFP4) return launch_one<D, TILE, PVT, MPSA_FMT_E4M3, MPSA_MODE_MXFP4>(a, st);
    if (a.mode == MPSA_MODE_MIXED)
        return a.fmt8 == MPSA_FMT_E5M2 ? launch_one<D, TILE, PVT, MPSA_FMT_E5M2, MPSA_MODE_MIXED>(a, st)
                                       : launch_one<D, TILE, PVT, MPSA_FMT_E4M3, MPSA_MODE_MIXED>(a, st);
    if (a.mode == MPSA_MODE_MXFP8)
        return a.fmt8 == MPSA_FMT_E5M2 ? launch_one<D, TILE, PVT, MPSA_FMT_E5M2, MPSA_MODE_MXFP8>(a, st)
                                       : launch_one<D, TILE, PVT, MPSA_FMT_E4M3, MPSA_MODE_MXFP8>(a, st);
    return a.fmt8 == MPSA_FMT_E5M2 ? launch_one<D, TILE, PVT, MPSA_FMT_E5M2, MPSA_MODE_DIAG>(a, st)
                                   : launch_one<D, TILE, PVT, MPSA_FMT_E4M3, MPSA_MODE_DIAG>(a, st);
}

template <int D, int TILE>
int launch_dt(const AttnArgs& a, int pv_dtype, hipStream_t st) {
    if (pv_dtype == MPSA_BF16) return launch_mode<D, TILE, MPSA_BF16>(a, st);
    return launch_mode<D, TILE, MPSA_F16>(a, st);
}

}  // namespace

// Causal runs of the general kernel: whether a head's rows are dealt out one by one over the XCDs instead of going to one of them
// in a contiguous range.  With a whole number of (batch, KV head) pairs per XCD ranges are even and keep a pair's K and V in one
// L2.  With any other number a range gives one XCD long rows and the next short ones; dealt out, everybody gets both, but
// pairs / gcd(pairs, 8) of them pass through every L2.  That costs more than it gains once there are more than six and the
// work is long: workgroups times 64-key tiles beyond 800 000, where an XCD is even enough by itself.
// Dealt -> contiguous, us, pairs x heads each, 64-key tiles of D = 128: 16384 tokens 2x4 383 -> 604, 6x4 1100 -> 1248, 9x4 1972 ->
// 1732, 11x4, 15x4 and 17x4 0.77, 0.61 and 0.59 of the time; 8192 tokens 9x4 453 -> 480, 15x4 and 52x4 0.89 and 0.70.
static bool rows_dealt(int64_t units, int64_t workgroups, int64_t tiles64) {
    return (units & 7) != 0 && (units / (units & -units) <= 6 || workgroups * tiles64 < 800000);
}

// paired_only: the shapes of mpsa_attn_fwd_q16, which takes no others
struct RawQ { const void* q; const int64_t* strides; int dtype; float pre; bool paired_only; };

static int attn_entry(int kernel, const RawQ* rq, const uint8_t* q4, const uint8_t* qs4, const uint8_t* q8, const uint8_t* qs8,
                      const uint8_t* k4, const uint8_t* ks4, const uint8_t* k8, const uint8_t* ks8, int fmt8,
                      const void* v_tiles, int pv_dtype, void* o, int o_dtype, const int64_t o_strides[4],
                      int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t n, int64_t D, int tile, int causal, int mode,
                      bool skip, float skip_thresh, int32_t* skipped, const int32_t* order, const int32_t* counts,
                      mpsa_stream_t stream) {
    if (mode != MPSA_MODE_MXFP4 && mode != MPSA_MODE_MXFP8 && mode != MPSA_MODE_DIAG && mode != MPSA_MODE_ROUTED && mode != MPSA_MODE_MIXED) return mpsa_fail(MPSA_EINVAL, "attn: unknown mode %d", mode);
    const bool routed = mode == MPSA_MODE_ROUTED;
    if (routed && (!order || !counts)) return mpsa_fail(MPSA_EINVAL, "attn: a routed run needs the visiting lists (order, counts)");
    if (routed && ((reinterpret_cast<uintptr_t>(order) | reinterpret_cast<uintptr_t>(counts)) & 3)) return mpsa_fail(MPSA_EALIGN, "attn: order and counts must be 4-byte aligned");
    const bool mixed = mode == MPSA_MODE_MIXED;
    const bool need4 = mode != MPSA_MODE_MXFP8, need8 = mode != MPSA_MODE_MXFP4;
    if (rq) {
        if (!rq->q || !rq->strides) return mpsa_fail(MPSA_EINVAL, "attn: null q");
        if (rq->dtype != pv_dtype) return mpsa_fail(MPSA_EINVAL, "attn: unquantized q must have the P.V dtype (the dtype of v)");
        if (rq->strides[3] != 1 || !mpsa_aligned16(rq->q) || (rq->strides[0] % 8) || (rq->strides[1] % 8) || (rq->strides[2] % 8))
            return mpsa_fail(MPSA_EALIGN, "attn: q rows must be contiguous and 16-byte aligned");
        if (mode == MPSA_MODE_ROUTED) return mpsa_fail(MPSA_EUNSUPPORTED, "attn: unquantized q is not taken in the routed mode (the router reads Q's scale bytes)");
        const bool k8_read = mode == MPSA_MODE_DIAG || mode == MPSA_MODE_MXFP8;       // the mixed mode multiplies 4-bit K only
        if ((need4 && (!k4 || !ks4)) || (k8_read && (!k8 || !ks8))) return mpsa_fail(MPSA_EINVAL, "attn: K operands missing");
    } else if (mixed) {
        if (!q8 || !qs8 || !k4 || !ks4) return mpsa_fail(MPSA_EINVAL, "attn: the mixed mode needs 8-bit Q and 4-bit K operands");
    } else if (routed) {
        // lists that name tiles of one precision only need that operand set only (the caller's promise); a set is whole or absent
        const bool has4 = q4 && qs4 && k4 && ks4, has8 = q8 && qs8 && k8 && ks8;
        const bool none4 = !q4 && !qs4 && !k4 && !ks4, none8 = !q8 && !qs8 && !k8 && !ks8;
        if (!(has4 || none4) || !(has8 || none8) || (none4 && none8)) return mpsa_fail(MPSA_EINVAL, "attn: a routed run needs the whole 4-bit operand set, the whole 8-bit one, or both");
    } else {
        if (need4 && (!q4 || !qs4 || !k4 || !ks4)) return mpsa_fail(MPSA_EINVAL, "attn: 4-bit operands missing");
        if (need8 && (!q8 || !qs8 || !k8 || !ks8)) return mpsa_fail(MPSA_EINVAL, "attn: 8-bit operands missing");
    }
    if (!v_tiles || !o || !o_strides) return mpsa_fail(MPSA_EINVAL, "attn: null pointer");
    if (need8 && (!routed || q8) && fmt8 != MPSA_FMT_E4M3 && fmt8 != MPSA_FMT_E5M2) return mpsa_fail(MPSA_EINVAL, "attn: 8-bit format must be E4M3 or E5M2");
    if (pv_dtype != MPSA_BF16 && pv_dtype != MPSA_F16) return mpsa_fail(MPSA_EINVAL, "attn: pv_dtype must be bf16 or f16");
    if (o_dtype != MPSA_BF16 && o_dtype != MPSA_F16 && o_dtype != MPSA_F32) return mpsa_fail(MPSA_EINVAL, "attn: bad output dtype");
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || n <= 0 || nq <= 0 || Hq % Hkv) return mpsa_fail(MPSA_EINVAL, "attn: bad shape (B=%lld Hq=%lld Hkv=%lld nq=%lld nk=%lld)", (long long)B, (long long)Hq, (long long)Hkv, (long long)nq, (long long)n);
    if (nq != n && (causal || mode == MPSA_MODE_DIAG)) return mpsa_fail(MPSA_EINVAL, "attn: causal masking and the diag mode need as many queries as keys (nq=%lld nk=%lld)", (long long)nq, (long long)n);
    if ((D != 64 && D != 128) || (tile != 64 && tile != 128)) return mpsa_fail(MPSA_EUNSUPPORTED, "attn: D=%lld tile=%d (both must be 64 or 128)", (long long)D, tile);
    if (o_strides[3] != 1 || (o_strides[0] % 4) || (o_strides[1] % 4) || (o_strides[2] % 4)) return mpsa_fail(MPSA_EALIGN, "attn: output rows must be contiguous and 8-byte aligned");
    const uintptr_t al = reinterpret_cast<uintptr_t>(q4) | reinterpret_cast<uintptr_t>(q8) | reinterpret_cast<uintptr_t>(k4) |
                         reinterpret_cast<uintptr_t>(k8) | reinterpret_cast<uintptr_t>(v_tiles) | reinterpret_cast<uintptr_t>(o);
    const uintptr_t al4 = reinterpret_cast<uintptr_t>(qs4) | reinterpret_cast<uintptr_t>(qs8) | reinterpret_cast<uintptr_t>(ks4) | reinterpret_cast<uintptr_t>(ks8);
    if ((al & 15) || (al4 & 3)) return mpsa_fail(MPSA_EALIGN, "attn: operands must be 16-byte (codes, v, o) / 4-byte (scales) aligned");
    const int64_t nt = (n + tile - 1) / tile, ntq = (nq + tile - 1) / tile;
    if (B * Hq * ntq >= (int64_t(1) << 31) || nt * tile >= (int64_t(1) << 30) || ntq * tile >= (int64_t(1) << 30)) return mpsa_fail(MPSA_EUNSUPPORTED, "attn: problem too large");
    AttnArgs a;
    a.q4 = q4; a.qs4 = qs4; a.q8 = q8; a.qs8 = qs8; a.k4 = k4; a.ks4 = ks4; a.k8 = k8; a.ks8 = ks8;
    a.v = v_tiles; a.o = o;
    a.o_sb = o_strides[0]; a.o_sh = o_strides[1]; a.o_sn = o_strides[2];
    a.B = (int)B; a.Hq = (int)Hq; a.Hkv = (int)Hkv; a.n = (int)n; a.nt = (int)nt; a.n_pad = (int)(nt * tile);
    a.nq = (int)nq; a.ntq = (int)ntq; a.nq_pad = (int)(ntq * tile);
    a.causal = causal ? 1 : 0; a.mode = mode; a.fmt8 = fmt8; a.o_dtype = o_dtype;
    a.d = (int)D; a.tile = tile;
    a.skip_thresh = skip_thresh; a.skipped = skipped;
    a.order = order; a.counts = counts;
    a.q_raw = nullptr; a.q_sb = a.q_sh = a.q_sn = 0; a.q_pre = 1.0f; a.q_sure = 0;
    if (causal && rows_dealt(B * Hkv, B * Hq * ntq, nt * tile / 64)) a.causal |= ROWS_DEALT;
    hipStream_t st = (hipStream_t)stream;
    if (rq) {
        a.q_raw = rq->q; a.q_sb = rq->strides[0]; a.q_sh = rq->strides[1]; a.q_sn = rq->strides[2]; a.q_pre = rq->pre;
        a.q_sure = mpsa_e2m1_sure(rq->pre, pv_dtype) ? 1 : 0;
        if (rq->paired_only && !attn_pp_supported(a, pv_dtype))
            return mpsa_fail(MPSA_EUNSUPPORTED, "attn: unquantized q needs the paired-tile kernel's shape (D = 128, tile = 128; "
                                                "causal: at least two tiles, unmasked: at least six); quantize q with mpsa_attn_prepare and call mpsa_attn_fwd");
    }
    if (routed) return attn_tile_supported(D, tile) ? attn_tile_launch(a, pv_dtype, st) : attn_routed_launch(a, pv_dtype, st);
    if (skip) {
        if (!(skip_thresh == skip_thresh)) return mpsa_fail(MPSA_EINVAL, "attn: skip_thresh is NaN");
        if (skipped && (reinterpret_cast<uintptr_t>(skipped) & 3)) return mpsa_fail(MPSA_EALIGN, "attn: skipped must be 4-byte aligned");
        return attn_skip_launch(a, pv_dtype, st);
    }
    kernel = mpsa_attn_kernel(kernel, B, Hq, Hkv, nq, n, D, tile, causal, mode);
    if (kernel < 0) return kernel;
    if (kernel == MPSA_ATTN_SHORT1) return attn_short_launch(a, pv_dtype, 1, st);
    if (kernel == MPSA_ATTN_SHORT2) return attn_short_launch(a, pv_dtype, 2, st);
    if (kernel == MPSA_ATTN_SHORT4) return attn_short_launch(a, pv_dtype, 4, st);
    if (kernel == MPSA_ATTN_PAIRED) return attn_pp_launch(a, pv_dtype, st);
    if (kernel == MPSA_ATTN_TILE) return attn_tile_launch(a, pv_dtype, st);
    if (rq) return mpsa_fail(MPSA_EUNSUPPORTED, "attn: the general kernel takes quantized q only; quantize it with mpsa_attn_prepare and call mpsa_attn_fwd");
    if (attn_tile_supported(D, tile)) return attn_tile_launch(a, pv_dtype, st);
    if (D == 64 && tile == 64)   return launch_dt<64, 64>(a, pv_dtype, st);
    if (D == 128 && tile == 64)  return launch_dt<128, 64>(a, pv_dtype, st);
    return launch_dt<64, 128>(a, pv_dtype, st);
}

extern "C" int mpsa_attn_fwd(const uint8_t* q4, const uint8_t* qs4, const uint8_t* q8, const uint8_t* qs8,
                             const uint8_t* k4, const uint8_t* ks4, const uint8_t* k8, const uint8_t* ks8, int fmt8,
                             const void* v_tiles, int pv_dtype, void* o, int o_dtype, const int64_t o_strides[4],
                             int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t n, int64_t D, int tile, int causal, int mode,
                             mpsa_stream_t stream) {
    return attn_entry(MPSA_ATTN_AUTO, nullptr, q4, qs4, q8, qs8, k4, ks4, k8, ks8, fmt8, v_tiles, pv_dtype, o, o_dtype, o_strides,
                      B, Hq, Hkv, nq, n, D, tile, causal, mode, false, 0.0f, nullptr, nullptr, nullptr, stream);
}

extern "C" int mpsa_attn_fwd_on(int kernel, const uint8_t* q4, const uint8_t* qs4, const uint8_t* q8, const uint8_t* qs8,
                                const uint8_t* k4, const uint8_t* ks4, const uint8_t* k8, const uint8_t* ks8, int fmt8,
                                const void* v_tiles, int pv_dtype, void* o, int o_dtype, const int64_t o_strides[4],
                                int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t n, int64_t D, int tile, int causal, int mode,
                                mpsa_stream_t stream) {
    return attn_entry(kernel, nullptr, q4, qs4, q8, qs8, k4, ks4, k8, ks8, fmt8, v_tiles, pv_dtype, o, o_dtype, o_strides,
                      B, Hq, Hkv, nq, n, D, tile, causal, mode, false, 0.0f, nullptr, nullptr, nullptr, stream);
}

extern "C" int mpsa_attn_fwd_skip(const uint8_t* q4, const uint8_t* qs4, const uint8_t* q8, const uint8_t* qs8,
                                  const uint8_t* k4, const uint8_t* ks4, const uint8_t* k8, const uint8_t* ks8, int fmt8,
                                  const void* v_tiles, int pv_dtype, void* o, int o_dtype, const int64_t o_strides[4],
                                  int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t n, int64_t D, int tile, int causal, int mode,
                                  float skip_thresh, int32_t* skipped, mpsa_stream_t stream) {
    return attn_entry(MPSA_ATTN_AUTO, nullptr, q4, qs4, q8, qs8, k4, ks4, k8, ks8, fmt8, v_tiles, pv_dtype, o, o_dtype, o_strides,
                      B, Hq, Hkv, nq, n, D, tile, causal, mode, true, skip_thresh, skipped, nullptr, nullptr, stream);
}

extern "C" int mpsa_attn_fwd_routed(const uint8_t* q4, const uint8_t* qs4, const uint8_t* q8, const uint8_t* qs8,
                                    const uint8_t* k4, const uint8_t* ks4, const uint8_t* k8, const uint8_t* ks8, int fmt8,
                                    const void* v_tiles, int pv_dtype, void* o, int o_dtype, const int64_t o_strides[4],
                                    int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t n, int64_t D, int tile, int causal,
                                    const int32_t* order, const int32_t* counts, mpsa_stream_t stream) {
    return attn_entry(MPSA_ATTN_AUTO, nullptr, q4, qs4, q8, qs8, k4, ks4, k8, ks8, fmt8, v_tiles, pv_dtype, o, o_dtype, o_strides,
                      B, Hq, Hkv, nq, n, D, tile, causal, MPSA_MODE_ROUTED, false, 0.0f, nullptr, order, counts, stream);
}

extern "C" int mpsa_attn_fwd_q16(const void* q, const int64_t q_strides[4], int q_dtype, float pre_scale_q,
                                 const uint8_t* k4, const uint8_t* ks4, const uint8_t* k8, const uint8_t* ks8, int fmt8,
                                 const void* v_tiles, int pv_dtype, void* o, int o_dtype, const int64_t o_strides[4],
                                 int64_t B, int64_t Hq, int64_t Hkv, int64_t n, int64_t D, int tile, int causal, int mode,
                                 mpsa_stream_t stream) {
    const RawQ rq = {q, q_strides, q_dtype, pre_scale_q, true};
    return attn_entry(MPSA_ATTN_AUTO, &rq, nullptr, nullptr, nullptr, nullptr, k4, ks4, k8, ks8, fmt8, v_tiles, pv_dtype, o, o_dtype, o_strides,
                      B, Hq, Hkv, n, n, D, tile, causal, mode, false, 0.0f, nullptr, nullptr, nullptr, stream);
}

extern "C" int mpsa_attn_fwd_q16_on(int kernel, const void* q, const int64_t q_strides[4], int q_dtype, float pre_scale_q,
                                    const uint8_t* k4, const uint8_t* ks4, const uint8_t* k8, const uint8_t* ks8, int fmt8,
                                    const void* v_tiles, int pv_dtype, void* o, int o_dtype, const int64_t o_strides[4],
                                    int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t nk, int64_t D, int tile, int causal, int mode,
                                    mpsa_stream_t stream) {
    const RawQ rq = {q, q_strides, q_dtype, pre_scale_q, false};
    return attn_entry(kernel, &rq, nullptr, nullptr, nullptr, nullptr, k4, ks4, k8, ks8, fmt8, v_tiles, pv_dtype, o, o_dtype, o_strides,
                      B, Hq, Hkv, nq, nk, D, tile, causal, mode, false, 0.0f, nullptr, nullptr, nullptr, stream);
}

extern "C" int mpsa_attn_fwd_q16_supported(int64_t B, int64_t Hq, int64_t Hkv, int64_t n, int64_t D, int tile, int causal, int mode) {
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || n <= 0 || Hq % Hkv || B * Hq * (n / 256 + 1) >= (int64_t(1) << 31)) return 0;
    if (mode != MPSA_MODE_DIAG && mode != MPSA_MODE_MXFP4 && mode != MPSA_MODE_MIXED && mode != MPSA_MODE_MXFP8) return 0;
    AttnArgs a = {};
    a.B = (int)B; a.Hq = (int)Hq; a.Hkv = (int)Hkv; a.n = (int)n; a.d = (int)D; a.tile = tile; a.causal = causal ? 1 : 0; a.mode = mode;
    a.nt = (int)((n + tile - 1) / (tile > 0 ? tile : 1)); a.n_pad = a.nt * tile;
    a.nq = a.n; a.ntq = a.nt; a.nq_pad = a.n_pad;
    return (tile == 64 || tile == 128) && attn_pp_supported(a, MPSA_BF16) ? 1 : 0;
}

static constexpr double SHORT_LIMIT = 16777216.0;         // blocks of 32 queries: a launch has fewer than 2^32 threads, a workgroup 256

// The kernel that is estimated to finish first: the short-sequence kernel (attn_fwd_short.hip) with one, two or four key splits,
// if there are no more blocks of queries than it takes (`fits`), or one that owns whole query tiles.  Microseconds
// of either side, fitted to measurements at 90 shapes (1 - 256 heads, 45 - 8192 keys, D = 64 and 128, masked and not).  A workgroup of the short kernel takes a fixed time and so
// much a stage, `full` with all of a CU's places filled, `alone` at the head of the longest chain; a tile kernel's time is its
// longest workgroup while there are no more of them than CUs.  With 32 heads and D = 128 four splits go up to 250 tokens, two
// to 1900; one split serves many queries over few keys, however many: 40 heads, 32760
// queries over 512 keys (whole calls) 303 us where the general kernel takes 365; 2 x 24 heads, 29157 over 100, 8-bit, 201
// and 319; and long sequences of many 64-wide heads, 4 x 32 of 12796 tokens, causal, 8-bit, 2.22 ms and 2.96.
//   Self-attention with D = 128 and tile = 128 has two kernels that own whole query tiles: one a workgroup and two workgroups a CU (attn_fwd_tile.hip), or
// two a workgroup of the whole CU (attn_fwd_pp.hip), which reads K and V half as often and is 1 to 7 % faster where either fills
// the chip evenly.  Half as large workgroups fill it more evenly: without the mask the chip works in rounds of 512 or 256
// workgroups, and a round that leaves one a CU takes 0.8 of a full one (32 heads of 2560 tokens, diag, 106 us in pairs, 86 in
// single tiles; 64 of 1500 76, 61; 32 of 4096 174, 172); under the mask 512 workgroups or fewer run in one round, a long row beside
// a short one (8 heads of 8192, 126 and 108; 32 of 2048 45 and 38); with 384 to 640 workgroups single tiles take 0.95 of the time where
// they are chosen, with 640 to 768 0.98 to 1.01, with 768 to 1024 1.04 and with more 0.98 to 1.0, so from there on pairs.  The constants are
// those with the least time lost over 1529 shapes of 700 to 20 000 tokens (all types, 1 - 256 heads); over 830 others (whole calls) the choice
// takes 1.4 % longer than the fastest kernel, which is what the fastest one besides the single tiles takes, too.  Where lengths differ, and
// unmasked below six tiles, the single-tile kernel is not among the candidates, and MPSA_ATTN_GENERAL, which is it there behind a
// quantization of Q, is priced as the kernel of attn_fwd_kernel.h: its constants are too high for D = 128 and tile = 128.
static int fastest_kernel(int64_t B, int64_t Hq, bool paired, bool fits, int64_t nq, int64_t nk, int64_t D, int tile, int causal) {
    const bool d128 = D == 128;
    auto tiles = [](int64_t n, int64_t t) { return (n + t - 1) / t; };
    const double heads = (double)(B * Hq);
    const int64_t qb = tiles(nq, 32), kb = tiles(nk, 32);
    struct Cost { int splits; double fixed, full, alone, places; };
    static const Cost costs[2][3] = {{{1, 3.6, 0.62, 0.41, 768.0}, {2, 3.6, 0.74, 0.44, 768.0}, {4, 3.4, 0.52, 0.44, 512.0}},
                                     {{1, 5.6, 0.85, 0.49, 512.0}, {2, 5.4, 0.86, 0.42, 512.0}, {4, 4.3, 0.48, 0.51, 256.0}}};
    double least = 1e300;
    int kernel = MPSA_ATTN_GENERAL;
    auto candidate = [&](int name, double us) {
        if (us < least) {
            least = us;
            kernel = name;
        }
    };
    for (const Cost& c : costs[d128]) {
        const double wgs = heads * (double)tiles(qb, 4 / c.splits), stages = (double)tiles(kb, c.splits);
        double load = wgs / c.places;
        if (c.splits == 4)    load = (double)(int64_t)(load + 1.0 - 1e-9);        // one workgroup a CU: whole rounds
        else if (load < 1.0)  load = 1.0;
        const double spread = c.fixed * load + c.full * wgs * (causal ? 0.5 * ((double)kb / c.splits + 1.0) : stages) / c.places;
        const double longest = c.fixed + c.alone * stages, us = spread > longest ? spread : longest;
        if (fits) candidate(c.splits == 1 ? MPSA_ATTN_SHORT1 : c.splits == 2 ? MPSA_ATTN_SHORT2 : MPSA_ATTN_SHORT4, us);
    }

    const double ntq = (double)tiles(nq, tile), ntk = (double)tiles(nk, tile);
    if (paired) {
        const double pairs = heads * (double)((int64_t)(ntq + 1.0) / 2), one = 10.4 + 1.61 * ntk;
        if (!causal)           candidate(MPSA_ATTN_PAIRED, (double)tiles((int64_t)pairs, 256) * one);
        else if (pairs <= 256.0)  candidate(MPSA_ATTN_PAIRED, one);
        else                      candidate(MPSA_ATTN_PAIRED, 24.0 + 2.1 * pairs * (ntk + 2.0) / 2.0 / 256.0);
        const double wgs = heads * ntq, rest = wgs - 512.0 * (double)(int64_t)(wgs / 512.0);
        const double rounds = (wgs - rest) / 512.0 + (rest == 0.0 ? 0.0 : rest <= 256.0 ? 0.8 : 1.0);
        const double longest = wgs > 256.0 ? 10.1 + 1.3 * ntk : 4.4 + 1.36 * ntk, spread = 12.1 + 0.31 * ntk + 2.1 * wgs * (ntk + 1.0) / 2.0 / 512.0;
        if (!causal)            candidate(MPSA_ATTN_TILE, rounds * (10.3 + 1.66 * ntk));
        else if (wgs <= 640.0)  candidate(MPSA_ATTN_TILE, spread > longest ? spread : longest);
    } else {                                                  // attn_fwd_kernel.h (fitted before attn_fwd_tile.hip was), and Q's quantization in front of it
        const bool t128 = tile == 128;
        const double wgs = heads * ntq, steps = wgs * (causal ? (ntk + 1.0) / 2.0 : ntk);
        const double step = t128 ? (d128 ? 1.5 : 1.2) : (d128 ? 0.6 : 0.45), slots = d128 && t128 ? 512.0 : 1024.0;
        const double full = 8.0 * wgs / slots + step * steps / 256.0, one = 8.0 + (t128 ? 1.0 : 0.75) * ntk;
        candidate(MPSA_ATTN_GENERAL, (full > one ? full : one) + 1.0 + heads * (double)nq * (double)D * 3.5 / 4.5e6);
    }
    return kernel;
}

// MPSA_ATTN_PP=0 in the environment leaves every call to the general kernel
static bool general_only() {
    static const bool on = [] {
        const char* v = getenv("MPSA_ATTN_PP");
        return v && v[0] == '0';
    }();
    return on;
}

extern "C" int mpsa_attn_kernel(int kernel, int64_t B, int64_t Hq, int64_t Hkv, int64_t nq, int64_t nk, int64_t D, int tile, int causal, int mode) {
    if (B <= 0 || Hq <= 0 || Hkv <= 0 || nq <= 0 || nk <= 0 || Hq % Hkv)
        return mpsa_fail(MPSA_EINVAL, "attn: bad shape (B=%lld Hq=%lld Hkv=%lld nq=%lld nk=%lld)", (long long)B, (long long)Hq, (long long)Hkv, (long long)nq, (long long)nk);
    if ((D != 64 && D != 128) || (tile != 64 && tile != 128)) return mpsa_fail(MPSA_EUNSUPPORTED, "attn: D=%lld tile=%d (both must be 64 or 128)", (long long)D, tile);
    if (mode < MPSA_MODE_MXFP4 || mode > MPSA_MODE_MIXED) return mpsa_fail(MPSA_EINVAL, "attn: unknown mode %d", mode);
    const bool listed = mode == MPSA_MODE_ROUTED;         // visiting lists: the general kernel's
    const bool paired = !listed && nq == nk && mpsa_attn_fwd_q16_supported(B, Hq, Hkv, nk, D, tile, causal, mode);
    const bool fits = (double)(B * Hq) * (double)((nq + 31) / 32) < SHORT_LIMIT;
    switch (kernel) {
        case MPSA_ATTN_AUTO: case MPSA_ATTN_SEQUENCE: {
            if (listed || general_only()) return MPSA_ATTN_GENERAL;
            return fastest_kernel(kernel == MPSA_ATTN_AUTO ? B : 1, Hq, paired, fits, nq, nk, D, tile, causal);
        }
        case MPSA_ATTN_GENERAL: return kernel;
        case MPSA_ATTN_TILE:
            if (!listed && attn_tile_supported(D, tile)) return kernel;
            return mpsa_fail(MPSA_EUNSUPPORTED, "attn: the tile kernel by its own name takes D = 128 and tile = 128, and no visiting lists");
        case MPSA_ATTN_PAIRED:
            if (paired) return kernel;
            return mpsa_fail(MPSA_EUNSUPPORTED, "attn: the paired-tile kernel takes self-attention with D = 128 and tile = 128, causal from two tiles on, unmasked from six, and no visiting lists");
        case MPSA_ATTN_SHORT1: case MPSA_ATTN_SHORT2: case MPSA_ATTN_SHORT4:
            if (!listed && fits) return kernel;
            return mpsa_fail(MPSA_EUNSUPPORTED, "attn: the short-sequence kernel takes no visiting lists, and at most %d blocks of 32 queries", (int)SHORT_LIMIT - 1);
        default: return mpsa_fail(MPSA_EINVAL, "attn: unknown kernel %d", kernel);
    }
}
