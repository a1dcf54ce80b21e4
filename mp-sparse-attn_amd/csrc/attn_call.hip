// One native call per attention call: the sequence-mean, preparation, routing and attention launches of
// ours/mxfp_attn_kernel.py::mxfp_attn_kernel behind one entry point with one workspace.
//
// What bounds a short call is the host: sixteen allocations, twenty context switches and six foreign calls of Python took
// 47 us for a 160-token prefill whose kernels took 15.  A caller keeps a description of the shapes (mpsa_attn_desc), hands
// over pointers and one block of memory, and everything else -- offsets into that block, which kernels run, their
// arguments -- happens here in about a microsecond next to the launches themselves.
#include "attn_common.h"

namespace {

// Byte offsets into the workspace, -1 where a call does not need the buffer.
struct Layout {
    int64_t q4, qs4, q8, qs8, k4, ks4, k8, ks8, v, mean, mean_work, work, cls, order, counts, skipped, total;
    int kernel;                       // MPSA_ATTN_*
    bool fuse_q;                      // Q quantized inside the attention kernel
    bool routed, ahead;               // tile router; skipping decided ahead
    int64_t ntq, ntk;
};

int64_t tiles(int64_t n, int tile) { return (n + tile - 1) / tile; }

int plan(int kernel, const mpsa_attn_desc* d, Layout* l) {
    if (!d) return mpsa_fail(MPSA_EINVAL, "attn call: null description");
    if (d->B <= 0 || d->Hq <= 0 || d->Hkv <= 0 || d->nq <= 0 || d->nk <= 0 || d->Hq % d->Hkv)
        return mpsa_fail(MPSA_EINVAL, "attn call: bad shape (B=%lld Hq=%lld Hkv=%lld nq=%lld nk=%lld)", (long long)d->B, (long long)d->Hq, (long long)d->Hkv, (long long)d->nq, (long long)d->nk);
    if ((d->D != 64 && d->D != 128) || (d->tile != 64 && d->tile != 128)) return mpsa_fail(MPSA_EUNSUPPORTED, "attn call: D=%lld tile=%d (both must be 64 or 128)", (long long)d->D, d->tile);
    if (d->mode < MPSA_MODE_MXFP4 || d->mode > MPSA_MODE_MIXED) return mpsa_fail(MPSA_EINVAL, "attn call: unknown mode %d", d->mode);
    l->routed = d->mode == MPSA_MODE_ROUTED;
    const bool skip = d->skip && !l->routed;
    l->ahead = skip && mpsa_skip_route_supported(d->nq, d->nk, d->D, d->tile, d->causal, d->mode);
    l->kernel = mpsa_attn_kernel(kernel, d->B, d->Hq, d->Hkv, d->nq, d->nk, d->D, d->tile, d->causal, d->mode);
    if (l->kernel < 0) return l->kernel;
    if (skip) {                       // the general kernel's, ahead of it or inside
        if (kernel != MPSA_ATTN_AUTO && kernel != MPSA_ATTN_SEQUENCE && l->kernel != MPSA_ATTN_GENERAL) return mpsa_fail(MPSA_EUNSUPPORTED, "attn call: tile skipping runs on the general kernel");
        l->kernel = MPSA_ATTN_GENERAL;
    }
    l->fuse_q = l->kernel != MPSA_ATTN_GENERAL;
    l->ntq = tiles(d->nq, d->tile);
    l->ntk = tiles(d->nk, d->tile);
    int64_t at = 0;
    auto take = [&](bool needed, int64_t bytes) {
        if (!needed) return (int64_t)-1;
        const int64_t o = at;
        at += (bytes + 255) & ~(int64_t)255;
        return o;
    };
    const int64_t qrows = d->B * d->Hq * l->ntq * d->tile, krows = d->B * d->Hkv * l->ntk * d->tile;
    // the mixed mode multiplies 8-bit Q with 4-bit K; the others use one set or both on either side
    const bool q4 = d->mode != MPSA_MODE_MXFP8 && d->mode != MPSA_MODE_MIXED, q8 = d->mode != MPSA_MODE_MXFP4;
    const bool k4 = d->mode != MPSA_MODE_MXFP8, k8 = d->mode != MPSA_MODE_MXFP4 && d->mode != MPSA_MODE_MIXED;
    l->q4 = take(q4 && !l->fuse_q, qrows * d->D / 2);
    l->qs4 = take(q4 && !l->fuse_q, qrows * d->D / 32);
    l->q8 = take(q8 && !l->fuse_q, qrows * d->D);
    l->qs8 = take(q8 && !l->fuse_q, qrows * d->D / 32);
    l->k4 = take(k4, krows * d->D / 2);
    l->ks4 = take(k4, krows * d->D / 32);
    l->k8 = take(k8, krows * d->D);
    l->ks8 = take(k8, krows * d->D / 32);
    l->v = take(true, krows * d->D * 2);
    l->mean = take(d->smooth_k, d->B * d->Hkv * d->D * 2);
    l->mean_work = take(d->smooth_k, mpsa_seq_mean_workspace(d->B, d->Hkv, d->nk, d->D));
    const int64_t pairs = d->B * d->Hq * l->ntq * l->ntk, rows = d->B * d->Hq * l->ntq;
    l->work = take(l->routed || l->ahead, l->routed ? mpsa_route_workspace(d->B, d->Hq, d->Hkv, d->nq, d->nk, d->D, d->tile)
                                                    : mpsa_skip_route_workspace(d->B, d->Hq, d->nq, d->nk, d->tile));
    l->cls = take(l->routed, pairs);
    l->order = take(l->routed || l->ahead, pairs * 4);
    l->counts = take(l->routed || l->ahead, rows * 16);
    l->skipped = take(skip && !l->ahead, rows * 4);
    l->total = at;
    return MPSA_OK;
}

// Share of the visited (query tile, key tile) pairs that a run left out: from the visiting lists' lengths (four a query
// tile) or from the skip counts (one a query tile).  One workgroup: a few thousand words at most tens of thousands.
__global__ __launch_bounds__(1024) void skipped_share_kernel(const int32_t* words, int64_t n, int64_t visited, int listed, float* share) {
    __shared__ long long part[16];
    long long s = 0;
    for (int64_t i = threadIdx.x; i < n; i += 1024) s += words[i];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 16; ++w) s += part[w];
        *share = (float)(listed ? visited - s : s) / (float)visited;
    }
}

}  // namespace

extern "C" int64_t mpsa_attn_call_workspace_on(int kernel, const mpsa_attn_desc* d) {
    Layout l;
    const int rc = plan(kernel, d, &l);
    return rc == MPSA_OK ? l.total : (int64_t)rc;
}

extern "C" int64_t mpsa_attn_call_workspace(const mpsa_attn_desc* d) { return mpsa_attn_call_workspace_on(MPSA_ATTN_AUTO, d); }

extern "C" int mpsa_attn_call_on(int kernel, const mpsa_attn_desc* d, const void* q, const void* k, const void* v, void* o, void* workspace,
                                 float* skipped_share, mpsa_stream_t stream) {
    Layout l;
    int rc = plan(kernel, d, &l);
    if (rc != MPSA_OK) return rc;
    if (!q || !k || !v || !o || !workspace) return mpsa_fail(MPSA_EINVAL, "attn call: null pointer");
    if (!mpsa_aligned16(workspace)) return mpsa_fail(MPSA_EALIGN, "attn call: the workspace must be 16-byte aligned");
    if (!skipped_share && attn_prompt_supported(d, l.kernel, q, k, v, o)) return attn_prompt_launch(d, q, k, v, o, (hipStream_t)stream);
    uint8_t* const w = static_cast<uint8_t*>(workspace);
    auto at = [&](int64_t off) { return off < 0 ? nullptr : w + off; };
    uint8_t *q4 = at(l.q4), *qs4 = at(l.qs4), *q8 = at(l.q8), *qs8 = at(l.qs8), *k4 = at(l.k4), *ks4 = at(l.ks4), *k8 = at(l.k8), *ks8 = at(l.ks8);
    int32_t *order = reinterpret_cast<int32_t*>(at(l.order)), *counts = reinterpret_cast<int32_t*>(at(l.counts)), *skipped = reinterpret_cast<int32_t*>(at(l.skipped));
    MeanSource mean = MEAN_NONE;
    const void* k_sub = nullptr;
    if (d->smooth_k) {
        mean = mpsa_mean_source(d->B, d->Hkv, d->nk, d->D);
        float* const sums = reinterpret_cast<float*>(at(l.mean_work));
        k_sub = mean == MEAN_SUMS ? static_cast<const void*>(sums) : at(l.mean);
        if (mean == MEAN_GIVEN)     rc = mpsa_seq_mean(k, d->dtype, d->B, d->Hkv, d->nk, d->D, d->k_strides, sums, at(l.mean), stream);
        else if (mean == MEAN_SUMS) rc = mpsa_seq_mean_partial(k, d->dtype, d->B, d->Hkv, d->nk, d->D, d->k_strides, sums, (hipStream_t)stream);
        if (rc != MPSA_OK) return rc;
    }
    rc = mpsa_prepare_operands(l.fuse_q ? nullptr : q, d->q_strides, k, d->k_strides, v, d->v_strides, d->dtype, d->B, d->Hq, d->Hkv, d->nq, d->nk,
                               d->D, d->tile, d->fmt8, d->pre_scale_q, mean, k_sub, l.q4 >= 0, l.q8 >= 0, l.k4 >= 0, l.k8 >= 0, q4, qs4, q8, qs8, k4, ks4, k8, ks8, at(l.v), (hipStream_t)stream);
    if (rc != MPSA_OK) return rc;
    if (l.fuse_q) {
        rc = mpsa_attn_fwd_q16_on(l.kernel, q, d->q_strides, d->dtype, d->pre_scale_q, k4, ks4, k8, ks8, d->fmt8, at(l.v), d->dtype, o, d->o_dtype, d->o_strides,
                                  d->B, d->Hq, d->Hkv, d->nq, d->nk, d->D, d->tile, d->causal, d->mode, stream);
    } else if (l.routed || l.ahead) {
        rc = l.routed ? mpsa_route_tiles(qs4, ks4, d->B, d->Hq, d->Hkv, d->nq, d->nk, d->D, d->tile, d->causal, d->route_thresh, d->skip ? d->skip_thresh : 0.0f,
                                         at(l.work), at(l.cls), order, counts, stream)
                      : mpsa_skip_route(q4, qs4, q8, qs8, k4, ks4, k8, ks8, d->fmt8, d->B, d->Hq, d->Hkv, d->nq, d->nk, d->D, d->tile, d->causal, d->mode,
                                        d->skip_thresh, at(l.work), nullptr, order, counts, nullptr, stream);
        if (rc != MPSA_OK) return rc;
        rc = mpsa_attn_fwd_routed(q4, qs4, q8, qs8, k4, ks4, k8, ks8, d->fmt8, at(l.v), d->dtype, o, d->o_dtype, d->o_strides,
                                  d->B, d->Hq, d->Hkv, d->nq, d->nk, d->D, d->tile, d->causal, order, counts, stream);
    } else if (d->skip) {
        rc = mpsa_attn_fwd_skip(q4, qs4, q8, qs8, k4, ks4, k8, ks8, d->fmt8, at(l.v), d->dtype, o, d->o_dtype, d->o_strides,
                                d->B, d->Hq, d->Hkv, d->nq, d->nk, d->D, d->tile, d->causal, d->mode, d->skip_thresh, skipped, stream);
    } else {
        rc = mpsa_attn_fwd_on(l.kernel, q4, qs4, q8, qs8, k4, ks4, k8, ks8, d->fmt8, at(l.v), d->dtype, o, d->o_dtype, d->o_strides,
                              d->B, d->Hq, d->Hkv, d->nq, d->nk, d->D, d->tile, d->causal, d->mode, stream);
    }
    if (rc != MPSA_OK || !skipped_share) return rc;
    const int64_t rows = d->B * d->Hq * l.ntq;
    const int64_t visited = d->B * d->Hq * (d->causal ? l.ntq * (l.ntq + 1) / 2 : l.ntq * l.ntk);
    const bool lists = l.routed || l.ahead;
    if (!lists && !skipped) return mpsa_fail(MPSA_EINVAL, "attn call: a share of skipped tiles needs a run that skips or routes");
    hipLaunchKernelGGL(skipped_share_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, lists ? counts : skipped, lists ? rows * 4 : rows, visited, lists ? 1 : 0, skipped_share);
    MPSA_CHECK_LAUNCH("attn call (skipped share)");
    return MPSA_OK;
}

extern "C" int mpsa_attn_call(const mpsa_attn_desc* d, const void* q, const void* k, const void* v, void* o, void* workspace,
                              float* skipped_share, mpsa_stream_t stream) {
    return mpsa_attn_call_on(MPSA_ATTN_AUTO, d, q, k, v, o, workspace, skipped_share, stream);
}
