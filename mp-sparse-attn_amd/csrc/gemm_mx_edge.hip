// The 256 x 256 kernel's instantiations for ragged M and N, and for 4-bit products with row-major scales that end in half a unit (gemm_mx_kernel.h).
#include "gemm_mx_kernel.h"

namespace {

template <int FMT, int FMTB, typename OutT>
void launch_scales(const GemmArgs& g, dim3 grid, hipStream_t st) {
    if constexpr (FMT == MPSA_FMT_E2M1) {
        if (g.K % 256) return g.packed ? launch_kernel<FMT, FMTB, OutT, false, true, true, true>(g, grid, st) : launch_kernel<FMT, FMTB, OutT, true, false, true, true>(g, grid, st);
    }
    if (g.packed)            launch_kernel<FMT, FMTB, OutT, false, true, true>(g, grid, st);
    else if (g.K % 512 == 0) launch_kernel<FMT, FMTB, OutT, false, false, true>(g, grid, st);
    else                     launch_kernel<FMT, FMTB, OutT, true, false, true>(g, grid, st);
}

template <int FMT, int FMTB>
void launch_fmt(const GemmArgs& g, int c_dtype, dim3 grid, hipStream_t st) {
    if (c_dtype == MPSA_BF16)        launch_scales<FMT, FMTB, __bf16>(g, grid, st);
    else if (c_dtype == MPSA_F8E5M2) launch_scales<FMT, FMTB, OutE5M2>(g, grid, st);
    else if (c_dtype == MPSA_F16)    launch_scales<FMT, FMTB, _Float16>(g, grid, st);
    else                             launch_scales<FMT, FMTB, float>(g, grid, st);
}

}  // namespace

void gemm_edge_launch(const GemmArgs& g, int64_t batches, int fmt_a, int fmt_b, int c_dtype, hipStream_t st) {
    const dim3 grid((unsigned)(((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN)), (unsigned)batches);
    const bool mixed = fmt_a != fmt_b;
    if (fmt_a == MPSA_FMT_E2M1)      launch_fmt<MPSA_FMT_E2M1, MPSA_FMT_E2M1>(g, c_dtype, grid, st);
    else if (fmt_a == MPSA_FMT_E4M3) mixed ? launch_fmt<MPSA_FMT_E4M3, MPSA_FMT_E2M1>(g, c_dtype, grid, st) : launch_fmt<MPSA_FMT_E4M3, MPSA_FMT_E4M3>(g, c_dtype, grid, st);
    else                             mixed ? launch_fmt<MPSA_FMT_E5M2, MPSA_FMT_E2M1>(g, c_dtype, grid, st) : launch_fmt<MPSA_FMT_E5M2, MPSA_FMT_E5M2>(g, c_dtype, grid, st);
}
