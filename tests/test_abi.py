"""The C-ABI library loads, exports every symbol include/mpsa.h declares, and rejects bad arguments on the
host (no kernel is launched; runs without a GPU)."""
import ctypes
import os
import re
import subprocess
import sys

import pytest
import torch

from conftest import ROOT
from ours import _lib


def _declared():
    text = open(os.path.join(ROOT, "include", "mpsa.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(mpsa_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol():
    names = _declared()
    assert "mpsa_attn_fwd" in names and "mpsa_quantize_mx" in names and len(names) >= 11
    handle = ctypes.CDLL(_lib.LIB_PATH)
    for n in names:
        assert hasattr(handle, n), f"{n} declared in mpsa.h but not exported"
    assert sorted(_lib.SIGNATURES) == names
    assert _lib.lib().mpsa_version() >= 100


def test_host_side_argument_validation():
    L = _lib.lib()
    null = ctypes.c_void_p(0)
    one = ctypes.c_void_p(16)           # never dereferenced: validation fails first
    st = (ctypes.c_int64 * 4)(1, 1, 32, 1)
    assert L.mpsa_quantize_mx(null, 0, 1, 1, 1, 32, st, null, 1.0, 4, 3, one, one, 1, null) == -1
    assert b"null" in L.mpsa_last_error()
    st_ok = (ctypes.c_int64 * 4)(64, 64, 64, 1)
    assert L.mpsa_quantize_mx(one, 0, 1, 1, 1, 48, st_ok, null, 1.0, 4, 3, one, one, 1, null) == -1      # D % 32
    assert L.mpsa_quantize_mx(one, 2, 1, 1, 1, 64, st_ok, null, 1.0, 4, 3, one, one, 1, null) == -1      # f32 input
    assert L.mpsa_quantize_mx(one, 0, 1, 1, 1, 64, st_ok, null, 1.0, 9, 3, one, one, 1, null) == -1      # bad format
    assert L.mpsa_quantize_mx(one, 0, 1, 1, 2, 64, st_ok, null, 1.0, 4, 3, one, one, 1, null) == -1      # out_rows < N
    assert L.mpsa_quantize_mx(ctypes.c_void_p(24), 0, 1, 1, 1, 64, st_ok, null, 1.0, 4, 3, one, one, 1, null) == -2
    assert L.mpsa_quantize_mx(one, 0, 1, 1, 1, 64, st_ok, ctypes.c_void_p(8), 1.0, 4, 3, one, one, 1, null) == -2   # sub alignment
    assert L.mpsa_seq_mean_workspace(2, 3, 1000, 64) == 2 * 3 * 4 * 64 * 4
    assert L.mpsa_seq_mean(one, 0, 1, 1, 8, 64, st_ok, null, one, null) == -1                      # no workspace
    assert L.mpsa_seq_mean(one, 0, 1, 1, 8, 96, st_ok, one, one, null) == -3                       # D = 96
    assert L.mpsa_gemm_mx(one, one, 4, one, one, 4, 100, 256, 96, one, 0, 256, null) == -3         # K % 64
    assert L.mpsa_gemm_mx(one, one, 4, one, one, 4, 256, 256, 128, one, 7, 256, null) == -1        # bad dtype
    assert L.mpsa_gemm_mx(one, one, 4, one, one, 3, 256, 256, 128, one, 0, 256, null) == -1        # bad format of B
    assert L.mpsa_gemm_mx_packed(one, one, 4, one, one, 4, 100, 256, 128, one, 0, 256, null) == -3  # packed: M % 128
    assert L.mpsa_fp8_encode(null, 4, 0, one, null) == -1
    assert L.mpsa_fp8_encode(one, 4, 4, one, null) == -1                                           # E2M1 is not an FP8 format
    assert L.mpsa_seq_mean_static(one, 0, 1, 64, 262144, 128, st_ok, one, null) == -3              # beyond the built-in array
    assert L.mpsa_v_tiles(one, 0, 1, 1, 128, 96, st_ok, 128, one, null) == -3                      # D = 96
    so = (ctypes.c_int64 * 4)(128 * 128, 128 * 128, 128, 1)
    args = [one] * 8 + [0, one, 0, one, 0, so, 1, 4, 3, 128, 128, 128, 128, 1, 2, null]
    assert L.mpsa_attn_fwd(*args) == -1                                                            # Hq % Hkv
    args = [null] * 4 + [one] * 4 + [0, one, 0, one, 0, so, 1, 4, 2, 128, 128, 128, 128, 1, 2, null]
    assert L.mpsa_attn_fwd(*args) == -1                                                            # diag needs 4-bit Q
    args = [one] * 8 + [0, one, 0, one, 0, so, 1, 4, 2, 128, 128, 96, 128, 1, 2, null]
    assert L.mpsa_attn_fwd(*args) == -3                                                            # D = 96
    args = [one] * 8 + [0, one, 0, one, 0, so, 1, 4, 2, 128, 256, 128, 128, 1, 0, null]
    assert L.mpsa_attn_fwd(*args) == -1                                                            # causal with nq != nk
    # tile skipping ahead of the attention kernel: the shapes it takes, the operands a mode multiplies, the lists' memory
    assert L.mpsa_skip_route_supported(8192, 8192, 128, 128, 1, 2) == 1 and L.mpsa_skip_route_supported(8192, 8192, 64, 128, 1, 2) == 0
    assert L.mpsa_skip_route_supported(8192, 8192, 128, 128, 1, 4) == 0                            # the mixed type
    assert L.mpsa_skip_route_supported(300, 77, 128, 128, 0, 0) == 1 and L.mpsa_skip_route_supported(300, 77, 128, 128, 0, 2) == 0
    assert L.mpsa_skip_route_supported(128 * 2049, 128 * 2049, 128, 128, 1, 0) == 0                # more key tiles than its LDS holds
    assert L.mpsa_skip_route_workspace(1, 4, 1000, 300, 128) == 4 * 8 * 3 * 4
    shape = [0, 1, 4, 2, 1024, 1024, 128, 128, 1]
    assert L.mpsa_skip_route(*([one] * 8 + shape + [4, 1.0, one, null, one, one, null, null])) == -3          # mixed
    assert L.mpsa_skip_route(*([one, one, null, null] + [one] * 4 + shape + [2, 1.0, one, null, one, one, null, null])) == -1   # diag without 8-bit Q
    assert L.mpsa_skip_route(*([one] * 8 + shape + [2, float("nan"), one, null, one, one, null, null])) == -1
    assert L.mpsa_skip_route(*([one] * 8 + shape + [2, 1.0, null, null, one, one, null, null])) == -1           # no workspace
    assert L.mpsa_skip_route(*([one] * 8 + shape + [2, 1.0, one, null, ctypes.c_void_p(18), one, null, null])) == -2   # order misaligned
    so2 = (ctypes.c_int64 * 4)(128 * 128, 128 * 128, 128, 1)
    routed = [one, one, null, one] + [one] * 4 + [0, one, 0, one, 0, so2, 1, 4, 2, 128, 128, 128, 128, 1, one, one, null]
    assert L.mpsa_attn_fwd_routed(*routed) == -1 and b"whole" in L.mpsa_last_error()               # half an operand set
    assert L.mpsa_e2m1_pack(null, 2, 3, 4, one, null) == -1                                         # null input
    assert L.mpsa_e2m1_pack(null, 0, 3, 4, null, null) == 0                                         # empty is fine
    assert L.mpsa_e2m1_encode(null, 4, one, null) == -1
    assert L.mpsa_e2m1_encode(null, 0, null, null) == 0                                            # empty is fine


def test_the_two_tensor_entry_points_refuse_what_two_calls_would():
    """mpsa_quantize_mx_pair and mpsa_e2m1_pack_pair, either operand bad: null jobs and pointers, shapes, formats, strides and
    alignment; what is empty on both sides is done without a launch."""
    L = _lib.lib()
    P = ctypes.pointer

    def job(x=16, B=1, H=2, N=128, D=128, strides=None, fmt=4, codes=16, scales=16, rows=None):
        return _lib.QuantizeJob(x, B, H, N, D, (ctypes.c_int64 * 4)(*(strides or (H * N * D, N * D, D, 1))), 1.0, fmt, 3 if fmt == 4 else 7, codes, scales, N if rows is None else rows)

    def pair(a, b, dtype=0, per_byte=0, five=0):
        return L.mpsa_quantize_mx_pair(a and P(a), b and P(b), dtype, per_byte, five, None)

    assert pair(None, job()) == -1 and pair(job(), None) == -1 and b"null job" in L.mpsa_last_error()
    assert pair(job(), job(), dtype=2) == -1                                                       # f32 inputs
    for bad, status in ((job(x=None), -1), (job(codes=None), -1), (job(scales=None), -1), (job(fmt=9), -1), (job(fmt=2), -1), (job(D=48), -1), (job(rows=127), -1),
                        (job(B=-1), -1), (job(strides=(32768, 16384, 128, 2)), -1), (job(x=24), -2), (job(strides=(32768, 16384, 132, 1)), -2), (job(codes=24), -2),
                        (job(H=65536), -3)):
        assert pair(bad, job(fmt=0)) == status and pair(job(fmt=1), bad) == status
    for five in (job(N=127), job(D=96)):                                                           # packed scales: rows and D in multiples of 128
        assert pair(five, job(), five=1) == -3 and pair(job(), five, five=1) == -3
    assert pair(job(N=0, x=None, codes=None, scales=None), job(B=0, x=None, codes=None, scales=None)) == 0

    one, null = ctypes.c_void_p(16), ctypes.c_void_p(0)
    pack = lambda a, na, pa, b, nb, pb: L.mpsa_e2m1_pack_pair(a, 1, na, pa, b, 1, nb, pb, None)
    assert pack(null, 16, one, one, 16, one) == -1 and pack(one, 16, null, one, 16, one) == -1
    assert pack(one, -1, one, one, 16, one) == -1 and pack(null, 0, null, null, 16, one) == -1 and pack(null, 0, null, one, -2, one) == -1
    assert pack(null, 0, null, null, 0, null) == 0


def test_python_entry_points_refuse_cpu_tensors_and_bad_arguments():
    from ours.mxfp import MXFP4Tensor, MXScaleTensor
    from ours.mxfp_attn import mxfp_attn
    from ours.mxfp_attn_kernel import mxfp_attn_kernel
    from ours.block_scaled_matmul import block_scaled_matmul, make_configs
    x = torch.zeros(1, 2, 128, 64, dtype=torch.bfloat16)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        mxfp_attn(x, x, x)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        MXFP4Tensor(data=torch.zeros(4))
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        MXScaleTensor(data=torch.ones(4))
    with pytest.raises(AssertionError, match="seq_len"):
        mxfp_attn(x[:, :, :64], x[:, :, :64], x[:, :, :64])
    with pytest.raises(AssertionError, match="headdim"):
        mxfp_attn(torch.zeros(1, 2, 128, 96), torch.zeros(1, 2, 128, 96), torch.zeros(1, 2, 128, 96))
    with pytest.raises(ValueError):
        MXFP4Tensor()
    with pytest.raises(ValueError, match="Unsupported dtype"):
        block_scaled_matmul(x, x, x, x, torch.int8, 256, 256, 128, make_configs("mxfp4"))
    with pytest.raises(ValueError, match="Invalid block scale type"):
        make_configs("nvfp4")
    assert make_configs("mixed")["ELEM_PER_BYTE_A"] == 1 and make_configs("mixed")["ELEM_PER_BYTE_B"] == 2
    t = MXFP4Tensor(data=torch.arange(16, dtype=torch.uint8).reshape(2, 8), dtype=torch.uint8)
    with pytest.raises(RuntimeError, match="no CPU"):
        t.to_packed_tensor(dim=1)


def test_kernels_by_name():
    """Which kernel a call takes, and what a named kernel refuses."""
    L, A, G = _lib.lib(), _lib.ATTN_KERNELS, _lib.GEMM_KERNELS
    attn = lambda kernel, B, Hq, Hkv, nq, nk, D, tile, causal, mode: L.mpsa_attn_kernel(A[kernel], B, Hq, Hkv, nq, nk, D, tile, causal, mode)
    assert attn("auto", 1, 32, 8, 160, 160, 128, 128, 1, _lib.MODE_DIAG) == A["short4"]
    assert attn("auto", 1, 32, 8, 1000, 1000, 128, 128, 1, _lib.MODE_DIAG) == A["short2"]
    assert attn("auto", 1, 32, 8, 8192, 8192, 128, 128, 1, _lib.MODE_DIAG) == A["paired"]
    assert attn("auto", 2, 16, 16, 4096, 333, 128, 128, 0, _lib.MODE_MXFP8) == A["short1"]
    # many queries over few keys: no end to the short-sequence kernel's range where its estimate is the better one
    for nq in (20000, 26000, 26300, 32760, 131072):
        assert attn("auto", 1, 40, 40, nq, 512, 128, 128, 0, _lib.MODE_MXFP4) == A["short1"]
    # unmasked self-attention below the paired-tile kernel's six tiles is no exception
    assert attn("auto", 1, 24, 24, 512, 512, 128, 128, 0, _lib.MODE_DIAG) == A["short2"] and attn("auto", 1, 8, 8, 300, 300, 128, 128, 0, _lib.MODE_MXFP4) == A["short4"]
    assert attn("short1", 64, 64, 64, 131072, 512, 128, 128, 0, _lib.MODE_MXFP4) == -3            # a launch's 2^32 threads
    assert attn("auto", 1, 40, 40, 32760, 32760, 128, 128, 0, _lib.MODE_ROUTED) == A["general"]
    for B in (1, 2, 4, 8, 64):
        assert attn("sequence", B, 32, 8, 200, 200, 128, 128, 1, _lib.MODE_DIAG) == attn("auto", 1, 32, 8, 200, 200, 128, 128, 1, _lib.MODE_DIAG)
        assert attn("sequence", B, 4, 4, 512, 512, 128, 128, 0, _lib.MODE_ROUTED) == A["general"]
    for kernel, i in A.items():
        if kernel not in ("auto", "sequence"):
            assert attn(kernel, 1, 8, 2, 1100, 1100, 128, 128, 1, _lib.MODE_DIAG) == i
    assert attn("paired", 1, 8, 2, 1100, 1100, 64, 128, 1, _lib.MODE_DIAG) == -3 and attn("paired", 1, 8, 2, 640, 640, 128, 128, 0, _lib.MODE_DIAG) == -3
    assert attn("short1", 1, 8, 2, 1100, 1100, 128, 128, 1, _lib.MODE_ROUTED) == -3 and attn("paired", 1, 8, 2, 1100, 1100, 128, 128, 1, _lib.MODE_ROUTED) == -3
    assert L.mpsa_attn_kernel(9, 1, 8, 2, 1100, 1100, 128, 128, 1, _lib.MODE_DIAG) == -1 and attn("auto", 1, 8, 3, 1100, 1100, 128, 128, 1, _lib.MODE_DIAG) == -1
    gemm = lambda kernel, fa, fb, M, N, K, heads=1: L.mpsa_gemm_kernel(G[kernel], fa, fb, 1, heads, M, N, K)
    assert gemm("auto", 4, 4, 16, 4096, 4096) == G["split1x1"] and gemm("split", 4, 4, 16, 4096, 4096) == G["split1x1"]
    assert gemm("auto", 0, 4, 1000, 14336, 4096) == G["tile256"] and gemm("auto", 4, 4, 8192, 8192, 8192) == G["tile256"]
    assert gemm("auto", 4, 4, 1000, 4096, 4096) == G["tile128"] and gemm("auto", 4, 4, 2048, 2048, 128, 16) == G["general"]
    assert gemm("auto", 4, 4, 256, 256, 192) == G["general"]
    for kernel in ("split", "split1x4", "tile128", "tile256"):
        assert gemm(kernel, 4, 4, 256, 256, 192) == -3
    assert gemm("tile256", 4, 0, 256, 256, 256) == -3 and gemm("tile256", 4, 4, 300, 256, 384) == -3 and gemm("tile256", 0, 4, 300, 256, 384) == G["tile256"]
    assert L.mpsa_gemm_kernel(13, 4, 4, 1, 1, 256, 256, 256) == -1 and L.mpsa_gemm_kernel(0, 4, 4, 1, 1, 256, 256, 96) == -3


@pytest.mark.parametrize("fmt_a,fmt_b", [(4, 4), (0, 0), (1, 1), (0, 4), (4, 0)])
def test_the_kernel_that_a_product_takes_can_be_named(fmt_a, fmt_b):
    L, halves = _lib.lib(), 0
    for M in (1, 16, 100, 256, 1000, 2304, 4224, 8192):
        for N in (8, 100, 128, 1000, 4096, 4224, 16400):
            for K in (64, 128, 256, 384, 640, 1152, 4096, 4224):
                for heads in (1, 8):
                    kernel = L.mpsa_gemm_kernel(0, fmt_a, fmt_b, 1, heads, M, N, K)
                    assert kernel > 0 and L.mpsa_gemm_kernel(kernel, fmt_a, fmt_b, 1, heads, M, N, K) == kernel, (M, N, K, heads)
                    halves += kernel == _lib.GEMM_KERNELS["tile256"] and K % 256 == 128 and M % 256 > 0
    assert fmt_a != 4 or fmt_b != 4 or halves > 0


def test_the_choice_of_matmul_kernels_at_few_rows_and_narrow_shapes():
    """Shapes at which the choice was measured to cost 9 to 39 %: one stage of K, several narrow products, and narrow ones with
    many rows."""
    L, G = _lib.lib(), _lib.GEMM_KERNELS
    pick = lambda fa, fb, heads, M, N, K: L.mpsa_gemm_kernel(0, fa, fb, 1, heads, M, N, K)
    for fa, fb in ((4, 4), (0, 4), (0, 0)):
        for heads, M, N in ((1, 16, 1024), (1, 16, 4096), (1, 4096, 16), (32, 64, 64), (1, 1, 4096), (8, 10, 256)):
            assert pick(fa, fb, heads, M, N, 128) in range(11, 45)          # tiles that split K
        for heads, M, N in ((1, 512, 4096), (1, 256, 16384), (16, 512, 512), (512, 128, 128)):
            assert pick(fa, fb, heads, M, N, 128) == G["general"]
    assert pick(4, 4, 1, 2399, 169, 6400) == G["split2x4"] and pick(4, 4, 32, 46, 128, 8832) == G["split2x2"]
    assert pick(0, 0, 8, 512, 128, 9344) == G["split2x4"] and pick(0, 0, 32, 25, 4608, 11904) == G["split2x4"]
    assert pick(4, 4, 2, 927, 8586, 1408) == G["general"] and pick(4, 4, 1, 3830, 128, 6016) == G["split2x4"]
    # and shapes at which a choice with the least error of its estimates took 26 to 36 % longer
    assert pick(4, 4, 1, 619, 6784, 3072) == G["tile128"] and pick(0, 0, 1, 821, 11136, 1024) == pick(0, 0, 1, 4925, 4480, 1024) == G["tile256"]
    assert pick(0, 4, 1, 420, 3072, 12288) == pick(4, 4, 1, 859, 1536, 14080) == G["split4x4"] and pick(4, 4, 23, 1862, 194, 640) == G["general"]


@pytest.mark.parametrize("name,value", [("MPSA_ATTN_PP", "0"), ("MPSA_GEMM_GENERAL", "1")])
def test_environment_switches_leave_everything_to_the_general_kernels(name, value):
    code = ("import sys; sys.path.insert(0, %r)\nfrom ours import _lib\nL = _lib.lib()\n"
            "print([L.mpsa_attn_kernel(0, 1, 32, 8, n, n, 128, 128, 1, 2) for n in (160, 1000, 8192)],"
            " [L.mpsa_gemm_kernel(0, 4, 4, 1, 1, m, 4096, 4096) for m in (16, 1000, 8192)])" % os.path.join(ROOT, "mp-sparse-attn_amd"))
    out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, **{name: value}), capture_output=True, text=True, check=True).stdout
    assert out.split("\n")[0] == ("[1, 1, 1] [11, 3, 4]" if name == "MPSA_ATTN_PP" else "[5, 4, 2] [1, 1, 1]")


def test_python_entry_points_refuse_unknown_kernels():
    from ours.mxfp_attn_kernel import _attn_kernel_id
    from ours.block_scaled_matmul import _gemm_kernel_id
    assert _attn_kernel_id("auto") == 0 and _gemm_kernel_id(None) == 0 and _gemm_kernel_id("split4x4") == 44
    for f in (_attn_kernel_id, _gemm_kernel_id):
        with pytest.raises(ValueError, match="unknown"):
            f("fastest")
