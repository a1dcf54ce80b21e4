"""mpsa_attn_call with an output over K's or V's memory: K and V are read before anything is stored, whichever kernels run."""
import ctypes

import pytest
import torch

from conftest import make_qkv
from ours import _lib
from ours.mxfp_attn_kernel import pre_scale_q

DEV = "cuda:0"


def describe(B, Hq, Hkv, nq, nk, D=128, nhd=False, o_dtype=_lib.BF16, mode=_lib.MODE_MXFP4, causal=False, o_strides=None):
    four = ctypes.c_int64 * 4
    strides = lambda H, N: four(N * H * D, D, H * D, 1) if nhd else four(H * N * D, N * D, D, 1)  # noqa: E731
    return _lib.AttnDesc(B, Hq, Hkv, nq, nk, D, strides(Hq, nq), strides(Hkv, nk), strides(Hkv, nk), o_strides or strides(Hq, nq), _lib.BF16, o_dtype,
                         128, causal, mode, _lib.FMT_E4M3, 0, 0, pre_scale_q(D, None), 0.0, 0.0)


@pytest.mark.parametrize("nhd", [False, True])
@pytest.mark.parametrize("o_dtype, size", [(_lib.BF16, 2), (_lib.F32, 4)])
def test_one_launch_wants_an_output_apart_from_k_and_v(nhd, o_dtype, size):
    rule = getattr(_lib.lib(), "_Z21attn_prompt_supportedPK14mpsa_attn_desciPKvS3_S3_S3_")
    rule.restype, rule.argtypes = ctypes.c_bool, [ctypes.POINTER(_lib.AttnDesc), ctypes.c_int] + [ctypes.c_void_p] * 4
    desc = describe(2, 4, 2, 100, 60, nhd=nhd, o_dtype=o_dtype)
    q, k, v = 1 << 20, 2 << 20, 3 << 20
    out, kv = 2 * 4 * 100 * 128 * size, 2 * 2 * 60 * 128 * 2
    one_launch = lambda o, d=desc: rule(d, _lib.ATTN_KERNELS["short4"], q, k, v, o)  # noqa: E731
    assert one_launch(4 << 20) and one_launch(q)                                     # (a workgroup reads its own queries first)
    for x in (k, v):
        assert one_launch(x - out) and one_launch(x + kv)                            # side by side
        assert not any(one_launch(x + at) for at in (0, 16 - out, kv - 16, kv // 2 // 16 * 16))
    # heads stored backwards: the first element is not the lowest
    back = (ctypes.c_int64 * 4)(4 * 100 * 128, -100 * 128, 128, 1)
    backwards = describe(2, 4, 2, 100, 60, o_dtype=o_dtype, o_strides=back)
    assert one_launch(k + kv + 3 * 100 * 128 * size, backwards) and not one_launch(k + kv + 3 * 100 * 128 * size - 16, backwards)


@pytest.mark.gpu
@pytest.mark.parametrize("mode", [_lib.MODE_MXFP4, _lib.MODE_DIAG])
@pytest.mark.parametrize("over", ["k", "v"])
@pytest.mark.parametrize("H, N, causal", [(8, 256, True), (8, 129, False), (32, 160, True)])
def test_output_over_k_or_v(mode, over, H, N, causal):
    desc = describe(1, H, H, N, N, mode=mode, causal=causal)
    named = _lib.ATTN_KERNELS["short4"]
    q, k, v = (t.to(DEV) for t in make_qkv(1, H, H, N, 128, 700 + N))
    work = torch.empty(_lib.lib().mpsa_attn_call_workspace_on(named, desc), dtype=torch.uint8, device=DEV)

    def call(out):
        _lib.check(_lib.lib().mpsa_attn_call_on(named, desc, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), work.data_ptr(), None, _lib.stream_ptr(q.device)))
        torch.cuda.synchronize()
        return out.cpu()
    want = call(torch.empty_like(q))
    assert torch.equal(call(k if over == "k" else v), want)
