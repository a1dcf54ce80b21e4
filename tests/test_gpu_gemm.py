"""HIP block-scaled matmul against the CPU oracle (dequantise + matmul).

Tolerances (float64 oracle; ``mag`` = |dq(A)| @ |dq(B)|^T, the sum of the magnitudes of all partial
products of an output element):

  * E2M1: every product and every partial sum is a small dyadic rational, the matrix cores add them
    exactly and the float32 result is bit-identical to the float64 one -> ``err <= 1e-7 * mag``.
  * E4M3 / E5M2: the scaled matrix instruction adds the products of a step in groups of 8 consecutive K elements and
    cuts every product of a group to 13 bits below the group's largest exponent (tests/mfma8_model.py;
    test_8bit_products_next_to_a_big_one_lose_their_low_bits pins it; measured on Gaussian operands:
    err / mag <= 1.5e-5 at K = 128, falling with K), so small outputs that are differences of large partial
    products cannot meet an elementwise rtol -> ``err <= 1e-3 * |want| + 3e-5 * mag``, i.e. the reference's
    rtol = 1e-3 (ours/block_scaled_matmul.py:440) plus a norm-wise term.
  * bf16 / f16 outputs add one rounding (2^-9 / 2^-11 relative)."""
import pytest
import torch

import oracle as O
from conftest import make_qkv
from ours import _lib
from ours.block_scaled_matmul import block_scaled_matmul, quantize_block_scaled_from_tensor, make_configs, pack_scale_5d
from ours.mxfp import MXFP4Tensor, MXScaleTensor

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TYPES = {"mxfp4": O.FMT_E2M1, "mxfp8": O.FMT_E4M3, "mxfp8e5": O.FMT_E5M2}


def _want_and_mag(ac, asc, bc, bsc, fmt):
    a = O.dequantize_mx(ac, asc, fmt, torch.float64)
    b = O.dequantize_mx(bc, bsc, fmt, torch.float64)
    return a @ b.T, a.abs() @ b.abs().T


def _assert_close(got, want, mag, fmt, out_rounding):
    err = (got.double() - want).abs()
    if fmt == O.FMT_E2M1:
        bound = 1e-7 * mag + out_rounding * want.abs()
    else:
        bound = (1e-3 + out_rounding) * want.abs() + 3e-5 * mag
    bad = err > bound
    assert not bad.any(), f"{bad.sum().item()} elements out of tolerance, worst err/mag {(err / mag.clamp_min(1e-30)).max().item():.3e}"


def _operands(M, N, K, bst, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K, generator=g).bfloat16()
    b = torch.randn(N, K, generator=g).bfloat16()
    return a, b, quantize_block_scaled_from_tensor(a.to(DEV), b.to(DEV), bst)


@pytest.mark.parametrize("bst", ["mxfp4", "mxfp8", "mxfp8e5"])
@pytest.mark.parametrize("shape", [(256, 256, 128), (512, 768, 1024), (256, 1024, 4096), (256, 512, 640), (512, 256, 1536)])
def test_quantize_then_matmul_matches_oracle(bst, shape):
    M, N, K = shape
    a, b, (ac, asc, bc, bsc, cfg) = _operands(M, N, K, bst, seed=M + K)
    fmt = TYPES[bst]
    oa, osa = O.quantize_mx(a, 1.0, fmt)
    ob, osb = O.quantize_mx(b, 1.0, fmt)
    assert torch.equal(ac.cpu(), oa) and torch.equal(bsc.cpu(), osb)
    want, mag = _want_and_mag(oa, osa, ob, osb, fmt)
    got = block_scaled_matmul(ac, asc, bc, bsc, torch.float32, M, N, K, cfg).cpu()
    _assert_close(got, want, mag, fmt, 0.0)
    got16 = block_scaled_matmul(ac, asc, bc, bsc, torch.bfloat16, M, N, K, cfg).cpu()
    _assert_close(got16, want, mag, fmt, 2 ** -8)
    gotf16 = block_scaled_matmul(ac, asc, bc, bsc, torch.float16, M, N, K, cfg).cpu()
    _assert_close(gotf16, want, mag, fmt, 2 ** -10)


def test_random_codes_and_scales_exact_integers():
    """Reference-tutorial style operands (random codes, random scales; ours/block_scaled_matmul.py:423-429):
    with scale exponents >= 0 the result is an integer/4 that float32 holds exactly -> bit-exact check."""
    M, N, K = 256, 256, 256
    a = MXFP4Tensor(size=(M, K), device=DEV).random()
    b = MXFP4Tensor(size=(N, K), device=DEV).random()
    sa = MXScaleTensor(size=(M, K // 32), device=DEV).random(low=1, high=8)
    sb = MXScaleTensor(size=(N, K // 32), device=DEV).random(low=1, high=8)
    got = block_scaled_matmul(a.to_packed_tensor(dim=1), sa.data, b.to_packed_tensor(dim=1), sb.data, torch.float32,
                              M, N, K, make_configs("mxfp4")).cpu()
    want = O.gemm_mx(O.pack_fp4(a.data.cpu()), sa.data.cpu(), O.pack_fp4(b.data.cpu()), sb.data.cpu(), O.FMT_E2M1,
                     acc_dtype=torch.float64)
    assert torch.equal(got.double(), want)
    # the helper classes' own decode gives the same reference (ours/block_scaled_matmul.py:382-392)
    ref = (a.to(torch.float32) * sa.to(torch.float32).repeat_interleave(32, 1)).cpu() @ \
          (b.to(torch.float32) * sb.to(torch.float32).repeat_interleave(32, 1)).cpu().T
    assert torch.equal(got, ref)


def test_identity_like_operand_selects_rows():
    """B = 2^k * one-hot rows: C[m, n] must be the dequantised A[m, k_n] -- catches any k / row permutation."""
    M, N, K = 256, 256, 512
    g = torch.Generator().manual_seed(3)
    a = torch.randn(M, K, generator=g).bfloat16()
    b = torch.zeros(N, K)
    cols = torch.randint(0, K, (N,), generator=g)
    b[torch.arange(N), cols] = 4.0
    ac, asc, bc, bsc, cfg = quantize_block_scaled_from_tensor(a.to(DEV), b.bfloat16().to(DEV), "mxfp8")
    got = block_scaled_matmul(ac, asc, bc, bsc, torch.float32, M, N, K, cfg).cpu()
    adq = O.dequantize_mx(*O.quantize_mx(a, 1.0, O.FMT_E4M3), O.FMT_E4M3)
    assert torch.equal(got, adq[:, cols] * 4.0)


@pytest.mark.parametrize("bst", ["mxfp4", "mxfp8"])
def test_c2_full_size_rows_against_oracle_and_linearity(bst):
    """8192^3: a slab of 256 rows and a slab of 256 columns against the float64 oracle, plus a checksum:
    sum_n C[m, n] must equal dq(A)[m, :] . sum_n dq(B)[n, :]."""
    M = N = K = 8192
    a, b, (ac, asc, bc, bsc, cfg) = _operands(M, N, K, bst, seed=1)
    fmt = TYPES[bst]
    got = block_scaled_matmul(ac, asc, bc, bsc, torch.bfloat16, M, N, K, cfg)
    ac_, asc_, bc_, bsc_ = ac.cpu(), asc.cpu(), bc.cpu(), bsc.cpu()
    rows = slice(4096 + 128, 4096 + 384)
    want_r, mag_r = _want_and_mag(ac_[rows], asc_[rows], bc_, bsc_, fmt)
    _assert_close(got[rows].cpu(), want_r, mag_r, fmt, 2 ** -8)
    cols = slice(7936, 8192)
    want_c, mag_c = _want_and_mag(ac_, asc_, bc_[cols], bsc_[cols], fmt)
    _assert_close(got[:, cols].cpu(), want_c, mag_c, fmt, 2 ** -8)
    got32 = block_scaled_matmul(ac, asc, bc, bsc, torch.float32, M, N, K, cfg)
    adq = O.dequantize_mx(ac_, asc_, fmt, torch.float64)
    bsum = O.dequantize_mx(bc_, bsc_, fmt, torch.float64).sum(dim=0)
    torch.testing.assert_close(got32.double().sum(dim=1).cpu(), adq @ bsum, atol=0.5, rtol=1e-4)


def test_errors():
    ac, asc, bc, bsc, cfg = _operands(256, 256, 128, "mxfp4", 0)[2]
    with pytest.raises(ValueError, match="Unsupported dtype"):
        block_scaled_matmul(ac, asc, bc, bsc, torch.int32, 256, 256, 128, cfg)
    L = _lib.lib()
    args = lambda K, packed=False: (_lib.ptr(ac), _lib.ptr(asc), 4, _lib.ptr(bc), _lib.ptr(bsc), 4, 256, 256, K, _lib.ptr(ac), 2, 256, None)
    assert L.mpsa_gemm_mx(*args(96)) == -3 and b"multiple of 64" in L.mpsa_last_error()
    assert L.mpsa_gemm_mx_packed(_lib.ptr(ac), _lib.ptr(asc), 4, _lib.ptr(bc), _lib.ptr(bsc), 4, 192, 256, 128, _lib.ptr(ac), 2, 256, None) == -3
    assert b"packed scales need" in L.mpsa_last_error()
    assert L.mpsa_gemm_mx(_lib.ptr(ac), _lib.ptr(asc), 9, _lib.ptr(bc), _lib.ptr(bsc), 4, 256, 256, 128, _lib.ptr(ac), 2, 256, None) == -1


def test_scale_5d_layout_and_matmul_with_packed_scales():
    """mpsa_scales_to_5d / _from_5d bit for bit against the reference's reshape/permute, and the matmul fed
    5-D packed scales gives the same bits as with linear ones."""
    from ours.block_scaled_matmul import pack_scale_5d, unpack_scale_5d
    g = torch.Generator().manual_seed(9)
    lin = torch.randint(0, 255, (3, 2, 384, 24), dtype=torch.uint8, generator=g)
    pk = pack_scale_5d(lin.to(DEV))
    assert torch.equal(pk.cpu(), O.scales_to_5d(lin))
    assert torch.equal(unpack_scale_5d(pk).cpu(), lin)
    M, N, K = 256, 512, 512
    a = torch.randn(M, K, generator=g).bfloat16()
    b = torch.randn(N, K, generator=g).bfloat16()
    ac, asc, bc, bsc, cfg = quantize_block_scaled_from_tensor(a.to(DEV), b.to(DEV), "mxfp4")
    c_lin = block_scaled_matmul(ac, asc, bc, bsc, torch.float32, M, N, K, cfg)
    c_pk = block_scaled_matmul(ac, pack_scale_5d(asc), bc, pack_scale_5d(bsc), torch.float32, M, N, K, cfg)
    assert torch.equal(c_lin, c_pk)
    with pytest.raises(RuntimeError, match="multiple of 128"):
        pack_scale_5d(lin[:, :, :100].contiguous().to(DEV))


@pytest.mark.parametrize("bst", ["mxfp4", "mxfp8", "mxfp8e5"])
@pytest.mark.parametrize("M,N,K", [(256, 256, 128), (512, 768, 384), (256, 512, 640), (768, 256, 1024), (512, 512, 2048)])
@pytest.mark.parametrize("kernel", [None, "tile256", "tile128", "split", "general"])
def test_packed_scale_kernel_path_equals_the_row_major_one(kernel, bst, M, N, K):
    """Both operands' scales in the reference's packed form go to the kernel as they are (512-byte chunks fetched
    whole, one 128-bit LDS read per lane and stage): every output bit equals the row-major path's, for every format,
    several tiles per dimension, K that is and is not a multiple of 512 (the row-major path then takes its own two
    variants), odd and even stage counts, and each output dtype, on every kernel."""
    from ours.block_scaled_matmul import pack_scale_5d
    g = torch.Generator().manual_seed(M + N + K)
    a = (torch.randn(M, K, generator=g) * torch.exp2(torch.randint(-6, 6, (M, 1), generator=g).float())).bfloat16()
    b = (torch.randn(N, K, generator=g) * torch.exp2(torch.randint(-6, 6, (1, K), generator=g).float())).bfloat16()
    ac, asc, bc, bsc, cfg = quantize_block_scaled_from_tensor(a.to(DEV), b.to(DEV), bst)
    cfg["KERNEL"] = kernel
    assert asc.unique().numel() > 4                               # scales that differ: a mixed-up byte would show
    a5, b5 = pack_scale_5d(asc), pack_scale_5d(bsc)
    for dt in (torch.float32, torch.bfloat16, torch.float16, torch.float8_e5m2):
        c_lin = block_scaled_matmul(ac, asc, bc, bsc, dt, M, N, K, cfg)
        c_pk = block_scaled_matmul(ac, a5, bc, b5, dt, M, N, K, cfg)
        assert torch.equal(c_lin.view(torch.uint8) if dt == torch.float8_e5m2 else c_lin,
                           c_pk.view(torch.uint8) if dt == torch.float8_e5m2 else c_pk), f"{bst} {M}x{N}x{K} {dt}"
    ac2, a52, bc2, b52, _ = quantize_block_scaled_from_tensor(a.to(DEV), b.to(DEV), bst, packed_scales=True)
    assert torch.equal(a52, a5) and torch.equal(b52, b5) and torch.equal(ac2, ac)


def test_e5m2_output_dtype():
    """The reference's third output dtype (ours/block_scaled_matmul.py:185-190): every byte equals torch's own
    float32 -> float8_e5m2 cast of the kernel's float32 result, overflow to infinity included."""
    M, N, K = 256, 256, 512
    g = torch.Generator().manual_seed(21)
    a = (torch.randn(M, K, generator=g) * 8).bfloat16()
    b = (torch.randn(N, K, generator=g) * 8).bfloat16()
    a[0] *= 64                                                   # one row large enough to overflow E5M2 (57344)
    ac, asc, bc, bsc, cfg = quantize_block_scaled_from_tensor(a.to(DEV), b.to(DEV), "mxfp4")
    c32 = block_scaled_matmul(ac, asc, bc, bsc, torch.float32, M, N, K, cfg)
    c8 = block_scaled_matmul(ac, asc, bc, bsc, torch.float8_e5m2, M, N, K, cfg)
    assert c8.dtype == torch.float8_e5m2
    want = c32.cpu().to(torch.float8_e5m2)
    assert torch.equal(c8.cpu().view(torch.uint8), want.view(torch.uint8))
    assert torch.isinf(want.float()).any() and (want.float().abs() < 1).any()
    # results down in E5M2's subnormal range (below 2^-14) and under its smallest step (2^-16)
    ac, asc, bc, bsc, cfg = quantize_block_scaled_from_tensor((a * 2.0 ** -14).bfloat16().to(DEV), (b * 2.0 ** -12).bfloat16().to(DEV), "mxfp4")
    c32 = block_scaled_matmul(ac, asc, bc, bsc, torch.float32, M, N, K, cfg)
    c8 = block_scaled_matmul(ac, asc, bc, bsc, torch.float8_e5m2, M, N, K, cfg)
    want = c32.cpu().to(torch.float8_e5m2)
    assert torch.equal(c8.cpu().view(torch.uint8), want.view(torch.uint8))
    mag = want.float().abs()
    assert ((mag > 0) & (mag < 2.0 ** -14)).any() and (mag == 0).any() and (mag >= 2.0 ** -14).any()


@pytest.mark.parametrize("bst", ["mxfp4", "mxfp8", "mxfp8e5"])
def test_batched_matmul_scores_with_grouped_heads(bst):
    """block_scaled_batched_matmul on attention-shaped operands (K = head dim 128): every (batch, head) slice
    equals the 2-D entry point's result bit for bit, grouped heads read the right B slice, and the scores match
    the oracle; the reference's packed 5-D scales are accepted."""
    from ours.batched_block_scaled_matmul import block_scaled_batched_matmul
    from ours.block_scaled_matmul import pack_scale_5d
    from ours.quant_mxint8 import quantize_mx
    B, H, Hkv, M, N, K = 2, 4, 2, 512, 256, 128
    q, k, _ = make_qkv(B, H, Hkv, M, K, seed=5)
    k = k[:, :, :N]
    cfg = make_configs(bst)
    fmt = {"mxfp4": O.FMT_E2M1, "mxfp8": O.FMT_E4M3, "mxfp8e5": O.FMT_E5M2}[bst]
    qc, qs = quantize_mx(q.to(DEV), O.q_pre_scale(K), fmt)
    kc, ks = quantize_mx(k.contiguous().to(DEV), 1.0, fmt)
    got = block_scaled_batched_matmul(qc, qs, kc, ks, torch.float32, B, H, M, N, K, cfg)
    assert got.shape == (B, H, M, N)
    for b in range(B):
        for h in range(H):
            one = block_scaled_matmul(qc[b, h], qs[b, h], kc[b, h // 2], ks[b, h // 2], torch.float32, M, N, K, cfg)
            assert torch.equal(got[b, h], one)
    want = O.gemm_mx(qc.cpu(), qs.cpu(), kc.cpu().repeat_interleave(2, dim=1), ks.cpu().repeat_interleave(2, dim=1), fmt)
    mag = O.gemm_mx(qc.cpu(), qs.cpu(), kc.cpu().repeat_interleave(2, dim=1), ks.cpu().repeat_interleave(2, dim=1), fmt,
                    acc_dtype=torch.float64).abs()
    assert ((got.cpu() - want).abs() <= 1e-3 * want.abs() + 3e-5 * mag.float().amax()).all()
    got5 = block_scaled_batched_matmul(qc, pack_scale_5d(qs), kc, pack_scale_5d(ks), torch.float32, B, H, M, N, K, cfg)
    assert torch.equal(got5, got)


def _oracle_operand(values, four_bit, f8):
    """CPU restatement of one packaged operand: the elementwise cast (E2M1 through the oracle's encoder, FP8 through
    torch's own cast -- a library routine, not the reference) and the bytes the kernel is handed."""
    x = values.float()
    if four_bit:
        return O.pack_fp4(O.encode_e2m1(x)), O.FMT_E2M1
    dt = torch.float8_e5m2 if f8 == O.FMT_E5M2 else torch.float8_e4m3fn
    return x.to(dt).view(torch.uint8), f8


@pytest.mark.parametrize("bst", ["mxfp8e5", "mxfp8", "mixed_e5", "mixed", "mxfp4"])
def test_reference_validate_call_sequence(bst):
    """validate_block_scaled_from_tensor(128, 256, 256) of the reference (ours/block_scaled_matmul.py:409-441, :498,
    seed 42 from :501): fp16 operands, float scale factors rand + 1e-8 in the packed 5-D layout,
    initialize_block_scaled_from_tensor with the reference's positional arguments, block_scaled_matmul to fp16.
    "mxfp8e5" is the reference's own 8-bit format; the result is compared with the oracle's product of the same codes
    and E8M0 bytes (the reference's assert_close bound, atol = rtol = 1e-3, is checked for the types with a 4-bit
    operand; the 8-bit x 8-bit bound is the norm-wise one used throughout this file)."""
    from ours.block_scaled_matmul import initialize_block_scaled_from_tensor
    M, N, K = 128, 256, 256
    torch.manual_seed(42)
    a_tensor = torch.randn((M, K), dtype=torch.float16)
    b_tensor = torch.randn((N, K), dtype=torch.float16)
    a_scale_tensor = torch.rand((M // 128, K // 32 // 4, 32, 4, 4)) + 1e-8
    b_scale_tensor = torch.rand((N // 128, K // 32 // 4, 32, 4, 4)) + 1e-8
    a_desc, a_scale, b_desc, b_scale, configs, reference = initialize_block_scaled_from_tensor(
        a_tensor.to(DEV), b_tensor.to(DEV), a_scale_tensor.to(DEV), b_scale_tensor.to(DEV), bst, False)
    assert reference is None
    output = block_scaled_matmul(a_desc, a_scale, b_desc, b_scale, torch.float16, M, N, K, configs)
    assert output.shape == (M, N) and output.dtype == torch.float16
    f8 = O.FMT_E5M2 if bst.endswith("e5") else O.FMT_E4M3
    a_codes, fa = _oracle_operand(a_tensor, bst == "mxfp4", f8)
    b_codes, fb = _oracle_operand(b_tensor, bst in ("mxfp4", "mixed", "mixed_e5"), f8)
    assert torch.equal(a_desc.cpu().view(torch.uint8), a_codes) and torch.equal(b_desc.cpu().view(torch.uint8), b_codes)
    sa, sb = O.encode_e8m0(a_scale_tensor), O.encode_e8m0(b_scale_tensor)
    assert torch.equal(a_scale.cpu(), sa) and torch.equal(b_scale.cpu(), sb)
    sa_lin, sb_lin = O.scales_from_5d(sa), O.scales_from_5d(sb)
    want = O.gemm_mx(a_codes, sa_lin, b_codes, sb_lin, fa, fb, acc_dtype=torch.float64)
    mag = O.dequantize_mx(a_codes, sa_lin, fa, torch.float64).abs() @ O.dequantize_mx(b_codes, sb_lin, fb, torch.float64).abs().T
    err = (output.cpu().double() - want).abs()
    if fa == O.FMT_E2M1 or fb == O.FMT_E2M1:
        # the reference's own bound holds where a 4-bit operand keeps the products short
        assert (err <= 1e-3 + 1e-3 * want.abs()).all(), err.max()
    assert (err <= (1e-3 + 2 ** -10) * want.abs() + 3e-5 * mag).all(), (err / mag).max()
    with pytest.raises(NotImplementedError, match="nvfp4"):
        initialize_block_scaled_from_tensor(a_tensor.to(DEV), b_tensor.to(DEV), a_scale_tensor.to(DEV), b_scale_tensor.to(DEV), "nvfp4")
    # compute_reference=True (ours/block_scaled_matmul.py:376-392, :404): the same packaged operands plus the triple
    # (fake-quant product, dq(A), dq(B)) in float32, made on the device from the packaged bytes.  The device reference
    # is itself pinned here: against the oracle's dequantization (exactly) and its float64 product.
    a2, sa2, b2, sb2, cfg2, reference = initialize_block_scaled_from_tensor(
        a_tensor.to(DEV), b_tensor.to(DEV), a_scale_tensor.to(DEV), b_scale_tensor.to(DEV), bst, compute_reference=True)
    assert torch.equal(a2, a_desc) and torch.equal(b2, b_desc) and torch.equal(sa2, a_scale) and torch.equal(sb2, b_scale) and cfg2 == configs
    ref, a_dq, b_dq = reference
    assert ref.dtype == torch.float32 and ref.shape == (M, N) and a_dq.shape == (M, K) and b_dq.shape == (N, K)
    assert torch.equal(a_dq.cpu(), O.dequantize_mx(a_codes, sa_lin, fa, torch.float32))
    assert torch.equal(b_dq.cpu(), O.dequantize_mx(b_codes, sb_lin, fb, torch.float32))
    assert ((ref.cpu().double() - want).abs() <= 1e-5 * mag).all()          # float32 accumulation of 256 products
    # the reference's own comparison (ours/block_scaled_matmul.py:440)
    if fa == O.FMT_E2M1 or fb == O.FMT_E2M1:
        torch.testing.assert_close(ref, output.to(torch.float32), atol=1e-3, rtol=1e-3)


@pytest.mark.parametrize("bst", ["mxfp4", "mixed", "mxfp8", "mixed_e5", "mxfp8e5"])
def test_validate_block_scaled_from_tensor_runs_the_reference_self_check(bst):
    """validate_block_scaled_from_tensor at the reference's own shape and seed (ours/block_scaled_matmul.py:498-501):
    packaging with compute_reference=True, the kernel's fp16 product, assert_close(atol = rtol = 1e-3) -- and the
    fake-quant reference it compares with is checked here against the oracle's float64 product of the same operands,
    which are regenerated on the CPU from the same seed."""
    from ours.block_scaled_matmul import validate_block_scaled_from_tensor
    M, N, K = 128, 256, 256
    torch.manual_seed(42)
    reference, output = validate_block_scaled_from_tensor(M, N, K, bst, device=DEV)
    assert reference.shape == (M, N) and output.dtype == torch.float16
    # the self-check drew its operands from the device generator; draw them again and rebuild them for the oracle
    torch.manual_seed(42)
    a_tensor = torch.randn((M, K), dtype=torch.float16, device=DEV).cpu()
    b_tensor = torch.randn((N, K), dtype=torch.float16, device=DEV).cpu()
    sa = (torch.rand((M // 128, K // 32 // 4, 32, 4, 4), device=DEV) + 1e-8).cpu()
    sb = (torch.rand((N // 128, K // 32 // 4, 32, 4, 4), device=DEV) + 1e-8).cpu()
    f8 = O.FMT_E5M2 if bst.endswith("e5") else O.FMT_E4M3
    a_codes, fa = _oracle_operand(a_tensor, bst == "mxfp4", f8)
    b_codes, fb = _oracle_operand(b_tensor, bst in ("mxfp4", "mixed", "mixed_e5"), f8)
    sa_lin, sb_lin = O.scales_from_5d(O.encode_e8m0(sa)), O.scales_from_5d(O.encode_e8m0(sb))
    want = O.gemm_mx(a_codes, sa_lin, b_codes, sb_lin, fa, fb, acc_dtype=torch.float64)
    mag = O.dequantize_mx(a_codes, sa_lin, fa, torch.float64).abs() @ O.dequantize_mx(b_codes, sb_lin, fb, torch.float64).abs().T
    assert ((reference.cpu().double() - want).abs() <= 1e-5 * mag).all()


def test_packaging_refuses_values_beyond_e4m3_and_casts_them_in_e5m2():
    """The reference's 8-bit cast is E5M2 (ours/block_scaled_matmul.py:334-336: finite up to 57344); this package's
    "mxfp8" / "mixed" cast to E4M3, where torch's cast makes NaN of magnitudes above 464: such input is refused with a
    pointer to the E5M2 types, under which the bytes are torch's E5M2 cast."""
    from ours.block_scaled_matmul import initialize_block_scaled_from_tensor
    M, N, K = 128, 128, 128
    g = torch.Generator().manual_seed(5)
    a = torch.randn(M, K, generator=g).to(torch.float16)
    b = torch.randn(N, K, generator=g).to(torch.float16)
    a[3, 7], a[100, 5], b[9, 9] = 1000.0, -30000.0, 449.0
    sa = torch.rand((1, 1, 32, 4, 4), generator=g) + 1e-8
    sb = torch.rand((1, 1, 32, 4, 4), generator=g) + 1e-8
    for bst in ("mxfp8", "mixed"):
        with pytest.raises(ValueError, match="mxfp8e5"):
            initialize_block_scaled_from_tensor(a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV), bst)
    a_desc, a_scale, b_desc, b_scale, configs, reference = initialize_block_scaled_from_tensor(
        a.to(DEV), b.to(DEV), sa.to(DEV), sb.to(DEV), "mxfp8e5", compute_reference=True)
    assert torch.equal(a_desc.cpu(), a.float().to(torch.float8_e5m2).view(torch.uint8))
    assert torch.equal(b_desc.cpu(), b.float().to(torch.float8_e5m2).view(torch.uint8))
    out = block_scaled_matmul(a_desc, a_scale, b_desc, b_scale, torch.float32, M, N, K, configs)
    assert torch.isfinite(out).all() and torch.isfinite(reference[0]).all()
    mag = reference[1].abs() @ reference[2].abs().T
    assert ((out - reference[0]).abs() <= 1e-3 * reference[0].abs() + 3e-5 * mag).all()
    # exactly +-448 still fits E4M3
    a2 = a.clamp(-448, 448)
    b2 = b.clamp(-448, 448)
    a_desc, *_ = initialize_block_scaled_from_tensor(a2.to(DEV), b2.to(DEV), sa.to(DEV), sb.to(DEV), "mxfp8")
    assert torch.equal(a_desc.cpu(), a2.float().to(torch.float8_e4m3fn).view(torch.uint8))


@pytest.mark.parametrize("fa,fb", [(O.FMT_E2M1, O.FMT_E2M1), (O.FMT_E4M3, O.FMT_E4M3), (O.FMT_E5M2, O.FMT_E5M2),
                                   (O.FMT_E4M3, O.FMT_E2M1), (O.FMT_E5M2, O.FMT_E2M1), (O.FMT_E2M1, O.FMT_E4M3),
                                   (O.FMT_E4M3, O.FMT_E5M2)])
@pytest.mark.parametrize("M,N,K", [(128, 256, 256), (100, 200, 192), (1, 1, 64), (384, 128, 640), (257, 129, 128)])
def test_edge_tiles_and_mixed_formats_against_oracle(fa, fb, M, N, K):
    """Shapes off the 256 x 256 tile (the reference's kernel masks its edge tiles, ours/block_scaled_matmul.py:154-267)
    and operands of different element formats (ELEM_PER_BYTE_A != ELEM_PER_BYTE_B, :318-324), through the C ABI."""
    from ours.quant_mxint8 import quantize_mx
    g = torch.Generator().manual_seed(M * 7 + N * 3 + K + fa + 10 * fb)
    a = (torch.randn(M, K, generator=g) * torch.exp2(torch.randint(-4, 4, (M, 1), generator=g).float())).bfloat16()
    b = (torch.randn(N, K, generator=g) * torch.exp2(torch.randint(-4, 4, (1, K), generator=g).float())).bfloat16()
    ac, asc = (t[0, 0] for t in quantize_mx(a[None, None].to(DEV), 1.0, fa))
    bc, bsc = (t[0, 0] for t in quantize_mx(b[None, None].to(DEV), 1.0, fb))
    out = torch.full((M, N + 3), 7.0, dtype=torch.float32, device=DEV)          # ldc > N: the padding must stay
    _lib.check(_lib.lib().mpsa_gemm_mx(_lib.ptr(ac), _lib.ptr(asc), fa, _lib.ptr(bc), _lib.ptr(bsc), fb, M, N, K,
                                       _lib.ptr(out), _lib.F32, N + 3, _lib.stream_ptr()))
    assert (out[:, N:] == 7.0).all()
    want = O.gemm_mx(ac.cpu(), asc.cpu(), bc.cpu(), bsc.cpu(), fa, fb, acc_dtype=torch.float64)
    mag = O.dequantize_mx(ac.cpu(), asc.cpu(), fa, torch.float64).abs() @ O.dequantize_mx(bc.cpu(), bsc.cpu(), fb, torch.float64).abs().T
    err = (out[:, :N].cpu().double() - want).abs()
    # E2M1 x E2M1 products and their float32 sums are exact.  With an 8-bit operand the matrix core aligns the 64
    # products of a step to the largest exponent and keeps about 16 bits below it; these operands carry a 2^8 spread
    # of magnitudes inside every MX block (the column gains of b), so more of the small products' bits fall off than
    # with the Gaussian operands of the other tests: measured err / sum|a||b| up to 5.5e-5 (E5M2 x E5M2).
    exact = fa == O.FMT_E2M1 and fb == O.FMT_E2M1
    bound = 1e-7 * mag if exact else 1e-3 * want.abs() + 1e-4 * mag
    assert (err <= bound).all(), f"worst err/mag {(err / mag.clamp_min(1e-30)).max().item():.3e}"


@pytest.mark.parametrize("K", [1024, 384])         # 16 scale bytes per row at a time (K % 512 == 0), and 4 per stage
@pytest.mark.parametrize("bst", ["mxfp4", "mxfp8", "mixed", "mixed_e5"])
def test_general_kernel_equals_the_staged_kernel_on_its_shapes(bst, K):
    """A 512 x 256 product on the LDS-staged 256 x 256 kernel, and on the general kernel whole and as two row slabs of 384 and
    128 rows: same K order, same matrix instruction, same bits -- for equal formats and for the reference's "mixed" type
    (8-bit A x 4-bit B, ours/block_scaled_matmul.py:318-324), with row-major and with packed scales.  So do ragged shapes on
    the staged kernel's edge variants, where it has them.  The other two kernels split K between waves: as close as float32
    additions in another order, and equal where those are exact (4-bit products)."""
    M, N = 512, 256
    a, b, (ac, asc, bc, bsc, cfg) = _operands(M, N, K, bst, seed=77)
    on = lambda kernel, dt=torch.float32, rows=slice(0, M), packed=False: block_scaled_matmul(
        ac[rows].contiguous(), (pack_scale_5d(asc) if packed else asc[rows].contiguous()), bc, pack_scale_5d(bsc) if packed else bsc, dt,
        len(range(*rows.indices(M))), N, K, dict(cfg, KERNEL=kernel))
    whole = on("tile256")
    assert torch.equal(whole, on("general"))
    assert torch.equal(whole, torch.cat([on("general", rows=slice(0, 384)), on("general", rows=slice(384, M))]))
    for kernel in ("tile256", "general"):
        assert torch.equal(whole, on(kernel, packed=True))
    for dt in (torch.bfloat16, torch.float16):
        assert torch.equal(on("tile256", dt), whole.to(dt))
    if bst != "mxfp4" or K % 256 == 0:
        assert torch.equal(whole[:300], on("tile256", rows=slice(0, 300)))
    for kernel in ("tile128", "split", None):
        got = on(kernel)
        assert torch.equal(whole, got) if bst == "mxfp4" else (whole - got).abs().max() <= 1e-5 * whole.abs().max()


@pytest.mark.parametrize("bst", ["mixed", "mixed_e5"])
@pytest.mark.parametrize("M,N,K", [(256, 256, 128), (512, 768, 1024), (256, 512, 640), (768, 256, 2048)])
@pytest.mark.parametrize("kernel", ["tile256", None])
def test_mixed_formats_on_the_staged_kernel_against_oracle(kernel, bst, M, N, K):
    """8-bit A x 4-bit B on whole 256 x 256 tiles (the LDS-staged kernel's mixed variant) against the float64 oracle."""
    f8 = O.FMT_E5M2 if bst.endswith("e5") else O.FMT_E4M3
    a, b, (ac, asc, bc, bsc, cfg) = _operands(M, N, K, bst, seed=M + N + K)
    oa, osa = O.quantize_mx(a, 1.0, f8)
    ob, osb = O.quantize_mx(b, 1.0, O.FMT_E2M1)
    assert torch.equal(ac.cpu(), oa) and torch.equal(bc.cpu(), ob) and torch.equal(asc.cpu(), osa) and torch.equal(bsc.cpu(), osb)
    want = O.gemm_mx(oa, osa, ob, osb, f8, O.FMT_E2M1, acc_dtype=torch.float64)
    mag = O.dequantize_mx(oa, osa, f8, torch.float64).abs() @ O.dequantize_mx(ob, osb, O.FMT_E2M1, torch.float64).abs().T
    got = block_scaled_matmul(ac, asc, bc, bsc, torch.float32, M, N, K, dict(cfg, KERNEL=kernel)).cpu()
    err = (got.double() - want).abs()
    assert (err <= 1e-3 * want.abs() + 3e-5 * mag).all(), f"worst err/mag {(err / mag.clamp_min(1e-30)).max().item():.3e}"


def test_batched_mixed_formats_with_grouped_heads():
    """The batched entry point with 8-bit A against 4-bit B (the reference's "mixed" Q.K^T) and grouped heads."""
    from ours.batched_block_scaled_matmul import block_scaled_batched_matmul
    from ours.quant_mxint8 import quantize_mx
    B, H, Hkv, M, N, K = 2, 4, 2, 128, 384, 128
    q, k, _ = make_qkv(B, H, Hkv, 384, K, seed=15)
    q = q[:, :, :M].contiguous()
    qc, qs = quantize_mx(q.to(DEV), O.q_pre_scale(K), O.FMT_E4M3)
    kc, ks = quantize_mx(k.to(DEV), 1.0, O.FMT_E2M1)
    got = block_scaled_batched_matmul(qc, qs, kc, ks, torch.float32, B, H, M, N, K, make_configs("mixed"))
    want = O.gemm_mx(qc.cpu(), qs.cpu(), kc.cpu().repeat_interleave(2, dim=1), ks.cpu().repeat_interleave(2, dim=1),
                     O.FMT_E4M3, O.FMT_E2M1, acc_dtype=torch.float64)
    mag = O.dequantize_mx(qc.cpu(), qs.cpu(), O.FMT_E4M3, torch.float64).abs() @ \
        O.dequantize_mx(kc.cpu().repeat_interleave(2, dim=1), ks.cpu().repeat_interleave(2, dim=1), O.FMT_E2M1, torch.float64).abs().transpose(-1, -2)
    assert ((got.cpu().double() - want).abs() <= 1e-3 * want.abs() + 3e-5 * mag).all()


@pytest.mark.parametrize("M,N,kernel", [(128, 256, "general"), (256, 256, "tile256"), (128, 256, "tile256"), (128, 256, "tile128"), (128, 256, "split"),
                                        (128, 256, "split4x4"), (256, 256, "auto")])
@pytest.mark.parametrize("fmt", [O.FMT_E4M3, O.FMT_E5M2])
def test_8bit_products_next_to_a_big_one_lose_their_low_bits(fmt, M, N, kernel):
    """What the matrix cores do with an 8-bit dot product whose terms differ by more than 2^13 (tests/mfma8_model.py),
    pinned through the C ABI on operands with two nonzero products per output: A is all ones, row n of B holds one big
    code and one small code.  A small product in the big one's group of 8 consecutive K elements arrives cut to a multiple
    of 2^(E - 13) (toward zero), one in any other group arrives whole.  The float32 product of the dequantized operands --
    the reference's arithmetic as oracle/ restates it -- keeps every bit here; this is the one place where the hardware's
    result and the oracle's differ by more than summation order."""
    from mfma8_model import product_8bit
    K = 128
    one, big = (0x38, 0x7E) if fmt == O.FMT_E4M3 else (0x3C, 0x78)           # 1.0; 448 (E4M3), 32768 (E5M2)
    # E4M3: 2^-6, 0.03515625, 0.234375, 0.25, -0.03515625, 0.5 (cut at 2^-5); E5M2: 1.25 * 2^-7, 5, 7, 8, 10, -5 (cut at 4)
    smalls = [0x08, 0x11, 0x27, 0x28, 0x91, 0x30] if fmt == O.FMT_E4M3 else [0x21, 0x45, 0x47, 0x48, 0x49, 0xC5]
    probes = [(kb, ks, c) for kb in (0, 5, 77) for ks in (kb + 1, kb - kb % 8 + 7 if kb % 8 != 7 else kb - 1, (kb + 8) % K, (kb + 64) % K) for c in smalls]
    assert len(probes) <= N
    a = torch.full((M, K), one, dtype=torch.uint8)
    b = torch.zeros((N, K), dtype=torch.uint8)
    for n, (kb, ks, c) in enumerate(probes):
        b[n, kb], b[n, ks] = big, c
    sc_a = torch.full((M, K // 32), 127, dtype=torch.uint8)
    sc_b = torch.full((N, K // 32), 127, dtype=torch.uint8)
    out = torch.empty((M, N), dtype=torch.float32, device=DEV)
    a_d, sa_d, b_d, sb_d = a.to(DEV), sc_a.to(DEV), b.to(DEV), sc_b.to(DEV)
    _lib.check(_lib.lib().mpsa_gemm_mx_on(_lib.GEMM_KERNELS[kernel], _lib.ptr(a_d), _lib.ptr(sa_d), fmt, _lib.ptr(b_d), _lib.ptr(sb_d), fmt, 0,
                                          1, 1, 1, M, N, K, _lib.ptr(out), _lib.F32, N, _lib.stream_ptr()))
    got = out.cpu()
    ad, bd = O.dequantize_mx(a, sc_a, fmt), O.dequantize_mx(b, sc_b, fmt)
    model = product_8bit(ad, bd)
    exact = (ad.double() @ bd.double().T).float()
    assert torch.equal(got, model)
    cut = kept = 0
    for n, (kb, ks, c) in enumerate(probes):
        same_group = kb // 8 == ks // 8
        if not same_group:
            assert got[0, n] == exact[0, n]
            kept += 1
        elif got[0, n] != exact[0, n]:
            assert abs(got[0, n] - float(bd[n, kb])) < abs(exact[0, n] - float(bd[n, kb]))      # cut toward zero
            cut += 1
    assert kept == len(probes) // 2 and cut >= len(probes) // 4
    if fmt == O.FMT_E4M3:                   # the literal cases quoted in tests/mfma8_model.py
        assert got[0, probes.index((0, 1, 0x08))] == 448.0 and got[0, probes.index((0, 8, 0x08))] == 448.015625
        assert got[0, probes.index((0, 1, 0x11))] == 448.03125 and got[0, probes.index((0, 1, 0x28))] == 448.25


@pytest.mark.parametrize("M,N,kernel", [(128, 256, "general"), (256, 256, "tile256"), (128, 256, "tile256"), (128, 256, "tile128"), (128, 256, "split"),
                                        (128, 256, "split4x4"), (256, 256, "auto")])
@pytest.mark.parametrize("fmt", [O.FMT_E4M3, O.FMT_E5M2])
def test_8bit_against_4bit_products_are_cut_the_same_way(fmt, M, N, kernel):
    """The same rule for the reference's "mixed" pair (8-bit A, E2M1 B): the probes sit in rows of A, B is all ones."""
    from mfma8_model import product_8bit
    K = 128
    big = 0x7E if fmt == O.FMT_E4M3 else 0x78
    smalls = [0x08, 0x11, 0x27, 0x28, 0x91, 0x30] if fmt == O.FMT_E4M3 else [0x21, 0x45, 0x47, 0x48, 0x49, 0xC5]
    probes = [(kb, ks, c) for kb in (0, 5, 77) for ks in (kb + 1, kb - kb % 8 + 7, (kb + 8) % K, (kb + 64) % K) for c in smalls]
    assert len(probes) <= M
    a = torch.zeros((M, K), dtype=torch.uint8)
    for m, (kb, ks, c) in enumerate(probes):
        a[m, kb], a[m, ks] = big, c
    b = torch.full((N, K // 2), 0x22, dtype=torch.uint8)                       # E2M1 1.0 in both nibbles
    sc_a = torch.full((M, K // 32), 127, dtype=torch.uint8)
    sc_b = torch.full((N, K // 32), 127, dtype=torch.uint8)
    out = torch.empty((M, N), dtype=torch.float32, device=DEV)
    a_d, sa_d, b_d, sb_d = a.to(DEV), sc_a.to(DEV), b.to(DEV), sc_b.to(DEV)
    _lib.check(_lib.lib().mpsa_gemm_mx_on(_lib.GEMM_KERNELS[kernel], _lib.ptr(a_d), _lib.ptr(sa_d), fmt, _lib.ptr(b_d), _lib.ptr(sb_d), O.FMT_E2M1, 0,
                                          1, 1, 1, M, N, K, _lib.ptr(out), _lib.F32, N, _lib.stream_ptr()))
    ad, bd = O.dequantize_mx(a, sc_a, fmt), O.dequantize_mx(b, sc_b, O.FMT_E2M1)
    assert torch.equal(out.cpu(), product_8bit(ad, bd))
    exact = (ad.double() @ bd.double().T).float()
    assert (out.cpu() != exact).any()



# a row count per tile height of the kernels behind mpsa_gemm_mx (16-row blocks with K split between the waves, 128 x 128,
# 256 x 256 with ragged edges), its remainders, and K with and without half a unit of 256: on the kernel that the shape takes and
# on every other one that takes it
@pytest.mark.parametrize("fmt_a,fmt_b", [(4, 4), (0, 4), (0, 0), (4, 1), (1, 4)])
@pytest.mark.parametrize("M,N,K", [(1, 16, 128), (16, 4095, 384), (17, 1025, 2176), (33, 4100, 1152), (65, 130, 4096), (129, 4096, 256),
                                   (300, 1000, 1408), (700, 2500, 1152), (900, 3200, 640), (1000, 14336, 256), (2303, 2817, 512),
                                   (2304, 2816, 128), (255, 257, 512), (384, 640, 1024)])
def test_every_kernel_at_its_edges(fmt_a, fmt_b, M, N, K):
    g = torch.Generator().manual_seed(M * 7 + N)
    a = torch.randn(M, K, generator=g).to(torch.bfloat16)
    b = torch.randn(N, K, generator=g).to(torch.bfloat16)
    (ac, sa), (bc, sb) = O.quantize_mx(a, 1.0, fmt_a), O.quantize_mx(b, 1.0, fmt_b)
    ad, sad, bd, sbd = (t.to(DEV) for t in (ac, sa, bc, sb))
    da = O.dequantize_mx(ac, sa, fmt_a, torch.float32).to(DEV).double()
    db = O.dequantize_mx(bc, sb, fmt_b, torch.float32).to(DEV).double()
    want, size = da @ db.t(), da.abs() @ db.abs().t()
    L = _lib.lib()
    kernels = [n for n, i in _lib.GEMM_KERNELS.items() if L.mpsa_gemm_kernel(i, fmt_a, fmt_b, 1, 1, M, N, K) > 0]
    staged = (fmt_a == fmt_b or fmt_b == 4) and not (fmt_a == fmt_b == 4 and K % 256 and (M % 256 or N % 256))
    assert ("tile256" in kernels) == staged and len(kernels) == len(_lib.GEMM_KERNELS) - (not staged)
    for packed in [False] + [True] * (M % 128 == 0 and N % 128 == 0):
        xa, xb = (pack_scale_5d(sad), pack_scale_5d(sbd)) if packed else (sad, sbd)
        for kernel in kernels:
            out = torch.full((M + 1, N), 7.0, device=DEV)        # one row more than the product has
            _lib.check(L.mpsa_gemm_mx_on(_lib.GEMM_KERNELS[kernel], _lib.ptr(ad), _lib.ptr(xa), fmt_a, _lib.ptr(bd), _lib.ptr(xb), fmt_b, packed,
                                         1, 1, 1, M, N, K, _lib.ptr(out), _lib.F32, N, _lib.stream_ptr()))
            err = (out[:M].double() - want).abs()
            assert bool((err <= (1e-7 if fmt_a == fmt_b == 4 else 1e-4) * size).all()), kernel
            assert bool((out[M] == 7.0).all()), kernel


def test_a_kernel_that_does_not_take_the_shape_is_refused():
    a, b, (ac, asc, bc, bsc, cfg) = _operands(256, 256, 192, "mxfp4", seed=1)
    for kernel in ("split", "split2x4", "tile128", "tile256"):
        with pytest.raises(_lib.MpsaError, match="K % 128"):
            block_scaled_matmul(ac, asc, bc, bsc, torch.float32, 256, 256, 192, dict(cfg, KERNEL=kernel))
    with pytest.raises(ValueError, match="unknown matmul kernel"):
        block_scaled_matmul(ac, asc, bc, bsc, torch.float32, 256, 256, 192, dict(cfg, KERNEL="fastest"))


@pytest.mark.parametrize("bst", ["mxfp4", "mxfp8", "mixed"])
def test_rows_do_not_depend_on_how_many_there_are(bst):
    """On the kernels that add up K in one order -- general, 256 x 256 -- by name, and for 4-bit products, whose sums are exact
    here, with the kernel left open."""
    M, N, K = 600, 640, 1024
    a, b, (ac, asc, bc, bsc, cfg) = _operands(M, N, K, bst, seed=5)
    on = lambda kernel, m: block_scaled_matmul(ac[:m].contiguous(), asc[:m].contiguous(), bc, bsc, torch.float32, m, N, K, dict(cfg, KERNEL=kernel))
    want = on("general", M)
    for kernel in ["general", "tile256"] + [None] * (bst == "mxfp4"):
        for m in (1, 16, 100, 256, 512, M):
            assert torch.equal(on(kernel, m), want[:m]), (kernel, m)


@pytest.mark.parametrize("kernel", ["general", "tile256", "tile128", "split", None])
def test_an_operand_of_more_than_4_gib(kernel):
    """Row offsets beyond 32 bits: the last rows of a 4.6 GB operand, and rows on either side of the 2^32nd byte."""
    M, N, K = 280000, 16, 16384
    g = torch.Generator(device=DEV).manual_seed(3)
    a = torch.randint(0, 0x77, (M, K), dtype=torch.uint8, device=DEV, generator=g)              # finite E4M3 codes
    b = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device=DEV, generator=g)
    sa = torch.randint(120, 124, (M, K // 32), dtype=torch.uint8, device=DEV, generator=g)
    sb = torch.randint(120, 124, (N, K // 32), dtype=torch.uint8, device=DEV, generator=g)
    out = block_scaled_matmul(a, sa, b, sb, torch.float32, M, N, K, dict(make_configs("mixed"), KERNEL=kernel))
    for rows in (slice(0, 4), slice(2 ** 32 // K - 4, 2 ** 32 // K + 4), slice(M - 4, M)):
        ac, bc = a[rows].cpu(), b.cpu()
        want = O.gemm_mx(ac, sa[rows].cpu(), bc, sb.cpu(), O.FMT_E4M3, O.FMT_E2M1, acc_dtype=torch.float64)
        mag = O.dequantize_mx(ac, sa[rows].cpu(), O.FMT_E4M3, torch.float64).abs() @ O.dequantize_mx(bc, sb.cpu(), O.FMT_E2M1, torch.float64).abs().T
        assert ((out[rows].cpu().double() - want).abs() <= 1e-3 * want.abs() + 1e-4 * mag).all(), (kernel, rows)


@pytest.mark.parametrize("bst", ["mxfp4", "mxfp8", "mixed"])
@pytest.mark.parametrize("packed", [False, True])
def test_batched_slices_equal_the_2d_product_on_every_kernel(bst, packed):
    from ours.batched_block_scaled_matmul import block_scaled_batched_matmul
    B, H, Hkv, M, N, K = 2, 4, 2, 384, 256, 640
    g = torch.Generator().manual_seed(8)
    a = torch.randn(B * H * M, K, generator=g).bfloat16().to(DEV)
    b = torch.randn(B * Hkv * N, K, generator=g).bfloat16().to(DEV)
    ac, sa, bc, sb, cfg = quantize_block_scaled_from_tensor(a, b, bst)
    ac, sa, bc, sb = ac.view(B, H, M, -1), sa.view(B, H, M, -1), bc.view(B, Hkv, N, -1), sb.view(B, Hkv, N, -1)
    if packed:
        sa, sb = pack_scale_5d(sa), pack_scale_5d(sb)
    fmt_a, fmt_b = (4 if cfg["ELEM_PER_BYTE_A"] == 2 else 0), (4 if cfg["ELEM_PER_BYTE_B"] == 2 else 0)
    names = [n for n, i in _lib.GEMM_KERNELS.items() if n not in ("auto", "split") and _lib.lib().mpsa_gemm_kernel(i, fmt_a, fmt_b, B, H, M, N, K) > 0]
    assert len(names) >= 8
    for kernel in names:
        on = dict(cfg, KERNEL=kernel)
        got = block_scaled_batched_matmul(ac, sa, bc, sb, torch.float32, B, H, M, N, K, on)
        for i in range(B):
            for h in range(H):
                one = block_scaled_matmul(ac[i, h], sa[i, h], bc[i, h // 2], sb[i, h // 2], torch.float32, M, N, K, on)
                assert torch.equal(got[i, h], one), (kernel, i, h)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kernel", ["general", "tile128", "tile256"])
@pytest.mark.parametrize("M,N,ldc", [(1, 8, 8), (31, 250, 256), (129, 129, 136), (257, 263, 264), (300, 520, 520), (256, 512, 520),
                                     (130, 77, 77), (257, 300, 303), (256, 256, 257)])
def test_16bit_results_are_the_float32_ones_rounded_once(kernel, M, N, ldc, dtype):
    """Rows in whole 16-byte pieces (row pitch a multiple of 8) and not, the last piece of a row cut, and nothing written
    past a row's end: the same bits as float32 results rounded once, and the gap between rows as it was."""
    K, L = 256, _lib.lib()
    g = torch.Generator().manual_seed(M + N)
    a = torch.randint(0, 256, (M, K // 2), dtype=torch.uint8, generator=g).to(DEV)
    b = torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, generator=g).to(DEV)
    sa = torch.randint(118, 130, (M, K // 32), dtype=torch.uint8, generator=g).to(DEV)
    sb = torch.randint(118, 130, (N, K // 32), dtype=torch.uint8, generator=g).to(DEV)

    def product(dt):
        c = torch.full((M + 1, ldc), 7.0, dtype=dt, device=DEV)
        _lib.check(L.mpsa_gemm_mx_on(_lib.GEMM_KERNELS[kernel], _lib.ptr(a), _lib.ptr(sa), 4, _lib.ptr(b), _lib.ptr(sb), 4, 0, 1, 1, 1, M, N, K,
                                     _lib.ptr(c), _lib.dtype_id(dt), ldc, _lib.stream_ptr(a.device)))
        return c

    got, want = product(dtype), product(torch.float32).to(dtype)
    assert torch.equal(got, want)


@pytest.mark.parametrize("fmt_a,fmt_b", [(4, 4), (0, 0), (1, 1), (0, 4), (1, 4)])
@pytest.mark.parametrize("batch,heads,heads_b,M,N", [(1, 1, 1, 128, 128), (1, 2, 1, 100, 130), (2, 4, 2, 1, 7), (1, 1, 1, 300, 4096), (2, 8, 4, 1024, 1024),
                                                     (1, 4, 4, 2000, 2040), (1, 8, 2, 1408, 1536), (1, 16, 16, 1030, 1025)])
def test_products_with_one_stage_of_k(batch, heads, heads_b, M, N, fmt_a, fmt_b):
    """K == 128 has a kernel of its own, which walks several tiles a workgroup where there are many: the general kernel's bits,
    whole and cut tiles, grouped heads, both scale layouts, and row pitches that it leaves to the general kernel."""
    K, L = 128, _lib.lib()
    packed_too = M % 128 == 0 and N % 128 == 0            # packed scales are whole chunks of 128 rows
    g = torch.Generator().manual_seed(M * N + fmt_a)

    def codes(rows, h, fmt):
        # 8-bit codes without infinities and NaN: exponent field below the top one
        c = torch.randint(0, 256, (batch, h, rows, K // 2 if fmt == 4 else K), generator=g, dtype=torch.uint8)
        return (c if fmt == 4 else c & 0xBF).to(DEV)

    a, b = codes(M, heads, fmt_a), codes(N, heads_b, fmt_b)
    sa, sb = (torch.randint(118, 130, (batch, h, rows, K // 32), generator=g, dtype=torch.uint8).to(DEV) for h, rows in ((heads, M), (heads_b, N)))
    for packed, dtype, ldc in [(p, d, l) for p in range(1 + packed_too) for d, l in ((torch.bfloat16, (N + 7) // 8 * 8), (torch.float16, N))]:
        got, want = (torch.full((batch, heads, M, ldc), 3.0, dtype=dtype, device=DEV) for _ in range(2))
        for out, kernel in ((got, "auto"), (want, "general")):
            _lib.check(L.mpsa_gemm_mx_on(_lib.GEMM_KERNELS[kernel], _lib.ptr(a), _lib.ptr(sa), fmt_a, _lib.ptr(b), _lib.ptr(sb), fmt_b, packed, batch, heads, heads_b, M, N, K,
                                         _lib.ptr(out), _lib.dtype_id(dtype), ldc, _lib.stream_ptr(a.device)))
        assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("fmt_a,fmt_b", [(4, 4), (0, 4), (1, 1), (0, 1)])
@pytest.mark.parametrize("batch,M,N", [(1, 16, 4096), (1, 256, 1024), (1, 257, 1024), (4, 128, 512), (5, 128, 512), (1, 500, 1000), (1, 512, 1032)])
def test_products_with_one_stage_of_k_run_on_the_kernel_that_is_said(batch, M, N, fmt_a, fmt_b):
    """K == 128 with up to 1024 blocks of 16 x 16 results, with more, and with more than 2048: the bits of the kernel that
    mpsa_gemm_kernel names, or from 1024 blocks on of the general one where 16-bit rows start on 16 bytes."""
    K, L = 128, _lib.lib()
    g = torch.Generator().manual_seed(M * N + fmt_a)
    codes = lambda rows, fmt: (torch.randint(0, 256, (batch, rows, K // 2 if fmt == 4 else K), generator=g, dtype=torch.uint8) & (0xFF if fmt == 4 else 0xBF)).to(DEV)
    a, b = codes(M, fmt_a), codes(N, fmt_b)
    sa, sb = (torch.randint(118, 130, (batch, rows, K // 32), generator=g, dtype=torch.uint8).to(DEV) for rows in (M, N))
    said = L.mpsa_gemm_kernel(0, fmt_a, fmt_b, 1, batch, M, N, K)
    blocks = (M + 15) // 16 * ((N + 15) // 16) * batch
    assert (said > 10) == (blocks <= 2048)
    stage = blocks > 1024 and (fmt_a == fmt_b or fmt_b == 4)
    for dtype, ldc, kernel in ((torch.bfloat16, N, 1 if stage else said), (torch.bfloat16, N + 1, said), (torch.float32, N, said)):
        got, want = (torch.full((batch, M, ldc), 3.0, dtype=dtype, device=DEV) for _ in range(2))
        for out, k in ((got, 0), (want, kernel)):
            _lib.check(L.mpsa_gemm_mx_on(k, _lib.ptr(a), _lib.ptr(sa), fmt_a, _lib.ptr(b), _lib.ptr(sb), fmt_b, 0, 1, batch, batch, M, N, K,
                                         _lib.ptr(out), _lib.dtype_id(dtype), ldc, _lib.stream_ptr(a.device)))
        assert torch.equal(got, want)


@pytest.mark.parametrize("fmt_a,fmt_b", [(4, 4), (0, 4), (1, 1)])
@pytest.mark.parametrize("M,N", [(256, 512), (300, 257), (1, 768), (3001, 4099), (1, 16392), (2176, 2176)])
@pytest.mark.parametrize("K", [128, 256, 384, 512, 640, 768, 896, 1024, 1152, 1280, 1664, 3968])
def test_256_wide_tiles_for_every_remainder_of_k(K, M, N, fmt_a, fmt_b):
    """Scale bytes come four words a row at a time (packed ones a chunk) and codes 256 (4-bit) or 128 elements at a time: every
    length of the last group and, with 4-bit codes, of the last unit gives the general kernel's bits, in the last row of either
    matrix too, and in 16-bit results, which go through the LDS that the codes came through.  Ragged 4-bit products that end in
    half a unit are taken from 64 tiles on."""
    L = _lib.lib()
    g = torch.Generator().manual_seed(K + M)
    if fmt_a == fmt_b == 4 and K % 256 == 128 and (M % 256 or N % 256) and ((M + 255) // 256) * ((N + 255) // 256) < 64:
        assert L.mpsa_gemm_kernel(_lib.GEMM_KERNELS["tile256"], fmt_a, fmt_b, 1, 1, M, N, K) == -3
        return

    def codes(rows, fmt):
        c = torch.randint(0, 256, (rows, K // 2 if fmt == 4 else K), dtype=torch.uint8, generator=g)
        return (c if fmt == 4 else c & 0xBF).to(DEV)

    a, b = codes(M, fmt_a), codes(N, fmt_b)
    sa, sb = (torch.randint(118, 130, (rows, K // 32), dtype=torch.uint8, generator=g).to(DEV) for rows in (M, N))
    for packed in range(1 + (M % 128 == 0 and N % 128 == 0)):
        xa, xb = (pack_scale_5d(sa), pack_scale_5d(sb)) if packed else (sa, sb)
        for dtype in [torch.float32] + [torch.bfloat16] * (N % 8 == 0):
            got, want = (torch.full((M + 1, N), 7.0, dtype=dtype, device=DEV) for _ in range(2))
            for out, kernel in ((got, "tile256"), (want, "general")):
                _lib.check(L.mpsa_gemm_mx_on(_lib.GEMM_KERNELS[kernel], _lib.ptr(a), _lib.ptr(xa), fmt_a, _lib.ptr(b), _lib.ptr(xb), fmt_b, packed, 1, 1, 1, M, N, K,
                                             _lib.ptr(out), _lib.dtype_id(dtype), N, _lib.stream_ptr(a.device)))
            assert torch.equal(got, want)
