"""HIP MX quantizer against the CPU oracle: packed codes and E8M0 scale bytes must be bit-identical."""
import pytest
import torch

import oracle as O
from conftest import make_qkv
from ours import _lib
from ours.quant_mxint8 import seq_mean, quantize_mx, quantize_mx_dual, quant_mxfp4, quant_mxfp8, quant_mxfp8e5, pre_scale_q

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
FMTS = [O.FMT_E2M1, O.FMT_E4M3, O.FMT_E5M2]


def _check(x, pre, fmt, **kw):
    codes, scales = quantize_mx(x.to(DEV), pre, fmt, **kw)
    want_c, want_s = O.quantize_mx(x, pre, fmt)
    n = x.shape[2]
    assert torch.equal(scales[:, :, :n].cpu(), want_s), "scale bytes differ"
    bad = (codes[:, :, :n].cpu() != want_c)
    assert not bad.any(), f"{bad.sum().item()} code bytes differ (fmt {fmt})"
    return codes, scales


@pytest.mark.parametrize("fmt", FMTS)
def test_c1_shapes(fmt):
    q, k, _ = make_qkv(1, 8, 8, 1024, 64, seed=0)
    assert pre_scale_q(64) == O.q_pre_scale(64)
    _check(q, O.q_pre_scale(64), fmt)
    _check(k, 1.0, fmt)


@pytest.mark.parametrize("fmt", FMTS)
def test_c3_shapes_with_outlier_channels(fmt):
    q, k, _ = make_qkv(1, 8, 2, 8192, 128, seed=2, outliers=True)
    _check(q, O.q_pre_scale(128), fmt)
    _check(k, 1.0, fmt)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_wide_dynamic_range_zero_blocks_and_tiny_values(dtype):
    g = torch.Generator().manual_seed(9)
    x = torch.randn(2, 3, 257, 128, generator=g) * torch.exp2(torch.randint(-14, 14, (2, 3, 257, 1), generator=g).float())
    x[0, 0, 5] = 0
    x[1, 2, 100, 32:64] = 0
    x[0, 1, 7, :32] = -0.0
    x[1, 1, 9, 64:96] = 6e-8 if dtype == torch.float16 else 1e-38
    x = x.to(dtype)
    for fmt in FMTS:
        _check(x, 1.0, fmt)
        _check(x, O.q_pre_scale(128), fmt)


def test_near_tie_values_follow_the_biased_compare():
    """Q-path style inputs: bf16 values whose float32 product with the pre-scale lands within 1e-6 of a grid
    midpoint are rare, so force them: pre-scale 1 and values at midpoints +- a few float32 ulps are not bf16 --
    instead use fp16 inputs with a pre-scale that maps them next to midpoints."""
    mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0])
    base = torch.tensor([0.5, 1.5, 2.5, 3.5, 5.0, 7.0, 10.0])       # fp16-exact; base * 0.5 = midpoint
    rows = []
    for ulps in range(-6, 7):
        pre = float(torch.tensor(0.5).view(torch.int32).add(ulps).view(torch.float32))
        row = torch.zeros(32)
        row[:7] = base
        row[7] = 16.0                                                # pins amax: 16*pre in [4,8)*... -> scale 2^-1.. checked by oracle
        rows.append((pre, row))
    for pre, row in rows:
        x = row.reshape(1, 1, 1, 32).to(torch.float16)
        _check(x, pre, O.FMT_E2M1)
    assert mids.numel() == 7


@pytest.mark.parametrize("emax", [7, 8, 20, -1])
@pytest.mark.parametrize("fmt,lim,kind", [(O.FMT_E4M3, 448.0, torch.float8_e4m3fn), (O.FMT_E5M2, 57344.0, torch.float8_e5m2)])
def test_8bit_codes_of_nan_infinity_and_values_past_the_maximum(fmt, lim, kind, emax):
    """The clamp to +-maximum in front of the 8-bit rounding, exactly: a NaN leaves it as the negative maximum and counts as zero
    in its block's largest magnitude, infinities and (under another emax) larger values saturate."""
    g = torch.Generator().manual_seed(emax + 2)
    x = torch.randn(1, 2, 96, 128, generator=g) * torch.exp2(torch.randint(-110, 126, (1, 2, 96, 4, 1), generator=g).expand(-1, -1, -1, -1, 32).reshape(1, 2, 96, 128).float())
    odd = torch.tensor([float("nan"), float("inf"), -float("inf"), -0.0])[torch.randint(0, 4, x.shape, generator=g)]
    x = torch.where(torch.rand(x.shape, generator=g) < 0.01, odd, x)
    x[0, 0, :2] = float("nan")
    x = x.to(torch.bfloat16)
    pre = 0.1275174
    y = (x.float() * pre).view(-1, 32)
    amax = y.nan_to_num(0.0, float("inf"), -float("inf")).abs().amax(1)
    e = torch.where(amax.isinf(), 128, torch.frexp(amax.nan_to_num(0.0, 1.0))[1] - 1)
    se = e - emax
    z = torch.ldexp(y.double(), -se[:, None].double())
    want = torch.where(z.isnan(), -lim, z.clamp(-lim, lim)).float().to(kind).view(torch.uint8)
    want[amax == 0] = 0
    scales = torch.where(amax == 0, 0, (se + 127).clamp(0, 254)).to(torch.uint8)
    codes, got = quantize_mx(x.to(DEV), pre, fmt, emax_elem=emax)
    assert torch.equal(got.cpu().view(-1), scales)
    assert torch.equal(codes.cpu().view(-1, 32), want)


def test_dual_equals_single_and_padding_rows_are_zero():
    q, _, _ = make_qkv(1, 4, 4, 200, 128, seed=4)
    pre = O.q_pre_scale(128)
    c4, s4, c8, s8 = quantize_mx_dual(q.to(DEV), pre, _lib.FMT_E4M3, out_rows=256)
    a4, b4 = _check(q, pre, O.FMT_E2M1, out_rows=256)
    a8, b8 = _check(q, pre, O.FMT_E4M3, out_rows=256)
    assert torch.equal(c4, a4) and torch.equal(s4, b4) and torch.equal(c8, a8) and torch.equal(s8, b8)
    for t in (c4, s4, c8, s8):
        assert t.shape[2] == 256 and (t[:, :, 200:] == 0).all()
    d4, t4, d5, t5 = quantize_mx_dual(q.to(DEV), pre, _lib.FMT_E5M2)
    w5, ws5 = O.quantize_mx(q, pre, O.FMT_E5M2)
    assert torch.equal(d5.cpu(), w5) and torch.equal(t5.cpu(), ws5) and torch.equal(d4, c4[:, :, :200])


def test_reference_style_entry_points_and_layouts():
    q, k, _ = make_qkv(2, 4, 2, 256, 64, seed=6)
    qd, kd = q.to(DEV), k.to(DEV)
    qc, qs, kc, ks = quant_mxfp4(qd, kd)
    wq, wqs = O.quantize_mx(q, O.q_pre_scale(64), O.FMT_E2M1)
    wk, wks = O.quantize_mx(k, 1.0, O.FMT_E2M1)
    assert torch.equal(qc.cpu(), wq) and torch.equal(qs.cpu(), wqs) and torch.equal(kc.cpu(), wk) and torch.equal(ks.cpu(), wks)
    # one code per byte, as the reference returns them
    qu, _, _, _ = quant_mxfp4(qd, kd, packed=False)
    assert qu.shape == q.shape and torch.equal(qu.cpu(), O.unpack_fp4(wq))
    # NHD: [B, L, H, D] input is read through its strides, outputs stay [B, H, L, *]
    qn, kn = qd.transpose(1, 2).contiguous(), kd.transpose(1, 2).contiguous()
    qc2, qs2, kc2, ks2 = quant_mxfp4(qn, kn, tensor_layout="NHD")
    assert torch.equal(qc2, qc) and torch.equal(ks2, ks)
    # custom softmax scale and the 8-bit siblings
    qc3, qs3, _, _ = quant_mxfp8(qd, kd, sm_scale=0.3)
    w3, ws3 = O.quantize_mx(q, O.q_pre_scale(64, 0.3), O.FMT_E4M3)
    assert torch.equal(qc3.cpu(), w3) and torch.equal(qs3.cpu(), ws3)
    qc5, _, kc5, ks5 = quant_mxfp8e5(qd, kd)
    assert qc5.dtype == torch.float8_e5m2
    w5, ws5 = O.quantize_mx(k, 1.0, O.FMT_E5M2)
    assert torch.equal(kc5.view(torch.uint8).cpu(), w5) and torch.equal(ks5.cpu(), ws5)
    with pytest.raises(ValueError, match="Unknown tensor layout"):
        quant_mxfp4(qd, kd, tensor_layout="DNH")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 8, 8192, 128), (2, 3, 1000, 64), (1, 2, 32760, 128), (1, 1, 7, 64)])
def test_smooth_k_mean_and_fused_subtraction(shape, dtype):
    """mpsa_seq_mean against the oracle's once-rounded mean (summation order may move the 16-bit result by one
    unit in the last place on rare channels: at most 1 ulp anywhere, equal on more than 99 %), and the
    quantizer's fused ``x - mean`` bit for bit against the oracle quantizing ``smooth_k(k, that mean)``."""
    B, H, N, D = shape
    g = torch.Generator().manual_seed(N + D)
    k = (torch.randn(B, H, N, D, generator=g) + torch.randn(1, H, 1, D, generator=g) * 2).to(dtype)
    got = seq_mean(k.to(DEV))
    assert got.shape == (B, H, D) and got.dtype == dtype
    want = O.seq_mean(k).squeeze(-2)
    same = (got.cpu() == want)
    assert same.float().mean().item() > 0.99
    ulp = torch.finfo(dtype).eps * want.float().abs().clamp_min(2.0 ** -14)
    assert ((got.cpu().float() - want.float()).abs() <= ulp).all()
    smoothed = O.smooth_k(k, got.cpu())
    for fmt in FMTS:
        codes, scales = quantize_mx(k.to(DEV), 1.0, fmt, sub=got)
        want_c, want_s = O.quantize_mx(smoothed, 1.0, fmt)
        assert torch.equal(scales.cpu(), want_s) and torch.equal(codes.cpu(), want_c), f"fmt {fmt}"
    c4, s4, c8, s8 = quantize_mx_dual(k.to(DEV), 1.0, O.FMT_E4M3, out_rows=N + 9, sub=got)
    w4, ws4 = O.quantize_mx(smoothed, 1.0, O.FMT_E2M1)
    w8, ws8 = O.quantize_mx(smoothed, 1.0, O.FMT_E4M3)
    assert torch.equal(c4[:, :, :N].cpu(), w4) and torch.equal(s4[:, :, :N].cpu(), ws4)
    assert torch.equal(c8[:, :, :N].cpu(), w8) and torch.equal(s8[:, :, :N].cpu(), ws8)
    assert not c4[:, :, N:].any() and not c8[:, :, N:].any() and not s4[:, :, N:].any()


def test_hardware_e2m1_conversion_agrees_with_the_explicit_rule_near_every_midpoint():
    """The quantizer's fast path (hardware FP4 conversion) must hand every value near a rounding boundary to
    the explicit rule: float32-dense sweeps around each of the seven midpoints, reached through a pre-scale
    that makes the scaled values arbitrary float32 numbers, and blocks whose scale is not a normal float32."""
    mids = torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0])
    rows = []
    for m in mids.tolist():
        base = torch.tensor(m, dtype=torch.float32)
        steps = torch.arange(-24, 25, dtype=torch.float32)
        vals = base + steps * 1.25e-7 * max(m, 1.0)            # a few float32 ulps either side, +-3e-6
        for chunk in vals.split(31):
            blk = torch.full((32,), 0.0)
            blk[0] = 6.0                                        # pins the shared exponent: scale 2^(2-3)... = 0.5
            blk[1:1 + chunk.numel()] = chunk
            rows.append(blk)
            rows.append(-blk)
    x = torch.stack(rows)                                       # [R, 32] float32 targets of x*pre / 2^se with se = -1
    # choose bf16 inputs and a pre-scale so that f32(x)*pre lands on arbitrary float32 values near the targets
    pre = 0.7310585975646973
    xin = (x * 0.5 / pre).bfloat16().view(1, 1, -1, 32)
    xin = torch.cat([xin, (xin.float() * 2.0 ** -120).bfloat16()], dim=2)       # tiny blocks: scale below 2^-126
    for p in (pre, 1.0, 0.9999998807907104, 1.0000001192092896):
        codes, scales = quantize_mx(xin.to(DEV), p, O.FMT_E2M1)
        want_c, want_s = O.quantize_mx(xin, p, O.FMT_E2M1)
        assert torch.equal(scales.cpu(), want_s) and torch.equal(codes.cpu(), want_c), f"pre {p}"
    # a dense float32 sweep through the pre-scale instead of the input: the scaled value walks across each midpoint
    one = torch.zeros(1, 1, 1, 32); one[..., 0] = 6.0
    for m in mids.tolist():
        xb = one.clone(); xb[..., 1:] = m
        xb = xb.bfloat16()
        for k in range(-40, 41):
            p = float(torch.tensor(1.0 + k * 2.0 ** -23, dtype=torch.float32))
            if (xb.float().abs().max() * p) >= 8.0:
                continue
            codes, scales = quantize_mx(xb.to(DEV), p, O.FMT_E2M1)
            want_c, want_s = O.quantize_mx(xb, p, O.FMT_E2M1)
            assert torch.equal(codes.cpu(), want_c) and torch.equal(scales.cpu(), want_s), f"mid {m} pre {p}"


@pytest.mark.parametrize("fmt", [O.FMT_E2M1, O.FMT_E4M3])
def test_c2_gemm_operand_full_size(fmt):
    """The 8192 x 8192 GEMM operand of the standalone config, quantized along K: every byte against the oracle."""
    g = torch.Generator().manual_seed(1)
    a = torch.randn(8192, 8192, generator=g).bfloat16()
    codes, scales = quantize_mx(a.to(DEV)[None, None], 1.0, fmt)
    codes, scales = codes[0, 0].cpu(), scales[0, 0].cpu()
    for r0 in range(0, 8192, 2048):                       # oracle in slabs to bound host memory
        wc, ws = O.quantize_mx(a[r0:r0 + 2048], 1.0, fmt)
        assert torch.equal(codes[r0:r0 + 2048], wc) and torch.equal(scales[r0:r0 + 2048], ws)


def test_empty_and_single_row_inputs():
    """Zero heads / zero rows are accepted and write nothing; one row works."""
    for shape in [(0, 2, 16, 64), (1, 0, 16, 64), (1, 2, 0, 64)]:
        x = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
        codes, scales = quantize_mx(x, 1.0, O.FMT_E2M1)
        assert codes.shape == (*shape[:3], 32) and scales.shape == (*shape[:3], 2)
    x = torch.randn(1, 1, 1, 32).bfloat16()
    _check(x, 1.0, O.FMT_E2M1)
    _check(x, 1.0, O.FMT_E4M3, out_rows=5)


@pytest.mark.parametrize("fmt", [0, 1, 4])
@pytest.mark.parametrize("B,H,L,rows,D", [(1, 1, 128, 128, 128), (2, 3, 200, 256, 128), (1, 2, 128, 384, 640)])
def test_layouts_written_directly_equal_the_separate_passes(fmt, B, H, L, rows, D):
    from ours.block_scaled_matmul import pack_scale_5d
    from ours.mxfp import MXFP4Tensor
    from ours.quant_mxint8 import _quantize_as, quantize_mx
    x = torch.randn(B, H, L, D, dtype=torch.bfloat16, device="cuda")
    codes, scales = quantize_mx(x, 1.0, fmt, out_rows=rows)
    wide, packed = _quantize_as(x, 1.0, fmt, out_rows=rows, code_per_byte=True, scales_5d=True)
    want = MXFP4Tensor(size=(1,)).unpack_packed_tensor(codes, 3, (B, H, rows, D)) if fmt == 4 else codes
    assert torch.equal(wide, want) and torch.equal(packed, pack_scale_5d(scales))


@pytest.mark.parametrize("rows", [-1, -5, 0, 99])
def test_fewer_output_rows_than_the_input_has_are_an_error(rows):
    x = torch.randn(1, 2, 100, 64, device=DEV).bfloat16()
    with pytest.raises(RuntimeError):
        quantize_mx(x, 1.0, O.FMT_E2M1, out_rows=rows)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("pre", [1.0, 0.1275174])
def test_small_blocks_on_either_side_of_the_step_by_step_conversion(fmt, pre):
    """Blocks whose scale is 2^-100 or less are converted step by step, the others by the scaled conversion: every exponent
    around that line, with elements down to subnormal ones, zeros and exact ties."""
    g = torch.Generator().manual_seed(4)
    x = torch.randn(1, 1, 64, 64, generator=g)
    x[..., ::7] = 0.0
    x[..., 3::16] = torch.tensor([0.25, 0.75, 1.25, 2.5])
    x[..., 5::16] *= 2.0 ** -24
    x = (x * torch.exp2(torch.arange(-126, -62).float())[None, None, :, None]).bfloat16()
    _check(x, pre, fmt)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("fmt_a,fmt_b", [(4, 4), (0, 0), (1, 1), (0, 4), (1, 4), (4, 0)])
@pytest.mark.parametrize("shape_a,shape_b", [((1, 1, 1, 32), (1, 1, 1, 32)), ((2, 3, 129, 64), (2, 1, 77, 64)), ((1, 5, 128, 128), (1, 2, 256, 128)), ((3, 64), (1000, 96)), ((256, 128), (128, 384))])
def test_two_tensors_in_one_launch_give_the_results_of_two(shape_a, shape_b, fmt_a, fmt_b, dtype):
    from ours.quant_mxint8 import quantize_pair
    g = torch.Generator().manual_seed(sum(shape_a))
    a, b = (torch.randn(*s, generator=g).to(dtype).to(DEV) for s in (shape_a, shape_b))
    whole = all(s[-1] % 128 == 0 and s[-2] % 128 == 0 for s in (shape_a, shape_b))
    for per_byte in (False, True):
        for five in ((False, True) if whole else (False,)):
            got = quantize_pair(a, b, 0.1275174, 1.0, fmt_a, fmt_b, per_byte, five)
            want = []
            for x, pre, fmt in ((a, 0.1275174, fmt_a), (b, 1.0, fmt_b)):
                from ours.quant_mxint8 import _quantize_as
                c, s = _quantize_as(x if x.dim() == 4 else x[None, None], pre, fmt, code_per_byte=per_byte, scales_5d=five)
                want += [c, s] if x.dim() == 4 else [c[0, 0], s[0, 0]]
            assert all(torch.equal(x, y) and x.shape == y.shape for x, y in zip(got, want))
    # rows of a wider tensor: strides of their own
    if len(shape_a) == 4:
        wide = torch.randn(*shape_a[:-1], shape_a[-1] + 8, generator=g).to(dtype).to(DEV)
        got = quantize_pair(wide[..., 8:], b, 1.0, 1.0, fmt_a, fmt_b)
        c, s = quantize_mx(wide[..., 8:].contiguous(), 1.0, fmt_a)
        assert torch.equal(got[0], c) and torch.equal(got[1], s)


def test_codes_of_two_tensors_packed_in_one_launch():
    from ours.mxfp_attn_kernel import initialize_block_scaled_batched_from_tensor
    g = torch.Generator().manual_seed(2)
    for M, N in ((128, 256), (256, 128)):
        a, b = (torch.randint(0, 16, (1, 2, rows, 128), generator=g, dtype=torch.uint8).to(DEV) for rows in (M, N))
        sa, sb = (torch.full((1, 2, rows // 128, 1, 32, 4, 4), 127, dtype=torch.uint8, device=DEV) for rows in (M, N))
        got = initialize_block_scaled_batched_from_tensor(a, b, sa, sb, "mxfp4")
        for codes, packed in ((a, got[0]), (b, got[2])):
            assert torch.equal(packed, codes[..., ::2] | codes[..., 1::2] << 4)
    odd = torch.randint(0, 16, (3, 7), generator=g, dtype=torch.uint8).to(DEV)
    even = torch.randint(0, 16, (3, 32), generator=g, dtype=torch.uint8).to(DEV)
    first, second = _lib.host().pack_pair(odd, even, _lib.raw_stream(odd))
    assert torch.equal(second, even[:, ::2] | even[:, 1::2] << 4)
    assert torch.equal(first[:, :3], odd[:, :6:2] | odd[:, 1::2] << 4) and torch.equal(first[:, 3], odd[:, 6])
