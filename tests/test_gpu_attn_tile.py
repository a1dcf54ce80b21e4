"""The single-tile attention kernel (csrc/attn_fwd_tile.hip) against kernels that share none of its loops, in the row orders that it has
for a few hundred causal workgroups, and with queries that its own quantization has to be careful with."""
import numpy as np
import pytest
import torch

import oracle as O
from conftest import attention_close, make_qkv
from ours.mxfp_attn_kernel import attention_from_operands, mxfp_attn_kernel, prepare_operands

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("bst", ["diag", "mxfp4", "mxfp8", "mixed"])
@pytest.mark.parametrize("B,Hq,Hkv,N", [(1, 100, 50, 300), (1, 100, 100, 600), (1, 32, 8, 1100), (1, 32, 8, 2000), (3, 20, 5, 1000), (1, 300, 300, 100), (1, 33, 11, 1030), (1, 32, 8, 2100)])
def test_causal_row_orders_of_a_few_hundred_workgroups(bst, B, Hq, Hkv, N):
    """300 to 512 workgroups, which have two layers of rows, the second in reverse, with heads that divide 256 and others, and 544,
    which have the plain order: every row of every head as the short-sequence kernel has it, and a list's rows as a fixed run's."""
    q, k, v = (t.to(DEV) for t in make_qkv(B, Hq, Hkv, N, 128, seed=N + Hq))
    run = lambda name: mxfp_attn_kernel(q, k, v, is_causal=True, block_scale_type=bst, tile=128, output_dtype=torch.float32, kernel=name)  # noqa: E731
    got, want = run("tile"), run("short1")
    attention_close(got, want.cpu(), f"{bst} {B}x{Hq}/{Hkv} {N}")
    if bst == "mxfp4":
        nt = -(-N // 128)
        i, j = np.meshgrid(np.arange(nt), np.arange(nt), indexing="ij")
        order, counts = O.route_order(np.broadcast_to(np.where(j > i, 255, 1), (B, Hq, nt, nt)).astype(np.uint8), N, 128, True)
        listed = torch.full((B, Hq, N, 128), float("nan"), dtype=torch.float32, device=DEV)
        attention_from_operands(prepare_operands(q, k, v, 128, "routed"), listed, True, route=(None, torch.from_numpy(order).to(DEV), torch.from_numpy(counts).to(DEV)))
        assert torch.equal(listed, run("general"))


@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("bst", ["diag", "mxfp4", "mxfp8", "mixed_e5"])
@pytest.mark.parametrize("N", [128, 300, 900])
def test_a_kernel_with_another_loop_gives_the_same(N, bst, causal):
    """The kernel that takes a tile's maximum before its exponentials, with a skipping rule that leaves nothing out."""
    q, k, v = (t.to(DEV) for t in make_qkv(1, 4, 2, N, 128, seed=3300 + N, dtype=torch.float16))
    ops = prepare_operands(q, k, v, 128, bst)
    a, b = (torch.full((1, 4, N, 128), float("nan"), dtype=torch.float32, device=DEV) for _ in range(2))
    attention_from_operands(ops, a, causal, kernel="tile")
    attention_from_operands(ops, b, causal, -1e30, skip_in_kernel=True)
    attention_close(a, b.cpu(), f"{bst} {N} causal={causal}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bst", ["diag", "mxfp4", "mxfp8", "mixed", "mxfp8e5"])
@pytest.mark.parametrize("rule", [False, True])
def test_rare_blocks_of_q_have_the_bits_of_prepared_q(bst, dtype, rule):
    """NaN of either sign, infinities, zeros among other values, blocks of zeros and too small for the conversions, a ragged last tile; under
    the default pre-scale, and under one that brings products within a rounding of a midpoint between two E2M1 codes."""
    N = 493
    scale = 1.25 / (1.0 + 5.0 / 128.0) / 1.4426950408889634 if rule else None
    q, k, v = make_qkv(1, 4, 2, N, 128, seed=3400, dtype=torch.float32)
    g = torch.Generator().manual_seed(N)
    q[:, 0, :64] *= (torch.rand(64, 128, generator=g) < 0.5).float()
    q[0, 0, 100:200] = (1.0 + 5.0 / 128.0) * torch.exp2(torch.randint(-4, 2, (100, 128), generator=g).float())
    q[0, 1, 80, 40], q[0, 1, 81, 41], q[0, 1, 82, 100], q[0, 2, 17, 3] = float("nan"), -float("nan"), float("inf"), float("-inf")
    q[0, 1, 90, 32:64], q[0, 2, 91, :32], q[0, 3, N - 1, 127] = 0.0, 6e-8 if dtype == torch.float16 else 1e-39, float("nan")
    q[0, 3, 200:204, :32] *= 1e-7 if dtype == torch.float16 else 1e-34
    q, k, v = (t.to(dtype).to(DEV) for t in (q, k, v))
    for causal in (True, False):
        a, b = (torch.empty((1, 4, N, 128), dtype=torch.float32, device=DEV) for _ in range(2))
        attention_from_operands(prepare_operands(q, k, v, 128, bst, scale), a, causal, kernel="tile")
        attention_from_operands(prepare_operands(q, k, v, 128, bst, scale, fuse_q=True), b, causal, kernel="tile")
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.nan_to_num(a, nan=0.0), torch.nan_to_num(b, nan=0.0)), causal
