"""GPU parity of the dense low-rank products (read from the factors as the caller holds them) and of the per-expert
weight-gradient launch, at the sizes where their launches change form."""

import pytest
import torch

from oracle import recipe as R
from tests.test_gpu_moe import test_moe_fwd_bwd_vs_oracle as check_experts
from tests.util_cases import close, gen, make_dense_module

pytestmark = pytest.mark.gpu
TOL = 1e-2


@pytest.mark.parametrize("bf16_factors", [False, True])
@pytest.mark.parametrize("M,N,K,r", [
    (65, 320, 64, 1),          # one unit of the contraction for sixteen waves
    (100, 64, 1088, 17),       # rows and units that fill no block; ranks of two tiles, the second nearly empty
    (1025, 256, 256, 40),      # wide factors: eight waves; two row splits of the weight gradients
    (4096, 128, 192, 16),      # the last size of short blocks
    (4097, 192, 128, 64),      # tall blocks and bf16 panels
])
def test_linear_training_at_the_edges(hip_device, M, N, K, r, bf16_factors):
    m, w_ref = make_dense_module("block_fp8", N, K, r, 2 * r, seed=M, device=hip_device)
    if bf16_factors:
        m.lora_A.data = m.lora_A.data.to(torch.bfloat16)
        m.lora_B.data = m.lora_B.data.to(torch.bfloat16)
    else:                      # a factor that starts 4 bytes off a 16-byte boundary (a view into a flat parameter)
        flat = torch.zeros(r * K + 1, device=hip_device)
        flat[1:] = m.lora_A.data.reshape(-1)
        m.lora_A.data = flat[1:].view(r, K)
    x = gen((M, K), 1.0, 1, torch.bfloat16)
    dy = gen((M, N), 1.0, 2, torch.bfloat16)
    xd = x.to(hip_device).requires_grad_(True)
    y = m(xd)
    y.backward(dy.to(hip_device))
    ex = R.linear_fwd_bwd_exact(x, w_ref, m.lora_A.detach().float().cpu(), m.lora_B.detach().float().cpu(), m.scaling, dy)
    close(y.detach().cpu(), ex["y"], TOL)
    close(xd.grad.cpu(), ex["dx"], TOL)
    close(m.lora_A.grad.float().cpu(), ex["dA"], TOL)
    close(m.lora_B.grad.float().cpu(), ex["dB"], TOL, rows="last" if r > 1 else "none")       # (rank 1: a row is one dot product)


@pytest.mark.parametrize("M,H,I,r", [
    (70, 128, 576, 16),        # nine units of columns for four waves, one column split
    (300, 256, 1600, 12),      # 25 units over three column splits
    (2047, 128, 512, 32),      # factors as they are, 2048: from panels
    (2048, 128, 512, 32),
])
def test_mlp_training_at_the_edges(hip_device, M, H, I, r):
    from xorl_amd.qlora import qlora_mlp_forward

    mods, w_ref = {}, {}
    for i, (k, (N, K)) in enumerate({"gate": (I, H), "up": (I, H), "down": (H, I)}.items()):
        mods[k], w_ref[k] = make_dense_module("nvfp4", N, K, r, 2 * r, seed=M + 10 * i, device=hip_device)
    x = gen((M, H), 1.0, 3, torch.bfloat16)
    dy = gen((M, H), 1.0, 4, torch.bfloat16)
    loras = {k: (m.lora_A.detach().cpu(), m.lora_B.detach().cpu()) for k, m in mods.items()}
    ex = R.mlp_fwd_bwd_exact(x, w_ref["gate"], w_ref["up"], w_ref["down"], loras, mods["gate"].scaling, dy)
    xd = x.to(hip_device).requires_grad_(True)
    y = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], xd)
    y.backward(dy.to(hip_device))
    close(y.detach().cpu(), ex["y"], TOL)
    close(xd.grad.cpu(), ex["dx"], TOL)
    for k, m in mods.items():
        close(m.lora_A.grad.cpu(), ex[f"dA_{k}"], TOL)
        close(m.lora_B.grad.cpu(), ex[f"dB_{k}"], TOL)


@pytest.mark.parametrize("over", [0, 1])      # 256 rows an expert on average: a block per expert; one more row: row chunks
@pytest.mark.parametrize("r,rp,transpose", [(16, 16, False), (33, 48, True)])
def test_expert_weight_gradients_either_side_of_the_rule(hip_device, r, rp, transpose, over):
    from xorl_amd import moe_functional as MF

    E, width = 4, 200
    counts = torch.tensor([0, 1, 33, 256 * E - 34 + over])
    ends = counts.cumsum(0)
    offsets = torch.cat([torch.zeros(1, dtype=torch.int64), ends]).to(torch.int32).to(hip_device)
    P = gen((int(ends[-1]), width), 1.0, 5, torch.bfloat16)
    Q = gen((int(ends[-1]), rp), 1.0, 6, torch.bfloat16)
    g = MF._wgrad(P.to(hip_device), Q.to(hip_device), r, offsets, E, transpose).cpu()
    for e in range(E):
        lo, hi = int(ends[e] - counts[e]), int(ends[e])
        ref = P[lo:hi].double().t() @ Q[lo:hi, :r].double()
        ref = ref.t() if transpose else ref
        if hi == lo:
            assert torch.count_nonzero(g[e]) == 0
        else:
            close(g[e], ref, 1e-2, rows="none")


@pytest.mark.parametrize("fmt,E,T,I,r,hybrid", [
    ("block_fp8", 3, 1500, 256, 24, False),     # row chunks; dA of gate and up side by side, 64 ranks wide
    ("block_fp8", 12, 200, 256, 16, True),      # a block per expert; the shared factors' gradients in a launch of their own
    ("nvfp4", 3, 1500, 192, 40, True),          # row chunks, every product by itself
    ("nf4", 12, 200, 192, 8, False),
])
def test_expert_factor_gradients_of_a_call(hip_device, fmt, E, T, I, r, hybrid):
    check_experts(hip_device, 0, fmt, E, T, 256, I, r, 2, hybrid)


@pytest.mark.parametrize("r,rp,transpose", [(16, 16, False), (33, 48, True)])
@pytest.mark.parametrize("counts", [
    [0, 1, 33, 2600, 0, 100, 0, 0, 0, 0, 0, 0],          # one expert over three and a bit of four chunks
    [1024, 1024, 0, 500, 1, 0, 0, 0, 0, 0, 0, 0],        # experts that end on the chunks' boundaries
    [1000, 24, 1030, 0, 0, 0, 0, 0, 0, 0, 0, 1000],      # a boundary crossed by six rows; the last expert crosses the last one
    [0, 0, 0, 3000, 0, 0, 0, 0, 0, 0, 0, 0],             # all rows in one
    [1025, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0],
])
def test_expert_weight_gradients_of_uneven_loads(hip_device, counts, r, rp, transpose):
    """Up to 256 rows an expert on average: the bits of the row chunks, which the same rows take under fewer experts."""
    from xorl_amd import moe_functional as MF

    width, counts = 200, torch.tensor(counts)
    offsets = lambda c: torch.cat([torch.zeros(1, dtype=torch.int64), c.cumsum(0)]).to(torch.int32).to(hip_device)
    R = int(counts.sum()) + 5                            # rows behind the last expert's belong to nobody
    P, Q = gen((R, width), 1.0, 5, torch.bfloat16), gen((R, rp), 1.0, 6, torch.bfloat16)
    assert R <= 256 * len(counts)
    got = MF._wgrad(P.to(hip_device), Q.to(hip_device), r, offsets(counts), len(counts), transpose)
    used = counts.nonzero().reshape(-1)
    lo = 0
    for e in range(len(counts)):
        ref = P[lo:lo + counts[e]].double().t() @ Q[lo:lo + counts[e], :r].double()
        lo += int(counts[e])
        if counts[e]:
            close(got[e].cpu(), ref.t() if transpose else ref, 1e-2, rows="none")
        else:
            assert torch.count_nonzero(got[e]) == 0
    if R > 256 * len(used):
        assert torch.equal(got[used.to(hip_device)], MF._wgrad(P.to(hip_device), Q.to(hip_device), r, offsets(counts[used]), len(used), transpose))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("fmt,M,N,K", [
    ("block_fp8", 97, 1168, 640),        # gemm_mid_kernel
    ("block_fp8", 97, 1168, 192),        # 128 x 128 tiles
    ("block_fp8", 2197, 6288, 192),      # gemm_dtl16_kernel
    ("nf4", 2600, 2832, 2816),           # gemm_dec_kernel
])
@pytest.mark.parametrize("r", [1, 7, 9, 20, 33, 63, 64])
def test_rows_of_the_right_factor_at_any_address(hip_device, fmt, M, N, K, r, dtype):
    """Eight ranks of a row of B are read at once where they lie in the row: B begins off a 16-byte boundary and ends its allocation,
    and every second of its rows is infinite, which no finite row's result may show."""
    from xorl_amd.functional import qlora_linear

    m, w = make_dense_module(fmt, N, K, 16, 32, seed=3, device=hip_device)
    A, B = gen((r, K), 0.02, 1).to(dtype), gen((N, r), 0.02, 2).to(dtype)
    B[1::2] = float("inf")
    b = torch.empty(N * r + 1, dtype=dtype, device=hip_device)[1:].view(N, r)
    b.copy_(B)
    x = gen((M, K), 1.0, 4, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        y = qlora_linear(x, m._quant_weight(), A.to(hip_device), b, r, 0.5)
    xf, Af, even = x.float(), A.to(hip_device).float().t(), B[::2].to(hip_device).float().t()
    u, au = xf @ Af, xf.abs() @ Af.abs()
    want = xf @ w[::2].to(hip_device).float().t() + 0.5 * (u @ even)
    # the result's rounding (2^-9, doubled for the fp32 sums) and, in the low-rank term, those of the inner factor's elements, of the
    # intermediate and of the outer factor's (2^-9 of the terms each, nothing cancelling)
    bound = 2 ** -8 * want.abs() + 0.5 * 2 ** -9 * ((au + 2 * u.abs()) @ even.abs()) + 1e-5 * want.abs().max()
    assert bool(((y[:, ::2].float() - want).abs() <= bound).all())
    assert not bool(torch.isfinite(y[:, 1::2]).any())


@pytest.mark.parametrize("bf16_factors", [False, True])
@pytest.mark.parametrize("M,N,K,r", [
    (65, 128, 4160, 64),       # forward over four splits of 65 units, the last one shorter
    (97, 4160, 192, 50),       # backward the same, ranks that fill no tile
    (300, 3136, 9216, 40),     # both, eight splits of the forward
])
def test_low_rank_products_in_splits(hip_device, M, N, K, r, bf16_factors):
    test_linear_training_at_the_edges(hip_device, M, N, K, r, bf16_factors)
