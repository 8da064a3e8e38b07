"""Dense products from 65 rows on whose weight is decoded in registers into the MFMA operand (xq_gemm_mid.h)."""

import pytest
import torch

from oracle import recipe as R
from tests.util_cases import dense_route, gen, make_dense_module

pytestmark = pytest.mark.gpu

FORMATS = ["int4", "nvfp4", "block_fp8", "nf4"]


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("M,N,K,r", [
    (65, 1152, 1408, 16),        # the fewest rows, a column tile cut in both directions, phases of unequal length
    (97, 2176, 2304, 64),        # a row past 96; every low-rank step of both phases; 9 steps a phase in the forward
    (130, 1024, 4224, 8),        # narrow: the contraction over several blocks, their shares uneven
    (385, 4224, 1152, 1),        # one row past six row tiles; the dgrad in seven splits
    (1000, 1280, 2048, 32),      # several row tiles
])
def test_forward_and_backward(hip_device, fmt, M, N, K, r):
    # (block-fp8 and nf4 products of a few of these sizes are shorter on the tile kernels)
    assert fmt in ("block_fp8", "nf4") or dense_route(fmt, True, M, N, K)[0] == dense_route(fmt, False, M, K, N)[0] == "mid"
    m, w_ref = make_dense_module(fmt, N, K, r, 32, seed=3, device=hip_device, bias=(M in (97, 385)))
    x, dy = gen((M, K), 1.0, 4, torch.bfloat16), gen((M, N), 1.0, 5, torch.bfloat16)
    xd = x.to(hip_device).requires_grad_(True)
    y = m(xd)
    y.backward(dy.to(hip_device))
    bias = m.bias.detach().cpu().to(torch.bfloat16) if m.bias is not None else None
    ex = R.linear_fwd_bwd_exact(x, w_ref, m.lora_A.detach().cpu(), m.lora_B.detach().cpu(), m.scaling, dy, bias)
    # operands are exact in bf16 and sums are fp32: what is left is the rounding of the result (2^-9) and of the
    # low-rank intermediate, as in every tile kernel
    for name, got, ref in (("y", y, ex["y"]), ("dx", xd.grad, ex["dx"]), ("dA", m.lora_A.grad, ex["dA"]), ("dB", m.lora_B.grad, ex["dB"])):
        err = R.max_rel_err(got.detach().cpu(), ref)
        assert err <= 1e-2, f"{name}: {err}"


@pytest.mark.parametrize("M,N,K,r", [
    (65, 1152, 384, 16),         # the shortest contraction that a forward brings here: three steps a phase
    (130, 2176, 448, 64),        # phases of four and three steps, half a scale block at the end
    (300, 960, 960, 8),
    (513, 4096, 576, 32),
])
def test_short_block_fp8_contractions(hip_device, M, N, K, r):
    assert dense_route("block_fp8", True, M, N, K)[0] == "mid"
    test_forward_and_backward(hip_device, "block_fp8", M, N, K, r)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("M,tile_rows", [(513, 96), (769, 128)])
def test_taller_row_tiles(hip_device, fmt, M, tile_rows):
    """Tiles of 96 and 128 rows, the last with 33 rows or one, its columns cut, phases of unequal length and three low-rank steps dealt to
    them: both directions of a product against fp32 products of the decoded weight.  Elementwise bound: the result's rounding (2^-9,
    doubled for the fp32 sums and the bias) and, in the low-rank term, those of the inner factor's elements, of the intermediate and of
    the outer factor's (2^-9 of the terms each, nothing cancelling)."""
    def check(got, x, w, inner, outer, bias):
        u, au = x @ inner, x.abs() @ inner.abs()
        want = x @ w + m.scaling * (u @ outer) + bias
        bound = 2 ** -8 * want.abs() + m.scaling * 2 ** -9 * ((au + 2 * u.abs()) @ outer.abs()) + 1e-5 * want.abs().max()
        assert bool(((got.float() - want).abs() <= bound).all())

    n, k = 7296, 704 if fmt == "block_fp8" else 640
    assert dense_route(fmt, True, M, n, k)[:2] == ("mid", tile_rows)
    m, w = make_dense_module(fmt, n, k, 48, 32, seed=5, device=hip_device, bias=True)
    x = gen((M, k), 1.0, 6, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        check(m(x), x.float(), w.to(hip_device).float().t(), m.lora_A.t(), m.lora_B.t(), m.bias.to(torch.bfloat16).float())
    k = 704
    assert dense_route(fmt, False, M, n, k)[:2] == ("mid", tile_rows)
    m, w = make_dense_module(fmt, k, n, 48, 32, seed=5, device=hip_device)
    dy = gen((M, k), 1.0, 7, torch.bfloat16).to(hip_device)
    x = torch.zeros(M, n, dtype=torch.bfloat16, device=hip_device).requires_grad_(True)
    m(x).backward(dy)
    with torch.no_grad():
        check(x.grad, dy.float(), w.to(hip_device).float(), m.lora_B, m.lora_A, 0.0)


@pytest.mark.parametrize("fmt", FORMATS)
def test_decodes_bit_for_bit(hip_device, fmt):
    """Rows of the identity: a forward returns the decoded weight's columns, a dgrad its rows, without a rounding."""
    rows, other = 640 if fmt == "nf4" else 1152, 1280
    assert dense_route(fmt, True, rows, other, rows)[0] == dense_route(fmt, False, rows, other, rows)[0] == "mid"
    eye = torch.eye(rows, dtype=torch.bfloat16, device=hip_device)
    m, w_ref = make_dense_module(fmt, other, rows, 8, 16, seed=7, device=hip_device)
    with torch.no_grad():
        m.lora_B.zero_()
    assert torch.equal(m(eye.requires_grad_(True)).detach().cpu(), w_ref.t())
    m, w_ref = make_dense_module(fmt, rows, other, 8, 16, seed=7, device=hip_device)
    with torch.no_grad():
        m.lora_B.zero_()
    x = torch.zeros(rows, other, dtype=torch.bfloat16, device=hip_device).requires_grad_(True)
    m(x).backward(eye.detach())
    assert torch.equal(x.grad.cpu(), w_ref)


@pytest.mark.parametrize("M,H,I,tile_rows,splits", [
    (385, 2048, 896, 64, 3),     # the second weight begins at the fifth step of phase 0 of the second split
    (300, 1920, 1664, 64, 4),    # ... at the sixth of phase 1 of the second split
    (769, 1664, 2432, 96, 4),    # ... at the ninth
])
def test_gradient_of_two_weights_in_one_product(hip_device, M, H, I, tile_rows, splits):
    """block-fp8 gate and up of an MLP: dX contracts over the rows of both, the second from the middle of a phase's steps on."""
    from xorl_amd.qlora import qlora_mlp_forward

    assert dense_route("block_fp8", False, M, H, 2 * I)[:4] == ("mid", tile_rows, 256, splits)
    steps, parts = 2 * I // 64, 2 * splits                           # (the first `steps % parts` parts are one step longer)
    begins = [p * (steps // parts) + min(p, steps % parts) for p in range(parts)]
    assert I // 64 not in begins
    r = 16
    mods, w = {}, {}
    for i, (k, (n, kk)) in enumerate({"gate": (I, H), "up": (I, H), "down": (H, I)}.items()):
        mods[k], w[k] = make_dense_module("block_fp8", n, kk, r, 32, seed=11 + i, device=hip_device)
    x, dy = gen((M, H), 1.0, 21, torch.bfloat16), gen((M, H), 1.0, 22, torch.bfloat16)
    xd = x.to(hip_device).requires_grad_(True)
    y = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], xd)
    y.backward(dy.to(hip_device))
    loras = {k: (m.lora_A.detach().cpu(), m.lora_B.detach().cpu()) for k, m in mods.items()}
    ex = R.mlp_fwd_bwd_exact(x, w["gate"], w["up"], w["down"], loras, mods["gate"].scaling, dy)
    assert R.max_rel_err(y.detach().cpu(), ex["y"]) <= 1e-2
    assert R.max_rel_err(xd.grad.cpu(), ex["dx"]) <= 2e-2       # (dgate and dup are bf16: one more rounding than above)


@pytest.mark.parametrize("rows", [0, 1])
def test_rows_at_any_pitch(hip_device, rows):
    """A slice of a wider activation, its rows at their pitch: the bits of the packed copy."""
    m, _ = make_dense_module("nvfp4", 1152, 1408, 16, 32, seed=5, device=hip_device)
    wide = gen((200, 3 * 1408), 1.0, 6, torch.bfloat16).to(hip_device)
    x = wide[rows:, 1408:2816]
    with torch.no_grad():
        assert torch.equal(m(x), m(x.contiguous()))
