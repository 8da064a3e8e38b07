"""Dense products under 65 .. some hundreds of rows: every weight value decoded in registers into the MFMA operand (xq_gemm_mid.h)."""

import pytest
import torch

from oracle import recipe as R
from tests.util_cases import gen, make_dense_module

pytestmark = pytest.mark.gpu

FORMATS = ["int4", "nvfp4", "block_fp8", "nf4"]


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("M,N,K,r", [
    (65, 1152, 1408, 16),        # the fewest rows, a column tile cut in both directions, phases of unequal length
    (97, 2176, 2304, 64),        # a row past 96; every low-rank step of both phases; 9 steps a phase in the forward
    (130, 1024, 4224, 8),        # narrow: the contraction over several blocks, their shares uneven
    (385, 4224, 1152, 1),        # row tiles of 96 and 128 rows with one row left
    (1000, 1280, 2048, 32),      # several row tiles
])
def test_forward_and_backward(hip_device, fmt, M, N, K, r):
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
    test_forward_and_backward(hip_device, "block_fp8", M, N, K, r)


@pytest.mark.parametrize("fmt", FORMATS)
def test_decodes_bit_for_bit(hip_device, fmt):
    """Rows of the identity: a forward returns the decoded weight's columns, a dgrad its rows, without a rounding."""
    rows, other = 1152, 1280
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


def test_gradient_of_two_weights_in_one_product(hip_device):
    """block-fp8 gate and up of an MLP: dX contracts over the rows of both, the second from the middle of a phase's steps on."""
    from xorl_amd.qlora import qlora_mlp_forward

    M, H, I, r = 200, 1280, 1152, 16
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
