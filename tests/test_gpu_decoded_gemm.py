"""Dense 4-bit weights under many rows: the weight decoded once into bf16 images, the products over those (xq_gemm_dec.h)."""

import ctypes

import pytest
import torch

from oracle import recipe as R
from tests.util_cases import dense_route, gen, make_dense_module

pytestmark = pytest.mark.gpu

FOUR_BIT = ["int4", "nvfp4", "nf4"]


@pytest.mark.parametrize("fmt,M,N,K,r", [
    *[(f, 640, 8192, 4096, 16) for f in FOUR_BIT],          # the fewest rows; K splits (nf4; the others decode in registers)
    *[(f, 1357, 4160, 3904, 64) for f in FOUR_BIT],         # rows, columns and K-steps that fill no tile or split evenly (nf4, nvfp4's forward)
    ("int4", 3432, 5120, 1152, 16), ("nvfp4", 3432, 5120, 1152, 64),       # 288-row tiles; 256-row ones in K splits in the dgrad
    ("nvfp4", 2305, 12352, 768, 8),                         # whole rounds of tiles and one row; K splits in the dgrad
    ("block_fp8", 6145, 1088, 3136, 32),                    # (the dgrad)
])
def test_forward_and_backward(hip_device, fmt, M, N, K, r):
    K = -(-K // 128) * 128 if fmt == "int4" else K              # (int4 groups are 128 wide and do not cross rows)
    m, w_ref = make_dense_module(fmt, N, K, r, 32, seed=3, device=hip_device, bias=(M == 1357))
    x, dy = gen((M, K), 1.0, 4, torch.bfloat16), gen((M, N), 1.0, 5, torch.bfloat16)
    xd = x.to(hip_device).requires_grad_(True)
    y = m(xd)
    y.backward(dy.to(hip_device))
    ex = R.linear_fwd_bwd_exact(x, w_ref, m.lora_A.detach().cpu(), m.lora_B.detach().cpu(), m.scaling, dy)
    want = ex["y"] + (m.bias.detach().cpu().to(ex["y"].dtype) if m.bias is not None else 0)
    # operands are exact in bf16 and sums are fp32: what is left is the rounding of the result (2^-9) and of the
    # low-rank intermediate, as in every tile kernel
    for name, got, ref in (("y", y, want), ("dx", xd.grad, ex["dx"]), ("dA", m.lora_A.grad, ex["dA"]), ("dB", m.lora_B.grad, ex["dB"])):
        err = R.max_rel_err(got.detach().cpu(), ref)
        assert err <= 1e-2, f"{name}: {err}"


@pytest.mark.parametrize("fmt,M,n,k,plan", [
    ("nvfp4", 4881, 3088, 1536, (288, 256, 1)),                                     # 288-row tiles, the last with one row, 16 columns past a whole one
    ("nvfp4", 5436, 3600, 1024, (320, 256, 1)),                      # 320-row tiles
    ("nvfp4", 3845, 5104, 1024, (256, 320, 1)),                      # 320-column tiles across the image's 256, the last one not full
    ("nvfp4", 5140, 4112, 1536, (256, 256, 1, 224, 256, 1)),         # 224-row tiles behind whole rounds of 256-row ones
    ("nvfp4", 1181, 2432, 7232, (256, 256, 5)), ("nvfp4", 7015, 1152, 6272, (288, 256, 2)),      # 256- and 288-row tiles in K splits
    ("block_fp8", 5572, 3200, 3072, (320, 256, 1)),         # below the rows from which it always decodes first
])
def test_tiles_that_fill_their_rounds(hip_device, fmt, M, n, k, plan):
    """Both directions of a [M, n] product over k, rows and columns that end inside a tile, against fp32 products of the decoded
    weight.  Elementwise bound: the result's rounding (2^-9, doubled for the fp32 sums and the bias) and, in the low-rank term, those
    of the inner factor's elements, of the intermediate and of the outer factor's (2^-9 of the terms each, nothing cancelling)."""
    def check(got, x, w, inner, outer, bias):
        u, au = x @ inner, x.abs() @ inner.abs()
        want = x @ w + m.scaling * (u @ outer) + bias
        bound = 2 ** -8 * want.abs() + m.scaling * 2 ** -9 * ((au + 2 * u.abs()) @ outer.abs()) + 1e-5 * want.abs().max()
        assert bool(((got.float() - want).abs() <= bound).all())

    assert dense_route(fmt, True, M, n, k) == ("image", *plan, *[0] * (6 - len(plan)))
    m, w = make_dense_module(fmt, n, k, 16, 32, seed=5, device=hip_device, bias=True)
    x = gen((M, k), 1.0, 6, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        check(m(x), x.float(), w.to(hip_device).float().t(), m.lora_A.t(), m.lora_B.t(), m.bias.to(torch.bfloat16).float())
    n = -(-n // 64) * 64                                        # (what the low-rank products of a module take)
    assert dense_route(fmt, False, M, n, k) == ("image", *plan, *[0] * (6 - len(plan)))
    m, w = make_dense_module(fmt, k, n, 16, 32, seed=5, device=hip_device)
    dy = gen((M, k), 1.0, 7, torch.bfloat16).to(hip_device)
    x = torch.zeros(M, n, dtype=torch.bfloat16, device=hip_device).requires_grad_(True)
    m(x).backward(dy)
    with torch.no_grad():
        check(x.grad, dy.float(), w.to(hip_device).float(), m.lora_B, m.lora_A, 0.0)


@pytest.mark.parametrize("fmt,rows,other", [*[(f, 4160, 1280) for f in FOUR_BIT], ("int4", 2304, 3840), ("nvfp4", 2304, 3840), ("block_fp8", 6208, 576)])
def test_decodes_bit_for_bit(hip_device, fmt, rows, other):
    """Rows of the identity: a forward returns the decoded weight's columns, a dgrad its rows, without a rounding."""
    # (4160 rows, 1280 others: int4 decodes in registers, and so does nvfp4's dgrad)
    assert other == 1280 or dense_route(fmt, True, rows, other, rows)[0] == dense_route(fmt, False, rows, other, rows)[0] == "image"
    eye = torch.eye(rows + (-rows % 128 if fmt == "int4" else 0), dtype=torch.bfloat16, device=hip_device)
    m, w_ref = make_dense_module(fmt, other, eye.shape[0], 8, 16, seed=7, device=hip_device)
    with torch.no_grad():
        m.lora_B.zero_()
        assert torch.equal(m(eye).cpu(), w_ref.t())
    m, w_ref = make_dense_module(fmt, rows, other, 8, 16, seed=7, device=hip_device)
    with torch.no_grad():
        m.lora_B.zero_()
    x = torch.zeros(rows, other, dtype=torch.bfloat16, device=hip_device).requires_grad_(True)
    m(x).backward(eye[:rows, :rows].contiguous())
    assert torch.equal(x.grad.cpu(), w_ref)


def test_without_room_for_the_image(hip_device):
    """A workspace of the size that was enough before still is: the tile kernel decodes then."""
    from xorl_amd import _C

    M, N, K = 8192, 2048, 1280
    m, _ = make_dense_module("int4", N, K, 16, 32, seed=3, device=hip_device)
    x = gen((M, K), 1.0, 4, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        want = m(x)
    got = torch.empty_like(want)
    L, w = _C.lib(), m._quant_weight().c()
    assert L.xq_linear_workspace_bytes(M, N, K, 16) > 2 * N * K
    _C.check(L.xq_linear_fwd_static(ctypes.byref(w), x.data_ptr(), K, M, m.lora_A.data_ptr(), m.lora_B.data_ptr(), _C.XQ_DT_F32, 16, m.scaling, None,
                                    got.data_ptr(), N, _C.stream_ptr(hip_device)))
    assert R.max_rel_err(got.float().cpu(), want.double().cpu()) <= 1e-2
