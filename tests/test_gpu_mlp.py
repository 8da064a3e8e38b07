"""GPU parity of the fused dense SwiGLU MLP (xq_mlp_fwd / xq_mlp_bwd through qlora_mlp_forward) against the float64
program of the oracle and against the three modules called one by one (same rounding points: the base products
are the same kernels' sums, so the two ways agree to bf16 rounding of reordered fp32 sums)."""

import pytest
import torch

from oracle import recipe as R
from tests.util_cases import close, dense_route, gate_up_joint, gen, make_dense_module

pytestmark = pytest.mark.gpu
TOL = 1e-2


def _mods(fmt, H, I, r, dev, bias=False, seed=0):
    mods, w_ref = {}, {}
    for i, (k, (N, K)) in enumerate({"gate": (I, H), "up": (I, H), "down": (H, I)}.items()):
        mods[k], w_ref[k] = make_dense_module(fmt, N, K, r, 2 * r, seed=seed + 10 * i, device=dev, bias=bias)
    return mods, w_ref


def _grads(mods):
    return {f"d{f}_{k}": getattr(m, f"lora_{f}").grad.clone() for k, m in mods.items() for f in ("A", "B")}


def _zero(mods):
    for m in mods.values():
        m.lora_A.grad = m.lora_B.grad = None


@pytest.mark.parametrize("tile_policy", [0, 1, 2], indirect=True)
@pytest.mark.parametrize("fmt,M,H,I,r", [
    ("block_fp8", 300, 256, 512, 16),      # fused gate/up/SwiGLU launch, fused dgrad (T = 128 tiles under policy 0)
    ("block_fp8", 1100, 512, 1024, 32),    # 2 rp = 64: both intermediates from one 64-row panel
    ("block_fp8", 130, 128, 192, 8),       # intermediate size not a multiple of 128: dgrads launch by launch
    ("block_fp8", 64, 256, 512, 40),       # 2 rp > 64: separate low-rank passes and dgrads
    ("nvfp4", 260, 256, 512, 16),          # 4-bit formats: the same program launch by launch
    ("int4", 200, 256, 384, 16),
    ("nf4", 200, 256, 384, 16),
])
def test_fused_mlp_vs_oracle_and_modules(hip_device, tile_policy, fmt, M, H, I, r):
    from xorl_amd.functional import silu_and_mul
    from xorl_amd.qlora import qlora_mlp_forward

    mods, w_ref = _mods(fmt, H, I, r, hip_device, seed=M)
    x = gen((M, H), 1.0, 71, torch.bfloat16)
    dy = gen((M, H), 1.0, 72, torch.bfloat16)
    loras = {k: (m.lora_A.detach().cpu(), m.lora_B.detach().cpu()) for k, m in mods.items()}
    ex = R.mlp_fwd_bwd_exact(x, w_ref["gate"], w_ref["up"], w_ref["down"], loras, mods["gate"].scaling, dy)

    xd = x.to(hip_device).requires_grad_(True)
    y = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], xd)
    y.backward(dy.to(hip_device))
    fused = {"y": y.detach().clone(), "dx": xd.grad.clone(), **_grads(mods)}
    close(fused["y"].cpu(), ex["y"], TOL)
    close(fused["dx"].cpu(), ex["dx"], TOL)
    for k in ("gate", "up", "down"):
        close(fused[f"dA_{k}"].cpu(), ex[f"dA_{k}"], TOL)
        close(fused[f"dB_{k}"].cpu(), ex[f"dB_{k}"], TOL)

    _zero(mods)
    xs = x.to(hip_device).requires_grad_(True)
    ys = mods["down"](silu_and_mul(mods["gate"](xs), mods["up"](xs)))
    ys.backward(dy.to(hip_device))
    sep = {"y": ys.detach(), "dx": xs.grad, **_grads(mods)}
    for name in fused:
        assert R.max_rel_err(fused[name].float().cpu(), sep[name].double().cpu()) <= 2 ** -7, name     # a bf16 step of the largest entry: dX is one rounded sum here, the sum of two rounded products there
    # a forward without grad (inference) gives the training forward's bits
    with torch.no_grad():
        assert torch.equal(qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], x.to(hip_device)), fused["y"])


@pytest.mark.parametrize("tile_policy", [0, 2], indirect=True)
@pytest.mark.parametrize("M,H,I,r,bias", [(300, 256, 512, 16, False), (1100, 512, 1024, 32, True), (2100, 512, 1536, 16, False)])
def test_gate_up_as_one_launch_or_two(hip_device, tile_policy, M, H, I, r, bias):
    """Block-fp8 gate and up as ONE launch with the SwiGLU in its epilogue, or as two launches followed by the pass that
    writes h and forms the down projection's low-rank intermediate (the default): same bits everywhere, and the
    one-launch form against the oracle."""
    from xorl_amd import _C
    from xorl_amd.qlora import qlora_mlp_forward

    mods, w_ref = _mods("block_fp8", H, I, r, hip_device, bias=bias, seed=M + 1)
    x = gen((M, H), 1.0, 81, torch.bfloat16)
    dy = gen((M, H), 1.0, 82, torch.bfloat16)
    got = {}
    try:
        # (the one-launch form lives in the tile kernel that all formats share: the bit-for-bit comparison keeps the two plain
        # launches on that kernel too; with the block-fp8 kernel of its own for them the sums run in another order)
        _C.check(_C.lib().xq_set_fp8_direct_tiles(0))
        for fused in (1, 0):
            _C.check(_C.lib().xq_set_mlp_gate_up_fused(fused))
            _zero(mods)
            xd = x.to(hip_device).requires_grad_(True)
            y = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], xd)
            y.backward(dy.to(hip_device))
            got[fused] = {"y": y.detach().clone(), "dx": xd.grad.clone(), **_grads(mods)}
        _C.check(_C.lib().xq_set_fp8_direct_tiles(1))
        _C.check(_C.lib().xq_set_mlp_gate_up_fused(0))
        _zero(mods)
        xd = x.to(hip_device).requires_grad_(True)
        y = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], xd)
        y.backward(dy.to(hip_device))
        direct = {"y": y.detach().clone(), "dx": xd.grad.clone(), **_grads(mods)}
    finally:
        _C.check(_C.lib().xq_set_mlp_gate_up_fused(0))
        _C.check(_C.lib().xq_set_fp8_direct_tiles(1))
    for name in got[0]:
        assert torch.equal(got[0][name], got[1][name]), name
        assert R.max_rel_err(direct[name].float().cpu(), got[0][name].double().cpu()) <= 2 ** -7, name     # same decoded operands, other summation order
    if bias:        # (the oracle's MLP program has no bias terms)
        return
    loras = {k: (m.lora_A.detach().cpu(), m.lora_B.detach().cpu()) for k, m in mods.items()}
    ex = R.mlp_fwd_bwd_exact(x, w_ref["gate"], w_ref["up"], w_ref["down"], loras, mods["gate"].scaling, dy)
    close(got[1]["y"].cpu(), ex["y"], TOL)
    close(got[1]["dx"].cpu(), ex["dx"], TOL)
    for k in ("gate", "up", "down"):
        close(got[1][f"dA_{k}"].cpu(), ex[f"dA_{k}"], TOL)
        close(got[1][f"dB_{k}"].cpu(), ex[f"dB_{k}"], TOL)


def test_fused_mlp_bias_no_lora_and_fallbacks(hip_device):
    from xorl_amd.qlora import qlora_mlp_forward

    H, I, M = 256, 512, 200
    mods, w_ref = _mods("block_fp8", H, I, 16, hip_device, bias=True, seed=3)
    x = gen((M, H), 1.0, 81, torch.bfloat16)
    dy = gen((M, H), 1.0, 82, torch.bfloat16)
    # biases on all three projections, against the float64 program
    Wg, Wu, Wd = (w_ref[k].double() for k in ("gate", "up", "down"))
    s = mods["gate"].scaling
    lin = lambda inp, W, m: inp @ W.t() + m.bias.detach().cpu().double() + s * ((inp @ m.lora_A.detach().cpu().double().t()) @ m.lora_B.detach().cpu().double().t())
    X = x.double()
    want = lin(torch.nn.functional.silu(lin(X, Wg, mods["gate"])) * lin(X, Wu, mods["up"]), Wd, mods["down"])
    with torch.no_grad():
        y = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], x.to(hip_device))
    close(y.cpu(), want, TOL)
    # frozen biases: the backward still returns dx and the factor gradients
    xd = x.to(hip_device).requires_grad_(True)
    qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], xd).backward(dy.to(hip_device))
    assert xd.grad is not None and mods["down"].lora_B.grad is not None
    # different active ranks: the helper calls the modules one by one and still agrees
    mods["up"].set_runtime_lora_config(8, 16)
    with torch.no_grad():
        y2 = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], x.to(hip_device))
    assert y2.shape == y.shape and bool(torch.isfinite(y2.float()).all())
    # empty batch
    with torch.no_grad():
        y0 = qlora_mlp_forward(mods["gate"], mods["down"].__class__(H, I, device=hip_device) if False else mods["up"], mods["down"],
                               torch.zeros(0, H, dtype=torch.bfloat16, device=hip_device))
    assert y0.shape == (0, H)


@pytest.mark.parametrize("backend", ["eager", "aot_eager"])
def test_fused_mlp_under_torch_compile(hip_device, backend):
    from xorl_amd.qlora import qlora_mlp_forward

    mods, _ = _mods("block_fp8", 256, 512, 16, hip_device, seed=9)
    x = gen((300, 256), 1.0, 91, torch.bfloat16).to(hip_device)
    dy = gen((300, 256), 1.0, 92, torch.bfloat16).to(hip_device)

    def run(fn):
        _zero(mods)
        xd = x.clone().requires_grad_(True)
        y = fn(mods["gate"], mods["up"], mods["down"], xd)
        y.backward(dy)
        return [y.detach().clone(), xd.grad.clone()] + list(_grads(mods).values())

    ref = run(qlora_mlp_forward)
    torch._dynamo.reset()
    got = run(torch.compile(qlora_mlp_forward, backend=backend, fullgraph=True))
    for a, b in zip(ref, got):
        assert torch.equal(a, b)


def test_gate_up_form_travels_with_the_saved_state(hip_device):
    """The form a forward ran gate and up in (one launch or two) fixes the layout of the saved low-rank intermediates;
    it travels to the backward in xq_mlp_saved, so flipping the process-wide default between a forward and its backward
    changes nothing: every gradient equals the undisturbed step's bit for bit, in both directions of the flip.  Between the two
    forms the bits are the same where the plain launches take the tile kernel of the joint one (xq_set_fp8_direct_tiles(0))."""
    from xorl_amd import _C
    from xorl_amd.qlora import qlora_mlp_forward

    M, H, I, r = 384, 512, 768, 16
    mods, _ = _mods("block_fp8", H, I, r, hip_device, bias=False, seed=77)
    x = gen((M, H), 1.0, 91, torch.bfloat16)
    dy = gen((M, H), 1.0, 92, torch.bfloat16)
    L = _C.lib()

    def step(fwd_mode, bwd_mode):
        _zero(mods)
        _C.check(L.xq_set_mlp_gate_up_fused(fwd_mode))
        xd = x.to(hip_device).requires_grad_(True)
        y = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], xd)
        _C.check(L.xq_set_mlp_gate_up_fused(bwd_mode))
        y.backward(dy.to(hip_device))
        return {"y": y.detach().clone(), "dx": xd.grad.clone(), **_grads(mods)}

    def equal(a, b, what):
        for name in a:
            assert torch.equal(a[name], b[name]), (*what, name)

    try:
        two, one = step(0, 0), step(1, 1)
        equal(step(0, 1), two, (0, 1))
        equal(step(1, 0), one, (1, 0))
        # the forms themselves: to the bit where both run on the same tile kernel
        _C.check(L.xq_set_fp8_direct_tiles(0))
        base = step(0, 0)
        for fwd_mode, bwd_mode in ((0, 1), (1, 0), (1, 1)):
            equal(step(fwd_mode, bwd_mode), base, (fwd_mode, bwd_mode))
    finally:
        _C.check(L.xq_set_fp8_direct_tiles(1))
        _C.check(L.xq_set_mlp_gate_up_fused(0))


def test_mlp_backward_rejects_a_saved_state_without_its_form(hip_device):
    """xq_mlp_bwd takes the form from the struct the forward filled; a struct that does not say (negative) is an argument error."""
    import ctypes
    from xorl_amd import _C
    from xorl_amd import functional as F

    M, H, I, r = 128, 256, 256, 16
    mods, _ = _mods("block_fp8", H, I, r, hip_device, bias=False, seed=5)
    banks = tuple(mods[k]._forward_quant_weight() for k in ("gate", "up", "down"))
    factors = tuple(t.detach().contiguous() for k in ("gate", "up", "down") for t in (mods[k].lora_A, mods[k].lora_B))
    x = gen((M, H), 1.0, 3, torch.bfloat16).to(hip_device)
    y, saved = F._mlp_fwd_impl(x, factors, (None, None, None), banks, r, 2.0, 0)
    with pytest.raises(ValueError, match="gate_up_fused"):
        F._mlp_bwd_impl(torch.ones_like(y), x, saved, factors, banks, r, 2.0, True, -1)


@pytest.mark.parametrize("M,H,I,r,bias", [
    (129, 192, 9280, 8, True), (300, 448, 9280, 64, False),       # part of a round of the chip; ragged rows and columns, three and seven K-steps
    (2309, 256, 7232, 24, False),                                   # more than two rounds
])
def test_gate_and_up_share_a_launch(hip_device, M, H, I, r, bias):
    """Block-fp8 gate and up as one launch of 128 x 256 tiles: against the three modules, whose projections are launches of their own
    (one rounded output each: a bf16 step of the largest entry), and without a bias against the float64 program."""
    from xorl_amd.functional import silu_and_mul
    from xorl_amd.qlora import qlora_mlp_forward

    mods, w_ref = _mods("block_fp8", H, I, r, hip_device, bias=bias, seed=M)
    x = gen((M, H), 1.0, 91, torch.bfloat16)
    xd = x.to(hip_device)
    with torch.no_grad():
        y = qlora_mlp_forward(mods["gate"], mods["up"], mods["down"], xd)
        sep = mods["down"](silu_and_mul(mods["gate"](xd), mods["up"](xd)))
    assert R.max_rel_err(y.float().cpu(), sep.double().cpu()) <= 2 ** -7
    assert R.max_rel_err(y[M // 128 * 128:].float().cpu(), sep[M // 128 * 128:].double().cpu()) <= 2 ** -7
    if not bias:
        loras = {k: (m.lora_A.detach().cpu(), m.lora_B.detach().cpu()) for k, m in mods.items()}
        ex = R.mlp_fwd_bwd_exact(x, w_ref["gate"], w_ref["up"], w_ref["down"], loras, mods["gate"].scaling, torch.zeros(M, H, dtype=torch.bfloat16))
        close(y.cpu(), ex["y"], TOL)


def _by_itself(m, x, dy, route):
    """(y, dx) of a projection on the kernel of `route`: "mid" by size, 256 or 128 forced tiles, or (head, tail rows) on 256 and on 128"""
    from xorl_amd import _C

    got = []
    try:
        for policy in {"mid": (0,), 256: (2,), 128: (3,)}.get(route, (2, 3)):
            _C.check(_C.lib().xq_set_tile_policy(policy))
            xd = x.detach().clone().requires_grad_(True)
            y = m(xd)
            got.append((y.detach(), torch.autograd.grad(y, xd, dy)[0]))
    finally:
        _C.check(_C.lib().xq_set_tile_policy(0))
    return got[0] if len(got) == 1 else tuple(torch.cat([a[:route[0]], b[route[0]:]]) for a, b in zip(*got))


@pytest.mark.parametrize("M,H,I,r,fwd,bwd,joint,bias", [
    (129, 192, 9280, 8, 128, "mid", False, False), (300, 448, 9280, 64, "mid", "mid", False, False),
    (1500, 384, 13120, 32, (1024, 476), (1024, 476), False, False),      # whole rounds of large tiles, the other rows on small ones
    (1000, 320, 9280, 16, 256, 256, True, False), (1000, 320, 9280, 64, 256, 256, True, True), (2300, 256, 12352, 24, 256, 256, True, True),
])
def test_mlp_products_sum_as_by_themselves(hip_device, M, H, I, r, fwd, bwd, joint, bias):
    """Gate, up and the dgrad of down, joint launch or not, are the bits of the same products by themselves on the kernels that their sizes
    choose.  Behind them: an fp32 factor gradient of gate, against float64 sums of the bf16 values that those bits give (fp32 sums
    of M products err by some sqrt(M) 2^-24; a flipped bf16 rounding in one value of a few hundred is 1e-4)."""
    from xorl_amd import functional as F
    from xorl_amd.qlora import qlora_mlp_forward

    for route, forward, n, k in ((fwd, True, I, H), (bwd, False, I, H)):
        here = dense_route("block_fp8", forward, M, n, k)
        # (a product by itself whose rows would be two launches, the second of small tiles, is free to be one of half tiles)
        assert here[0] == "mid" if route == "mid" else here[:3] == ("tiles", 128, 256) if isinstance(route, tuple) else here == ("tiles", route, route, 1, 0, 0, 0)
    assert gate_up_joint(M, H, I) == joint
    mods, w_ref = _mods("block_fp8", H, I, r, hip_device, bias=bias, seed=M)
    x, dy = gen((M, H), 1.0, 95, torch.bfloat16).to(hip_device), gen((M, H), 1.0, 96, torch.bfloat16).to(hip_device)
    m3 = [mods[k] for k in ("gate", "up", "down")]
    factors = [t.detach() for m in m3 for t in (m.lora_A, m.lora_B)]
    _, saved = F._mlp_fwd_impl(x, factors, [m.bias.detach().to(torch.bfloat16) if bias else None for m in m3], [m._quant_weight() for m in m3], r, m3[0].scaling, 0)
    zero = torch.zeros(M, I, dtype=torch.bfloat16, device=hip_device)
    g, u = (_by_itself(m, x, zero, fwd)[0] for m in m3[:2])
    assert torch.equal(saved[0], torch.cat([g, u], 1))
    # the backward
    xd = x.clone().requires_grad_(True)
    y = qlora_mlp_forward(*m3, xd)
    dB = torch.autograd.grad(y, m3[0].lora_B, dy)[0]
    dh = _by_itself(m3[2], saved[1], dy, bwd)[1]
    g.requires_grad_(True)
    dg = torch.autograd.grad(F.silu_and_mul(g, u), g, dh)[0]
    rp = saved[2].shape[1] // 2
    want = dg.double().t() @ saved[2].flatten()[:M * rp].view(M, rp)[:, :r].double()
    assert float((dB.double() - want).norm() / want.norm()) <= 2e-5
    if joint and not bias:
        loras = {k: (m.lora_A.detach().cpu(), m.lora_B.detach().cpu()) for k, m in mods.items()}
        ex = R.mlp_fwd_bwd_exact(x.cpu(), w_ref["gate"], w_ref["up"], w_ref["down"], loras, m3[0].scaling, dy.cpu())
        close(y.detach().cpu(), ex["y"], TOL)
        close(dB.cpu(), ex["dB_gate"], TOL)
