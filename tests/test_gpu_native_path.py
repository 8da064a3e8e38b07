"""The compiled host path (csrc/xq_torch.cpp) against the Python path over the same library calls: the same bits, forward and
backward, for every module kind; calls it leaves to the Python path still work."""

import pytest
import torch

from tests.test_gpu_moe import _make_experts, _zipf_routing
from tests.util_cases import gen, make_dense_module

pytestmark = pytest.mark.gpu


class _Declines:
    """Stands in for the extension and leaves every call to the Python path."""

    def __getattr__(self, name):
        return lambda *a: None


@pytest.fixture
def both_paths(monkeypatch):
    import xorl_amd.moe_functional as MF
    import xorl_amd.qlora.linear as LIN
    import xorl_amd.qlora.moe_experts as EXP

    def run(fn):
        got = fn()
        with monkeypatch.context() as mp:
            for mod in (MF, LIN, EXP):
                mp.setattr(mod, "native", lambda: _Declines())
            want = fn()
        assert len(got) == len(want)
        for a, b in zip(got, want):
            assert a.dtype == b.dtype and torch.equal(a, b)
        return got

    return run


@pytest.mark.parametrize("fmt,bias", [("block_fp8", False), ("nvfp4", True), ("int4", False), ("nf4", True)])
@pytest.mark.parametrize("shape", [(1, 512), (2, 9, 512), (65, 512)])
def test_linear(hip_device, both_paths, fmt, bias, shape):
    m, _ = make_dense_module(fmt, 256, 512, 16, 32, 3, hip_device, bias=bias)
    x = gen(shape, 1.0, 4, torch.bfloat16).to(hip_device)
    dy = gen((*shape[:-1], 256), 1.0, 5, torch.bfloat16).to(hip_device)

    def infer():
        with torch.no_grad():
            return [m(x), m(x.transpose(0, -1).contiguous().transpose(0, -1))]      # a layout that needs a packed copy

    def train():
        xr = x.clone().requires_grad_(True)
        y = m(xr)
        return [y.detach(), *torch.autograd.grad(y, [xr, m.lora_A, m.lora_B], dy)]

    both_paths(infer)
    both_paths(train)


@pytest.mark.parametrize("fmt", ["block_fp8", "nvfp4"])
@pytest.mark.parametrize("M", [1, 33, 200])
def test_mlp_and_joint_linears(hip_device, both_paths, fmt, M):
    from xorl_amd.qlora import qlora_linears_forward, qlora_mlp_forward

    H, I = 512, 768
    mods = [make_dense_module(fmt, n, k, 8, 16, 11 + i, hip_device)[0] for i, (n, k) in enumerate(((I, H), (I, H), (H, I)))]
    x = gen((M, H), 1.0, 4, torch.bfloat16).to(hip_device)
    dy = gen((M, H), 1.0, 5, torch.bfloat16).to(hip_device)

    def infer():
        with torch.no_grad():
            return [qlora_mlp_forward(*mods, x), *qlora_linears_forward(mods[:2], x)]

    def train():
        xr = x.clone().requires_grad_(True)
        y = qlora_mlp_forward(*mods, xr)
        return [y.detach(), *torch.autograd.grad(y, [xr] + [p for m in mods for p in m.get_lora_parameters()], dy)]

    both_paths(infer)
    both_paths(train)


@pytest.mark.parametrize("fmt,hybrid,rw_dtype", [("block_fp8", False, torch.bfloat16), ("nvfp4", True, torch.float32), ("nf4", False, torch.float64)])
@pytest.mark.parametrize("T", [3, 300])
def test_experts(hip_device, both_paths, fmt, hybrid, rw_dtype, T):
    E, H, I, topk = 6, 256, 256, 2
    m, _ = _make_experts(fmt, E, H, I, 8, hybrid, 7, hip_device)
    rw, sel = _zipf_routing(T, E, topk, seed=2)
    rw, sel = rw.to(rw_dtype).to(hip_device), sel.long().to(hip_device)
    x = gen((T, H), 1.0, 4, torch.bfloat16).to(hip_device)
    dy = gen((T, H), 1.0, 5, torch.bfloat16).to(hip_device)

    def infer():
        with torch.no_grad():
            return [m(x, rw, sel)]

    def train():
        xr, rr = x.clone().requires_grad_(True), rw.clone().requires_grad_(True)
        y = m(xr, rr, sel)
        return [y.detach(), *torch.autograd.grad(y, [xr, rr, *m.get_lora_parameters()], dy)]

    both_paths(train)
    if T == 3:      # (the Python path reaches _moe_infer with its banks)
        import xorl_amd.moe_functional as MF

        got = infer()[0]
        with torch.no_grad():
            gA, gB = m._active_lora_views("gate_proj")
            uA, uB = m._active_lora_views("up_proj")
            dA, dB = m._active_lora_views("down_proj")
            want = MF.moe_experts_qlora_forward(E, rw, sel, x, m._bank("gate"), m._bank("up"), m._bank("down"), gA, gB, uA, uB, dA, dB,
                                                m._active_scaling())
        assert torch.equal(got, want)
    else:
        both_paths(infer)


def test_calls_left_to_the_python_path(hip_device):
    from xorl_amd import _C

    m, _ = make_dense_module("int4", 128, 256, 16, 32, 3, hip_device)
    x = gen((4, 256), 1.0, 4, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        full = m(x)
        m.set_runtime_lora_config(8, 16)                       # an active rank below the stored one
        part = m(x)
    assert full.shape == part.shape and not torch.equal(full, part)
    with pytest.raises(_C.XqError):
        m(x.float())
    with pytest.raises(_C.XqError):
        m(x[:, :128].contiguous())


def test_backward_reads_the_weight_where_it_is_then(hip_device):
    """Sharded training frees the packed bytes after a forward and gathers them again before its backward, elsewhere."""
    m, _ = make_dense_module("int4", 128, 256, 16, 32, 3, hip_device)
    x = gen((70, 256), 1.0, 4, torch.bfloat16).to(hip_device).requires_grad_(True)
    dy = gen((70, 128), 1.0, 5, torch.bfloat16).to(hip_device)
    want = torch.autograd.grad(m(x), [x, m.lora_A, m.lora_B], dy)
    y, y2, packed = m(x), m(x), m.packed_weight_f32
    copy, storage = packed.detach().clone(), packed.untyped_storage()
    nbytes = storage.nbytes()
    storage.resize_(0)
    other = torch.zeros_like(copy)                 # takes the block that was given back
    with pytest.raises(RuntimeError, match="freed or resized"):
        torch.autograd.grad(y2, [x, m.lora_A, m.lora_B], dy)
    storage.resize_(nbytes)
    assert packed.data_ptr() != other.data_ptr()
    with torch.no_grad():
        packed.copy_(copy)
    for a, b in zip(torch.autograd.grad(y, [x, m.lora_A, m.lora_B], dy), want):
        assert torch.equal(a, b)


def test_tangents_and_transforms_are_refused_as_before(hip_device):
    import torch.autograd.forward_ad as fwAD

    m, _ = make_dense_module("int4", 128, 256, 16, 32, 3, hip_device)
    x = gen((4, 256), 1.0, 4, torch.bfloat16).to(hip_device)
    with fwAD.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        m(fwAD.make_dual(x, torch.ones_like(x)))
    with pytest.raises(RuntimeError):
        torch.vmap(lambda s: m(x) * s)(torch.ones(2, device=hip_device))


def test_strided_activations_are_read_in_place(hip_device, both_paths):
    """A [B, S, K] slice of a wider last dimension: the bits of the packed copy, and not the memory of one, in either direction."""
    B, S, K, N = 2, 320, 4096, 128
    m, _ = make_dense_module("block_fp8", N, K, 16, 32, 3, hip_device)
    wide = gen((B, S, 2 * K), 1.0, 4, torch.bfloat16).to(hip_device)
    wide_dy = gen((B, S, 3 * N), 1.0, 5, torch.bfloat16).to(hip_device)
    x, dy = wide[..., K:], wide_dy[..., N:2 * N]

    def step(x, dy):
        xr = x.detach().requires_grad_(True)
        y = m(xr)
        return [y.detach(), *torch.autograd.grad(y, [xr, m.lora_A, m.lora_B], dy)]

    def infer(x):
        with torch.no_grad():
            return [m(x), m(x[:, :1]), m(x[:1, 3]), m(x[:, ::2])]

    def peak(fn, *args):
        # The autograd engine's device thread lets go of a finished pass's graph task, and with it of the gradients, a moment
        # after the caller has them.  Where it is late, `before` holds the last pass's results and the reading is too low by
        # them, never too high: the highest of several counts.  Bytes as requested: what the allocator rounds up depends on the
        # blocks that happen to be free.
        readings = []
        for _ in range(4):
            fn(*args)
            torch.cuda.synchronize()
            before = torch.cuda.memory_stats()["requested_bytes.all.current"]
            torch.cuda.reset_peak_memory_stats()
            fn(*args)
            torch.cuda.synchronize()
            readings.append(torch.cuda.memory_stats()["requested_bytes.all.peak"] - before)
        return max(readings)

    packed = x.contiguous(), dy.contiguous()
    for a, b in zip(both_paths(lambda: step(x, dy)), step(*packed)):
        assert torch.equal(a, b)
    for a, b in zip(both_paths(lambda: infer(x)), infer(packed[0])):
        assert torch.equal(a, b)
    assert peak(step, x, dy) == peak(step, *packed)
    assert peak(lambda t: m(t).detach(), x) == peak(lambda t: m(t).detach(), packed[0])
    # layouts that do need one: rows a varying pitch apart, a pitch that is no multiple of 16 bytes, rows that start off one
    odd = gen((B * S, K + 4), 1.0, 6, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        for t in (x.transpose(0, 1), wide[:, ::3, :K], odd[:, :K], wide[..., 4:K + 4]):
            for a, b in zip(both_paths(lambda: [m(t)]), [m(t.contiguous())]):
                assert torch.equal(a, b)


def test_overridden_methods_are_called(hip_device, monkeypatch):
    """What a subclass, an instance or a patched class puts in the place of the methods that the native path stands for runs, in the
    module call, the joint call and the MLP; a subclass that replaces nothing stays native."""
    from xorl_amd._native import native
    from xorl_amd.qlora import Int4QLoRALinear, qlora_linears_forward, qlora_mlp_forward

    def module(cls, seed, n=256, k=256):
        m, _ = make_dense_module("int4", n, k, 16, 32, seed, hip_device)
        m.__class__ = cls
        return m

    class Same(Int4QLoRALinear):
        def extra_repr(self):
            return "same"

    class NoUpdate(Int4QLoRALinear):
        def _active_scaling(self):
            return 0.0

    class Other(Int4QLoRALinear):
        def _forward_quant_weight(self):
            return self.other._quant_weight()

    class Held(Int4QLoRALinear):
        @property
        def lora_B(self):
            return self._parameters["lora_B"] * 0.0

    x = gen((4, 256), 1.0, 4, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        plain, other = module(Int4QLoRALinear, 3), module(Int4QLoRALinear, 5)
        want, base = plain(x), module(Int4QLoRALinear, 3)
        base.lora_B.zero_()
        base = base(x)
        assert not torch.equal(want, base)
        assert native().linear(module(Same, 3), x) is not None
        for cls in (NoUpdate, Held):
            m = module(cls, 3)
            assert torch.equal(m(x), base)
            assert torch.equal(qlora_linears_forward([m, m], x)[1], base)
            assert torch.equal(qlora_mlp_forward(plain, plain, m, x), qlora_mlp_forward(plain, plain, m.eval(), x))
            assert native().mlp(plain, plain, m, x) is None
        m = module(Other, 3)
        object.__setattr__(m, "other", other)
        copy = module(Int4QLoRALinear, 5)
        copy.lora_A.copy_(m.lora_A)
        copy.lora_B.copy_(m.lora_B)
        assert torch.equal(m(x), copy(x))
        m = module(Int4QLoRALinear, 3)
        m._active_scaling = lambda: 0.0
        assert torch.equal(m(x), base)
        with monkeypatch.context() as mp:
            mp.setattr(Int4QLoRALinear, "_active_scaling", lambda self: 0.0)
            assert torch.equal(plain(x), base)
        assert torch.equal(plain(x), want)

    e, _ = _make_experts("block_fp8", 4, 256, 256, 8, False, 7, hip_device)
    rw, sel = _zipf_routing(40, 4, 2, seed=2)
    rw, sel = rw.to(hip_device), sel.long().to(hip_device)
    x = gen((40, 256), 1.0, 4, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        want = e(x, rw, sel)
        e._active_scaling = lambda: 0.0
        got = e(x, rw, sel)
        assert native().moe(e, x, rw, sel, False) is None and not torch.equal(got, want)
        del e._active_scaling
        for p in e.get_lora_parameters():
            p.zero_()
        assert torch.equal(got, e(x, rw, sel))


def test_block_fp8_calls_take_no_memory_for_an_image(hip_device):
    """Below 6144 rows a block-fp8 weight is not decoded first: a module call's scratch stays below the decoded weight's size."""
    from xorl_amd.qlora import QLoRALinear

    M, N, K = 2048, 12288, 4096
    x = torch.randn(M, K, dtype=torch.bfloat16, device=hip_device)
    lin = torch.nn.Linear(K, N, bias=False, dtype=torch.bfloat16, device=hip_device)
    for fmt, image in (("block_fp8", False), ("int4", True)):
        m = QLoRALinear.from_module(lin, r=16, lora_alpha=32, quant_format=fmt)
        with torch.no_grad():
            y = m(x)
            torch.cuda.synchronize()
            del y
            before = torch.cuda.memory_allocated()
            torch.cuda.reset_peak_memory_stats()
            y = m(x)
            torch.cuda.synchronize()
        scratch = torch.cuda.max_memory_allocated() - before - y.numel() * 2
        assert (scratch >= 2 * N * K) == image, (fmt, scratch)
