"""xq_quantize against the torch quantizers on the CPU (checked byte for byte against the oracle in
tests/test_quantizers_cpu.py): codes, scales and global scale are the same bytes."""

import pytest
import torch

from xorl_amd import quantize as Q

pytestmark = pytest.mark.gpu


def _weight(shape, dtype, seed):
    """N(0, 0.02) with a zero group, values on code boundaries (multiples of an eighth of a block maximum of 6), magnitudes from
    denormal to huge, and signed zeros."""
    g = torch.Generator().manual_seed(seed)
    w = torch.randn(*shape, generator=g) * 0.02
    flat = w.view(-1)
    flat[:128] = 0.0
    n = min(flat.numel() - 128, 512)
    flat[128:128 + n] = torch.randint(-48, 49, (n,), generator=g) / 8.0
    if flat.numel() > 2048:
        flat[1024:1280] = torch.randn(256, generator=g) * 1e-20
        flat[1280:1536] = torch.randn(256, generator=g) * 1e4
        flat[1536:1600] = -0.0
    return w.to(dtype)


def _same(got, want):
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.shape == b.shape and a.is_cuda
        assert torch.equal(a.cpu().view(torch.uint8), b.view(torch.uint8))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(1, 128), (3, 640), (130, 896), (513, 4096)])
def test_flat(hip_device, dtype, shape):
    w = _weight(shape, dtype, 1)
    d = w.to(hip_device)
    for fn in (lambda x: Q.nf4_quantize(x), lambda x: Q.nvfp4_quantize(x), lambda x: Q.int4_quantize_sym(x, 128),
               lambda x: Q.int4_quantize(x, 128), lambda x: Q.int4_quantize(x, 32), lambda x: Q.block_fp8_quantize_gkn(x),
               lambda x: Q.block_fp8_quantize_gkn(x, amax_scale=1.25)):
        _same(fn(d), fn(w))
    _same(Q.nvfp4_quantize(d, global_amax=torch.tensor([0.2])), Q.nvfp4_quantize(w, global_amax=torch.tensor([0.2])))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(64, 8), (192, 136), (1024, 640), (2048, 768)])
def test_gkn(hip_device, dtype, shape):
    w = _weight(shape, dtype, 2)
    d = w.to(hip_device)
    for fn in (Q.nf4_quantize_gkn, Q.nvfp4_quantize_gkn, lambda x: Q.int4_quantize_gkn(x, 64), lambda x: Q.int4_quantize_gkn(x, 32)):
        _same(fn(d), fn(w))
    _same(Q.nvfp4_quantize_gkn(d, global_amax=torch.tensor([0.2])), Q.nvfp4_quantize_gkn(w, global_amax=torch.tensor([0.2])))


def test_edges_of_the_dispatch(hip_device):
    """Row counts that leave a 64-row tile partly empty, edge tiles of block fp8, and shapes that stay on torch ops."""
    w = _weight((80, 72), torch.float32, 3)
    d = w.to(hip_device)
    _same(Q.nvfp4_quantize_gkn(d), Q.nvfp4_quantize_gkn(w))
    _same(Q.block_fp8_quantize_gkn(d), Q.block_fp8_quantize_gkn(w))
    w = _weight((12, 100), torch.bfloat16, 4)
    d = w.to(hip_device)
    _same(Q.block_fp8_quantize_gkn(d), Q.block_fp8_quantize_gkn(w))          # columns not a multiple of 8
    _same(Q.int4_quantize(d, -1), Q.int4_quantize(w, -1))                    # a group that is no power of two
    w = _weight((1 << 12, 1 << 13), torch.bfloat16, 5)                        # more runs than the grid has threads
    d = w.to(hip_device)
    for fn in (Q.nvfp4_quantize, Q.nf4_quantize):
        _same(fn(d), fn(w))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("values", [(float("nan"),), (float("inf"), float("-inf")), (float("-inf"), float("nan"))])
def test_nan_and_infinity_stay_visible(hip_device, monkeypatch, dtype, values):
    """A damaged weight: the scales and codes of the torch forms on the same device.  (An e4m3 NaN counts as one whatever its sign.)"""
    w = _weight((192, 640), dtype, 6)
    w[7, 130], w[100, 3] = values[0], values[-1]
    d = w.to(hip_device)
    amax = torch.tensor([0.2])
    calls = [lambda: Q.nf4_quantize(d), lambda: Q.nvfp4_quantize(d), lambda: Q.nvfp4_quantize(d, global_amax=amax),
             lambda: Q.nvfp4_quantize(d, global_amax=amax * float("nan")), lambda: Q.int4_quantize_sym(d, 128),
             lambda: Q.int4_quantize(d, 128), lambda: Q.int4_quantize(d, 32), lambda: Q.block_fp8_quantize_gkn(d),
             lambda: Q.nf4_quantize_gkn(d), lambda: Q.nvfp4_quantize_gkn(d), lambda: Q.nvfp4_quantize_gkn(d, global_amax=amax),
             lambda: Q.int4_quantize_gkn(d, 64), lambda: Q.int4_quantize_gkn(d, 32)]
    got = [fn() for fn in calls]
    with monkeypatch.context() as mp:
        mp.setattr(torch.compiler, "is_compiling", lambda: True)          # leaves every call to the torch forms
        want = [fn() for fn in calls]
    for i, (a, b) in enumerate(zip(got, want)):
        assert any(not torch.isfinite(t.float()).all() for t in b) or i in (2, 10)      # a given amax: an infinite block saturates
        for s, t in zip(a, b):
            assert s.dtype == t.dtype and s.shape == t.shape, i
            if s.dtype == torch.uint8:
                assert torch.equal(s, t), i
            else:
                assert torch.equal(s.float().isnan(), t.float().isnan()), i
                assert torch.equal(s.float().nan_to_num(0.0, None, None), t.float().nan_to_num(0.0, None, None)), i
