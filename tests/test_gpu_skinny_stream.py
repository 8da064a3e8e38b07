"""GPU parity of the streaming skinny forward (M <= 64, two launches): joint forwards give the bits of the separate ones,
and the gate + up launch whose epilogue writes h = SwiGLU gives the MLP of the oracle."""

import pytest
import torch

from oracle import recipe as R
from tests.util_cases import close, gen, make_dense_module, skinny_route

pytestmark = pytest.mark.gpu


@pytest.fixture
def stream_only(hip_device):
    """the two-launch organisation at every M"""
    from xorl_amd._C import lib
    lib().xq_set_skinny_one_launch(0)
    yield
    lib().xq_set_skinny_one_launch(1)


@pytest.mark.parametrize("M", [1, 3, 16, 17, 33, 64])
@pytest.mark.parametrize("fmt,H,I,r", [
    ("int4", 1152, 1152, 16),      # 9 steps of 128: uneven splits
    ("nvfp4", 2944, 1088, 40),     # 68 row tiles: an uneven row block, a cut column block; ranks in three units of 16, the last one cut
    ("block_fp8", 1024, 1280, 64), # the widest low-rank term
    ("nf4", 1024, 1536, 1),
])
def test_joint_launches(stream_only, hip_device, fmt, H, I, r, M):
    from xorl_amd.functional import silu_and_mul
    from xorl_amd.qlora import qlora_linears_forward, qlora_mlp_forward

    bias = fmt in ("int4", "nf4")
    mods, w_ref = {}, {}
    for i, (k, (N, K)) in enumerate({"gate": (I, H), "up": (I, H), "down": (H, I)}.items()):
        mods[k], w_ref[k] = make_dense_module(fmt, N, K, r, 2 * r, seed=M + 10 * i, device=hip_device, bias=bias)
    g, u, d = mods["gate"], mods["up"], mods["down"]
    x = gen((M, H), 1.0, 71, torch.bfloat16)
    xd = x.to(hip_device)
    with torch.no_grad():
        yg, yu = g(xd), u(xd)
        for a, b in zip(qlora_linears_forward([g, u], xd), (yg, yu)):
            assert torch.equal(a, b)
        y = qlora_mlp_forward(g, u, d, xd)
        assert torch.equal(qlora_mlp_forward(g, u, d, xd), y)
        ref = d(silu_and_mul(yg, yu))
    close(y.cpu(), ref.cpu().double(), 1e-2)
    if not bias:
        loras = {k: (m.lora_A.detach().cpu(), m.lora_B.detach().cpu()) for k, m in mods.items()}
        ex = R.mlp_fwd_bwd_exact(x, w_ref["gate"], w_ref["up"], w_ref["down"], loras, g.scaling, torch.zeros(M, H, dtype=torch.bfloat16))
        close(y.cpu(), ex["y"], 1e-2)


@pytest.mark.parametrize("fmt,M,K", [("int4", 33, 65664), ("nvfp4", 64, 66560), ("block_fp8", 17, 131200), ("nf4", 2, 262272)])
def test_a_contraction_of_more_than_64_splits(hip_device, fmt, M, K):
    m, w_ref = make_dense_module(fmt, 64, K, 16, 32, seed=M, device=hip_device)
    x = gen((M, K), 1.0, 72, torch.bfloat16)
    with torch.no_grad():
        y = m(x.to(hip_device))
    ex = R.linear_fwd_bwd_exact(x, w_ref, m.lora_A.detach().cpu(), m.lora_B.detach().cpu(), m.scaling, torch.zeros(M, 64, dtype=torch.bfloat16))
    close(y.cpu(), ex["y"], 1e-2)


@pytest.mark.parametrize("fmt,name,off", [("nvfp4", "weight_block_scales", 1), ("nf4", "weight_scales", 4), ("int4", "weight_scales", 2),
                                          ("block_fp8", "weight_block_scales", 4)])
@pytest.mark.parametrize("M,K", [(1, 1152), (1, 2048), (4, 1152), (4, 2048), (20, 1152), (64, 1152)])     # 2048: the one-launch kernels
def test_scales_at_their_elements_alignment(hip_device, fmt, name, off, M, K):
    """Scales that start anywhere an element may (a view into a larger buffer) are read where they are."""
    m, _ = make_dense_module(fmt, 512, K, 16, 32, seed=M, device=hip_device)
    x = gen((M, K), 1.0, 73, torch.bfloat16).to(hip_device)
    with torch.no_grad():
        want = m(x)
        s = getattr(m, name)
        flat = torch.zeros(s.numel() + 16, dtype=torch.uint8, device=hip_device)
        moved = flat[off:off + s.numel()].view(s.shape)
        moved.copy_(s)
        setattr(m, name, moved)
        assert moved.data_ptr() % 8 == off and torch.equal(m(x), want)


def test_fp32_nvfp4_scales_at_four_bytes(hip_device):
    """(sources merged at load keep fp32 block scales)"""
    m, _ = make_dense_module("nvfp4", 512, 1152, 16, 32, seed=3, device=hip_device)
    s = m.weight_block_scales.view(torch.float8_e4m3fn).float().view(torch.uint8).reshape(512, -1)
    m._scale_dtypes["weight_block_scales"] = torch.float32
    flat = torch.zeros(s.numel() + 16, dtype=torch.uint8, device=hip_device)
    for M in (4, 40):
        x = gen((M, 1152), 1.0, 74, torch.bfloat16).to(hip_device)
        with torch.no_grad():
            m.weight_block_scales = s
            want = m(x)
            m.weight_block_scales = flat[4:4 + s.numel()].view(s.shape)
            m.weight_block_scales.copy_(s)
            assert torch.equal(m(x), want)


@pytest.mark.parametrize("fmt,N,K,r,Ms", [
    ("int4", 16, 1152, 64, (17, 64)),            # one row tile, four rank tiles: blocks that only form a low-rank part; an odd last step
    ("nf4", 48, 1024, 40, (20, 49)),             # fewer steps than waves once K is split
    ("int4", 12288, 5248, 16, (33, 64)),         # six and five steps a wave: a second window of scales, odd ranges, six row tiles
    ("nvfp4", 12320, 5248, 24, (48, 64)),        # the same with byte scales; a last row block that is partly past the end
    ("block_fp8", 12288, 4096, 16, (32, 64)),    # several half steps of x in flight, and one
    ("nvfp4", 24560, 1152, 16, (64,)),           # six row tiles, the last block's past the end
    ("nf4", 7824, 2944, 64, (24, 56)),           # 23 steps: three and two a wave; rows of x that end inside eight
])
def test_waves_that_split_the_contraction(hip_device, fmt, N, K, r, Ms):
    m, w_ref = make_dense_module(fmt, N, K, r, 2 * r, seed=N + K, device=hip_device)
    A, B = m.lora_A.detach().cpu(), m.lora_B.detach().cpu()
    for M in Ms:
        wide = gen((M, K + 64), 1.0, M, torch.bfloat16)           # rows that do not follow each other
        with torch.no_grad():
            y = m(wide.to(hip_device)[:, :K])
            assert torch.equal(m(wide[:, :K].contiguous().to(hip_device)), y)
        ex = R.linear_fwd_bwd_exact(wide[:, :K].contiguous(), w_ref, A, B, m.scaling, torch.zeros(M, N, dtype=torch.bfloat16))
        close(y.cpu(), ex["y"], 1e-2)                             # (the bound of every forward above)


@pytest.mark.parametrize("K", [1152, 2048])                       # a depth of the streaming kernels and one of the one-launch kernels
def test_rows_of_x_a_gigabyte_apart(hip_device, K):
    """Eight rows 2^29 elements apart (32-bit offsets of the rows would repeat every four): the packed copy's result."""
    m, w_ref = make_dense_module("int4", 512, K, 16, 32, seed=K, device=hip_device)
    g, u = (make_dense_module("int4", 1024, K, 16, 32, seed=s, device=hip_device)[0] for s in (5, 6))
    d = make_dense_module("int4", K, 1024, 16, 32, seed=7, device=hip_device)[0]
    from xorl_amd.qlora import qlora_linears_forward, qlora_mlp_forward

    x = gen((8, K), 1.0, 75, torch.bfloat16)
    pitch = 1 << 29
    far = torch.empty(7 * pitch + K, dtype=torch.bfloat16, device=hip_device).as_strided((8, K), (pitch, 1))
    far.copy_(x.to(hip_device))
    for M in (1, 2, 3, 8):
        with torch.no_grad():
            packed = x[:M].to(hip_device)
            close(m(far[:M]).cpu(), R.linear_fwd_bwd_exact(x[:M], w_ref, m.lora_A.detach().cpu(), m.lora_B.detach().cpu(), m.scaling,
                                                           torch.zeros(M, 512, dtype=torch.bfloat16))["y"], 1e-2)
            for a, b in zip(qlora_linears_forward([g, u], far[:M]), qlora_linears_forward([g, u], packed)):
                close(a.cpu(), b.cpu().double(), 1e-2)
            close(qlora_mlp_forward(g, u, d, far[:M]).cpu(), qlora_mlp_forward(g, u, d, packed).cpu().double(), 1e-2)


@pytest.mark.parametrize("fmt,N,K,tiles", [                       # rows of x: the plan's row tiles
    ("int4", 6272, 5120, {33: 5, 49: 5}),
    ("int4", 8320, 5120, {17: 7, 33: 7}),
    ("int4", 28800, 1024, {17: 8}),
    ("nf4", 16512, 2944, {3: 5}),                                 # the nf4 levels beside odd numbers of tiles
    ("nf4", 16512, 1024, {17: 5}),
    ("nf4", 6272, 5120, {33: 5, 49: 5}),
    ("nf4", 8320, 5120, {17: 7}),
    ("nf4", 28800, 1024, {3: 8}),
    ("block_fp8", 27648, 2944, {17: 7}),                          # an odd number of steps
])
def test_five_seven_and_eight_row_tiles(hip_device, fmt, N, K, tiles):
    m, w_ref = make_dense_module(fmt, N, K, 24, 48, seed=N + K, device=hip_device)
    A, B = m.lora_A.detach().cpu(), m.lora_B.detach().cpu()
    for M, rt in tiles.items():
        assert skinny_route(fmt, N, K, M, K, r=24)[2] == rt
        x = gen((M, K), 1.0, M, torch.bfloat16)
        with torch.no_grad():
            y = m(x.to(hip_device))
        ex = R.linear_fwd_bwd_exact(x, w_ref, A, B, m.scaling, torch.zeros(M, N, dtype=torch.bfloat16))
        close(y.cpu(), ex["y"], 1e-2)                             # (the bound of every forward above)
