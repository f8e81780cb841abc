"""The matrix-core kernels of the general family (groups of any width, 9 to 256 taps, any element alignment) at the
edges of their tiles: lengths around a block of 16 rows, a tile of 256 and the filter's reach, filter lengths around
the depths of the product (17, 81, 145), group widths around the two channels of a wave and the 32 of a workgroup.

Bars: nothing is rounded between load and store, so a 16-bit output is off by at most half a unit in the last place
of the largest value (2^-8 / 2^-11 of it) and fp32 outputs meet the fp32 bar."""
import pytest
import torch

from helpers import TOL_DH, assert_close, oracle_bwd, oracle_fwd
from savanna_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BAR = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
TYPES = {"f32": (torch.float32, None), "bf16": (torch.bfloat16, None), "f16": (torch.float16, None),
         "bf16w": (torch.bfloat16, torch.float32), "f16w": (torch.float16, torch.float32)}
SHAPES = [                    # bs, L, g, dg, hl
    (1, 1, 3, 1, 9),
    (1, 15, 5, 3, 17),
    (2, 16, 2, 8, 18),
    (1, 257, 33, 1, 81),      # one channel per filter, a channel block and one more
    (1, 256, 3, 31, 82),
    (3, 700, 4, 9, 128),
    (1, 1500, 2, 24, 145),    # several tiles, reach longer than the first
    (2, 513, 5, 7, 146),
    (1, 1111, 1, 40, 241),
    (1, 900, 17, 2, 256),
    (1, 300, 40, 1, 256),     # the deepest product with one filter per channel (fp32 and f16: vector kernels)
]


@pytest.mark.parametrize("types", list(TYPES))
@pytest.mark.parametrize("bs,L,g,dg,hl", SHAPES)
def test_fwd_bwd(gcg_lib, bs, L, g, dg, hl, types):
    dtype, filt = TYPES[types]
    gen = torch.Generator().manual_seed(hl + L)
    x, B, C, dy = (torch.randn(bs, L, g, dg, generator=gen).to(dtype) for _ in range(4))
    h = (torch.randn(g, 1, hl, generator=gen) / hl ** 0.5).to(filt or dtype)
    dev = [t.to(DEV) for t in (x, B, C, h)]
    bx, y2, y = _lib.fwd(*dev, return_bx=True, return_y2=True)
    got = _lib.bwd(dy.to(DEV), *dev)
    again = _lib.bwd(dy.to(DEV), *dev)
    torch.cuda.synchronize()
    for o, r, n in zip((bx, y2, y), oracle_fwd(x, B, C, h), ("Bx", "y2", "y")):
        assert_close(o, r, BAR[dtype], n)
    ref = oracle_bwd(dy, x, B, C, h)
    for o, r, n in zip(got, ref, ("dx", "dB", "dC")):
        assert_close(o, r, BAR[dtype], n)
    assert_close(got[3], ref[3], TOL_DH[torch.float32] if got[3].dtype == torch.float32 else BAR[dtype], "dh")
    for a, b in zip(got, again):
        assert torch.equal(a, b)


@pytest.mark.parametrize("layout", ["interleaved", "planar"])
@pytest.mark.parametrize("bs,L,g,dg,hl", [(2, 300, 7, 3, 128), (1, 600, 3, 20, 200)])
def test_feature_layouts_give_the_same_bits(gcg_lib, bs, L, g, dg, hl, layout):
    gen = torch.Generator().manual_seed(5)
    x, B, C, dy = (torch.randn(bs, L, g, dg, generator=gen).to(torch.bfloat16).to(DEV) for _ in range(4))
    h = (torch.randn(g, 1, hl, generator=gen) / hl ** 0.5).to(torch.bfloat16).to(DEV)
    dim = -1 if layout == "interleaved" else 2
    feat = torch.stack([C, B, x], dim=dim).contiguous()
    fwd, bwd = ((_lib.fwd_interleaved, _lib.bwd_interleaved) if layout == "interleaved" else
                (_lib.fwd_planar, _lib.bwd_planar))
    assert torch.equal(fwd(feat, h), _lib.fwd(x, B, C, h)[2])
    dfeat, dh = bwd(dy, feat, h)
    dx, dB, dC, dh_s = _lib.bwd(dy, x, B, C, h)
    for a, b in zip(dfeat.unbind(dim), (dC, dB, dx)):
        assert torch.equal(a, b)
    assert torch.equal(dh, dh_s)


@pytest.mark.parametrize("types", ["f32", "bf16w", "f16w"])
@pytest.mark.parametrize("bs,L,g,dg,hl", [(1, 4096, 64, 8, 128), (4, 16384, 9, 14, 30), (1, 8192, 16, 32, 256), (2, 3000, 7, 5, 17)])
def test_filter_gradient_has_no_bias(gcg_lib, bs, L, g, dg, hl, types):
    """dh (kept in fp32) against its 64-bit sum.  A sum of P terms of random sign, added one after the other with rounding
    to nearest, is off by 2^-24 sqrt(P / 6) of its size; the bar is that for the vector kernels' P = 64-row partial sums,
    and 1.5 units for the roundings within them.  A rounding that always goes one way adds up like P instead."""
    dtype, filt = TYPES[types]
    gen = torch.Generator(device=DEV).manual_seed(hl)
    x, B, C, dy = (torch.randn(bs, L, g, dg, generator=gen, device=DEV).to(dtype) for _ in range(4))
    h = torch.randn(g, 1, hl, generator=gen, device=DEV).to(filt or dtype)
    dh = _lib.bwd(dy, x, B, C, h)[3][:, 0].double()
    u, g2 = x.double() * B.double(), dy.double() * C.double()
    exact = torch.stack([(g2[:, lag:] * u[:, :L - lag]).sum((0, 1, 3)) for lag in reversed(range(hl))], dim=1)
    assert (dh - exact).norm() <= 2.0 ** -24 * (1.5 + (bs * L / 64 / 6) ** 0.5) * exact.norm()
