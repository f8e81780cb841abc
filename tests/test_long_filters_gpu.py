"""The vector kernels (gcg_direct.hip) beyond 256 taps, where nothing else runs: the second and later passes over the taps
of the forward (128 a pass) and of the backward (32), filters longer than the sequence, and a last block of one tap.

Bars: nothing is rounded between load and store, so a 16-bit output is off by at most half a unit in the last place of
the largest value (2^-8 / 2^-11 of it) and fp32 outputs meet the fp32 bar."""
import pytest
import torch

from helpers import TOL_DH, assert_close, oracle_bwd, oracle_fwd
from savanna_amd import _lib
from test_general_shapes_gpu import BAR, TYPES

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
SHAPES = [                    # bs, L, g, dg, hl
    (1, 700, 3, 16, 257),
    (2, 333, 5, 7, 300),      # odd groups across the blocks of 64 channels, a ragged last tile
    (1, 1100, 2, 33, 513),
    (1, 100, 9, 1, 300),      # longer than the sequence
    (1, 1, 2, 24, 400),
    (3, 65, 1, 80, 385),      # one row past a tile, a group wider than a block
]


@pytest.mark.parametrize("types", list(TYPES))
@pytest.mark.parametrize("bs,L,g,dg,hl", SHAPES)
def test_fwd_bwd(gcg_lib, bs, L, g, dg, hl, types):
    dtype, filt = TYPES[types]
    gen = torch.Generator().manual_seed(hl + L)
    x, B, C, dy = (torch.randn(bs, L, g, dg, generator=gen).to(dtype) for _ in range(4))
    h = (torch.randn(g, 1, hl, generator=gen) / hl ** 0.5).to(filt or dtype)
    assert _lib.select_algo(bs, L, g, dg, hl, dtype) == "direct"
    dev = [t.to(DEV) for t in (x, B, C, h)]
    got = _lib.fwd(*dev, return_bx=True, return_y2=True)
    grads = _lib.bwd(dy.to(DEV), *dev)
    for o, r, n in zip(got, oracle_fwd(x, B, C, h), ("Bx", "y2", "y")):
        assert_close(o, r, BAR[dtype], n)
    ref = oracle_bwd(dy, x, B, C, h)
    for o, r, n in zip(grads, ref, ("dx", "dB", "dC")):
        assert_close(o, r, BAR[dtype], n)
    assert_close(grads[3], ref[3], TOL_DH[torch.float32] if grads[3].dtype == torch.float32 else BAR[dtype], "dh")


@pytest.mark.parametrize("layout", ["interleaved", "planar"])
@pytest.mark.parametrize("bs,L,g,dg,hl", [(2, 300, 7, 3, 257), (1, 600, 3, 20, 400)])
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
