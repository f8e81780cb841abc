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
    (1, 300, 40, 1, 256),     # the deepest product with one filter per channel (backward in fp32 arithmetic on fp32 and f16
                              # tensors: vector kernels)
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


def _taps_form(u, taps, step):
    """Sum over lags of taps[lag] * u[t - step * lag] in 64 bits, zero outside the sequence: where a term is infinite or NaN
    the sum is, and nowhere else."""
    out, L = torch.zeros_like(u), u.shape[1]
    for lag in range(taps.shape[1]):
        past = torch.zeros_like(u)
        if step > 0:
            past[:, lag:] = u[:, :max(L - lag, 0)]
        else:
            past[:, :max(L - lag, 0)] = u[:, lag:]
        out += past * taps[:, lag].view(1, 1, -1, 1)
    return out


@pytest.mark.parametrize("types", list(TYPES))
@pytest.mark.parametrize("where", ["x", "dy", "h"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), "large"])
@pytest.mark.parametrize("bs,L,g,dg,hl", [(2, 300, 5, 3, 17), (1, 1500, 3, 10, 100), (1, 700, 20, 2, 256)])
def test_values_beyond_the_finite_range(gcg_lib, bs, L, g, dg, hl, value, where, types):
    """An infinity or NaN reaches the rows its taps reach and no other, as the kind it is in the tap-by-tap sum, and what
    stays finite is as exact as ever; the largest finite values give finite products."""
    dtype, filt = TYPES[types]
    gen = torch.Generator().manual_seed(hl)
    x, B, C, dy = (torch.randn(bs, L, g, dg, generator=gen).to(dtype) for _ in range(4))
    h = (torch.rand(g, 1, hl, generator=gen) / hl + 0.1 / hl).to(filt or dtype)
    if value == "large":
        value = torch.finfo((filt or dtype) if where == "h" else dtype).max
        B[:, L // 2], C[:, L // 2], C[:, L - 1] = 1, 1, 1            # (the sample itself is the large value)
        if where == "h":
            x, dy = x / 16, dy / 16
    t = {"x": x, "dy": dy, "h": h}[where]
    if where == "h":
        t[g // 2, 0, hl // 2] = value
    else:
        for b, row, c in ((0, L // 2, 1), (bs - 1, L - 1, 0)):
            t[b, row, g // 2, c] = value
    dev = [v.to(DEV) for v in (x, B, C, h)]
    bx, y2, y = _lib.fwd(*dev, return_bx=True, return_y2=True)
    dx, dB, dC, dh = _lib.bwd(dy.to(DEV), *dev)
    # the gated products are fp32 in the kernels: an infinite one may be a finite 64-bit value
    u, g2 = (x.float() * B.float()).double(), (dy.float() * C.float()).double()
    taps = h[:, 0].double().flip(-1)                                 # by lag
    ry2, rdu = _taps_form(u, taps, 1), _taps_form(g2, taps, -1)
    terms = [g2[:, lag:] * u[:, :max(L - lag, 0)] for lag in reversed(range(hl))]
    rdh = torch.stack([t.sum((0, 1, 3)) for t in terms], dim=1)
    most = torch.stack([t.abs().sum((0, 1, 3)) for t in terms], dim=1)    # (partial sums of dh may pass the limit where it does not)
    big = torch.finfo(torch.float32).max
    for name, got, ref in (("y2", y2, ry2), ("y", y, C.double() * ry2), ("dx", dx, B.double() * rdu), ("dB", dB, x.double() * rdu),
                           ("dC", dC, dy.double() * ry2), ("dh", dh[:, 0], rdh)):
        got, limit = got.cpu(), torch.finfo(got.dtype).max
        sure = ~((ref.abs() > limit / 4) & (ref.abs() < 4 * big))        # (around the type's limit either is right)
        if name == "dh":
            sure &= ~(most.isfinite() & (most > big / 4))
        ref = torch.where(ref.abs() > limit, ref * float("inf"), ref)
        fin = ref.isfinite()
        assert torch.equal(got.isfinite()[sure], fin[sure]), name
        if name != "dh":                                                 # (its order of summation decides between inf and NaN)
            kind = sure & ~fin
            assert torch.equal(got[kind].isnan(), ref[kind].isnan()), name
            assert torch.equal(got[kind].double().nan_to_num(0, 1, -1), ref[kind].nan_to_num(0, 1, -1)), name
        small = fin & (ref.abs() < 1e4) & got.isfinite()
        assert_close(got[small], ref[small], BAR[got.dtype], name)


@pytest.mark.parametrize("types", ["f32", "bf16"])
@pytest.mark.parametrize("bs,L,g,dg,hl", [(36, 4, 52, 54, 246), (6, 5, 653, 12, 255), (84, 20, 64, 32, 256)])
def test_backward_in_several_launches(gcg_lib, bs, L, g, dg, hl, types):
    """Batches launched in parts so that the sums of dh fit the static scratch: as exact as in one launch, with the same
    bits from the static scratch and from a workspace, and timed from the first launch to the end of the last."""
    dtype, filt = TYPES[types]
    gen = torch.Generator().manual_seed(hl)
    x, B, C, dy = (torch.randn(bs, L, g, dg, generator=gen).to(dtype) for _ in range(4))
    h = (torch.randn(g, 1, hl, generator=gen) / hl ** 0.5).to(filt or dtype)
    dev = [t.to(DEV) for t in (dy, x, B, C, h)]
    start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    start.record(), stop.record()                    # (creates them)
    got = _lib.bwd(*dev)
    torch.cuda.synchronize()
    _lib.time_next_kernel(start.cuda_event, stop.cuda_event)
    again = [torch.full_like(t, float("nan")) for t in got]
    _lib.bwd_static(*dev, *again)
    torch.cuda.synchronize()
    assert 0 < start.elapsed_time(stop) < 1000
    for a, b in zip(got, again):
        assert torch.equal(a, b)
    for o, r, n in zip(got, oracle_bwd(dy, x, B, C, h), ("dx", "dB", "dC", "dh")):
        assert_close(o, r, TOL_DH[dtype] if n == "dh" else BAR[dtype], n)


@pytest.mark.parametrize("types,which", [("f32", "x"), ("bf16w", "x"), ("f32", "h"), ("bf16w", "h")])
def test_values_near_the_smallest_normal_one(gcg_lib, types, which):
    """Gated products or taps around 2^-122 keep the bits that larger ones have, through all planes of the split."""
    bs, L, g, dg, hl = 1, 1000, 8, 6, 64
    dtype, filt = TYPES[types]
    gen = torch.Generator().manual_seed(8)
    x, B, C, dy = (torch.randn(bs, L, g, dg, generator=gen).to(dtype) for _ in range(4))
    h, up = torch.randn(g, 1, hl, generator=gen), 2.0 ** 122
    if which == "x":
        x = x / up
    else:
        h = h / up
    _, y2, y = _lib.fwd(*(t.to(DEV) for t in (x, B, C, h)), return_y2=True)
    dx, _, _, dh = _lib.bwd(*(t.to(DEV) for t in (dy, x, B, C, h)))
    u, taps = (x.float() * B.float()).double(), h[:, 0].double().flip(-1)
    g2 = (dy.float() * C.float()).double()
    ref, rdx = _taps_form(u, taps, 1), B.double() * _taps_form(g2, taps, -1)
    assert_close(y2.cpu().double() * up, ref * up, BAR[dtype], "y2")
    assert_close(y.cpu().double() * up, C.double() * ref * up, BAR[dtype], "y")
    if which == "h":
        assert_close(dx.cpu().double() * up, rdx * up, BAR[dtype], "dx")
    else:
        rdh = torch.stack([(g2[:, lag:] * u[:, :L - lag]).sum((0, 1, 3)) for lag in reversed(range(hl))], dim=1)
        assert_close(dh[:, 0].cpu().double() * up, rdh * up, TOL_DH[torch.float32], "dh")


@pytest.mark.parametrize("types", ["f32", "bf16w"])
def test_large_results_of_moderate_values(gcg_lib, types):
    """y2 and du of 2^85 and a filter gradient of 2^90 are beyond what the scaled products hold and within fp32."""
    bs, L, g, dg, hl = 1, 600, 3, 6, 40
    dtype, filt = TYPES[types]
    gen = torch.Generator().manual_seed(9)
    x, B, C, dy = (torch.randn(bs, L, g, dg, generator=gen).to(dtype) for _ in range(4))
    h = torch.randn(g, 1, hl, generator=gen) * 2.0 ** 45
    x, dy = x * 2.0 ** 40, dy * 2.0 ** 40
    _, y2, _ = _lib.fwd(*(t.to(DEV) for t in (x, B, C, h)), return_y2=True)
    dx, _, _, dh = _lib.bwd(*(t.to(DEV) for t in (dy, x, B, C, h)))
    u, g2, taps = (x.float() * B.float()).double(), (dy.float() * C.float()).double(), h[:, 0].double().flip(-1)
    assert_close(y2, _taps_form(u, taps, 1), BAR[dtype], "y2")
    assert_close(dx, B.double() * _taps_form(g2, taps, -1), BAR[dtype], "dx")
    rdh = torch.stack([(g2[:, lag:] * u[:, :L - lag]).sum((0, 1, 3)) for lag in reversed(range(hl))], dim=1)
    assert_close(dh[:, 0], rdh, TOL_DH[torch.float32], "dh")
