"""Rows that do not start and end on 128-byte lines: the kernels' accesses of their own give the same bits.

The channels of a filter group do not depend on the groups beside it, so a narrow tensor's results are those of the same
channels inside a wider one whose rows are whole lines.
"""
import pytest
import torch

from savanna_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _pair(bs, L, g, wide, dg, dtype, gen, lead=(), tail=()):
    """A tensor of `wide` groups and its first `g` groups by themselves."""
    w = torch.randn(bs, L, *lead, wide, dg, *tail, generator=gen, device=DEV).to(dtype)
    return w, w.narrow(2 + len(lead), 0, g).contiguous()


@pytest.mark.parametrize("dtype,arith", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                         (torch.bfloat16, torch.float32), (torch.float16, torch.float32),
                                         (torch.float32, torch.float32)])
@pytest.mark.parametrize("hl", [2, 7, 20, 40, 70, 97, 128])
@pytest.mark.parametrize("g", [5, 6])
def test_separate_tensors(dtype, arith, hl, g):
    bs, L, wide, dg = 2, 333, 8, 16
    gen = torch.Generator(device=DEV).manual_seed(hl + g)
    ops = [_pair(bs, L, g, wide, dg, dtype, gen) for _ in range(4)]
    h = (torch.randn(wide, 1, hl, generator=gen, device=DEV) / hl ** 0.5).to(arith)
    (dyw, xw, Bw, Cw), (dyn, xn, Bn, Cn) = ([p[i] for p in ops] for i in (0, 1))
    assert torch.equal(_lib.fwd(xw, Bw, Cw, h)[2][..., :g, :], _lib.fwd(xn, Bn, Cn, h[:g].contiguous())[2])
    rw, rn = _lib.bwd(dyw, xw, Bw, Cw, h), _lib.bwd(dyn, xn, Bn, Cn, h[:g].contiguous())
    for a, b in zip(rw[:3], rn[:3]):
        assert torch.equal(a[..., :g, :], b)
    # dh: the same products, in sums that may be cut differently; one rounding to the filter's type
    eps = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11, torch.float32: 1e-5}[arith]
    assert (rw[3][:g].float() - rn[3].float()).abs().max() <= eps * rw[3].float().abs().max()


@pytest.mark.parametrize("dtype,arith", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32)])
@pytest.mark.parametrize("hl", [5, 128])
@pytest.mark.parametrize("g", [5, 6])
def test_planar_features(dtype, arith, hl, g):
    bs, L, wide, dg = 2, 333, 8, 16
    gen = torch.Generator(device=DEV).manual_seed(hl + g)
    fw, fn = _pair(bs, L, g, wide, dg, dtype, gen, lead=(3,))
    dyw, dyn = _pair(bs, L, g, wide, dg, dtype, gen)
    h = (torch.randn(wide, 1, hl, generator=gen, device=DEV) / hl ** 0.5).to(arith)
    assert torch.equal(_lib.fwd_planar(fw, h)[..., :g, :], _lib.fwd_planar(fn, h[:g].contiguous()))
    rw, rn = _lib.bwd_planar(dyw, fw, h), _lib.bwd_planar(dyn, fn, h[:g].contiguous())
    assert torch.equal(rw[0][..., :g, :], rn[0])


@pytest.mark.parametrize("dtype,arith", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("bs,L,g,wide", [(1, 700, 5, 8), (2, 3001, 29, 32), (3, 90, 54, 64), (1, 40000, 11, 16)])
@pytest.mark.parametrize("planar", [False, True])
def test_register_window_kernels(dtype, arith, bs, L, g, wide, planar):
    """Run lengths and workgroups of one to four waves, chosen by the width: operator on interleaved features, short mixer."""
    dg, hl = 16, 7
    gen = torch.Generator(device=DEV).manual_seed(L + g)
    lay = {"lead": (3,)} if planar else {"tail": (3,)}
    cut = (lambda t: t[..., :g, :]) if planar else (lambda t: t[:, :, :g])
    rw, rn = _pair(bs, L, g, wide, dg, dtype, gen, **lay)
    dyw, dyn = _pair(bs, L, g, wide, dg, dtype, gen)
    h = (torch.randn(wide, 1, hl, generator=gen, device=DEV) / hl ** 0.5).to(arith)
    hn = h[:g].contiguous()
    wf = torch.randn(3, wide, dg, 3, generator=gen, device=DEV).to(dtype) / 2
    wfw, wfn = ((t if planar else t.permute(1, 2, 0, 3)).reshape(-1, 1, 3).contiguous() for t in (wf, wf[:, :g]))
    if not planar:
        assert torch.equal(_lib.fwd_interleaved(rw, h)[:, :, :g], _lib.fwd_interleaved(rn, hn))
        assert torch.equal(cut(_lib.bwd_interleaved(dyw, rw, h)[0]), _lib.bwd_interleaved(dyn, rn, hn)[0])
    assert torch.equal(_lib.mixer_se_fwd(rw, wfw, h, planar)[:, :, :g], _lib.mixer_se_fwd(rn, wfn, hn, planar))
    a, b = _lib.mixer_se_bwd(dyw, rw, wfw, h, planar), _lib.mixer_se_bwd(dyn, rn, wfn, hn, planar)
    assert torch.equal(cut(a[0]), b[0])
    # filter gradients: the same fp32 products in sums that are cut differently (errors of sums grow like the root of
    # their terms, as the sums themselves do), one rounding to the filter's type
    ulp = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11, torch.float32: 1e-5}
    dwa = a[1].reshape(3, wide, dg, 3) if planar else a[1].reshape(wide, dg, 3, 3).permute(2, 0, 1, 3)
    dwb = b[1].reshape(3, g, dg, 3) if planar else b[1].reshape(g, dg, 3, 3).permute(2, 0, 1, 3)
    assert (dwa[:, :g].float() - dwb.float()).abs().max() <= ulp[dtype] * dwa.float().abs().max()
    assert (a[2][:g].float() - b[2].float()).abs().max() <= ulp[arith] * a[2].float().abs().max()


# layout, tensors' and filter's type, groups, taps, sequences
BEYOND = [("separate", "bfloat16", "bfloat16", 29, 7, 1), ("separate", "bfloat16", "float32", 29, 3, 2),
          ("separate", "float16", "float16", 27, 8, 1), ("separate", "float32", "float32", 31, 7, 1),
          ("separate", "float32", "float32", 256, 4, 2), ("interleaved", "float16", "float16", 64, 7, 2),
          ("extra", "bfloat16", "bfloat16", 29, 7, 2), ("extra", "float16", "float32", 27, 4, 1), ("extra", "float32", "float32", 31, 7, 1),
          ("interleaved", "float16", "float16", 61, 7, 1), ("interleaved", "bfloat16", "bfloat16", 28, 8, 2),
          ("interleaved", "float32", "float32", 30, 7, 1), ("interleaved", "float32", "float32", 31, 3, 2),
          ("time_major", "bfloat16", "bfloat16", 29, 7, 2), ("time_major", "float16", "float32", 29, 3, 3),
          ("planar", "float16", "float16", 27, 7, 1), ("planar", "bfloat16", "float32", 29, 8, 2)]


@pytest.mark.parametrize("layout,dtype,arith,g,hl,bs", BEYOND)
def test_window_forward_beyond_the_cache(layout, dtype, arith, g, hl, bs):
    """Tensors that together exceed the last-level cache are walked in another form; a row depends on the hl - 1 before it, so
    pieces of the result are those of the same rows by themselves.  (Pieces start at a multiple of eight rows: the walks are
    unrolled by eight, and an f16 y2 is converted from the sum or folded into its last step by the row's place among them.)"""
    dg, dtype = 16, getattr(torch, dtype)
    row = g * dg * dtype.itemsize
    L = (1 << 26) // (row * bs) + 1003
    gen = torch.Generator(device=DEV).manual_seed(g + hl)
    h = (torch.randn(g, 1, hl, generator=gen, device=DEV) / hl ** 0.5).to(getattr(torch, arith))
    shape = {"interleaved": (bs, L, g, dg, 3), "planar": (bs, L, 3, g, dg), "time_major": (L, bs, g, dg)}.get(layout, (bs, L, g, dg))
    time = 0 if layout == "time_major" else 1
    ops = [torch.empty(shape, device=DEV, dtype=dtype).normal_(generator=gen) for _ in range(1 if len(shape) == 5 else 3)]
    f = {"interleaved": lambda a: [_lib.fwd_interleaved(a[0], h)], "planar": lambda a: [_lib.fwd_planar(a[0], h)],
         "time_major": lambda a: [_lib.fwd_time_major(*a, h)], "separate": lambda a: [_lib.fwd(*a, h)[2]],
         "extra": lambda a: list(_lib.fwd(*a, h, return_bx=True, return_y2=True))}[layout]
    assert 4 * bs * L * row > 1 << 28
    ys = f(ops)
    n = min(4000, L // 4)
    for t0, t1 in ((0, n), (n, 2 * n), (L // 2 + 5, L // 2 + 5 + n), (L - n, L)):
        first = max(t0 - hl + 1, 0) // 8 * 8
        parts = f([t.narrow(time, first, t1 - first).clone() for t in ops])
        for y, part in zip(ys, parts):
            assert torch.equal(y[:, t0:t1], part[:, t0 - first:])
