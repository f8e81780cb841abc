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
