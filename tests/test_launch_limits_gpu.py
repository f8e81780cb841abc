"""Launches of 2^32 work-items and more, of which the runtime would run what is left modulo 2^32: narrow tensors of very many rows
are walked in longer runs, and what no plan holds is refused."""
import pytest
import torch

from savanna_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _pieces(f, x, y, hl, n=2000):
    """Pieces of y against f on the same rows by themselves (a row depends on the hl - 1 before it)."""
    L = x.shape[1]
    for b in range(x.shape[0]):
        assert torch.equal(y[b:b + 1, :n], f(x[b:b + 1, :n].clone()))
        for t0 in (n, L // 2 + 5, L - n):
            part = f(x[b:b + 1, t0 - hl + 1:t0 + n].clone())
            assert torch.equal(y[b:b + 1, t0:t0 + n], part[:, hl - 1:])


def _tensor(rows, bs, copies):
    torch.cuda.empty_cache()
    need = (copies + 1) * rows * 8
    if torch.cuda.mem_get_info()[0] < need + (4 << 30):
        pytest.skip(f"needs {need >> 30} GiB of device memory")
    gen = torch.Generator(device=DEV).manual_seed(1)
    return torch.empty(bs, rows // bs, 1, 4, device=DEV, dtype=torch.bfloat16).normal_(generator=gen)


@pytest.mark.parametrize("interleaved", [False, True])
def test_window_forward(interleaved):
    """Rows of four channels off the 128-byte lines, beyond the last-level cache: runs of 16 rows would be 2^26 waves."""
    hl, bs = 3, 4
    h = torch.randn(1, 1, hl, device=DEV).to(torch.bfloat16)
    if interleaved:
        flat = _tensor(3 * ((1 << 30) + 4000), bs, 3)
        x = flat.view(bs, -1, 1, 4, 3)
        f = lambda t: _lib.fwd_interleaved(t, h)
    else:
        x = _tensor((1 << 30) + 4000, bs, 1)
        f = lambda t: _lib.fwd(t, t, t, h)[2]
    _pieces(f, x, f(x), hl)


def test_featurizer_forward():
    """Runs of 64 rows of four channels: 2^26 waves at 2^32 rows."""
    w = torch.randn(1, 1, 3, device=DEV).to(torch.bfloat16)
    x = _tensor((1 << 32) + 4096, 16, 1)
    f = lambda t: _lib.dwconv_fwd(t, w)
    _pieces(f, x, f(x), 3)


@pytest.mark.parametrize("hl", [3, 40])
def test_more_sequences_than_a_launch_holds(hl):
    bs = (1 << 26) + 8
    x = _tensor(bs, bs, 3)
    h = torch.randn(1, 1, hl, device=DEV).to(torch.bfloat16)
    with pytest.raises(RuntimeError, match="hipError 9"):          # hipErrorInvalidConfiguration
        _lib.fwd(x, x, x, h, algo="window" if hl <= 8 else "direct")
