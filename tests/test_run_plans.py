"""How the matrix-core backward cuts a sequence into runs, seen through the scratch its partial sums need."""
import pytest

from savanna_amd import _lib

STATIC = _lib.STATIC_SCRATCH_BYTES


def scratch(bs, L, g, hl):
    return _lib.load().gcg_bwd_workspace_bytes(bs, L, g, 16, hl, _lib.GCG_BF16, _lib.ALGO_MFMA)


@pytest.mark.parametrize("bs,nsteps,hl", [(854, 75, 9), (858, 75, 9), (1023, 31, 9), (257, 63, 128), (769, 63, 33),
                                          (255, 300, 9), (300, 129, 64)])
def test_static_scratch_holds_what_it_held(bs, nsteps, hl):
    """Columns of 64 channels: launches that fill the chip with runs of 16 steps are not cut further."""
    assert 0 < scratch(bs, 32 * nsteps, 4, hl) <= STATIC


@pytest.mark.parametrize("cols", [1, 3, 64, 100, 255])
@pytest.mark.parametrize("hl", [9, 128])
def test_small_launches_stay_far_below_it(cols, hl):
    for nsteps in (1, 7, 16, 31, 75, 200):
        assert 0 < scratch(cols, 32 * nsteps, 4, hl) <= 2304 * 2048 + 4096
