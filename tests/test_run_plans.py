"""How the matrix-core backwards cut their work into runs and launches, seen through the scratch their partial sums need."""
import random
import time

import pytest

from savanna_amd import _lib

STATIC = _lib.STATIC_SCRATCH_BYTES


CODES = [_lib.GCG_F32, _lib.GCG_BF16, _lib.GCG_F16, _lib.GCG_BF16_F32, _lib.GCG_F16_F32]


def scratch(bs, L, g, hl):
    return _lib.load().gcg_bwd_workspace_bytes(bs, L, g, 16, hl, _lib.GCG_BF16, _lib.ALGO_MFMA)


def vector_scratch(bs, L, g, dg, hl):
    """The vector kernels': one slot of a filter for each that a block of 64 channels touches, runs of 64 rows or more."""
    blocks, tiles = (g * dg + 63) // 64, (L + 63) // 64
    tps = -(-tiles // min(max(4096 // (bs * blocks), 1), tiles))
    filters = 64 // dg if 64 % dg == 0 else min(63 // dg + 2, 64)
    return -(-bs * -(-tiles // tps) * blocks * filters * hl * 4 // 256) * 256


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


def test_register_window_backward_stays_in_static_scratch():
    """Runs cut to fill the SIMDs leave no more partial sums than 8 MiB hold, or than runs of a power of two up to 1024 rows
    that give 2^17 lanes work."""
    rng = random.Random(7)
    for _ in range(3000):
        bs, L, g = int(2 ** rng.uniform(0, 6)), int(2 ** rng.uniform(0, 18)), int(2 ** rng.uniform(0, 10))
        dg, hl = rng.choice([4, 8, 12, 16, 32, 64]), rng.randint(1, 8)
        most = 0
        for v in (1, 2, 4):
            ts = 1024
            while ts > 8 and bs * -(-L // ts) * (g * dg // v) < 1 << 17:
                ts >>= 1
            most = max(most, bs * -(-L // ts) * (g * dg // v))
        got = _lib.load().gcg_bwd_workspace_bytes(bs, L, g, dg, hl, _lib.GCG_BF16, _lib.ALGO_NAMES["window"])
        assert 0 < got <= max(STATIC, most * hl * 4 + 256), (bs, L, g, dg, hl)


@pytest.mark.parametrize("code", CODES)
@pytest.mark.parametrize("bs,L,g,dg,hl", [(21, 160, 256, 32, 256), (49, 1, 64, 24, 256), (6, 5, 653, 12, 255), (47, 189, 124, 63, 111),
                                          (22, 215, 147, 43, 226), (127, 1634, 839, 6, 15), (36, 4, 52, 54, 246),
                                          (1, 100, 8000, 64, 255), (3, 7, 2730, 64, 250)])
def test_general_family_stays_in_static_scratch(code, bs, L, g, dg, hl):
    """Where the vector kernels' sums fit it, those of the matrix-core kernels with their narrower blocks do too."""
    assert vector_scratch(bs, L, g, dg, hl) <= STATIC
    for algo in (_lib.ALGO_NAMES["direct"], _lib.ALGO_AUTO):
        assert 0 < _lib.load().gcg_bwd_workspace_bytes(bs, L, g, dg, hl, code, algo) <= STATIC


def test_launches_beyond_the_grid_stay_with_the_vector_kernels():
    """A launch holds 2^32 - 1 work-items.  65536 rows of 65 blocks in workgroups of 1024 are more: the vector kernels' 33
    blocks in workgroups of 256 are not."""
    size = lambda *s: _lib.load().gcg_bwd_workspace_bytes(*s, _lib.GCG_BF16, _lib.ALGO_NAMES["direct"])
    assert size(65536, 16, 86, 24, 64) == vector_scratch(65536, 16, 86, 24, 64)
    assert size(63000, 16, 86, 24, 64) != vector_scratch(63000, 16, 86, 24, 64)


def test_query_for_either_alignment_costs_no_search():
    """Under AUTO the query that every backward call makes also sizes for misaligned tensors; that takes a fraction of the
    call (0.16 us against 0.12 of its own at a million rows, where a search over all run lengths took 1.3)."""
    query = _lib.load().gcg_bwd_workspace_bytes

    def best(*args):
        times = []
        for _ in range(40):
            t = time.perf_counter()
            for _ in range(500):
                query(*args)
            times.append(time.perf_counter() - t)
        return min(times)

    shape = (1, 1 << 20, 256, 16, 128, _lib.GCG_BF16)
    assert best(*shape, _lib.ALGO_AUTO) < 1.6 * best(*shape, _lib.ALGO_MFMA)
