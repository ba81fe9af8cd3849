"""Read-backs into ordinary host memory at the sizes where their path changes: a few words, one chunk,
the first size copied out by several threads, whole and broken chunks, more chunks than the pinned
ring holds, and several handles reading at once (one of them has the ring)."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import cugip_amd
from tests.gpu_util import say

pytestmark = pytest.mark.gpu

CHUNK = (4 << 20) // 4  # int32 voxels of one chunk
THREADED = (3 << 19) // 4


def random_grid(nx, ny, seed):
    rng = np.random.default_rng(seed)
    cs, ct = (rng.integers(0, 1 << 20, (1, ny, nx)).astype(np.int32) for _ in range(2))
    return cs, ct, rng.integers(0, 1 << 20, (3, 1, ny, nx)).astype(np.int32)


def readback(nx, ny, seed, repeats=1):
    cs, ct, cn = random_grid(nx, ny, seed)
    with cugip_amd.GridGraph() as g:
        g.set_grid(cs, ct, cn)
        for _ in range(repeats):
            a, b, c, d = g.capacities()
            assert np.array_equal(a, cs) and np.array_equal(b, ct) and np.array_equal(c, cn) and np.array_equal(d, cn)
    return True


@pytest.mark.parametrize("n", [1, 256, 257, THREADED - 1, THREADED, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK + 5,
                               5 * CHUNK + 77])
def test_readback_sizes(n):
    say(f"read-back of {n} words")
    assert readback(n, 1, n)


def test_readback_of_several_handles_at_once():
    say("read-backs of several handles at once")
    with ThreadPoolExecutor(max_workers=6) as pool:
        assert all(pool.map(lambda i: readback(1000 + i, 1500, i, 5), range(6)))
