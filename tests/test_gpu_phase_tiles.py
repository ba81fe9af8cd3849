"""Where a grid's size changes the launches. Discharge phases and sweeps on both sides of the tile count
up to which they take their colour class whole instead of a compacted list, host-driven and
(6-connected) device-driven: the flow equals the capacity of the cut it returns (integers, so the flow
is maximum), and both engines give the same. The init on both sides of the workgroup count that
decides how many z-levels a workgroup takes."""
import numpy as np
import pytest

import cugip_amd
from perf.cases import HALF
from tests.gpu_util import say

pytestmark = pytest.mark.gpu

LIMIT = 32768  # tiles


def cut_capacity(cs, ct, cn, inside, conn):
    total = int(cs[~inside].sum(dtype=np.int64)) + int(ct[inside].sum(dtype=np.int64))
    nz, ny, nx = cs.shape
    for j, (dx, dy, dz) in enumerate(HALF[conn]):
        here = tuple(slice(max(0, -o), n - max(0, o)) for o, n in ((dz, nz), (dy, ny), (dx, nx)))
        there = tuple(slice(max(0, o), n - max(0, -o)) for o, n in ((dz, nz), (dy, ny), (dx, nx)))
        total += int(cn[j][here][inside[here] != inside[there]].sum(dtype=np.int64))
    return total


@pytest.mark.parametrize("conn,tile,across", [(6, (16, 4, 4), 4), (26, (32, 4, 2), 4)])
@pytest.mark.parametrize("extra", [0, 1])
def test_phases_around_the_whole_colour_limit(conn, tile, across, extra):
    # 2 x 2 ragged tiles across, LIMIT / 4 (+ 1) along z
    nx, ny = tile[0] + 1, tile[1] + 1
    nz = (LIMIT // across + extra) * tile[2] - 1
    say(f"phases of {conn} connections, {LIMIT + across * extra} tiles")
    rng = np.random.default_rng(conn + extra)
    cs, ct = (np.maximum(rng.integers(-300, 200, (nz, ny, nx)), 0).astype(np.int32) for _ in range(2))
    cn = rng.integers(0, 60, (conn // 2, nz, ny, nx)).astype(np.int32)
    results = []
    for engine in (cugip_amd.ENGINE_TILES, cugip_amd.ENGINE_GRAPH)[:2 if conn == 6 else 1]:
        with cugip_amd.GridGraph() as g:
            g.set_grid(cs, ct, cn, conn=conn)
            g.set_policy(engine=engine, tile_x=tile[0], tile_y=tile[1], tile_z=tile[2])
            flow = g.max_flow()
            st = g.stats
            tiles = 1
            for n, t in ((nx, st.tile_x), (ny, st.tile_y), (nz, st.tile_z)):
                tiles *= -(-n // t)
            assert tiles == LIMIT + across * extra
            inside = g.source_set().reshape(cs.shape).astype(bool)
        assert flow == cut_capacity(cs, ct, cn, inside, conn)
        results.append((flow, inside))
    for flow, inside in results[1:]:
        assert flow == results[0][0] and np.array_equal(inside, results[0][1])


@pytest.mark.parametrize("conn", [6, 26])
@pytest.mark.parametrize("nz", [8 * 4095, 8 * 4095 + 1])
def test_init_around_the_deep_chunk_limit(conn, nz):
    # one strip (rectangle) of columns, 4095 and 4096 chunks of 8 levels
    say(f"init of 9 x 3 x {nz}, {conn} connections")
    rng = np.random.default_rng(conn)
    cs, ct = (np.maximum(rng.integers(-300, 200, (nz, 3, 9)), 0).astype(np.int32) for _ in range(2))
    cn = rng.integers(0, 60, (conn // 2, nz, 3, 9)).astype(np.int32)
    with cugip_amd.GridGraph() as g:
        g.set_grid(cs, ct, cn, conn=conn)
        flow = g.max_flow()
        inside = g.source_set().reshape(cs.shape).astype(bool)
    assert flow == cut_capacity(cs, ct, cn, inside, conn)
