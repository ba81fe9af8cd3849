"""The one-launch solve of generic graphs at the sizes and shapes where its paths part: one workgroup
or several, each lane-group width (by the mean degree), degrees beyond a pass, steps that one
workgroup runs alone, lists longer than the LDS stage, the round cap, and the staged launches of a
traced solve. Flow, S_min and T_min are integers and equal the CPU solver's."""
import numpy as np
import pytest

import cugip_amd
import oracle
from tests.gpu_util import say

pytestmark = pytest.mark.gpu


def handle(g):
    n, ea, eb, fwd, bwd, cs, ct = g
    gr = cugip_amd.Graph()
    gr.set_vertex_count(n)
    gr.set_nweights(np.stack([ea, eb], 1), fwd, bwd)
    gr.set_tweights(cs, ct)
    return gr


def check(g, **policy):
    with handle(g) as gr:
        if policy:
            gr.set_policy(**policy)
        ref = oracle.bk(*g)
        for _ in range(2):  # (a second solve starts from the state the first one left)
            assert gr.max_flow() == ref[0]
            assert np.array_equal(gr.source_set(), ref[1]) and np.array_equal(gr.fill_segments(1, 0), ref[2])


def graph(rng, ea, eb, n, share=0.1, tcap=400, cap=100):
    ea, eb = np.minimum(ea, eb).astype(np.int32), np.maximum(ea, eb).astype(np.int32)
    fwd, bwd = (rng.integers(0, cap, ea.size).astype(np.int32) for _ in range(2))
    cs, ct = ((rng.integers(0, tcap, n) * (rng.random(n) < share)).astype(np.int32) for _ in range(2))
    return n, ea, eb, fwd, bwd, cs, ct


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 8192, 70000])
@pytest.mark.parametrize("degree", [2, 7, 20, 70])
def test_sizes_and_degrees(n, degree):
    if n * degree > 1000000:
        degree = 14
    say(f"generic solve n {n} degree {degree}")
    rng = np.random.default_rng(n + degree)
    m = n * degree // 2
    check(graph(rng, rng.integers(0, n, m), rng.integers(0, n, m), n, tcap=100 * degree))


@pytest.mark.parametrize("minimal_residual", [0.0, 6.0])
def test_long_chain(minimal_residual):
    """3000 levels of a handful of vertices: nearly every step is run by workgroup 0 alone."""
    n = 3000
    say(f"generic chain of {n}, threshold {minimal_residual}")
    rng = np.random.default_rng(5)
    g = list(graph(rng, np.arange(n - 1), np.arange(1, n), n, share=0.0))
    g[3] += 5
    g[5][0], g[5][40], g[6][n - 1], g[6][1500] = 1000, 30, 1000, 3
    check(tuple(g), minimal_residual=minimal_residual)


def test_hubs():
    """Vertices of thousands of arcs next to leaves (many passes of a lane group), and one step that
    wakes more vertices than a workgroup keeps in LDS."""
    say("generic hubs")
    rng = np.random.default_rng(6)
    n = 30000
    leaves = np.arange(3, n)
    g = list(graph(rng, np.concatenate([np.zeros(leaves.size, int), leaves % 2 + 1]), np.concatenate([leaves, leaves]),
                   n, share=0.3))
    g[5][0], g[6][1], g[6][2] = 500000, 300000, 300000
    check(tuple(g))


def test_round_cap():
    say("generic round cap")
    rng = np.random.default_rng(7)
    n, m = 3000, 9000
    g = graph(rng, rng.integers(0, n, m), rng.integers(0, n, m), n)
    with handle(g) as gr:
        gr.set_policy(max_rounds=1)  # the relabel that finds the end is the second one at the earliest
        with pytest.raises(cugip_amd.CgpError) as e:
            gr.max_flow()
        assert e.value.code == cugip_amd.CGP_ERR_NOT_CONVERGED
        gr.set_policy(max_rounds=1 << 16)
        assert gr.max_flow() == oracle.bk(*g)[0]


@pytest.mark.parametrize("n", [900, 20000])
def test_traced_solve_stage_by_stage(n):
    say(f"generic traced solve n {n}")
    rng = np.random.default_rng(n)
    m = 4 * n
    g = graph(rng, rng.integers(0, n, m), rng.integers(0, n, m), n)
    ref = oracle.bk(*g)
    events = []
    with handle(g) as gr:
        gr.set_trace(lambda ev, it, done, flow, ls: events.append((ev, it, done, flow, ls)))
        assert gr.max_flow() == ref[0]
        assert np.array_equal(gr.source_set(), ref[1]) and np.array_equal(gr.fill_segments(1, 0), ref[2])
        labels = gr.labels()
    relabels = [e for e in events if e[0] == cugip_amd.TRACE_AFTER_RELABEL]
    pushes = [e for e in events if e[0] == cugip_amd.TRACE_AFTER_PUSH]
    assert len(relabels) == len(pushes) and [p[2] for p in pushes] == [0] * (len(pushes) - 1) + [1]
    assert all(a[3] <= b[3] for a, b in zip(pushes, pushes[1:])) and pushes[-1][3] == ref[0]
    # the last relabel's level starts are the counts of the exact labels
    finite = labels[labels < cugip_amd.LABEL_UNREACHABLE]
    counts = np.bincount(finite, minlength=2)[1:] if finite.size else np.zeros(1, int)
    assert list(relabels[-1][4]) == [0] + list(np.cumsum(counts))
