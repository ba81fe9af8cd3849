"""Performance cases of the graph cut: what a program that uses this package has it do, through the
package's public classes, over the sizes it is used at.

A case's "kind" names the entry point:
  resident  max_flow_noalloc: capacities and cut stay in device memory (a serving loop that may not
            allocate), 6- or 26-connected, symmetric or directed n-links
  grid      GridGraph: repeated solves of a grid the handle holds, with the cut read back as the
            sink-side segmentation ("tmin", fill_segments) or the source set ("smin")
  segment   GridGraph from a host volume to a host segmentation, set-up included
  batch     GridBatch: independent grids of uneven sizes solved together
  generic   Graph: a sparse irregular graph (region adjacency) through the CSR path
  predict   Cnn.predict: learned cut proposal of a volume, its probabilities and certificate
  gradient  Cnn.gradients: one training step's loss and gradient against the solved cut

Flows and cuts are exact integers; only the network's outputs are floating.
"""
import math
import os

import numpy as np
import torch

import cugip_amd

# half neighbourhoods (dx, dy, dz) of the n-link planes, in the order of cap_n
HALF = {
    6: [(-1, 0, 0), (0, -1, 0), (0, 0, -1)],
    26: [(-1, -1, -1), (0, -1, -1), (1, -1, -1), (-1, 0, -1), (0, 0, -1), (1, 0, -1), (-1, 1, -1), (0, 1, -1),
         (1, 1, -1), (-1, -1, 0), (0, -1, 0), (1, -1, 0), (-1, 0, 0)],
}
BATCH_LO, BATCH_HI = 32, 128  # edge lengths of the batch workload


def listed():
    return [
        # one object patch per request of a serving loop: launch latency and host waits dominate
        {"name": "resident6_patch", "kind": "resident", "nx": 33, "ny": 30, "nz": 28, "conn": 6, "directed": False},
        # a whole organ crop, near the largest grid the no-allocation entry holds
        {"name": "resident6_crop", "kind": "resident", "nx": 118, "ny": 110, "nz": 105, "conn": 6, "directed": False},
        # a crop with full neighbourhoods and directed contrast (bright-to-dark edges)
        {"name": "resident26_directed", "kind": "resident", "nx": 77, "ny": 71, "nz": 64, "conn": 26,
         "directed": True},
        # one image through the whole pipeline, host volume to host segmentation, odd sizes
        {"name": "segment6_image", "kind": "segment", "nx": 131, "ny": 125, "nz": 119, "conn": 6},
        # the benchmark's instance size, solved again and again with the reference's fill_segments
        {"name": "grid6_256cube", "kind": "grid", "nx": 256, "ny": 256, "nz": 256, "conn": 6, "cut": "tmin"},
        # a middle-sized 26-connected volume
        {"name": "grid26_middle", "kind": "grid", "nx": 194, "ny": 190, "nz": 157, "conn": 26, "cut": "smin"},
        # the largest configuration of the benchmark
        {"name": "grid26_512x512x384", "kind": "grid", "nx": 512, "ny": 512, "nz": 384, "conn": 26, "cut": "smin"},
        # a queue of uneven volumes solved as one batch
        {"name": "batch6_56grids", "kind": "batch", "count": 56},
        # region adjacency graph of an oversegmented slice stack
        {"name": "generic_20k", "kind": "generic", "vertices": 19683},
        # the benchmark's irregular graph
        {"name": "generic_1m", "kind": "generic", "vertices": 1000000},
        # learned proposal of a volume
        {"name": "predict_image", "kind": "predict", "nx": 131, "ny": 125, "nz": 119},
        # one training sample
        {"name": "gradient_crop", "kind": "gradient", "nx": 98, "ny": 96, "nz": 91},
    ]


def _edges(rng, lo, hi, aspect=1.35):
    """Three edge lengths around one log-uniform edge, any integer, odd ones among them."""
    base = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return [max(8, int(round(base * math.exp(rng.uniform(-1, 1) * math.log(aspect) / 2)))) for _ in range(3)]


def draw(rng):
    kind = rng.choice(["resident", "resident", "grid", "grid", "segment", "batch", "generic", "predict", "gradient"])
    if kind == "resident":
        conn = rng.choice([6, 26])
        nx, ny, nz = _edges(rng, 20, 98 if conn == 6 else 68)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "conn": conn, "directed": rng.random() < 0.4}
    if kind == "grid":
        conn = rng.choice([6, 26])
        nx, ny, nz = _edges(rng, 48, 300 if conn == 6 else 240)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "conn": conn, "cut": rng.choice(["tmin", "smin"])}
    if kind == "segment":
        nx, ny, nz = _edges(rng, 40, 220)
        return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "conn": rng.choice([6, 6, 26])}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(3, 60)}
    if kind == "generic":
        return {"kind": kind, "vertices": int(math.exp(rng.uniform(math.log(2000), math.log(800000))))}
    nx, ny, nz = _edges(rng, 32, 180 if kind == "predict" else 110)
    return {"kind": kind, "nx": nx, "ny": ny, "nz": nz}


# ---- inputs ---------------------------------------------------------------------------------------


def _volume(nx, ny, nz, seed):
    """uint8 device volume: 3-8 ellipsoids at 180 on 60, semi-axes 8-25 % of the shortest edge, with
    N(0, 25^2) noise (the synthetic instances' distribution)."""
    r = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)
    short = min(nx, ny, nz)
    ax = [torch.arange(n, device="cuda", dtype=torch.float32) for n in (nz, ny, nx)]
    inside = torch.zeros((nz, ny, nx), dtype=torch.bool, device="cuda")
    for _ in range(int(r.integers(3, 9))):
        q = []
        for a, n in zip(ax, (nz, ny, nx)):
            c, s = r.integers(0, n), max(1.0, r.uniform(0.08, 0.25) * short)
            q.append(((a - float(c)) / float(s)) ** 2)
        inside |= q[0][:, None, None] + q[1][None, :, None] + q[2][None, None, :] <= 1.0
    v = torch.randn((nz, ny, nx), generator=gen, device="cuda").mul_(25.0).add_(60.0)
    v += inside * 120.0
    return v.round_().clamp_(0, 255).to(torch.uint8)


def _capacities(vol, conn, directed):
    """Device capacities of a volume by the default tables: Boykov-Jolly t-links, contrast-sensitive
    n-links; directed: an edge towards a brighter voxel keeps a quarter of its capacity."""
    w = cugip_amd.default_volume_weights()
    table = [torch.tensor(list(t), dtype=torch.int32, device="cuda") for t in w.nlink]
    v = vol.to(torch.int64)
    cs = torch.tensor(list(w.tlink_source), dtype=torch.int32, device="cuda")[v]
    ct = torch.tensor(list(w.tlink_sink), dtype=torch.int32, device="cuda")[v]
    nz, ny, nx = vol.shape
    cn = torch.zeros((conn // 2, nz, ny, nx), dtype=torch.int32, device="cuda")
    cnb = torch.zeros_like(cn) if directed else None
    for j, (dx, dy, dz) in enumerate(HALF[conn]):
        own = tuple(slice(max(0, -d), n - max(0, d)) for d, n in ((dz, nz), (dy, ny), (dx, nx)))
        nbr = tuple(slice(max(0, d), n - max(0, -d)) for d, n in ((dz, nz), (dy, ny), (dx, nx)))
        diff = v[nbr] - v[own]
        c = table[(dx != 0) + (dy != 0) + (dz != 0) - 1][diff.abs()]
        cn[j][own] = torch.where(diff > 0, c // 4, c) if directed else c
        if directed:
            cnb[j][own] = torch.where(diff < 0, c // 4, c)
    return cs, ct, cn, cnb


def _irregular_graph(vertices, seed):
    """Lattice neighbours plus one random vertex within 2 steps per axis, capacities 1-99 each way, a
    tenth of the vertices with a source link and a tenth with a sink link (the benchmark's graph)."""
    rng = np.random.default_rng(seed)
    k = max(4, int(round(vertices ** (1.0 / 3.0))))
    n = k ** 3
    z, y, x = (c.reshape(-1) for c in np.indices((k, k, k)))
    v = np.arange(n, dtype=np.int64)
    ends = []
    for dx, dy, dz in [(1, 0, 0), (0, 1, 0), (0, 0, 1)]:
        ok = (x + dx < k) & (y + dy < k) & (z + dz < k)
        ends.append((v[ok], v[ok] + dx + dy * k + dz * k * k))
    off = rng.integers(-2, 3, (n, 3))
    p = [np.clip(c + off[:, i], 0, k - 1) for i, c in enumerate((x, y, z))]
    u = (p[2] * k + p[1]) * k + p[0]
    ends.append((v[u != v], u[u != v]))
    edges = np.stack([np.concatenate([e[i] for e in ends]) for i in (0, 1)], 1)
    edges.sort(axis=1)
    fwd, bwd = (rng.integers(1, 100, len(edges)).astype(np.int32) for _ in range(2))
    cs, ct = ((rng.integers(0, 400, n) * (rng.random(n) < 0.1)).astype(np.int32) for _ in range(2))
    return n, edges, fwd, bwd, cs, ct


def _batch_shapes(case):
    return cugip_amd.batch_shapes(case["count"], case["count"], BATCH_LO, BATCH_HI)


def _network_parameters(case, seed):
    if case["kind"] == "predict":
        return np.load(os.path.join(os.path.dirname(cugip_amd.__file__), "cnn_weights.npy"))
    return cugip_amd.Cnn.init_params(seed)  # a step early in a training run


def _grid_from(vol, conn):
    g = cugip_amd.GridGraph()
    g.set_grid_volume(vol.cpu().numpy(), conn=conn)
    return g


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    if kind == "resident":
        vol = _volume(case["nx"], case["ny"], case["nz"], seed)
        s["shape"] = tuple(vol.shape)
        s["caps"] = _capacities(vol, case["conn"], case["directed"])
        s["source_set"] = torch.empty(s["shape"], dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
    elif kind == "grid":
        s["graph"] = _grid_from(_volume(case["nx"], case["ny"], case["nz"], seed), case["conn"])
    elif kind == "segment":
        s["volume"] = _volume(case["nx"], case["ny"], case["nz"], seed).cpu().numpy()
        s["graph"] = cugip_amd.GridGraph()
    elif kind == "batch":
        shapes = _batch_shapes(case)
        caps = [_capacities(_volume(nx, ny, nz, seed * 64 + i), 6, False) for i, (nz, ny, nx) in enumerate(shapes)]
        torch.cuda.synchronize()
        s["graph"] = cugip_amd.GridBatch()
        s["graph"].set_batch_device(shapes, 6, [tuple(t.data_ptr() for t in c[:3]) for c in caps])
    elif kind == "generic":
        n, edges, fwd, bwd, cs, ct = _irregular_graph(case["vertices"], seed)
        s["graph"] = cugip_amd.Graph()
        s["graph"].set_vertex_count(n)
        s["graph"].set_nweights(edges, fwd, bwd)
        s["graph"].set_tweights(cs, ct)
    else:
        vol = _volume(case["nx"], case["ny"], case["nz"], seed)
        s["graph"] = _grid_from(vol, 6)
        if kind == "gradient":
            s["graph"].max_flow()
        s["net"] = cugip_amd.Cnn()
        s["net"].set_params(_network_parameters(case, seed))
    return s


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "resident":
        cs, ct, cn, cnb = s["caps"]
        flow = cugip_amd.max_flow_noalloc(s["shape"], case["conn"], cs.data_ptr(), ct.data_ptr(), cn.data_ptr(),
                                          cnb.data_ptr() if cnb is not None else None, s["source_set"].data_ptr())
        return {"flow": flow, "source_set": s["source_set"]}
    if kind == "grid":
        flow = s["graph"].max_flow()
        return {"flow": flow, "cut": s["graph"].fill_segments() if case["cut"] == "tmin" else s["graph"].source_set()}
    if kind == "segment":
        s["graph"].set_grid_volume(s["volume"], conn=case["conn"])
        return {"flow": s["graph"].max_flow(), "segments": s["graph"].fill_segments()}
    if kind == "batch":
        flows = s["graph"].solve()
        return {"flows": np.array(flows), "cuts": [s["graph"].batch_source_set(i) for i in range(len(flows))]}
    if kind == "generic":
        return {"flow": s["graph"].max_flow(), "segments": s["graph"].fill_segments()}
    if kind == "predict":
        side, prob, certificate = s["net"].predict(s["graph"], None)
        return {"side": side, "prob": prob, "certificate": certificate}
    loss, grad = s["net"].gradients(s["graph"], None)
    return {"loss": loss, "grad": grad}


def work(case):
    """Inputs read once and outputs written once; flops of the network's products only."""
    kind = case["kind"]
    if kind == "batch":
        return {"bytes": 21 * sum(a * b * c for a, b, c in _batch_shapes(case)), "flops": 0}
    if kind == "generic":
        k = max(4, int(round(case["vertices"] ** (1.0 / 3.0))))
        edges = 3 * k * k * (k - 1) + k ** 3  # (one edge in 125 or so of the random ones is a loop)
        return {"bytes": edges * 16 + k ** 3 * 9, "flops": 0}
    vox = case["nx"] * case["ny"] * case["nz"]
    if kind in ("resident", "grid"):
        planes = case["conn"] // 2 * (2 if case.get("directed") else 1)
        return {"bytes": vox * (4 * (2 + planes) + 1), "flops": 0}
    if kind == "segment":
        return {"bytes": vox * 2, "flops": 0}
    forward = 2 * (27 * 3 * 16 + 3 * 27 * 16 * 16 + 16)
    if kind == "predict":
        return {"bytes": vox * (1 + 8 + 1 + 4), "flops": vox * forward}
    # gradient: the forward pass, the weight gradients (as many products) and the input gradients of
    # layers 2-4
    return {"bytes": vox * (1 + 8 + 1), "flops": vox * (2 * forward + 2 * 3 * 27 * 16 * 16)}


def exact(case, seed):
    """The network's probabilities in float64 (flows, cuts and the thresholded side are integers; the
    gradient's labels are a cut, which only a solver gives)."""
    if case["kind"] != "predict":
        return None
    vol = _volume(case["nx"], case["ny"], case["nz"], seed)
    cs, ct, _, _ = _capacities(vol, 6, False)
    p = torch.tensor(_network_parameters(case, seed), dtype=torch.float64, device="cuda")
    x = torch.stack([vol.double() / 255.0, cs.double() / 1000.0, ct.double() / 1000.0, torch.zeros_like(vol).double()], -1)
    nz, ny, nx = vol.shape
    at = 0
    for cin in (4, 16, 16, 16):
        weights = p[at:at + 27 * cin * 16].reshape(27, cin, 16)
        bias = p[at + 27 * cin * 16:at + 27 * cin * 16 + 16]
        at += 27 * cin * 16 + 16
        pad = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
        x = bias.expand(nz, ny, nx, 16).clone()
        for t in range(27):
            z0, y0, x0 = t // 9, t // 3 % 3, t % 3
            x += pad[z0:z0 + nz, y0:y0 + ny, x0:x0 + nx] @ weights[t]
        x.relu_()
    prob = torch.sigmoid(x @ p[at:at + 16] + p[at + 16])
    return {"side": None, "prob": prob.reshape(-1), "certificate": None}
