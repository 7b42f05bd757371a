"""The work this solver is measured on, through its public entry points.

A case is one multicut problem (or several) and the call that solves it:

  entry    "torch"   rama_py.rama_torch: tensors in, tensors out (the Python
                     interface of RAMA's users)
           "device"  rama_amd.solve_device: device pointers in and out, what
                     a C++ program with resident graphs calls
           "host"    rama_amd.solve: host arrays in and out
           "batch"   rama_amd.solve_batch: many host instances in one call
           "serve"   rama_amd.Server: requests submitted one after the other,
                     then waited for
  preset   the solver's own presets: P (primal), PD (default), PD+, D (lower
           bound only)
  graph    the generators of rama_amd/instances.py, redone on the GPU because
           inputs are made many times: "grid2d" (4-neighbourhood, or with the
           long-range offsets 9 and 27), "grid3d" (6-neighbourhood), both with
           a Voronoi partition and logit-Beta costs, and "er" (random graph of
           average degree 8, N(0.3, 1) costs)

Sizes run from the 64x64 grid (8,064 edges) to the 192^3 grid (21,123,072).
"""
import math

import numpy as np
import torch

import rama_amd
from rama_amd import rama_py

# Cluster densities of the generators: nodes per Voronoi seed.
NODES_PER_SEED_2D = 1049
NODES_PER_SEED_3D = 354


def listed():
    return [
        # the smallest call: the 64x64 grid, as a PyTorch program makes it
        # inside a training loop (latency, launches, read-backs)
        {"name": "torch_pd_grid_64x64", "entry": "torch", "preset": "PD", "graph": "grid2d", "a": 64, "b": 64, "long": False},
        # a small scattered graph with odd size, primal only, from host arrays
        {"name": "host_p_er_5003", "entry": "host", "preset": "P", "graph": "er", "a": 5003, "b": 0, "long": False},
        # a small superpixel-like grid with the best-quality preset
        {"name": "torch_pdplus_grid_187x211", "entry": "torch", "preset": "PD+", "graph": "grid2d", "a": 187, "b": 211, "long": False},
        # an ordinary correlation-clustering graph with ids in gaps, which the
        # solver renumbers first (sanitize_graph)
        {"name": "host_pd_er_50021_gaps", "entry": "host", "preset": "PD", "graph": "er", "a": 50021, "b": 0, "long": False, "gaps": True},
        # an image segmentation graph of ordinary size with long-range edges
        {"name": "torch_pd_long_257x509", "entry": "torch", "preset": "PD", "graph": "grid2d", "a": 257, "b": 509, "long": True},
        # a volume of ordinary size, best quality
        {"name": "device_pdplus_grid3d_71", "entry": "device", "preset": "PD+", "graph": "grid3d", "a": 71, "b": 0, "long": False},
        # the primal heuristic alone on a large image
        {"name": "device_p_long_1024x2048", "entry": "device", "preset": "P", "graph": "grid2d", "a": 1024, "b": 2048, "long": True},
        # the headline workload: 12,469,248 edges with the default preset
        {"name": "device_pd_long_1024x2048", "entry": "device", "preset": "PD", "graph": "grid2d", "a": 1024, "b": 2048, "long": True},
        # the lower bound alone on the same graph
        {"name": "device_d_long_1024x2048", "entry": "device", "preset": "D", "graph": "grid2d", "a": 1024, "b": 2048, "long": True},
        # the largest: a 192^3 volume with the best-quality preset
        {"name": "device_pdplus_grid3d_192", "entry": "device", "preset": "PD+", "graph": "grid3d", "a": 192, "b": 0, "long": False},
        # many instances in one call: half grids, half random graphs
        {"name": "batch_pd_48_mixed", "entry": "batch", "preset": "PD", "graph": "mixed", "a": 48, "b": 60000, "long": False},
        # a burst of requests at the serving loop
        {"name": "serve_pd_24_burst", "entry": "serve", "preset": "PD", "graph": "mixed", "a": 24, "b": 60000, "long": False},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges: any preset at any size, grids of any
    shape, every entry.  The largest sizes go with the device entry."""
    kind = rng.choice(["grid2d", "grid2d", "long", "long", "grid3d", "er", "er", "mixed"])
    preset = rng.choice(["P", "PD", "PD", "PD+", "D"])
    if kind == "mixed":
        entry = rng.choice(["batch", "batch", "serve"])
        return {"entry": entry, "preset": "PD", "graph": "mixed", "a": rng.randint(8, 48), "b": _log_uniform(rng, 4000, 60000), "long": False}
    if kind == "er":
        n = _log_uniform(rng, 2000, 500000)
        entry = rng.choice(["torch", "host", "device"])
        case = {"entry": entry, "preset": preset, "graph": "er", "a": n, "b": 0, "long": False}
        if rng.random() < 0.3:
            case["gaps"] = True
        return case
    if kind == "grid3d":
        d = _log_uniform(rng, 14, 160)
        entry = "device" if d > 80 else rng.choice(["torch", "host", "device"])
        return {"entry": entry, "preset": preset, "graph": "grid3d", "a": d, "b": 0, "long": False}
    n = _log_uniform(rng, 4096, 2000000)
    aspect = math.exp(rng.uniform(-0.7, 0.7))
    h = max(30, int(round(math.sqrt(n) * aspect)))
    w = max(30, n // h)
    entry = "device" if n > 400000 else rng.choice(["torch", "host", "device"])
    return {"entry": entry, "preset": preset, "graph": "grid2d", "a": h, "b": w, "long": kind == "long"}


# ------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _gamma(k, n, g):
    """n Gamma(k) variates for a whole k: a sum of k exponentials."""
    s = torch.zeros(n, dtype=torch.float64, device="cuda")
    for _ in range(k):
        s -= torch.log1p(-torch.rand(n, generator=g, device="cuda", dtype=torch.float64))
    return s


def _beta(a, b, n, g):
    x = _gamma(a, n, g)
    return x / (x + _gamma(b, n, g))


def _voronoi(shape, n_seeds, g):
    """The nearest of n_seeds uniform points for every node of the grid, on
    coordinates centred on the grid."""
    size = torch.tensor(shape, dtype=torch.float32, device="cuda")
    seeds = (torch.rand(n_seeds, len(shape), generator=g, device="cuda") - 0.5) * size
    norm = (seeds * seeds).sum(1)
    axes = [torch.arange(s, dtype=torch.float32, device="cuda") - 0.5 * s for s in shape]
    pts = torch.stack([t.reshape(-1) for t in torch.meshgrid(*axes, indexing="ij")], dim=1)
    label = torch.empty(len(pts), dtype=torch.int64, device="cuda")
    step = max(1, (1 << 28) // n_seeds)
    for b in range(0, len(pts), step):
        label[b:b + step] = torch.addmm(norm, pts[b:b + step], seeds.t(), alpha=-2.0).argmin(1)
    return label


def _grid(shape, offsets):
    idx = torch.arange(math.prod(shape), dtype=torch.int64, device="cuda").reshape(shape)
    I, J = [], []
    for off in offsets:
        I.append(idx[tuple(slice(0, s - o) for s, o in zip(shape, off))].reshape(-1))
        J.append(idx[tuple(slice(o, s) for s, o in zip(shape, off))].reshape(-1))
    return torch.cat(I), torch.cat(J)


def _costs(p):
    p = p.clamp(1e-3, 1.0 - 1e-3)
    return torch.log((1.0 - p) / p).to(torch.float32)


def _grid2d(h, w, long, g):
    offsets = [(0, 1), (1, 0)] + ([(9, 0), (0, 9), (27, 0), (0, 27)] if long else [])
    label = _voronoi((h, w), max(2, round(h * w / NODES_PER_SEED_2D)), g)
    i, j = _grid((h, w), offsets)
    m = len(i)
    inside = _beta(2, 8, m, g)
    across = _beta(8, 2, m, g)
    flip = torch.rand(m, generator=g, device="cuda") < 0.10
    return i, j, _costs(torch.where((label[i] == label[j]) | flip, inside, across))


def _grid3d(d, g):
    shape = (d, d, d)
    label = _voronoi(shape, max(2, round(d ** 3 / NODES_PER_SEED_3D)), g)
    i, j = _grid(shape, [(0, 0, 1), (0, 1, 0), (1, 0, 0)])
    m = len(i)
    mix = torch.rand(m, generator=g, device="cuda") < 0.7
    inside = torch.where(mix, _beta(2, 8, m, g), _beta(5, 5, m, g))
    across = _beta(8, 2, m, g)
    return i, j, _costs(torch.where(label[i] == label[j], inside, across))


def _er(n, g):
    m = 4 * n
    keys = torch.empty(0, dtype=torch.int64, device="cuda")
    while len(keys) < m:
        a, b = torch.randint(0, n, (2, int(1.1 * m) + 16), generator=g, device="cuda")
        k = torch.minimum(a, b) * n + torch.maximum(a, b)
        keys = torch.unique(torch.cat([keys, k[a != b]]))
    keys = keys[torch.randperm(len(keys), generator=g, device="cuda")[:m]].sort().values
    c = 0.3 + torch.randn(m, generator=g, device="cuda")
    return keys // n, keys % n, c


def _graph(case, g):
    if case["graph"] == "grid2d":
        i, j, c = _grid2d(case["a"], case["b"], case["long"], g)
    elif case["graph"] == "grid3d":
        i, j, c = _grid3d(case["a"], g)
    else:
        i, j, c = _er(case["a"], g)
    if case.get("gaps"):
        # half of the ids are in use, the last one among them
        n = case["a"]
        ids = torch.randperm(2 * n - 1, generator=g, device="cuda")[:n].sort().values
        ids[-1] = 2 * n - 1
        i, j = ids[i], ids[j]
    return i.to(torch.int32).contiguous(), j.to(torch.int32).contiguous(), c.contiguous()


def _mixed(case, g):
    """`a` instances of log-uniform size from 1000 to b nodes: even ones 2D
    grids, odd ones random graphs, as host arrays."""
    rng = np.random.Generator(np.random.PCG64(case["a"]))
    out = []
    for k, u in enumerate(rng.uniform(size=case["a"])):
        n = int(1000 * (case["b"] / 1000) ** u)
        if k % 2 == 0:
            h = max(2, math.isqrt(n))
            i, j, c = _grid2d(h, max(2, -(-n // h)), False, g)
        else:
            i, j, c = _er(n, g)
        out.append(tuple(t.cpu().numpy() for t in (i.to(torch.int32), j.to(torch.int32), c)))
    return out


def prepare(case, seed):
    g = _generator(seed)
    state = {"entry": case["entry"]}
    if case["entry"] in ("batch", "serve"):
        state["instances"] = _mixed(case, g)
        state["options"] = rama_amd.options(case["preset"], verbose=0)
        if case["entry"] == "serve":
            state["server"] = rama_amd.Server(workers=8, opts=state["options"])
        return state
    i, j, c = _graph(case, g)
    gaps = bool(case.get("gaps"))
    if case["entry"] == "torch":
        o = rama_py.multicut_solver_options(case["preset"])
        o.verbose = False
        o.sanitize_graph = gaps
        state["options"] = o
        state["graph"] = (i, j, c)
        return state
    state["options"] = rama_amd.options(case["preset"], verbose=0, sanitize_graph=int(gaps))
    if case["entry"] == "host":
        state["graph"] = tuple(t.cpu().numpy() for t in (i, j, c))
    else:
        nodes = int(torch.maximum(i.max(), j.max())) + 2
        state["graph"] = (i, j, c)
        state["labels"] = torch.empty(nodes, dtype=torch.int32, device="cuda")
    return state


def run(state):
    entry = state["entry"]
    if entry == "torch":
        labels, bound = rama_py.rama_torch(*state["graph"], state["options"])
        return {"labels": labels, "bound": bound}
    if entry == "device":
        i, j, c = state["graph"]
        labels = state["labels"]
        n, bound, _, _ = rama_amd.solve_device(i.data_ptr(), j.data_ptr(), c.data_ptr(), c.numel(), labels.data_ptr(), labels.numel(),
                                               state["options"], device=0, stream=torch.cuda.current_stream().cuda_stream)
        return {"labels": labels[:n], "bound": bound}
    if entry == "host":
        labels, bound, _, _ = rama_amd.solve(*state["graph"], state["options"])
        return {"labels": labels, "bound": bound}
    if entry == "batch":
        done = rama_amd.solve_batch(state["instances"], state["options"], workers=8)
    else:
        server = state["server"]
        tickets = [server.submit(*x) for x in state["instances"]]
        done = [server.wait(t)[:2] for t in tickets]
    return {"labels": np.concatenate([x[0] for x in done]), "bounds": np.array([x[1] for x in done])}


# -------------------------------------------------------------------- work

def _sizes(case):
    """(nodes, edges) of a case; of a mixed set, about."""
    a, b = case["a"], case["b"]
    if case["graph"] == "grid2d":
        offs = [(0, 1), (1, 0)] + ([(9, 0), (0, 9), (27, 0), (0, 27)] if case["long"] else [])
        return a * b, sum((a - x) * (b - y) for x, y in offs)
    if case["graph"] == "grid3d":
        return a ** 3, 3 * a * a * (a - 1)
    if case["graph"] == "er":
        return a * (2 if case.get("gaps") else 1), 4 * a
    mean = (b - 1000) / math.log(b / 1000)
    return int(a * mean), int(3 * a * mean)


def work(case):
    """Each edge (two ids, one cost) read once, each label written once (the
    lower bound alone: no labels).  The solver has no dense product."""
    nodes, edges = _sizes(case)
    return {"bytes": 12 * edges + (0 if case["preset"] == "D" else 4 * nodes), "flops": 0}


def exact(case, seed):
    """Where the bound has a closed form: the primal preset's bound is the sum
    of the negative costs.  The others come out of a search and a message
    passing that stop by their own rounding; labels are whole numbers."""
    if case["preset"] != "P" or case["entry"] in ("batch", "serve"):
        return None
    c = _graph(case, _generator(seed))[2].to(torch.float64)
    bound = c.clamp(max=0.0).sum()
    return {"labels": None, "bound": bound.reshape(1) if case["entry"] == "torch" else float(bound)}
