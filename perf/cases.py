"""Workloads of the message-passing hot path, as calls through the package's public entry points.

Four kinds, each over the range of sizes that atomistic models meet:

``harmonics``    ``o3.spherical_harmonics`` of edge vectors, alone or with the gradient that forces need
``message``      gather -> per-edge-weighted tensor product -> scatter-sum over a graph, forward or training step
``dense``        ``o3.FullyConnectedTensorProduct`` with shared weights on a batch of rows, forward or training step
``convolution``  a whole interaction block (self-connection, radial network, message, mixing)

``listed()`` holds the cases that are timed, ``draw(rng)`` makes more of the same ranges, ``prepare(case, seed)`` builds
what a program has in hand before the call, ``run(state)`` is one pass, ``work(case)`` and ``tolerance(case)`` say what a
pass cannot do without and how far two correct results may lie apart.
"""
import math

import torch

from e3nn_amd import nn, o3
from e3nn_amd.nn.message import message_tensor_product

DEVICE = "cuda:0"
CUTOFF = 5.0  # of the neighbour lists, in the unit of the positions
DENSITY = 50_000 / 86.8**3  # atoms per unit volume: about 37 neighbours inside the cutoff, away from the surface
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}

# node features of a message step, highest degree of the edge harmonics, and whether all paths onto one irrep are summed
# into one output block (the narrow sets) or every path keeps a block of its own (the wide one)
MESSAGES = {
    "narrow": ("16x0e+16x1o+16x2e", 2, True),
    "medium": ("32x0e+32x1o+32x2e", 2, True),
    "wide": ("128x0e+128x1o+128x2e+128x3o", 3, False),
}
# both inputs and the output of a dense product
PRODUCTS = {
    "small": ("16x0e+16x1o", "0e+1o+2e", "16x0e+16x1o+16x2e"),
    "mixed": ("64x0e+32x1o", "32x0e+32x1o+32x2e", "64x0e+64x1o+64x1e+64x2e"),
    "wide": ("128x0e+128x1o+128x2e",) * 3,
}


def listed():
    return [
        # edge attributes of a large neighbour list, evaluated once per step
        {"name": "harmonics_forward", "kind": "harmonics", "vectors": 4_000_000, "lmax": 3, "backward": False},
        # the same with the gradient that carries forces back to the positions; not a round number of vectors
        {"name": "harmonics_forces", "kind": "harmonics", "vectors": 1_876_963, "lmax": 2, "backward": True},
        # one molecule, as in single-structure inference: nothing but launches and latency
        {"name": "message_molecule", "kind": "message", "set": "medium", "nodes": 33, "edges": 526, "graph": "cutoff", "dtype": "f32",
         "index_bits": 64, "grouped": True, "backward": False},
        # a large atomistic system, inference
        {"name": "message_bulk", "kind": "message", "set": "medium", "nodes": 50_000, "edges": 1_876_964, "graph": "cutoff", "dtype": "f32",
         "index_bits": 64, "grouped": True, "backward": False},
        # ... and a training step on it: every gradient; edge list in the order of a pair list
        {"name": "message_bulk_training", "kind": "message", "set": "medium", "nodes": 50_000, "edges": 1_876_964, "graph": "cutoff",
         "dtype": "f32", "index_bits": 64, "grouped": False, "backward": True},
        # 128 channels up to l = 3 on a random graph, half-precision storage, inference
        {"name": "message_wide_bf16", "kind": "message", "set": "wide", "nodes": 20_000, "edges": 500_000, "graph": "random", "dtype": "bf16",
         "index_bits": 32, "grouped": False, "backward": False},
        # ... and the training step in full precision
        {"name": "message_wide_training", "kind": "message", "set": "wide", "nodes": 20_000, "edges": 500_000, "graph": "random",
         "dtype": "f32", "index_bits": 32, "grouped": False, "backward": True},
        # the smallest dense layer: vectors against harmonics
        {"name": "dense_small", "kind": "dense", "set": "small", "rows": 4096, "dtype": "f32", "backward": False},
        # 128 channels on both sides, half-precision storage, inference
        {"name": "dense_wide_bf16", "kind": "dense", "set": "wide", "rows": 65_536, "dtype": "bf16", "backward": False},
        # ... and the training step in full precision: the largest piece of work here
        {"name": "dense_wide_training", "kind": "dense", "set": "wide", "rows": 65_536, "dtype": "f32", "backward": True},
        # a step of molecular dynamics on a mid-sized system: the neighbour list is new, then harmonics and one block
        {"name": "convolution_step", "kind": "convolution", "nodes": 5_003, "edges": 176_852, "graph": "cutoff", "new_graph": True,
         "backward": False},
        # a training step of a block on a large system
        {"name": "convolution_training", "kind": "convolution", "nodes": 50_000, "edges": 1_876_964, "graph": "cutoff", "new_graph": False,
         "backward": True},
    ]  # fmt: skip


def _spread(rng, lo, hi):
    """A whole number between lo and hi, uniform in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _edges_within_cutoff(nodes):
    """Expected number of ordered pairs inside the cutoff among uniform points of a cube (an even number)."""
    side = (nodes / DENSITY) ** (1 / 3)
    r = min(CUTOFF / side, 1.0)
    # probability that two points of the unit cube lie within r <= 1 of each other
    p = 4 / 3 * math.pi * r**3 - 3 / 2 * math.pi * r**4 + 8 / 5 * r**5 - r**6 / 6
    return 2 * int(nodes * (nodes - 1) * p / 2)


def draw(rng):
    kind = rng.choice(["harmonics", "message", "message", "dense", "convolution"])
    if kind == "harmonics":
        return {"kind": kind, "vectors": _spread(rng, 100, 4_000_000), "lmax": rng.randint(1, 3), "backward": rng.random() < 0.5}
    if kind == "message":
        name = rng.choice(list(MESSAGES))
        graph = "random" if name == "wide" or rng.random() < 0.2 else "cutoff"
        nodes = _spread(rng, 20, 20_000 if name == "wide" else 50_000)
        edges = min(500_000, nodes * rng.randint(4, 60)) if graph == "random" else _edges_within_cutoff(nodes)
        return {"kind": kind, "set": name, "nodes": nodes, "edges": edges, "graph": graph, "dtype": rng.choice(["f32", "f32", "bf16"]),
                "index_bits": rng.choice([32, 64]), "grouped": rng.random() < 0.5, "backward": rng.random() < 0.5}  # fmt: skip
    if kind == "dense":
        name = rng.choice(list(PRODUCTS))
        dtype = "f32" if name == "small" else rng.choice(["f32", "bf16"])
        return {"kind": kind, "set": name, "rows": _spread(rng, 64, 65_536), "dtype": dtype, "backward": rng.random() < 0.5}
    nodes = _spread(rng, 20, 50_000)
    return {"kind": kind, "nodes": nodes, "edges": _edges_within_cutoff(nodes), "graph": "cutoff", "new_graph": rng.random() < 0.5,
            "backward": rng.random() < 0.5}  # fmt: skip


# ------------------------------------------------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEVICE)


def _neighbour_list(nodes, edges, gen):
    """Uniform positions in a cube and the ``edges / 2`` closest pairs (all pairs inside the cutoff, give or take the few
    that make the number of edges the same for every seed), as a list of pairs: every pair once, then every pair reversed."""
    pos = torch.rand(nodes, 3, generator=gen, device=DEVICE) * (nodes / DENSITY) ** (1 / 3)
    reach = 1.1 * CUTOFF if nodes > 2000 else math.inf
    a, b, dist = [], [], []
    for lo in range(0, nodes, 1024):
        rows = pos[lo : lo + 1024]
        d2 = sum((rows[:, None, c] - pos[None, lo:, c]).square_() for c in range(3))
        i, j = torch.nonzero(torch.triu(d2 < reach**2, diagonal=1), as_tuple=True)
        a.append(i + lo)
        b.append(j + lo)
        dist.append(d2[i, j])
    a, b = torch.cat(a), torch.cat(b)
    closest = torch.sort(torch.sort(torch.cat(dist), stable=True)[1][: edges // 2])[0]
    a, b = a[closest], b[closest]
    return pos, torch.cat([a, b]), torch.cat([b, a])


def _radial_basis(r):
    """Eight Bessel functions of the distance, scaled to unit second moment as the radial networks want them."""
    n = torch.arange(1, 9, device=DEVICE)
    x = r.clamp(min=1e-3)[:, None]
    basis = math.sqrt(2.0 / CUTOFF) * torch.sin(n * (math.pi / CUTOFF) * x) / x
    return (basis / basis.square().mean().sqrt().clamp(min=1e-6)).contiguous()


def _graph(case, gen):
    """(edge vectors, sources, destinations) of a case."""
    if case["graph"] == "random":
        src = torch.randint(0, case["nodes"], (case["edges"],), generator=gen, device=DEVICE)
        dst = torch.randint(0, case["nodes"], (case["edges"],), generator=gen, device=DEVICE)
    else:
        pos, src, dst = _neighbour_list(case["nodes"], case["edges"], gen)
    if case.get("grouped", True):  # as a neighbour search per node emits them
        dst, order = torch.sort(dst, stable=True)
        src = src[order]
    vec = _randn(gen, case["edges"], 3) if case["graph"] == "random" else pos[src] - pos[dst]
    idx = torch.int32 if case.get("index_bits", 64) == 32 else torch.int64
    return vec, src.to(idx), dst.to(idx)


def _prepare_harmonics(case, gen):
    direction = torch.nn.functional.normalize(_randn(gen, case["vectors"], 3), dim=1)
    vec = direction * torch.exp(0.5 * _randn(gen, case["vectors"], 1))
    state = {"vec": vec.requires_grad_(case["backward"]), "sh": o3.SphericalHarmonics(list(range(case["lmax"] + 1)), True, "component")}
    if case["backward"]:
        state["cotangent"] = _randn(gen, case["vectors"], (case["lmax"] + 1) ** 2)
    return state


def _message_product(name):
    features, lmax, merged = MESSAGES[name]
    sh = o3.Irreps.spherical_harmonics(lmax)
    return message_tensor_product(features, sh, irreps_out=features) if merged else message_tensor_product(features, sh, keep="0e+1o+2e+3o")


def _prepare_message(case, gen):
    dtype, tp = DTYPES[case["dtype"]], _message_product(case["set"])
    lmax = MESSAGES[case["set"]][1]
    vec, src, dst = _graph(case, gen)
    edges = nn.DstSortedEdges(src, dst, case["nodes"])
    state = {
        "tp": tp,
        "edges": edges,
        "x": _randn(gen, case["nodes"], tp.irreps_in1.dim).to(dtype).requires_grad_(case["backward"]),
        "w": _randn(gen, edges.num_edges, tp.weight_numel).to(dtype).requires_grad_(case["backward"]),
    }
    # the harmonics are formed inside the kernel where the set and the precision allow it, stored otherwise
    if case["set"] != "wide" and dtype == torch.float32:
        state["vec"] = vec.requires_grad_(case["backward"])
    else:
        # half-precision training differentiates an energy: node features and weights, not the geometry
        state["attr"] = o3.spherical_harmonics(list(range(lmax + 1)), vec, True, "component").to(dtype)
        state["attr"].requires_grad_(case["backward"] and dtype == torch.float32)
    if case["backward"]:
        state["cotangent"] = _randn(gen, case["nodes"], tp.irreps_out.dim).to(dtype)
    return state


def _prepare_dense(case, gen):
    dtype = DTYPES[case["dtype"]]
    tp = o3.FullyConnectedTensorProduct(*PRODUCTS[case["set"]])
    tp = tp.to(DEVICE)
    with torch.no_grad():
        tp.weight.copy_(_randn(gen, tp.weight_numel))
    tp = tp.to(dtype)
    x1 = _randn(gen, case["rows"], tp.irreps_in1.dim)
    x2 = _randn(gen, case["rows"], tp.irreps_in2.dim)
    if case["set"] == "small":
        x2 = o3.spherical_harmonics([0, 1, 2], _randn(gen, case["rows"], 3), True, "component")
    state = {"tp": tp, "x1": x1.to(dtype).requires_grad_(case["backward"]), "x2": x2.to(dtype).requires_grad_(case["backward"])}
    tp.weight.requires_grad_(case["backward"])
    if case["backward"]:
        state["cotangent"] = _randn(gen, case["rows"], tp.irreps_out.dim).to(dtype)
    return state


def _prepare_convolution(case, gen):
    features = MESSAGES["medium"][0]
    conv = nn.Convolution(features, "4x0e", o3.Irreps.spherical_harmonics(2), features, [8, 64], 37.5).to(DEVICE)
    with torch.no_grad():
        for p in conv.parameters():  # the values of a trained block: none of its branches is switched off
            p.copy_(_randn(gen, *p.shape))
    vec, src, dst = _graph(case, gen)
    species = torch.randint(0, 4, (case["nodes"],), generator=gen, device=DEVICE)
    state = {
        "conv": conv, "src": src, "dst": dst, "nodes": case["nodes"], "vec": vec, "scalars": _radial_basis(vec.norm(dim=1)),
        "species": torch.nn.functional.one_hot(species, 4).float(),
        "x": _randn(gen, case["nodes"], conv.irreps_node_input.dim).requires_grad_(case["backward"]),
        "edges": None if case["new_graph"] else nn.DstSortedEdges(src, dst, case["nodes"]),
    }  # fmt: skip
    if case["backward"]:
        state["cotangent"] = _randn(gen, case["nodes"], conv.irreps_node_output.dim)
    return state


def prepare(case, seed):
    make = {"harmonics": _prepare_harmonics, "message": _prepare_message, "dense": _prepare_dense, "convolution": _prepare_convolution}
    state = make[case["kind"]](case, _generator(seed))
    state["kind"] = case["kind"]
    return state


# ------------------------------------------------------------------------------------------------------------- passes
def _with_gradients(state, out, inputs):
    if "cotangent" not in state:
        return out
    return (out, *torch.autograd.grad(out, inputs, state["cotangent"]))


def run(state):
    if state["kind"] == "harmonics":
        return _with_gradients(state, state["sh"](state["vec"]), (state["vec"],))
    if state["kind"] == "message":
        tp, x, w, edges = state["tp"], state["x"], state["w"], state["edges"]
        if "vec" in state:
            out = tp.forward_gather_scatter_sh(x, state["vec"], w, edges, True, "component")
            return _with_gradients(state, out, (x, state["vec"], w))
        out = tp.forward_gather_scatter(x, state["attr"], w, edges=edges)
        return _with_gradients(state, out, tuple(t for t in (x, state["attr"], w) if t.requires_grad))
    if state["kind"] == "dense":
        tp, x1, x2 = state["tp"], state["x1"], state["x2"]
        return _with_gradients(state, tp(x1, x2), (x1, x2, tp.weight))
    conv, x, edges = state["conv"], state["x"], state["edges"]
    with torch.set_grad_enabled("cotangent" in state):
        if edges is None:
            edges = nn.DstSortedEdges(state["src"], state["dst"], state["nodes"])
        attr = o3.spherical_harmonics([0, 1, 2], state["vec"], True, "component")
        out = conv(x, state["species"], state["src"], state["dst"], attr, state["scalars"], edges=edges)
    return _with_gradients(state, out, (x, *conv.parameters()))


# -------------------------------------------------------------------------------------------------- what a pass needs
def _message_counts(tp):
    """(multiply-adds of one edge, weights per edge) of a uvu product: one per Clebsch-Gordan non-zero and channel, and
    one per output component and channel for the weight."""
    macs = 0
    for t in tp.instructions:
        mul, (l1, l2, l3) = t.path_shape[0], (tp.irreps_in1[t.i_in1].ir.l, tp.irreps_in2[t.i_in2].ir.l, tp.irreps_out[t.i_out].ir.l)
        macs += mul * (int((o3.wigner_3j(l1, l2, l3).abs() > 1e-9).sum()) + 2 * l3 + 1)
    return macs, tp.weight_numel


def work(case):
    if case["kind"] == "harmonics":
        n, c = case["vectors"], (case["lmax"] + 1) ** 2
        bytes_ = n * 4 * (3 + c) + (n * 4 * (3 + c) if case["backward"] else 0)
        return {"bytes": bytes_, "flops": n * c * (12 if case["backward"] else 4)}
    if case["kind"] == "message":
        tp, size = _message_product(case["set"]), DTYPES[case["dtype"]].itemsize
        macs, weights = _message_counts(tp)
        e, n = case["edges"], case["nodes"]
        stored = case["set"] == "wide" or case["dtype"] != "f32"
        edge_in = tp.irreps_in2.dim * size if stored else 12
        rows = n * size * (tp.irreps_in1.dim + tp.irreps_out.dim)
        once = e * (weights * size + edge_in) + rows
        indices = 2 * e * case["index_bits"] // 8
        # a training step reads the cotangent beside these and writes a gradient for every input
        return {"bytes": indices + once * (2 if case["backward"] else 1), "flops": 2 * e * macs * (4 if case["backward"] else 1)}
    if case["kind"] == "dense":
        tp, size = o3.FullyConnectedTensorProduct(*PRODUCTS[case["set"]]), DTYPES[case["dtype"]].itemsize
        macs = 0
        for t in tp.instructions:  # the cheapest order of the contraction
            ls = (tp.irreps_in1[t.i_in1].ir.l, tp.irreps_in2[t.i_in2].ir.l, tp.irreps_out[t.i_out].ir.l)
            macs += math.prod(t.path_shape) * (2 * min(ls) + 1)
        once = size * (case["rows"] * (tp.irreps_in1.dim + tp.irreps_in2.dim + tp.irreps_out.dim) + tp.weight_numel)
        return {"bytes": once * (2 if case["backward"] else 1), "flops": 2 * case["rows"] * macs * (4 if case["backward"] else 1)}
    n, e = case["nodes"], case["edges"]
    features = o3.Irreps(MESSAGES["medium"][0])
    macs, weights = _message_counts(message_tensor_product(features, o3.Irreps.spherical_harmonics(2), keep="0e+1o+2e"))
    per_edge = macs + 8 * 64 + 64 * weights
    per_node = sum(32 * 32 * 4 * ir.dim for _, ir in features) * 2 + sum(32 * 32 * 4 * ir.dim * k for k, (_, ir) in zip((3, 4, 4), features))
    once = e * (12 + 16 + 8 * 4) + n * 4 * (2 * features.dim + 4)
    return {"bytes": once + (n * 4 * 2 * features.dim if case["backward"] else 0),
            "flops": 2 * (e * per_edge + n * per_node) * (3 if case["backward"] else 1)}  # fmt: skip


def tolerance(case):
    """About four times the largest error seen against the same pass in 64 bits (2-norm of each output)."""
    if case.get("dtype") == "bf16":
        return {"rel": 8e-3}  # seen: 1.66e-3 (the rounding of the result) to 2.2e-3
    if case["kind"] in ("harmonics", "message"):
        return {"rel": 7e-7}  # seen: up to 1.7e-7, sums of a few dozen terms
    return {"rel": 8e-6}  # seen: up to 1.7e-6, sums over up to 128 x 128 channel pairs or all rows
