"""What the speed of this framework is measured on: the calls that an N-body or
FMM program makes on its trees, from the smallest to the largest in use.

Kinds of case:

* ``step``: one time step of a simulation: build the tree from new positions,
  its geometry, and the far and near lists of the dual-tree walk.
* ``build``: the tree alone, with reordered particles (sorting and neighbour
  programs, and every step that keeps old lists).
* ``upward``: the node data of a tree that is kept while the particles move or
  carry new masses: boxes, their level-major views, and mass moments.
* ``dense``, ``grouped``: the two M2L layouts of a far list.
* ``batch``: a step for many independent systems of uneven size, called
  directly or replayed as a captured graph on moved positions.
* ``predict``, ``train``: the capacity model that sizes a walk's streams.

The order of the entries inside one row of a far or near list is not
specified. The listed nodes come back as the sum of a 32-bit weight per node
over every row (as a monopole pass sums masses over each row), modulo 2^32,
next to all counts and offsets: the same entries in another order give the
same sums. Arrays whose length follows from the particles are kept in arrays
of fixed length, as a program does that allocates once.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import yggdrax_amd as ygg
from yggdrax_amd import batch, dense_interactions, grouped_interactions, learned, tree_moments
from yggdrax_amd.tree import device_topology

# Steps of at most this many particles take the default options of the walk
# (dense neighbour positions among them).
SMALL = 20_000
# Room for far entries, per node.
FAR_ROOM = 2048


# ---- the cases -------------------------------------------------------------

def _step(points, leaf, theta, mac, octree, cloud, config=False):
    return {"kind": "step", "points": points, "leaf": leaf, "theta": theta, "mac": mac,
            "octree": octree, "cloud": cloud, "config": config}


def listed():
    return [
        # the reference's own 512-point example with its fixed capacities:
        # latency of a whole step
        dict(_step(512, 16, 0.6, "dehnen", True, "uniform", True), name="step_octree_512"),
        # a small system with every option at its default (leaf size 8, "bh"
        # criterion, dense neighbour positions), odd size
        dict(_step(10_007, 8, 0.7, "bh", False, "uniform"), name="step_radix_10007"),
        # an ordinary system: a clustered snapshot of 10^5 particles
        dict(_step(100_003, 32, 0.5, "dehnen", True, "clustered"), name="step_octree_100003"),
        # a Plummer sphere of 2^20 particles, the usual single-galaxy run
        dict(_step(1 << 20, 32, 0.5, "dehnen", False, "plummer"), name="step_radix_1m"),
        # the benchmark workload: 2^24 clustered particles
        dict(_step(1 << 24, 64, 0.5, "dehnen", True, "clustered"), name="step_octree_16m"),
        # a deep radix tree with the default leaf size over an odd particle count
        {"kind": "build", "points": 3_000_017, "leaf": 8, "octree": False, "cloud": "uniform",
         "name": "build_radix_3m"},
        # node data refreshed on a kept tree
        {"kind": "upward", "points": 4_000_003, "leaf": 32, "cloud": "plummer",
         "masses": "float32", "name": "upward_4m"},
        # M2L buffers for a padded, level-by-level downward sweep
        {"kind": "dense", "points": 1 << 18, "leaf": 32, "theta": 0.5, "cloud": "plummer",
         "name": "dense_262k"},
        # far pairs by displacement class, for one translation operator per class
        {"kind": "grouped", "points": 1 << 20, "leaf": 32, "theta": 0.5, "cloud": "plummer",
         "name": "grouped_1m"},
        # 1024 independent systems of 256 to 65536 particles, every step replayed
        # on new positions
        {"kind": "batch", "systems": 1024, "smallest": 256, "largest": 65536, "leaf": 32,
         "theta": 0.6, "graph": True, "name": "batch_graph_1024"},
        # stream sizes of the benchmark tree predicted per node
        {"kind": "predict", "points": 1 << 24, "leaf": 64, "cloud": "clustered",
         "name": "predict_16m"},
        # one optimiser step of the capacity model at its training batch
        {"kind": "train", "rows": 4096, "name": "train_4096"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 6 + ["build"] * 2 + ["upward", "dense", "grouped", "batch",
                                                      "batch", "predict", "train"])
    cloud = rng.choice(["uniform", "plummer", "clustered"])
    if kind == "step":
        leaf = rng.choice([8, 16, 32, 64])
        points = _log(rng, 200, (1 << 17) * leaf)  # at most 2^18 nodes
        theta = round(rng.uniform(0.5, 0.8), 2)
        return _step(points, leaf, theta, rng.choice(["bh", "dehnen", "dehnen", "engblom"]),
                     rng.random() < 0.5, cloud, points < 2000 and rng.random() < 0.5)
    if kind == "build":
        return {"kind": kind, "points": _log(rng, 200, 1 << 23),
                "leaf": rng.choice([4, 8, 16, 33, 64]), "octree": rng.random() < 0.5,
                "cloud": cloud}
    if kind == "upward":
        return {"kind": kind, "points": _log(rng, 1000, 1 << 23), "leaf": rng.choice([8, 16, 32, 64]),
                "cloud": cloud, "masses": rng.choice(["float32", "float32", "float64"])}
    if kind in ("dense", "grouped"):
        return {"kind": kind, "points": _log(rng, 500, 1 << (17 if kind == "dense" else 19)),
                "leaf": rng.choice([16, 32, 64]), "theta": round(rng.uniform(0.5, 0.8), 2),
                "cloud": rng.choice(["uniform", "plummer"])}
    if kind == "batch":
        smallest = _log(rng, 100, 1000)
        return {"kind": kind, "systems": _log(rng, 2, 512), "smallest": smallest,
                "largest": _log(rng, 2 * smallest, 30_000), "leaf": rng.choice([16, 32]),
                "theta": round(rng.uniform(0.5, 0.8), 2), "graph": rng.random() < 0.4}
    if kind == "predict":
        return {"kind": kind, "points": _log(rng, 1000, 1 << 23), "leaf": rng.choice([16, 32, 64]),
                "cloud": cloud}
    return {"kind": kind, "rows": _log(rng, 200, 40_000)}


# ---- inputs ----------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) % (1 << 62))


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _plummer(g, n, a, cut=20.0):
    """n points of Plummer spheres of scale radius a (a number, or one per
    point) cut at `cut` scale radii: the enclosed mass r^3 / (r^2 + a^2)^1.5
    inverted."""
    u = _rand(g, n) * (cut * cut / (1.0 + cut * cut)) ** 1.5
    r = a / torch.sqrt(u.clamp_min(1e-30) ** (-2.0 / 3.0) - 1.0)
    z = 2.0 * _rand(g, n) - 1.0
    phi = 2.0 * math.pi * _rand(g, n)
    s = torch.sqrt(1.0 - z * z)
    return r[:, None] * torch.stack([s * torch.cos(phi), s * torch.sin(phi), z], 1)


def _cloud(cloud, n, seed):
    """float32 positions [n, 3] and masses [n] on the GPU. The clusters of a
    clustered cloud (64 Plummer spheres over 6 binary orders of scale radius,
    Dirichlet weights, 10 % uniform background) are the same for every seed;
    its particles are not."""
    g = _gen(seed)
    if cloud == "uniform":
        return (2.0 * _rand(g, n, 3) - 1.0).float(), (0.5 + _rand(g, n)).float()
    if cloud == "plummer":
        return _plummer(g, n, 1.0).float(), torch.full((n,), 1.0 / n, device="cuda")
    layout = np.random.Generator(np.random.PCG64(3))
    radii = torch.from_numpy(10.0 ** layout.uniform(-3.0, -1.0, 64)).cuda()
    centres = torch.from_numpy(layout.uniform(-1.0, 1.0, (64, 3))).cuda()
    edges = torch.from_numpy(np.cumsum(0.9 * layout.dirichlet(np.full(64, 0.5)))).cuda()
    u = _rand(g, n)
    k = torch.searchsorted(edges, u, right=True)
    inside = k < 64
    k = k.clamp(max=63)
    pos = torch.where(inside[:, None], centres[k] + _plummer(g, n, radii[k]),
                      2.0 * _rand(g, n, 3) - 1.0)
    mass = torch.exp(0.5 * torch.randn(n, generator=g, device="cuda"))
    return pos.float(), mass


def _weights(n):
    return torch.randint(-(1 << 31), 1 << 31, (n,), generator=_gen(7), device="cuda",
                         dtype=torch.int64).to(torch.int32)


def _tree(case, seed, octree=False):
    pos, mass = _cloud(case["cloud"], case["points"], seed)
    build = ygg.build_octree if octree else ygg.build_tree
    tree, pos, mass, _ = build(pos, mass, leaf_size=case["leaf"], return_reordered=True)
    return tree, pos, mass


def _far_list(tree, geom, theta, seed):
    """The tree's far list, the order inside its rows made from the seed."""
    inter, _ = ygg.build_interactions_and_neighbors(tree, geom, theta=theta, mac_type="dehnen",
                                                    neighbor_positions=False, strict_int32=False)
    T = tree.num_nodes
    rank = torch.empty(T, dtype=torch.int64, device="cuda")
    rank[tree.nodes_by_level] = torch.arange(T, device="cuda")
    mixed = torch.randperm(T, generator=_gen(seed), device="cuda")
    order = torch.argsort(rank[inter.targets] * T + mixed[inter.sources])
    return inter._replace(sources=inter.sources[order])


def _moved(pos, seed):
    """Positions some time after the tree was built."""
    return pos + 1e-4 * torch.randn(pos.shape, generator=_gen(seed), device="cuda")


def _systems(case, seed):
    """Plummer spheres of log-uniform size, scale radii 0.05 to 0.5."""
    layout = np.random.Generator(np.random.PCG64(4))
    sizes = np.rint(np.exp(layout.uniform(math.log(case["smallest"]), math.log(case["largest"]),
                                          case["systems"]))).astype(np.int64)
    radii = torch.from_numpy(np.repeat(layout.uniform(0.05, 0.5, case["systems"]), sizes)).cuda()
    offsets = np.concatenate([[0], np.cumsum(sizes)])
    pos = _plummer(_gen(seed), int(offsets[-1]), radii).float()
    mass = torch.from_numpy(np.repeat((1.0 / sizes).astype(np.float32), sizes)).cuda()
    return pos, mass, offsets


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "build"):
        pos, mass = _cloud(case["cloud"], case["points"], seed)
        leaves = -(-case["points"] // case["leaf"])
        state = {"case": case, "pos": pos, "mass": mass, "weights": _weights(2 * leaves)}
        if kind == "step":
            T = 2 * leaves - 1
            room = dict(dtype=torch.int32, device="cuda")
            state["room"] = {"targets": torch.zeros(T * min(T, FAR_ROOM), **room),
                             "target_levels": torch.zeros(T * min(T, FAR_ROOM), **room),
                             "level_offsets": torch.zeros(1025, **room)}
        return state
    if kind == "upward":
        # the tree is one for all seeds, the particles have moved since
        tree, pos, _ = _tree(case, 11)
        mass = torch.exp(0.5 * torch.randn(case["points"], generator=_gen(seed + 1),
                                           device="cuda", dtype=torch.float64))
        return {"case": case, "tree": tree, "pos": _moved(pos, seed),
                "mass": mass.to(getattr(torch, case["masses"]))}
    if kind in ("dense", "grouped"):
        # one tree and far list for all seeds: for the displacements the
        # particles have moved since, for the classes the rows are in another order
        tree, pos, _ = _tree(case, 11)
        geom = ygg.compute_tree_geometry(tree, pos)
        far = _far_list(tree, geom, case["theta"], seed)
        if kind == "dense":
            geom = ygg.compute_tree_geometry(tree, _moved(pos, seed))
        return {"case": case, "tree": tree, "geom": geom, "far": far}
    if kind == "batch":
        pos, mass, offsets = _systems(case, seed)
        state = {"case": case, "pos": pos, "mass": mass, "offsets": offsets}
        leaves = -(-np.diff(offsets) // case["leaf"])
        state["weights"] = _weights(2 * int(leaves.max()) - 1)
        # where each system's first and last offset lies in the lists' offsets
        last = np.cumsum(2 * leaves) - 1, np.cumsum(leaves + 1) - 1
        state["last"] = [torch.from_numpy(v).cuda() for v in last]
        state["rows"] = [torch.from_numpy(np.delete(np.arange(v[-1] + 1), v)).cuda() for v in last]
        state["system"] = [torch.from_numpy(np.repeat(np.arange(case["systems"]), v)).cuda()
                           for v in (2 * leaves - 1, leaves)]
        if case["graph"]:
            g = _gen(seed + 1)
            start = pos * (1.0 + 1e-3 * torch.randn(pos.shape, generator=g, device="cuda"))
            state["graph"] = batch.BatchedGraph(start, mass, offsets, leaf_size=case["leaf"],
                                                theta=case["theta"], mac_type="dehnen")
        return state
    if kind == "predict":
        tree, pos, _ = _tree(case, seed, octree=True)
        model = learned.CapacityModel.load()
        model.device_weights(pos.device)
        return {"case": case, "tree": tree, "geom": ygg.compute_tree_geometry(tree, pos),
                "model": model}
    g = _gen(seed)
    rows = case["rows"]
    # features in the range of those of real trees, counts of a Poisson process
    x = torch.rand((rows, 8), generator=g, device="cuda")
    rate = 4.0 * torch.rand((rows, 3), generator=g, device="cuda") ** 4
    y = torch.poisson(rate, generator=g)
    mask = (torch.rand((rows, 3), generator=g, device="cuda") > 0.25).float()
    return {"case": case, "x": x, "y": y, "mask": mask,
            "trainer": learned.Trainer(learned.init_params(int(seed) % 1000), rows)}


# ---- one pass --------------------------------------------------------------

def _whole(t):
    """Every tensor of a named tuple; 64-bit codes as signed words."""
    out = {}
    for name, v in zip(t._fields, t):
        if isinstance(v, torch.Tensor):
            out[name] = v.view(torch.int64) if v.dtype == torch.uint64 else v
        elif v is not None:
            out[name] = int(v)
    return out


def _row_sums(weights, entries, start, count):
    """Sum of the weights of each row's entries, modulo 2^32."""
    run = torch.empty(entries.numel() + 1, dtype=torch.int32, device=entries.device)
    run[0] = 0
    torch.cumsum(weights[entries], 0, dtype=torch.int32, out=run[1:])
    return run[start + count] - run[start]


def _run_step(s):
    c = s["case"]
    build = ygg.build_octree if c["octree"] else ygg.build_tree
    tree, pos, mass, inverse = build(s["pos"], s["mass"], leaf_size=c["leaf"],
                                     return_reordered=True)
    out = {"tree": _whole(tree.topology), "positions": pos, "masses": mass, "inverse": inverse}
    if c["kind"] == "build":
        return out
    geom = ygg.compute_tree_geometry(tree, pos)
    out["geometry"] = _whole(geom)
    small = c["points"] <= SMALL
    kw = {} if small else {"neighbor_positions": False, "strict_int32": False}
    if c["config"]:
        kw["traversal_config"] = ygg.DualTreeTraversalConfig(8192, 256, 2048, 2048)
    far, near = ygg.build_interactions_and_neighbors(tree, geom, theta=c["theta"],
                                                     mac_type=c["mac"], **kw)
    out["far"] = {"offsets": far.offsets, "counts": far.counts}
    for k, room in s["room"].items():
        v = getattr(far, k)
        room[:v.numel()].copy_(v)
        out["far"][k] = room
    out["near"] = {k: getattr(near, k) for k in ("offsets", "counts", "leaf_indices",
                                                 "particle_order_leaf_indices",
                                                 "particle_order_to_native_leaf")}
    T, L = tree.num_nodes, tree.num_leaves
    out["far_rows"] = _row_sums(s["weights"], far.sources, far.offsets[:T], far.counts)
    out["near_rows"] = _row_sums(s["weights"], near.neighbors, near.offsets[:L], near.counts)
    if small:  # rows of native leaf positions, -1 past the end
        out["near_positions"] = s["weights"][near.neighbor_leaf_positions + 1].sum(1)
    return out


def _run_batch(s):
    c = s["case"]
    if c["graph"]:
        trees, geom, lists = s["graph"].replay(s["pos"], s["mass"])
    else:
        trees = batch.build_octree_batched(s["pos"], s["mass"], s["offsets"],
                                           leaf_size=c["leaf"])
        geom = batch.compute_tree_geometry_batched(trees)
        lists = batch.build_interactions_and_neighbors_batched(trees, geom, c["theta"],
                                                               mac_type="dehnen")
    rad = ("parent", "left_child", "right_child", "node_ranges", "node_level", "nodes_by_level",
           "leaf_codes")
    octa = ("oct_parent", "oct_child_counts", "oct_valid_mask", "oct_node_codes",
            "oct_node_depths", "oct_nodes_by_level", "oct_leaf_mask", "oct_leaf_nodes",
            "radix_node_to_oct", "leaf_indices", "leaf_position")
    out = {"tree": {**{k: trees.rad[k] for k in rad}, **{k: trees.octa[k] for k in octa},
                    "codes": trees.sorted_codes, "permutation": trees.perm_local},
           "positions": trees.positions_sorted, "masses": trees.masses_sorted,
           "inverse": trees.inverse_permutation,
           "geometry": {k: getattr(geom, k) for k in ("center", "half_extent", "radius",
                                                      "max_extent")},
           "far": {"offsets": lists.far_offsets, "counts": lists.far_counts,
                   "level_offsets": lists.far_level_offsets},
           "near": {"offsets": lists.near_offsets, "counts": lists.near_counts}}
    # a graph's lists end before their buffers do
    far, near = lists.stats["far_total"], lists.stats["near_total"]
    for k, (entries, offsets, counts) in enumerate((
            (lists.sources[:far], lists.far_offsets, lists.far_counts),
            (lists.neighbors[:near], lists.near_offsets, lists.near_counts))):
        total = offsets[s["last"][k]]
        base = torch.cumsum(total, 0) - total
        start = base[s["system"][k]] + offsets[s["rows"][k]]
        out[("far_rows", "near_rows")[k]] = _row_sums(s["weights"], entries, start, counts)
    return out


def run(state):
    kind = state["case"]["kind"]
    if kind in ("step", "build"):
        return _run_step(state)
    if kind == "batch":
        return _run_batch(state)
    if kind == "upward":
        geom = ygg.compute_tree_geometry(state["tree"], state["pos"])
        levels = ygg.geometry_to_level_major(state["tree"], geom)
        moments = tree_moments.compute_tree_mass_moments(state["tree"], state["pos"],
                                                         state["mass"])
        return {"geometry": _whole(geom), "levels": _whole(levels), "moments": _whole(moments)}
    if kind == "dense":
        d = dense_interactions.densify_interactions(state["tree"], state["geom"], state["far"])
        return {"levels": _whole(d.geometry), "sources": d.m2l_sources, "counts": d.m2l_counts,
                "displacements": d.m2l_displacements, "mask": d.m2l_mask}
    if kind == "grouped":
        return _whole(grouped_interactions.build_grouped_interactions(
            state["tree"], state["geom"], state["far"]))
    if kind == "predict":
        return state["model"].predict_nodes(state["tree"], state["geom"])
    t = state["trainer"]
    t.step(state["x"], state["y"], state["mask"], 3e-3)
    return {"loss": t.loss, "gradients": t.g, "weights": t.p, "first": t.m, "second": t.v}


# ---- what a pass cannot do without ------------------------------------------

def _nbytes(v):
    if isinstance(v, dict):
        return sum(_nbytes(x) for x in v.values())
    return v.numel() * v.element_size() if isinstance(v, torch.Tensor) else 8


MLP_WEIGHTS = 8 * 64 + 64 * 64 + 64 * 64 + 64 * 3


def work(case):
    """Bytes of the inputs and of the outputs of a pass (the listed nodes of
    every row among them, whatever stands for them in the outputs), each once;
    the products of the layers of the model. The lengths of the lists depend
    on the particles, so they are taken from one pass."""
    state = prepare(case, 1)
    out = run(state)
    kind = case["kind"]
    if kind == "train":
        # every weight and moment read and written, the batch read
        return {"bytes": _nbytes(out) * 2 + case["rows"] * 14 * 4,
                "flops": 6.0 * MLP_WEIGHTS * case["rows"]}
    if kind == "predict":
        T = state["tree"].num_nodes
        # level, range, parent, child, box, radius and extent of each node
        return {"bytes": _nbytes(out) + T * 40, "flops": 2 * 2.0 * MLP_WEIGHTS * T}
    if kind in ("step", "build", "batch"):
        moved = _nbytes(state["pos"]) + _nbytes(state["mass"])
        if "far" in out:
            # sources, targets and their levels; neighbours
            moved += 24 * int(out["far"]["counts"].sum()) + 8 * int(out["near"]["counts"].sum())
        for k in state.get("room", ()):
            del out["far"][k]
        if "near_positions" in out:
            moved += 8 * int(out["near"]["counts"].max()) * out["near"]["counts"].numel()
        for k in ("far_rows", "near_rows", "near_positions"):
            out.pop(k, None)
        return {"bytes": moved + _nbytes(out), "flops": 0}
    if kind == "upward":
        T = state["tree"].num_nodes
        return {"bytes": _nbytes(state["pos"]) + _nbytes(state["mass"]) + 8 * T + _nbytes(out),
                "flops": 0}
    far = state["far"]
    read = _nbytes(far.sources) + (_nbytes(far.targets) if kind == "grouped" else
                                   _nbytes(far.counts) + _nbytes(far.offsets))
    return {"bytes": read + 12 * state["tree"].num_nodes + _nbytes(out), "flops": 0}


def tolerance(case):
    """Whole numbers are the same always; so are boxes, which are the least
    and largest coordinates. Mass moments are float64 sums rounded once.
    The model's layers take each activation as two bfloat16 parts (4e-5 off
    float64 as measured); the gradients are float32 sums over the rows of the
    batch, and an element of them near zero moves its weight by up to the
    learning rate."""
    kind = case["kind"]
    if kind in ("step", "build", "batch", "dense", "grouped"):
        return "exact"
    if kind == "upward":
        return {"rel": 4e-7}
    if kind == "predict":
        return {"rel": 1.5e-4}
    return {"rel": 4e-6, "max": 0.05}


# ---- the same in 64 bits -----------------------------------------------------

def _range_boxes(pos, first, last):
    """Least and largest coordinates of pos[first : last + 1] for many ranges,
    from tables of the minima over 2^k elements."""
    n = pos.shape[0]
    length = last - first + 1
    k_of = torch.log2(length.double()).floor().long()
    k_of = torch.where((1 << k_of) > length, k_of - 1, k_of)
    lo = torch.empty((first.numel(), 3), dtype=torch.float64, device=pos.device)
    hi = torch.empty_like(lo)
    a, b = pos, pos
    for k in range(int(k_of.max()) + 1):
        if k:
            h = 1 << (k - 1)
            a = torch.minimum(a[:-h], a[h:])
            b = torch.maximum(b[:-h], b[h:])
        i = (k_of == k).nonzero()[:, 0]
        p, q = first[i], last[i] + 1 - (1 << k)
        lo[i] = torch.minimum(a[p], a[q]).double()
        hi[i] = torch.maximum(b[p], b[q]).double()
    return lo, hi


def _geometry64(pos, first, last):
    lo, hi = _range_boxes(pos, first, last)
    half = (0.5 * (hi - lo)).clamp_min(1e-6)
    return {"center": 0.5 * (lo + hi), "half_extent": half,
            "radius": torch.sqrt((half * half).sum(1)), "max_extent": half.max(1)[0]}


def _levels64(tree, geom):
    counts = torch.diff(tree.level_offsets[: int(tree.num_levels) + 1])
    widest = int(counts.max())
    out = {}
    for name, field in (("centers", "center"), ("half_extents", "half_extent"),
                        ("radii", "radius"), ("max_extents", "max_extent")):
        v = geom[field].double()
        out[name] = torch.zeros((counts.numel(), widest, *v.shape[1:]), dtype=torch.float64,
                                device=v.device)
        for l, k in enumerate(counts.tolist()):
            at = int(tree.level_offsets[l])
            out[name][l, :k] = v[tree.nodes_by_level[at:at + k]]
    return out


def _range_sums(values, first, last):
    """Sums of values[first : last + 1], as differences of prefix sums that are
    exact: the terms as whole multiples of 2^-40 of the largest, in int64."""
    scale = 2.0 ** 38 / float(values.abs().max())
    total = torch.zeros((values.shape[0] + 1, *values.shape[1:]), dtype=torch.int64,
                        device=values.device)
    total[1:] = torch.cumsum(torch.round(values * scale).to(torch.int64), 0)
    return (total[last + 1] - total[first]).double() / scale


def _layers(p):
    out, at = [], 0
    for i, o in ((8, 64), (64, 64), (64, 64), (64, 3)):
        out.append((p[at:at + i * o].reshape(o, i), p[at + i * o:at + i * o + o]))
        at += i * o + o
    return out


def _bf16(p):
    return torch.as_tensor(p).cuda().bfloat16().double()


def _mlp64(layers, x):
    acts = [x]
    for k, (w, b) in enumerate(layers):
        x = x @ w.T + b
        x = x.clamp_min(0) if k < 3 else x
        acts.append(x)
    return acts


def _predict64(tree, geom, model):
    T, NI = tree.num_nodes, int(tree.num_internal_nodes)
    size = (tree.node_ranges[:, 1] - tree.node_ranges[:, 0] + 1).double()
    parent = tree.parent
    up = parent.clamp_min(0)
    node = torch.arange(T, device=parent.device)
    left, right = tree.left_child, tree.right_child
    sibling = torch.where(left[up] == node, right[up], left[up])
    sib = torch.where(parent >= 0, size[sibling], 0.0)
    half = geom.half_extent.double()
    ext, rad = geom.max_extent.double(), geom.radius.double()
    density = size / (8.0 * half.prod(1)).clamp_min(1e-30)
    x = torch.zeros((T, 8), dtype=torch.float64, device=parent.device)
    x[:, 0] = tree.node_level.double() / 64
    x[:, 1] = torch.log2(size) / 24
    x[:, 2] = torch.log2(ext / ext[0]) / 32 + 1
    x[:, 3] = torch.log2(rad / rad[0]) / 32 + 1
    x[:, 5] = torch.log2(1 + sib) / 24
    x[:, 6] = (torch.log2((density / density[0]).clamp_min(1e-30)) / 64).clamp(-1, 1)
    x[NI:, 7] = 1
    layers = _layers(_bf16(model.params))
    far = float(model.scale[0]) * torch.exp2(_mlp64(layers, x)[-1][:, 0].clamp_max(30))
    x[:, 4] = torch.log2(1 + torch.where(parent >= 0, far[up], 0.0)) / 16
    return _mlp64(layers, x)[-1]


def _train64(state, seed):
    start = torch.from_numpy(learned.init_params(int(seed) % 1000)).cuda()
    layers = _layers(_bf16(start))
    x, t, mask = (state[k].double() for k in ("x", "y", "mask"))
    acts = _mlp64(layers, x)
    y, ln2, rows = acts[-1], math.log(2.0), x.shape[0]
    yc = y.clamp_max(30)
    rate = torch.exp2(yc)
    loss = (mask * (rate - t * yc * ln2)).sum() / rows
    d = torch.where(y > 30, 0.0, mask * (rate - t) * ln2 / rows)
    grads = []
    for k in (3, 2, 1, 0):
        grads = [(d.T @ acts[k]).reshape(-1), d.sum(0)] + grads
        d = (d @ layers[k][0]) * (acts[k] > 0)
    g = torch.cat(grads)
    return {"loss": loss.reshape(1), "gradients": g,
            "weights": start.double() - 3e-3 * g / (g.abs() + 1e-8),
            "first": 0.1 * g, "second": 0.001 * g * g}


def _classes64(tree, geom, far):
    """Displacements of the classes of a far list, in the order of their keys."""
    extent = (tree.bounds_max.double() - tree.bounds_min.double())
    level = tree.node_level
    lt, ls = level[far.targets], level[far.sources]
    cell = (extent / torch.exp2(lt.double())[:, None]).clamp_min(1e-12)
    delta = geom.center[far.targets].double() - geom.center[far.sources].double()
    i = torch.round(delta / cell)
    if float(i.abs().max()) >= 2.0 ** 31:
        return None
    i = i.long()
    high = (lt * 4096 + ls << 32) + (i[:, 0] + (1 << 31))
    low = (i[:, 1] << 32) + (i[:, 2] + (1 << 31))
    order = torch.sort(low, stable=True)[1]
    order = order[torch.sort(high[order], stable=True)[1]]
    high, low = high[order], low[order]
    first = torch.ones_like(high, dtype=torch.bool)
    first[1:] = (high[1:] != high[:-1]) | (low[1:] != low[:-1])
    order = order[first]
    return i[order].double() * cell[order]


def _without(v):
    """The layout of an answer with no value that has one in 64 bits."""
    return {k: _without(x) for k, x in v.items()} if isinstance(v, dict) else None


def exact(case, seed):
    """Boxes, sums, displacements and the model in float64 from the same
    inputs (the tree's ranges, whole numbers, are an input here)."""
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "train":
        return _train64(state, seed)
    if kind == "predict":
        return _predict64(state["tree"], state["geom"], state["model"])
    if kind == "build":
        return None
    out = _without(run(state))
    if kind == "step":
        c = state["case"]
        build = ygg.build_octree if c["octree"] else ygg.build_tree
        tree, pos, _, _ = build(state["pos"], state["mass"], leaf_size=c["leaf"],
                                return_reordered=True)
        out["geometry"] = _geometry64(pos, *tree.node_ranges.long().T)
        return out
    if kind == "batch":
        trees = batch.build_octree_batched(state["pos"], state["mass"], state["offsets"],
                                           leaf_size=case["leaf"])
        base = torch.from_numpy(state["offsets"][:-1]).cuda()[state["system"][0]]
        first, last = (base + trees.rad["node_ranges"][:, k].long() for k in (0, 1))
        out["geometry"] = _geometry64(trees.positions_sorted, first, last)
        return out
    tree = state["tree"]
    if kind == "upward":
        first, last = tree.node_ranges.long().T
        geom = _geometry64(state["pos"], first, last)
        out["geometry"] = geom
        out["levels"].update(_levels64(tree, geom))
        mass = state["mass"]
        # m x is a product in the wider of the two types
        term = (mass[:, None] * state["pos"].to(mass.dtype)).double()
        total = _range_sums(mass.double(), first, last)
        out["moments"] = {"mass": total,
                          "center_of_mass": _range_sums(term, first, last) / total[:, None]}
        return out
    geom = state["geom"]
    if kind == "dense":
        out["levels"].update(_levels64(tree, {k: getattr(geom, k) for k in geom._fields}))
        far, lev = state["far"], int(tree.num_levels)
        counts = torch.diff(tree.level_offsets[: lev + 1])
        k = max(1, int(far.counts.max()))
        d = torch.zeros((lev * int(counts.max()), k, 3), dtype=torch.float64,
                        device=far.counts.device)
        slot = torch.empty(tree.num_nodes, dtype=torch.int64, device=d.device)
        for l, m in enumerate(counts.tolist()):
            at = int(tree.level_offsets[l])
            slot[tree.nodes_by_level[at:at + m]] = (l * int(counts.max())
                                                    + torch.arange(m, device=d.device))
        t = far.targets
        at = torch.arange(t.numel(), device=d.device) - far.offsets[t]
        d[slot[t], at] = geom.center[t].double() - geom.center[far.sources].double()
        out["displacements"] = d.reshape(lev, -1, k, 3)
        return out
    out["class_displacements"] = _classes64(tree, geom, state["far"])
    return out
