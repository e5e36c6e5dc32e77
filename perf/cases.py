"""Timed cases of the package's public operators: what a point-cloud network asks of it in training and inference.

A case is a dict of plain values; its "op" names the call pattern below, the other entries its sizes and options.
Every operator of the package has one listed case; `draw` gives further cases between the smallest and the largest
sizes these calls have in use, odd ones among them, and with the options the listed cases leave at their defaults.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "torch-points-kernels_amd"))
import torch_points_kernels as tpk  # noqa: E402

DEVICE = "cuda"


def listed():
    return [
        # A set-abstraction layer on two small clouds: sample centres, find their neighbours, group the features,
        # send a gradient back.  The smallest calls of all: launches and host work are what they cost.
        {"name": "set_abstraction_small", "op": "set_abstraction", "b": 2, "n": 1024, "npoint": 256, "nsample": 32,
         "c": 64, "cloud": "uniform"},
        # Down-sampling a batch of large, unevenly dense clouds (the package's headline workload).
        {"name": "sample_clusters", "op": "sample", "b": 16, "n": 16384, "npoint": 4096, "cloud": "clusters"},
        # Neighbourhoods in packed indoor scans of very different sizes: a kernel-point or sparse network's input.
        {"name": "ball_query_packed_scenes", "op": "ball_packed", "clouds": 4, "smallest": 20000, "largest": 100000,
         "query_share": 4, "radius": 0.05, "nsample": 64, "sort": False},
        # Feature propagation, first half: the three nearest known points of every point of the dense cloud.
        {"name": "three_nn_dense", "op": "three_nn", "b": 16, "n": 16384, "m": 4096, "cloud": "uniform"},
        # Feature propagation, second half: interpolation of the coarse features, with its gradient.
        {"name": "interpolate_dense", "op": "interpolate", "b": 16, "c": 128, "n": 16384, "m": 4096},
        # Grouping of features at neighbour indices, with its gradient.
        {"name": "group_features", "op": "group", "b": 16, "c": 128, "n": 4096, "npoint": 1024, "nsample": 32,
         "index": "uniform"},
        # Completion loss on a batch of surface scans, with the gradients of both clouds.
        {"name": "chamfer_surfaces", "op": "chamfer", "b": 32, "n": 16384, "m": 16384, "double": False},
        # Neighbour graph of a batch of clouds of odd size (every point's 16 nearest in its own cloud).
        {"name": "knn_graph", "op": "knn", "b": 8, "n": 4099, "m": 4099, "k": 16, "cloud": "uniform"},
        # Instance proposals of three rooms with objects of eight classes: region growing class by class.
        {"name": "region_grow_rooms", "op": "region_grow", "samples": 3, "n": 100000, "classes": 8, "objects": 24,
         "order": "reference"},
        # Scoring those proposals against the annotated instances.
        {"name": "instance_iou_proposals", "op": "instance_iou", "samples": 4, "n": 75000, "instances": 50,
         "proposals": 500, "size": 2000},
        # Grid completion: occupancy grids of a batch of padded clouds, with the gradient of the points ...
        {"name": "gridding_batch", "op": "gridding", "b": 32, "n": 2048, "scale": 32, "double": False},
        # ... and the features of the grid's vertices around every point, with the gradient of the maps.
        {"name": "cubic_sampling_batch", "op": "cubic", "b": 32, "n": 2048, "c": 64, "scale": 16, "neighborhood": 1},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["set_abstraction", "sample", "ball_dense", "ball_packed", "three_nn", "interpolate", "group",
                     "chamfer", "knn", "region_grow", "instance_iou", "gridding", "cubic"])
    cloud = rng.choice(["uniform", "clusters", "sphere"])
    if op == "set_abstraction":
        n = _log(rng, 512, 8192)
        return {"op": op, "b": _log(rng, 1, 16), "n": n, "npoint": max(16, n // rng.choice([2, 4, 8])),
                "nsample": rng.choice([16, 24, 32, 64]), "c": _log(rng, 3, 128), "cloud": cloud}
    if op == "sample":
        n = _log(rng, 256, 50000)
        return {"op": op, "b": _log(rng, 1, 16), "n": n, "npoint": max(16, min(4096, n // rng.choice([2, 4, 8, 16]))),
                "cloud": cloud}
    if op == "ball_dense":
        n = _log(rng, 512, 16384)
        return {"op": op, "b": _log(rng, 1, 16), "n": n, "m": max(32, n // rng.choice([1, 2, 4, 8])),
                "nsample": rng.choice([16, 32, 48, 64]), "sort": rng.random() < 0.3, "cloud": cloud}
    if op == "ball_packed":
        smallest = _log(rng, 2000, 20000)
        return {"op": op, "clouds": rng.randint(1, 4), "smallest": smallest, "largest": _log(rng, smallest, 100000),
                "query_share": rng.choice([1, 2, 4, 8]), "radius": round(rng.uniform(0.04, 0.1), 3),
                "nsample": rng.choice([16, 32, 64]), "sort": rng.random() < 0.3}
    if op == "three_nn":
        n = _log(rng, 256, 16384)
        return {"op": op, "b": _log(rng, 1, 16), "n": n, "m": max(16, n // rng.choice([1, 2, 4, 8, 16])), "cloud": cloud}
    if op == "interpolate":
        n = _log(rng, 256, 16384)
        return {"op": op, "b": _log(rng, 1, 16), "c": _log(rng, 16, 512) if n <= 4096 else _log(rng, 16, 128), "n": n,
                "m": max(16, n // rng.choice([2, 4, 8, 16]))}
    if op == "group":
        n = _log(rng, 256, 4096)
        return {"op": op, "b": _log(rng, 1, 16), "c": _log(rng, 3, 128), "n": n, "npoint": max(16, n // rng.choice([2, 4, 8])),
                "nsample": rng.choice([16, 20, 32]), "index": rng.choice(["uniform", "ball"])}
    if op == "chamfer":
        double = rng.random() < 0.2
        n = _log(rng, 256, 2048 if double else 16384)
        return {"op": op, "b": _log(rng, 1, 32), "n": n, "m": rng.choice([n, n, max(128, n // 2), max(128, (2 * n) // 3)]),
                "double": double}
    if op == "knn":
        n = _log(rng, 256, 16384)
        return {"op": op, "b": _log(rng, 1, 8), "n": n, "m": max(64, n // rng.choice([1, 1, 2, 4])),
                "k": rng.choice([4, 8, 16, 20, 32]), "cloud": cloud}
    if op == "region_grow":
        return {"op": op, "samples": rng.randint(1, 3), "n": _log(rng, 4000, 100000), "classes": rng.randint(1, 12),
                "objects": rng.randint(12, 40), "order": rng.choice(["reference", "reference", "index"])}
    if op == "instance_iou":
        return {"op": op, "samples": rng.randint(1, 4), "n": _log(rng, 4000, 75000), "instances": rng.randint(5, 60),
                "proposals": _log(rng, 10, 500), "size": _log(rng, 100, 2000)}
    if op == "gridding":
        scale = rng.choice([16, 32, 32, 64])
        return {"op": op, "b": _log(rng, 1, 32 if scale < 64 else 8), "n": _log(rng, 512, 16384), "scale": scale,
                "double": rng.random() < 0.15}
    return {"op": op, "b": _log(rng, 1, 32), "n": _log(rng, 256, 2048), "c": rng.choice([16, 32, 64, 33]),
            "scale": rng.choice([8, 12, 16]), "neighborhood": 1}


# ---- inputs ----------------------------------------------------------------------------------------------------

def _clouds(kind, b, n, g):
    """(b, n, 3): uniform in the unit cube; 8 Gaussian clusters over a thin background; or a noisy unit sphere."""
    if kind == "uniform":
        return torch.rand(b, n, 3, generator=g, device=DEVICE)
    if kind == "sphere":
        p = torch.randn(b, n, 3, generator=g, device=DEVICE)
        return p / p.norm(dim=2, keepdim=True) + 0.02 * torch.randn(b, n, 3, generator=g, device=DEVICE)
    centres = torch.rand(b, 8, 3, generator=g, device=DEVICE)
    which = torch.randint(0, 8, (b, n, 1), generator=g, device=DEVICE).expand(-1, -1, 3)
    p = torch.gather(centres, 1, which) + 0.05 * torch.randn(b, n, 3, generator=g, device=DEVICE)
    background = torch.rand(b, n, 1, generator=g, device=DEVICE) < 0.1
    return torch.where(background, torch.rand(b, n, 3, generator=g, device=DEVICE), p).contiguous()


def _radius(kind, n, neighbours):
    """A radius that holds about this many points of such a cloud of n."""
    if kind == "sphere":
        return 2.0 * math.sqrt(neighbours / n)
    density = n if kind == "uniform" else n * 20.0
    return (neighbours / (density * 4.19)) ** (1.0 / 3.0)


def _scene(n, g):
    """One indoor scan of an 8 m room: points of 6 axis-aligned planes, a fifth of them spread over the room."""
    p = 8.0 * torch.rand(n, 3, generator=g, device=DEVICE)
    axis = torch.randint(0, 3, (6,), generator=g, device=DEVICE)
    offset = 8.0 * torch.rand(6, generator=g, device=DEVICE)
    which = torch.randint(0, 6, (n,), generator=g, device=DEVICE)
    off_plane = offset[which] + 0.01 * torch.randn(n, generator=g, device=DEVICE)
    flat = p.scatter(1, axis[which].unsqueeze(1), off_plane.unsqueeze(1))
    return torch.where(torch.rand(n, 1, generator=g, device=DEVICE) < 0.2, p, flat).contiguous()


def _rooms(case, g):
    """Rooms whose points lie on the sides of boxes (the objects), in no order; a class per object."""
    n, objects = case["n"], case["objects"]
    pos, labels = [], []
    for _ in range(case["samples"]):
        centre = torch.rand(objects, 3, generator=g, device=DEVICE) * torch.tensor([8.0, 8.0, 3.0], device=DEVICE)
        extent = 0.3 + 1.2 * torch.rand(objects, 3, generator=g, device=DEVICE)
        kind = torch.randint(0, case["classes"], (objects,), generator=g, device=DEVICE)
        which = torch.randint(0, objects, (n,), generator=g, device=DEVICE)
        p = torch.rand(n, 3, generator=g, device=DEVICE) - 0.5
        side = torch.randint(0, 3, (n, 1), generator=g, device=DEVICE)
        p = p.scatter(1, side, torch.sign(torch.rand(n, 1, generator=g, device=DEVICE) - 0.5) * 0.5)
        p = p * extent[which] + centre[which] + 0.004 * torch.randn(n, 3, generator=g, device=DEVICE)
        pos.append(p)
        labels.append(kind[which])
    batch = torch.arange(case["samples"], device=DEVICE).repeat_interleave(n)
    return torch.cat(pos).contiguous(), torch.cat(labels), batch


def _packed_sizes(case):
    k = case["clouds"]
    step = (case["largest"] / case["smallest"]) ** (1.0 / max(1, k - 1))
    return [int(case["smallest"] * step ** i) for i in range(k)] if k > 1 else [case["largest"]]


def prepare(case, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    op = case["op"]
    s = {"case": case}
    if op == "set_abstraction":
        s["xyz"] = _clouds(case["cloud"], case["b"], case["n"], g)
        s["features"] = torch.randn(case["b"], case["c"], case["n"], generator=g, device=DEVICE).requires_grad_()
        s["grad"] = torch.randn(case["b"], case["c"], case["npoint"], case["nsample"], generator=g, device=DEVICE)
        s["radius"] = _radius(case["cloud"], case["n"], 0.8 * case["nsample"])
    elif op == "sample":
        s["xyz"] = _clouds(case["cloud"], case["b"], case["n"], g)
    elif op == "ball_dense":
        s["xyz"] = _clouds(case["cloud"], case["b"], case["n"], g)
        s["centres"] = s["xyz"][:, : case["m"]].contiguous()
        s["radius"] = _radius(case["cloud"], case["n"], 0.8 * case["nsample"])
    elif op == "ball_packed":
        x, y, bx, by = [], [], [], []
        for i, n in enumerate(_packed_sizes(case)):
            cloud = _scene(n, g)
            q = torch.sort(torch.randperm(n, generator=g, device=DEVICE)[: n // case["query_share"]]).values
            x.append(cloud)
            y.append(cloud[q])
            bx.append(torch.full((n,), i, dtype=torch.int64, device=DEVICE))
            by.append(torch.full((q.numel(),), i, dtype=torch.int64, device=DEVICE))
        s["x"], s["y"], s["batch_x"], s["batch_y"] = (torch.cat(v).contiguous() for v in (x, y, bx, by))
    elif op == "three_nn":
        s["unknown"] = _clouds(case["cloud"], case["b"], case["n"], g)
        # the coarse cloud is a subset of the dense one, as sampling leaves it, or a scan of its own
        s["known"] = _clouds(case["cloud"], case["b"], case["m"], g) if case["cloud"] == "uniform" else s["unknown"][:, : case["m"]].contiguous()
    elif op == "interpolate":
        dist, s["idx"] = tpk.three_nn(_clouds("uniform", case["b"], case["n"], g), _clouds("uniform", case["b"], case["m"], g))
        near = 1.0 / (dist + 1e-8)
        s["weight"] = (near / near.sum(dim=2, keepdim=True)).contiguous()
        s["features"] = torch.randn(case["b"], case["c"], case["m"], generator=g, device=DEVICE).requires_grad_()
        s["grad"] = torch.randn(case["b"], case["c"], case["n"], generator=g, device=DEVICE)
    elif op == "group":
        shape = (case["b"], case["npoint"], case["nsample"])
        if case["index"] == "uniform":
            s["idx"] = torch.randint(0, case["n"], shape, generator=g, device=DEVICE)
        else:
            xyz = _clouds("uniform", case["b"], case["n"], g)
            radius = _radius("uniform", case["n"], 0.8 * case["nsample"])
            s["idx"] = tpk.ball_query(radius, case["nsample"], xyz, xyz[:, : case["npoint"]].contiguous())[0]
        s["features"] = torch.randn(case["b"], case["c"], case["n"], generator=g, device=DEVICE).requires_grad_()
        s["grad"] = torch.randn(case["b"], case["c"], case["npoint"], case["nsample"], generator=g, device=DEVICE)
    elif op == "chamfer":
        p = _clouds("sphere", case["b"], max(case["n"], case["m"]), g)
        q = p[:, :, [1, 2, 0]] * torch.tensor([1.0, -1.0, -1.0], device=DEVICE)  # a rotation
        jittered = torch.rand(*q.shape[:2], 1, generator=g, device=DEVICE) < 0.05
        q = torch.where(jittered, q + 0.1 * torch.randn(q.shape, generator=g, device=DEVICE), q)
        kind = torch.float64 if case["double"] else torch.float32
        s["xyz1"] = p[:, : case["n"]].to(kind).contiguous().requires_grad_()
        s["xyz2"] = q[:, : case["m"]].to(kind).contiguous().requires_grad_()
    elif op == "knn":
        s["support"] = _clouds(case["cloud"], case["b"], case["n"], g)
        s["queries"] = s["support"][:, : case["m"]].contiguous()
    elif op == "region_grow":
        s["pos"], s["labels"], s["batch"] = _rooms(case, g)
        s["radius"] = 0.06 * math.sqrt(case["objects"] / 24 * 1e5 / case["n"])
    elif op == "instance_iou":
        n, total = case["n"], case["n"] * case["samples"]
        s["batch"] = torch.arange(case["samples"], device=DEVICE).repeat_interleave(n)
        s["gt"] = torch.randint(0, case["instances"] + 1, (total,), generator=g, device=DEVICE)
        s["gt"][::n] = case["instances"]  # every instance number occurs in every sample's range
        rows = torch.randint(0, n, (case["proposals"], case["size"]), generator=g, device=DEVICE)
        cut = torch.randint(case["size"] // 2, case["size"] + 1, (case["proposals"],), generator=g, device=DEVICE).tolist()
        s["proposals"] = [rows[p, : cut[p]] + n * (p % case["samples"]) for p in range(case["proposals"])]
    elif op == "gridding":
        kind = torch.float64 if case["double"] else torch.float32
        p = (_clouds("sphere", case["b"], case["n"], g) * 0.7).clamp(-0.99, 0.99)
        filled = torch.randint((7 * case["n"]) // 8, case["n"] + 1, (case["b"], 1), generator=g, device=DEVICE)
        p = torch.where((torch.arange(case["n"], device=DEVICE) < filled).unsqueeze(2), p, torch.zeros_like(p))  # padding
        s["cloud"] = p.to(kind).contiguous().requires_grad_()
        s["grad"] = torch.randn(case["b"], (2 * case["scale"]) ** 3, generator=g, device=DEVICE, dtype=kind)
    else:
        c, m = case["c"], case["scale"]
        s["cloud"] = (_clouds("sphere", case["b"], case["n"], g) * 0.7).clamp(-0.99, 0.99).contiguous()
        s["maps"] = torch.randn(case["b"], c, m, m, m, generator=g, device=DEVICE).requires_grad_()
        s["grad"] = torch.randn(case["b"], case["n"], (2 * case["neighborhood"]) ** 3, c, generator=g, device=DEVICE)
    return s


# ---- one pass --------------------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    op = case["op"]
    if op == "set_abstraction":
        sampled = tpk.furthest_point_sample(s["xyz"], case["npoint"])
        centres = torch.gather(s["xyz"], 1, sampled.long().unsqueeze(2).expand(-1, -1, 3))
        idx, dist = tpk.ball_query(s["radius"], case["nsample"], s["xyz"], centres)
        grouped = tpk.grouping_operation(s["features"], idx)
        return sampled, idx, dist, grouped, torch.autograd.grad(grouped, s["features"], s["grad"])[0]
    if op == "sample":
        return tpk.furthest_point_sample(s["xyz"], case["npoint"])
    if op == "ball_dense":
        return tpk.ball_query(s["radius"], case["nsample"], s["xyz"], s["centres"], sort=case["sort"])
    if op == "ball_packed":
        return tpk.ball_query(case["radius"], case["nsample"], s["x"], s["y"], mode="partial_dense", batch_x=s["batch_x"],
                              batch_y=s["batch_y"], sort=case["sort"])
    if op == "three_nn":
        return tpk.three_nn(s["unknown"], s["known"])
    if op == "interpolate":
        out = tpk.three_interpolate(s["features"], s["idx"], s["weight"])
        return out, torch.autograd.grad(out, s["features"], s["grad"])[0]
    if op == "group":
        out = tpk.grouping_operation(s["features"], s["idx"])
        return out, torch.autograd.grad(out, s["features"], s["grad"])[0]
    if op == "chamfer":
        loss = tpk.chamfer_dist.chamfer_dist(s["xyz1"], s["xyz2"])
        return (loss,) + torch.autograd.grad(loss, (s["xyz1"], s["xyz2"]))
    if op == "knn":
        return tpk.knn(s["support"], s["queries"], case["k"])
    if op == "region_grow":
        clusters = tpk.region_grow(s["pos"], s["labels"], s["batch"], radius=s["radius"], member_order=case["order"])
        # a network takes its proposals as one index and their sizes, here padded to what the room could hold
        members = torch.cat(clusters) if clusters else s["labels"].new_empty(0)
        sizes = np.zeros(s["pos"].shape[0] // 32, dtype=np.int64)
        sizes[: len(clusters)] = [c.shape[0] for c in clusters]
        return torch.nn.functional.pad(members, (0, s["pos"].shape[0] - members.shape[0]), value=-1), sizes
    if op == "instance_iou":
        return tpk.instance_iou(s["proposals"], s["gt"], s["batch"])
    if op == "gridding":
        grid = tpk.gridding(s["cloud"], case["scale"])
        return grid, torch.autograd.grad(grid, s["cloud"], s["grad"])[0]
    sampled = tpk.cubic_feature_sampling(s["cloud"], s["maps"], case["neighborhood"])
    return sampled, torch.autograd.grad(sampled, s["maps"], s["grad"])[0]


# ---- what a pass cannot do without -----------------------------------------------------------------------------

def work(case):
    """Bytes of the inputs and outputs, each once, and the arithmetic of the results themselves (a distance is 8
    operations): a search is not charged for the pairs that it can rule out."""
    op = case["op"]
    b, n, c = case.get("b", 1), case.get("n", 0), case.get("c", 1)
    if op == "set_abstraction":
        slots = b * case["npoint"] * case["nsample"]
        return {"bytes": 12 * b * n + 4 * b * case["npoint"] + 20 * slots + 8 * b * c * n + 8 * c * slots,
                "flops": 10 * b * n + 8 * slots + c * slots}
    if op == "sample":
        return {"bytes": 12 * b * n + 4 * b * case["npoint"], "flops": 10 * b * n}
    if op == "ball_dense":
        slots = b * case["m"] * case["nsample"]
        return {"bytes": 12 * b * (n + case["m"]) + 12 * slots, "flops": 8 * slots}
    if op == "ball_packed":
        points = sum(_packed_sizes(case))
        queries = sum(k // case["query_share"] for k in _packed_sizes(case))
        return {"bytes": 20 * (points + queries) + 12 * queries * case["nsample"], "flops": 8 * queries * case["nsample"]}
    if op == "three_nn":
        return {"bytes": 12 * b * (n + case["m"]) + 24 * b * n, "flops": 27 * b * n}
    if op == "interpolate":
        return {"bytes": 8 * b * c * (n + case["m"]) + 24 * b * n, "flops": 12 * b * c * n}
    if op == "group":
        slots = b * case["npoint"] * case["nsample"]
        return {"bytes": 8 * b * c * (n + case["npoint"] * case["nsample"]) + 8 * slots, "flops": c * slots}
    if op == "chamfer":
        size = 8 if case["double"] else 4
        return {"bytes": 6 * size * b * (n + case["m"]) + size, "flops": 20 * b * (n + case["m"])}
    if op == "knn":
        return {"bytes": 12 * b * (n + case["m"]) + 12 * b * case["m"] * case["k"], "flops": 8 * b * case["m"] * case["k"]}
    if op == "region_grow":
        points = case["samples"] * n
        return {"bytes": 36 * points, "flops": 8 * 8 * points}
    if op == "instance_iou":
        return {"bytes": 16 * case["samples"] * n + 6 * case["proposals"] * case["size"]
                + 4 * case["proposals"] * case["samples"] * case["instances"],
                "flops": case["proposals"] * (case["size"] + 3 * case["instances"])}
    if op == "gridding":
        size = 8 if case["double"] else 4
        return {"bytes": size * b * (6 * n + 2 * (2 * case["scale"]) ** 3), "flops": 100 * b * n}
    slots = b * n * (2 * case["neighborhood"]) ** 3
    return {"bytes": 12 * b * n + 8 * b * c * case["scale"] ** 3 + 8 * c * slots, "flops": c * slots}


def tolerance(case):
    """Indices, counts and copies are exact, and so are squared distances, which round every operation on its own;
    sums of 32-bit terms may be formed in another order."""
    if case["op"] in ("sample", "ball_dense", "ball_packed", "knn", "region_grow"):
        return "exact"
    if case["op"] in ("three_nn", "instance_iou"):
        return {"rel": 1e-6}
    if case.get("double"):
        return {"rel": 1e-12}
    return {"rel": 1e-5}
