"""The work that users of this package have it do, as a list of cases that can be timed and compared.

Kinds of cases (every size is a plain value of the case):
  stack      `layers` x [SubmanifoldConvolution(3) + BatchNormReLU] on a voxel scene whose rulebook is in hand
  structure  InputLayer (mode 4) and the 3^3 and stride-2 rulebooks of `levels` scales, from host coordinates
  unet       full forward of the U-Net (InputLayer .. OutputLayer, classifier), points on the GPU
  session    a full forward over the first part of a scene, then `frames` incremental frames of a sensor sweep
  residual   one residual frame (reference-style increment) against a saved scene
  labels     label fusion: two frames of class scores folded into an empty table, then the labels of one of them
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("ins-conv_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

CLASSES = 20


def listed():
    return [
        # one narrow layer on a small scene: a launch or two, latency
        {"name": "ssc_16_20k", "kind": "stack", "n": 20000, "c": 16, "layers": 1},
        # the layer stacks of the benchmark: bandwidth (32 channels) and matrix cores (64)
        {"name": "stack_32_500k", "kind": "stack", "n": 500000, "c": 32, "layers": 4},
        {"name": "stack_64_500k", "kind": "stack", "n": 500000, "c": 64, "layers": 4},
        # a width between the scales of the benchmark's network and a ragged number of sites
        {"name": "stack_48_60011", "kind": "stack", "n": 60011, "c": 48, "layers": 4},
        # a scan becomes a sparse tensor: hash grid, both rulebooks of every scale, per-voxel mean of the colours
        {"name": "structure_220k", "kind": "structure", "n": 200000, "dup": 0.1, "levels": 5, "c": 3},
        # a small network on one object: every layer is a short launch
        {"name": "unet_m16_6k", "kind": "unet", "n": 6000, "m": 16, "levels": 4, "dup": 0.1, "batch": 1},
        # two rooms in one batch, ragged
        {"name": "unet_m16_batch2_37k", "kind": "unet", "n": 37001, "m": 16, "levels": 5, "dup": 0.07, "batch": 2},
        # the benchmark's network on a room, and on the largest scene it is used on
        {"name": "unet_m32_150k", "kind": "unet", "n": 150000, "m": 32, "levels": 7, "dup": 0.1, "batch": 1},
        {"name": "unet_m32_500k", "kind": "unet", "n": 500000, "m": 32, "levels": 7, "dup": 0.1, "batch": 1},
        # a scanning session: full pass, then frames as the sensor moves on (host coordinates, as scanners deliver them)
        {"name": "session_150k", "kind": "session", "n": 150000, "m": 32, "levels": 7, "frames": 6, "new": 3000, "old": 1500},
        # the approximate kind of incremental frame, against a saved scene of 148k voxels
        {"name": "residual_150k", "kind": "residual", "n": 150000, "m": 32, "levels": 7, "new": 2200, "old": 1500},
        # what follows the network in a mapping program: fusing its labels per voxel
        {"name": "labels_220k", "kind": "labels", "n": 200000, "dup": 0.1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["stack", "stack", "structure", "unet", "unet", "session", "residual", "labels"])
    if kind == "stack":
        c = rng.choice([16, 32, 48, 64, 96, 128])
        return {"kind": kind, "n": _log(rng, 2000, min(500000, 500000 * 64 // c)), "c": c, "layers": rng.randint(1, 4)}
    if kind == "structure":
        return {"kind": kind, "n": _log(rng, 2000, 200000), "dup": rng.choice([0.0, 0.1, 0.5]), "levels": rng.randint(2, 6), "c": rng.choice([1, 3, 6, 32])}
    if kind == "labels":
        return {"kind": kind, "n": _log(rng, 2000, 200000), "dup": rng.choice([0.0, 0.1, 0.5])}
    m, levels = rng.choice([(16, 3), (16, 4), (16, 5), (32, 5), (32, 7)])
    if kind == "unet":
        return {"kind": kind, "n": _log(rng, 3000, 400000), "m": m, "levels": levels, "dup": rng.choice([0.0, 0.1]), "batch": rng.choice([1, 1, 2, 3])}
    case = {"kind": kind, "n": _log(rng, 20000, 150000), "m": m, "levels": levels}
    if kind == "session":
        case["frames"] = rng.randint(2, 6)
    most = case["n"] // 4 // case.get("frames", 1)
    case["new"] = _log(rng, 300, min(5000, most))
    case["old"] = _log(rng, 100, 2000)
    return case


# ---- scenes -----------------------------------------------------------------------------------
def _sheet(a, b):
    ga, gb = np.meshgrid(a, b, indexing="ij")
    return ga.ravel(), gb.ravel()


def _room(rng, n):
    """Exactly `n` distinct voxels of a room - floor, four walls, boxes on the floor, surfaces bent by up to a
    voxel - in the proportions of the benchmark's room, in scan order (distance from a corner)."""
    s = math.sqrt(n / 150000.0)
    dx, dy, dz = max(12, int(270 * s)), max(12, int(220 * s)), max(8, int(80 * s))
    xs, ys, zs = np.arange(dx), np.arange(dy), np.arange(1, dz)
    parts, normal = [], []

    def face(axis, at, a, b):
        p = np.empty((len(a) * len(b), 3), np.int64)
        i, j = [k for k in range(3) if k != axis]
        p[:, i], p[:, j] = _sheet(a, b)
        p[:, axis] = at
        parts.append(p)
        normal.append(np.full(len(p), axis))

    face(2, 0, xs, ys)
    for at in (0, dx - 1):
        face(0, at, ys, zs)
    for at in (0, dy - 1):
        face(1, at, xs, zs)
    have, lo_side, hi_side = sum(len(p) for p in parts), max(3, int(15 * s)), max(5, int(60 * s))
    while True:
        side = np.minimum(rng.integers(lo_side, hi_side, 3), [dx - 4, dy - 4, dz - 3])
        lo = np.array([rng.integers(2, dx - side[0] - 1), rng.integers(2, dy - side[1] - 1), 1])
        r = [np.arange(lo[k], lo[k] + side[k]) for k in range(3)]
        for axis in range(3):
            a, b = [r[k] for k in range(3) if k != axis]
            for at in (lo[axis], lo[axis] + side[axis] - 1):
                face(axis, at, a, b)
        have += 2 * int(side[0] * side[1] + side[1] * side[2] + side[0] * side[2])
        if have < 1.15 * n:
            continue
        p, ax = np.concatenate(parts), np.concatenate(normal)
        ph = rng.uniform(0, 6.28, 3)
        wave = np.sin(p[:, 0] * 0.11 + ph[0]) + np.sin(p[:, 1] * 0.13 + ph[1]) + np.sin(p[:, 2] * 0.17 + ph[2])
        q = p + 1024
        q[np.arange(len(q)), ax] += np.where(wave > 1.0, 1, np.where(wave < -1.0, -1, 0))
        key = (q[:, 0] << 32) | (q[:, 1] << 16) | q[:, 2]
        _, first = np.unique(key, return_index=True)
        if len(first) >= n:
            q = q[np.sort(first)[:n]]
            d = ((q - np.array([1044, 1044, 1054])) ** 2).sum(1)
            return q[np.argsort(d, kind="stable")]
        have = int(len(first) * have / len(p))  # boxes overlap: more of them


def _points(rng, vox, dup):
    """The voxels and repeated observations of some of them, in random order."""
    idx = np.concatenate([np.arange(len(vox)), rng.integers(0, len(vox), int(dup * len(vox)))])
    return vox[rng.permutation(idx)]


def _sweep(rng, case):
    """Frame 0: the scene up to the frames' new voxels; each later frame the next `new` voxels along the sweep
    and `old` re-observed ones."""
    vox, frames = _room(rng, case["n"]), case.get("frames", 1)
    seen = len(vox) - frames * case["new"]
    out = [vox[rng.permutation(seen)]]
    for _ in range(frames):
        idx = np.concatenate([np.arange(seen, seen + case["new"]), rng.integers(0, seen, case["old"])])
        out.append(vox[rng.permutation(idx)])
        seen += case["new"]
    return out


def _colours(rng, n, c=3):
    return torch.from_numpy(rng.random((n, c), np.float32)).cuda()


# ---- state in hand before the call --------------------------------------------------------------
def _network(case, seed, residual=False):
    import sparseconvnet as scn
    from workloads.netdefs import NaiveUNet

    model = NaiveUNet(m=case["m"], levels=case["levels"], seed=seed % 1000, classes=CLASSES).cuda()
    points = int(1.2 * case["n"])
    net = scn.compile(model.sparseModel, capacity_sites=max(1 << 18, 2 * points), residual=residual)
    return model, net


def prepare(case, seed):
    import sparseconvnet as scn

    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = {"kind": kind, "case": dict(case)}
    if kind == "stack":
        c, n = case["c"], case["n"]
        vox = _room(rng, n)[rng.permutation(n)]
        g = torch.Generator(device="cuda").manual_seed(seed)
        feats = torch.randn((n, c), generator=g, device="cuda")
        s["x"] = scn.InputLayer(3, 4096, mode=4)([torch.from_numpy(vox), feats, 1])
        s["x"].features = s["x"].features.clone()
        torch.manual_seed(seed)
        s["net"] = scn.Sequential()
        for _ in range(case["layers"]):
            s["net"].add(scn.SubmanifoldConvolution(3, c, c, 3, False))
            bn = scn.BatchNormReLU(c)
            bn.running_mean.normal_(0, 1)
            bn.running_var.uniform_(0.5, 2.0)
            s["net"].add(bn)
        s["net"] = s["net"].cuda().eval()
        s["x"].metadata.ssc_plan(s["x"].metadata.ssc_rulebook(s["x"].spatial_size))
    elif kind == "structure":
        # (one room per size, scanned in another order by every seed: the coarser scales hold a fixed number of sites)
        pts = _points(rng, _room(np.random.default_rng(case["n"]), case["n"]), case["dup"])
        s["coords"] = torch.from_numpy(pts)
        s["feats"] = _colours(rng, len(pts), case["c"])
        s["layer"] = scn.InputLayer(3, 4096, mode=4)
        s["sizes"] = [torch.LongTensor([4096 >> l] * 3) for l in range(case["levels"])]
    elif kind == "unet":
        s["batch"] = b = case["batch"]
        rooms = [_points(rng, _room(rng, case["n"] // b), case["dup"]) for _ in range(b)]
        pts = np.concatenate(rooms)
        if b > 1:
            pts = np.concatenate([pts, np.repeat(np.arange(b), [len(r) for r in rooms])[:, None]], 1)
            pts = pts[rng.permutation(len(pts))]
        s["coords"] = torch.from_numpy(pts.astype(np.int32)).cuda()
        s["feats"] = _colours(rng, len(pts))
        s["model"], s["net"] = _network(case, seed)
    elif kind in ("session", "residual"):
        frames = _sweep(rng, case)
        s["frames"] = [[torch.from_numpy(p), _colours(rng, len(p)), 1] for p in frames]
        s["model"], s["net"] = _network(case, seed, residual=kind == "residual")
        if kind == "residual":
            with torch.no_grad():
                s["net"](s["frames"][0], increment=False)
    else:
        vox = _room(rng, case["n"])
        s["frames"] = []
        for _ in range(2):
            pts = _points(rng, vox, case["dup"])
            score = torch.softmax(3 * torch.from_numpy(rng.standard_normal((len(pts), CLASSES), np.float32)).cuda(), 1)
            s["frames"].append((torch.from_numpy(pts).cuda(), score))
        s["table"] = scn.SCN.Result_3()
    return s


# ---- one pass ---------------------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    with torch.no_grad():
        if kind == "stack":
            return state["net"](state["x"]).features
        if kind == "structure":
            x = state["layer"]([state["coords"], state["feats"], 1])
            m, sizes = x.metadata, state["sizes"]
            out = [x.features]
            for fine, coarse in zip(sizes, sizes[1:] + [None]):
                sc = m.ssc_rulebook(fine)
                # (coords_view is memory of the grid, which goes away with its Metadata: the program keeps a copy)
                out += [sc.coords_view().clone(), sc.nbr.t[:sc.n]]
                if coarse is not None:
                    _, c, d = m.down_rulebook(fine, coarse)
                    out += [d.parent.t[:sc.n], d.offset.t[:sc.n], d.child.t[:c.n]]
            return out
        if kind == "unet":
            return state["model"].linear(state["net"]([state["coords"], state["feats"], state["batch"]], increment=False))
        if kind == "session":
            return [state["model"].linear(state["net"](f, increment=i > 0)) for i, f in enumerate(state["frames"])]
        if kind == "residual":
            return state["model"].linear(state["net"](state["frames"][1], increment="residual"))
        table = state["table"]
        table.clear()
        for pts, score in state["frames"]:
            table.update(pts, score)
        return table.multiQuery(state["frames"][0][0])


# ---- what a pass cannot do without ----------------------------------------------------------------------
_RULES = 9.0  # occupied cells in the 3^3 neighbourhood of a voxel on a surface, itself included
_SHRINK = 0.262  # sites of a scale per site of the next finer one


def _unet(n, m, levels):
    """(flops, weight floats) of the U-Net on n sites: the 3^3 layers, strided layers and shortcuts of every scale."""
    flops = weights = 0.0
    sites = [n * _SHRINK ** l for l in range(levels)]
    for l, k in enumerate(sites):
        w = m * (l + 1)
        below = m * (l + 2)
        ssc = [(w, w)] * 4 + ([(3, w)] if l == 0 else [])
        if l + 1 < levels:
            ssc += [(2 * w, w)] + [(w, w)] * 3
            flops += 2 * k * 2 * w * below + 2 * k * 2 * w * w  # strided down and up; 1x1 shortcut
            weights += 2 * 8 * w * below + 2 * w * w
        for a, b in ssc:
            flops += 2 * _RULES * k * a * b
            weights += 27 * a * b
    return flops, weights


def work(case):
    kind, n = case["kind"], case["n"]
    if kind == "stack":
        c, layers = case["c"], case["layers"]
        return {"bytes": 4.0 * (2 * n * c + layers * 27 * c * c + 27 * n), "flops": 2.0 * _RULES * n * c * c * layers}
    points = n * (1 + case.get("dup", 0.0))
    if kind == "structure":
        sites = sum(n * _SHRINK ** l for l in range(case["levels"]))
        per_site = 16 + 27 * 4 + 8 + 8 * 4 * _SHRINK  # coordinates, neighbours, parent and offset, children
        return {"bytes": points * (24 + 4 * case["c"]) + 4.0 * n * case["c"] + sites * per_site, "flops": points * case["c"]}
    if kind == "labels":
        return {"bytes": 2 * points * (24 + 4 * CLASSES) + n * 24.0 + points * 12, "flops": 2.0 * points * CLASSES}
    m, levels = case["m"], case["levels"]
    if kind == "unet":
        flops, weights = _unet(n, m, levels)
        return {"bytes": 4 * weights + points * (16 + 12 + 4 * CLASSES), "flops": flops + 2 * points * m * CLASSES}
    frame = case["new"] + case["old"]
    if kind == "session":
        # a change anywhere reaches every site of the coarse scales and, through them, every site of the decoder
        flops, weights = _unet(n, m, levels)
        frames = case["frames"]
        p = n + frames * case["old"]
        return {"bytes": (1 + frames) * 4 * weights + p * (24 + 12 + 4 * CLASSES), "flops": (1 + 0.75 * frames) * flops}
    flops, weights = _unet(frame, m, levels)
    return {"bytes": 4 * weights + frame * (24 + 12 + 4 * CLASSES), "flops": flops}


def tolerance(case):
    """About four times the largest distance seen between this path and the same path with 64-bit sums."""
    kind = case["kind"]
    if kind == "labels":
        return "exact"
    if kind == "structure":
        return {"rel": 5e-7}  # the per-voxel means: a handful of 32-bit sums and one division
    if kind == "stack":
        return {"rel": 1e-6, "max": 2e-5}  # seen: rel 1.3e-7 (16 channels, one layer) to 2.6e-7 (48, four), max 5.0e-6
    return {"rel": 1.6e-6, "max": 2.4e-5}  # seen on logits: rel 2.6e-7 (4 scales, 6k) to 4.0e-7 (7 scales, 150k), max 5.8e-6
