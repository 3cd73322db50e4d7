"""The calls whose speed counts: relaxations, their seeds and grids, batches and the adjoint, over their real sizes.

Every case is one call that a meshing program makes through the package's entry
points, or the short chain of calls it makes for one volume:

  plan      a grid and seeds resident on the device, relaxed and downloaded
            (Plan.run + Plan.download): the repeated use of one volume
  relax     relax(grid, nodes) from host arrays: relax_cl's own contract
  batch     relax_batch over many uneven volumes from host arrays
  chain     labels to relaxed nodes: grid build, seeding, plan, relaxation, download
  grid      gridbuild.build: a label volume to a host Grid
  seed      Resident.seed: seeds of a grid on the device
  thin      thin(grid, nodes, factor)
  adjoint   RelaxLoss forward and backward: a training step of a sizing field

The volumes are the repository's own kinds (nested, randomly oriented ellipsoids with
perturbed boundaries; softmax probability maps; gray-scale shells; concentric balls),
made here on the device so that one costs a fraction of a second. A case fixes its
anatomy, so that the number of nodes is the case's; the seed draws the label numbers of
the volume (atlas labels, ascending), the voxel size's unit (a power of two) where nodes
are seeded, thinned or a grid is built, and the start positions (a jitter of the interior
nodes) where given nodes are relaxed.

Results of the relaxation, the seeding, the thinning and the grid build are the
reference's own bits by this package's contract, so those cases are compared exactly
and have no 64-bit counterpart (types, resets and rebuilds are decided by comparisons
of the 32-bit values; one bit more of precision is another trajectory). The adjoint's
loss and gradients are ordinary computed numbers: `exact` gives them in 64 bits.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from trussnet_amd import adjoint, gridbuild, relax, volumes
from trussnet_amd._abi import GridParams, Nodes, RelaxParams

K = 24   # list entries a node


def _relax_case(name, kind, source, nx, ny, nz, lo, hi, iters, **more):
    c = {"name": name, "kind": kind, "source": source, "nx": nx, "ny": ny, "nz": nz, "lo": lo, "hi": hi, "iters": iters,
         "vx": 1.0, "vy": 1.0, "vz": 1.0, "nlab": 3, "fire": True, "voxel": False, "dptol": 0.0}
    c.update(more)
    return c


def listed():
    return [
        # a phantom or a quick preview: 3 k nodes, where launches and latency are everything
        _relax_case("plan_small", "plan", "balls", 64, 64, 64, 3.0, 3.0, 50, nlab=2),
        # the production size: a 256^3 six-label volume, sizes graded off the interfaces, 2 M nodes
        _relax_case("plan_large", "plan", "ellipsoids", 256, 256, 256, 1.5, 6.0, 100, nlab=6),
        # a tissue-probability atlas on its usual grid: junctions and corners everywhere
        _relax_case("plan_prob", "plan", "prob", 182, 218, 182, 1.8, 1.8, 100, nlab=6),
        # a thresholded gray-scale scan, automatic (curvature) sizing
        _relax_case("plan_gray", "plan", "gray", 256, 256, 256, 1.5, 6.0, 100, nlab=3),
        # the exact staircase of a label volume (voxel_trap), rebuilds at almost every iteration
        _relax_case("plan_voxel", "plan", "ellipsoids", 160, 168, 152, 1.5, 4.0, 50, nlab=4, voxel=True),
        # the plain call of the pipeline: an odd-sized anisotropic scan from host arrays, the
        # default parameters (FIRE, the convergence stop)
        _relax_case("relax_scan", "relax", "ellipsoids", 121, 137, 94, 2.5, 2.5, 500, nlab=4, vx=0.9, vy=0.9, vz=1.3,
                    dptol=2e-3),
        # a study: uneven volumes of 32 to 160 voxels, each with its own size, in one call
        {"name": "batch_study", "kind": "batch", "count": 20, "edge_lo": 32, "edge_hi": 160, "h_lo": 2.0, "h_hi": 5.0,
         "iters": 100},
        # the whole front end for one labelled volume
        _relax_case("chain_volume", "chain", "ellipsoids", 192, 200, 176, 1.5, 6.0, 100, nlab=6),
        # its first stage alone, as a host pipeline takes it
        {"name": "grid_volume", "kind": "grid", "nx": 200, "ny": 208, "nz": 190, "nlab": 6, "hmin": 1.5, "hbase": 4.5,
         "hmax": 6.0},
        # its second stage alone at the production size
        {"name": "seed_large", "kind": "seed", "nx": 256, "ny": 256, "nz": 256, "nlab": 6, "lo": 1.5, "hi": 6.0},
        # the optional thinning of those seeds
        {"name": "thin_mid", "kind": "thin", "nx": 192, "ny": 192, "nz": 192, "nlab": 5, "lo": 1.5, "hi": 5.0,
         "factor": 0.8},
        # a training step on 200 k nodes: 64 smoothed steps forward and their adjoint
        {"name": "adjoint_200k", "kind": "adjoint", "edge": 58, "iters": 64, "every": 8, "grid": 32},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["plan"] * 6 + ["relax", "relax", "batch", "chain", "grid", "seed", "thin", "adjoint", "adjoint"])
    if kind == "adjoint":
        return {"kind": kind, "edge": _log_int(rng, 12, 58), "iters": rng.randint(8, 64), "every": rng.randint(1, 16),
                "grid": rng.randint(5, 32)}
    if kind == "batch":
        lo = rng.randint(24, 60)
        return {"kind": kind, "count": _log_int(rng, 2, 20), "edge_lo": lo, "edge_hi": rng.randint(lo + 1, 150),
                "h_lo": 2.2, "h_hi": round(rng.uniform(2.5, 5.0), 2), "iters": rng.randint(20, 100)}
    n = [_log_int(rng, 40, 190) for _ in range(3)]
    nlab = rng.randint(2, 6)
    lo = round(rng.uniform(1.5, 3.0), 2)
    if kind == "grid":
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "nlab": nlab, "hmin": lo, "hbase": 2.0 * lo,
                "hmax": 3.0 * lo}
    if kind in ("seed", "thin"):
        c = {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "nlab": nlab, "lo": lo, "hi": round(lo * rng.uniform(1, 4), 2)}
        if kind == "thin":
            c["factor"] = round(rng.uniform(0.4, 1.1), 2)
        return c
    source = rng.choice(["ellipsoids", "ellipsoids", "balls", "prob", "gray"])
    v = [1.0, 1.0, 1.0]
    if source == "ellipsoids" and rng.random() < 0.4:
        v = [round(rng.uniform(0.8, 1.3), 2) for _ in range(3)]
    hi = lo if source in ("balls", "prob") else round(lo * rng.uniform(1, 4), 2)
    c = _relax_case("", kind, source, n[0], n[1], n[2], lo, hi, rng.randint(10, 100),
                    nlab=2 if source == "balls" else (3 if source == "gray" else nlab), vx=v[0], vy=v[1], vz=v[2],
                    fire=rng.random() < 0.8, voxel=source == "ellipsoids" and rng.random() < 0.2,
                    dptol=2e-3 if rng.random() < 0.3 else 0.0)
    del c["name"]
    return c


# --- volumes -----------------------------------------------------------------------------

def _smooth(f, sigma):
    """Gaussian smoothing with wrap-around, unit standard deviation."""
    r = int(math.ceil(3.0 * sigma))
    w = [math.exp(-0.5 * (k / sigma) ** 2) for k in range(-r, r + 1)]
    for ax in range(3):
        g = torch.zeros_like(f)
        for k in range(-r, r + 1):
            g += torch.roll(f, k, ax) * w[k + r]
        f = g
    return f / f.std()


def _noise(shape, sigma, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return _smooth(torch.randn(shape, generator=gen, device="cuda"), sigma)


def _axes(nx, ny, nz):
    z, y, x = (torch.arange(m, dtype=torch.float32, device="cuda") for m in (nz, ny, nx))
    return x[None, None, :], y[None, :, None], z[:, None, None]


def _anatomy(*sizes):
    """The seed of a case's volume: its own, the same for every seed of the inputs."""
    a = 17
    for v in sizes:
        a = (a * 1000003 + int(round(1000 * v))) % (1 << 31)
    return a


def _relabelled(lab, seed):
    """Labels 1.. replaced by ascending atlas numbers drawn by the seed (0 stays the exterior)."""
    m = int(lab.max())
    ids = np.sort(np.random.default_rng(seed).choice(np.arange(1, 1000), m, replace=False))
    return torch.from_numpy(np.concatenate([[0], ids])).cuda()[lab.long()]


def _unit(seed):
    """A voxel's unit: a power of two, by which every length scales without a rounding."""
    return 2.0 ** int(np.random.default_rng(seed + 1).integers(-3, 4))


def _jittered(nodes, labels, vs, h, seed):
    """The nodes with the interior ones moved by up to 0.1 h where that keeps their voxel's label."""
    rng = np.random.default_rng(seed + 2)
    P = nodes.P + rng.uniform(-0.1 * h, 0.1 * h, nodes.P.shape).astype(np.float32)
    v = np.floor(P / np.array(vs, np.float32) + 0.5).astype(np.int64)
    dims = np.array(labels.shape[::-1])
    ok = (nodes.typ == 0) & ((v >= 0) & (v < dims)).all(1)
    v = np.clip(v, 0, dims - 1)
    ok &= labels[v[:, 2], v[:, 1], v[:, 0]] == nodes.lab
    return Nodes(np.where(ok[:, None], P, nodes.P), nodes.lab, nodes.typ, nodes.part, nodes.part3)


def _ellipsoids(nx, ny, nz, nlab):
    """Labels of nested, randomly oriented ellipsoids with perturbed boundaries, and
    about the distance (voxels) from the nearest interface; (nz, ny, nx) tensors."""
    seed = _anatomy(nx, ny, nz, nlab)
    rng = np.random.default_rng(seed)
    x, y, z = _axes(nx, ny, nz)
    edge = np.array([nx, ny, nz], np.float64)
    frac = np.linspace(0.47, 0.09, nlab)[:, None] * rng.uniform(0.85, 1.1, (nlab, 3))
    frac = -np.sort(-frac, axis=0)
    bump = 3.0 * _noise((nz, ny, nx), 4.0, seed)
    lab = torch.zeros((nz, ny, nx), dtype=torch.int32, device="cuda")
    dist = torch.full((nz, ny, nx), 1e6, device="cuda")
    for k in range(nlab):
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        c = (edge - 1) / 2 + rng.uniform(-0.025, 0.025, 3) * edge
        a = frac[k] * edge.min()
        d = [x - c[0], y - c[1], z - c[2]]
        u = [sum(float(q[i, j]) * d[i] for i in range(3)) / float(a[j]) for j in range(3)]
        s = (torch.sqrt(u[0] ** 2 + u[1] ** 2 + u[2] ** 2) - 1.0) * float(a.mean()) + bump
        lab[s < 0] = k + 1
        dist = torch.minimum(dist, s.abs())
    return lab, dist


def _host(t, dtype):
    return t.cpu().numpy().astype(dtype)


def _volume(case, seed):
    """Keyword arguments of gridbuild.build for the case's volume (host arrays)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    unit = _unit(seed) if case["kind"] in ("seed", "thin", "chain") else 1.0
    vs = tuple(unit * case.get(k, 1.0) for k in ("vx", "vy", "vz"))
    lo, hi = unit * case["lo"], unit * case["hi"]
    source = case.get("source", "ellipsoids")
    own = _anatomy(nx, ny, nz, case["nlab"])
    kw = {"vs": vs, "prm": GridParams(hbase=0.5 * (lo + hi) if hi > lo else lo, hmin=lo, hmax=hi)}
    if source == "balls":
        x, y, z = _axes(nx, ny, nz)
        c = [(m - 1) / 2 for m in (nx, ny, nz)]
        r = torch.sqrt((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2)
        m = min(nx, ny, nz)
        lab = (r < 0.375 * m).to(torch.int32) + (r < 0.1875 * m).to(torch.int32)
    elif source == "prob":
        f = torch.stack([_noise((nz, ny, nx), 6.0, own + k) for k in range(case["nlab"])])
        p = torch.softmax(f, 0)
        lab = p.argmax(0)
        kw["prob"] = p.cpu().numpy()
    elif source == "gray":
        x, y, z = _axes(nx, ny, nz)
        c = [(m - 1) / 2 for m in (nx, ny, nz)]
        r = torch.sqrt((x - c[0]) ** 2 + (y - c[1]) ** 2 + (z - c[2]) ** 2)
        g = 1.0 - r / (0.45 * min(nx, ny, nz)) + 0.06 * _noise((nz, ny, nx), 3.0, own)
        lab = sum((g >= t).to(torch.int32) for t in volumes.GRAY_THRESHOLDS)
        kw["gray"] = g.cpu().numpy()
        kw["thresholds"] = volumes.GRAY_THRESHOLDS
    else:
        lab, dist = _ellipsoids(nx, ny, nz, case["nlab"])
        if hi > lo and case["kind"] != "chain":   # graded off the interfaces, as a user's sizing field
            kw["hvox"] = _host(unit * torch.clamp(case["lo"] + 0.03 * dist, max=case["hi"]), np.float32)
    if source in ("ellipsoids", "balls"):
        lab = _relabelled(lab, seed)
    kw["labels"] = _host(lab, np.uint16)
    return kw


def _relax_params(case):
    return RelaxParams(max_iters=case["iters"], dptol=case["dptol"], fire=case["fire"], voxel_trap=case["voxel"])


def _kuhn_tets(m):
    """Six tetrahedra a cell of an m^3 lattice (x fastest)."""
    i = np.arange(m - 1)
    z, y, x = np.meshgrid(i, i, i, indexing="ij")
    base = (x + m * (y + m * z)).ravel()
    step = (1, m, m * m)
    tets = []
    for p in ((0, 1, 2), (1, 2, 0), (2, 0, 1), (0, 2, 1), (2, 1, 0), (1, 0, 2)):
        a = base + step[p[0]]
        b = a + step[p[1]]
        tets.append(np.stack([base, a, b, b + step[p[2]]], axis=1))
    return np.concatenate(tets).astype(np.int32)


def _adjoint_inputs(case, seed):
    """A jittered lattice with its fixed surface, its K-nearest lists, tetrahedra and sizing grid."""
    m, s = case["edge"], 2.0
    ext = (m - 1) * s
    n = int(ext) + 1
    P = volumes.jittered_points(n, s, 0.2, seed)
    # nodes off the volume's edge by half a voxel at most stay inside it
    P = np.clip(P, 0.0, ext).astype(np.float32)
    i = np.arange(m)
    z, y, x = np.meshgrid(i, i, i, indexing="ij")
    rim = ((np.minimum(np.minimum(x, y), z) == 0) | (np.maximum(np.maximum(x, y), z) == m - 1)).ravel()
    h = 1.1 * s
    res = gridbuild.build_resident(np.ones((n, n, n), np.uint16), prm=GridParams(hbase=h, hmin=h, hmax=h))
    nodes = Nodes(P, np.ones(P.shape[0], np.uint16), np.where(rim, 1, 0).astype(np.uint8),
                  np.full((P.shape[0], 2), 0xFFFF, np.uint16))
    with res.plan(nodes) as plan:
        rb = plan.rebuild()
    res.close()
    g = case["grid"]
    spacing = (ext / (g - 1),) * 3
    rng = np.random.default_rng(seed)
    u = np.arange(g) / g
    wave = (np.sin(2 * np.pi * (u[None, None, :] + rng.uniform())) * np.cos(2 * np.pi * (u[None, :, None] + rng.uniform()))
            * np.cos(2 * np.pi * u[:, None, None]))
    theta = (h * (1.0 + 0.1 * wave)).astype(np.float32)
    return P, theta, rb["nbr"].reshape(-1, K), rb["nnb"], nodes.typ, _kuhn_tets(m), spacing


def prepare(case, seed):
    kind = case["kind"]
    if kind == "adjoint":
        P, theta, nbr, nnb, typ, tets, spacing = _adjoint_inputs(case, seed)
        prm = adjoint.AdjParams(iters=case["iters"], ckpt_every=case["every"])
        pb = adjoint.Problem(nbr, nnb, typ, tets, theta.shape, (0.0, 0.0, 0.0), spacing, prm)
        return {"kind": kind, "problem": pb, "x0": torch.from_numpy(P).cuda().requires_grad_(),
                "theta": torch.from_numpy(theta).cuda().requires_grad_()}
    if kind == "batch":
        grids, nodes = [], []
        # evenly spread edges and sizes, paired out of order
        edges = np.linspace(case["edge_lo"], case["edge_hi"], case["count"]).astype(int)
        sizes = np.linspace(case["h_lo"], case["h_hi"], case["count"])[(np.arange(case["count"]) * 7) % case["count"]]
        for k, (n, h) in enumerate(zip(edges.tolist(), sizes.tolist())):
            lab, _ = _ellipsoids(n, n, n, 2 + k % 3)
            lab = _host(_relabelled(lab, seed + k), np.uint16)
            grids.append(gridbuild.build(lab, prm=GridParams(hbase=h, hmin=h, hmax=h)))
            nodes.append(_jittered(relax.seed(grids[-1]), lab, (1.0, 1.0, 1.0), h, seed + k))
        return {"kind": kind, "grids": grids, "nodes": nodes, "prm": RelaxParams(max_iters=case["iters"], dptol=0.0)}
    if kind == "grid":
        lab, _ = _ellipsoids(case["nx"], case["ny"], case["nz"], case["nlab"])
        unit = _unit(seed)
        return {"kind": kind, "labels": _host(_relabelled(lab, seed), np.uint16), "vs": (unit, unit, unit),
                "prm": GridParams(hbase=unit * case["hbase"], hmin=unit * case["hmin"], hmax=unit * case["hmax"])}
    kw = _volume(case, seed)
    if kind == "chain":
        return {"kind": kind, "volume": kw, "prm": _relax_params(case)}
    if kind in ("relax", "thin"):
        grid = gridbuild.build(**kw)
        nodes = relax.seed(grid)
        if kind == "thin":
            return {"kind": kind, "grid": grid, "nodes": nodes, "factor": case["factor"]}
        nodes = _jittered(nodes, kw["labels"], kw["vs"], case["lo"], seed)
        return {"kind": kind, "grid": grid, "nodes": nodes, "prm": _relax_params(case)}
    res = gridbuild.build_resident(**kw)
    if kind == "seed":
        return {"kind": kind, "grid": res}
    prm = _relax_params(case)
    plan = res.plan(_jittered(res.seed(prm), kw["labels"], kw["vs"], case["lo"], seed), prm)
    res.close()
    return {"kind": kind, "plan": plan}


def _nodes(x):
    out = {"P": x.P, "lab": x.lab.view(np.int16), "typ": x.typ, "part": x.part.view(np.int16)}
    if x.part3 is not None:
        out["part3"] = x.part3.view(np.int16)
    return out


def _relaxed(x, st):
    return {"P": x.P, "typ": x.typ, "part": x.part.view(np.int16), "iters": st["iters"], "rebuilds": st["rebuilds"],
            "last_move": st["last_move"]}


def run(state):
    kind = state["kind"]
    if kind == "plan":
        st = state["plan"].run()
        return _relaxed(state["plan"].download(), st)
    if kind == "relax":
        return _relaxed(*relax.relax(state["grid"], state["nodes"], state["prm"]))
    if kind == "batch":
        out = relax.relax_batch(state["grids"], state["nodes"], state["prm"])
        return [[x.P, x.typ, x.part.view(np.int16)] for x, _ in out]
    if kind == "chain":
        res = gridbuild.build_resident(**state["volume"])
        seeds = res.seed(state["prm"])
        with res.plan(seeds, state["prm"]) as plan:
            res.close()
            st = plan.run()
            out = _relaxed(plan.download(), st)
        out["lab"] = seeds.lab.view(np.int16)
        return out
    if kind == "grid":
        g = gridbuild.build(state["labels"], state["vs"], state["prm"])
        return {"bl_cnt": g.bl_cnt, "bl_lab": g.bl_lab.view(np.int16), "bl_slot": g.bl_slot, "phi": g.phi, "h": g.h,
                "grade": g.grade}
    if kind == "seed":
        return _nodes(state["grid"].seed())
    if kind == "thin":
        return _nodes(relax.thin(state["grid"], state["nodes"], state["factor"]))
    x0, theta = state["x0"], state["theta"]
    loss = adjoint.RelaxLoss.apply(x0, theta, state["problem"])
    gx, gt = torch.autograd.grad(loss, (x0, theta))
    return {"loss": loss.detach(), "grad_x": gx, "grad_theta": gt}


# --- what a pass cannot do without --------------------------------------------------------

def _seed_count(case):
    """About the nodes of a case's volume: sqrt(2) / h^3 a mm^3, graded by the distance off the interfaces."""
    nx, ny, nz, nlab, lo, hi = (case[k] for k in ("nx", "ny", "nz", "nlab", "lo", "hi"))
    cell = case.get("vx", 1.0) * case.get("vy", 1.0) * case.get("vz", 1.0)
    edge = min(nx, ny, nz)
    source = case.get("source", "ellipsoids")
    if source == "prob":
        inside = nx * ny * nz * (1.0 - 1.0 / nlab)
    else:
        inside = 4.0 / 3.0 * math.pi * ({"balls": 0.375, "gray": 0.36}.get(source, 0.46) * edge) ** 3
    if hi > lo and source == "ellipsoids" and case["kind"] != "chain":
        reach = 0.38 * edge / max(1, nlab - 1) / 2
        d = np.linspace(0.0, reach, 64)
        density = float(np.mean(np.minimum(lo + 0.03 * d, hi) ** -3.0))
    elif hi > lo:   # automatic sizing: between the smallest and the base size
        density = (0.5 * (lo + 0.5 * (lo + hi))) ** -3.0
    else:
        density = lo ** -3.0
    return math.sqrt(2.0) * density * inside * cell


def _relax_work(n, voxels, iters):
    # one iteration: 21 list entries (84), their neighbours' positions once (16), position, velocity and size
    # read and written (64), type, label, partners, list length (11), reference position (16); 21 bars of
    # about 20 operations and a move of about 200. Rebuilds come about every fifth iteration: the same state
    # once more, with the lists written. The field is read once.
    return {"bytes": n * (iters * 191.0 + (iters / 5.0) * 263.0) + 8.0 * voxels,
            "flops": n * iters * 620.0 + n * (iters / 5.0) * 24 * 40.0}


def work(case):
    kind = case["kind"]
    if kind == "adjoint":
        n = case["edge"] ** 3
        # a forward step: lists once and positions in and out; the backward takes about twice that; RelaxLoss
        # returns the loss and both gradients
        return {"bytes": 3.0 * case["iters"] * n * (24 * 4 + 4 + 32.0), "flops": 3.0 * case["iters"] * n * 24 * 30.0}
    if kind == "batch":
        edges = np.linspace(case["edge_lo"], case["edge_hi"], case["count"])
        sizes = np.linspace(case["h_lo"], case["h_hi"], case["count"])[(np.arange(case["count"]) * 7) % case["count"]]
        total = {"bytes": 0.0, "flops": 0.0}
        for e, h in zip(edges, sizes):
            n = math.sqrt(2.0) / h ** 3 * 4.0 / 3.0 * math.pi * (0.46 * e) ** 3
            w = _relax_work(n, e ** 3, case["iters"])
            total = {k: total[k] + w[k] for k in total}
        return total
    voxels = case["nx"] * case["ny"] * case["nz"]
    if kind == "grid":   # labels in; sizes, grades and the fields of about a third of the bricks' labels out
        return {"bytes": voxels * (2.0 + 4.0 + 1.0 + 4.0), "flops": voxels * 400.0}
    n = _seed_count(case)
    if kind in ("seed", "thin"):
        return {"bytes": voxels * 11.0 + n * 21.0 * (1 if kind == "seed" else 2), "flops": voxels * 10.0 + n * 400.0}
    w = _relax_work(n, voxels, case["iters"] if case["dptol"] == 0.0 else 0.5 * case["iters"])
    if kind == "chain":
        w = {"bytes": w["bytes"] + voxels * 22.0, "flops": w["flops"] + voxels * 410.0}
    return w


# --- how far another correct implementation may be off -------------------------------------

def tolerance(case):
    if case["kind"] == "adjoint":
        # measured against 64 bits: loss 3e-8, gradients up to 1.4e-6 off in norm
        return {"rel": 6e-6, "max": 1e-3}
    return "exact"


def _sizes64(theta, x, spacing):
    """Sizes at x: trilinear in theta with smoothstep cell fractions, positions clamped to the grid."""
    g = torch.tensor(theta.shape[::-1], device=x.device)
    u = torch.minimum(torch.clamp(x / torch.tensor(spacing, dtype=x.dtype, device=x.device), min=0.0), (g - 1).to(x.dtype))
    i = torch.minimum(torch.floor(u.detach()).long(), g - 2)
    f = u - i
    f = f * f * (3.0 - 2.0 * f)
    flat = theta.reshape(-1)
    h = 0.0
    for c in range(8):
        b = [c & 1, (c >> 1) & 1, c >> 2]
        w = 1.0
        for a in range(3):
            w = w * (f[:, a] if b[a] else 1.0 - f[:, a])
        h = h + w * flat[(i[:, 0] + b[0]) + g[0] * ((i[:, 1] + b[1]) + g[1] * (i[:, 2] + b[2]))]
    return h


def _bars64(x, theta, spacing, prm, i, j, c):
    h = _sizes64(theta, x, spacing)
    e = x[i] - x[j]
    l = torch.sqrt((e * e).sum(1))
    u = c * 0.5 * (h[i] + h[j]) - l
    return e, l, u, torch.nn.functional.softplus(u, beta=prm.beta, threshold=1e3)


def _step64(x, theta, spacing, prm, i, j, c, moves):
    e, l, u, sp = _bars64(x, theta, spacing, prm, i, j, c)
    F = torch.zeros_like(x).index_add(0, i, (sp / l)[:, None] * e)
    D = 1.0 + torch.zeros_like(x[:, 0]).index_add(0, i, torch.sigmoid(prm.beta * u))
    return x + moves[:, None] * prm.dt * F / D[:, None]


def exact(case, seed):
    if case["kind"] != "adjoint":
        return None   # compared bit for bit: no 64-bit counterpart
    from torch.utils.checkpoint import checkpoint

    P, theta, nbr, nnb, typ, tets, spacing = _adjoint_inputs(case, seed)
    prm = adjoint.AdjParams(iters=case["iters"], ckpt_every=case["every"])
    dev = "cuda"
    # (the library reads spacing and the scalars as 32-bit values)
    spacing = tuple(float(np.float32(s)) for s in spacing)
    fscale, fsurf, eps = float(np.float32(prm.fscale)), float(np.float32(prm.fsurf)), float(np.float32(prm.eps_v))
    x0 = torch.from_numpy(P).to(dev, torch.float64).requires_grad_()
    th = torch.from_numpy(theta).to(dev, torch.float64).requires_grad_()
    n = P.shape[0]
    used = np.arange(K)[None, :] < nnb[:, None]
    i = torch.from_numpy(np.repeat(np.arange(n), nnb)).to(dev)
    j = torch.from_numpy(nbr[used].astype(np.int64)).to(dev)
    t = torch.from_numpy(typ).to(dev)
    c = torch.where((t[i] != 0) & (t[j] != 0), fsurf, fscale).to(torch.float64)
    moves = (t == 0).to(torch.float64)
    x = x0
    for _ in range(case["iters"]):
        x = checkpoint(_step64, x, th, spacing, prm, i, j, c, moves, use_reentrant=False)
    sp = _bars64(x, th, spacing, prm, i, j, c)[3]
    energy = 0.5 * (sp * sp).sum() / n
    v = torch.from_numpy(tets.astype(np.int64)).to(dev)
    p = [x[v[:, k]] for k in range(4)]
    a, b, d = p[1] - p[0], p[2] - p[0], p[3] - p[0]
    vol = (a * torch.linalg.cross(b, d)).sum(1) / 6.0
    vs = torch.sqrt(vol * vol + eps * eps)
    s = sum(((p[m] - p[o]) ** 2).sum(1) for m in range(4) for o in range(m + 1, 4))
    quality = (1.0 - 12.0 * (3.0 * vs) ** (2.0 / 3.0) / s).mean()
    loss = energy + prm.wq * quality
    gx, gt = torch.autograd.grad(loss, (x0, th))
    return {"loss": loss.detach(), "grad_x": gx, "grad_theta": gt}
