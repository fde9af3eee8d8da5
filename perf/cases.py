"""What users of vdock have it do, as cases that can be timed and checked.

Every case is one call sequence through the Python front end (vdock.Context), over the sizes the
benchmark and the tests use: single conformations to a million, 10-atom fragments to 80-atom
peptides, 20 A boxes to 70 A boxes, one ligand to a screening batch.

    kind     one pass                                         stands for
    score    vd_eval on host arrays                           rescoring a few poses; a caller's own optimiser
    adjoint  vd_eval on device arrays (torch tensors)         large resident sets of conformations
    maps     set_receptor, grid_populate, scores on the maps  a new receptor, or a new box
    search   local_search from given starts                   minimising poses without docking
    refine   postprocess of given poses                       the FP64 step after a search
    dock     dock, every chain's result back                  one ligand (kernel_monte's role)
    screen   dock_batch, postprocess_docked, every mode back  a library of ligands, the whole call

Inputs come from the seed alone: receptors and ligands from the library's own generators, poses
and ligand sizes from numpy.  torch is imported first: libvdock then runs on the HIP runtime that
torch has loaded, and the two exchange device pointers.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "vina-cuda_amd"))
import vdock  # noqa: E402

# (receptor atoms, cube edge, cavity radius, box edge): the three scenes of the benchmark.  The
# largest box at 0.375 A has 188^3 points per map.
SCENES = {"small": (2000, 36.0, 8.0, 20.0), "medium": (8000, 60.0, 10.0, 30.0), "large": (20000, 90.0, 25.0, 70.0)}
GRID = 0.375


def listed():
    return [
        # one pose scored, host arrays: the latency of a call (a caller's own optimiser makes one per step)
        {"name": "score_one", "kind": "score", "scene": "medium", "heavy": 32, "tors": 8, "n": 1},
        # a ragged set of poses of a large flexible ligand, more atoms than a wavefront has lanes
        {"name": "score_peptide_5003", "kind": "score", "scene": "medium", "heavy": 75, "tors": 24, "n": 5003},
        # the adjoint microbenchmark: 2^20 resident conformations
        {"name": "adjoint_2e20", "kind": "adjoint", "scene": "medium", "heavy": 40, "tors": 12, "n": 1 << 20},
        # a new receptor in an ordinary box (81^3 points), and in the largest box of the benchmark
        {"name": "maps_81", "kind": "maps", "scene": "medium", "heavy": 24, "tors": 5, "n": 1001},
        {"name": "maps_188", "kind": "maps", "scene": "large", "heavy": 40, "tors": 10, "n": 1001},
        # poses minimised without a search
        {"name": "search_2000", "kind": "search", "scene": "medium", "heavy": 32, "tors": 8, "n": 2000, "dense": False},
        # the FP64 refinement of the pose lists of 60 ligands
        {"name": "refine_60x20", "kind": "refine", "scene": "medium", "heavy": 60, "tors": 16, "ligands": 60, "poses": 20},
        # one ligand with few chains (a workgroup per chain leaves most of the GPU idle), and the
        # default 8,192 chains of the command line
        {"name": "dock_512", "kind": "dock", "scene": "small", "heavy": 20, "tors": 5, "chains": 512, "policy": "vina"},
        {"name": "dock_8192", "kind": "dock", "scene": "medium", "heavy": 32, "tors": 8, "chains": 8192, "policy": "vina"},
        # libraries: the headline's ligands and box, the same under dense BFGS, and the large box
        # under the QuickVina2 policy
        {"name": "screen_vina", "kind": "screen", "scene": "medium", "heavy": 60, "tors": 16, "ligands": 256,
         "chains": 256, "policy": "vina"},
        {"name": "screen_bfgs", "kind": "screen", "scene": "medium", "heavy": 60, "tors": 16, "ligands": 96,
         "chains": 256, "policy": "bfgs"},
        {"name": "screen_qvina2_large", "kind": "screen", "scene": "large", "heavy": 80, "tors": 24, "ligands": 200,
         "chains": 128, "policy": "qvina2"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges; heavy and tors are a ligand's, or a library's largest."""
    kind = rng.choice(["score", "score", "adjoint", "maps", "maps", "search", "refine", "dock", "dock", "screen", "screen"])
    heavy = rng.randint(10, 75)
    c = {"kind": kind, "scene": rng.choice(["small", "medium", "medium", "large"]), "heavy": heavy,
         "tors": rng.randint(0, min(24, heavy // 3))}
    if kind == "score":
        c["n"] = _log_int(rng, 1, 20000)
    elif kind == "adjoint":
        c["n"] = _log_int(rng, 30000, 500000)
    elif kind == "maps":
        c["n"] = _log_int(rng, 100, 2000)
    elif kind == "search":
        c.update(n=_log_int(rng, 50, 5000), dense=rng.random() < 0.3)
    elif kind == "refine":
        c.update(ligands=_log_int(rng, 1, 60), poses=rng.randint(1, 20))
    elif kind == "dock":
        c.update(chains=_log_int(rng, 100, 8192 * 32 // max(32, heavy)), policy=rng.choice(["vina", "vina", "bfgs", "qvina2"]))
    else:
        c.update(heavy=rng.randint(20, 75), policy=rng.choice(["vina", "vina", "bfgs", "qvina2"]), chains=rng.choice([32, 100, 128]),
                 ligands=_log_int(rng, 3, 80))
        c["tors"] = rng.randint(2, min(20, c["heavy"] // 3))
    return c


# ---- inputs ---------------------------------------------------------------------------------
def _scene(case, seed):
    n, cube, cavity, box = SCENES[case["scene"]]
    xyz, xs = vdock.synth_receptor(n, cube, cavity, 1000 + seed)
    return xyz, xs, vdock.box_from_center([0, 0, 0], [box] * 3, GRID)


def _ligand(case, seed):
    return vdock.synth_ligand(case["heavy"], case["tors"], 2000 + seed)


def _library(case, seed):
    """PDBQT texts of a library: heavy atoms uniform in [10, heavy], torsions in [0, min(tors, heavy / 3)]."""
    rng = np.random.default_rng(3000 + seed)
    out = []
    for i in range(case["ligands"]):
        heavy = int(rng.integers(10, case["heavy"] + 1))
        out.append(vdock.synth_ligand(heavy, int(rng.integers(0, min(case["tors"], heavy // 3) + 1)), 100000 * (seed % 1000) + i))
    return out


def _torsions(text):
    return text.count("\nBRANCH")


def _poses(text, n, box, seed):
    """Poses [n][7 + T]: root atom in the middle of the box (0.3 of each edge), any orientation, any torsions."""
    rng = np.random.default_rng(4000 + seed)
    lo, hi = np.array(box.begin), np.array(box.end)
    c = np.empty((n, 7 + _torsions(text)), dtype=np.float32)
    c[:, :3] = (lo + hi) / 2 + rng.uniform(-0.15, 0.15, (n, 3)) * (hi - lo)
    q = rng.normal(size=(n, 4))
    c[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    c[:, 7:] = rng.uniform(-np.pi, np.pi, (n, c.shape[1] - 7))
    return c


def _params(case, seed):
    kw = {"seed": seed & 0x7FFFFFFF}
    if case.get("policy") == "bfgs" or case.get("dense"):
        kw["local_search"] = vdock.VD_LS_BFGS
    if case.get("policy") == "qvina2":
        kw["policy"] = vdock.VD_MC_QVINA2
    if "chains" in case:
        kw["chains"] = case["chains"]
    return vdock.default_params(**kw)


def prepare(case, seed):
    kind = case["kind"]
    xyz, xs, box = _scene(case, seed)
    ctx = vdock.Context(0)
    s = {"kind": kind, "ctx": ctx, "xyz": xyz, "xs": xs, "box": box}
    if kind in ("refine", "screen"):
        texts = _library(case, seed)
        s["ids"] = [ctx.add_ligand(t) for t in texts]
        s["tors"], s["atoms"] = case["tors"], 2 * case["heavy"]   # with hydrogens: at most one per heavy atom
    else:
        text = _ligand(case, seed)
        s["id"] = ctx.add_ligand(text)
    if kind != "maps":
        ctx.set_receptor(xyz, xs)
        ctx.grid_populate(box)
    if kind in ("search", "dock", "screen"):
        s["params"] = _params(case, seed)
    if kind in ("score", "maps", "search"):
        s["conf"] = _poses(text, case["n"], box, seed)
    elif kind == "adjoint":
        conf = _poses(text, case["n"], box, seed)
        s["conf"] = torch.from_numpy(conf).cuda()
        s["e"] = torch.zeros(case["n"], dtype=torch.float32, device="cuda")
        s["g"] = torch.zeros((case["n"], conf.shape[1] - 1), dtype=torch.float32, device="cuda")
        torch.cuda.synchronize()
    elif kind == "refine":
        # rough poses, as a search with few steps leaves them: one short search from random ones
        s["confs"] = []
        p = vdock.default_params(bfgs_steps=4)
        for k, (i, t) in enumerate(zip(s["ids"], texts)):
            start = _poses(t, case["poses"], box, seed + 7 * k)
            s["confs"].append(ctx.local_search(i, start, p)[1])
    return s


def _modes(ctx, s):
    """Every ligand's modes after a post-processing call, in arrays of one shape for any library:
    at most 9 modes of a ligand, rows of the library's largest ligand."""
    n = len(s["ids"])
    count = np.zeros(n, dtype=np.int32)
    pose = np.full((n, 9), -1, dtype=np.int32)
    score = np.zeros((n, 9, 3), dtype=np.float32)
    conf = np.zeros((n, 9, 7 + s["tors"]), dtype=np.float32)
    coords = np.zeros((n, 9, s["atoms"], 3), dtype=np.float32)
    for k in range(n):
        modes, cf, xyz = ctx.post_results(k)
        m = count[k] = len(modes)
        pose[k, :m] = [x.pose for x in modes]
        score[k, :m] = [(x.e, x.rmsd_lb, x.rmsd_ub) for x in modes]
        conf[k, :m, :cf.shape[1]] = cf
        coords[k, :m, :xyz.shape[1]] = xyz
    return {"count": count, "pose": pose, "score": score, "conf": conf, "coords": coords}


def run(s):
    ctx, kind = s["ctx"], s["kind"]
    if kind == "score":
        return ctx.eval(s["id"], s["conf"])
    if kind == "adjoint":
        ctx.eval_device(s["id"], s["conf"].data_ptr(), s["e"].data_ptr(), s["g"].data_ptr(), len(s["e"]))
        return s["e"], s["g"]
    if kind == "maps":
        ctx.set_receptor(s["xyz"], s["xs"])
        ctx.grid_populate(s["box"])
        return ctx.eval(s["id"], s["conf"])
    if kind == "search":
        e, conf, st = ctx.local_search(s["id"], s["conf"], s["params"])
        return e, conf, int(st.evals)
    if kind == "refine":
        ctx.postprocess(s["ids"], s["confs"])
        return _modes(ctx, s)
    if kind == "dock":
        e, conf, heavy, st = ctx.dock(s["id"], s["params"])
        return e, conf, heavy, int(st.evals)
    st = ctx.dock_batch(s["ids"], s["params"])
    best = ctx.batch_best()
    ctx.postprocess_docked(20)
    return {"best": best, "evals": int(st.evals), **_modes(ctx, s)}


# ---- work -----------------------------------------------------------------------------------
def work(case):
    """Inputs read once and outputs written once; operations of the evaluations.  One evaluation:
    about 120 per atom (its place, eight map corners, its part of the adjoint) and 35 per pair of
    atoms (A^2 / 3 pairs).  A search does about two evaluations per iteration, a chain one search
    per step, a refinement about 100 evaluations with 80 receptor atoms for each ligand atom."""
    kind = case["kind"]
    n_rec, _, _, edge = SCENES[case["scene"]]
    points = (math.ceil(edge / GRID) + 1) ** 3
    lib = kind in ("refine", "screen")
    A = 1.2 * (10 + case["heavy"]) / 2 if lib else 1.2 * case["heavy"]
    T = case["tors"] / 2.5 if lib else case["tors"]
    per_eval = 120 * A + 35 * A * A / 3
    io = 4.0 * (14 + 2 * T)
    maps = 68.0 * points
    if kind in ("score", "adjoint"):
        return {"bytes": case["n"] * io + min(maps, case["n"] * A * 32), "flops": case["n"] * per_eval}
    if kind == "maps":
        return {"bytes": 16.0 * n_rec + maps + case["n"] * io, "flops": points * 80 * 25 + case["n"] * per_eval}
    depth, iters = (max(1.0, (0.24 * A + 0.29 * T - 3.41) * 2), (30 + A) / 3)
    if kind == "search":
        return {"bytes": 2 * case["n"] * io, "flops": case["n"] * iters * 2 * per_eval}
    if kind == "refine":
        n = case["ligands"] * case["poses"]
        return {"bytes": n * (io + 12 * A), "flops": n * 100 * (per_eval + A * 80 * 20)}
    n = case["chains"] * case.get("ligands", 1)
    return {"bytes": n * (io + 12 * A) + maps, "flops": n * depth * iters * 2 * per_eval}


# ---- energies and gradients in 64 bits ------------------------------------------------------
# The scoring function, the interpolation on its tables and maps, and the adjoint, written out
# for exact() from their definitions: Vina's terms on tables over 32 r^2, the sum over receptor
# atoms at each grid point from the table's mean of neighbouring entries, trilinear maps.
_RADIUS = np.array([1.9, 1.9, 1.8, 1.8, 1.8, 1.8, 1.7, 1.7, 1.7, 1.7, 2.0, 2.1, 1.5, 1.8, 2.0, 2.2, 1.2])
_HYDROPHOBIC, _ACCEPTOR, _DONOR = {0, 12, 13, 14, 15}, {4, 5, 8, 9}, {3, 5, 7, 9, 16}
_BINS = 2051


def _tables(device):
    """smooth value, derivative / r and map value, each [17][17][bins]."""
    w = vdock.DEFAULT_WEIGHTS
    r = np.sqrt(np.arange(_BINS) / 32.0)
    e = np.zeros((17, 17, _BINS))
    for a in range(17):
        for b in range(17):
            d = r - (_RADIUS[a] + _RADIUS[b])
            t = w[0] * np.exp(-(d / 0.5) ** 2) + w[1] * np.exp(-((d - 3.0) / 2.0) ** 2) + w[2] * np.where(d < 0, d * d, 0.0)
            if a in _HYDROPHOBIC and b in _HYDROPHOBIC:
                t = t + w[3] * np.clip(1.5 - d, 0.0, 1.0)
            if (a in _DONOR and b in _ACCEPTOR) or (b in _DONOR and a in _ACCEPTOR):
                t = t + w[4] * np.clip(d / -0.7, 0.0, 1.0)
            e[a, b] = t
    dor = np.zeros_like(e)
    dor[..., 1:-1] = (e[..., 2:] - e[..., :-2]) / ((r[2:] - r[:-2]) * r[1:-1])
    fast = 0.5 * (e + np.concatenate([e[..., 1:], np.zeros((17, 17, 1))], axis=-1))
    return [torch.from_numpy(t).to(device) for t in (e, dor, fast)]


def _model(text):
    """Atoms (local place, node, XS type), nodes (parent, origin and axis in the parent's frame) and
    pairs (variable distance, more than three bonds apart) of a generated ligand's PDBQT text.  The
    far atom of a rotatable bond belongs to the near side's node, and is its own side's origin."""
    place, kind, serial, nodes, rows, stack = [], [], {}, [[-1, None, None]], {0: []}, [0]
    pending = []
    ends = []   # per node: the two atoms on its axis
    for line in text.splitlines():
        if line.startswith("ATOM"):
            i = len(place)
            place.append([float(line[30:38]), float(line[38:46]), float(line[46:54])])
            kind.append(line[77:].strip())
            serial[int(line[6:11])] = i
            if pending:   # the far atom of the branch just opened
                frm, parent = pending.pop()
                rows[parent].append(i)
                ends.append((frm, i))
                nodes.append([parent, i, frm])
                rows[len(nodes) - 1] = []
                stack.append(len(nodes) - 1)
            else:
                rows[stack[-1]].append(i)
        elif line.startswith("BRANCH"):
            pending.append((serial[int(line.split()[1])], stack[-1]))
        elif line.startswith("ENDBRANCH"):
            stack.pop()
    x = np.array(place)
    n = len(x)
    # a branch of one atom turns nothing that has a place of its own: it is no node
    keep = [k for k in range(len(nodes)) if k == 0 or rows[k] or any(m[0] == k for m in nodes[1:])]
    index = {k: j for j, k in enumerate(keep)}
    node_of = np.zeros(n, dtype=int)
    for k in keep:
        node_of[rows[k]] = index[k]
    parent = [index.get(nodes[k][0], -1) for k in keep]
    origin = np.array([x[nodes[k][1]] if k else x[0] for k in keep])
    axis = np.array([x[nodes[k][1]] - x[nodes[k][2]] if k else [0.0, 0.0, 0.0] for k in keep])
    axis[1:] /= np.linalg.norm(axis[1:], axis=1, keepdims=True)
    cov = {"C": 0.77, "N": 0.75, "NA": 0.75, "OA": 0.73, "F": 0.71, "Cl": 0.99, "HD": 0.37}
    c = np.array([cov[k] for k in kind])
    d = np.linalg.norm(x[:, None] - x[None], axis=-1)
    bond = (d < 1.1 * (c[:, None] + c[None])) & ~np.eye(n, dtype=bool)
    xs = np.full(n, 17)
    for i in range(n):
        near = [kind[j] for j in np.flatnonzero(bond[i])]
        donor, acceptor = "HD" in near, kind[i] in ("NA", "OA")
        if kind[i] == "C":
            xs[i] = 1 if any(k not in ("C", "HD") for k in near) else 0
        elif kind[i] in ("N", "NA"):
            xs[i] = 2 + donor + 2 * acceptor
        elif kind[i] == "OA":
            xs[i] = 6 + donor + 2 * acceptor
        elif kind[i] in ("F", "Cl"):
            xs[i] = 12 if kind[i] == "F" else 13
    reach = np.eye(n, dtype=bool)
    for _ in range(3):
        reach = reach | (reach.astype(int) @ bond.astype(int) > 0)
    rigid = node_of[:, None] == node_of[None]
    for k, j in index.items():
        if k:
            for a in ends[k - 1]:
                rigid[a, node_of == j] = True
                rigid[node_of == j, a] = True
            rigid[ends[k - 1][0], ends[k - 1][1]] = rigid[ends[k - 1][1], ends[k - 1][0]] = True
    typed = xs < 17
    ok = ~rigid & ~reach & typed[:, None] & typed[None]
    pairs = np.argwhere(np.triu(ok, 1))
    return x - origin[node_of], node_of, xs, parent, origin, axis, pairs


def _map_values(points, xyz, xs, fast):
    """Values of the 17 maps at points [m][3]."""
    out = torch.zeros((len(points), 17), dtype=torch.float64, device=points.device)
    order = torch.argsort(points[:, 2])
    flat = fast.permute(0, 2, 1).contiguous().reshape(-1, 17)
    step = 2048
    for a in range(0, len(order), step):
        sel = order[a:a + step]
        p = points[sel]
        near = (xyz[:, 2] >= p[:, 2].min() - 8) & (xyz[:, 2] <= p[:, 2].max() + 8)
        q, t = xyz[near], xs[near]
        r2 = ((p[:, None] - q[None]) ** 2).sum(-1)
        i, j = torch.nonzero(r2 <= 64.0, as_tuple=True)
        rows = flat[t[j] * _BINS + (32.0 * r2[i, j]).long()]
        part = torch.zeros((len(sel), 17), dtype=torch.float64, device=points.device)
        part.index_add_(0, i, rows)
        out[sel] = part
    return out


def _rotation(q):
    q = q / q.norm(dim=-1, keepdim=True)
    w, x, y, z = q.unbind(-1)
    return torch.stack([w * w + x * x - y * y - z * z, 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), w * w - x * x + y * y - z * z, 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), w * w - x * x - y * y + z * z], -1).reshape(q.shape[:-1] + (3, 3))


def _curl(e, d, v=10.0):
    t = torch.where(e > 0, v / (v + e.clamp(min=0.0)), torch.ones_like(e))
    return e * t, d * (t * t)[..., None]


def _frames(conf, parent, origin, axis):
    """Per node: rotation and origin in the lab, and the lab axis of its torsion."""
    R, O, X = [_rotation(conf[:, 3:7])], [conf[:, :3]], [torch.zeros_like(conf[:, :3])]
    for k in range(1, len(parent)):
        p = parent[k]
        h = conf[:, 6 + k] / 2
        local = _rotation(torch.cat([torch.cos(h)[:, None], torch.sin(h)[:, None] * axis[k]], -1))
        X.append(R[p] @ axis[k])
        O.append(O[p] + R[p] @ (origin[k] - origin[p]))
        R.append(R[p] @ local)
    return torch.stack(R, 1), torch.stack(O, 1), torch.stack(X, 1)


def _energies(text, conf, xyz, xs_rec, box, slope=1e6):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    smooth, dor, fast = _tables(dev)
    local, node_of, xs, parent, origin, axis, pairs = _model(text)
    f64 = lambda a: torch.as_tensor(np.asarray(a, dtype=np.float64), device=dev)  # noqa: E731
    local, origin, axis, conf = f64(local), f64(origin), f64(axis), f64(conf)
    xyz, xs_rec = f64(xyz), torch.as_tensor(np.asarray(xs_rec, dtype=np.int64), device=dev)
    node = torch.as_tensor(node_of, device=dev)
    typed = torch.as_tensor(np.flatnonzero(xs < 17), device=dev)
    t_of = torch.as_tensor(xs[xs < 17], device=dev)
    pa, pb = (torch.as_tensor(pairs[:, k].copy(), device=dev) for k in (0, 1))
    ta, tb = (torch.as_tensor(xs[pairs[:, k]], device=dev) for k in (0, 1))
    lo, n_cells = f64(list(box.begin)), torch.tensor(list(box.n), device=dev)
    factor = n_cells / f64(np.array(box.end) - np.array(box.begin))
    dims = n_cells + 1
    below = torch.zeros((len(parent), len(parent)), dtype=torch.float64, device=dev)
    for k in range(len(parent)):   # below[k][j]: node j lies in the subtree of k
        j = k
        while j >= 0:
            below[j, k] = 1.0
            j = parent[j]
    corner = torch.tensor([[i, j, k] for k in (0, 1) for j in (0, 1) for i in (0, 1)], device=dev)
    step = max(1, 12_000_000 // max(1, len(pairs) + 8 * len(xs)))
    places, cells = [], []
    for a in range(0, len(conf), step):
        R, O, X = _frames(conf[a:a + step], parent, origin, axis)
        x = O[:, node] + (R[:, node] @ local[None, :, :, None])[..., 0]
        s = (x[:, typed] - lo) * factor
        cell = torch.minimum(s.clamp(min=0.0).long(), n_cells - 1)
        places.append((x, s, O, X))
        c = cell[:, :, None] + corner
        cells.append(torch.unique((c[..., 2] * dims[1] + c[..., 1]) * dims[0] + c[..., 0]))
    need = torch.unique(torch.cat(cells))
    grid = torch.stack([need % dims[0], need // dims[0] % dims[1], need // (dims[0] * dims[1])], -1)
    values = _map_values(lo + grid / factor, xyz, xs_rec, fast)
    where = torch.zeros(int(dims.prod()), dtype=torch.int64, device=dev)
    where[need] = torch.arange(len(need), device=dev)
    es, gs = [], []
    for x, s, O, X in places:
        f = torch.zeros_like(x)
        inside = (s >= 0) & (s < n_cells)
        out = torch.where(s < 0, -1.0, torch.where(inside, 0.0, 1.0)).double()
        miss = torch.where(s < 0, -s, torch.where(inside, torch.zeros_like(s), s - n_cells))
        cell = torch.minimum(s.clamp(min=0.0).long(), n_cells - 1)
        u = torch.where(inside, s - cell, torch.where(s < 0, torch.zeros_like(s), torch.ones_like(s)))
        c = cell[:, :, None] + corner
        v = values[where[(c[..., 2] * dims[1] + c[..., 1]) * dims[0] + c[..., 0]], t_of[None, :, None]]
        w = torch.where(corner.bool(), u[:, :, None], 1 - u[:, :, None])
        sign = corner * 2.0 - 1.0
        e = (v * w.prod(-1)).sum(-1)
        d = torch.stack([(v * sign[:, k] * w[..., [m for m in range(3) if m != k]].prod(-1)).sum(-1) for k in range(3)], -1)
        e, d = _curl(e, d)
        d = factor * torch.where(inside, d, torch.zeros_like(d)) + slope * out
        total = (e + slope * (miss / factor).sum(-1)).sum(-1)
        f[:, typed] = d
        r = x[:, pb] - x[:, pa]
        r2 = (r * r).sum(-1)
        near = r2 < 64.0
        b = (32.0 * r2).clamp(max=2047.0)
        i = torch.where(near, b.long(), torch.zeros_like(pa))
        rem = b - i
        e = smooth[ta, tb, i] + rem * (smooth[ta, tb, i + 1] - smooth[ta, tb, i])
        k = dor[ta, tb, i] + rem * (dor[ta, tb, i + 1] - dor[ta, tb, i])
        e, d = _curl(e, k[..., None] * r)
        total = total + (e * near).sum(-1)
        d = d * near[..., None]
        f.index_add_(1, pb, d)
        f.index_add_(1, pa, -d)
        one = torch.zeros((x.shape[0], len(parent), 6), dtype=torch.float64, device=dev)
        one.index_add_(1, node, torch.cat([f, torch.cross(x - O[:, :1], f, dim=-1)], -1))
        sub = torch.einsum("kj,cjx->ckx", below, one)
        M = sub[..., 3:] - torch.cross(O - O[:, :1], sub[..., :3], dim=-1)
        tors = (M * X).sum(-1)[:, 1:]
        es.append(total)
        gs.append(torch.cat([sub[:, 0], tors], -1))
    return torch.cat(es), torch.cat(gs)


def exact(case, seed):
    """Energies and gradients in 64 bits; searches and refinements have no such value (which
    minimum a pose ends in is decided by comparisons)."""
    if case["kind"] not in ("score", "adjoint", "maps"):
        return None
    xyz, xs, box = _scene(case, seed)
    text = _ligand(case, seed)
    return _energies(text, _poses(text, case["n"], box, seed), xyz, xs, box)
