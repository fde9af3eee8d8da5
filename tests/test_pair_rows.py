"""The rows of the device's pair table are shared by type pairs of equal radius sum, hydrophobic
match and hydrogen-bond match: the tables of such type pairs are equal bit for bit under any
weights (CPU), and ligands of every atom type score as the FP64 oracle scores them (GPU)."""
import numpy as np
import pytest

import oracle as orc
from helpers import intra_cutoff_bound

RADIUS = [1.9, 1.9, 1.8, 1.8, 1.8, 1.8, 1.7, 1.7, 1.7, 1.7, 2.0, 2.1, 1.5, 1.8, 2.0, 2.2, 1.2]
HYDROPHOBIC, ACCEPTOR, DONOR = {0, 12, 13, 14, 15}, {4, 5, 8, 9}, {3, 5, 7, 9, 16}


@pytest.mark.parametrize("weights", [(-0.035579, -0.005156, 0.840245, -0.035069, -0.587439, 0.05846),
                                     (0.3, -1.7, 0.0, 0.11, 2.9, 0.0)])
def test_type_pairs_of_one_class_have_one_table(weights):
    import vdock
    ctx = vdock.Context(-1)
    ctx.set_weights(weights)
    rows = {}
    for b in range(17):
        for a in range(b + 1):
            key = (RADIUS[a] + RADIUS[b], a in HYDROPHOBIC and b in HYDROPHOBIC,
                   (a in DONOR and b in ACCEPTOR) or (b in DONOR and a in ACCEPTOR))
            table = np.stack(ctx.lut(a + b * (b + 1) // 2)[:2]).tobytes()
            assert rows.setdefault(key, table) == table, (a, b)
    assert len(rows) < 60


KINDS = ["C", "S", "P", "F", "Cl", "Br", "I", "N", "NA", "OA", "SA", "A", "Zn", "HD"]


def chain_ligand(n, start, step):
    """n atoms in a zigzag, three to a rigid piece, their AutoDock types taken in turn from KINDS."""
    lines, opened = ["ROOT"], []
    for i in range(n):
        if i and i % 3 == 0:
            if i == 3:
                lines.append("ENDROOT")
            lines.append("BRANCH %3d %3d" % (i, i + 1))
            opened.append((i, i + 1))
        kind = KINDS[(start + step * i) % len(KINDS)]
        xyz = (1.5 * i, 0.9 * (i % 2), 0.35 * (i % 5))
        lines.append("ATOM  %5d  %-3s UNL     1    %8.3f%8.3f%8.3f  0.00  0.00    %+6.3f %-2s" % (i + 1, "X", *xyz, 0.0, kind))
    if not opened:
        lines.append("ENDROOT")
    lines += ["ENDBRANCH %3d %3d" % b for b in reversed(opened)]
    return "\n".join(lines + ["TORSDOF %d" % len(opened)]) + "\n"


@pytest.mark.gpu
@pytest.mark.parametrize("n,start,step", [(3, 0, 1), (16, 0, 1), (17, 3, 5), (28, 0, 3), (30, 5, 9), (64, 1, 1), (65, 7, 3)])
def test_every_atom_type_scores_as_the_oracle(ctx, n, start, step):
    import vdock
    print("chain of", n, start, step, flush=True)
    text = chain_ligand(n, start, step)
    box = vdock.box_from_center([0, 0, 0], [120, 120, 120], 8.0)
    maps = np.zeros((17,) + box.dims[::-1], dtype=np.float32)
    ctx.grid_upload(box, maps)
    lid, lig = ctx.add_ligand(text), orc.Ligand(text)
    b, e, dims = box.as_tuple()
    grid = orc.Grid(orc.Lut(), b, e, dims)
    grid.set_maps(maps.astype(np.float64))
    rng = np.random.default_rng(n)
    conf = np.zeros((40, 7 + lig.T), dtype=np.float32)
    conf[:, :3] = rng.uniform(-1, 1, (40, 3))
    q = rng.normal(size=(40, 4))
    conf[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    conf[:, 7:] = rng.uniform(-np.pi, np.pi, (40, lig.T))
    for cpw in (0, 1):
        energy, grad = ctx.eval(lid, conf, chains_per_wave=cpw)
        for k in range(40):
            ref, gref, _, _ = orc.eval_deriv(grid, lig, conf[k].astype(np.float64))
            assert abs(energy[k] - ref) <= max(1e-4, 1e-3 * abs(ref)) + intra_cutoff_bound(lig, conf[k])
            assert np.abs(grad[k] - gref).max() <= 1e-3 * max(1.0, np.abs(gref).max()) + 1e-4


@pytest.mark.gpu
@pytest.mark.parametrize("types", [range(17), (0,), (1, 10, 11, 2, 6), (12, 13, 14, 15), (3, 7, 16), (4, 8), (5, 9)])
def test_maps_of_every_receptor_type(module_ctx, types):
    """The map kernel's rows, by class of receptor type: plain, hydrophobic, donor, acceptor, both.
    Tolerance as test_gpu_core.py: 1e-4 relative plus the change of an r^2 within 0.003 bins of an edge."""
    import vdock
    print("receptor types", list(types), flush=True)
    xyz, _ = vdock.synth_receptor(700, 26.0, 3.0, 9)
    xs = np.array([list(types)[i % len(types)] for i in range(len(xyz))], dtype=np.int32)
    box = vdock.box_from_center([1.0, -2.0, 0.5], [5.5, 3.0, 4.2], 0.375)
    module_ctx.set_receptor(xyz, xs)
    module_ctx.grid_populate(box)
    maps = module_ctx.grid_download()
    b, e, n = box.as_tuple()
    grid = orc.Grid(orc.Lut(), b, e, n)
    grid.set_receptor(xyz.astype(np.float64), xs)
    slack = grid.populate_with_slack(0.003)
    ref = grid.maps()
    assert (np.abs(maps - ref) <= 1e-4 * np.maximum(1.0, np.abs(ref)) + slack).all()
