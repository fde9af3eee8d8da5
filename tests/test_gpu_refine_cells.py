"""The refinement's receptor lists, built on the device: wherever an atom of a pose lies in the box, the
inter energy of the refined pose is the FP64 oracle's direct sum over the receptor.  An atom missing
from a list, or listed twice, changes the sum; the bound is that of the refinement's
other comparisons with the oracle (energies and coordinates come back in FP32)."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


# (receptor atoms, cube, cavity, box): empty lists; rows of more than 64 atoms; one cell; more than 64
# rows of bins per cell; unequal edges; a box beside the receptor
@pytest.mark.parametrize("n,cube,cavity,center,size", [
    (3, 60.0, 10.0, (0, 0, 0), (12.0, 12.0, 12.0)), (2500, 14.0, 0.5, (0, 0, 0), (6.0, 9.0, 3.0)),
    (1000, 30.0, 4.0, (1.0, 2.0, 3.0), (1.2, 0.8, 1.9)), (1500, 36.0, 6.0, (0.5, -1.0, 0.0), (7.1, 23.9, 11.3)),
    (1500, 36.0, 6.0, (22.0, 0, 0), (10.0, 10.0, 10.0))])
def test_every_receptor_atom_is_listed_once(ctx, n, cube, cavity, center, size):
    import vdock
    print("receptor", n, "box", size, flush=True)
    xyz, xs = vdock.synth_receptor(n, cube, cavity, 5)
    ctx.set_receptor(xyz, xs)
    box = vdock.box_from_center(list(center), list(size), 0.375)
    ctx.grid_populate(box)
    b, e, dims = box.as_tuple()
    g = orc.Grid(orc.Lut(), b, e, dims)
    g.set_receptor(xyz.astype(np.float64), xs)
    text = vdock.synth_ligand(1, 0, 3)
    lid, lig = ctx.add_ligand(text), orc.Ligand(text)
    lo, hi = np.array(box.begin), np.array(box.end)
    conf = np.zeros((60, 7), dtype=np.float32)
    conf[:, 3] = 1
    conf[:, :3] = lo + np.random.default_rng(9).uniform(0, 1, (60, 3)) * (hi - lo)
    conf[0, :3], conf[1, :3] = lo, hi
    _, out, res = ctx.refine(lid, conf, vdock.post_params(max_steps=1))
    seen = 0
    for x, r in zip(out, res):
        if not r.inside:
            continue
        ei = orc.noncache_eval(g, lig, x.astype(np.float64))
        assert abs(r.e_inter - ei) <= 1e-3 + 1e-5 * abs(ei), (x, r.e_inter, ei)
        seen += 1
    assert seen >= 10
