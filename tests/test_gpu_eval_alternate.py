"""vd_eval of several ligands in turn: a ligand's record is copied ahead of its kernel without a wait in
between.  Every call gives what the same call gives in a context of its own, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# records from a few hundred bytes to some 40 KB, every lane count
LIGANDS = [(90, 24, 1), (3, 0, 2), (60, 9, 3), (1, 0, 4), (40, 20, 5)]


def poses(n, T, seed):
    rng = np.random.default_rng(seed)
    c = np.zeros((n, 7 + T), dtype=np.float32)
    c[:, :3] = rng.uniform(-6, 6, (n, 3))
    q = rng.normal(size=(n, 4))
    c[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    c[:, 7:] = rng.uniform(-np.pi, np.pi, (n, T))
    return c


@pytest.mark.parametrize("n", [1, 30, 40000])   # the last beyond the arrays the kernel reads in place
def test_ligands_in_turn(module_ctx, n):
    import vdock
    from vdock import workloads
    ctx = module_ctx
    workloads.small_scene(vdock, ctx)
    texts = [vdock.synth_ligand(*s) for s in LIGANDS]
    ids = [ctx.add_ligand(t) for t in texts]
    confs = [poses(n, ctx.ligand_info(i).n_torsions, k) for k, i in enumerate(ids)]
    want = []
    for t, c in zip(texts, confs):
        own = vdock.Context(0)
        workloads.small_scene(vdock, own)
        want.append(own.eval(own.add_ligand(t), c))
        own.close()
    print("poses", n, flush=True)
    for order in ([0, 1, 2, 3, 4], [4, 3, 0, 1, 0, 2], [2, 2, 1, 4, 4]):
        for k in order:
            e, g = ctx.eval(ids[k], confs[k])
            assert np.array_equal(e, want[k][0]) and np.array_equal(g, want[k][1]), (n, LIGANDS[k])
    with pytest.raises(vdock.VdockError):   # a refused call leaves the kept record as it is
        ctx.eval(10**6, confs[0])
    e, g = ctx.eval(ids[4], confs[4])
    assert np.array_equal(e, want[4][0]) and np.array_equal(g, want[4][1])
