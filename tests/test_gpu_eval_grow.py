"""vd_eval on host arrays that grow from call to call, past the size up to which the kernel reads and
writes them in place: every call gives what one call on all poses gives, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heavy,tors", [(20, 5), (60, 16)])
def test_growing_arrays(module_ctx, heavy, tors):
    import vdock
    from vdock import workloads
    ctx = module_ctx
    workloads.small_scene(vdock, ctx)
    lid = ctx.add_ligand(vdock.synth_ligand(heavy, tors, 6))
    T = ctx.ligand_info(lid).n_torsions
    rng = np.random.default_rng(heavy)
    sizes = [1, 2, 3, 100, 101, 700, 3000, 9000, 20000, 50000, 7, 9001]
    c = np.zeros((max(sizes), 7 + T), dtype=np.float32)
    c[:, :3] = rng.uniform(-6, 6, (len(c), 3))
    q = rng.normal(size=(len(c), 4))
    c[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    c[:, 7:] = rng.uniform(-np.pi, np.pi, (len(c), T))
    own = vdock.Context(0)   # nothing taken yet
    workloads.small_scene(vdock, own)
    mine = own.add_ligand(vdock.synth_ligand(heavy, tors, 6))
    e, g = ctx.eval(lid, c)
    for n in sizes:
        a, b = own.eval(mine, c[-n:])
        assert np.array_equal(a, e[-n:]) and np.array_equal(b, g[-n:]), n
    own.close()
