"""Dense BFGS: the matrix takes the LDS of the launch's largest ligand, and the 64-lane class of a batch
runs at three waves per SIMD.  Chains must not change: each ligand of a batch is compared bit for bit
with its own launch, where the matrix is sized for it alone and the budget is two."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# a library's ligands, (heavy atoms, torsions, seed): the smallest and largest matrix of a class side by side
@pytest.mark.parametrize("lanes,specs", [
    (64, [(60, 16, 1), (24, 10, 2), (70, 20, 3)]),
    (64, [(150, 57, 5), (30, 11, 6), (120, 40, 4)]),
    (16, [(8, 0, 7), (20, 9, 8), (12, 1, 9)]),
    (32, [(14, 3, 10), (40, 25, 11)])])
def test_batch_equals_single_launches(module_ctx, lanes, specs):
    import vdock
    from vdock import workloads
    print("lanes", lanes, specs, flush=True)
    ctx = module_ctx
    workloads.small_scene(vdock, ctx)
    ids = [ctx.add_ligand(vdock.synth_ligand(*s)) for s in specs]
    kw = dict(chains=9, search_depth=4, bfgs_steps=7, seed=3, local_search=0)
    ctx.dock_batch(ids, vdock.default_params(chains_per_wave=64 // lanes, **kw))
    launches = ctx.last_launches()
    assert [l.lanes_per_chain for l in launches] == [lanes]
    assert launches[0].waves_per_simd == 3 or lanes < 64 or specs[0][0] > 100   # LDS for two only
    batch = [ctx.batch_results(k) for k in range(len(ids))]
    for k, i in enumerate(ids):
        e, conf, heavy, _ = ctx.dock(i, vdock.default_params(chains_per_wave=64 // lanes, **kw))
        assert np.isfinite(e).all()
        for a, b in zip(batch[k], (e, conf, heavy)):
            assert np.array_equal(a, b), specs[k]
