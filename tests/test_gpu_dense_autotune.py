"""The autotuner under dense BFGS: every ligand's chains are those of a fixed shape, bit for bit, in a
batch (whose 64-lane class runs at three waves per SIMD, as it is timed) and in a launch of its own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec", [(20, 4, 1), (40, 12, 2), (75, 24, 3)])
def test_tuned_dense_chains_are_those_of_a_fixed_shape(module_ctx, spec):
    import vdock
    from vdock import workloads
    ctx = module_ctx
    workloads.small_scene(vdock, ctx)
    lid = ctx.add_ligand(vdock.synth_ligand(*spec))
    kw = dict(chains=12, search_depth=3, bfgs_steps=6, seed=4, local_search=0)
    print("ligand", spec, flush=True)
    ctx.set_autotune(True)
    ctx.dock_batch([lid], vdock.default_params(**kw))
    record, = ctx.last_launches()
    got = ctx.batch_results(0)
    alone = ctx.dock(lid, vdock.default_params(**kw))
    single, = ctx.last_launches()
    ctx.set_autotune(False)
    assert single.waves_per_simd == 2
    # LDS decides whether a third wave fits where there are 64 lanes
    assert record.waves_per_simd == (3 if record.wide else 2) or record.lanes_per_chain == 64
    for r, launch in ((got, record), (alone[:3], single)):
        want = ctx.dock(lid, vdock.default_params(chains_per_wave=64 // launch.lanes_per_chain, **kw))
        for a, b in zip(r, want[:3]):
            assert np.array_equal(a, b)
