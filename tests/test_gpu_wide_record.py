"""What vd_last_launches says of wide launches -- that they are wide, the budget their kernel is built
for, the name a profiler lists -- and, by that, that a batch really docked wide where its results are
compared with the 16-lane kernel's bit for bit: with one chain per ligand, where the number of items
tells nothing."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIGANDS = [(17, 1, 2), (20, 9, 3), (33, 7, 4), (60, 9, 7), (66, 5, 8)]


@pytest.fixture(scope="module")
def docked(module_ctx):
    import vdock
    from vdock import workloads
    workloads.small_scene(vdock, module_ctx)
    return module_ctx, [module_ctx.add_ligand(vdock.synth_ligand(*s)) for s in LIGANDS]


@pytest.mark.parametrize("policy,local_search,mode", [(0, 0, 0), (0, 1, 1), (1, 1, 2)])
@pytest.mark.parametrize("chains", [1, 5])
def test_record_of_a_wide_launch(docked, policy, local_search, mode, chains):
    import vdock
    ctx, ids = docked
    print("mode", mode, "chains", chains, flush=True)
    kw = dict(chains=chains, policy=policy, local_search=local_search, search_depth=5, seed=2)
    ctx.dock_batch(ids, vdock.default_params(**kw))
    launches = ctx.last_launches()
    got = [ctx.batch_results(k) for k in range(len(ids))]
    first = launches[0]
    assert first.wide == 1 and first.kernel == "vd_mc_wide_kernel<16, %d, 3>" % mode
    assert (first.lanes_per_chain, first.waves_per_simd, first.items) == (16, 3, first.ligands * chains)
    assert all(r.wide == 0 and r.kernel.startswith("vd_mc_kernel<16, %d, " % mode) for r in launches[1:])
    assert sum(r.ligands for r in launches) == len(ids) and first.ligands >= len(ids) - 2
    # left to themselves and four to a wavefront
    ctx.dock_batch(ids, vdock.default_params(chains_per_wave=4, **kw))
    assert [r.wide for r in ctx.last_launches()] == [0]
    for k in range(len(ids)):
        for a, b in zip(got[k], ctx.batch_results(k)):
            assert np.array_equal(a, b), LIGANDS[k]
