"""Wide launches -- a batch's heaviest 16-lane ligands, one chain per wavefront -- give the results of
the 16-lane kernel bit for bit.  All but the lightest ligands of a batch this small are docked wide
when the launch shape is left to the library; vd_dock with four chains per wavefront runs the 16-lane kernel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (heavy atoms, torsions, seed): just beyond 16 atoms, around 64 lanes, two atoms per lane, rigid
# (no pairs), fewer pairs than a pass holds
LIGANDS = [(17, 0, 1), (17, 1, 2), (20, 9, 3), (33, 7, 4), (52, 9, 5), (54, 8, 6), (60, 9, 7), (66, 5, 8)]


@pytest.fixture(scope="module")
def docked(module_ctx):
    import vdock
    from vdock import workloads
    workloads.small_scene(vdock, module_ctx)
    ids = [module_ctx.add_ligand(vdock.synth_ligand(*s)) for s in LIGANDS]
    atoms = [module_ctx.ligand_info(i).n_atoms for i in ids]
    print("atoms", atoms, flush=True)
    assert min(atoms) > 16 and max(atoms) > 64
    return module_ctx, ids


@pytest.mark.parametrize("policy,local_search,depth", [(0, 1, 6), (1, 1, 70), (0, 0, 4)])
@pytest.mark.parametrize("chains", [1, 6, 33])
def test_wide_equals_narrow_bit_for_bit(docked, policy, local_search, depth, chains):
    import vdock
    ctx, ids = docked
    print("policy", policy, "search", local_search, "chains", chains, flush=True)
    kw = dict(chains=chains, policy=policy, local_search=local_search, search_depth=depth, seed=5)
    st = ctx.dock_batch(ids, vdock.default_params(**kw))
    launches = ctx.last_launches()
    # the wide launch comes first, an item per chain; at most the lightest ligands are left out of it
    assert all(l.lanes_per_chain == 16 for l in launches) and len(launches) <= 2
    assert launches[0].items % chains == 0 and launches[0].items >= (len(ids) - 2) * chains
    wide = [ctx.batch_results(k) for k in range(len(ids))]
    evals = 0
    for k, i in enumerate(ids):
        e, conf, heavy, s = ctx.dock(i, vdock.default_params(chains_per_wave=4, **kw))
        evals += s.evals
        for a, b in zip(wide[k], (e, conf, heavy)):
            assert np.array_equal(a, b), LIGANDS[k]
    assert st.evals == evals


def test_three_launches_at_once(docked):
    """Wide, 16-lane and 64-lane launches of one batch against the 16- and 64-lane ones in turn (no
    launch goes wide without overlap): equal results."""
    import vdock
    ctx, _ = docked
    specs = [(60, 9, 7)] + [(18, 2, 100 + k) for k in range(40)] + [(40, 12, 8), (30, 11, 9)]
    ids = [ctx.add_ligand(vdock.synth_ligand(*s)) for s in specs]
    p = vdock.default_params(chains=320, seed=3, search_depth=3)
    got = []
    for on in (True, False):
        ctx.set_class_overlap(on)
        ctx.dock_batch(ids, p)
        got.append([ctx.batch_results(k) for k in range(len(ids))])
        print("items per launch", [l.items for l in ctx.last_launches()], flush=True)
        assert len(ctx.last_launches()) == (3 if on else 2)
    ctx.set_class_overlap(True)
    for a, b in zip(*got):
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
