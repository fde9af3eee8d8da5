"""Captured batches (vd_set_graphs) follow the maps: another box captures the batch again, the same box
populated again is read by the replay; every pass gives the eager results bit for bit."""
import numpy as np
import pytest

from helpers import say

pytestmark = pytest.mark.gpu


def results(ctx, n):
    return [ctx.batch_results(k) for k in range(n)]


def same(a, b):
    return all(np.array_equal(x, y) for ra, rb in zip(a, b) for x, y in zip(ra, rb))


def test_graph_follows_the_box(module_ctx):
    import vdock
    ctx = module_ctx
    ctx.set_receptor(*vdock.synth_receptor(2000, 36.0, 8.0, 42))
    ids = [ctx.add_ligand(vdock.synth_ligand(14 + 5 * k, 2 + 2 * k, 300 + k)) for k in range(4)]
    p = vdock.default_params(chains=64, search_depth=3, bfgs_steps=8, seed=5, chains_per_wave=4, waves_per_simd=3)
    first = vdock.box_from_center([0, 0, 0], [12, 12, 12], 0.375)
    # a larger box moves the maps, a smaller one leaves them where they are
    boxes = [first, vdock.box_from_center([1, 0, 0], [17, 15, 16], 0.375),
             vdock.box_from_center([0, 1, 0], [9, 11, 10], 0.375), first, first]
    ref = []
    for box in boxes:
        ctx.grid_populate(box)
        ctx.dock_batch(ids, p)
        ref.append(results(ctx, len(ids)))
    ctx.set_graphs(True)
    try:
        for k, box in enumerate(boxes):
            ctx.grid_populate(box)
            for r in range(3):
                say("graph", "box", k, "pass", r)
                ctx.dock_batch(ids, p)
                assert same(results(ctx, len(ids)), ref[k])
    finally:
        ctx.set_graphs(False)
