"""vd_eval's ways in and out -- small host arrays read and written by the kernel, large ones copied,
device pointers -- and its kept ligand record give the same numbers bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIRECT = 4 << 20   # bytes of host arrays up to which the kernel reads and writes them itself


def poses(n, T, seed):
    rng = np.random.default_rng(seed)
    c = np.zeros((n, 7 + T), dtype=np.float32)
    c[:, :3] = rng.uniform(-6, 6, (n, 3))
    q = rng.normal(size=(n, 4))
    c[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    c[:, 7:] = rng.uniform(-np.pi, np.pi, (n, T))
    return c


def through_device(ctx, lid, c, cpw):
    n, m = c.shape
    ptrs = [ctx.alloc(4 * n * k) for k in (m, 1, m - 1)]
    try:
        ctx._check(ctx.lib.vd_copy(ctx.h, ptrs[0], c.ctypes.data, c.nbytes, 0))
        ctx.eval_device(lid, *ptrs, n, chains_per_wave=cpw)
        return ctx.to_host(ptrs[1], (n,)), ctx.to_host(ptrs[2], (n, m - 1))
    finally:
        for p in ptrs:
            ctx.free(p)


@pytest.mark.parametrize("heavy,tors,cpw", [(1, 0, 0), (12, 0, 4), (20, 9, 4), (20, 5, 2), (30, 10, 0), (75, 24, 1)])
def test_every_path_gives_the_same_numbers(module_ctx, heavy, tors, cpw):
    import vdock
    from vdock import workloads
    ctx = module_ctx
    workloads.small_scene(vdock, ctx)
    lid = ctx.add_ligand(vdock.synth_ligand(heavy, tors, 3))
    other = ctx.add_ligand(vdock.synth_ligand(9, 2, 4))
    T = ctx.ligand_info(lid).n_torsions
    edge = DIRECT // 4 // (14 + 2 * T)   # poses that just fit
    print("ligand", heavy, T, "poses", edge, flush=True)
    c = poses(edge + 1, T, heavy)
    e, g = through_device(ctx, lid, c, cpw)
    for n in (1, 2, 5, 64, edge, edge + 1):
        a, b = ctx.eval(lid, c[:n], chains_per_wave=cpw)
        assert np.array_equal(a, e[:n]) and np.array_equal(b, g[:n]), n
        ctx.eval(other, poses(3, ctx.ligand_info(other).n_torsions, n))   # another ligand's record in between
    assert ctx.eval_last_ms() > 0
    ctx.set_weights([2 * w for w in vdock.DEFAULT_WEIGHTS])
    workloads.small_scene(vdock, ctx)
    e2, g2 = through_device(ctx, lid, c[:50], cpw)
    a, b = ctx.eval(lid, c[:50], chains_per_wave=cpw)
    ctx.set_weights(vdock.DEFAULT_WEIGHTS)
    assert np.array_equal(a, e2) and np.array_equal(b, g2)
    if heavy > 9:
        assert not np.array_equal(a, e[:50])
