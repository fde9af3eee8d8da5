"""The two forms of the refinement kernel -- four wavefronts per pose for launches of few poses, one
for many -- give the same poses, coordinates and energies bit for bit (the few-pose form is compared
with the FP64 oracle in test_gpu_post.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MANY = 8 * 256 + 13   # more poses than the four-wavefront form takes on 256 CUs


@pytest.fixture(scope="module")
def scene(module_ctx):
    import vdock
    from vdock import workloads
    workloads.small_scene(vdock, module_ctx)
    return module_ctx


# atoms beyond a wavefront's lanes, one and several rounds of pair chunks, no pairs at all, one
# atom, a deep tree
@pytest.mark.parametrize("heavy,tors,seed", [(1, 0, 1), (3, 0, 2), (9, 2, 3), (24, 3, 4), (50, 9, 5), (60, 16, 6),
                                             (66, 8, 7), (90, 24, 8)])
def test_both_forms_agree_bit_for_bit(scene, heavy, tors, seed):
    import vdock
    print("ligand", heavy, tors, flush=True)
    lid = scene.add_ligand(vdock.synth_ligand(heavy, tors, seed))
    T = scene.ligand_info(lid).n_torsions
    rng = np.random.default_rng(seed)
    conf = np.zeros((7, 7 + T), dtype=np.float32)
    conf[:, :3] = rng.uniform(-9, 9, (7, 3))   # some outside the 20 A box
    q = rng.normal(size=(7, 4))
    conf[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
    conf[:, 7:] = rng.uniform(-np.pi, np.pi, (7, T))
    p = vdock.post_params(max_steps=6)
    few = scene.refine(lid, conf, p)
    pick = np.arange(MANY) % 7
    many = scene.refine(lid, conf[pick], p)
    for a, b in zip(few[:2], many[:2]):
        assert np.array_equal(a[pick], b)
    key = [(r.e, r.e_inter, r.e_intra, r.inside) for r in few[2]]
    assert [key[k] for k in pick] == [(r.e, r.e_inter, r.e_intra, r.inside) for r in many[2]]


@pytest.mark.parametrize("poses", [3, 400])
def test_heaviest_first_keeps_every_pose_in_its_place(scene, poses):
    """Workgroups start with the heaviest ligands' poses: a library gives what each ligand gives alone."""
    import vdock
    specs = [(9, 2, 21), (50, 9, 22), (1, 0, 23), (24, 3, 24), (33, 8, 25), (12, 4, 26)]
    ids, confs = [], []
    for s in specs:
        ids.append(scene.add_ligand(vdock.synth_ligand(*s)))
        T = scene.ligand_info(ids[-1]).n_torsions
        rng = np.random.default_rng(s[2])
        c = np.zeros((poses, 7 + T), dtype=np.float32)
        c[:, :3] = rng.uniform(-6, 6, (poses, 3))
        q = rng.normal(size=(poses, 4))
        c[:, 3:7] = q / np.linalg.norm(q, axis=1, keepdims=True)
        c[:, 7:] = rng.uniform(-np.pi, np.pi, (poses, T))
        confs.append(c)
    p = vdock.post_params(max_steps=3)
    print("poses", poses, flush=True)
    scene.postprocess(ids, confs, p)
    both = [scene.post_results(k) for k in range(len(ids))]
    for k, i in enumerate(ids):
        scene.postprocess([i], [confs[k]], p)
        modes, conf, xyz = scene.post_results(0)
        assert [(m.pose, m.e, m.rmsd_lb, m.rmsd_ub) for m in modes] == [(m.pose, m.e, m.rmsd_lb, m.rmsd_ub) for m in both[k][0]]
        assert np.array_equal(conf, both[k][1]) and np.array_equal(xyz, both[k][2])
