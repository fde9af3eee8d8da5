"""The launch rules on the host: the header is compiled into a small library of its own, so every line
is checked without a device.  256 compute units, an MI355X's."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import ROOT

CUS = 256
SHIM = """
#include "launch_rules.h"
extern "C" {
int refine_waves(int n_cu, long long poses, long long atoms) { return vd::refine_waves(n_cu, poses, atoms); }
size_t grown_size(size_t have, size_t need, size_t least, size_t most) { return vd::grown_size(have, need, least, most); }
int dense_waves(int lanes, int batch) { return vd::dense_waves(lanes, batch != 0); }
int trial_waves(int lanes, int rilc, int batch, int* out) {
  const std::vector<int> w = vd::trial_waves(lanes, rilc != 0, batch != 0);
  std::copy(w.begin(), w.end(), out);
  return (int)w.size();
}
// (lanes, waves, wide) per ligand -> launches (size, first ligand of each to out), overlap
int classes(int n, const int* lanes, const int* waves, const int* wide, int* out, int* overlap) {
  std::vector<vd::LigPlan> plans;
  for (int k = 0; k < n; ++k) plans.push_back(vd::LigPlan{k, lanes[k], waves[k], 1, 1, 1, 1, 1, wide[k] != 0});
  const vd::Classes c = vd::batch_classes(plans);
  for (const auto& e : c) { *out++ = (int)e.second.size(); *out++ = e.second[0]; }
  *overlap = vd::may_overlap(c);
  return (int)c.size();
}
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC",
                           "-I", os.path.join(ROOT, "vina-cuda_amd", "csrc"), "-o", str(d / "shim.so"), str(d / "shim.cpp")])
    return C.CDLL(str(d / "shim.so"))


# (atoms of every ligand, poses, wavefronts per pose): sizes at which one of the two took at least 1.1
# times the other's time
@pytest.mark.parametrize("atoms,poses,waves", [
    (1, 20, 1), (3, 500, 1), (6, 1000, 1), (11, 500, 4), (11, 1000, 1), (11, 2000, 1), (14, 1000, 4), (14, 2000, 1),
    (17, 1100, 4), (17, 1800, 1), (21, 1400, 4), (24, 1100, 4), (24, 2000, 1), (28, 1500, 4), (34, 2000, 4), (42, 2000, 4),
    (64, 2000, 4), (64, 2049, 1), (64, 5120, 1), (42, 20, 4)])
def test_refinement_takes_the_faster_form(rules, atoms, poses, waves):
    f = rules.refine_waves
    f.argtypes = [C.c_int, C.c_longlong, C.c_longlong]
    assert f(CUS, poses, atoms * poses) == waves
    assert f(CUS, 0, 0) == 1


def classes(rules, plans):
    n = len(plans)
    a = [(C.c_int * n)(*col) for col in zip(*plans)]
    out, overlap = (C.c_int * (2 * n))(), C.c_int()
    k = rules.classes(n, *a, out, C.byref(overlap))
    return [(out[2 * i], out[2 * i + 1]) for i in range(k)], bool(overlap.value)


def test_wide_ligands_of_any_budget_share_one_launch(rules):
    # two 16-lane budgets, as the autotuner may choose, heavy ligands in both
    assert classes(rules, [(16, 3, 0), (16, 4, 0), (16, 3, 1), (16, 4, 1)]) == ([(2, 2), (1, 0), (1, 1)], True)
    assert classes(rules, [(16, 3, 1), (64, 3, 0), (16, 3, 0)]) == ([(1, 0), (1, 2), (1, 1)], True)
    assert classes(rules, [(16, 3, 1), (16, 2, 1)]) == ([(2, 0)], False)


def test_classes_that_run_one_after_the_other(rules):
    assert classes(rules, [(16, 3, 0), (64, 3, 0)]) == ([(1, 0), (1, 1)], True)
    assert classes(rules, [(16, 3, 0)]) == ([(1, 0)], False)
    assert classes(rules, [(16, 3, 0), (32, 3, 0), (64, 3, 0)])[1] is False
    assert classes(rules, [(16, 3, 1), (16, 3, 0), (32, 3, 0), (64, 3, 0)])[1] is False


@pytest.mark.parametrize("lanes", [16, 32, 64])
@pytest.mark.parametrize("batch", [0, 1])
def test_autotuner_times_what_the_call_runs(rules, lanes, batch):
    out = (C.c_int * 4)()
    trials = out[:rules.trial_waves(lanes, 0, batch, out)]
    assert trials == [rules.dense_waves(lanes, batch)] == [3 if lanes == 64 and batch else 2]
    assert out[:rules.trial_waves(lanes, 1, batch, out)] == [3, 4, 2]


def test_growing_arrays_cost_few_allocations(rules):
    f = rules.grown_size
    f.argtypes, f.restype = [C.c_size_t] * 4, C.c_size_t
    least, most = 4096, 1 << 20
    have, allocations = 0, 0
    for need in range(1, most + 1, 97):
        new = f(have, need, least, most)
        assert need <= new <= most and new >= least
        allocations += new != have
        have = new
    assert allocations <= 10
    assert f(0, 300000, least, most) == 300000   # the first one takes what it needs
    assert f(5000, 100, least, most) == 5000
    assert f(900000, 1000000, least, most) == most
