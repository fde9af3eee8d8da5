// Launch shapes chosen by size, as plain host functions (no HIP types), so that each line can be checked
// without a device.
#pragma once
#include <algorithm>
#include <cstddef>
#include <map>
#include <tuple>
#include <vector>

namespace vd {

// The size to give a buffer of `have` elements that must hold `need`: at least twice what it had, within
// [least, most], so that arrays that grow from call to call cost a few allocations and not one each
// (60 calls of vd_eval on 100, 150, ... 3,050 poses, page-locked memory: 30 ms taken to size, 4.0 grown,
// 5.9 when the arrays were copied to device buffers taken to size).
inline size_t grown_size(size_t have, size_t need, size_t least, size_t most) {
  if (need <= have) return have;
  return std::max({need, least, std::min(2 * have, most)});
}

// How a ligand of a batch is docked: id; lanes per chain, waves per SIMD; MC steps, local-search
// iterations; torsions, heavy atoms, chains; wide: one chain per wavefront in 16-lane arithmetic.
struct LigPlan { int id, G, W, depth, bfgs, T, H, chains; bool wide = false; };

// The launch classes of a persistent batch: ligand indices per launch form, wide launches first.  There
// is one wide kernel per mode, whatever budget the ligand would have narrow, so all wide ligands go in
// one launch (under the autotuner two 16-lane classes may have two budgets).
struct ClassKey {
  int narrow, G, W;   // narrow: 0 for a wide launch; lanes per chain, waves per SIMD (wide: 0, its kernel's own)
  bool operator<(const ClassKey& o) const { return std::tie(narrow, G, W) < std::tie(o.narrow, o.G, o.W); }
};
using Classes = std::map<ClassKey, std::vector<int>>;
inline Classes batch_classes(const std::vector<LigPlan>& plans) {
  Classes classes;
  for (size_t k = 0; k < plans.size(); ++k) {
    const LigPlan& p = plans[k];
    classes[p.wide ? ClassKey{0, p.G, 0} : ClassKey{1, p.G, p.W}].push_back((int)k);
  }
  return classes;
}

// Overlap applies to batches of exactly two classes, besides a wide launch.  Measured on the
// screening batch (a 16-lane class whose waves mostly wait, a 64-lane class that keeps the vector
// units busy): 3 % shorter steps.  With more classes it lost: on a 4,096-ligand batch of five classes a
// fourth stream shared a hardware queue with the third (four queues per process), and capped classes
// that outlast the uncapped one keep half their CU slots empty to the end.
inline bool may_overlap(const Classes& classes) {
  const bool wide = !classes.empty() && classes.begin()->first.narrow == 0;
  return classes.size() == 2 || (wide && classes.size() == 3);
}

// Waves per SIMD of a dense-BFGS launch: three (168 registers, 144 bytes of spills) for the 64-lane class
// of a batch (nine batches of 96 ligands 1,427 -> 1,311 ms); on 16 lanes a third loses (123 -> 130 ms),
// and a launch of one ligand rarely has the chains for it (24 atoms, 2,048 chains 18.4 -> 19.2 ms).
inline int dense_waves(int G, bool batch) { return G == 64 && batch ? 3 : 2; }

// The budgets the autotuner times for G lanes per chain, in order of preference: those that the call
// would run.
inline std::vector<int> trial_waves(int G, bool rilc, bool batch) {
  return rilc ? std::vector<int>{3, 4, 2} : std::vector<int>{dense_waves(G, batch)};
}

// Wavefronts per pose of a refinement launch of `poses` poses with `pose_atoms` atoms in all, on n_cu
// compute units.  A pose takes some 100 evaluations one after the other, so a launch takes at least as
// long as its longest pose: four wavefronts per pose halve that (20 poses of a 63-atom ligand 4.1 ->
// 2.0 ms), at the price of the slots in which three wait while the first walks the tree.  As long as one
// wavefront per pose would leave no pose waiting for a slot (eight per CU at the kernel's registers) the
// shorter pose is the shorter launch for ligands of some 35 atoms and more: 2,000 poses of 63-atom ligands
// 14.8 -> 12.6 ms, of 41-atom ones 7.5 -> 6.8; beyond, throughput counts (5,120 poses 19.7 -> 20.5, 10.7
// -> 12.1 ms).  A smaller ligand's team shares less work, and two or three teams per CU already take
// longer than eight single wavefronts.  Time of one wavefront over time of four, by atoms: 6 atoms 0.95 at
// 20 poses, 0.52 at 2,000; 11 atoms 1.14 up to 600 poses, 1.11 at 800, 0.90 at 1,000, 0.58 at 2,000; 14
// 1.33 at 1,000, 1.02 at 1,200, 0.82 at 2,000; 21 1.19 at 1,400, 1.02 at 1,700, 0.94 at 2,000; 24 1.20 at
// 1,100, 0.88 at 1,500; 28 1.26 at 1,400, 1.12 at 2,000.  The line runs between, from 3 poses per CU at
// 10 atoms to 8 at 30.
inline int refine_waves(int n_cu, long long poses, long long pose_atoms) {
  if (poses <= 0) return 1;
  const double atoms = (double)pose_atoms / poses;
  if (atoms < 10) return 1;
  return poses <= std::min(8.0, 3.0 + 0.25 * (atoms - 10)) * n_cu ? 4 : 1;
}

}  // namespace vd
