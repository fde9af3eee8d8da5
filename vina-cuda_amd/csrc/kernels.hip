// kernels.hip -- HIP kernels of libvdock for gfx950 and their launch wrappers.
//
//  vd_grid_kernel     17-map precompute (replaces kernel1/kernel_grid, V11/inc/cuda/kernel1.cu:93-249;
//                     CPU semantics cache::populate, V11/lib/cache.cpp:148-208)
//  vd_eval_kernel     energy + adjoint gradient of given conformations (m_eval_deriv_update,
//                     V11/inc/cuda/quasi_newton.cuh:1294-1339; model::eval_deriv, model.cpp:1324-1334)
//  vd_mc_kernel       Monte Carlo + local search chains (kernel2_update, V11/inc/cuda/kernel2.cu:219-564),
//                     either one work item per workgroup (plain per-ligand launch) or a persistent
//                     grid pulling (ligand, chain block) items from a device queue.
//  vd_nc_lists_kernel the receptor atoms near every cell of the refinement
//  vd_refine_kernel   refinement of the kept poses against the receptor atoms and the parts of
//                     their final score (refine_structure + eval_adjusted, V11/main/main.cpp:139-157,
//                     425-440; the reference runs these on the CPU).
#include <hip/hip_runtime.h>
#include "dock_device.hpp"
#include "refine_device.hpp"
#include "kernels.h"

using namespace vdk;

namespace {

// ------------------------------------------------------------------------------------------
// Grid maps.  A workgroup is one wavefront and owns a compact tile of points (x fastest), two
// lanes per point: lane l works on point l / 2 and half l % 2 of the map types.  The receptor atoms
// that can reach the tile
// come from a host-built cell list (cells of VD_GCELL A over the box grown by the 8 A cutoff, one
// contiguous atom range per x-row of cells).  Each range is read 64 atoms at a time, one per lane
// in a single coalesced load; a ballot of the lanes whose atom lies within the cutoff of the tile
// box lists the atoms worth a pass, and the loop takes them in index order (GU per pass, their
// table reads before any is added), reading each atom from its lane with readlane.  For
// every atom within the cutoff of a point, one row of the map LUT gives the contribution to all 17
// maps: 4 values per half for a receptor type that neither is hydrophobic nor bonds, up to 6 for the
// others, 16 and 8 bytes per lane.  Every point adds its atoms in the order of the cell list,
// whatever the tile shape, so it does not change a map value.
// What bounds it is the L2's delivery to the L1s (a wavefront's 32 points read 32 rows far apart:
// 4e7 requests at 81^3, some 20 TB/s), with the vector units 70 % busy.  Rows of all 17 values (68
// bytes) took 232 us at 81^3 and 1.91 ms at 188^3, these 202 us and 1.64 ms; one lane per point
// 236 us and 1.79 ms, four atoms per pass 224 us and 1.79 ms, loads not masked by the cutoff 210 us
// and 1.70 ms.
// FEW: a launch of few tiles is bound by the length of a wavefront's chain of waits instead, and takes
// as long as its longest.  Two things shorten that chain: all rows of cells are looked up at once, a
// row per lane, and every lane reads, those out of reach the row of zeros at the table's start, so that
// no branch stands between the reads of a pass (around masked reads the compiler has the second atom's
// wait for the first's).  Kernel times with masked reads -> FEW: a 1 A box 21.6 -> 18.4 us, 8 A 34 ->
// 28.5, 16 A 59.6 -> 50, 24 A 134 -> 127, 35 A 296 -> 297, 40 A 422 -> 425, 70 A 1,385 -> 1,431; in a
// cavity, whose tiles reach few atoms, 30 A 63.5 -> 59.6, 35 A 106 -> 96, 40 A 149 -> 153.
constexpr int GU = 2;   // receptor atoms per pass of the grid kernel's loop

__device__ __forceinline__ float lane_f(float v, int j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}

struct GridTile { static constexpr int TX = 4, TY = 4, TZ = 2; };   // points of a wavefront

// One lane's half of a row, and its addition to the lane's sums: acc[k] += value of index pick k.
struct HalfRow { float4 a; float2 b; };
// A row of twelve floats leaves its second half at a multiple of 8 bytes only, and the read has to say
// so (global memory takes a 16-byte load at 8-byte alignment whole).  Copied in this form the two loads
// of a masked read stay in order, and a plain row's sums wait for the first only; through a vector type
// of alignment 8 they were swapped.
__device__ __forceinline__ HalfRow load_half(const float* r) {
  HalfRow v;
  __builtin_memcpy(&v.a, __builtin_assume_aligned(r, 8), 16);
  __builtin_memcpy(&v.b, __builtin_assume_aligned(r + 4, 8), 8);
  return v;
}
template <int I> __device__ __forceinline__ float value(const HalfRow& v) {
  if constexpr (I == 0) return v.a.x;
  else if constexpr (I == 1) return v.a.y;
  else if constexpr (I == 2) return v.a.z;
  else if constexpr (I == 3) return v.a.w;
  else if constexpr (I == 4) return v.b.x;
  else return v.b.y;
}
struct HalfSums { float s0, s1, s2, s3, s4, s5, s6, s7, s8; };
template <int P0, int P1, int P2, int P3, int P4, int P5, int P6, int P7, int P8>
__device__ __forceinline__ void add_picked(HalfSums& s, const HalfRow v, float v5) {
  s.s0 += value<P0>(v); s.s1 += value<P1>(v); s.s2 += value<P2>(v);
  s.s3 += value<P3>(v); s.s4 += value<P4>(v); s.s5 += v5;
  s.s6 += value<P6>(v); s.s7 += value<P7>(v); s.s8 += value<P8>(v);
}
// The classes are uniform branches of nine additions each.  The empty asm statements keep the
// additions in their branches (merged behind them, they took up to eleven register moves).
#define VD_KEEP(text)   asm volatile(text : "+v"(s.s0), "+v"(s.s1), "+v"(s.s2), "+v"(s.s3), "+v"(s.s4), "+v"(s.s5), "+v"(s.s6), "+v"(s.s7), "+v"(s.s8))
__device__ __forceinline__ void add_row(uint32_t meta, HalfSums& s, const HalfRow v) {
  const uint32_t cls = (meta >> 24) & 3u;
  if (cls == 0) {
    add_picked<VD_GRID_PICK_PLAIN>(s, v, v.a.y);
    VD_KEEP("; plain");
  } else if (cls == 1) {
    add_picked<VD_GRID_PICK_HYDROPHOBIC>(s, v, v.a.z);
    VD_KEEP("; hydrophobic");
  } else {
    add_picked<VD_GRID_PICK_BONDING>(s, v, (meta & VD_GRID_DONOR) ? v.a.w : v.a.z);
    VD_KEEP("; bonding");
  }
}
#undef VD_KEEP

template <bool FEW>
__global__ __launch_bounds__(64) void vd_grid_kernel(const float4* __restrict__ atoms, const int2* __restrict__ cells,
                                                     GridCells gc, const float* __restrict__ lut, float* __restrict__ maps,
                                                     vd_grid_desc gd, int tiles_x, int tiles_y) {
  constexpr int TX = GridTile::TX, TY = GridTile::TY, TZ = GridTile::TZ;
  const int tile = blockIdx.x, lane = threadIdx.x;
  const int pt = lane / 2, q = lane % 2;
  const int tx0 = (tile % tiles_x) * TX, ty0 = ((tile / tiles_x) % tiles_y) * TY, tz0 = (tile / (tiles_x * tiles_y)) * TZ;
  const int lx = pt % TX, ly = (pt / TX) % TY, lz = pt / (TX * TY);
  const int x = tx0 + lx, y = ty0 + ly, z = tz0 + lz;
  const bool inside = x < gd.dim[0] && y < gd.dim[1] && z < gd.dim[2];
  // probe coordinates as grid::index_to_argument (V11/lib/grid.h:49-53), relative to the cell origin
  const float px = gd.init[0] + gd.factor_inv[0] * x - gc.origin[0];
  const float py = gd.init[1] + gd.factor_inv[1] * y - gc.origin[1];
  const float pz = gd.init[2] + gd.factor_inv[2] * z - gc.origin[2];
  // tile bounds (relative), grown by the cutoff, -> cell range
  const float lo_x = gd.init[0] + gd.factor_inv[0] * tx0 - gc.origin[0], hi_x = lo_x + gd.factor_inv[0] * (TX - 1);
  const float lo_y = gd.init[1] + gd.factor_inv[1] * ty0 - gc.origin[1], hi_y = lo_y + gd.factor_inv[1] * (TY - 1);
  const float lo_z = gd.init[2] + gd.factor_inv[2] * tz0 - gc.origin[2], hi_z = lo_z + gd.factor_inv[2] * (TZ - 1);
  const float cut = 8.0f, inv = 1.0f / gc.cell;
  const int cx0 = max(0, (int)floorf((lo_x - cut) * inv)), cx1 = min(gc.n[0] - 1, (int)floorf((hi_x + cut) * inv));
  const int cy0 = max(0, (int)floorf((lo_y - cut) * inv)), cy1 = min(gc.n[1] - 1, (int)floorf((hi_y + cut) * inv));
  const int cz0 = max(0, (int)floorf((lo_z - cut) * inv)), cz1 = min(gc.n[2] - 1, (int)floorf((hi_z + cut) * inv));
  HalfSums acc = {};
  const int ny = cy1 - cy0 + 1, rows = ny * max(0, cz1 - cz0 + 1);
  for (int outer = FEW ? 0 : cz0; FEW ? 64 * outer < rows : outer <= cz1; ++outer) {
    // few tiles: every lane looks up a row, and those that hold atoms are taken in turn
    uint64_t left = 0;
    int row_begin = 0, row_end = 0;
    if constexpr (FEW) {
      const int r = 64 * outer + lane;
      if (r < rows) {
        const int first = ((cz0 + r / ny) * gc.n[1] + cy0 + r % ny) * gc.n[0];
        row_begin = cells[first + cx0].x; row_end = cells[first + cx1].y;
      }
      left = __ballot(row_end > row_begin);
    }
    for (int cy = cy0; FEW ? left != 0 : cy <= cy1; ++cy) {
      int begin, end;   // cells of one x-row are contiguous
      if constexpr (FEW) {
        const int i = __builtin_ctzll(left);
        left &= left - 1;
        begin = __builtin_amdgcn_readlane(row_begin, i); end = __builtin_amdgcn_readlane(row_end, i);
      } else {
        const int first = (outer * gc.n[1] + cy) * gc.n[0];
        begin = cells[first + cx0].x; end = cells[first + cx1].y;
      }
      for (int base = begin; base < end; base += 64) {
        // this lane's atom of the chunk, and whether it can reach the tile at all
        const int k = base + lane;
        const float4 mine = k < end ? atoms[k] : make_float4(0, 0, 0, 0);
        const float ddx = fmaxf(fmaxf(lo_x - mine.x, mine.x - hi_x), 0.0f);
        const float ddy = fmaxf(fmaxf(lo_y - mine.y, mine.y - hi_y), 0.0f);
        const float ddz = fmaxf(fmaxf(lo_z - mine.z, mine.z - hi_z), 0.0f);
        uint64_t todo = __ballot(k < end && ddx * ddx + ddy * ddy + ddz * ddz <= VD_CUTOFF_SQR);
        while (todo) {
          // the next GU atoms of the list, in index order (fewer when fewer are left)
          int j[GU];
          bool has[GU];
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            has[u] = todo != 0;
            j[u] = has[u] ? __builtin_ctzll(todo) : 0;
            todo &= todo - 1;
          }
          HalfRow v[GU];
          uint32_t meta[GU];
          bool use[GU];
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            const float ax = lane_f(mine.x, j[u]), ay = lane_f(mine.y, j[u]), az = lane_f(mine.z, j[u]);
            meta[u] = (uint32_t)__builtin_amdgcn_readlane(__float_as_int(mine.w), j[u]);
            const float dx = ax - px, dy = ay - py, dz = az - pz;
            const float r2 = dx * dx + dy * dy + dz * dz;
            use[u] = has[u] && inside && r2 <= VD_CUTOFF_SQR;
            const uint32_t type_rows = 4 * (meta[u] & 0xFFFFFFu);
            if (FEW || use[u]) {
              // a plain row's lane reads past its own 16 bytes; the table ends with room for that
              const uint32_t bin = (uint32_t)(VD_LUT_FACTOR * r2);
              const uint32_t half = ((meta[u] >> 24) & 3u) == 0 ? 4u : 6u;   // uniform
              const uint32_t o = __umul24(bin, 2 * half) + half * q;
              v[u] = load_half(FEW ? lut + (use[u] ? type_rows + o : 0u) : lut + type_rows + o);
            }
          }
#pragma unroll
          for (int u = 0; u < GU; ++u) {
            if (!FEW && !use[u]) continue;
            add_row(meta[u], acc, v[u]);
          }
        }
      }
    }
  }
  if (inside) {
    const size_t o = (size_t)x + (size_t)gd.dim[0] * ((size_t)y + (size_t)gd.dim[1] * z);
    constexpr int types[2][VD_GRID_PER_HALF] = {VD_GRID_TYPES};
    const float sum[VD_GRID_PER_HALF] = {acc.s0, acc.s1, acc.s2, acc.s3, acc.s4, acc.s5, acc.s6, acc.s7, acc.s8};
#pragma unroll
    for (int k = 0; k < VD_GRID_PER_HALF; ++k) {
      const int t = q ? types[1][k] : types[0][k];
      if (t >= 0) maps[(size_t)t * gd.plane + o] = sum[k];
    }
  }
}

// Edge records of the maps (the layout the searches read, described at EvalK).  blockIdx.z = type,
// blockIdx.y = a run of kEdgeRun planes of cells, thread = a record of the plane: point (i, j) of
// the plane's first dim0 (dim1 - 1) points, whose offset is the same in the map's plane, so there
// is nothing to divide and every load and store of a wavefront is one run of addresses.  A thread
// walks its planes and keeps the last one's two values.  Bound by the 16-byte stores: 188^3 maps
// 1.08 -> 0.45 ms (1.8 GB written instead of 3.6), 81^3 52 -> 31 us.
constexpr int kEdgeRun = 8;
__global__ __launch_bounds__(256) void vd_edge_kernel(const float* __restrict__ maps, float4* __restrict__ edges,
                                                      vd_grid_desc gd) {
  const int d0 = gd.dim[0], d01 = gd.dim[0] * gd.dim[1], row = d0 * (gd.dim[1] - 1), planes = gd.dim[2] - 1;
  const int p = blockIdx.x * 256 + threadIdx.x;
  if (p >= row) return;
  const int k0 = blockIdx.y * kEdgeRun, k1 = min(k0 + kEdgeRun, planes);
  const float* b = maps + (long long)blockIdx.z * gd.plane + (long long)k0 * d01 + p;
  float4* o = edges + ((long long)blockIdx.z * planes + k0) * row + p;
  float lo0 = b[0], lo1 = b[d0];
#pragma unroll 4
  for (int k = k0; k < k1; ++k) {
    b += d01;
    const float hi0 = b[0], hi1 = b[d0];
    *o = make_float4(lo0, lo1, hi0, hi1);
    o += row;
    lo0 = hi0; lo1 = hi1;
  }
}

// ------------------------------------------------------------------------------------------
// LDS layout of one wave: ligand (atoms 4A, node_o 4N, node_a 4N floats), the conformation
// stash, then per chain group the node area 12N, xyz 4A, frc 4A, the pair-force exchange row
// 4(G+1), and for dense BFGS 2G and H.  The node area holds the frame rows from the kinematics
// until the atoms are placed, then the per-node force and moment sums of the adjoint (8N): an
// evaluation reads the frames only in its intermolecular pass, which ends (with a fence) before
// the sums are cleared.  The pair words stay in global memory (read once per evaluation,
// coalesced, L2-resident).
__host__ __device__ inline int lig_floats(int A, int N) { return 4 * A + 8 * N + kStashSlots * kStashSlotFloats; }
// H is n x n for the n = 6 + torsions = 5 + nodes of the launch's largest ligand, to a multiple of four: with
// G x G floats (16 KB of 64 lanes) seven 64-lane waves fitted a CU's LDS, which now takes all its
// registers allow (4,096 chains of a 60-atom ligand with 16 torsions 154 -> 130 ms; nine batches of 96
// ligands 1,470 -> 1,385 ms).
__host__ __device__ inline int dense_floats(int N, int G) { return 2 * G + ((N + 5) * (N + 5) < G * G ? ((N + 5) * (N + 5) + 3) / 4 * 4 : G * G); }
__host__ __device__ inline int group_floats(int A, int N, int G, int dense) {
  return 12 * N + 8 * A + 4 * (G + 1) + (dense ? dense_floats(N, G) : 0);
}
// a wide launch's one group: the exchange row has a slot per lane
__host__ __device__ inline int wide_floats(int A, int N, int dense) {
  return group_floats(A, N, 16, dense) + 4 * (64 - 16);
}

template <int G>
__device__ __forceinline__ void stage_ligand(const float4* __restrict__ blob, const vd_lig_header& h, float* lds, int lane) {
  float4* dst = reinterpret_cast<float4*>(lds);
  for (int i = lane; i < h.n_atoms; i += 64) dst[i] = blob[h.off_atoms + i];
  for (int i = lane; i < 2 * h.n_nodes; i += 64) dst[h.n_atoms + i] = blob[h.off_nodes + i];
}

template <int G>
__device__ __forceinline__ void make_views(const float4* __restrict__ blob, const vd_lig_header& h, float* lds, int Amax,
                                           int Nmax, int dense, int group, LigView& L, Scratch& S, float*& H) {
  float4* base = reinterpret_cast<float4*>(lds);
  L.atom = base; L.node_o = base + h.n_atoms; L.node_a = base + h.n_atoms + h.n_nodes;
  L.pairs = reinterpret_cast<const uint4*>(reinterpret_cast<const uint32_t*>(blob) + h.off_pairs);
  L.A = h.n_atoms; L.N = h.n_nodes; L.C = h.n_chunks; L.T = h.n_torsions; L.H = h.n_heavy; L.rounds = h.jump_rounds;
  L.rows = h.pair_rows;
  S.stash = lds + lig_floats(Amax, Nmax) - kStashSlots * kStashSlotFloats;
  float* g = lds + lig_floats(Amax, Nmax) + group * group_floats(Amax, Nmax, G, dense);
  S.frame = reinterpret_cast<float4*>(g);
  S.nacc = S.frame;
  S.xyz = reinterpret_cast<float4*>(g + 12 * Nmax);
  S.frc = S.xyz + Amax;
  S.fx = S.frc + Amax;
  H = reinterpret_cast<float*>(S.fx + G + 1);
  L.ent = nullptr;
}

// Writes a chain's best energy, conformation and heavy-atom coordinates (call after
// set_coords of the best conformation).
template <int G>
__device__ void write_chain(const LigView& L, const Scratch& S, const Conf& best, float best_e, uint32_t chain, int l,
                            float* out_e, float* out_conf, float* out_heavy) {
  if (l == 0) {
    out_e[chain] = best_e;
    float* c = out_conf + (size_t)chain * (7 + L.T);
    c[0] = best.px; c[1] = best.py; c[2] = best.pz; c[3] = best.q.w; c[4] = best.q.x; c[5] = best.q.y; c[6] = best.q.z;
  }
  if (l >= 1 && l <= L.T) out_conf[(size_t)chain * (7 + L.T) + 6 + l] = best.tor;
  for (int i = l; i < L.A; i += G) {
    const uint32_t meta = fbits(L.atom[i].w);
    if ((meta >> 16) & 1u) {
      const int slot = (meta >> 17) & 255;
      float* o = out_heavy + ((size_t)chain * L.H + slot) * 3;
      const float4 y = S.xyz[i];
      o[0] = best.px + y.x; o[1] = best.py + y.y; o[2] = best.pz + y.z;
    }
  }
}

// Initial conformation of a chain: the caller's (the role of kernel_monte's ric,
// V11/inc/cuda/kernel2.cuh:27; the reference host draws them at main_procedure_cu.cpp:584-635), or
// conf::randomize (V11/lib/conf.h:127-130, 214-217; random_orientation, V11/lib/quaternion.cpp:206-219)
// from the shared random stream.  `given` points at the chain's 7+T numbers or is null.
template <int G>
__device__ Conf initial_conf(const vd_mc_consts& P, uint32_t stream, uint32_t chain, int l, int T,
                             const float* given = nullptr) {
  Conf c;
  if (given) {
    c.px = given[0]; c.py = given[1]; c.pz = given[2];
    c.q = qnormalize(Quat{given[3], given[4], given[5], given[6]});
    c.tor = (l >= 1 && l <= T) ? given[6 + l] : 0.0f;
    return c;
  }
  const U4 w = philox(chain, VD_INIT_STEP, 0, 0, P.seed, stream);
  c.px = P.box_lo[0] + (P.box_hi[0] - P.box_lo[0]) * u01(w.x);
  c.py = P.box_lo[1] + (P.box_hi[1] - P.box_lo[1]) * u01(w.y);
  c.pz = P.box_lo[2] + (P.box_hi[2] - P.box_lo[2]) * u01(w.z);
  c.q = Quat{1, 0, 0, 0};
  bool done = false;
  for (uint32_t a = 0; a < 8 && !done; ++a) {
    const U4 v = philox(chain, VD_INIT_STEP, 1, a, P.seed, stream);
    const float r0 = sqrtf(-2.0f * logf(u01(v.x) + 1.0f / 16777216.0f)), r1 = sqrtf(-2.0f * logf(u01(v.z) + 1.0f / 16777216.0f));
    float s0, c0, s1, c1;
    sincosf(2.0f * kPi * u01(v.y), &s0, &c0); sincosf(2.0f * kPi * u01(v.w), &s1, &c1);
    const float n0 = r0 * c0, n1 = r0 * s0, n2 = r1 * c1, n3 = r1 * s1;
    const float nrm = sqrtf(n0 * n0 + n1 * n1 + n2 * n2 + n3 * n3);
    if (nrm > 1e-6f) { c.q = Quat{n0 / nrm, n1 / nrm, n2 / nrm, n3 / nrm}; done = true; }
  }
  c.tor = 0.0f;
  if (l >= 1 && l <= T) {
    const int j = l - 1;
    const U4 v = philox(chain, VD_INIT_STEP, 2 + (uint32_t)(j / 4), 0, P.seed, stream);
    const uint32_t word = (j % 4 == 0) ? v.x : (j % 4 == 1) ? v.y : (j % 4 == 2) ? v.z : v.w;
    c.tor = -kPi + 2.0f * kPi * u01(word);
  }
  return c;
}

// One MC chain per group with the reference GPU schedule (V11/inc/cuda/kernel2.cu:219-426):
// mutate -> local search -> Metropolis(T) -> on accept, if better than the best so far: second
// local search, keep the best.  Mutation as V11/lib/mutate.cpp:62-127 (see initial_conf for the
// random stream); the orientation step uses the gyration radius of the current conformation.
// ls_only: one local search from the starting conformation, no MC steps (vd_local_search).
// The local search is RILC-BFGS with the Lewis-Overton line search (quasi_newton.cuh:1710-1806,
// 2172-2389) or, with POL = -1, dense BFGS with its backtracking line search (--rilc_bfgs 0,
// kernel2.cu:427-563 with bfgs_optimized, quasi_newton.cuh:2391-2499; H is the group's matrix,
// see dense_minus_hv).  It runs as a flat state machine: every pass evaluates one conformation
// per chain group and each group then advances its own state (start of a local search,
// line-search trial, end of a BFGS iteration, end of a local search, Metropolis step, next
// mutation) as far as it can without another evaluation.  Chains of a wavefront thus never wait
// for each other's line searches or local searches; they only wait at the end of the chain.  The
// gyration radius of each evaluated conformation comes from the evaluation itself and travels
// with the conformation.
// POL: -1 dense BFGS; 0 Vina; 1 QuickVina2 gate at the start of every local search (see
// History); 2 QuickVina-W gate (qvw_interesting) with its records: the searched start point, each
// BFGS iteration's end point and the point where the search stops go to the chain's own buffer,
// the search's last point to the ligand's global buffer (QVW/inc/cuda/quasi_newton.cuh:2236-2410).
// WIDE: the four rows of the wavefront carry one chain (G = 16; see pair_terms_wide).
template <int G, int POL, bool WIDE = false>
__device__ void mc_chain_flat(const LigView& L, const Scratch& S, const EvalK& K, const vd_mc_consts& P, int depth,
                              int max_steps, uint32_t stream, uint32_t chain, bool valid, int l, float* out_e,
                              float* out_conf, float* out_heavy, int& evals, History* hist, const GlobalHist* gh,
                              const float* given, bool ls_only, float* H) {
  const uint32_t k0 = P.seed, k1 = stream;
  const int n_ent = P.mutation_quirk ? (1 + L.T) : (2 + L.T);
  float* const vbuf = H;   // dense BFGS: 2 G floats, then the matrix
  H += 2 * G;
  enum { kMutate = 0, kStart = 1, kTrial = 2, kDone = 3 };
  // MC state; the current conformation lives in the stash (kSlotTmp)
  {
    const Conf c0 = initial_conf<G>(P, stream, chain, l, L.T, given);
    stash_put<G>(S.stash, kSlotTmp, c0);
    stash_put<G>(S.stash, kSlotBest, c0);
    set_coords<G>(L, S, c0, l);
  }
  float rg = gyration_radius<G>(L, S, l);
  float tmp_e = 0.0f, best_e = INFINITY, u_metro = 0.0f;
  // ls_kind: 1 the search of a mutated candidate, 2 the second search of an accepted one,
  // 0 a lone search from the starting conformation (ls_only)
  int step = 0, phase = (valid && depth > 0) ? kMutate : kDone, ls_kind = 1;
  if (ls_only) {
    phase = valid ? kStart : kDone;
    ls_kind = 0;
  }
  // local-search state
  Conf x = stash_get<G>(S.stash, kSlotTmp);
  float x_rg = rg, g = 0.0f, d = 0.0f, gp = 0.0f;
  float fx = 0.0f, fxp = 0.0f, fx_orig = 0.0f, orig_rg = 0.0f, prev_rg = 0.0f;
  float stp = 0.0f, finit = 0.0f, dgtest = 0.0f, dstest = 0.0f, mu = 0.0f, nu = 0.0f;
  bool brackt = false;
  int count = 0, k = 0;
  float dn_pg = 0.0f;   // dense BFGS: p.g of the iteration's direction
  int dn_step = 0;      // dense BFGS: iterations done in this search
  while (__any(phase != kDone)) {
    // (1) MC step start: draws and mutation (mutate.cpp:62-127); the candidate is evaluated next
    const bool mut = phase == kMutate;
    if (__any(mut)) {
      const U4 w = philox(chain, (uint32_t)step, 0, 0, k0, k1);
      const int which = min((int)(u01(w.x) * (float)n_ent), n_ent - 1);
      const float tor = -kPi + 2.0f * kPi * u01(w.z);
      float sx = 0.0f, sy = 0.0f, sz = 0.0f;
      bool need = mut && which <= 1;
      for (uint32_t a = 0; a < 64 && __any(need); ++a) {   // P(64 rejections) ~ 1e-20
        const U4 v = philox(chain, (uint32_t)step, 1, a, k0, k1);
        const float vx = 2.0f * u01(v.x) - 1.0f, vy = 2.0f * u01(v.y) - 1.0f, vz = 2.0f * u01(v.z) - 1.0f;
        if (need && vx * vx + vy * vy + vz * vz < 1.0f) { sx = vx; sy = vy; sz = vz; need = false; }
      }
      if (mut) {
        Conf cand = stash_get<G>(S.stash, kSlotTmp);
        if (which == 0) { cand.px += P.amplitude * sx; cand.py += P.amplitude * sy; cand.pz += P.amplitude * sz; }
        else if (which == 1) { if (rg > kEpsFl) { const float f = P.amplitude / rg; cand.q = qincrement(cand.q, f * sx, f * sy, f * sz); } }
        else if (l == which - 1) cand.tor = tor;
        x = cand; u_metro = u01(w.y); ls_kind = 1; phase = kStart;
      }
    }
    // (2) one evaluation per group: the search start point, or the line-search trial point
    const bool trial = phase == kTrial, start = phase == kStart;
    const Conf xt = increment<G>(stash_get<G>(S.stash, kSlotPrev), d, stp, l, L.T);
    const Conf xe = csel(trial, xt, x);
    // A trial that fails the line search's decrease test is only a value: its gradient is looked at
    // after the test passes, or when the tenth trial ends the search.  The adjoint (node scan, subtree
    // sums) of a pass is left out when no chain of the wavefront wants it: dense BFGS, 64-lane class
    // 98 -> 83 ms, RILC-BFGS 59 -> 56.5 ms alone; four chains seldom all fail together (under 2 %).
    float ge, rge;
    bool decrease = false;
    const float fe = eval_deriv<G, WIDE>(L, S, K, xe, l, ge, &rge, [&](float e) {
      decrease = POL < 0 ? e - fxp < 1e-4f * stp * dn_pg : !(e > finit + stp * dgtest);
      return start || (trial && (decrease || count + 1 >= 10));
    });
    // (3) consume it
    bool ls_done = false, iter_end = false, begin = false;
    int result = -1;
    if (start || trial) { ++evals; x = xe; fx = fe; g = ge; x_rg = rge; }
    if (trial) ++count;
    if (start) { fx_orig = fe; orig_rg = rge; stash_put<G>(S.stash, kSlotOrig, x); }
    bool search = start;
    if constexpr (POL == 1) {
      if (__any(start)) {
        const bool interesting = hist_interesting<G>(*hist, x, fx, g, l, L.T, start);
        hist_add<G>(*hist, x, fx, g, l, L.T, start && interesting);
        search = start && interesting;
      }
    }
    if constexpr (POL == 2) {
      if (__any(start)) {
        const bool interesting = qvw_interesting<G>(*hist, *gh, x, fx, g, l, L.T, start);
        hist_add<G>(*hist, x, fx, g, l, L.T, start && interesting);
        search = start && interesting;
      }
    }
    bool rec_own = false, rec_glob = false;   // QuickVina-W records of this pass
    if constexpr (POL < 0) {   // dense BFGS (quasi_newton.cuh:2391-2499); x, fx, g hold the point evaluated
      // a search starts from the identity matrix; no step limit -> the start point is the result
      dense_identity<G>(H, l, L.T, start);
      if (start) { dn_step = 0; if (max_steps > 0) begin = true; else ls_done = true; }
      // backtracking: accept when f1 - f0 < 1e-4 alpha p.g, else halve alpha; after ten trials the
      // last point is taken (alpha halved once more)
      if (trial) {
        if (!decrease) stp *= 0.5f;
        if (decrease || count >= 10) iter_end = true;
      }
      if (__any(iter_end)) {   // end of an iteration: the step is taken; the update
        const float y = g - gp;
        const float gnorm = sqrtf(gsum<G>(gp * gp));
        bool upd = false;
        if (iter_end) { if (!(gnorm >= 1e-5f)) ls_done = true; else upd = true; }
        const float yy = gsum<G>(y * y), yp = gsum<G>(y * d);
        dense_set_diag<G>(H, stp * yp / yy, l, L.T, iter_end && dn_step == 0 && upd && fabsf(yy) > kEpsFl);   // first step: scaled diagonal
        const float mhy = dense_minus_hv<G>(H, vbuf, y, l, L.T);
        const float yhy = -gsum<G>(y * mhy);
        const float r = 1.0f / (stp * yp);
        dense_update<G>(H, vbuf, mhy, d, stp, r, yhy, iter_end && upd && !(stp * yp < kEpsFl), l, L.T);
        if (iter_end && !ls_done) { ++dn_step; if (dn_step < max_steps) begin = true; else ls_done = true; }
      }
      if (__any(begin)) {      // an iteration starts at x: p = -H g
        if (begin) { stash_put<G>(S.stash, kSlotPrev, x); gp = g; fxp = fx; prev_rg = x_rg; }
        const float pn = dense_minus_hv<G>(H, vbuf, g, l, L.T);
        const float pg = gsum<G>(pn * g);
        if (begin) { d = pn; dn_pg = pg; stp = 1.0f; count = 0; phase = kTrial; }
      }
    }
    if constexpr (POL >= 0) {
    if (__any(start)) {
      const float gg = gsum<G>(g * g);
      if (start) {
        d = -g;
        if (search && sqrtf(gg) >= 1e-5f) { stp = 1.0f / sqrtf(gg); k = 1; begin = true; }
        else ls_done = true;
      }
    }
    if (__any(trial)) {   // Lewis-Overton line search (quasi_newton.cuh:2172-2389)
      const float gtd = gsum<G>(g * d);
      if (trial) {
        bool done = false;
        if (!decrease) { nu = stp; brackt = true; }
        else if (gtd < dstest) { mu = stp; }
        else { result = count; done = true; }
        if (!done && count >= 10) { result = (fx > finit) ? -1 : count; done = true; }
        if (!done) stp = brackt ? 0.5f * (mu + nu) : 2.0f * stp;
        iter_end = done;
      }
    }
    if (__any(iter_end)) {   // end of a BFGS iteration, direction update (quasi_newton.cuh:2342-2350)
      const float gnorm = sqrtf(gsum<G>(g * g));
      bool update = false;
      if (iter_end) {
        if (result < 0) {
          x = stash_get<G>(S.stash, kSlotPrev); g = gp; fx = fxp; x_rg = prev_rg; ls_done = true;
          rec_own = rec_glob = true;
        }
        else if (!(gnorm >= 1e-5f)) ls_done = true;
        else if ((max_steps != 0 && max_steps <= k) || k >= 1000) { ls_done = true; rec_own = rec_glob = true; }   // 1000: hard bound
        else { ++k; update = true; rec_own = true; }
      }
      const float sv = stp * d, y = g - gp;
      const float ys = gsum<G>(y * sv), yy = gsum<G>(y * y), ss = gsum<G>(sv * sv), gpgp = gsum<G>(gp * gp);
      const float nd = -g;
      const float alpha = gsum<G>(sv * nd) / ys;
      const float nd2 = (nd + alpha * y) * (ys / yy);
      const float beta = gsum<G>(y * nd2) / ys;
      const float nd3 = nd2 + (alpha - beta) * sv;
      if (update) { d = (ys > ss * sqrtf(gpgp) * 1.0e-6f) ? nd3 : nd; stp = 1.0f; begin = true; }
    }
    if (__any(begin)) {      // a BFGS iteration starts: its line search begins at x along d
      if (begin) { stash_put<G>(S.stash, kSlotPrev, x); gp = g; fxp = fx; prev_rg = x_rg; }
      const float dginit = gsum<G>(g * d);
      if (begin) {
        if (0.0f < dginit) { ls_done = true; rec_own = rec_glob = true; }   // no descent: the iteration fails, x stays
        else {
          finit = fx; dgtest = 1e-4f * dginit; dstest = 0.1f * dginit;
          mu = 0.0f; nu = 1.0e20f; brackt = false; count = 0; phase = kTrial;
        }
      }
    }
    }   // RILC-BFGS
    if constexpr (POL == 2) {
      if (__any(rec_own)) hist_add<G>(*hist, x, fx, g, l, L.T, rec_own);
      if (__any(rec_glob)) glob_add<G>(*gh, x, fx, g, l, L.T, rec_glob);
    }
    if (ls_done) {           // end of a local search: keep the better of its start and its result
      if (!(fx <= fx_orig)) { fx = fx_orig; x = stash_get<G>(S.stash, kSlotOrig); x_rg = orig_rg; }
      bool step_done = true;
      if (ls_kind == 0) {    // a lone local search: its result is the chain's output
        stash_put<G>(S.stash, kSlotBest, x); best_e = fx; phase = kDone; step_done = false;
      } else if (ls_kind == 1) {    // Metropolis (kernel2.cu:364-392)
        const bool accept = step == 0 || fx < tmp_e || u_metro < expf((tmp_e - fx) / P.temperature);
        if (accept) { stash_put<G>(S.stash, kSlotTmp, x); tmp_e = fx; rg = x_rg; }
        if (accept && tmp_e < best_e) { ls_kind = 2; phase = kStart; step_done = false; }   // second search of x
      } else {
        stash_put<G>(S.stash, kSlotTmp, x); tmp_e = fx; rg = x_rg;
        if (tmp_e < best_e) { stash_put<G>(S.stash, kSlotBest, x); best_e = tmp_e; }
      }
      if (step_done) { ++step; phase = step < depth ? kMutate : kDone; }
    }
  }
  const Conf best = stash_get<G>(S.stash, kSlotBest);
  set_coords<G>(L, S, best, l);
  if (valid && (!WIDE || threadIdx.x < G)) write_chain<G>(L, S, best, best_e, chain, l, out_e, out_conf, out_heavy);
}

// W = minimum waves per SIMD the register allocation must allow (2 = unconstrained); a tuning knob:
// more resident waves hide more latency, at the price of register spills.
template <int G, int MODE, int W>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(W, 8))) void vd_mc_kernel(McArgs a) {
  extern __shared__ float4 lds4[];
  float* lds = reinterpret_cast<float*>(lds4);
  constexpr int CPW = 64 / G;
  const int lane = threadIdx.x, group = lane / G, l = lane % G;
  int cur = -1;
  for (int it = 0;; ++it) {
    int item;
    if (a.queue) {
      int v = 0;
      if (lane == 0) v = atomicAdd(a.queue, 1);
      item = __shfl(v, 0);
    } else {
      item = (it == 0) ? (int)blockIdx.x : a.n_items;
    }
    if (item >= a.n_items) break;
    // (ligand slot, first chain of the block); without an item list, one ligand's chain blocks in order
    const int2 wi = a.items ? a.items[item] : make_int2(0, item * CPW);
    const vd_lig_header h = a.headers[wi.x];
    if (wi.x != cur) {
      __syncthreads();
      stage_ligand<G>(a.blob, h, lds, lane);
      __syncthreads();
      cur = wi.x;
    }
    LigView L; Scratch S; float* H;
    make_views<G>(a.blob, h, lds, a.Amax, a.Nmax, MODE == 0, group, L, S, H);
    const uint32_t chain = (uint32_t)(wi.y + group);
    const bool valid = (int)chain < a.P.chains;
    const float* given = (a.init_conf && valid) ? a.init_conf + a.out_off[wi.x].y + (size_t)chain * (7 + h.n_torsions)
                                                : nullptr;
    int evals = 0;
    History hist;
    if constexpr (MODE == 2) hist.init(a.hist + ((long long)blockIdx.x * CPW + group) * a.hist_stride, h.n_torsions);
    if constexpr (MODE == 3) hist.init(a.hist + ((long long)blockIdx.x * CPW + group) * a.hist_stride, h.n_torsions, 5);
    GlobalHist gh{};
    if constexpr (MODE == 3) {
      gh.base = a.glob + a.out_off[wi.x].w; gh.per_axis = h.reserved; gh.T = h.n_torsions;
      for (int k = 0; k < 3; ++k) { gh.lo[k] = a.P.box_lo[k]; gh.hi[k] = a.P.box_hi[k]; }
    }
    mc_chain_flat<G, MODE - 1>(L, S, a.K, a.P, h.search_depth, h.bfgs_steps, a.streams[wi.x], chain, valid, l,
                               a.out_e + a.out_off[wi.x].x, a.out_conf + a.out_off[wi.x].y,
                               a.out_heavy + a.out_off[wi.x].z, evals, &hist, &gh, given, a.ls_only != 0, H);
    if (a.slot_evals) {
      int sum = 0;
      for (int gi = 0; gi < CPW; ++gi) sum += __shfl(evals, gi * G);
      if (lane == 0) atomicAdd(a.slot_evals + wi.x, (unsigned long long)sum);
    }
  }
}

// A wide launch's chains: items are (ligand slot, chain).  Three waves per SIMD (168 registers; 236
// bytes of spills under dense BFGS, 184 under RILC-BFGS, 336 with the QuickVina2 history) against two
// (217 and none under RILC-BFGS): large-box QuickVina2 batch of 200 ligands 149 against 163 ms, dense
// BFGS of 96 the same.
// Its template arguments are vd_mc_kernel's: lanes whose arithmetic it takes, mode, waves per SIMD.
template <int G, int MODE, int W>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(W, 8))) void vd_mc_wide_kernel(McArgs a) {
  static_assert(G == 16, "");
  extern __shared__ float4 lds4[];
  float* lds = reinterpret_cast<float*>(lds4);
  const int lane = threadIdx.x, l = lane & 15;
  int cur = -1;
  for (int it = 0;; ++it) {
    int item = 0;
    if (lane == 0) item = atomicAdd(a.queue, 1);
    item = __shfl(item, 0);
    if (item >= a.n_items) break;
    const int2 wi = a.items[item];
    const vd_lig_header h = a.headers[wi.x];
    if (wi.x != cur) {
      __syncthreads();
      stage_ligand<16>(a.blob, h, lds, lane);
      __syncthreads();
      cur = wi.x;
    }
    LigView L; Scratch S; float* H;
    make_views<16>(a.blob, h, lds, a.Amax, a.Nmax, MODE == 0, 0, L, S, H);
    H += 4 * (64 - 16);
    L.ent = reinterpret_cast<const uint2*>(reinterpret_cast<const uint32_t*>(a.blob) + h.off_ent);
    int evals = 0;
    History hist;
    if constexpr (MODE == 2) hist.init(a.hist + (long long)blockIdx.x * a.hist_stride, h.n_torsions);
    GlobalHist gh{};
    mc_chain_flat<16, MODE - 1, true>(L, S, a.K, a.P, h.search_depth, h.bfgs_steps, a.streams[wi.x], (uint32_t)wi.y, true, l,
                                      a.out_e + a.out_off[wi.x].x, a.out_conf + a.out_off[wi.x].y,
                                      a.out_heavy + a.out_off[wi.x].z, evals, &hist, &gh, nullptr, false, H);
    if (lane == 0) atomicAdd(a.slot_evals + wi.x, (unsigned long long)evals);
  }
}

// HOST: the conformations lie in host memory, two microseconds away: a conformation's 7 + T <= G
// numbers in one load, a number per lane, a conformation ahead, handed round by broadcasts.  On the
// device every lane reads what it needs, when it needs it: the broadcasts (through the LDS for groups of
// 32) cost resident conformations up to 4 % (300,000 poses, kernel: 24-atom ligand on 64 lanes 605 ->
// 599 us, 34 atoms on 32 lanes 619 -> 600, 42 atoms 791 -> 780).
template <int G, bool HOST>
__global__ __launch_bounds__(64) void vd_eval_kernel(EvalArgs a) {
  extern __shared__ float4 lds4[];
  float* lds = reinterpret_cast<float*>(lds4);
  constexpr int CPW = 64 / G;
  const int lane = threadIdx.x, group = lane / G, l = lane % G;
  if (blockIdx.x == 0 && lane == 0) a.clock[0] = (unsigned long long)wall_clock64();
  const vd_lig_header& h = a.header;
  LigView L; Scratch S; float* H;
  make_views<G>(a.blob, h, lds, h.n_atoms, h.n_nodes, 0, group, L, S, H);
  const int T = h.n_torsions, nc = 7 + T, ng = 6 + T;
  const auto numbers = [&](long long c) { return l < nc ? a.conf[(c < a.n_conf ? c : 0) * nc + l] : 0.0f; };
  const long long stride = (long long)gridDim.x * CPW;
  float next = HOST ? numbers((long long)blockIdx.x * CPW + group) : 0.0f;
  stage_ligand<G>(a.blob, h, lds, lane);
  __syncthreads();
  for (long long base = (long long)blockIdx.x * CPW; base < a.n_conf; base += stride) {
    const long long c = base + group;
    const bool valid = c < a.n_conf;
    Conf cf;
    if constexpr (HOST) {
      const float x = next;
      if (base + stride < a.n_conf) next = numbers(c + stride);
      cf.px = gbcast<G, 0>(x); cf.py = gbcast<G, 1>(x); cf.pz = gbcast<G, 2>(x);
      cf.q = Quat{gbcast<G, 3>(x), gbcast<G, 4>(x), gbcast<G, 5>(x), gbcast<G, 6>(x)};
      const float tor = gget<G>(x, min(l + 6, G - 1));
      cf.tor = (l >= 1 && l <= T) ? tor : 0.0f;
    } else {
      const float* x = a.conf + (valid ? c : 0) * nc;
      cf.px = x[0]; cf.py = x[1]; cf.pz = x[2]; cf.q = Quat{x[3], x[4], x[5], x[6]};
      cf.tor = (l >= 1 && l <= T) ? x[6 + l] : 0.0f;
    }
    float g;
    const float e = eval_deriv<G>(L, S, a.K, cf, l, g);
    if (valid) {
      if (l == 0) a.e[c] = e;
      float* go = a.grad + c * ng;
      if (l >= 1 && l <= T) go[5 + l] = g;
      if (l >= G - 6) go[l - (G - 6)] = g;
    }
  }
  // a word per workgroup: a maximum of 4,096 workgroups over one word took 45 us of a launch
  if (lane == 0) a.clock[1 + blockIdx.x] = (unsigned long long)wall_clock64();
}

// ------------------------------------------------------------------------------------------
// Receptor lists of the refinement's cells, one wavefront per cell: every lane looks up the atom range
// of one x-row of bins, then the rows that hold atoms are taken in order, 64 atoms at a time, and the
// lanes whose atom lies within the cutoff of the cell's brick write it behind the ones before.  The
// order is that of the sorted atoms, with rounded products and sums throughout (no fused ones), so a
// cell lists the atoms that a loop over its bins on the host lists, in that order.  The same loop counts
// (fill = false) and writes; both wait on short rows (two atoms of a row of ten bins, 64 lanes).  The
// lists of a 70 A box (42,875 cells, 215 MB) took the host 260 ms to build and copy, this takes 2; of a
// 30 A box (8,000 atoms) 25 and 1 ms.
template <bool FILL>
__global__ __launch_bounds__(256) void vd_nc_lists_kernel(NcLists b, int* __restrict__ start, double4* __restrict__ list) {
  const int lane = threadIdx.x & 63;
  const long long cell = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (cell >= (long long)b.n[0] * b.n[1] * b.n[2]) return;
  const int x = (int)(cell % b.n[0]), y = (int)(cell / b.n[0] % b.n[1]), z = (int)(cell / b.n[0] / b.n[1]);
  const int id[3] = {x, y, z};
  double lo[3], hi[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    lo[k] = __dadd_rn(b.lo[k], __dmul_rn(b.cell[k], (double)id[k]));
    hi[k] = __dadd_rn(b.lo[k], __dmul_rn(b.cell[k], (double)(id[k] + 1)));
  }
  const int x1 = min(b.nb[0] - 1, x + b.reach[0]);
  const int ny = min(b.nb[1] - 1, y + b.reach[1]) - y + 1, nz = min(b.nb[2] - 1, z + b.reach[2]) - z + 1;
  auto first = [&](long long bin) {   // the first atom of bin or a later one
    int i = 0, n = b.n_atoms;
    while (n > 0) {
      const int h = n / 2;
      if (b.bin[i + h] < bin) { i += h + 1; n -= h + 1; } else n = h;
    }
    return i;
  };
  const long long rows = (long long)ny * nz;
  int count = 0;
  const long long base = FILL ? start[cell] : 0;
  for (long long r0 = 0; r0 < rows; r0 += 64) {
    int s = 0, e = 0;
    if (r0 + lane < rows) {
      const int ry = y + (int)((r0 + lane) % ny), rz = z + (int)((r0 + lane) / ny);
      const long long row = ((long long)rz * b.nb[1] + ry) * b.nb[0];
      s = first(row + x); e = first(row + x1 + 1);
    }
    for (unsigned long long m = __ballot(e > s); m; m &= m - 1) {
      const int q = __ffsll(m) - 1, rs = __shfl(s, q), re = __shfl(e, q);
      for (int i0 = rs; i0 < re; i0 += 64) {
        bool in = false;
        double4 a;
        if (i0 + lane < re) {
          a = b.atoms[i0 + lane];
          const double v[3] = {a.x, a.y, a.z};
          double dd = 0;
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            const double d = v[k] < lo[k] ? lo[k] - v[k] : (v[k] > hi[k] ? v[k] - hi[k] : 0.0);
            dd = __dadd_rn(dd, __dmul_rn(d, d));
          }
          in = !(dd >= b.cut2);
        }
        const unsigned long long w = __ballot(in);
        if (FILL && in) list[base + count + __popcll(w & ((1ULL << lane) - 1))] = a;
        count += __popcll(w);
      }
    }
  }
  if (!FILL && lane == 0) start[cell] = count;
}

// ------------------------------------------------------------------------------------------
// After the search: refine_structure (V11/main/main.cpp:139-157) of one pose per workgroup of NW
// wavefronts, in FP64: dense BFGS on the receptor atoms themselves with the out-of-box slope
// raised 1e2 -> 1e10 until the heavy atoms lie within the box (a pose that never gets inside
// reports max_fl), then the parts of the final score at the refined pose (fast tables, slope
// a.final_slope).
template <int NW>
__global__ __launch_bounds__(64 * NW) void vd_refine_kernel(RefineArgs a) {
  extern __shared__ double lds_d[];
  const int pose = a.order[blockIdx.x], l = threadIdx.x & 63, w = threadIdx.x >> 6;
  const vdr::RefHeader h = a.hdr[a.pose_lig[pose]];
  vdr::Pose P;
  vdr::carve(P, lds_d, a.Amax, a.Nmax);
  vdr::Team M{};
  P.pairs = a.pairs + h.off_pairs;
  P.A = h.A; P.N = h.N; P.T = h.T; P.C = h.C; P.n = 6 + h.T;
  for (int i = threadIdx.x; i < h.A; i += 64 * NW) const_cast<double4*>(P.atom)[i] = a.geo[h.off_atoms + i];
  for (int i = threadIdx.x; i < h.N; i += 64 * NW) {
    const_cast<double4*>(P.node_o)[i] = a.geo[h.off_atoms + h.A + i];
    const_cast<double4*>(P.node_a)[i] = a.geo[h.off_atoms + h.A + h.N + i];
  }
  for (int i = threadIdx.x; i < VD_XS_SIZE * VD_XS_SIZE; i += 64 * NW) P.rows[i] = a.K.rows[i];
  if constexpr (NW > 1) {
    vdr::carve_team(M, lds_d + vdr::pose_lds_doubles(a.Amax, a.Nmax, a.nmax));
    M.ent = a.ent + h.off_ent;
    for (int i = threadIdx.x; i < 3 * vdr::kTeamChunks; i += 64 * NW) {
      double* z = M.f + i / 3 * vdr::kTeamChunkDoubles + i % 3 * 66 + 64;
      z[0] = 0.0; z[1] = -0.0;
    }
    __syncthreads();
    if (w > 0) { vdr::team_serve<NW>(P, a.K, M, w, l); return; }
  }
  vdr::wave_sync();
  vdr::load_links(P, l);
  const double* ci = a.conf_in + a.conf_off[pose];
  vdr::Conf x;
  x.pos = vdr::D3{ci[0], ci[1], ci[2]};
  x.q = vdr::DQ{ci[3], ci[4], ci[5], ci[6]};
  x.tor = (l >= 6 && l < 6 + h.T) ? ci[7 + (l - 6)] : 0.0;
  vdr::wave_sync();
  double e = 0, slope = 100;
  bool inside = false;
  int evals = 0;
  for (int p = 0; p < 5; ++p, slope *= 100) {
    e = vdr::bfgs<NW>(P, a.K, M, slope, x, h.max_steps, l, evals);
    vdr::set_coords(P, a.K, x, l);
    inside = vdr::within(P, a.K, l);
    if (inside) break;
  }
  if constexpr (NW > 1) {
    if (l == 0) *M.serve = 0;
    __syncthreads();
  }
  if (!inside) e = vdr::kMaxFl;
  const double e_inter = vdr::lane_sum<64>(vdr::nc_inter<true>(P, a.K, a.final_slope, l >> 4, 4, l));
  const double e_intra = vdr::lane_sum<64>(vdr::pair_terms<true>(P, a.K, l));
  double* co = a.conf_out + a.conf_off[pose];
  if (l == 0) {
    co[0] = x.pos.x; co[1] = x.pos.y; co[2] = x.pos.z; co[3] = x.q.a; co[4] = x.q.b; co[5] = x.q.c; co[6] = x.q.d;
    a.res[pose] = make_double4(e, e_inter, e_intra, inside ? 1.0 : 0.0);
    a.evals[pose] = evals;
  }
  if (l >= 6 && l < 6 + h.T) co[7 + (l - 6)] = x.tor;
  double* xyz = a.coords_out + a.coords_off[pose];
  for (int i = l; i < h.A; i += 64) {
    const double4 y = P.xyz[i];
    xyz[3 * i] = y.x; xyz[3 * i + 1] = y.y; xyz[3 * i + 2] = y.z;
  }
}

}  // namespace

// Device memory of the no-allocation docking entry point (vd_dock_noalloc): one array per device,
// held until the process ends.  Host code never passes the array's name to a kernel or a copy: it
// takes the device address from scratch_address once per device and uses that.
static __device__ __align__(256) unsigned char scratch[VD_NOALLOC_SCRATCH_BYTES];

namespace vdl {

hipError_t scratch_address(void** p) { return hipGetSymbolAddress(p, HIP_SYMBOL(scratch)); }

hipError_t launch_nc_lists(bool fill, const NcLists& b, int* start, double4* list, hipStream_t s) {
  const long long cells = (long long)b.n[0] * b.n[1] * b.n[2];
  if (cells <= 0 || cells > 0x7fffffffLL * 4) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((cells + 3) / 4));
  if (fill) hipLaunchKernelGGL(vd_nc_lists_kernel<true>, grid, dim3(256), 0, s, b, start, list);
  else hipLaunchKernelGGL(vd_nc_lists_kernel<false>, grid, dim3(256), 0, s, b, start, list);
  return hipGetLastError();
}

int refine_lds_bytes(int waves, int Amax, int Nmax, int nmax) {
  return 8 * (vdr::pose_lds_doubles(Amax, Nmax, nmax) + (waves > 1 ? vdr::team_lds_doubles() : 0));
}

hipError_t launch_refine(int waves, const RefineArgs& a, int poses, hipStream_t s) {
  const int lds = refine_lds_bytes(waves, a.Amax, a.Nmax, a.nmax);
  switch (waves) {
    case 1: hipLaunchKernelGGL(vd_refine_kernel<1>, dim3(poses), dim3(64), lds, s, a); break;
    case 4: hipLaunchKernelGGL(vd_refine_kernel<4>, dim3(poses), dim3(256), lds, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

int mc_lds_bytes(int G, int Amax, int Nmax, int dense) {
  return 4 * (lig_floats(Amax, Nmax) + (64 / G) * group_floats(Amax, Nmax, G, dense));
}

hipError_t launch_grid(const float4* atoms, const int2* cells, const GridCells& gc, const float* lut, float* maps,
                       const vd_grid_desc& gd, int n_cu, hipStream_t s) {
  using T = GridTile;
  const int tx = (gd.dim[0] + T::TX - 1) / T::TX, ty = (gd.dim[1] + T::TY - 1) / T::TY, tz = (gd.dim[2] + T::TZ - 1) / T::TZ;
  if (tx * ty * tz <= 112 * n_cu)   // 35 A boxes and smaller; both sides are given above vd_grid_kernel
    hipLaunchKernelGGL(vd_grid_kernel<true>, dim3(tx * ty * tz), dim3(64), 0, s, atoms, cells, gc, lut, maps, gd, tx, ty);
  else
    hipLaunchKernelGGL(vd_grid_kernel<false>, dim3(tx * ty * tz), dim3(64), 0, s, atoms, cells, gc, lut, maps, gd, tx, ty);
  return hipGetLastError();
}

hipError_t launch_edges(const float* maps, float4* edges, const vd_grid_desc& gd, hipStream_t s) {
  const int row = gd.dim[0] * (gd.dim[1] - 1), planes = gd.dim[2] - 1;
  if (row <= 0 || planes <= 0) return hipSuccess;
  hipLaunchKernelGGL(vd_edge_kernel, dim3((row + 255) / 256, (planes + kEdgeRun - 1) / kEdgeRun, VD_XS_SIZE), dim3(256), 0, s,
                     maps, edges, gd);
  return hipGetLastError();
}

template <bool HOST>
static void launch_eval_form(int G, const EvalArgs& a, int blocks, int lds, hipStream_t s) {
  switch (G) {
    case 64: hipLaunchKernelGGL((vd_eval_kernel<64, HOST>), dim3(blocks), dim3(64), lds, s, a); break;
    case 32: hipLaunchKernelGGL((vd_eval_kernel<32, HOST>), dim3(blocks), dim3(64), lds, s, a); break;
    default: hipLaunchKernelGGL((vd_eval_kernel<16, HOST>), dim3(blocks), dim3(64), lds, s, a);
  }
}
hipError_t launch_eval(int G, bool host, const EvalArgs& a, int blocks, hipStream_t s) {
  if (G != 64 && G != 32 && G != 16) return hipErrorInvalidValue;
  const int lds = mc_lds_bytes(G, a.header.n_atoms, a.header.n_nodes, 0);
  if (host) launch_eval_form<true>(G, a, blocks, lds, s);
  else launch_eval_form<false>(G, a, blocks, lds, s);
  return hipGetLastError();
}

int wide_lds_bytes(int Amax, int Nmax, int dense) { return 4 * (lig_floats(Amax, Nmax) + wide_floats(Amax, Nmax, dense)); }

hipError_t launch_mc_wide(const McArgs& a, int blocks, hipStream_t s) {
  const int lds = wide_lds_bytes(a.Amax, a.Nmax, a.P.local_search == 0);
  if (!a.queue || !a.items || (a.P.policy == 1 && !a.hist) || a.P.policy == 2) return hipErrorInvalidValue;
  if (a.P.local_search == 0) hipLaunchKernelGGL((vd_mc_wide_kernel<16, 0, kWideWaves>), dim3(blocks), dim3(64), lds, s, a);
  else if (a.P.policy == 1) hipLaunchKernelGGL((vd_mc_wide_kernel<16, 2, kWideWaves>), dim3(blocks), dim3(64), lds, s, a);
  else hipLaunchKernelGGL((vd_mc_wide_kernel<16, 1, kWideWaves>), dim3(blocks), dim3(64), lds, s, a);
  return hipGetLastError();
}

int max_resident_wide_blocks(int mode, int lds_bytes) {
  int n = 0;
  const hipError_t e =
      mode == 0 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, vd_mc_wide_kernel<16, 0, kWideWaves>, 64, lds_bytes)
      : mode == 2 ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, vd_mc_wide_kernel<16, 2, kWideWaves>, 64, lds_bytes)
                  : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, vd_mc_wide_kernel<16, 1, kWideWaves>, 64, lds_bytes);
  return e == hipSuccess ? n : 0;
}

// The budgets compiled: dense BFGS runs at three waves per SIMD on 64 lanes only (plan_for).
template <int G, int MODE, int W> constexpr int kBudget = MODE == 0 && G < 64 ? 2 : W;
template <int MODE, int W>
static hipError_t launch_mc_mode(int G, const McArgs& a, int blocks, int lds, hipStream_t s) {
  switch (G) {
    case 64: hipLaunchKernelGGL((vd_mc_kernel<64, MODE, kBudget<64, MODE, W>>), dim3(blocks), dim3(64), lds, s, a); break;
    case 32: hipLaunchKernelGGL((vd_mc_kernel<32, MODE, kBudget<32, MODE, W>>), dim3(blocks), dim3(64), lds, s, a); break;
    case 16: hipLaunchKernelGGL((vd_mc_kernel<16, MODE, kBudget<16, MODE, W>>), dim3(blocks), dim3(64), lds, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_mc(int G, int W, const McArgs& a, int blocks, hipStream_t s) {
  const int lds = mc_lds_bytes(G, a.Amax, a.Nmax, a.P.local_search == 0);
  if (a.P.local_search == 0) return W == 3 ? launch_mc_mode<0, 3>(G, a, blocks, lds, s) : launch_mc_mode<0, 2>(G, a, blocks, lds, s);
  if (a.P.policy == 1) {
    if (!a.hist) return hipErrorInvalidValue;
    switch (W) {
      case 3: return launch_mc_mode<2, 3>(G, a, blocks, lds, s);
      case 4: return launch_mc_mode<2, 4>(G, a, blocks, lds, s);
      default: return launch_mc_mode<2, 2>(G, a, blocks, lds, s);
    }
  }
  if (a.P.policy == 2) {
    if (!a.hist || !a.glob) return hipErrorInvalidValue;
    switch (W) {
      case 3: return launch_mc_mode<3, 3>(G, a, blocks, lds, s);
      case 4: return launch_mc_mode<3, 4>(G, a, blocks, lds, s);
      default: return launch_mc_mode<3, 2>(G, a, blocks, lds, s);
    }
  }
  switch (W) {
    case 3: return launch_mc_mode<1, 3>(G, a, blocks, lds, s);
    case 4: return launch_mc_mode<1, 4>(G, a, blocks, lds, s);
    default: return launch_mc_mode<1, 2>(G, a, blocks, lds, s);
  }
}

template <int MODE, int W>
static const void* mc_fn_mode(int G) {
  switch (G) {
    case 64: return reinterpret_cast<const void*>(&vd_mc_kernel<64, MODE, kBudget<64, MODE, W>>);
    case 32: return reinterpret_cast<const void*>(&vd_mc_kernel<32, MODE, kBudget<32, MODE, W>>);
    case 16: return reinterpret_cast<const void*>(&vd_mc_kernel<16, MODE, kBudget<16, MODE, W>>);
    default: return nullptr;
  }
}

// The instantiation launch_mc launches for (G, W, a), the same dispatch.
const void* mc_kernel_fn(int G, int W, const McArgs& a) {
  if (a.P.local_search == 0) return W == 3 ? mc_fn_mode<0, 3>(G) : mc_fn_mode<0, 2>(G);
  const int mode = a.P.policy == 1 ? 2 : a.P.policy == 2 ? 3 : 1;
  const int w = (W == 3 || W == 4) ? W : 2;
  switch (mode * 8 + w) {
    case 1 * 8 + 2: return mc_fn_mode<1, 2>(G);
    case 1 * 8 + 3: return mc_fn_mode<1, 3>(G);
    case 1 * 8 + 4: return mc_fn_mode<1, 4>(G);
    case 2 * 8 + 2: return mc_fn_mode<2, 2>(G);
    case 2 * 8 + 3: return mc_fn_mode<2, 3>(G);
    case 2 * 8 + 4: return mc_fn_mode<2, 4>(G);
    case 3 * 8 + 2: return mc_fn_mode<3, 2>(G);
    case 3 * 8 + 3: return mc_fn_mode<3, 3>(G);
    default: return mc_fn_mode<3, 4>(G);
  }
}

__global__ void vd_fill_int(int* p, int v) { *p = v; }
__global__ void vd_zero_u64_kernel(unsigned long long* p, int n) {
  for (int i = threadIdx.x; i < n; i += blockDim.x) p[i] = 0ull;
}
hipError_t zero_u64(unsigned long long* p, int n, hipStream_t s) {
  hipLaunchKernelGGL(vd_zero_u64_kernel, dim3(1), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

// Clears QuickVina-W global buffers: counters 0, conformation numbers 1e30 (never near),
// energies 0, zero-derivative masks all ones (an entry nobody wrote never explains a point).
__global__ void vd_glob_init_kernel(float* base, const long long* off, const int* per_axis, const int* T, int n) {
  for (int k = blockIdx.y; k < n; k += gridDim.y) {
  const long long cells = (long long)per_axis[k] * per_axis[k] * per_axis[k];
  const int t = T[k];
  float* b = base + off[k];
  const long long per_cell = 8LL * (12 + t);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < cells + cells * per_cell;
       i += (long long)gridDim.x * blockDim.x) {
    if (i < cells) { reinterpret_cast<int*>(b)[i] = 0; continue; }
    const long long j = (i - cells) % per_cell;      // position inside the cell's record
    float v = 0.0f;
    if (j < 8LL * (7 + t)) v = 1e30f;
    else if (j >= 8LL * (8 + t) && j < 8LL * (8 + t) + 16) v = __uint_as_float(0xFFFFFFFFu);   // Z masks
    b[i] = v;
  }
  }
}
hipError_t glob_init(float* base, const long long* off, const int* per_axis, const int* T, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(vd_glob_init_kernel, dim3(64, std::min(n, 1024)), dim3(256), 0, s, base, off, per_axis, T, n);
  return hipGetLastError();
}

// Random conformations of the adjoint benchmark: translation uniform in the box, orientation a
// normalised 4-Gaussian (uniform on rotations), torsions uniform in [-pi, pi).
__global__ void vd_random_confs_kernel(float* conf, long long n, int T, uint32_t seed, float3 lo, float3 hi) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  float* x = conf + c * (7 + T);
  const uint32_t cl = (uint32_t)c, ch = (uint32_t)(c >> 32);
  U4 w = philox(cl, ch, 0xFFFFFFFEu, 0, seed, 0x5EEDu);
  x[0] = lo.x + (hi.x - lo.x) * u01(w.x); x[1] = lo.y + (hi.y - lo.y) * u01(w.y); x[2] = lo.z + (hi.z - lo.z) * u01(w.z);
  w = philox(cl, ch, 0xFFFFFFFEu, 1, seed, 0x5EEDu);
  const float r0 = sqrtf(-2.0f * logf(u01(w.x) + 1.0f / 16777216.0f)), r1 = sqrtf(-2.0f * logf(u01(w.z) + 1.0f / 16777216.0f));
  float s0, c0, s1, c1;
  sincosf(2.0f * kPi * u01(w.y), &s0, &c0); sincosf(2.0f * kPi * u01(w.w), &s1, &c1);
  float q0 = r0 * c0, q1 = r0 * s0, q2 = r1 * c1, q3 = r1 * s1;
  const float inv = rsqrtf(fmaxf(q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3, 1e-30f));
  x[3] = q0 * inv; x[4] = q1 * inv; x[5] = q2 * inv; x[6] = q3 * inv;
  for (int j = 0; j < T; j += 4) {
    w = philox(cl, ch, 0xFFFFFFFEu, 2 + (uint32_t)(j / 4), seed, 0x5EEDu);
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
    for (int k = 0; k < 4 && j + k < T; ++k) x[7 + j + k] = -kPi + 2.0f * kPi * u01(ws[k]);
  }
}
hipError_t random_confs(float* conf, long long n, int T, uint32_t seed, const float lo[3], const float hi[3], hipStream_t s) {
  const int threads = 256;
  const long long blocks = (n + threads - 1) / threads;
  hipLaunchKernelGGL(vd_random_confs_kernel, dim3((unsigned)blocks), dim3(threads), 0, s, conf, n, T, seed,
                     make_float3(lo[0], lo[1], lo[2]), make_float3(hi[0], hi[1], hi[2]));
  return hipGetLastError();
}
hipError_t reset_counter(int* p, hipStream_t s) {
  hipLaunchKernelGGL(vd_fill_int, dim3(1), dim3(1), 0, s, p, 0);
  return hipGetLastError();
}

template <int MODE, int W>
static int occupancy(int G, int lds_bytes) {
  int n = 0;
  hipError_t e = hipErrorInvalidValue;
  switch (G) {
    case 64: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, vd_mc_kernel<64, MODE, kBudget<64, MODE, W>>, 64, lds_bytes); break;
    case 32: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, vd_mc_kernel<32, MODE, kBudget<32, MODE, W>>, 64, lds_bytes); break;
    case 16: e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, vd_mc_kernel<16, MODE, kBudget<16, MODE, W>>, 64, lds_bytes); break;
    default: break;
  }
  return e == hipSuccess ? n : 0;
}

// mode: 0 dense BFGS, 1 RILC-BFGS, 2 RILC-BFGS with the QuickVina2 history, 3 with QuickVina-W's
int max_resident_mc_blocks(int G, int W, int mode, int lds_bytes) {
  if (mode == 0) return W == 3 ? occupancy<0, 3>(G, lds_bytes) : occupancy<0, 2>(G, lds_bytes);
  if (mode == 2) return W == 3 ? occupancy<2, 3>(G, lds_bytes) : W == 4 ? occupancy<2, 4>(G, lds_bytes) : occupancy<2, 2>(G, lds_bytes);
  if (mode == 3) return W == 3 ? occupancy<3, 3>(G, lds_bytes) : W == 4 ? occupancy<3, 4>(G, lds_bytes) : occupancy<3, 2>(G, lds_bytes);
  return W == 3 ? occupancy<1, 3>(G, lds_bytes) : W == 4 ? occupancy<1, 4>(G, lds_bytes) : occupancy<1, 2>(G, lds_bytes);
}

}  // namespace vdl
