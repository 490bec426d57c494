// Work-unit evaluation stages (device functions).  A work unit is one thread block holding one
// or more whole systems in LDS.  The stages run in order, separated by block barriers:
//   stage_load      system table, tile tasks, parameters, coordinates -> LDS, accumulators zeroed
//   stage_psi       Born-radius integrals over 16 x 16 pair tiles (both directions per pair)
//   stage_radii     effective Born radii, GB self energies, self part of dE/dR (per atom, FP64)
//   stage_pairs     Coulomb + Lennard-Jones (exclusion masked) and GB pair energy / force / dE/dR
//   stage_chain     OBC chain rule on dE/dR (per atom, FP64)
//   stage_deriv     forces from the radius derivatives over the pair tiles
//   stage_valence   bonds, angles, cosine dihedrals and attenuated 1:4 pairs
// Forces, psi and dE/dR are accumulated in LDS as 64-bit fixed-precision integers, so the
// result does not depend on which lanes or work units processed which tiles.
#pragma once

#include <type_traits>

#include "mm_device.h"

namespace stormm_amd {

template <typename T> struct StageCtx {
  WuLds<T> L;
  WuDesc wu;
  int tid, nthr;
  int crd_shift;     // right shift from global fixed precision to LDS coordinates
  int org_shift;     // right shift from global fixed precision to the stored origins
  T crd_scale;       // LDS coordinate unit in Angstroms (single precision)
  int cycle;         // minimization cycle of this evaluation (clash-damping schedule)
  int rst_step;      // restraint step number when the kit gives no per-system cycle counts
  bool gb;
  int part = 0, parts = 1;  // this block's share of the unit's tile tasks and valence chunks
  bool move_pending = false;  // stage_load adds L.move[slot] x direction first
  __device__ StageCtx(unsigned char *smem, int maxa, int waves) : L(smem, maxa, waves) {}
};

// Slot of the unit's system that holds item t, given the running total F of each system's items
// over the earlier systems: the last system whose total does not exceed t.
template <int WuSys::*F>
__device__ __forceinline__ int find_slot(const WuSys *sys, int n, int t) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (sys[mid].*F <= t) {
      lo = mid;
    }
    else {
      hi = mid;
    }
  }
  return lo;
}

template <typename T>
__device__ __forceinline__ bool clash_params(const MMKit &k, int sys_index, int cycle, T &d,
                                             T &r);

// A coordinate after the pending line move mf (0: none), x += rint(mf * direction) with the
// normalized direction in the force arrays (line_movement.cui:343-360).
__device__ __forceinline__ long long moved(const long long *crd, const long long *dir, int g,
                                           double mf) {
  const long long x = crd[g];
  return (mf != 0.0) ? x + static_cast<long long>(__builtin_rint(mf *
                                                                 static_cast<double>(dir[g])))
                     : x;
}

// Work-unit set-up: system table, tile tasks, per-atom parameters, coordinates relative to a
// per-system origin (its first atom's position, with the bits below the LDS resolution cleared),
// and all accumulators zeroed.  Every thread takes its system's origin from the first atom
// itself, so that after the system table the tasks, parameters and coordinates all arrive in one
// round trip to memory: the set-up is latency, 4 us of a block's time with a barrier and a round
// trip for each of them.
// PHASE, in an evaluation in parts: the pair phase also loads the atoms' Born-radius integrals, the
// derivative phase their dE/dR and dR/dpsi.
enum PartPhase : int { kPartPsi = 0, kPartPairs = 1, kPartDeriv = 2, kWhole = 3 };
template <typename T, bool CLASH, int PHASE = kWhole>
__device__ __forceinline__ void stage_load(StageCtx<T> &c, const MMKit &k) {
  WuLds<T> &L = c.L;
  const WuDesc &wu = c.wu;
  {
    constexpr int kWords = sizeof(WuSys) / sizeof(int4);
    const int4 *src = reinterpret_cast<const int4 *>(k.wu_sys + wu.sys_first);
    int4 *dst = reinterpret_cast<int4 *>(L.sys);
    for (int e = c.tid; e < wu.sys_count * kWords; e += c.nthr) {
      dst[e] = src[e];
    }
  }
  for (int e = c.tid; e < wu.sys_count * 16; e += c.nthr) {
    L.nrg[e] = 0;
  }
  if (c.tid < kStageCounters) {
    L.work[c.tid] = 0;
  }
  __syncthreads();
  if (CLASH && c.tid < wu.sys_count) {
    T d, r;
    const bool on = clash_params<T>(k, L.sys[c.tid].sys_index, c.cycle, d, r);
    L.clash_d[c.tid] = on ? d : T(0);
    L.clash_r[c.tid] = on ? r : T(0);
    L.clash_on[c.tid] = on ? 1 : 0;
  }
  // A thread's atoms (at most two: blocks hold at least 256 threads), their moved coordinates
  // kept until every thread has read the unmoved ones.
  constexpr int kPer = kMaxWuAtoms / kMinEvalBlock;
  long long at[kPer][3];
  int owned[kPer];
#pragma unroll
  for (int it = 0; it < kPer; it++) {
    const int a = c.tid + (it * c.nthr);
    owned[it] = -1;
    if (a >= wu.lds_atoms) {
      continue;
    }
    const int s = find_slot<&WuSys::lds_base>(L.sys, wu.sys_count, a);
    const int gs = L.sys[s].global_start;
    const int local = a - L.sys[s].lds_base;
    const bool valid = local < L.sys[s].natom;
    const int g = gs + local;
    L.gidx[a] = valid ? g : -1;
    L.slot[a] = s;
    // In double precision the tile loops read j atoms from LDS as they come, so the padding slots
    // hold their far-away position themselves.
    const auto far = (sizeof(T) == 8) ? -FarAway<T>::kCrd : T(0);
    AtomPos<T> pos = {static_cast<typename Prec<T>::crd_t>(far),
                      static_cast<typename Prec<T>::crd_t>(far),
                      static_cast<typename Prec<T>::crd_t>(far), T(0)};
    AtomNb<T> nb = {T(0), T(0), T(0), T(1)};
    AtomRad<T> rr = {T(1), T(1)};
    if (valid) {
      nb.q = static_cast<T>(k.q[g]);
      if (wu.lj_table) {
        nb.p1 = static_cast<T>(k.lj_type[g]);
      }
      else {
        nb.p1 = static_cast<T>(0.5 * k.ljp1[g]);  // half sigma: sigma_ij = p1_i + p1_j
        nb.p2 = static_cast<T>(k.ljp2[g]);
      }
      const double rho = k.rho[g];
      rr.rho = static_cast<T>(rho);
      rr.irho = (rho > 0.0) ? static_cast<T>(Prec<double>::rcp(rho)) : T(0);
      pos.scr = static_cast<T>(k.scr[g]);
      bool ok;
      if (k.xcrd_ovrf != nullptr) {
        // 95-bit coordinates: origins kept in units of 2^-(gpos_bits - org_shift) A.
        auto wide = [&](const long long *crd, const int *ovr, int d) {
          const __int128 v = (i95_value(crd[gs], ovr[gs]) >> c.crd_shift) << c.crd_shift;
          const long long o = static_cast<long long>(v >> c.org_shift);
          if (local == 0) {
            L.org[3 * s + d] = o;
          }
          return i95_value(crd[g], ovr[g]) - (static_cast<__int128>(o) << c.org_shift);
        };
        const __int128 dx = wide(k.xcrd, k.xcrd_ovrf, 0);
        const __int128 dy = wide(k.ycrd, k.ycrd_ovrf, 1);
        const __int128 dz = wide(k.zcrd, k.zcrd_ovrf, 2);
        ok = CrdConv<T>::in_range_wide(dx, c.crd_shift) &&
             CrdConv<T>::in_range_wide(dy, c.crd_shift) &&
             CrdConv<T>::in_range_wide(dz, c.crd_shift);
        pos.x = CrdConv<T>::to_lds_wide(dx, c.crd_shift);
        pos.y = CrdConv<T>::to_lds_wide(dy, c.crd_shift);
        pos.z = CrdConv<T>::to_lds_wide(dz, c.crd_shift);
      }
      else {
        const double mf = c.move_pending ? L.move[s] : 0.0;
        const long long mask = ~((1LL << c.crd_shift) - 1LL);
        const long long gx = moved(k.xcrd, k.xfrc, g, mf);
        const long long gy = moved(k.ycrd, k.yfrc, g, mf);
        const long long gz = moved(k.zcrd, k.zfrc, g, mf);
        const long long ox = moved(k.xcrd, k.xfrc, gs, mf) & mask;
        const long long oy = moved(k.ycrd, k.yfrc, gs, mf) & mask;
        const long long oz = moved(k.zcrd, k.zfrc, gs, mf) & mask;
        if (local == 0) {
          L.org[3 * s + 0] = ox;
          L.org[3 * s + 1] = oy;
          L.org[3 * s + 2] = oz;
        }
        if (mf != 0.0) {
          owned[it] = g;
          at[it][0] = gx;
          at[it][1] = gy;
          at[it][2] = gz;
        }
        ok = CrdConv<T>::in_range(gx, ox, c.crd_shift) &&
             CrdConv<T>::in_range(gy, oy, c.crd_shift) &&
             CrdConv<T>::in_range(gz, oz, c.crd_shift);
        pos.x = CrdConv<T>::to_lds(gx, ox, c.crd_shift);
        pos.y = CrdConv<T>::to_lds(gy, oy, c.crd_shift);
        pos.z = CrdConv<T>::to_lds(gz, oz, c.crd_shift);
      }
      if (!ok) {
        atomicOr(k.status, static_cast<int>(kStatusCoordinateRange));
      }
    }
    AtomRec<T> &r = L.atom[a];
    r.pos = pos;
    r.nb = nb;
    r.rr = rr;
    r.psi = 0;
    r.fx = r.fy = r.fz = 0;
    r.dedr = 0;
    inv_radius(L, a) = T(1);
    if (PHASE == kPartPairs && valid && c.gb) {
      r.psi = k.part_psi[g];
    }
    if (PHASE == kPartDeriv && valid) {
      r.psi = __double_as_longlong(k.part_drdpsi[g]);
      r.dedr = k.part_dedr[g];
    }
  }
  // The unit's tile tasks, read once per evaluation: the clean off-diagonal tasks of every
  // system, then their other off-diagonal tasks, then the diagonal ones, each with its system's
  // LDS base added and its slot in the low bits of y.
  for (int t = c.tid; t < wu.task_count; t += c.nthr) {
    int s, idx;
    if (t < wu.clean_count) {
      s = find_slot<&WuSys::clean_pre>(L.sys, wu.sys_count, t);
      idx = L.sys[s].task_first + (t - L.sys[s].clean_pre);
    }
    else if (t < wu.offd_count) {
      const int to = t - wu.clean_count;
      s = find_slot<&WuSys::offd_pre>(L.sys, wu.sys_count, to);
      idx = L.sys[s].task_first + L.sys[s].clean_count + (to - L.sys[s].offd_pre);
    }
    else {
      const int td = t - wu.offd_count;
      s = find_slot<&WuSys::diag_pre>(L.sys, wu.sys_count, td);
      idx = L.sys[s].task_first + L.sys[s].offd_count + (td - L.sys[s].diag_pre);
    }
    int4 tk = k.tasks[idx];
    const int base = L.sys[s].lds_base;
    tk.x += base | (base << 16);
    tk.y |= s;
    L.tasks[t] = tk;
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kPer; it++) {
    if (owned[it] >= 0) {
      k.xcrd[owned[it]] = at[it][0];
      k.ycrd[owned[it]] = at[it][1];
      k.zcrd[owned[it]] = at[it][2];
    }
  }
}

template <typename T>
__device__ __forceinline__ void init_ctx(StageCtx<T> &c, const MMKit &k, int wu_index, int terms) {
  c.wu = k.wu[wu_index];
  c.tid = threadIdx.x;
  c.nthr = blockDim.x;
  if (sizeof(T) == 4) {
    c.crd_shift = (k.gpos_bits > kLdsCrdBits) ? (k.gpos_bits - kLdsCrdBits) : 0;
    c.crd_scale = T(ldexp(1.0, -(k.gpos_bits - c.crd_shift)));
  }
  else {
    c.crd_shift = k.gpos_bits;
    c.crd_scale = T(1);
  }
  c.org_shift = (k.xcrd_ovrf != nullptr) ? (k.gpos_bits - kOriginBits) : 0;
  c.gb = (k.igb != 0) && ((terms & kTermNonbonded) != 0);
  c.cycle = k.clash_cycle;
  c.rst_step = k.rst_step;
}

// Clash-damping parameters of one system for this evaluation
// (src/MolecularMechanics/hpc_minimization.cu:269-274): the floor and ratio shrink linearly to
// zero over the first clash_cycles cycles.  The damped potentials apply when either value
// exceeds 10^-6, the threshold at which the reference launches its damped kernels
// (src/Potential/hpc_nonbonded_potential.cu:1476 in double precision, :1662 in single).
template <typename T>
__device__ __forceinline__ bool clash_params(const MMKit &k, int sys_index, int cycle,
                                             T &dist, T &ratio) {
  double d = k.clash_r0, r = k.clash_ratio;
  if (k.clash_cycles > 0) {
    const int i = (k.clash_step != nullptr) ? k.clash_step[sys_index] + k.clash_step_offset
                                            : cycle;
    if (i < k.clash_cycles) {
      const double progress = static_cast<double>(k.clash_cycles - i) /
                              static_cast<double>(k.clash_cycles);
      d *= progress;
      r *= progress;
    }
    else {
      d = 0.0;
      r = 0.0;
    }
  }
  dist = static_cast<T>(d);
  ratio = static_cast<T>(r);
  if (sizeof(T) == 8) {
    return d >= 1.0e-6 || r >= 1.0e-6;
  }
  return static_cast<float>(d) > 0.000001f || static_cast<float>(r) > 0.000001f;
}

// Rotation-step mask of a 16-bit mask over the j atoms of a tile: bit ks of the result is bit
// (il - ks) mod 16 of jmask, the j atom lane il holds after ks rotations.  The reversed mask,
// rotated right by 15 - il, puts those bits in step order.
__device__ __forceinline__ unsigned step_mask(unsigned jmask, int il) {
  const unsigned r = __brev(jmask) >> 16;
  const int sh = (15 - il) & 15;
  return ((r >> sh) | (r << (16 - sh))) & 0xffffu;
}

// Number of rotation steps the wave runs for its current tasks: 16 when any of its rows holds
// an off-diagonal tile, 8 when all hold diagonal tiles.
__device__ __forceinline__ int wave_steps(bool diag) {
  const unsigned long long offd = __ballot(!diag);
  return (offd != 0ULL) ? 16 : 8;
}

// A tile task as seen by one lane of its 16-lane row.  Lane il starts with j lane jl0: il on an
// off-diagonal tile, il - 1 (mod 16) on a diagonal one, so that a diagonal tile's step ks meets
// the atom ks + 1 lanes back and its first 8 steps hold every pair of the tile once (the 8th
// step, which meets each pair twice, on lanes 0..7 only) and no atom paired with itself.  Bit ks
// of `valid` is set when the lane's pair at rotation step ks exists.
struct TileTask {
  int ib, jb, slot, ni, nj, i, jl0, j0, nsteps;
  bool diag, ivalid;
  unsigned valid;
  __device__ __forceinline__ TileTask(const Task &tk, int il) {
    ib = tk.x & 0xffff;
    jb = tk.x >> 16;
    slot = tk.y & 0xff;
    diag = ((tk.y >> 8) & 1) != 0;
    ni = (tk.y >> 12) & 0xff;
    nj = (tk.y >> 20) & 0xff;
    ivalid = il < ni;
    i = ib + il;
    jl0 = (il - (diag ? 1 : 0)) & 15;
    j0 = jb + jl0;
    const unsigned jm = (nj >= 16) ? 0xffffu : ((1u << nj) - 1u);
    unsigned v = step_mask(jm, jl0);
    if (diag) {
      v &= (il < 8) ? 0xffu : 0x7fu;
    }
    valid = ivalid ? v : 0u;
    nsteps = wave_steps(diag);
  }
  // The j lane whose sums a lane holds after the last step (the j sums move one lane per step).
  __device__ __forceinline__ int jl_home() const {
    return (jl0 - (nsteps - 1)) & 15;
  }
};

// Coordinates (Angstroms) and screened radii of lane il's i atom and first j atom of a tile.  The
// padding slots of a partial tile (lanes past ni on the i side, past nj on the j side) are put far
// away, so that their pairs are far-field pairs with terms of exactly zero in the Born-integral
// and derivative loops, which need no pair mask on off-diagonal tiles.
template <typename T>
__device__ __forceinline__ void tile_coords(const StageCtx<T> &c, const TileTask &tt, T &xi,
                                            T &yi, T &zi, T &xj, T &yj, T &zj, T &si, T &sj) {
  const AtomRec<T> *atom = c.L.atom;
  const AtomPos<T> bi = atom[tt.ib].pos, bj = atom[tt.jb].pos;
  const AtomPos<T> pi = atom[tt.i].pos, pj = atom[tt.j0].pos;
  const auto ox = tile_centre(bi.x, bj.x);
  const auto oy = tile_centre(bi.y, bj.y);
  const auto oz = tile_centre(bi.z, bj.z);
  const bool jvalid = tt.jl0 < tt.nj;
  xi = tt.ivalid ? tile_crd(pi.x, ox, c.crd_scale) : FarAway<T>::kCrd;
  yi = tt.ivalid ? tile_crd(pi.y, oy, c.crd_scale) : FarAway<T>::kCrd;
  zi = tt.ivalid ? tile_crd(pi.z, oz, c.crd_scale) : FarAway<T>::kCrd;
  xj = jvalid ? tile_crd(pj.x, ox, c.crd_scale) : -FarAway<T>::kCrd;
  yj = jvalid ? tile_crd(pj.y, oy, c.crd_scale) : -FarAway<T>::kCrd;
  zj = jvalid ? tile_crd(pj.z, oz, c.crd_scale) : -FarAway<T>::kCrd;
  si = pi.scr;
  sj = pj.scr;
}

// The j atom that a lane meets K rotation steps on: in double precision its record's fields, read
// from LDS, in single precision nothing (the rotated registers serve).
template <typename T> struct JAtom {
  AtomPos<T> pos;
  AtomNb<T> nb;
  T irad, sd;
  T s2, s3;                 // screened radius squared and cubed
};
template <int K> __device__ __forceinline__ JAtom<double> j_atom(const JRecords &j) {
  const AtomRec<double> &r = j.at<K>();
  JAtom<double> a;
  a.pos = r.pos;
  a.nb = r.nb;
  a.irad = r.irad;
  a.sd = r.sd;
  a.s2 = r.pos.scr * r.pos.scr;
  a.s3 = a.s2 * r.pos.scr;
  return a;
}
struct NoRecords {
  __device__ __forceinline__ NoRecords(AtomRec<float> *, int) {}
  template <int K> __device__ __forceinline__ void rotate() {}
};
template <int K> __device__ __forceinline__ JAtom<float> j_atom(const NoRecords &) {
  return JAtom<float>();
}
template <typename T>
using JSource = std::conditional_t<sizeof(T) == 8, JRecords, NoRecords>;
// A j value at step K: the record's field, or the register rotated K lanes (at the place of its
// use, so that the rotation folds into the instruction that reads it).
template <int K> __device__ __forceinline__ double j_value(double field, double) {
  return field;
}
template <int K> __device__ __forceinline__ float j_value(float, float reg) {
  return row_ror<K>(reg);
}
// Moves a register of j values on by K lanes (single precision).
template <int K> __device__ __forceinline__ void j_rotate(double &) {}
template <int K> __device__ __forceinline__ void j_rotate(float &reg) { reg = row_ror<K>(reg); }

// True on every lane when `b` holds on every active lane of the wavefront.
__device__ __forceinline__ bool wave_all(bool b) {
  return __ballot(!b) == 0ULL;
}

__device__ __forceinline__ bool step_bit(unsigned mask, int ks) {
  return ((mask >> ks) & 1u) != 0u;
}

// ------------------------------------------------------------------------------------------

// Tile task t of the work unit, placed at its system's LDS base and tagged with its slot
// (staged in LDS by stage_load).
template <typename T>
__device__ __forceinline__ Task fetch_task(const StageCtx<T> &c, const MMKit &, int t) {
  return c.L.tasks[t];
}

// Task dealing for the Born-integral stages: pass tb gives the four 16-lane rows of a
// wavefront four consecutive tasks; rows past the end of the list get an empty diagonal task,
// so every lane of a wavefront runs the same passes and rotation steps (the near queue below
// needs the whole wavefront at each step).
template <typename T>
__device__ __forceinline__ Task wave_task(const StageCtx<T> &c, const MMKit &k, int t) {
  if (t < c.wu.task_count) {
    return fetch_task(c, k, t);
  }
  return make_int4(0, 1 << 8, -1, 0);
}

// Work items of a stage are taken by the wavefronts of the block one at a time from a counter in
// LDS, so a wavefront that finishes early takes more items (the result does not depend on which
// wavefront took which item: every contribution goes to integer accumulators).
// In an evaluation in parts a block takes every parts-th item.
template <typename T>
__device__ __forceinline__ int next_item(const StageCtx<T> &c, int counter, int lane) {
  int item = 0;
  if (lane == 0) {
    item = atomicAdd(&c.L.work[counter], 1);
  }
  return (__builtin_amdgcn_readfirstlane(item) * c.parts) + c.part;
}

// Item i of a stage holding `quads` tile-task quads and `chunks` chunks of 64 valence terms, the
// chunks spread evenly among the quads so that latency-bound valence work overlaps the
// arithmetic of the tiles on the other wavefronts.  Returns the chunk index for a valence item
// and -1 - (quad index) for a tile item.
__device__ __forceinline__ int stage_item(int i, int quads, int chunks) {
  if (chunks == 0) {
    return -1 - i;
  }
  const unsigned total = static_cast<unsigned>(quads + chunks);
  const int c0 = static_cast<int>((static_cast<unsigned>(i) * chunks) / total);
  const int c1 = static_cast<int>((static_cast<unsigned>(i + 1) * chunks) / total);
  return (c1 > c0) ? c0 : (-1 - (i - c0));
}

template <typename T, bool FORCES, bool CLASH>
__device__ __forceinline__ void valence_term(StageCtx<T> &c, const MMKit &k, int kind, int t);

// Chunks of 64 valence terms of the unit: its bonds, then its angles, then its dihedrals, each
// kind starting a chunk of its own.
template <typename T> __device__ __forceinline__ int valence_chunks(const StageCtx<T> &c) {
  const WuDesc &wu = c.wu;
  return ((wu.bond_count + 63) >> 6) + ((wu.angl_count + 63) >> 6) +
         ((wu.term_count - wu.bond_count - wu.angl_count + 63) >> 6);
}

// Valence chunk `chunk` (wavefront-uniform), one term per lane.
template <typename T, bool FORCES, bool CLASH>
__device__ __forceinline__ void valence_chunk(StageCtx<T> &c, const MMKit &k, int chunk,
                                              int lane) {
  const int cb = (c.wu.bond_count + 63) >> 6;
  const int ca = (c.wu.angl_count + 63) >> 6;
  const int kind = (chunk < cb) ? kVBond : (chunk < cb + ca) ? kVAngle : kVDihedral;
  const int local = chunk - ((kind == kVBond) ? 0 : (kind == kVAngle) ? cb : cb + ca);
  valence_term<T, FORCES, CLASH>(c, k, kind, (local << 6) + lane);
}

// Near-field pair queue of a wavefront.  An entry packs the byte offsets of the pair's atom
// records (in double precision halved, to fit 16 bits) and which of the two directions (onto i,
// onto j) lies within 4 screened radii: j << 16 | i | near_i << 1 | near_j, where the offsets'
// low bits are free.
constexpr unsigned kNearI = 2u;
constexpr unsigned kNearJ = 1u;
template <typename T> struct NearIndex {
  static constexpr int kShift = (sizeof(T) == 4) ? 0 : 1;
  static constexpr unsigned kMask = 0xfff8u;
  static_assert(((kMaxWuAtoms - 1) * sizeof(AtomRec<T>)) >> kShift <= 0xffffu,
                "record offsets do not fit a near-queue entry");
  static_assert(((sizeof(AtomRec<T>) >> kShift) & ~kMask) == 0,
                "record offsets need their low bits for the near flags");
  // The halves of an entry's two parts, which nearq_push doubles.
  static __device__ __forceinline__ unsigned half_i(int i) {
    return static_cast<unsigned>(i) * static_cast<unsigned>(sizeof(AtomRec<T>) >> (kShift + 1));
  }
  static __device__ __forceinline__ int half_j(int j) {
    return static_cast<int>(half_i(j) << 16);
  }
  static __device__ __forceinline__ AtomRec<T> &record(AtomRec<T> *atom, unsigned off) {
    return *reinterpret_cast<AtomRec<T> *>(reinterpret_cast<unsigned char *>(atom) +
                                           (off << kShift));
  }
};

// LDS byte address of a pointer into the block's dynamic LDS.
__device__ __forceinline__ unsigned lds_address(const void *p) {
  return static_cast<unsigned>(reinterpret_cast<size_t>(
      (const __attribute__((address_space(3))) unsigned char *)p));
}

// Appends the entries of the lanes with a direction that is not far, in lane order, to the queue
// at LDS byte address q holding n entries (both wavefront-uniform).  All 64 lanes must run it.
// ei = half_i(i); ej = half_j of the j atom at step 0, rotated K lanes here.  Five
// vector instructions: the two flags enter as carries of the additions that join the indices
// (the first reads ej through DPP) and the store runs under the lanes' own mask, set and restored
// with scalar instructions inside one statement, so that the step stays one basic block.  A push
// made of selects and spare slots for the lanes without an entry took nine of a Born-integral
// step's 37 instructions; the stages are bound by vector-instruction issue.
template <int K>
__device__ __forceinline__ void nearq_push(unsigned q, int &n, bool far_i, bool far_j,
                                           unsigned ei, int ej) {
  // From the comparisons the step selects by: a ballot of their negations compares once more.
  const unsigned long long mi = ~__builtin_amdgcn_ballot_w64(far_i);
  const unsigned long long mj = ~__builtin_amdgcn_ballot_w64(far_j);
  const unsigned long long m = mi | mj;
  const unsigned lo = static_cast<unsigned>(m), hi = static_cast<unsigned>(m >> 32);
  const unsigned base = q + (static_cast<unsigned>(n) << 2);
  unsigned entry, slot;
  unsigned long long all;
  // The two scalar instructions ahead of the DPP read cover the wait that a vector write of ej
  // just before would need.
  if constexpr (K == 0) {
    asm volatile("s_mov_b64 vcc, %[mi]\n\t"
                 "v_addc_co_u32_e32 %[e], vcc, %[ej], %[ei], vcc\n\t"
                 "s_mov_b64 vcc, %[mj]\n\t"
                 "v_addc_co_u32_e32 %[e], vcc, %[e], %[e], vcc\n\t"
                 "v_mbcnt_lo_u32_b32 %[s], %[lo], 0\n\t"
                 "v_mbcnt_hi_u32_b32 %[s], %[hi], %[s]\n\t"
                 "v_lshl_add_u32 %[s], %[s], 2, %[base]\n\t"
                 "s_mov_b64 %[x], exec\n\t"
                 "s_mov_b64 exec, %[m]\n\t"
                 "ds_write_b32 %[s], %[e]\n\t"
                 "s_mov_b64 exec, %[x]"
                 : [e] "=&v"(entry), [s] "=&v"(slot), [x] "=&s"(all)
                 : [mi] "s"(mi), [mj] "s"(mj), [m] "s"(m), [lo] "s"(lo), [hi] "s"(hi),
                   [base] "s"(base), [ei] "v"(ei), [ej] "v"(ej)
                 : "vcc", "memory");
  }
  else {
    asm volatile("s_mov_b64 vcc, %[mi]\n\t"
                 "s_nop 0\n\t"
                 "v_addc_co_u32_dpp %[e], vcc, %[ej], %[ei], vcc row_ror:%[k] row_mask:0xf "
                 "bank_mask:0xf\n\t"
                 "s_mov_b64 vcc, %[mj]\n\t"
                 "v_addc_co_u32_e32 %[e], vcc, %[e], %[e], vcc\n\t"
                 "v_mbcnt_lo_u32_b32 %[s], %[lo], 0\n\t"
                 "v_mbcnt_hi_u32_b32 %[s], %[hi], %[s]\n\t"
                 "v_lshl_add_u32 %[s], %[s], 2, %[base]\n\t"
                 "s_mov_b64 %[x], exec\n\t"
                 "s_mov_b64 exec, %[m]\n\t"
                 "ds_write_b32 %[s], %[e]\n\t"
                 "s_mov_b64 exec, %[x]"
                 : [e] "=&v"(entry), [s] "=&v"(slot), [x] "=&s"(all)
                 : [mi] "s"(mi), [mj] "s"(mj), [m] "s"(m), [lo] "s"(lo), [hi] "s"(hi),
                   [base] "s"(base), [ei] "v"(ei), [ej] "v"(ej), [k] "n"(K)
                 : "vcc", "memory");
  }
  n += __popcll(m);
}

// The Born-integral and derivative stages run their rotation steps in groups of kStepGroup with
// compile-time rotation counts inside a group; the j-side data move kStepGroup lanes between
// groups, and the near-pair queue is drained after each group, taking 64 entries at a time from
// its end.  Before a group the queue holds at most 63 entries, and a group pushes at most 64 in
// each step.
constexpr int kStepGroup = 4;
static_assert(63 + (kStepGroup * 64) <= kNearQueue, "near queue too short for a step group");

// Geometry of a queued pair, recomputed from the LDS coordinates.
template <typename T> struct NearPair {
  AtomRec<T> &i, &j;
  bool near_i, near_j;
  T dx, dy, dz, r2, invr, r, si, sj;
  __device__ __forceinline__ NearPair(const StageCtx<T> &c, unsigned e)
      : i(NearIndex<T>::record(c.L.atom, e & NearIndex<T>::kMask)),
        j(NearIndex<T>::record(c.L.atom, e >> 16)) {
    using P = Prec<T>;
    near_i = (e & kNearI) != 0u;
    near_j = (e & kNearJ) != 0u;
    const AtomPos<T> pi = i.pos, pj = j.pos;
    dx = crd_delta(pj.x, pi.x, c.crd_scale);
    dy = crd_delta(pj.y, pi.y, c.crd_scale);
    dz = crd_delta(pj.z, pi.z, c.crd_scale);
    si = pi.scr;
    sj = pj.scr;
    r2 = (dx * dx) + (dy * dy) + (dz * dz);
    invr = P::rsqrt(r2);
    r = r2 * invr;
  }
};

// Near-field Born-integral terms of the first `count` queued pairs, one pair per lane.
template <typename T>
__device__ __forceinline__ void psi_drain(StageCtx<T> &c, const unsigned *q, int count,
                                          int lane) {
  if (lane < count) {
    const NearPair<T> p(c, q[lane]);
    const AtomRad<T> ri = p.i.rr, rj = p.j.rr;
    if (p.near_i) {
      const T t = psi_near(p.r, p.r2, p.invr, ri.rho, ri.irho, p.sj);
      lds_add(&p.i.psi, fixed_contrib(t, kPsiBits));
    }
    if (p.near_j) {
      const T t = psi_near(p.r, p.r2, p.invr, rj.rho, rj.irho, p.si);
      lds_add(&p.j.psi, fixed_contrib(t, kPsiBits));
    }
  }
}

// Born-radius integrals (src/Potential/nonbonded_potential.tpp:560-650).  Each lane evaluates
// the far-field series of its pair at every rotation step and queues the pair when either
// direction is within 4 screened radii; full wavefronts of queued pairs are evaluated together.
// The series terms of one task are summed in the working precision (at most 16 small terms per
// lane) and added to the fixed-precision accumulators once per task.  With x = (s / r)^2 for the
// sphere of screened radius s on the other atom, the far-field term is -s^3 / r^4 times the
// series in x, and r > 4 s is x < 1/16.
// Chunks of valence terms (`val_chunks`, possibly 0) are taken as work items alongside the tiles.
template <typename T, bool FORCES, bool CLASH>
__device__ __forceinline__ void stage_psi(StageCtx<T> &c, const MMKit &k, int val_chunks) {
  using P = Prec<T>;
  WuLds<T> &L = c.L;
  const int il = c.tid & 15;
  const int lane = c.tid & 63;
  // Wavefront-uniform, so the queue's base address stays in scalar registers.
  const int wave = __builtin_amdgcn_readfirstlane(c.tid >> 6);
  const unsigned *q = L.nearq + (wave * kNearQueueStride);
  const unsigned qaddr = lds_address(q);
  int qn = 0;
  const double psi_scale = ldexp(1.0, kPsiBits);
  const int quads = (c.wu.task_count + 3) >> 2;
  const int items = quads + val_chunks;
  for (int item = next_item(c, 0, lane); item < items; item = next_item(c, 0, lane)) {
    const int it = stage_item(item, quads, val_chunks);
    if (it >= 0) {
      valence_chunk<T, FORCES, CLASH>(c, k, it, lane);
      continue;
    }
    const TileTask tt(wave_task(c, k, ((-1 - it) << 2) + ((c.tid >> 4) & 3)), il);
    T xi, yi, zi, xj, yj, zj, si, sj;
    tile_coords(c, tt, xi, yi, zi, xj, yj, zj, si, sj);
    const T si2 = si * si;
    const T si3 = si2 * si;
    T sj2 = sj * sj;
    T sj3 = sj2 * sj;
    const unsigned ei = NearIndex<T>::half_i(tt.i);
    int ej = NearIndex<T>::half_j(tt.j0);
    T acci = T(0), accj = T(0);
    unsigned vbits = tt.valid;
    JSource<T> jrec(c.L.atom, tt.j0);
    // Off-diagonal tiles need no pair mask (their padding atoms sit far away); a wavefront whose
    // four tiles are all off-diagonal runs the 16 steps without one.  On diagonal tiles the mask
    // removes each lane's own atom and the second copy of each pair.
    auto run = [&](auto mc) {
      constexpr bool MASKED = decltype(mc)::value;
      const int nsteps = MASKED ? tt.nsteps : kTile;
      for (int g = 0; g < nsteps; g += kStepGroup) {
        auto step = [&](auto kc) {
          constexpr int K = decltype(kc)::value;
          if (MASKED && g + K >= nsteps) {
            return;
          }
          // An absent pair is put far away: both directions are then far-field with terms
          // that round to exactly zero, so no validity test follows.
          const bool valid = !MASKED || (((vbits >> K) & 1u) != 0u);
          const JAtom<T> aj = j_atom<K>(jrec);
          const T dx = j_value<K>(aj.pos.x, xj) - xi;
          const T dy = j_value<K>(aj.pos.y, yj) - yi;
          const T dz = j_value<K>(aj.pos.z, zj) - zi;
          const T r2c = (dx * dx) + (dy * dy) + (dz * dz);
          const T r2 = valid ? r2c : FarAway<T>::kR2;
          const T invr2 = P::rcp(r2);
          const T invr4 = invr2 * invr2;
          const T x_i = j_value<K>(aj.s2, sj2) * invr2;
          const T x_j = si2 * invr2;
          const bool far_i = x_i < T(0.0625);
          const bool far_j = x_j < T(0.0625);
          const T ti = psi_series(x_i) * (j_value<K>(aj.s3, sj3) * invr4);
          const T tj = psi_series(x_j) * (si3 * invr4);
          acci -= far_i ? ti : T(0);
          accj = row_rotate(accj) - (far_j ? tj : T(0));
          nearq_push<K>(qaddr, qn, far_i, far_j, ei, ej);
        };
        unrolled_steps(step, std::integer_sequence<int, 0, 1, 2, 3>{});
        settle(acci);
        vbits >>= kStepGroup;
        jrec.template rotate<kStepGroup>();
        j_rotate<kStepGroup>(xj);
        j_rotate<kStepGroup>(yj);
        j_rotate<kStepGroup>(zj);
        j_rotate<kStepGroup>(sj2);
        j_rotate<kStepGroup>(sj3);
        ej = row_ror<kStepGroup>(ej);
        while (qn >= 64) {
          psi_drain(c, q + (qn - 64), 64, lane);
          qn -= 64;
        }
      }
    };
    if (wave_all(!tt.diag)) {
      run(std::false_type{});
    }
    else {
      run(std::true_type{});
    }
    if (tt.ivalid) {
      lds_add(&L.atom[tt.i].psi, Prec<double>::fixed(static_cast<double>(acci) * psi_scale));
    }
    // After the last step the j sums sit nsteps - 1 lanes right of the lanes that loaded them.
    const int jl_home = tt.jl_home();
    if (jl_home < tt.nj) {
      lds_add(&L.atom[tt.jb + jl_home].psi,
              Prec<double>::fixed(static_cast<double>(accj) * psi_scale));
    }
  }
  psi_drain(c, q, qn, lane);
  __syncthreads();
}

// ------------------------------------------------------------------------------------------
// Effective radii (src/Potential/nonbonded_potential.tpp:731-781), self energies and the self
// part of the radius derivative accumulator (:784-806), all in double precision.
template <typename T, bool FORCES>
__device__ __forceinline__ void stage_radii(StageCtx<T> &c, const MMKit &k, double coulomb_inv_scaled) {
  WuLds<T> &L = c.L;
  const double nrg_scale = ldexp(1.0, k.nrg_bits);
  const double inv_diel = 1.0 / k.dielectric;
  for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
    const int g = L.gidx[a];
    if (g < 0) {
      continue;
    }
    const double psi = static_cast<double>(L.atom[a].psi) * ldexp(1.0, -kPsiBits);
    const BornRadius b = born_radius(k.igb, k.gb_alpha, k.gb_beta, k.gb_gamma, k.rho[g],
                                     k.pbr[g], psi);
    const double R = b.R;
    if (FORCES && k.igb != 1) {
      // Kept for the chain rule in the accumulator slot whose psi is no longer needed.
      L.atom[a].psi = __double_as_longlong(b.dr_dpsi);
    }
    L.atom[a].nb.rad = static_cast<T>(R);
    inv_radius(L, a) = static_cast<T>(b.inv_R);
    // q holds charge * sqrt(Coulomb), so q^2 = Coulomb * charge^2.
    const double qg = k.q[g];
    const double expmkf = ((k.kappa != 0.0) ? Prec<double>::exp(-kGbKscale * k.kappa * R) : 1.0) *
                          inv_diel;
    const double dielfac = 1.0 - expmkf;
    const double atmq2h = 0.5 * qg * qg;
    const double atmqd2h = atmq2h * dielfac;
    const double contrib = -atmqd2h / R;
    if (c.part != 0) {
      continue;  // the unit's first part adds the self terms
    }
    lds_add(&L.nrg[L.slot[a] * 16 + kGb], static_cast<long long>(__builtin_rint(contrib *
                                                                                  nrg_scale)));
    if (FORCES) {
      const double sdi = atmqd2h - (kGbKscale * k.kappa * atmq2h * expmkf * R);
      L.atom[a].dedr = static_cast<long long>(__builtin_rint(sdi * ldexp(1.0, kDedrBits)));
    }
  }
  (void)coulomb_inv_scaled;
  __syncthreads();
}

// ------------------------------------------------------------------------------------------
// Coulomb + Lennard-Jones (src/Potential/nonbonded_potential.tpp:174-231,312-373) and the GB
// pair energy, force and radius derivative (:811-972).  Every lane evaluates its pair at every
// step; absent and excluded pairs are removed by zeroing the charge product and the LJ
// coefficients, and the squared distance of an absent pair is replaced by 1 to keep the
// arithmetic finite.  Forces are summed per lane in the working precision and converted to fixed
// precision once per task.
// Damped Coulomb and Lennard-Jones of one pair at distance r (clash damping,
// src/Potential/nonbonded_potential_tilegroups.cui:536-602): inside clash distance cd the
// Coulomb potential becomes the parabola qq (ca (r + 1)^2 + cb), and inside ratio * sigma the
// Lennard-Jones potential becomes a (r + 1)^4 + b, each meeting the plain potential and its
// slope at the boundary.  fmag receives dE/dr / r.
template <typename T, bool FORCES>
__device__ __forceinline__ void clash_pair(T r, T qq, T lja, T ljb, T sigma, T cd, T ca, T cb,
                                           T ratio, T &e_qq, T &e_lj, T &fmag) {
  const T tiny = T(1.0e-10);   // constants::tiny, src/Constants/scaling.h:26
  if (r < cd) {
    e_qq += qq * ((ca * (r + T(1)) * (r + T(1))) + cb);
    if (FORCES && r > tiny) {
      fmag += qq * ((T(2) * ca) + (T(2) * ca / r));
    }
  }
  else {
    e_qq += qq / r;
    if (FORCES) {
      fmag -= qq / (r * r * r);
    }
  }
  const T vdw_limit = ratio * sigma;
  if (r < vdw_limit) {
    const T invrlim = T(1) / vdw_limit;
    const T invrlim2 = invrlim * invrlim;
    const T invrlim6 = invrlim2 * invrlim2 * invrlim2;
    const T aparm = (((T(6) * ljb) - (T(12) * lja * invrlim6)) * invrlim * invrlim6) /
                    ((((((T(4) * vdw_limit) + T(12)) * vdw_limit) + T(12)) * vdw_limit) + T(4));
    const T r_plus_one = r + T(1);
    const T arpo_three = aparm * r_plus_one * r_plus_one * r_plus_one;
    const T rlimit_plus_one = vdw_limit + T(1);
    const T arlimit_po_four = aparm * (rlimit_plus_one * rlimit_plus_one * rlimit_plus_one *
                                       rlimit_plus_one);
    const T bparm = (((lja * invrlim6) - ljb) * invrlim6) - arlimit_po_four;
    e_lj += (arpo_three * r_plus_one) + bparm;
    if (FORCES && r > tiny) {
      fmag += T(4) * arpo_three / r;
    }
  }
  else {
    const T invr2 = T(1) / (r * r);
    const T invr4 = invr2 * invr2;
    e_lj += ((lja * invr4 * invr2) - ljb) * invr4 * invr2;
    if (FORCES) {
      fmag += ((T(6) * ljb) - (T(12) * lja * invr4 * invr2)) * invr4 * invr4;
    }
  }
}

// CLASH selects the kernels that damp Coulomb and Lennard-Jones for the systems whose clash
// flag is set in this evaluation; the other systems take the plain potentials.  The rotation
// steps run in groups of kStepGroup with compile-time rotation counts, as in stage_psi: within a
// group the j-side data stay put and are read through DPP operands; the j-side accumulators move
// one lane per step.  The radius-derivative sums hold dE/dR / R and are scaled
// by the atom's radius at the end.
template <typename T, bool FORCES, bool LJTABLE, bool GB, bool CLASH>
__device__ __forceinline__ void stage_pairs(StageCtx<T> &c, const MMKit &k) {
  using P = Prec<T>;
  WuLds<T> &L = c.L;
  const int row = c.tid >> 4;
  const int nrows = c.nthr >> 4;
  const int il = c.tid & 15;
  const T frc_scale = T(ldexp(1.0, k.frc_bits));
  const T dedr_scale = T(ldexp(1.0, kDedrBits));
  const T nrg_scale = T(ldexp(1.0, k.nrg_bits));
  const T inv_diel = T(1.0 / k.dielectric);
  const T kap = T(k.kappa * kGbKscale);
  const bool use_kappa = (k.kappa != 0.0);
  const T dielfac0 = T(1) - inv_diel;
  // The steps leave out the 1/2 of the radius derivatives (a power of two: no rounding).
  const T dri_scale = T(0.5) * dedr_scale;
  for (int t = row + (c.part * nrows); t < c.wu.task_count; t += nrows * c.parts) {
    const Task tk = fetch_task(c, k, t);
    const TileTask tt(tk, il);
    const unsigned emask = (tk.z >= 0 && tt.ivalid) ? k.masks[tk.z + il] : 0u;
    const unsigned nbmask = tt.valid & ~step_mask(emask, tt.jl0);
    T xi, yi, zi, xj, yj, zj, si, sj;
    tile_coords(c, tt, xi, yi, zi, xj, yj, zj, si, sj);
    const AtomNb<T> ni = L.atom[tt.i].nb, nj = L.atom[tt.j0].nb;
    const T qi = ni.q, p1i = ni.p1, p2i = ni.p2, Ri = ni.rad;
    T qj = nj.q, p1j = nj.p1, p2j = nj.p2, Rj = nj.rad;
    // exp(-r^2 / (4 Ri Rj)) = GbExp(r^2 * (1 / Rj) * (scale / Ri)).
    T iRj = GB ? inv_radius(L, tt.j0) : T(0);
    const T iRi = GB ? inv_radius(L, tt.i) * GbExp<T>::kScale : T(0);
    JSource<T> jrec(c.L.atom, tt.j0);
    T fxi = T(0), fyi = T(0), fzi = T(0), dri = T(0);
    T fxj = T(0), fyj = T(0), fzj = T(0), drj = T(0);
    // Each lane sums its energies over the task in the calculation precision and converts the
    // sums to fixed precision once, as the reference does per tile
    // (src/Potential/nonbonded_potential_tilegroups.cui:461-464,640-645).
    T e_qq = T(0), e_lj = T(0), e_gb = T(0);
    // The row of the system's A / B table that atom i's type selects (a per-lane pointer, so
    // the steps need no kernel-argument registers to address it).
    const double2 *ljrow = nullptr;
    if (LJTABLE) {
      ljrow = k.ljab + L.sys[tt.slot].lj_off +
              (static_cast<int>(p1i) * L.sys[tt.slot].lj_nt);
    }
    bool clash_on = false;
    T cd = T(0), ca = T(0), cb = T(0), cratio = T(0);
    if (CLASH) {
      clash_on = (L.clash_on[tt.slot] != 0);
      cd = L.clash_d[tt.slot];
      cratio = L.clash_r[tt.slot];
      ca = T(-0.5) / (cd * cd * (cd + T(1)));
      cb = (T(1) / cd) - (ca * (cd + T(1)) * (cd + T(1)));
    }
    // The clash-damped kernels evaluate both potentials in one step (damping is per system, so a
    // wavefront's rows can differ): they rotate every step to stay within the register budget.
    constexpr int kGroup = CLASH ? 1 : kStepGroup;
    unsigned vbits = tt.valid, nbbits = nbmask;
    // A wavefront whose four tiles are all clean (off-diagonal, 16 x 16 atoms, no excluded pair)
    // runs the 16 steps without pair masks.
    auto run = [&](auto mc, auto kc) {
      constexpr bool MASKED = decltype(mc)::value;
      constexpr bool KAPPA = decltype(kc)::value;
      const int nsteps = MASKED ? tt.nsteps : kTile;
      for (int g = 0; g < nsteps; g += kGroup) {
        auto step = [&](auto sc) {
          constexpr int K = decltype(sc)::value;
          if (MASKED && g + K >= nsteps) {
            return;
          }
          const bool valid = !MASKED || (((vbits >> K) & 1u) != 0u);
          const bool nbok = !MASKED || (((nbbits >> K) & 1u) != 0u);
          const JAtom<T> aj = j_atom<K>(jrec);
          const T dx = j_value<K>(aj.pos.x, xj) - xi;
          const T dy = j_value<K>(aj.pos.y, yj) - yi;
          const T dz = j_value<K>(aj.pos.z, zj) - zi;
          const T r2c = (dx * dx) + (dy * dy) + (dz * dz);
          const T r2 = valid ? r2c : T(1);
          const T qiqj = j_value<K>(aj.nb.q, qj) * qi;
          T fmag = T(0);
          if (GB) {
            const T qgb = valid ? qiqj : T(0);
            const T rr = j_value<K>(aj.nb.rad, Rj) * Ri;
            const T efac = GbExp<T>::eval(r2 * (j_value<K>(aj.irad, iRj) * iRi));
            const T fgb2 = r2 + (rr * efac);
            const T fgbi = P::rsqrt(fgb2);
            // egb = qq (1 - exp(-kappa fgb) / diel) / fgb, temp6 = -(dE/dfgb) / fgb.
            T egb, temp6;
            if (KAPPA) {
              const T fgbk = -kap * fgb2 * fgbi;
              const T expmkf = P::exp(fgbk) * inv_diel;
              const T dielfac = T(1) - expmkf;
              const T qf = qgb * fgbi;
              egb = qf * dielfac;
              temp6 = qf * fgbi * fgbi * (dielfac + (fgbk * expmkf));
            }
            else {
              egb = qgb * fgbi * dielfac0;
              temp6 = egb * fgbi * fgbi;
            }
            e_gb -= egb;
            if (FORCES) {
              fmag += temp6 * (T(1) - (T(0.25) * efac));
              const T temp5 = efac * temp6 * (rr + (T(0.25) * r2));
              dri += temp5;
              drj = row_rotate(drj) + temp5;
            }
          }
          const T qnb = nbok ? qiqj : T(0);
          if (CLASH && clash_on) {
            const T pj1 = j_value<K>(aj.nb.p1, p1j);
            const T pj2 = j_value<K>(aj.nb.p2, p2j);
            T lja, ljb, sigma;
            if (LJTABLE) {
              const double2 ab = ljrow[static_cast<int>(pj1)];
              lja = nbok ? static_cast<T>(ab.x) : T(0);
              ljb = nbok ? static_cast<T>(ab.y) : T(0);
              sigma = (ljb > T(1.0e-6)) ? P::sqrt(P::cbrt(lja / ljb)) : T(0);
            }
            else {
              const T sig = p1i + pj1;
              const T sig2 = sig * sig;
              const T sig6 = sig2 * sig2 * sig2;
              const T e4 = nbok ? p2i * pj2 : T(0);
              ljb = e4 * sig6;
              lja = ljb * sig6;
              sigma = (ljb > T(1.0e-6)) ? sig : T(0);
            }
            clash_pair<T, FORCES>(P::sqrt(r2), qnb, lja, ljb, sigma, cd, ca, cb, cratio, e_qq, e_lj,
                                  fmag);
          }
          else {
            const T invr = P::rsqrt(r2);
            const T invr2 = invr * invr;
            const T eqq = qnb * invr;
            e_qq += eqq;
            if (LJTABLE) {
              const double2 ab = ljrow[static_cast<int>(j_value<K>(aj.nb.p1, p1j))];
              const T lja = nbok ? static_cast<T>(ab.x) : T(0);
              const T ljb = nbok ? static_cast<T>(ab.y) : T(0);
              const T invr4 = invr2 * invr2;
              e_lj += ((lja * invr4 * invr4) - (ljb * invr2)) * invr4;
              if (FORCES) {
                fmag += ((T(6) * ljb) - (T(12) * lja * invr4 * invr2)) * invr4 * invr4;
              }
            }
            else {
              const T sig = j_value<K>(aj.nb.p1, p1j) + p1i;
              const T s2 = sig * sig * invr2;
              const T s6 = s2 * s2 * s2;
              const T e4c = j_value<K>(aj.nb.p2, p2j) * p2i;
              const T e4 = nbok ? e4c : T(0);
              const T e4s6 = e4 * s6;
              e_lj += e4s6 * (s6 - T(1));
              if (FORCES) {
                fmag += e4s6 * (T(6) - (T(12) * s6)) * invr2;
              }
            }
            if (FORCES) {
              fmag -= eqq * invr2;
            }
          }
          if (FORCES) {
            const T fdx = fmag * dx;
            const T fdy = fmag * dy;
            const T fdz = fmag * dz;
            fxi += fdx;
            fyi += fdy;
            fzi += fdz;
            fxj = row_rotate(fxj) - fdx;
            fyj = row_rotate(fyj) - fdy;
            fzj = row_rotate(fzj) - fdz;
          }
        };
        unrolled_steps(step, std::make_integer_sequence<int, kGroup>{});
        vbits >>= kGroup;
        nbbits >>= kGroup;
        jrec.template rotate<kGroup>();
        j_rotate<kGroup>(xj);
        j_rotate<kGroup>(yj);
        j_rotate<kGroup>(zj);
        j_rotate<kGroup>(qj);
        j_rotate<kGroup>(p1j);
        j_rotate<kGroup>(p2j);
        if (GB) {
          j_rotate<kGroup>(Rj);
          j_rotate<kGroup>(iRj);
        }
      }
    };
    // The kappa choice is made here too, so that no branch splits the steps.
    const bool clean = wave_all(!tt.diag && tt.ni == kTile && tt.nj == kTile && tk.z < 0);
    if (GB && use_kappa) {
      if (clean) {
        run(std::false_type{}, std::true_type{});
      }
      else {
        run(std::true_type{}, std::true_type{});
      }
    }
    else if (clean) {
      run(std::false_type{}, std::false_type{});
    }
    else {
      run(std::true_type{}, std::false_type{});
    }
    if (FORCES) {
      if (tt.ivalid) {
        AtomRec<T> &ri = L.atom[tt.i];
        lds_add(&ri.fx, P::fixed(fxi * frc_scale));
        lds_add(&ri.fy, P::fixed(fyi * frc_scale));
        lds_add(&ri.fz, P::fixed(fzi * frc_scale));
        if (GB) {
          lds_add(&ri.dedr, P::fixed(Ri * dri * dri_scale));
        }
      }
      // After the last step the j sums sit nsteps - 1 lanes right of the lanes that loaded them.
      const int jl_home = tt.jl_home();
      if (jl_home < tt.nj) {
        AtomRec<T> &rj = L.atom[tt.jb + jl_home];
        lds_add(&rj.fx, P::fixed(fxj * frc_scale));
        lds_add(&rj.fy, P::fixed(fyj * frc_scale));
        lds_add(&rj.fz, P::fixed(fzj * frc_scale));
        if (GB) {
          lds_add(&rj.dedr, P::fixed(rj.nb.rad * drj * dri_scale));
        }
      }
    }
    const long long vqq = row_sum(P::fixed(e_qq * nrg_scale));
    const long long vlj = row_sum(P::fixed(e_lj * nrg_scale));
    const long long vgb = GB ? row_sum(P::fixed(e_gb * nrg_scale)) : 0LL;
    if (il == 0) {
      lds_add(&L.nrg[tt.slot * 16 + kElec], vqq);
      lds_add(&L.nrg[tt.slot * 16 + kVdw], vlj);
      if (GB) {
        lds_add(&L.nrg[tt.slot * 16 + kGb], vgb);
      }
    }
  }
  __syncthreads();
}

// ------------------------------------------------------------------------------------------
// OBC chain rule on the accumulated radius derivatives, src/Potential/nonbonded_potential.tpp:
// 985-1017.  The HCT model uses the accumulated values as they stand.  The factor takes the place
// of the atom's dR/dpsi.
template <typename T>
__device__ __forceinline__ void stage_chain(StageCtx<T> &c, const MMKit &k) {
  WuLds<T> &L = c.L;
  for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
    const int g = L.gidx[a];
    if (g < 0) {
      L.atom[a].sd = T(0);
      continue;
    }
    double sdi = static_cast<double>(L.atom[a].dedr) * ldexp(1.0, -kDedrBits);
    if (k.igb != 1) {
      // The radii stage left dR/dpsi in the psi slot.
      sdi *= __longlong_as_double(L.atom[a].psi);
    }
    L.atom[a].sd = static_cast<T>(sdi);
  }
  __syncthreads();
}

// ------------------------------------------------------------------------------------------
// Near-field radius-derivative forces of the first `count` queued pairs, one pair per lane.
template <typename T>
__device__ __forceinline__ void deriv_drain(StageCtx<T> &c, const unsigned *q, int count,
                                            int lane, int frc_bits) {
  if (lane < count) {
    const NearPair<T> p(c, q[lane]);
    const AtomRad<T> ri = p.i.rr, rj = p.j.rr;
    const T invr2 = p.invr * p.invr;
    T fmag = T(0);
    if (p.near_i) {
      fmag += dpsi_near(p.r, p.r2, p.invr, invr2, ri.rho, ri.irho, p.sj) * p.i.sd;
    }
    if (p.near_j) {
      fmag += dpsi_near(p.r, p.r2, p.invr, invr2, rj.rho, rj.irho, p.si) * p.j.sd;
    }
    const long long fx = fixed_contrib(fmag * p.dx, frc_bits);
    const long long fy = fixed_contrib(fmag * p.dy, frc_bits);
    const long long fz = fixed_contrib(fmag * p.dz, frc_bits);
    lds_add(&p.i.fx, -fx);
    lds_add(&p.i.fy, -fy);
    lds_add(&p.i.fz, -fz);
    lds_add(&p.j.fx, fx);
    lds_add(&p.j.fy, fy);
    lds_add(&p.j.fz, fz);
  }
}

// Forces from the Born-radius derivatives, src/Potential/nonbonded_potential.tpp:1018-1292,
// with the same far-field / queued near-field split and step groups as stage_psi.  Far-field
// forces are summed per lane in the working precision and converted to fixed precision once per
// task.
template <typename T>
// Always inlined: kept whole inside the kernels that evaluate forces.
__device__ __forceinline__ void stage_deriv(StageCtx<T> &c, const MMKit &k) {
  using P = Prec<T>;
  WuLds<T> &L = c.L;
  const int il = c.tid & 15;
  const int lane = c.tid & 63;
  // Wavefront-uniform, so the queue's base address stays in scalar registers.
  const int wave = __builtin_amdgcn_readfirstlane(c.tid >> 6);
  const unsigned *q = L.nearq + (wave * kNearQueueStride);
  const unsigned qaddr = lds_address(q);
  int qn = 0;
  const T frc_scale = T(ldexp(1.0, k.frc_bits));
  const int quads = (c.wu.task_count + 3) >> 2;
  for (int item = next_item(c, 1, lane); item < quads; item = next_item(c, 1, lane)) {
    const TileTask tt(wave_task(c, k, (item << 2) + ((c.tid >> 4) & 3)), il);
    T xi, yi, zi, xj, yj, zj, si, sj;
    tile_coords(c, tt, xi, yi, zi, xj, yj, zj, si, sj);
    const T sdi = L.atom[tt.i].sd;
    const T si2 = si * si;
    const T si3 = si2 * si;
    T sj2 = sj * sj;
    T sj3 = sj2 * sj;
    T sdj = L.atom[tt.j0].sd;
    const unsigned ei = NearIndex<T>::half_i(tt.i);
    int ej = NearIndex<T>::half_j(tt.j0);
    T fxi = T(0), fyi = T(0), fzi = T(0);
    T gxj = T(0), gyj = T(0), gzj = T(0);
    unsigned vbits = tt.valid;
    JSource<T> jrec(c.L.atom, tt.j0);
    // Wavefronts of four off-diagonal tiles run without a pair mask, as in stage_psi.
    auto run = [&](auto mc) {
      constexpr bool MASKED = decltype(mc)::value;
      const int nsteps = MASKED ? tt.nsteps : kTile;
      for (int g = 0; g < nsteps; g += kStepGroup) {
        auto step = [&](auto kc) {
          constexpr int K = decltype(kc)::value;
          if (MASKED && g + K >= nsteps) {
            return;
          }
          // Absent pairs are put far away, as in stage_psi.
          const bool valid = !MASKED || (((vbits >> K) & 1u) != 0u);
          const JAtom<T> aj = j_atom<K>(jrec);
          const T dx = j_value<K>(aj.pos.x, xj) - xi;
          const T dy = j_value<K>(aj.pos.y, yj) - yi;
          const T dz = j_value<K>(aj.pos.z, zj) - zi;
          const T r2c = (dx * dx) + (dy * dy) + (dz * dz);
          const T r2 = valid ? r2c : FarAway<T>::kR2;
          const T invr2 = P::rcp(r2);
          const T invr6 = invr2 * invr2 * invr2;
          const T x_i = j_value<K>(aj.s2, sj2) * invr2;
          const T x_j = si2 * invr2;
          const bool far_i = x_i < T(0.0625);
          const bool far_j = x_j < T(0.0625);
          // Both series are evaluated on every lane and selected, which keeps the step free of
          // branches.
          const T ti = dpsi_series(x_i) * (j_value<K>(aj.s3, sj3) * (invr6 * sdi));
          const T tj = dpsi_series(x_j) * (j_value<K>(aj.sd, sdj) * (invr6 * si3));
          const T fmag = (far_i ? ti : T(0)) + (far_j ? tj : T(0));
          const T fdx = fmag * dx;
          const T fdy = fmag * dy;
          const T fdz = fmag * dz;
          fxi -= fdx;
          fyi -= fdy;
          fzi -= fdz;
          gxj = row_rotate(gxj) + fdx;
          gyj = row_rotate(gyj) + fdy;
          gzj = row_rotate(gzj) + fdz;
          nearq_push<K>(qaddr, qn, far_i, far_j, ei, ej);
        };
        unrolled_steps(step, std::integer_sequence<int, 0, 1, 2, 3>{});
        settle(fxi);
        settle(fyi);
        settle(fzi);
        vbits >>= kStepGroup;
        jrec.template rotate<kStepGroup>();
        j_rotate<kStepGroup>(xj);
        j_rotate<kStepGroup>(yj);
        j_rotate<kStepGroup>(zj);
        j_rotate<kStepGroup>(sj2);
        j_rotate<kStepGroup>(sj3);
        j_rotate<kStepGroup>(sdj);
        ej = row_ror<kStepGroup>(ej);
        while (qn >= 64) {
          deriv_drain(c, q + (qn - 64), 64, lane, k.frc_bits);
          qn -= 64;
        }
      }
    };
    if (wave_all(!tt.diag)) {
      run(std::false_type{});
    }
    else {
      run(std::true_type{});
    }
    if (tt.ivalid) {
      AtomRec<T> &ri = L.atom[tt.i];
      lds_add(&ri.fx, P::fixed(fxi * frc_scale));
      lds_add(&ri.fy, P::fixed(fyi * frc_scale));
      lds_add(&ri.fz, P::fixed(fzi * frc_scale));
    }
    const int jl_home = tt.jl_home();
    if (jl_home < tt.nj) {
      AtomRec<T> &rj = L.atom[tt.jb + jl_home];
      lds_add(&rj.fx, P::fixed(gxj * frc_scale));
      lds_add(&rj.fy, P::fixed(gyj * frc_scale));
      lds_add(&rj.fz, P::fixed(gzj * frc_scale));
    }
  }
  deriv_drain(c, q, qn, lane, k.frc_bits);
  __syncthreads();
}

// ------------------------------------------------------------------------------------------
// Valence terms.  They are O(N) work, so both precision models evaluate them in double
// precision: a single-precision r - r0 or theta - theta0 near equilibrium loses most of its
// significant bits.  Displacements come from the LDS coordinates (exact in the double-precision
// model; 2^-24 Angstrom steps in the single-precision model, far finer than the bits such a
// difference keeps in single precision).
// ------------------------------------------------------------------------------------------
struct Vec3 {
  double x, y, z;
};
__device__ __forceinline__ Vec3 cross(const Vec3 &a, const Vec3 &b) {
  return {(a.y * b.z) - (a.z * b.y), (a.z * b.x) - (a.x * b.z), (a.x * b.y) - (a.y * b.x)};
}
__device__ __forceinline__ double dot(const Vec3 &a, const Vec3 &b) {
  return (a.x * b.x) + (a.y * b.y) + (a.z * b.z);
}

struct Vec3f {
  float x, y, z;
};
__device__ __forceinline__ Vec3f cross(const Vec3f &a, const Vec3f &b) {
  return {(a.y * b.z) - (a.z * b.y), (a.z * b.x) - (a.x * b.z), (a.x * b.y) - (a.y * b.x)};
}
__device__ __forceinline__ float dot(const Vec3f &a, const Vec3f &b) {
  return (a.x * b.x) + (a.y * b.y) + (a.z * b.z);
}

template <typename T> struct ValenceCtxT {
  AtomRec<T> *atom;
  const int *gidx;
  double crd_scale;
  float crd_scale_f;
  __device__ __forceinline__ explicit ValenceCtxT(const StageCtx<T> &c)
      : atom(c.L.atom), gidx(c.L.gidx), crd_scale(static_cast<double>(c.crd_scale)),
        crd_scale_f(static_cast<float>(c.crd_scale)) {}
  // Absolute position (A) of LDS atom a of a system whose coordinate origin is org (fixed
  // precision at inv_gpos).
  __device__ __forceinline__ Vec3 absolute(int a, const long long *org, double inv_gpos) const {
    const AtomPos<T> p = atom[a].pos;
    return {(static_cast<double>(org[0]) * inv_gpos) + (static_cast<double>(p.x) * crd_scale),
            (static_cast<double>(org[1]) * inv_gpos) + (static_cast<double>(p.y) * crd_scale),
            (static_cast<double>(org[2]) * inv_gpos) + (static_cast<double>(p.z) * crd_scale)};
  }
  // Single-precision displacement: the LDS coordinates' difference is exact, then rounded once.
  __device__ __forceinline__ Vec3f dispf(int from, int to) const {
    const AtomPos<T> a = atom[from].pos, b = atom[to].pos;
    return {static_cast<float>(b.x - a.x) * crd_scale_f,
            static_cast<float>(b.y - a.y) * crd_scale_f,
            static_cast<float>(b.z - a.z) * crd_scale_f};
  }
  __device__ __forceinline__ Vec3 disp(int from, int to) const {
    const AtomPos<T> a = atom[from].pos, b = atom[to].pos;
    return {(static_cast<double>(b.x) - static_cast<double>(a.x)) * crd_scale,
            (static_cast<double>(b.y) - static_cast<double>(a.y)) * crd_scale,
            (static_cast<double>(b.z) - static_cast<double>(a.z)) * crd_scale};
  }
  __device__ __forceinline__ void add(int a, long long vx, long long vy, long long vz) const {
    AtomRec<T> &r = atom[a];
    lds_add(&r.fx, vx);
    lds_add(&r.fy, vy);
    lds_add(&r.fz, vz);
  }
};

__device__ __forceinline__ long long fix64(double v) { return round_to_ll(v); }

// Harmonic bond, src/Potential/valence_potential.tpp:9-96.
template <bool FORCES, typename V>
__device__ __forceinline__ double eval_bond(const V &v, int i, int j, double kb,
                                            double r0, double fscale) {
  const Vec3 d = v.disp(i, j);
  using D = Prec<double>;
  const double d2 = dot(d, d);
  const double inv = D::rsqrt(d2);
  const double dr = (d2 > 0.0) ? D::root(d2, inv) : 0.0;
  const double dl = dr - r0;
  if (FORCES) {
    const double fmag = D::quotient(2.0 * kb * dl, dr, inv);
    const long long ix = fix64(fmag * d.x * fscale);
    const long long iy = fix64(fmag * d.y * fscale);
    const long long iz = fix64(fmag * d.z * fscale);
    v.add(i, ix, iy, iz);
    v.add(j, -ix, -iy, -iz);
  }
  return kb * dl * dl;
}

// Harmonic angle, src/Potential/valence_potential.tpp:170-287.
template <bool FORCES, typename V>
__device__ __forceinline__ double eval_angle(const V &v, int i, int j, int kk,
                                             double ka, double th0, double fscale) {
  const Vec3 ba = v.disp(j, i);
  const Vec3 bc = v.disp(j, kk);
  using D = Prec<double>;
  const double mgba = dot(ba, ba);
  const double mgbc = dot(bc, bc);
  const double mg2 = mgba * mgbc;
  const double invmg = D::rsqrt(mg2);
  const double invbabc = D::quotient(1.0, D::root(mg2, invmg), invmg);
  double costheta = dot(ba, bc) * invbabc;
  costheta = (costheta < -1.0) ? -1.0 : ((costheta > 1.0) ? 1.0 : costheta);
  const double theta = acos(costheta);
  const double dtheta = theta - th0;
  if (FORCES) {
    const double sin2 = 1.0 - (costheta * costheta);
    const double invsin = D::rsqrt(sin2);
    const double dA = D::quotient(-2.0 * ka * dtheta, D::root(sin2, invsin), invsin);
    const double sqba = D::quotient(dA, mgba, D::rcp(mgba));
    const double sqbc = D::quotient(dA, mgbc, D::rcp(mgbc));
    const double mbabc = dA * invbabc;
    const long long iax = fix64(((bc.x * mbabc) - (costheta * ba.x * sqba)) * fscale);
    const long long iay = fix64(((bc.y * mbabc) - (costheta * ba.y * sqba)) * fscale);
    const long long iaz = fix64(((bc.z * mbabc) - (costheta * ba.z * sqba)) * fscale);
    const long long icx = fix64(((ba.x * mbabc) - (costheta * bc.x * sqbc)) * fscale);
    const long long icy = fix64(((ba.y * mbabc) - (costheta * bc.y * sqbc)) * fscale);
    const long long icz = fix64(((ba.z * mbabc) - (costheta * bc.z * sqbc)) * fscale);
    v.add(i, -iax, -iay, -iaz);
    v.add(j, iax + icx, iay + icy, iaz + icz);
    v.add(kk, -icx, -icy, -icz);
  }
  return ka * dtheta * dtheta;
}

// Cosine dihedral, src/Potential/valence_potential.tpp:359-578: E = A (1 + cos(n theta - phase))
// with the force factor A n sin(n theta - phase).  The reference recovers the signed angle
// theta with an arccosine (src/Math/rounding.tpp:24-59) and then takes the sine and cosine of
// n theta - phase.  For the integer periodicities used here both functions follow exactly from
// cos(theta) and sin(theta) by the multiple-angle expansion (cos theta + i sin theta)^n, and the
// phase enters through its precomputed cosine and sine.  cos(theta) is the normalized dot
// product of the two plane normals and the signed sin(theta) their cross product projected on
// the central bond (the reference's sign convention for theta), so no inverse or forward
// trigonometric function is evaluated.
template <bool FORCES, typename V>
__device__ __forceinline__ double eval_dihedral(const V &v, int i, int j, int kk, int l,
                                                const DiheParam &dp, double fscale) {
  const Vec3 ab = v.disp(i, j);
  const Vec3 bc = v.disp(j, kk);
  const Vec3 cd = v.disp(kk, l);
  Vec3 crabbc = cross(ab, bc);
  Vec3 crbccd = cross(bc, cd);
  const double inv12 = 1.0 / sqrt(dot(crabbc, crabbc) * dot(crbccd, crbccd));
  const double mgbc = sqrt(dot(bc, bc));
  const Vec3 scr = cross(crabbc, crbccd);
  const double cth = dot(crabbc, crbccd) * inv12;
  const double sth = dot(scr, bc) * inv12 / mgbc;
  double cn = 1.0, sn = 0.0;
  for (int p = 0; p < dp.period; p++) {
    const double t = (cn * cth) - (sn * sth);
    sn = (sn * cth) + (cn * sth);
    cn = t;
  }
  const double cos_sangle = (cn * dp.cos_phase) + (sn * dp.sin_phase);
  if (FORCES) {
    const double sin_sangle = (sn * dp.cos_phase) - (cn * dp.sin_phase);
    const double fr = dp.amp * static_cast<double>(dp.period) * sin_sangle;
    const double mgab = sqrt(dot(ab, ab));
    const double mgcd = sqrt(dot(cd, cd));
    const double invab = 1.0 / mgab;
    const double invbc = 1.0 / mgbc;
    const double invcd = 1.0 / mgcd;
    const double cosb = -dot(ab, bc) * invab * invbc;
    const double cosc = -dot(bc, cd) * invbc * invcd;
    // src/Constants/symbol_values.h:72-82 (asymptotic_to_one_lf, inverse_one_minus_asymptote)
    const double isinb2 = (cosb * cosb < 0.99999904632568359375) ? fr / (1.0 - (cosb * cosb)) :
                                                                   fr * 1048576.0;
    const double isinc2 = (cosc * cosc < 0.99999904632568359375) ? fr / (1.0 - (cosc * cosc)) :
                                                                   fr * 1048576.0;
    const double invabc = invab * invbc;
    const double invbcd = invbc * invcd;
    crabbc = {crabbc.x * invabc, crabbc.y * invabc, crabbc.z * invabc};
    crbccd = {crbccd.x * invbcd, crbccd.y * invbcd, crbccd.z * invbcd};
    const double fa = -invab * isinb2;
    const double fb1 = (mgbc - (mgab * cosb)) * invabc * isinb2;
    const double fb2 = cosc * invbc * isinc2;
    const double fd = -invcd * isinc2;
    const long long fix = fix64(crabbc.x * fa * fscale);
    const long long fiy = fix64(crabbc.y * fa * fscale);
    const long long fiz = fix64(crabbc.z * fa * fscale);
    v.add(i, fix, fiy, fiz);
    const long long flx = fix64(-fd * crbccd.x * fscale);
    const long long fly = fix64(-fd * crbccd.y * fscale);
    const long long flz = fix64(-fd * crbccd.z * fscale);
    v.add(l, flx, fly, flz);
    const long long fjx = fix64(((fb1 * crabbc.x) - (fb2 * crbccd.x)) * fscale);
    const long long fjy = fix64(((fb1 * crabbc.y) - (fb2 * crbccd.y)) * fscale);
    const long long fjz = fix64(((fb1 * crabbc.z) - (fb2 * crbccd.z)) * fscale);
    v.add(j, fjx, fjy, fjz);
    v.add(kk, -(fix + fjx + flx), -(fiy + fjy + fly), -(fiz + fjz + flz));
  }
  return dp.amp * (1.0 + cos_sangle);
}

// Attenuated 1:4 pair, src/Potential/valence_potential.tpp:1288-1419; with clash damping on,
// the damped potentials of src/Potential/valence_potential.cui:930-1040, whose sigma comes from
// the attenuated coefficients.
template <bool FORCES, bool CLASH, typename V>
__device__ __forceinline__ void eval_14(const V &v, const MMKit &k, bool lj_table, int2 lj,
                                        int i, int l, double inv_scee, double inv_scnb,
                                        double fscale, bool clash_on, double cd, double cratio,
                                        double &ele, double &vdw) {
  const int gi = v.gidx[i], gl = v.gidx[l];
  const Vec3 d = v.disp(i, l);
  const double r2 = dot(d, d);
  const double qiqj = k.q[gi] * k.q[gl] * inv_scee;
  double lja, ljb, sigma_lb = 0.0;
  if (lj_table) {
    const double2 ab = k.ljab14[lj.x + (k.lj_type[gi] * lj.y) + k.lj_type[gl]];
    lja = ab.x * inv_scnb;
    ljb = ab.y * inv_scnb;
  }
  else {
    sigma_lb = 0.5 * (k.ljp1[gi] + k.ljp1[gl]);
    const double sig2 = sigma_lb * sigma_lb;
    const double sig6 = sig2 * sig2 * sig2;
    ljb = k.ljp2[gi] * k.ljp2[gl] * inv_scnb * sig6;
    lja = ljb * sig6;
  }
  double fmag = 0.0;
  if (CLASH && clash_on) {
    ele = 0.0;
    vdw = 0.0;
    const double sigma = (ljb > 1.0e-6) ? (lj_table ? sqrt(cbrt(lja / ljb)) : sigma_lb) : 0.0;
    const double ca = -0.5 / (cd * cd * (cd + 1.0));
    const double cb = (1.0 / cd) - (ca * (cd + 1.0) * (cd + 1.0));
    clash_pair<double, FORCES>(sqrt(r2), qiqj, lja, ljb, sigma, cd, ca, cb, cratio, ele, vdw,
                               fmag);
  }
  else {
    const double invr2 = 1.0 / r2;
    const double invr = sqrt(invr2);
    const double invr4 = invr2 * invr2;
    ele = qiqj * invr;
    vdw = (lja * invr4 * invr4 * invr4) - (ljb * invr4 * invr2);
    if (FORCES) {
      fmag = ((6.0 * ljb) - (12.0 * lja * invr4 * invr2)) * invr4 * invr4;
      fmag -= qiqj * invr * invr2;
    }
  }
  if (FORCES) {
    const long long ix = fix64(fmag * d.x * fscale);
    const long long iy = fix64(fmag * d.y * fscale);
    const long long iz = fix64(fmag * d.z * fscale);
    v.add(i, ix, iy, iz);
    v.add(l, -ix, -iy, -iz);
  }
}

// Single-precision forms of the cosine dihedral and the attenuated 1:4 pair for the
// single-precision model, as the reference evaluates them there (valence_potential.cui:540-640,
// 930-1040 with TCALC = float).  Their energies carry no cancellation (a cosine series and
// pair potentials at 1:4 distances), unlike r - r0 and theta - theta0 of the bonds and angles,
// which stay in double precision.  Guards: asymptotic_to_one_f and
// inverse_one_minus_asymptote_f (src/Constants/symbol_values.h:72-82).
template <bool FORCES, typename V>
__device__ __forceinline__ float eval_dihedral_f(const V &v, int i, int j, int kk, int l,
                                                 const DiheParam &dp, int frc_bits) {
  using P = Prec<float>;
  const Vec3f ab = v.dispf(i, j);
  const Vec3f bc = v.dispf(j, kk);
  const Vec3f cd = v.dispf(kk, l);
  Vec3f crabbc = cross(ab, bc);
  Vec3f crbccd = cross(bc, cd);
  const float inv12 = P::rsqrt(dot(crabbc, crabbc) * dot(crbccd, crbccd));
  const float invbc = P::rsqrt(dot(bc, bc));
  const Vec3f scr = cross(crabbc, crbccd);
  const float cth = dot(crabbc, crbccd) * inv12;
  const float sth = dot(scr, bc) * inv12 * invbc;
  float cn = 1.0f, sn = 0.0f;
  for (int p = 0; p < dp.period; p++) {
    const float t = (cn * cth) - (sn * sth);
    sn = (sn * cth) + (cn * sth);
    cn = t;
  }
  const float cph = static_cast<float>(dp.cos_phase);
  const float sph = static_cast<float>(dp.sin_phase);
  const float amp = static_cast<float>(dp.amp);
  const float cos_sangle = (cn * cph) + (sn * sph);
  if (FORCES) {
    const float sin_sangle = (sn * cph) - (cn * sph);
    const float fr = amp * static_cast<float>(dp.period) * sin_sangle;
    const float invab = P::rsqrt(dot(ab, ab));
    const float invcd = P::rsqrt(dot(cd, cd));
    const float mgab = dot(ab, ab) * invab;
    const float mgbc = dot(bc, bc) * invbc;
    const float cosb = -dot(ab, bc) * invab * invbc;
    const float cosc = -dot(bc, cd) * invbc * invcd;
    constexpr float kAsym = 0.99999904632568359375f;
    constexpr float kInvAsym = 1048576.0f;
    const float isinb2 = (cosb * cosb < kAsym) ? fr * P::rcp(1.0f - (cosb * cosb)) : fr * kInvAsym;
    const float isinc2 = (cosc * cosc < kAsym) ? fr * P::rcp(1.0f - (cosc * cosc)) : fr * kInvAsym;
    const float invabc = invab * invbc;
    const float invbcd = invbc * invcd;
    crabbc = {crabbc.x * invabc, crabbc.y * invabc, crabbc.z * invabc};
    crbccd = {crbccd.x * invbcd, crbccd.y * invbcd, crbccd.z * invbcd};
    const float fa = -invab * isinb2;
    const float fb1 = (mgbc - (mgab * cosb)) * invabc * isinb2;
    const float fb2 = cosc * invbc * isinc2;
    const float fd = -invcd * isinc2;
    const long long fix = fixed_contrib(crabbc.x * fa, frc_bits);
    const long long fiy = fixed_contrib(crabbc.y * fa, frc_bits);
    const long long fiz = fixed_contrib(crabbc.z * fa, frc_bits);
    v.add(i, fix, fiy, fiz);
    const long long flx = fixed_contrib(-fd * crbccd.x, frc_bits);
    const long long fly = fixed_contrib(-fd * crbccd.y, frc_bits);
    const long long flz = fixed_contrib(-fd * crbccd.z, frc_bits);
    v.add(l, flx, fly, flz);
    const long long fjx = fixed_contrib((fb1 * crabbc.x) - (fb2 * crbccd.x), frc_bits);
    const long long fjy = fixed_contrib((fb1 * crabbc.y) - (fb2 * crbccd.y), frc_bits);
    const long long fjz = fixed_contrib((fb1 * crabbc.z) - (fb2 * crbccd.z), frc_bits);
    v.add(j, fjx, fjy, fjz);
    v.add(kk, -(fix + fjx + flx), -(fiy + fjy + fly), -(fiz + fjz + flz));
  }
  return amp * (1.0f + cos_sangle);
}

template <bool FORCES, bool CLASH, typename V>
__device__ __forceinline__ void eval_14_f(const V &v, const MMKit &k, bool lj_table, int2 lj,
                                          int i, int l, float inv_scee, float inv_scnb,
                                          int frc_bits, bool clash_on, float cd, float cratio,
                                          float &ele, float &vdw) {
  using P = Prec<float>;
  const int gi = v.gidx[i], gl = v.gidx[l];
  const Vec3f d = v.dispf(i, l);
  const float r2 = dot(d, d);
  const float qiqj = static_cast<float>(k.q[gi] * k.q[gl]) * inv_scee;
  float lja, ljb, sigma_lb = 0.0f;
  if (lj_table) {
    const double2 ab = k.ljab14[lj.x + (k.lj_type[gi] * lj.y) + k.lj_type[gl]];
    lja = static_cast<float>(ab.x) * inv_scnb;
    ljb = static_cast<float>(ab.y) * inv_scnb;
  }
  else {
    sigma_lb = 0.5f * static_cast<float>(k.ljp1[gi] + k.ljp1[gl]);
    const float sig2 = sigma_lb * sigma_lb;
    const float sig6 = sig2 * sig2 * sig2;
    ljb = static_cast<float>(k.ljp2[gi] * k.ljp2[gl]) * inv_scnb * sig6;
    lja = ljb * sig6;
  }
  float fmag = 0.0f;
  if (CLASH && clash_on) {
    ele = 0.0f;
    vdw = 0.0f;
    const float sigma = (ljb > 1.0e-6f) ? (lj_table ? P::sqrt(P::cbrt(lja / ljb)) : sigma_lb)
                                        : 0.0f;
    const float ca = -0.5f / (cd * cd * (cd + 1.0f));
    const float cb = (1.0f / cd) - (ca * (cd + 1.0f) * (cd + 1.0f));
    clash_pair<float, FORCES>(P::sqrt(r2), qiqj, lja, ljb, sigma, cd, ca, cb, cratio, ele, vdw,
                              fmag);
  }
  else {
    const float invr = P::rsqrt(r2);
    const float invr2 = invr * invr;
    const float invr4 = invr2 * invr2;
    ele = qiqj * invr;
    vdw = (lja * invr4 * invr4 * invr4) - (ljb * invr4 * invr2);
    if (FORCES) {
      fmag = ((6.0f * ljb) - (12.0f * lja * invr4 * invr2)) * invr4 * invr4;
      fmag -= qiqj * invr * invr2;
    }
  }
  if (FORCES) {
    const long long ix = fixed_contrib(fmag * d.x, frc_bits);
    const long long iy = fixed_contrib(fmag * d.y, frc_bits);
    const long long iz = fixed_contrib(fmag * d.z, frc_bits);
    v.add(i, ix, iy, iz);
    v.add(l, -ix, -iy, -iz);
  }
}

// ------------------------------------------------------------------------------------------
// Flat-bottom restraints, src/Restraints/restraint_util.tpp:8-77 and
// src/Potential/valence_potential.tpp:1555-2088 (non-periodic systems: no imaging), in double
// precision like the other valence terms.
// ------------------------------------------------------------------------------------------
// Weights of a restraint's initial and final parameters at `step`.
__device__ __forceinline__ double2 restraint_mixture(int step, int init_step, int final_step) {
  if (step < init_step) {
    return make_double2(0.0, 0.0);
  }
  if (init_step == final_step) {
    return make_double2(1.0, 0.0);
  }
  if (step < final_step) {
    const double wslide = static_cast<double>(step - init_step) /
                          static_cast<double>(final_step - init_step);
    return make_double2(1.0 - wslide, wslide);
  }
  return make_double2(0.0, 1.0);
}

// Stiffness, displacement beyond the flat bottom and penalty at coordinate value dr.
__device__ __forceinline__ double3 restraint_delta(const stormm_restraint &t, double2 w,
                                                   double dr) {
  const double r1 = (w.x * t.init_r[0]) + (w.y * t.final_r[0]);
  const double r2 = (w.x * t.init_r[1]) + (w.y * t.final_r[1]);
  const double r3 = (w.x * t.init_r[2]) + (w.y * t.final_r[2]);
  const double r4 = (w.x * t.init_r[3]) + (w.y * t.final_r[3]);
  const double k2 = (w.x * t.init_k[0]) + (w.y * t.final_k[0]);
  const double k3 = (w.x * t.init_k[1]) + (w.y * t.final_k[1]);
  if (dr < r1) {
    const double dl = r1 - r2;
    return make_double3(k2, dl, k2 * ((dl * dl) + (2.0 * dl * (dr - r1))));
  }
  if (dr < r2) {
    const double dl = dr - r2;
    return make_double3(k2, dl, k2 * dl * dl);
  }
  if (dr < r3) {
    return make_double3(0.0, 0.0, 0.0);
  }
  if (dr < r4) {
    const double dl = dr - r3;
    return make_double3(k3, dl, k3 * dl * dl);
  }
  const double dl = r4 - r3;
  return make_double3(k3, dl, k3 * ((dl * dl) + (2.0 * dl * (dr - r4))));
}

// Minimum image of an angle over 2 pi, src/Structure/local_arrangement.tpp:42-58.
__device__ __forceinline__ double image_angle(double x) {
  constexpr double kTwoPi = 6.283185307179586476925286766559;
  double xf = x / kTwoPi;
  xf -= ((xf >= 0.5) ? ceil(xf - 0.5) : 0.0) + ((xf < -0.5) ? floor(xf + 0.5) : 0.0);
  return (xf - ((xf >= 0.5) ? 1.0 : 0.0)) * kTwoPi;
}

// One restraint of the system at LDS base `base`; returns its penalty.
template <bool FORCES, typename V>
__device__ __forceinline__ double eval_restraint(const V &v, const stormm_restraint &t, int base,
                                 const long long *org, double inv_gpos, int step,
                                 double fscale) {
  const double2 w = restraint_mixture(step, t.init_step, t.final_step);
  const int i = base + t.atoms[0], j = base + t.atoms[1];
  const int kk = base + t.atoms[2], l = base + t.atoms[3];
  if (t.kind == STORMM_RESTRAINT_POSITION) {
    const Vec3 p = v.absolute(i, org, inv_gpos);
    const Vec3 d = {p.x - ((w.x * t.init_target[0]) + (w.y * t.final_target[0])),
                    p.y - ((w.x * t.init_target[1]) + (w.y * t.final_target[1])),
                    p.z - ((w.x * t.init_target[2]) + (w.y * t.final_target[2]))};
    const double dr = sqrt(dot(d, d));
    const double3 e = restraint_delta(t, w, dr);
    if (FORCES) {
      if (dr < 1.0e-10) {
        // On the target: split the force among the three axes (valence_potential.tpp:1610-1626).
        const long long f = fix64(2.0 * e.x * e.y / sqrt(3.0) * fscale);
        v.add(i, -f, -f, -f);
      }
      else {
        const double fmag = 2.0 * e.x * e.y / dr;
        v.add(i, -fix64(fmag * d.x * fscale), -fix64(fmag * d.y * fscale),
              -fix64(fmag * d.z * fscale));
      }
    }
    return e.z;
  }
  if (t.kind == STORMM_RESTRAINT_DISTANCE) {
    const Vec3 d = v.disp(i, j);
    const double dr = sqrt(dot(d, d));
    const double3 e = restraint_delta(t, w, dr);
    if (FORCES) {
      const double fmag = 2.0 * e.x * e.y / dr;
      const long long fx = fix64(fmag * d.x * fscale);
      const long long fy = fix64(fmag * d.y * fscale);
      const long long fz = fix64(fmag * d.z * fscale);
      v.add(i, fx, fy, fz);
      v.add(j, -fx, -fy, -fz);
    }
    return e.z;
  }
  if (t.kind == STORMM_RESTRAINT_ANGLE) {
    const Vec3 ba = v.disp(j, i);
    const Vec3 bc = v.disp(j, kk);
    const double mgba = dot(ba, ba);
    const double mgbc = dot(bc, bc);
    const double invbabc = 1.0 / sqrt(mgba * mgbc);
    double costheta = dot(ba, bc) * invbabc;
    costheta = (costheta < -1.0) ? -1.0 : ((costheta > 1.0) ? 1.0 : costheta);
    const double3 e = restraint_delta(t, w, acos(costheta));
    if (FORCES) {
      const double dA = -2.0 * e.x * e.y / sqrt(1.0 - (costheta * costheta));
      const double sqba = dA / mgba;
      const double sqbc = dA / mgbc;
      const double mbabc = dA * invbabc;
      const long long iax = fix64(((bc.x * mbabc) - (costheta * ba.x * sqba)) * fscale);
      const long long iay = fix64(((bc.y * mbabc) - (costheta * ba.y * sqba)) * fscale);
      const long long iaz = fix64(((bc.z * mbabc) - (costheta * ba.z * sqba)) * fscale);
      const long long icx = fix64(((ba.x * mbabc) - (costheta * bc.x * sqbc)) * fscale);
      const long long icy = fix64(((ba.y * mbabc) - (costheta * bc.y * sqbc)) * fscale);
      const long long icz = fix64(((ba.z * mbabc) - (costheta * bc.z * sqbc)) * fscale);
      v.add(i, -iax, -iay, -iaz);
      v.add(j, iax + icx, iay + icy, iaz + icz);
      v.add(kk, -icx, -icy, -icz);
    }
    return e.z;
  }
  // Dihedral: the signed angle from the plane normals, imaged to the restraint's centre.
  const Vec3 ab = v.disp(i, j);
  const Vec3 bc = v.disp(j, kk);
  const Vec3 cd = v.disp(kk, l);
  Vec3 crabbc = cross(ab, bc);
  Vec3 crbccd = cross(bc, cd);
  double costheta = dot(crabbc, crbccd) / sqrt(dot(crabbc, crabbc) * dot(crbccd, crbccd));
  const Vec3 scr = cross(crabbc, crbccd);
  costheta = (costheta < -1.0) ? -1.0 : ((costheta > 1.0) ? 1.0 : costheta);
  double theta = (dot(scr, bc) > 0.0) ? acos(costheta) : -acos(costheta);
  const double midpoint = 0.5 * ((w.x * (t.init_r[1] + t.init_r[2])) +
                                 (w.y * (t.final_r[1] + t.final_r[2])));
  theta += image_angle(theta - midpoint) - (theta - midpoint);
  const double3 e = restraint_delta(t, w, theta);
  if (FORCES) {
    const double fr = -2.0 * e.x * e.y;
    const double mgab = sqrt(dot(ab, ab));
    const double mgbc = sqrt(dot(bc, bc));
    const double mgcd = sqrt(dot(cd, cd));
    const double invab = 1.0 / mgab;
    const double invbc = 1.0 / mgbc;
    const double invcd = 1.0 / mgcd;
    const double cosb = -dot(ab, bc) * invab * invbc;
    const double cosc = -dot(bc, cd) * invbc * invcd;
    // src/Constants/symbol_values.h:72-82 (asymptotic_to_one_lf, inverse_one_minus_asymptote)
    const double isinb2 = (cosb * cosb < 0.99999904632568359375) ? fr / (1.0 - (cosb * cosb)) :
                                                                   fr * 1048576.0;
    const double isinc2 = (cosc * cosc < 0.99999904632568359375) ? fr / (1.0 - (cosc * cosc)) :
                                                                   fr * 1048576.0;
    const double invabc = invab * invbc;
    const double invbcd = invbc * invcd;
    crabbc = {crabbc.x * invabc, crabbc.y * invabc, crabbc.z * invabc};
    crbccd = {crbccd.x * invbcd, crbccd.y * invbcd, crbccd.z * invbcd};
    const double fa = -invab * isinb2;
    const double fb1 = (mgbc - (mgab * cosb)) * invabc * isinb2;
    const double fb2 = cosc * invbc * isinc2;
    const double fd = -invcd * isinc2;
    const long long fix = fix64(crabbc.x * fa * fscale);
    const long long fiy = fix64(crabbc.y * fa * fscale);
    const long long fiz = fix64(crabbc.z * fa * fscale);
    const long long flx = fix64(-fd * crbccd.x * fscale);
    const long long fly = fix64(-fd * crbccd.y * fscale);
    const long long flz = fix64(-fd * crbccd.z * fscale);
    const long long fjx = fix64(((fb1 * crabbc.x) - (fb2 * crbccd.x)) * fscale);
    const long long fjy = fix64(((fb1 * crabbc.y) - (fb2 * crbccd.y)) * fscale);
    const long long fjz = fix64(((fb1 * crabbc.z) - (fb2 * crbccd.z)) * fscale);
    v.add(i, fix, fiy, fiz);
    v.add(l, flx, fly, flz);
    v.add(j, fjx, fjy, fjz);
    v.add(kk, -(fix + fjx + flx), -(fiy + fjy + fly), -(fiz + fjz + flz));
  }
  return e.z;
}

// Valence term t of the work unit (nothing when t is past the unit's last term).  A kind's
// parameters lie in term order, so they are fetched together with the term's atoms.
template <typename T, bool FORCES, bool CLASH>
__device__ __forceinline__ void valence_term(StageCtx<T> &c, const MMKit &k, int kind, int t) {
  const int n = c.wu.sys_count;
  const int count = (kind == kVBond) ? c.wu.bond_count :
                    (kind == kVAngle) ? c.wu.angl_count :
                                        c.wu.term_count - c.wu.bond_count - c.wu.angl_count;
  if (t >= count) {
    return;
  }
  const double fscale = ldexp(1.0, k.frc_bits);
  const double nrg_scale = ldexp(1.0, k.nrg_bits);
  const ValenceCtxT<T> v(c);
  // The system's terms of this kind, in its template's bonds / angles / dihedrals order.
  const int slot = (kind == kVBond) ? find_slot<&WuSys::bond_pre>(c.L.sys, n, t) :
                   (kind == kVAngle) ? find_slot<&WuSys::angl_pre>(c.L.sys, n, t) :
                                       find_slot<&WuSys::dihe_pre>(c.L.sys, n, t);
  const WuSys &ws = c.L.sys[slot];
  const int local = t - ((kind == kVBond) ? ws.bond_pre :
                         (kind == kVAngle) ? ws.angl_pre : ws.dihe_pre);
  const int kind_first = (kind == kVBond) ? 0 :
                         (kind == kVAngle) ? ws.bond_count : ws.bond_count + ws.angl_count;
  const int par = local + ((kind == kVBond) ? ws.bond_par :
                           (kind == kVAngle) ? ws.angl_par : ws.dihe_par);
  const int4 vt = k.vterms[ws.term_first + kind_first + local];
  const int i = ws.lds_base + (vt.y & 0xffff), j = ws.lds_base + (vt.y >> 16);
  const int kk = ws.lds_base + (vt.z & 0xffff), l = ws.lds_base + (vt.z >> 16);
  long long *nrg = &c.L.nrg[slot * 16];
  if (kind == kVBond) {
    const double2 p = k.bond_par[par];
    lds_add(&nrg[kBond], fix64(eval_bond<FORCES>(v, i, j, p.x, p.y, fscale) * nrg_scale));
  }
  else if (kind == kVAngle) {
    const double2 p = k.angl_par[par];
    lds_add(&nrg[kAngle], fix64(eval_angle<FORCES>(v, i, j, kk, p.x, p.y, fscale) * nrg_scale));
  }
  else if (std::is_same<T, float>::value) {
    const DiheParam p = k.dihe_par[par];
    const float e = eval_dihedral_f<FORCES>(v, i, j, kk, l, p, k.frc_bits);
    lds_add(&nrg[p.improper ? kImproperDihedral : kProperDihedral],
            fix64(static_cast<double>(e) * nrg_scale));
    const double2 a14 = k.dihe14[par];
    if (a14.x > 0.0) {
      float ele, vdw;
      const bool con = CLASH && (c.L.clash_on[slot] != 0);
      eval_14_f<FORCES, CLASH>(v, k, c.wu.lj_table != 0, make_int2(ws.lj_off, ws.lj_nt), i, l,
                               static_cast<float>(a14.x), static_cast<float>(a14.y), k.frc_bits,
                               con, con ? static_cast<float>(c.L.clash_d[slot]) : 0.0f,
                               con ? static_cast<float>(c.L.clash_r[slot]) : 0.0f, ele, vdw);
      lds_add(&nrg[kElec14], fix64(static_cast<double>(ele) * nrg_scale));
      lds_add(&nrg[kVdw14], fix64(static_cast<double>(vdw) * nrg_scale));
    }
  }
  else {
    const DiheParam p = k.dihe_par[par];
    const double e = eval_dihedral<FORCES>(v, i, j, kk, l, p, fscale);
    lds_add(&nrg[p.improper ? kImproperDihedral : kProperDihedral], fix64(e * nrg_scale));
    const double2 a14 = k.dihe14[par];
    if (a14.x > 0.0) {
      double ele, vdw;
      const bool con = CLASH && (c.L.clash_on[slot] != 0);
      eval_14<FORCES, CLASH>(v, k, c.wu.lj_table != 0, make_int2(ws.lj_off, ws.lj_nt), i, l,
                             a14.x, a14.y, fscale, con,
                             con ? static_cast<double>(c.L.clash_d[slot]) : 0.0,
                             con ? static_cast<double>(c.L.clash_r[slot]) : 0.0, ele, vdw);
      lds_add(&nrg[kElec14], fix64(ele * nrg_scale));
      lds_add(&nrg[kVdw14], fix64(vdw * nrg_scale));
    }
  }
}

// Valence terms on their own (evaluations without pair tiles), in chunks of 64 per wavefront.
template <typename T, bool FORCES, bool CLASH>
__device__ __forceinline__ void stage_valence(StageCtx<T> &c, const MMKit &k) {
  const int lane = c.tid & 63;
  const int chunks = valence_chunks(c);
  for (int item = next_item(c, 2, lane); item < chunks; item = next_item(c, 2, lane)) {
    valence_chunk<T, FORCES, CLASH>(c, k, item, lane);
  }
  __syncthreads();
}

// Restraints of the unit's systems, one thread each, in a stage of their own so that their
// double-precision code stays out of the register budget of the tile loops.
template <typename T, bool FORCES>
__device__ __forceinline__ void stage_restraints(StageCtx<T> &c, const MMKit &k) {
  const double fscale = ldexp(1.0, k.frc_bits);
  const double nrg_scale = ldexp(1.0, k.nrg_bits);
  const double inv_gpos = ldexp(1.0, -(k.gpos_bits - c.org_shift));
  const ValenceCtxT<T> v(c);
  for (int r = c.tid; r < c.wu.rst_count; r += c.nthr) {
    int slot = 0, u = r;
    while (u >= c.L.sys[slot].rst_count) {
      u -= c.L.sys[slot].rst_count;
      slot++;
    }
    const WuSys &ws = c.L.sys[slot];
    const int step = (k.rst_step_sys != nullptr) ?
                         minimizer_step(k.rst_step_sys[ws.sys_index] + k.rst_cycle_offset,
                                        k.rst_move, k.rst_clash_cycles) :
                         c.rst_step;
    const double e = eval_restraint<FORCES>(v, k.rst[ws.rst_first + u], ws.lds_base,
                                            &c.L.org[3 * slot], inv_gpos, step, fscale);
    lds_add(&c.L.nrg[slot * 16 + kRestraint], fix64(e * nrg_scale));
  }
  __syncthreads();
}

// The pair stage for the unit's Lennard-Jones form and solvent.
template <typename T, bool FORCES, bool CLASH>
__device__ __forceinline__ void evaluate_pairs(StageCtx<T> &c, const MMKit &k) {
  if (c.wu.lj_table != 0) {
    if (c.gb) {
      stage_pairs<T, FORCES, true, true, CLASH>(c, k);
    }
    else {
      stage_pairs<T, FORCES, true, false, CLASH>(c, k);
    }
  }
  else if (c.gb) {
    stage_pairs<T, FORCES, false, true, CLASH>(c, k);
  }
  else {
    stage_pairs<T, FORCES, false, false, CLASH>(c, k);
  }
}

// ------------------------------------------------------------------------------------------
// One evaluation of the selected terms on the coordinates currently in global memory, leaving
// forces (FORCES) and energies in the LDS accumulators.  RESTRAINTS = false leaves the restraint
// stage out of the instantiation (for callers that never see restrained work units).
template <typename T, bool FORCES, bool CLASH, bool RESTRAINTS = true>
__device__ __forceinline__ void evaluate_wu(StageCtx<T> &c, const MMKit &k, int terms) {
  stage_load<T, CLASH>(c, k);
  // With GB the valence terms ride along with the Born-integral tiles.
  const bool val = (terms & kTermValence) != 0;
  if (c.gb) {
    stage_psi<T, FORCES, CLASH>(c, k, val ? valence_chunks(c) : 0);
    stage_radii<T, FORCES>(c, k, 0.0);
  }
  if (terms & kTermNonbonded) {
    evaluate_pairs<T, FORCES, CLASH>(c, k);
  }
  if (FORCES && c.gb) {
    stage_chain<T>(c, k);
    stage_deriv<T>(c, k);
  }
  if (val && !c.gb) {
    stage_valence<T, FORCES, CLASH>(c, k);
  }
  if (RESTRAINTS && val && c.wu.rst_count > 0) {
    stage_restraints<T, FORCES>(c, k);
  }
}

// ------------------------------------------------------------------------------------------
// Results out: forces added to the global fixed-precision arrays (one owning block per atom)
// and energies added to the ScoreCard rows of the block's systems.
template <typename T, bool FORCES>
__device__ __forceinline__ void stage_store(StageCtx<T> &c, const MMKit &k, bool eval_energy) {
  WuLds<T> &L = c.L;
  if (FORCES && k.xfrc_ovrf != nullptr) {
    // 95-bit forces: the LDS sums scaled to the stored precision, added to (or replacing) the
    // stored values and split into word and overflow word.
    long long *frc[3] = {k.xfrc, k.yfrc, k.zfrc};
    int *ovr[3] = {k.xfrc_ovrf, k.yfrc_ovrf, k.zfrc_ovrf};
    for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
      const int g = L.gidx[a];
      if (g >= 0) {
        const long long sum[3] = {L.atom[a].fx, L.atom[a].fy, L.atom[a].fz};
        for (int d = 0; d < 3; d++) {
          __int128 v = static_cast<__int128>(sum[d]) << k.frc_store_shift;
          if (!k.store_overwrite) {
            v += i95_value(frc[d][g], ovr[d][g]);
          }
          i95_split(v, &frc[d][g], &ovr[d][g]);
        }
      }
    }
  }
  else if (FORCES) {
    for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
      const int g = L.gidx[a];
      if (g >= 0) {
        if (k.store_overwrite) {
          k.xfrc[g] = L.atom[a].fx;
          k.yfrc[g] = L.atom[a].fy;
          k.zfrc[g] = L.atom[a].fz;
        }
        else {
          k.xfrc[g] += L.atom[a].fx;
          k.yfrc[g] += L.atom[a].fy;
          k.zfrc[g] += L.atom[a].fz;
        }
      }
    }
  }
  if (eval_energy) {
    for (int e = c.tid; e < c.wu.sys_count * kNrgSlots; e += c.nthr) {
      const int s = e / kNrgSlots;
      const int comp = e - (s * kNrgSlots);
      const long long v = L.nrg[s * 16 + comp];
      long long *dst = &k.scorecard[(static_cast<size_t>(L.sys[s].sys_index) * kScoreStride) +
                                    comp];
      if (k.store_overwrite) {
        *dst = v;
      }
      else if (v != 0) {
        *dst += v;
      }
    }
  }
}

}  // namespace stormm_amd
