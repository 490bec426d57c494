// Evaluation in parts: several blocks share one work unit where the units are fewer than the
// compute units and a unit is large (the conformers of one large molecule, the tail of a serving
// pool).  One block per unit then leaves most of the device idle: 24 systems of 487 atoms kept 24
// of 256 compute units busy.  The unit's Born radii need the sums of all its parts, and so do the
// radius derivatives, so the evaluation runs as two or three launches (Born-radius integrals;
// valence, radii and pairs; derivative forces) that pass those sums through per-atom arrays in
// device memory.  All sums are fixed-precision integers, so results equal one block's bit for bit.
// Measured against one block of 1024 threads per unit: an evaluation of 24 systems of 487 atoms
// 161 -> 60 us with its fills (15, 27 and 17 us for the three launches; in double precision and
// without the fills 234 -> 58 us), 20 served cycles of 160 systems of
// 16-416 atoms 21.1 -> 17.1 ms.  Below about 250 atoms the two extra launches and set-ups cost
// more than the idle compute units (33 systems of 149 atoms: 61 us against 50).
#include <algorithm>

#include "mm_eval.h"
#include "kernels.h"

namespace stormm_amd {

__device__ __forceinline__ void global_add(long long *addr, long long v) {
  if (v != 0) {
    atomicAdd(reinterpret_cast<unsigned long long *>(addr), static_cast<unsigned long long>(v));
  }
}

// True in every thread when all systems of the unit have stopped (k.done).  Its coordinates no
// longer change, so its forces and ScoreCard rows already hold what the evaluation would write
// and its integrals are zero: the block returns, as k_min_cycle's does.
__device__ __forceinline__ bool unit_stopped(const MMKit &k, int unit) {
  if (k.done == nullptr) {
    return false;
  }
  const WuDesc &wu = k.wu[unit];
  const int tid = static_cast<int>(threadIdx.x);
  const bool runs = tid < wu.sys_count && k.done[k.wu_sys[wu.sys_first + tid].sys_index] == 0;
  return __syncthreads_or(runs ? 1 : 0) == 0;
}

// This part's force and energy sums added to the global arrays.
template <typename T, bool FORCES>
__device__ __forceinline__ void part_store(StageCtx<T> &c, const MMKit &k, bool eval_energy) {
  WuLds<T> &L = c.L;
  if (FORCES) {
    for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
      const int g = L.gidx[a];
      if (g >= 0) {
        global_add(&k.xfrc[g], L.atom[a].fx);
        global_add(&k.yfrc[g], L.atom[a].fy);
        global_add(&k.zfrc[g], L.atom[a].fz);
      }
    }
  }
  if (eval_energy) {
    for (int e = c.tid; e < c.wu.sys_count * kNrgSlots; e += c.nthr) {
      const int s = e / kNrgSlots;
      const int comp = e - (s * kNrgSlots);
      global_add(&k.scorecard[(static_cast<size_t>(L.sys[s].sys_index) * kScoreStride) + comp],
                 L.nrg[s * 16 + comp]);
    }
  }
}

// Phase 0, Born-radius integrals: this part's share of the tiles, added to part_psi.  A unit's
// first part also clears what the later phases add to: dE/dR, and, when the launch overwrites,
// the forces and energies (this phase adds to neither).
template <typename T, bool FORCES>
__global__ void __launch_bounds__((EvalBlockLimit<T, false>::value))
    k_part_psi(MMKit k, int terms, int eval_energy) {
  extern __shared__ __align__(16) unsigned char smem[];
  StageCtx<T> c(smem, k.maxa, static_cast<int>(blockDim.x >> 6));
  const WuPart wp = k.parts[blockIdx.x];
  if (unit_stopped(k, wp.unit)) {
    return;
  }
  init_ctx<T>(c, k, wp.unit, terms);
  c.part = wp.part;
  c.parts = wp.parts;
  stage_load<T, false, kPartPsi>(c, k);
  WuLds<T> &L = c.L;
  if (c.part == 0) {
    for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
      const int g = L.gidx[a];
      if (FORCES && g >= 0) {
        if (c.gb) {
          k.part_dedr[g] = 0;
        }
        if (k.store_overwrite) {
          k.xfrc[g] = 0;
          k.yfrc[g] = 0;
          k.zfrc[g] = 0;
        }
      }
    }
    if (k.store_overwrite && eval_energy) {
      for (int e = c.tid; e < c.wu.sys_count * kNrgSlots; e += c.nthr) {
        const int s = e / kNrgSlots;
        k.scorecard[(static_cast<size_t>(L.sys[s].sys_index) * kScoreStride) +
                    (e - (s * kNrgSlots))] = 0;
      }
    }
  }
  if (!c.gb) {
    return;
  }
  stage_psi<T, false, false>(c, k, 0);
  for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
    if (L.gidx[a] >= 0) {
      global_add(&k.part_psi[L.gidx[a]], L.atom[a].psi);
    }
  }
}

// Phase 1: radii from the summed integrals (every part; the first adds the self terms and keeps
// dR/dpsi), this part's share of the valence terms and pairs; the first part takes the restraints.
template <typename T, bool FORCES, bool CLASH>
__global__ void __launch_bounds__((EvalBlockLimit<T, FORCES && CLASH>::value))
    k_part_pairs(MMKit k, int terms, int eval_energy) {
  extern __shared__ __align__(16) unsigned char smem[];
  StageCtx<T> c(smem, k.maxa, static_cast<int>(blockDim.x >> 6));
  const WuPart wp = k.parts[blockIdx.x];
  if (unit_stopped(k, wp.unit)) {
    return;
  }
  init_ctx<T>(c, k, wp.unit, terms);
  c.part = wp.part;
  c.parts = wp.parts;
  stage_load<T, CLASH, kPartPairs>(c, k);
  WuLds<T> &L = c.L;
  if (c.gb) {
    stage_radii<T, FORCES>(c, k, 0.0);
    if (FORCES && c.part == 0 && k.igb != 1) {
      for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
        if (L.gidx[a] >= 0) {
          k.part_drdpsi[L.gidx[a]] = __longlong_as_double(L.atom[a].psi);
        }
      }
    }
  }
  if (terms & kTermValence) {
    if (c.part == 0 && c.wu.rst_count > 0) {
      stage_restraints<T, FORCES>(c, k);
    }
    // The valence chunks go to the block's last wavefronts, the tile tasks to its first ones (a
    // share is often less than one round of tiles), with no barrier between the two.
    const int waves = c.nthr >> 6;
    const int chunks = valence_chunks(c);
    const int wave = __builtin_amdgcn_readfirstlane(c.tid >> 6);
    for (int i = c.part + (c.parts * (waves - 1 - wave)); i < chunks; i += c.parts * waves) {
      valence_chunk<T, FORCES, CLASH>(c, k, i, c.tid & 63);
    }
  }
  evaluate_pairs<T, FORCES, CLASH>(c, k);
  part_store<T, FORCES>(c, k, eval_energy != 0);
  if (FORCES && c.gb) {
    for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
      if (L.gidx[a] >= 0) {
        global_add(&k.part_dedr[L.gidx[a]], L.atom[a].dedr);
      }
    }
  }
}

// Phase 2: this part's share of the derivative forces.  The first part returns the Born-radius
// integrals, which no phase reads any more, to zero for the next evaluation.
template <typename T>
__global__ void __launch_bounds__((EvalBlockLimit<T, false>::value))
    k_part_deriv(MMKit k, int terms) {
  extern __shared__ __align__(16) unsigned char smem[];
  StageCtx<T> c(smem, k.maxa, static_cast<int>(blockDim.x >> 6));
  const WuPart wp = k.parts[blockIdx.x];
  if (unit_stopped(k, wp.unit)) {
    return;
  }
  init_ctx<T>(c, k, wp.unit, terms);
  c.part = wp.part;
  c.parts = wp.parts;
  stage_load<T, false, kPartDeriv>(c, k);
  if (c.part == 0) {
    for (int a = c.tid; a < c.wu.lds_atoms; a += c.nthr) {
      if (c.L.gidx[a] >= 0) {
        k.part_psi[c.L.gidx[a]] = 0;
      }
    }
  }
  stage_chain<T>(c, k);
  stage_deriv<T>(c, k);
  part_store<T, true>(c, k, false);
}

template <typename T, bool HEAVY = false, typename F, typename... Args>
static hipError_t launch_parts(F fn, const MMKit &k, hipStream_t stream, Args... args) {
  const int block = eval_block<T, HEAVY>(k, k.nparts);
  const size_t lds = WuLds<T>::bytes(k.maxa, block / 64);
  const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void *>(fn),
                                             hipFuncAttributeMaxDynamicSharedMemorySize,
                                             static_cast<int>(lds));
  if (err != hipSuccess) {
    return err;
  }
  hipLaunchKernelGGL(fn, dim3(k.nparts), dim3(block), lds, stream, k, args...);
  return hipGetLastError();
}

template <typename T>
static hipError_t launch_mm_parts_t(const MMKit &k, int terms, bool force, int eval_energy,
                                    hipStream_t stream) {
  const bool gb = (k.igb != 0) && (terms & kTermNonbonded) != 0;
  const bool clash = (k.clash_variant != 0);
  hipError_t err = hipSuccess;
  if (gb || k.store_overwrite) {
    err = launch_parts<T>(force ? k_part_psi<T, true> : k_part_psi<T, false>, k, stream, terms,
                          eval_energy);
  }
  if (err == hipSuccess) {
    err = (force && clash)
              ? launch_parts<T, true>(k_part_pairs<T, true, true>, k, stream, terms, eval_energy)
              : launch_parts<T>(force ? k_part_pairs<T, true, false>
                                      : clash ? k_part_pairs<T, false, true>
                                              : k_part_pairs<T, false, false>,
                                k, stream, terms, eval_energy);
  }
  if (err == hipSuccess && gb && force) {
    err = launch_parts<T>(k_part_deriv<T>, k, stream, terms);
  }
  return err;
}

hipError_t launch_mm_parts(int precision, const MMKit &k, int terms, int eval_force,
                           int eval_energy, hipStream_t stream) {
  return (precision == 0)
             ? launch_mm_parts_t<double>(k, terms, eval_force != 0, eval_energy, stream)
             : launch_mm_parts_t<float>(k, terms, eval_force != 0, eval_energy, stream);
}

}  // namespace stormm_amd
