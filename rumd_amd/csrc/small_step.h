// One kernel per step for small samples: the list check and, when due, the
// list build, the pair forces, the leapfrog / Nose-Hoover update and the
// previous step's thermostat update, over an N2 list or over all pairs.
//
// Reference: one pass of the run loop, sample.CalcF then itg.Integrate
// (Python/rumd/Simulation.py:583-597), with calculateNBL_N2
// (src/NeighborList.cu:1001-1099), Calcf_NBL_tp (src/PairPotential.cu:350-515),
// integrateNVTAlgorithm and updateNVTThermostatState
// (src/IntegratorNVT.cu:364-437).
//
// A small sample's step is bound by launches and by the chain of dependent
// reads, not by work: four kernels (build, forces, integrator, thermostat) took
// 13 us a step at n = 500 without a list, 18 at n = 1000 and 19 at n = 4099,
// most of it between them; one takes 7.5, 8.4 and 12 (rebuilds included).  The
// host class takes it over N2 lists of at most 5,000 particles: above, the
// build's O(n^2) scan is the step's time and the four kernels' build is faster
// at it.
// None of the four needs a grid-wide barrier inside a step:
//  - a list of the N2 method belongs to one particle and is built from the
//    positions alone, so the workgroup that owns the particle rebuilds it when
//    a rebuild is due and goes on to its forces;
//  - the new positions go to a second array (the others still read the old);
//  - the thermostat's update after step k-1 is a sum of n / 16 partials: every
//    workgroup of step k forms it for itself, in the one fixed order, and the
//    first stores the state for step k+1;
//  - the rebuild request alternates between words, so that one step reads one
//    (no workgroup changes it), sets the next and clears the one before.
// rumdx_small_steps_end, after the last step of a chain, stores the
// thermostat state and the request where the other entry points read them.
//
// 16 particles per workgroup.  An N2 list is spread over 16 lanes, as in
// k_pair_nbl (same order of sums, hence the same bits); all pairs take a wave
// per particle, as in k_pair_all.
#pragma once

#include "force_kernels.h"

namespace rumdx {
namespace {

struct SmallStep {
  const float4* r;
  float4* f;
  float4* w;
  uint32_t* nbl;
  uint32_t* num_nbrs;
  float4* last_r;
  uint32_t* flags;
  const float* cut_skin2;
  const float* params;
  uint32_t nt;
  uint32_t n, nvp, max_nbrs;
  Exclusions ex;
  const uint32_t* request;   // this step's rebuild request (null: no list)
  uint32_t* set_request;     // the next step's
  uint32_t* clear_request;   // the last step's (null in the first step)
  const rumdx_nh_state* nh;  // state before the update that is due (or to use as it is)
  rumdx_nh_state* nh_out;    // where the updated state goes
  const double* partials_in; // the last step's kinetic-energy partials (null: no update due)
  float omega2;
  uint32_t dof;
  NvtFuse fz;                // fz.nh is null with the thermostat off; fz.nb_flags is not used
};

// The update of k_nvt_finish by every thread of the workgroup, from the same
// sums in the same order (sum_partials): threads 0..255 add partials k, k +
// 256, ..., each wave its lanes, and every thread the four waves' totals.
__device__ __forceinline__ rumdx_nh_state thermostat_update(const SmallStep& a, double* s_red) {
  rumdx_nh_state st = *a.nh;
  if (a.partials_in != nullptr) {
    const uint32_t np = (a.n + kSmallGroup - 1u) / kSmallGroup;
    double v = 0.0;
    if (threadIdx.x < kBlock)
      for (uint32_t k = threadIdx.x; k < np; k += kBlock) v += a.partials_in[k];
    v = wave_sum(v);
    if ((threadIdx.x & 63u) == 0 && threadIdx.x < kBlock) s_red[threadIdx.x >> 6] = v;
    __syncthreads();
    double tot = 0.0;
    for (uint32_t k = 0; k < kBlock / 64; ++k) tot += s_red[k];
    nh_advance(st, tot, a.fz.dt, a.omega2, a.dof);
  }
  return st;
}

// Rebuilds the lists of the workgroup's particles (k_build_n2's criterion and
// order): 16 lanes per particle test 16 candidates at a time from positions
// staged in LDS.
constexpr uint32_t kSmallTile = 512;

__device__ __forceinline__ void small_build(const SmallStep& a, const Box& bx, uint32_t i, bool live, float4 ri,
                                            float4* s_r, const float* s_cut) {
  const uint32_t part = threadIdx.x & 15u;
  const float* cut = s_cut + a.nt * __float_as_uint(ri.w);
  const ExclusionRange er = live ? a.ex.of(i) : ExclusionRange{};
  uint32_t cnt = 0;
  for (uint32_t base = 0; base < a.n; base += kSmallTile) {
    __syncthreads();
    for (uint32_t q = threadIdx.x; q < kSmallTile; q += blockDim.x) s_r[q] = a.r[min(base + q, a.n - 1u)];
    __syncthreads();
    const uint32_t m = min(a.n - base, kSmallTile);
    for (uint32_t q0 = 0; q0 < m; q0 += 16u) {
      const uint32_t j = base + q0 + part;
      const float4 rj = s_r[q0 + part];
      bool in = live && j < a.n && j != i && min_image_d2_f32(ri, rj, bx) < cut[__float_as_uint(rj.w)];
      if (in) in = !a.ex.excludes(er, j);
      const uint32_t hit =
          static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(in) >> (threadIdx.x & 48u)) & 0xffffu;
      if (in) {
        const uint32_t k = cnt + static_cast<uint32_t>(__builtin_popcount(hit & ((1u << part) - 1u)));
        if (k < a.max_nbrs) a.nbl[static_cast<size_t>(k) * a.nvp + i] = j;
      }
      cnt += static_cast<uint32_t>(__builtin_popcount(hit));
    }
  }
  if (live && part == 0) {
    a.last_r[i] = ri;
    a.num_nbrs[i] = cnt < a.max_nbrs ? cnt : a.max_nbrs;
    if (cnt >= a.max_nbrs) a.flags[RUMDX_FLAG_OVERFLOW] = 1u;
    if (cnt > __hip_atomic_load(a.flags + RUMDX_FLAG_MAXLEN, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(a.flags + RUMDX_FLAG_MAXLEN, cnt);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.flags[RUMDX_FLAG_BUILDS] += 1u;
    a.flags[RUMDX_FLAG_PRUNE] = 1u;
  }
  __syncthreads();  // the lists are read by other lanes below
}

// WANT: the step's forces, energies and virials are stored; otherwise the next
// step replaces them before anything can read them, and only the update uses
// the forces.
template <class PP, bool ALL, bool WANT>
__global__ __launch_bounds__(ALL ? 1024 : 256) void k_small_step(PP pp, SmallStep a, Box bx) {
  constexpr uint32_t kLg = ALL ? 6u : 4u;
  static_assert((kSmallGroup << kLg) == (ALL ? 1024u : 256u), "16 particles per workgroup");
  extern __shared__ float4 s_dyn[];
  float4* s_r = s_dyn;                      // kSmallTile
  float4* s_tab = s_dyn + kSmallTile;       // kRow nt^2
  float* s_cut = reinterpret_cast<float*>(s_tab + PP::kRow * a.nt * a.nt);  // nt^2 (lists)
  __shared__ float4 s_f[kSmallGroup];
  __shared__ double s_red[kBlock / 64];
  const uint32_t g = threadIdx.x >> kLg, part = threadIdx.x & ((1u << kLg) - 1u);
  const uint32_t i = blockIdx.x * kSmallGroup + g;
  const bool live = i < a.n;
  const bool rebuild = !ALL && *a.request != 0u;
  // the particle this thread will advance, its state read ahead of the forces
  const uint32_t own_i = blockIdx.x * kSmallGroup + threadIdx.x;
  const bool owner = threadIdx.x < kSmallGroup && own_i < a.n;
  NvtIn own{};
  if (owner) {
    own.r = a.r[own_i];
    own.v = a.fz.v[own_i];
    own.lo = a.fz.rlo != nullptr ? a.fz.rlo[own_i] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (!ALL) own.last_r = rebuild ? own.r : a.last_r[own_i];
  }
  const float4 ri = a.r[live ? i : a.n - 1u];
  pp.load_table(s_tab, a.params, a.nt);
  if (rebuild)
    for (uint32_t k = threadIdx.x; k < a.nt * a.nt; k += blockDim.x) s_cut[k] = a.cut_skin2[k];
  float ps = 0.f;
  if (a.fz.nh != nullptr) {
    const rumdx_nh_state st = thermostat_update(a, s_red);
    ps = static_cast<float>(st.ps);
    if (a.nh_out != nullptr && blockIdx.x == 0 && threadIdx.x == 0) *a.nh_out = st;
  }
  __syncthreads();  // the tables
  if (rebuild) small_build(a, bx, i, live, ri, s_r, s_cut);

  const float4* prow = s_tab + PP::kRow * __float_as_uint(ri.w) * a.nt;
  const double xi = ri.x, yi = ri.y, zi = ri.z;
  Acc acc;
  if (ALL) {
    for (uint32_t base = 0; base < a.n; base += kSmallTile) {
      if (base != 0) __syncthreads();
      for (uint32_t q = threadIdx.x; q < kSmallTile && base + q < a.n; q += blockDim.x) s_r[q] = a.r[base + q];
      __syncthreads();
      const uint32_t m = live ? min(a.n - base, kSmallTile) : 0u;
      for (uint32_t q = part; q < m; q += 64u)
        if (base + q != i) pair_term<false>(pp, xi, yi, zi, s_r[q], prow, bx, acc);
    }
  } else if (live) {
    list_forces<false>(pp, i, part, kLg, xi, yi, zi, a.r, a.nbl, a.num_nbrs[i], a.n, a.nvp, a.max_nbrs, prow, bx,
                       a.ex, acc);
  }
  combine_lanes<false>(acc, kLg);
  if (live && part == 0) {
    s_f[g] = make_float4(acc.fx, acc.fy, acc.fz, 0.f);
    if (WANT) store_result<false, true>(i, acc, a.f, a.w, nullptr);
  }
  __syncthreads();
  if (threadIdx.x < kSmallGroup) {
    double ke2 = 0.0;
    if (owner) {
      float4 rn;
      bool moved;
      ke2 = static_cast<double>(nvt_advance(own_i, s_f[threadIdx.x], own, a.fz, ps, bx, rn, moved, !ALL));
      if (!ALL && moved) *a.set_request = 1u;
    }
    if (a.fz.nh != nullptr) {
      const double s = group_sum(ke2);
      if (threadIdx.x == 0) a.fz.partials[blockIdx.x] = s;
    }
  }
  if (!ALL && blockIdx.x == 0 && threadIdx.x == 0 && a.clear_request != nullptr) *a.clear_request = 0u;
}

}  // namespace
}  // namespace rumdx
