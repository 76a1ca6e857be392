// LJ 12-6 pair force / energy / virial (gfx950): the pair policy of
// Pot_IPL_12_6 / Pot_LJ_12_6 and its entry point rumdx_pair_lj.
//
// Reference: Pot_IPL_12_6::ComputeInteraction (include/rumd/PairPotential.h:161-168),
// fij (include/rumd/PairPotential.h:1198-1244).  The pair arithmetic is
// VALU-bound, so the LDS table holds pre-multiplied constants: per type pair
// {rc^2, 12 A12, 6 A6, s(rc) rc}, which a step that wants forces alone reads,
// and {A12, A6, -u(rc), -(u(rc) + s(rc) rc^2)}, the last two being the energy
// shifts of the shifted-potential and shifted-force cut-offs.
#include <type_traits>

#include "force_kernels.h"
#include "small_step.h"

// Waves per SIMD of the 12-6 tile kernel (five fit a 2040-particle halo).
#ifndef RUMDX_TILE_WAVES_PER_EU
#define RUMDX_TILE_WAVES_PER_EU 5
#endif

namespace rumdx {
namespace {

template <int CUT>
struct LjPair {
  static constexpr uint32_t kRow = 2;
  static constexpr int kWavesPerEU = RUMDX_TILE_WAVES_PER_EU;
  static constexpr bool kTunedWaves = true;

  __device__ __forceinline__ void load_table(float4* s_tab, const float* __restrict__ params, uint32_t nt) const {
    for (uint32_t k = threadIdx.x; k < nt * nt; k += blockDim.x) {
      const float* q = params + static_cast<size_t>(k) * RUMDX_NUM_PARAM;
      const float rc = q[0], a12 = q[1], a6 = q[2];
      const float src = q[RUMDX_NUM_PARAM - 2], ucut = q[RUMDX_NUM_PARAM - 1];
      s_tab[2 * k] = make_float4(rc * rc, 12.f * a12, 6.f * a6, src);
      s_tab[2 * k + 1] = make_float4(a12, a6, -ucut, -fmaf(src, rc, ucut));
    }
  }

  // The LJ term of one pair given its displacement (fij with
  // ComputeInteraction inlined): u = A12 r^-12 + A6 r^-6, s = -u'(r)/r,
  // shifted as the cut-off method asks (SP: u - u(rc); SF: s - s(rc) rc/r and
  // u - u(rc) + s(rc) rc (r - rc)).  Branch-free; pairs at or beyond rc are
  // masked.  FINE refines 1/r^2 from the squared rsq by one Newton step (two
  // operations): the seventh power of its error enters the force, and the
  // callers that form displacements in FP64 are not bound by the arithmetic.
  template <bool STR, bool FINE>
  __device__ __forceinline__ void core(float dx, float dy, float dz, float d2, uint32_t tj, const float4* prow,
                                       Acc& a) const {
    const float4 pa = prow[2 * tj];
    const float4 pb = prow[2 * tj + 1];
    // SF needs 1/r anyway: one rsq gives both 1/r and 1/r^2
    float rinv = 0.f, inv2;
    if (CUT == RUMDX_CUTOFF_SF) {
      rinv = __builtin_amdgcn_rsqf(d2);
      inv2 = rinv * rinv;
      if (FINE) inv2 = fmaf(inv2, fmaf(-d2, inv2, 1.f), inv2);
    } else {
      inv2 = __builtin_amdgcn_rcpf(d2);
    }
    const float inv6 = inv2 * inv2 * inv2;
    float s = (inv6 * inv2) * fmaf(pa.y, inv6, pa.z);
    float u;
    if (CUT == RUMDX_CUTOFF_SP) {
      u = fmaf(inv6, fmaf(pb.x, inv6, pb.y), pb.z);
    } else if (CUT == RUMDX_CUTOFF_SF) {
      u = fmaf(inv6, fmaf(pb.x, inv6, pb.y), pb.w);
      s = fmaf(-pa.w, rinv, s);
      u = fmaf(pa.w, d2 * rinv, u);
    } else {
      u = inv6 * fmaf(pb.x, inv6, pb.y);
    }
    const bool in = d2 < pa.x;
    s = in ? s : 0.f;
    u = in ? u : 0.f;
    accumulate<STR>(dx, dy, dz, d2, s, u, a);
  }
};

}  // namespace
}  // namespace rumdx

extern "C" int rumdx_pair_lj(const rumdx_particles* p, const rumdx_nblist* nb, const float* params_dev,
                             uint32_t ntypes, const float box[8], int cutoff_method, int initialize,
                             int calc_stresses, void* stream) {
  using namespace rumdx;
  const char* entry = "rumdx_pair_lj";
  const int rc = check_pair_args(entry, p, nb, params_dev, ntypes, box, calc_stresses);
  if (rc != RUMDX_OK) return rc;
  if (p->n == 0) return RUMDX_OK;
  const Box bx = make_box(box);
  const hipStream_t st = as_stream(stream);
  const bool init = initialize != 0, str = calc_stresses != 0;
  switch (cutoff_method) {
    case RUMDX_CUTOFF_NS:
      return dispatch_pair(LjPair<RUMDX_CUTOFF_NS>{}, entry, p, nb, params_dev, ntypes, bx, init, str, st);
    case RUMDX_CUTOFF_SP:
      return dispatch_pair(LjPair<RUMDX_CUTOFF_SP>{}, entry, p, nb, params_dev, ntypes, bx, init, str, st);
    case RUMDX_CUTOFF_SF:
      return dispatch_pair(LjPair<RUMDX_CUTOFF_SF>{}, entry, p, nb, params_dev, ntypes, bx, init, str, st);
    default: return fail(RUMDX_E_INVALID, "rumdx_pair_lj: invalid cutoff method");
  }
}

// One NVT step of a sample whose only force term is this 12-6 potential over a
// sorted list: the forces at the positions p->r_dev, and in the same kernel
// each particle's leapfrog / Nose-Hoover update with the skin check, the new
// positions going to r_out_dev; then the thermostat update from the per-tile
// kinetic-energy sums.  Per particle the arithmetic is that of rumdx_pair_lj
// followed by rumdx_nvt_step.
namespace rumdx {
namespace {

// The fused step without the thermostat's update; want: energies and virials
// are stored too.
int pair_lj_nvt(const char* entry, const rumdx_particles* p, const rumdx_nblist* nb, const float* params_dev,
                uint32_t ntypes, const float* box, int cutoff_method, float* r_out_dev, const rumdx_nh_state* nh_dev,
                float dt, uint32_t thermostat_on_mask, bool want, void* workspace_dev, void* stream) {
  const std::string e(entry);
  const int rc = check_pair_args(entry, p, nb, params_dev, ntypes, box, 0);
  if (rc != RUMDX_OK) return rc;
  if (nb == nullptr || nb->nbl16_dev == nullptr)
    return fail(RUMDX_E_INVALID, e + ": needs a list of the sorted method");
  if (nb->flags_dev == nullptr || nb->last_r_dev == nullptr)
    return fail(RUMDX_E_INVALID, e + ": neighbour list not allocated");
  if (p->v_dev == nullptr || p->im_dev == nullptr || r_out_dev == nullptr)
    return fail(RUMDX_E_INVALID, e + ": particle arrays not allocated");
  if (r_out_dev == p->r_dev)
    return fail(RUMDX_E_INVALID, e + ": r_out_dev must not alias the positions the forces read");
  if (cutoff_method != RUMDX_CUTOFF_NS && cutoff_method != RUMDX_CUTOFF_SP && cutoff_method != RUMDX_CUTOFF_SF)
    return fail(RUMDX_E_INVALID, e + ": invalid cutoff method");
  const bool thermo = thermostat_on_mask != 0u;
  if (thermo && (nh_dev == nullptr || workspace_dev == nullptr))
    return fail(RUMDX_E_INVALID, e + ": thermostat state and workspace required");
  // one kinetic-energy partial per tile in the workspace's partials
  if (thermo && static_cast<size_t>(nb->ntiles) > Workspace::partial_doubles(p->n))
    return fail(RUMDX_E_INVALID, e + ": more tiles than the workspace holds partials");
  if (p->n == 0) return RUMDX_OK;
  NvtFuse fz{};
  fz.r_out = reinterpret_cast<float4*>(r_out_dev);
  fz.v = reinterpret_cast<float4*>(p->v_dev);
  fz.im = reinterpret_cast<float4*>(p->im_dev);
  fz.rlo = reinterpret_cast<float4*>(p->rlo_dev);
  fz.nh = thermo ? nh_dev : nullptr;
  fz.partials = thermo ? Workspace::partials(workspace_dev) : nullptr;
  fz.last_r = reinterpret_cast<const float4*>(nb->last_r_dev);
  fz.nb_flags = nb->flags_dev;
  fz.skin2_over_4 = static_cast<float>(0.25 * static_cast<double>(nb->skin) * static_cast<double>(nb->skin));
  fz.prune_r = reinterpret_cast<const float4*>(inner_prune_r(nb));
  fz.inner2 = inner_check2(nb);
  fz.dt = dt;
  fz.on_mask = thermostat_on_mask;
  const Box bx = make_box(box);
  const hipStream_t st = as_stream(stream);
  const uint32_t lpp = nb->lanes_per_particle;
  const uint32_t lgp = lpp >= 8u ? 3u : lpp >= 4u ? 2u : lpp >= 2u ? 1u : 0u;
  const auto launch = [&](auto pp) {
    if (want)
      launch_tiles<decltype(pp), false, true, kFuseStore>(pp, p, nb, params_dev, ntypes, bx, lgp, fz, st);
    else
      launch_tiles<decltype(pp), false, true, kFuseInner>(pp, p, nb, params_dev, ntypes, bx, lgp, fz, st);
  };
  switch (cutoff_method) {
    case RUMDX_CUTOFF_NS: launch(LjPair<RUMDX_CUTOFF_NS>{}); break;
    case RUMDX_CUTOFF_SP: launch(LjPair<RUMDX_CUTOFF_SP>{}); break;
    default: launch(LjPair<RUMDX_CUTOFF_SF>{}); break;
  }
  return check_launch(entry);
}

}  // namespace
}  // namespace rumdx

extern "C" int rumdx_pair_lj_nvt_due(const rumdx_particles* p, const rumdx_nblist* nb, const float* params_dev,
                                     uint32_t ntypes, const float box[8], int cutoff_method, float* r_out_dev,
                                     const rumdx_nh_state* nh_dev, float dt, uint32_t thermostat_on_mask,
                                     int store_forces, void* workspace_dev, void* stream) {
  return rumdx::pair_lj_nvt("rumdx_pair_lj_nvt_due", p, nb, params_dev, ntypes, box, cutoff_method, r_out_dev, nh_dev,
                            dt, thermostat_on_mask, store_forces != 0, workspace_dev, stream);
}

extern "C" int rumdx_pair_lj_nvt(const rumdx_particles* p, const rumdx_nblist* nb, const float* params_dev,
                                 uint32_t ntypes, const float box[8], int cutoff_method, float* r_out_dev,
                                 rumdx_nh_state* nh_dev, float dt, uint32_t thermostat_on_mask, float omega2,
                                 uint32_t dof, void* workspace_dev, void* stream) {
  using namespace rumdx;
  const bool thermo = thermostat_on_mask != 0u;
  if (thermo && nh_dev != nullptr && workspace_dev != nullptr && dof == 0)
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_nvt: zero degrees of freedom");
  const int rc = pair_lj_nvt("rumdx_pair_lj_nvt", p, nb, params_dev, ntypes, box, cutoff_method, r_out_dev, nh_dev, dt,
                             thermostat_on_mask, true, workspace_dev, stream);
  if (rc != RUMDX_OK || !thermo || p->n == 0) return rc;
  const rumdx_nh_update due{nh_dev, workspace_dev, nb->ntiles, dof, dt, omega2};
  return rumdx_nvt_finish(&due, stream);
}

namespace rumdx {
namespace {

// The words a chain's rebuild request alternates between: step k reads word
// k, sets word k + 1 and clears word k - 1; word 0 is the list's own flag.
uint32_t* request_word(const rumdx_nblist* nb, uint32_t k) {
  return nb->flags_dev + (k == 0u ? RUMDX_FLAG_REBUILD : RUMDX_FLAG_CHAIN + (k - 1u) % 3u);
}

// End of a chain of m steps: the due thermostat update into nh, and the
// request of the last step where the next list update reads it.
__global__ __launch_bounds__(kBlock) void k_small_end(const double* __restrict__ partials, uint32_t np,
                                                      const rumdx_nh_state* from, rumdx_nh_state* nh, float dt,
                                                      float omega2, uint32_t dof, uint32_t* request,
                                                      uint32_t* last_request, uint32_t* flag) {
  __shared__ double s_red[kBlock / 64];
  if (nh != nullptr) {
    const double tot = sum_partials(partials, np, 1, s_red);
    if (threadIdx.x == 0) {
      rumdx_nh_state st = *from;
      nh_advance(st, tot, dt, omega2, dof);
      *nh = st;
    }
  }
  if (request != nullptr && threadIdx.x == 0) {
    const uint32_t due = *request;
    *last_request = 0u;
    *request = 0u;
    if (due != 0u) *flag = 1u;
  }
}

template <int CUT, bool ALL>
void launch_small(const SmallStep& a, const Box& bx, bool want, hipStream_t st) {
  using PP = LjPair<CUT>;
  const size_t lds = sizeof(float4) * (kSmallTile + PP::kRow * a.nt * a.nt) + sizeof(float) * a.nt * a.nt;
  const dim3 grid((a.n + kSmallGroup - 1u) / kSmallGroup), block(ALL ? 1024 : 256);
  if (want)
    hipLaunchKernelGGL((k_small_step<PP, ALL, true>), grid, block, lds, st, PP{}, a, bx);
  else
    hipLaunchKernelGGL((k_small_step<PP, ALL, false>), grid, block, lds, st, PP{}, a, bx);
}

int check_small(const char* entry, const rumdx_particles* p, const rumdx_nblist* nb, const rumdx_nh_state* nh_dev,
                uint32_t thermostat_on_mask, uint32_t dof, const void* workspace_dev) {
  const std::string e(entry);
  if (p == nullptr || workspace_dev == nullptr) return fail(RUMDX_E_INVALID, e + ": null argument");
  if (p->n > kSmallStepMax) return fail(RUMDX_E_INVALID, e + ": more than RUMDX_SMALL_STEP_MAX particles");
  if (nb != nullptr && (nb->nbl_dev == nullptr || nb->flags_dev == nullptr || nb->last_r_dev == nullptr ||
                        nb->num_nbrs_dev == nullptr || nb->cut_skin2_dev == nullptr))
    return fail(RUMDX_E_INVALID, e + ": needs a list of the N2 method, or none");
  if (thermostat_on_mask != 0u && nh_dev == nullptr) return fail(RUMDX_E_INVALID, e + ": thermostat state required");
  if (thermostat_on_mask != 0u && dof == 0) return fail(RUMDX_E_INVALID, e + ": zero degrees of freedom");
  return RUMDX_OK;
}

}  // namespace
}  // namespace rumdx

extern "C" int rumdx_pair_lj_small_step(const rumdx_particles* p, rumdx_nblist* nb, const float* params_dev,
                                        uint32_t ntypes, const float box[8], int cutoff_method, float* r_out_dev,
                                        rumdx_nh_state* nh_dev, float dt, uint32_t thermostat_on_mask, float omega2,
                                        uint32_t dof, uint32_t step, int store_forces, void* workspace_dev,
                                        void* stream) {
  using namespace rumdx;
  const char* entry = "rumdx_pair_lj_small_step";
  int rc = check_pair_args(entry, p, nb, params_dev, ntypes, box, 0);
  if (rc != RUMDX_OK) return rc;
  rc = check_small(entry, p, nb, nh_dev, thermostat_on_mask, dof, workspace_dev);
  if (rc != RUMDX_OK) return rc;
  if (p->v_dev == nullptr || p->im_dev == nullptr || r_out_dev == nullptr || r_out_dev == p->r_dev)
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_small_step: particle arrays not allocated or r_out_dev aliases r");
  if (cutoff_method != RUMDX_CUTOFF_NS && cutoff_method != RUMDX_CUTOFF_SP && cutoff_method != RUMDX_CUTOFF_SF)
    return fail(RUMDX_E_INVALID, "rumdx_pair_lj_small_step: invalid cutoff method");
  if (p->n == 0) return RUMDX_OK;
  SmallStep a{};
  a.r = reinterpret_cast<const float4*>(p->r_dev);
  a.f = reinterpret_cast<float4*>(p->f_dev);
  a.w = reinterpret_cast<float4*>(p->w_dev);
  a.params = params_dev;
  a.nt = ntypes;
  a.n = p->n;
  a.nvp = p->nvp;
  a.fz.r_out = reinterpret_cast<float4*>(r_out_dev);
  a.fz.v = reinterpret_cast<float4*>(p->v_dev);
  a.fz.im = reinterpret_cast<float4*>(p->im_dev);
  a.fz.rlo = reinterpret_cast<float4*>(p->rlo_dev);
  a.fz.dt = dt;
  a.fz.on_mask = thermostat_on_mask;
  if (nb != nullptr) {
    a.nbl = nb->nbl_dev;
    a.num_nbrs = nb->num_nbrs_dev;
    a.last_r = reinterpret_cast<float4*>(nb->last_r_dev);
    a.flags = nb->flags_dev;
    a.cut_skin2 = nb->cut_skin2_dev;
    a.max_nbrs = nb->max_nbrs;
    a.ex = Exclusions{p->unsorted_index_dev, nb->excl_start_dev, nb->excl_ids_dev};
    a.request = request_word(nb, step);
    a.set_request = request_word(nb, step + 1u);
    a.clear_request = step > 0u ? request_word(nb, step - 1u) : nullptr;
    a.fz.skin2_over_4 = static_cast<float>(0.25 * static_cast<double>(nb->skin) * static_cast<double>(nb->skin));
  }
  if (thermostat_on_mask != 0u) {
    double* partials = Workspace::partials(workspace_dev);
    rumdx_nh_state* states = Workspace::states(workspace_dev);
    const uint32_t np = ke_partials(p->n);
    a.nh = step > 1u ? states + (step - 1u) % 2u : nh_dev;
    a.nh_out = step > 0u ? states + step % 2u : nullptr;
    a.partials_in = step > 0u ? partials + static_cast<size_t>((step - 1u) % 2u) * np : nullptr;
    a.omega2 = omega2;
    a.dof = dof;
    a.fz.nh = nh_dev;
    a.fz.partials = partials + static_cast<size_t>(step % 2u) * np;
  }
  const Box bx = make_box(box);
  const hipStream_t st = as_stream(stream);
  const bool want = store_forces != 0;
  const auto launch = [&](auto cut) {
    if (nb != nullptr)
      launch_small<decltype(cut)::value, false>(a, bx, want, st);
    else
      launch_small<decltype(cut)::value, true>(a, bx, want, st);
  };
  switch (cutoff_method) {
    case RUMDX_CUTOFF_NS: launch(std::integral_constant<int, RUMDX_CUTOFF_NS>{}); break;
    case RUMDX_CUTOFF_SP: launch(std::integral_constant<int, RUMDX_CUTOFF_SP>{}); break;
    default: launch(std::integral_constant<int, RUMDX_CUTOFF_SF>{}); break;
  }
  return check_launch(entry);
}

extern "C" int rumdx_small_steps_end(const rumdx_particles* p, rumdx_nblist* nb, rumdx_nh_state* nh_dev, float dt,
                                     uint32_t thermostat_on_mask, float omega2, uint32_t dof, uint32_t steps,
                                     void* workspace_dev, void* stream) {
  using namespace rumdx;
  const char* entry = "rumdx_small_steps_end";
  const int rc = check_small(entry, p, nb, nh_dev, thermostat_on_mask, dof, workspace_dev);
  if (rc != RUMDX_OK) return rc;
  if (p->n == 0 || steps == 0) return RUMDX_OK;
  const bool thermo = thermostat_on_mask != 0u;
  if (!thermo && nb == nullptr) return RUMDX_OK;
  const uint32_t np = ke_partials(p->n);
  hipLaunchKernelGGL(k_small_end, dim3(1), dim3(kBlock), 0, as_stream(stream),
                     Workspace::partials(workspace_dev) + static_cast<size_t>((steps - 1u) % 2u) * np, np,
                     steps > 1u ? Workspace::states(workspace_dev) + (steps - 1u) % 2u : nh_dev,
                     thermo ? nh_dev : nullptr, dt, omega2, dof, nb != nullptr ? request_word(nb, steps) : nullptr,
                     nb != nullptr ? request_word(nb, steps - 1u) : nullptr,
                     nb != nullptr ? nb->flags_dev + RUMDX_FLAG_REBUILD : nullptr);
  return check_launch(entry);
}
