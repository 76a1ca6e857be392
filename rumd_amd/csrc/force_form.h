// The pair policy of the potential forms in pot_forms.h and the launch of one
// form's force kernels.
//
// Reference: fij (include/rumd/PairPotential.h:1198-1244) around each class's
// ComputeInteraction; the reference generates one CalcF kernel per potential
// from a common skeleton (src/Generate_PP_FunctionBodies.py:3-127).  Here the
// skeleton is the shared kernels of force_kernels.h.  The kernels of a run's
// steps (no stresses, initialising) are compiled per form, so the eight pairs of
// a list group overlap; with the form as an argument every pair ended at a
// branch over the forms (43.7 us at Buckingham N = 30,011, then 23.2 us with
// the reciprocal and root of pot_forms.h, 17.8 in smaller tiles; 63.9 -> 31.9 at
// N = 150,000).  The other variants take the form as an argument (FORM = 0), one
// set for all.
//
// Per type pair the LDS table holds three float4: {rc^2, p1, p2, p3},
// {p4, p5, p6, p7}, {s(rc) rc, shift, p8, p9}, with the energy shift u(rc) for
// SP and s(rc) rc^2 + u(rc) for SF.
#pragma once

#include "force_kernels.h"
#include "pot_forms.h"

namespace rumdx {

// Everything one force launch needs (rumdx_pair_form's arguments, checked).
struct FormCall {
  const rumdx_particles* p;
  const rumdx_nblist* nb;
  const float* params;
  uint32_t nt;
  Box bx;
  int form;
  int cutoff;
  hipStream_t st;
};

// The initialising launch without stresses of one form, each defined in the
// source that instantiates it (force_form_*.hip).
template <int FORM>
int launch_form(const FormCall& c);

namespace {

constexpr const char* kFormEntry = "rumdx_pair_form";

template <int CUT, int FORM>
struct FormPair {
  int form;  // read when FORM is 0
  static constexpr uint32_t kRow = 3;
  static constexpr int kWavesPerEU = FORM != 0 ? 4 : 3;
  static constexpr bool kTunedWaves = false;

  __device__ __forceinline__ void load_table(float4* s_tab, const float* __restrict__ params, uint32_t nt) const {
    for (uint32_t k = threadIdx.x; k < nt * nt; k += blockDim.x) {
      const float* q = params + static_cast<size_t>(k) * RUMDX_NUM_PARAM;
      const float rc = q[0], src = q[RUMDX_NUM_PARAM - 2], ucut = q[RUMDX_NUM_PARAM - 1];
      s_tab[3 * k] = make_float4(rc * rc, q[1], q[2], q[3]);
      s_tab[3 * k + 1] = make_float4(q[4], q[5], q[6], q[7]);
      s_tab[3 * k + 2] = make_float4(src, CUT == RUMDX_CUTOFF_SF ? fmaf(src, rc, ucut) : ucut, q[8], q[9]);
    }
  }

  // fij: the form's s and u, shifted as the cut-off method asks (SP: u -
  // u(rc); SF: s - s(rc) rc / r, u + s(rc) rc (r - rc) - u(rc), the last two
  // terms as s(rc) rc r - (s(rc) rc^2 + u(rc))); pairs at or beyond rc are
  // masked.
  template <bool STR, bool FINE>
  __device__ __forceinline__ void core(float dx, float dy, float dz, float d2, uint32_t tj, const float4* prow,
                                       Acc& a) const {
    const float4 c0 = prow[3 * tj];
    const float4 c1 = prow[3 * tj + 1];
    const float4 c2 = prow[3 * tj + 2];
    const float p[10] = {0.f, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w, c2.z, c2.w};
    float u;
    float s = FORM != 0 ? pot_form_of<FORM, float>(d2, p, u) : pot_form<float>(form, d2, p, u);
    if (CUT == RUMDX_CUTOFF_SP) {
      u -= c2.y;
    } else if (CUT == RUMDX_CUTOFF_SF) {
      const float r = pf_sqrt(d2);
      s -= c2.x * pf_rcp(r);
      u += fmaf(c2.x, r, -c2.y);
    }
    const bool in = d2 < c0.x;
    accumulate<STR>(dx, dy, dz, d2, in ? s : 0.f, in ? u : 0.f, a);
  }
};

template <int FORM>
int launch_form_cut(const FormCall& c) {
  switch (c.cutoff) {
    case RUMDX_CUTOFF_NS:
      return launch_pair<FormPair<RUMDX_CUTOFF_NS, FORM>, false, true>({}, kFormEntry, c.p, c.nb, c.params, c.nt, c.bx, c.st);
    case RUMDX_CUTOFF_SP:
      return launch_pair<FormPair<RUMDX_CUTOFF_SP, FORM>, false, true>({}, kFormEntry, c.p, c.nb, c.params, c.nt, c.bx, c.st);
    default:
      return launch_pair<FormPair<RUMDX_CUTOFF_SF, FORM>, false, true>({}, kFormEntry, c.p, c.nb, c.params, c.nt, c.bx, c.st);
  }
}

}  // namespace
}  // namespace rumdx

#define RUMDX_DEFINE_FORM(F)                       \
  template <>                                      \
  int rumdx::launch_form<F>(const FormCall& c) {   \
    return launch_form_cut<F>(c);                  \
  }
