// Pair force / energy / virial of the potential forms in pot_forms.h
// (gfx950): the entry point rumdx_pair_form and the variants that take the
// form as an argument (stresses, or added to the forces there are).
#include "force_form.h"

namespace rumdx {
#define RUMDX_DECLARE_FORM(F) \
  template <>                 \
  int launch_form<F>(const FormCall& c);
RUMDX_ALL_FORMS(RUMDX_DECLARE_FORM)
#undef RUMDX_DECLARE_FORM

namespace {

template <int CUT>
int launch_any_form(const FormCall& c, bool init, bool str) {
  const FormPair<CUT, 0> pp{c.form};
  if (str) return init ? launch_pair<FormPair<CUT, 0>, true, true>(pp, kFormEntry, c.p, c.nb, c.params, c.nt, c.bx, c.st)
                       : launch_pair<FormPair<CUT, 0>, true, false>(pp, kFormEntry, c.p, c.nb, c.params, c.nt, c.bx, c.st);
  return launch_pair<FormPair<CUT, 0>, false, false>(pp, kFormEntry, c.p, c.nb, c.params, c.nt, c.bx, c.st);
}

}  // namespace
}  // namespace rumdx

extern "C" int rumdx_pair_form(const rumdx_particles* p, const rumdx_nblist* nb, const float* params_dev,
                               uint32_t ntypes, const float box[8], int form, int cutoff_method, int initialize,
                               int calc_stresses, void* stream) {
  using namespace rumdx;
  const int rc = check_pair_args(kFormEntry, p, nb, params_dev, ntypes, box, calc_stresses);
  if (rc != RUMDX_OK) return rc;
  if (!pot_form_known(form)) return fail(RUMDX_E_INVALID, "rumdx_pair_form: unknown potential form");
  if (p->n == 0) return RUMDX_OK;
  if (cutoff_method != RUMDX_CUTOFF_NS && cutoff_method != RUMDX_CUTOFF_SP && cutoff_method != RUMDX_CUTOFF_SF)
    return fail(RUMDX_E_INVALID, "rumdx_pair_form: invalid cutoff method");
  const FormCall c{p, nb, params_dev, ntypes, make_box(box), form, cutoff_method, as_stream(stream)};
  const bool init = initialize != 0, str = calc_stresses != 0;
  if (init && !str) {
    switch (form) {
#define RUMDX_FORM_CASE(F) \
  case F: return launch_form<F>(c);
      RUMDX_ALL_FORMS(RUMDX_FORM_CASE)
#undef RUMDX_FORM_CASE
    }
  }
  switch (cutoff_method) {
    case RUMDX_CUTOFF_NS: return launch_any_form<RUMDX_CUTOFF_NS>(c, init, str);
    case RUMDX_CUTOFF_SP: return launch_any_form<RUMDX_CUTOFF_SP>(c, init, str);
    default: return launch_any_form<RUMDX_CUTOFF_SF>(c, init, str);
  }
}
