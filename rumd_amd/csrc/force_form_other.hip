// Force kernels of the potential forms, compiled per form: the remaining forms.
#include "force_form.h"

RUMDX_DEFINE_FORM(RUMDX_POT_GIRIFALCO)
RUMDX_DEFINE_FORM(RUMDX_POT_DZUGUTOV)
RUMDX_DEFINE_FORM(RUMDX_POT_FERMI_JAGLA)
RUMDX_DEFINE_FORM(RUMDX_POT_REP_SHOULDER)
