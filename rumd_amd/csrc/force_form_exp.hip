// Force kernels of the potential forms, compiled per form: exponential and Coulomb forms.
#include "force_form.h"

RUMDX_DEFINE_FORM(RUMDX_POT_BUCKINGHAM)
RUMDX_DEFINE_FORM(RUMDX_POT_YUKAWA)
RUMDX_DEFINE_FORM(RUMDX_POT_EXP)
RUMDX_DEFINE_FORM(RUMDX_POT_SAAP)
RUMDX_DEFINE_FORM(RUMDX_POT_SF_COULOMB)
