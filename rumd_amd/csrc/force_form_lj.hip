// Force kernels of the potential forms, compiled per form: Lennard-Jones variants and logarithmic forms.
#include "force_form.h"

RUMDX_DEFINE_FORM(RUMDX_POT_LJ_SMOOTH_2_4)
RUMDX_DEFINE_FORM(RUMDX_POT_GLJ_M_N)
RUMDX_DEFINE_FORM(RUMDX_POT_LJ_GAUSS)
RUMDX_DEFINE_FORM(RUMDX_POT_LJ_LN)
RUMDX_DEFINE_FORM(RUMDX_POT_IPL6_LN)
