// Force kernels of the potential forms, compiled per form: inverse power laws and the Gaussian.
#include "force_form.h"

RUMDX_DEFINE_FORM(RUMDX_POT_IPL_N)
RUMDX_DEFINE_FORM(RUMDX_POT_IPL_12)
RUMDX_DEFINE_FORM(RUMDX_POT_IPL_9)
RUMDX_DEFINE_FORM(RUMDX_POT_IPL_18)
RUMDX_DEFINE_FORM(RUMDX_POT_GAUSS)
