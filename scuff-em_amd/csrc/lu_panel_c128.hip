// the exact LU's panel for complex128 matrices
#include "lu_panel.inc"

namespace scuffx {
template const void *panel_x_kernel<double2>(bool);
template const void *panel_l_kernel<double2>(int *);
}
