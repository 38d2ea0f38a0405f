// the exact LU's panel for real matrices
#include "lu_panel.inc"

namespace scuffx {
template const void *panel_x_kernel<double>(bool);
template const void *panel_l_kernel<double>(int *);
}
