// the exact LU's panel for complex64 matrices
#include "lu_panel.inc"

namespace scuffx {
template const void *panel_x_kernel<float2>(bool);
template const void *panel_l_kernel<float2>(int *);
}
