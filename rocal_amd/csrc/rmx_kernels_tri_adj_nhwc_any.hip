// K2t streaming path, lanes that own neighbouring columns, source rows at any byte phase (see rmx_kernels_tri_adj_impl.h).
#include "rmx_kernels_tri_adj_impl.h"

namespace rmx {
RMX_TADJ_UNIT(RMX_NHWC, true, tadj_unit_nhwc_any)
}  // namespace rmx
