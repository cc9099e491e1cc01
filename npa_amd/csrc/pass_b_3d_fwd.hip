// Lane-split pass-B forward kernels for 3D clamped grids.
#include "perception_pass_b.hpp"

namespace sphops {
namespace pk {
template void pass_b_forward<3, false>(const Grid&, int, const OpPtrs&, hipStream_t);
}  // namespace pk
}  // namespace sphops
