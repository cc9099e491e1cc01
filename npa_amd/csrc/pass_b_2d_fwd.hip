// Lane-split pass-B forward kernels for 2D clamped grids.
#include "perception_pass_b.hpp"

namespace sphops {
namespace pk {
template void pass_b_forward<2, false>(const Grid&, int, const OpPtrs&, hipStream_t);
}  // namespace pk
}  // namespace sphops
