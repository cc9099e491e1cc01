// Lane-split pass-B backward kernels for 2D clamped grids.
#include "perception_pass_b.hpp"

namespace sphops {
namespace pk {
template void pass_b_backward<2, false>(const Grid&, int, bool, const OpPtrs&, hipStream_t);
}  // namespace pk
}  // namespace sphops
