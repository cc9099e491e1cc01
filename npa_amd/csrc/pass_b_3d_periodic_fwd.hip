// Lane-split pass-B forward kernels for 3D periodic grids.
#include "perception_pass_b.hpp"

namespace sphops {
namespace pk {
template void pass_b_forward<3, true>(const Grid&, int, const OpPtrs&, hipStream_t);
}  // namespace pk
}  // namespace sphops
