// Lane-split pass-B backward kernels for 3D periodic grids.
#include "perception_pass_b.hpp"

namespace sphops {
namespace pk {
template void pass_b_backward<3, true>(const Grid&, int, bool, const OpPtrs&, hipStream_t);
}  // namespace pk
}  // namespace sphops
