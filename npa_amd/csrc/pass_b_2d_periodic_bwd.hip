// Lane-split pass-B backward kernels for 2D periodic grids.
#include "perception_pass_b.hpp"

namespace sphops {
namespace pk {
template void pass_b_backward<2, true>(const Grid&, int, bool, const OpPtrs&, hipStream_t);
}  // namespace pk
}  // namespace sphops
