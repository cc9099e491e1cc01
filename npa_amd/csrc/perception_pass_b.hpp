// Launchers of the lane-split pass-B kernels (perception_kernels.hpp), one
// instantiation per channel width; included by the pass-B translation units
// only, which compile beside those of the other operators.
#pragma once

#include "perception_kernels.hpp"

namespace sphops {
namespace pk {

// f(slice width, 32-bit row offsets) for a.C channels; 64-bit offsets are
// compiled for 16 and 32 channels (split_ok admits no others that need them).
template <class F>
inline void with_slice(const Grid& g, uint32_t C, F&& f) {
  const bool off32 = row_offsets_fit_32(g, C);
  using std::integral_constant;
#define SPHOPS_SLICE(CW, O32) return f(integral_constant<int, CW>{}, integral_constant<bool, O32>{})
  if (off32) {
    switch (C) {
      case 8: SPHOPS_SLICE(2, true);
      case 12: SPHOPS_SLICE(3, true);
      case 16: SPHOPS_SLICE(4, true);
      case 20: SPHOPS_SLICE(5, true);
      case 24: SPHOPS_SLICE(6, true);
      case 32: SPHOPS_SLICE(8, true);
    }
  } else {
    switch (C) {
      case 16: SPHOPS_SLICE(4, false);
      case 32: SPHOPS_SLICE(8, false);
    }
  }
#undef SPHOPS_SLICE
  throw Error("no lane-split kernel for this channel count");
}

template <int D, bool P>
void pass_b_forward(const Grid& g, int parts, const OpPtrs& a, hipStream_t st) {
  const uint32_t wgs = schedule_groups(a.nwaves2, a.nwaves2_dev);
  if (wgs == 0) return;
  with_slice(g, a.C, [&](auto cw, auto off) {
    constexpr int CW = decltype(cw)::value;
    constexpr bool O32 = decltype(off)::value;
#define SPHOPS_FWD_QUAD(PARTS) \
  hipLaunchKernelGGL((k_blur_hybrid_fwd_quad<D, P, CW, O32, PARTS>), dim3(wgs), dim3(kThreads), 0, st, g.p, a)
    if (parts == 3) SPHOPS_FWD_QUAD(3);
    else if (parts == 2) SPHOPS_FWD_QUAD(2);
    else if (parts == 4) SPHOPS_FWD_QUAD(4);
    else if constexpr (CW % 4 != 0) SPHOPS_FWD_QUAD(1);
    else throw Error("blur alone runs on the grouped kernel at this channel count");
#undef SPHOPS_FWD_QUAD
  });
  SPHOPS_LAUNCHED();
}

template <int D, bool P>
void pass_b_backward(const Grid& g, int parts, bool full, const OpPtrs& a, hipStream_t st) {
  const uint32_t wgs = schedule_groups(a.nwaves2, a.nwaves2_dev);
  if (wgs == 0) return;
  with_slice(g, a.C, [&](auto cw, auto off) {
    constexpr int CW = decltype(cw)::value;
    constexpr bool O32 = decltype(off)::value;
#define SPHOPS_BWD_QUAD(FULL, PARTS) \
  hipLaunchKernelGGL((k_blur_hybrid_bwd_quad<D, P, CW, FULL, O32, PARTS>), dim3(wgs), dim3(kThreads), 0, st, g.p, a)
    if (full) {
      if (parts == 3) SPHOPS_BWD_QUAD(true, 3);
      else if (parts == 2) SPHOPS_BWD_QUAD(true, 2);
      else SPHOPS_BWD_QUAD(true, 1);
    } else {
      if (parts == 3) SPHOPS_BWD_QUAD(false, 3);
      else if (parts == 2) SPHOPS_BWD_QUAD(false, 2);
      else SPHOPS_BWD_QUAD(false, 1);
    }
#undef SPHOPS_BWD_QUAD
  });
  SPHOPS_LAUNCHED();
}

}  // namespace pk
}  // namespace sphops
