// The NPA MLP (models/npa.py:63-78 of the reference: Linear, ReLU, Linear)
// over one row per particle, for gfx950: y = relu(z W1^T + b1) W2^T + b2 with
// 128 hidden units, and its gradients, on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32), three kernels of one pass over the rows each.
//
// As separate layers the step reads and writes the 128-wide rows six times
// (first layer, ReLU + second layer, its input gradient, two weight
// gradients, the first layer's input gradient).  Here a row's hidden values
// stay in registers between the two products of a kernel: the products are
// arranged so that the result layout of the first is the operand layout of
// the second.  For a 32 x 32 tile, lane l supplies A[m = l % 32][k = l / 32]
// and B[k = l / 32][n = l % 32], and result register r of lane l holds row 8
// (r / 4) + 4 (l / 32) + r % 4, column l % 32.  So register r is a valid
// operand with the tile's columns as m or n and the rows {8 (r / 4) + r % 4,
// that + 4} as the k pair, and a lane's four registers of one r / 4 are four
// consecutive rows: the other operand comes in 16-byte pieces.
//
// * forward: hidden^T = W1 z^T (rows of z as n), then y^T = W2 relu(hidden)^T;
// * input gradient: dh^T = W2^T dy^T masked by hidden > 0, then dz^T = W1^T dh^T;
// * weight gradients: dh = dy W2 masked (rows as k of the next products),
//   then dW1 = dh^T z, db1 and dW2 = dy^T relu(hidden), one band of 32 hidden
//   units per wave, partial sums per chunk of rows added in a fixed order.
//
// Forward and input gradient keep their weights in LDS as operand images (one
// 16-byte read a lane feeds four matrix instructions) and walk row tiles of
// 32, one per wave at a time.  Bounds: 240 matrix instructions of 64 cycles a
// tile forward (padding included), 240 for the input gradient, 304 for the
// weight gradients: 0.2 + 0.2 + 0.26 ms for 2^20 rows of 83 -> 128 -> 19, beside 0.19 ms of memory
// traffic for each of the first two.  Measured inside a training step: 0.30 +
// 0.28 + 0.36 ms, where the separate kernels took 0.51 (library product,
// ReLU + second layer), 0.66 (its input gradient, library product) and 0.39;
// forward and backward back to back 1.54 -> 0.94 ms (0.95 with the next row
// tile's operands loaded under the second product only, before the weight
// gradients' shorter sums, which cost 0.03).
#include "sphops_internal.hpp"
#include "sphops_device.hpp"

#include <type_traits>
#include <utility>

namespace sphops {

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 32;            // matrix-core tile side
constexpr int kHid = kMlpHidden;  // 128
constexpr int kHT = kHid / kT;    // hidden tiles
constexpr int kMlpThreads = 256;  // of the backward kernels
constexpr int kMlpWaves = kMlpThreads / 64;

// Buffer resource over `bytes` from base: loads past it return 0, stores past
// it are dropped; kPast is an offset past any of them.
constexpr uint32_t kPast = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const float* base, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float load1(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ f32x4 load4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
__device__ __forceinline__ void store1(__amdgpu_buffer_rsrc_t r, uint32_t off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, off, 0, 0);
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void store4(__amdgpu_buffer_rsrc_t r, uint32_t off, f32x4 v) {
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, off, 0, 0);
}

__device__ __forceinline__ f32x16 mma(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// relu as torch computes it: NaN stays NaN
__device__ __forceinline__ float relu(float v) { return v <= 0.0f ? 0.0f : v; }

// Four columns loaded `shift` before their place, moved up and zero-filled
// (4 or more: none of them exist).
__device__ __forceinline__ f32x4 move_up(f32x4 t, int shift) {
  if (shift & 1) t = f32x4{t[1], t[2], t[3], 0.0f};
  if (shift & 2) t = f32x4{t[2], t[3], 0.0f, 0.0f};
  if (shift >= 4) t = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  return t;
}

// A lane's share of row c of a row tile of `width` >= 4 columns, G = ceil(width
// / 8): columns 8 g + 4 h .. + 3 (h the lane's half) for each group g, in
// 16-byte loads (dword-aligned).  The last group's load is moved back to end
// with the row, so that it stays inside it, and its values moved up and
// zero-filled.
template <int G>
struct RowLoad {
  uint32_t off, off_last;  // bytes
  int shift;               // columns the last load was moved back by; 4 or more: none of them exist
  __device__ __forceinline__ RowLoad(int width, int c, int h) {
    const int k = 8 * (G - 1) + 4 * h, at = min(k, width - 4);
    off = (uint32_t)(c * width + 4 * h) * 4u;
    off_last = (uint32_t)(c * width + at) * 4u;
    shift = k - at;
  }
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, f32x4 (&v)[G]) const {
#pragma unroll
    for (int g = 0; g < G - 1; ++g) v[g] = load4(r, off + 32u * g);
    v[G - 1] = load4(r, off_last);
  }
  // after the loads, before the first use
  __device__ __forceinline__ void settle(f32x4 (&v)[G]) const { v[G - 1] = move_up(v[G - 1], shift); }
};

// Result columns of a transposed tile back to row c: registers 4 q .. 4 q + 3
// are columns col0 + 8 q + 4 h .. + 3.
__device__ __forceinline__ void store_row(__amdgpu_buffer_rsrc_t r, int width, int col0, int c, int h, f32x16 acc) {
  const uint32_t row = (uint32_t)(c * width);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int k = col0 + 8 * q + 4 * h;
    const f32x4 v = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    if (col0 + 8 * q + 8 <= width) {  // uniform
      store4(r, (row + (uint32_t)k) * 4u, v);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) store1(r, k + j < width ? (row + (uint32_t)(k + j)) * 4u : kPast, v[j]);
    }
  }
}

// Fills an operand image of N entries (entry i = load(i)) by T threads, kBatch
// entries a thread in flight: a workgroup builds its images before its first
// row tile, and one entry at a time that took longer than the tiles of few
// rows (see k_mlp_forward and k_mlp_input_grad).
template <int N, int T, class Load>
__device__ __forceinline__ void build_image(f32x4* image, Load load) {
  constexpr int kBatch = 8;
#pragma unroll 1
  for (int i0 = 0; i0 < N; i0 += kBatch * T) {
    f32x4 v[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) v[u] = load(min(i0 + u * T + (int)threadIdx.x, N - 1));
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int i = i0 + u * T + (int)threadIdx.x;
      if (i < N) image[i] = v[u];
    }
  }
}

// ---------------------------------------------------------------- forward

// Threads a workgroup: the operand images of wide rows (G > 13) leave room for
// one workgroup per CU, which then gets two waves a SIMD by itself, unless the
// row tiles are no more than a wave each for the chip's SIMDs: two waves on a
// SIMD take turns at the matrix core (300 rows of 163 columns: 33 us with 512
// threads a workgroup, 21 with 256).
constexpr int forward_threads(int g, int64_t tiles) { return g > 13 && tiles > 1024 ? 512 : 256; }

// G: groups of 8 input columns; OT: output tiles.  a (rows x 128), the
// pre-activations for the backward, may be null.
template <int G, int OT, int kThreads>
__global__ __launch_bounds__(kThreads, G > 13 ? kThreads / 256 : 2) void k_mlp_forward(const float* __restrict__ z,
                                                                const float* __restrict__ w1,
                                                                const float* __restrict__ b1,
                                                                const float* __restrict__ w2,
                                                                const float* __restrict__ b2, float* __restrict__ a,
                                                                float* __restrict__ y, int64_t rows, int nin,
                                                                int nout, int64_t tiles) {
  __shared__ f32x4 w1img[G][kHT][64];        // lane l: W1[32 t + l % 32][8 g + 4 (l / 32) ..]
  __shared__ f32x4 w2img[kHT * 4][OT][64];   // lane l: W2[32 o + l % 32][8 p + 4 (l / 32) ..]
  __shared__ f32x4 b1s[kHid / 4];
  __shared__ f32x4 b2s[OT * kT / 4];
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const __amdgpu_buffer_rsrc_t rw1 = rows_rsrc(w1, kHid * nin * 4), rw2 = rows_rsrc(w2, nout * kHid * 4);
  build_image<G * kHT * 64, kThreads>(&w1img[0][0][0], [&](int i) {
    const int l = i & 63, t = (i >> 6) % kHT, g = (i >> 6) / kHT, k = 8 * g + 4 * (l >> 5), at = min(k, nin - 4);
    return move_up(load4(rw1, (uint32_t)((kT * t + (l & 31)) * nin + at) * 4u), k - at);
  });
  build_image<kHT * 4 * OT * 64, kThreads>(&w2img[0][0][0], [&](int i) {
    const int l = i & 63, o = (i >> 6) % OT, p = (i >> 6) / OT, n = kT * o + (l & 31);
    return load4(rw2, n < nout ? (uint32_t)(n * kHid + 8 * p + 4 * (l >> 5)) * 4u : kPast);
  });
  if (threadIdx.x < kHid) reinterpret_cast<float*>(b1s)[threadIdx.x] = b1 != nullptr ? b1[threadIdx.x] : 0.0f;
  if (threadIdx.x < OT * kT)
    reinterpret_cast<float*>(b2s)[threadIdx.x] =
        b2 != nullptr && (int)threadIdx.x < nout ? b2[threadIdx.x] : 0.0f;
  __syncthreads();

  const int64_t step = (int64_t)gridDim.x * (kThreads / 64);
  int64_t tile = (int64_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kThreads / 64) + threadIdx.x / 64));
  // the next row tile's z is loaded while this one computes: all along, into
  // registers of its own, where they fit (kAhead), else under the second
  // product
  constexpr bool kAhead = G <= 11;
  f32x4 zv[G], zn[kAhead ? G : 1];
  const RowLoad<G> rl(nin, c, h);
  auto load = [&](int64_t t, f32x4 (&v)[G]) {
    const int64_t r0 = t * kT, nr = t < tiles ? min<int64_t>(kT, rows - r0) : 0;
    rl.load(rows_rsrc(z + (nr > 0 ? r0 * nin : 0), nr * nin * 4), v);
  };
  load(tile, zv);
  for (; tile < tiles; tile += step) {
    rl.settle(zv);
    if constexpr (kAhead) {
      __builtin_amdgcn_sched_barrier(0);
      load(tile + step, zn);
      __builtin_amdgcn_sched_barrier(0);
    }
    f32x16 acc[kHT];
#pragma unroll
    for (int t = 0; t < kHT; ++t) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 b = b1s[8 * t + 2 * q + h];
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[t][4 * q + j] = b[j];
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      f32x4 w[kHT];
#pragma unroll
      for (int t = 0; t < kHT; ++t) w[t] = w1img[g][t][lane];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
#pragma unroll
        for (int t = 0; t < kHT; ++t) acc[t] = mma(w[t][j], zv[g][j], acc[t]);
      }
    }
    if constexpr (!kAhead) {
      __builtin_amdgcn_sched_barrier(0);
      load(tile + step, zv);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int64_t r0 = tile * kT, nr = min<int64_t>(kT, rows - r0);
    if (a != nullptr) {
      const __amdgpu_buffer_rsrc_t ra = rows_rsrc(a + r0 * kHid, nr * kHid * 4);
#pragma unroll
      for (int t = 0; t < kHT; ++t) store_row(ra, kHid, kT * t, c, h, acc[t]);
    }
    f32x16 out[OT];
#pragma unroll
    for (int o = 0; o < OT; ++o) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 b = b2s[8 * o + 2 * q + h];
#pragma unroll
        for (int j = 0; j < 4; ++j) out[o][4 * q + j] = b[j];
      }
    }
#pragma unroll
    for (int p = 0; p < kHT * 4; ++p) {
      f32x4 w[OT];
#pragma unroll
      for (int o = 0; o < OT; ++o) w[o] = w2img[p][o][lane];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float v = relu(acc[p / 4][4 * (p % 4) + j]);
#pragma unroll
        for (int o = 0; o < OT; ++o) out[o] = mma(w[o][j], v, out[o]);
      }
    }
    const __amdgpu_buffer_rsrc_t ry = rows_rsrc(y + r0 * nout, nr * nout * 4);
#pragma unroll
    for (int o = 0; o < OT; ++o) store_row(ry, nout, kT * o, c, h, out[o]);
    if constexpr (kAhead) {
#pragma unroll
      for (int g = 0; g < G; ++g) zv[g] = zn[g];
    }
  }
}

// --------------------------------------------------------- input gradient

// CT: tiles of 32 input columns; GO: groups of 8 outputs.
template <int CT, int GO>
__global__ __launch_bounds__(kMlpThreads, CT > 3 ? 1 : 2) void k_mlp_input_grad(
    const float* __restrict__ dy, const float* __restrict__ w1, const float* __restrict__ w2,
    const float* __restrict__ a, float* __restrict__ dz, int64_t rows, int nin, int nout, int64_t tiles) {
  constexpr int kThreads = kMlpThreads;
  __shared__ f32x4 w1img[kHT * 4][CT][64];  // lane l: W1[8 p + 4 (l / 32) + j][32 ct + l % 32], j = 0..3
  __shared__ f32x4 w2img[GO][kHT][64];      // lane l: W2[8 g + 4 (l / 32) + j][32 t + l % 32]
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const __amdgpu_buffer_rsrc_t rw1 = rows_rsrc(w1, kHid * nin * 4), rw2 = rows_rsrc(w2, nout * kHid * 4);
  build_image<kHT * 4 * CT * 64, kThreads>(&w1img[0][0][0], [&](int i) {
    const int l = i & 63, ct = (i >> 6) % CT, p = (i >> 6) / CT, n = kT * ct + (l & 31);
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[j] = load1(rw1, n < nin ? (uint32_t)((8 * p + 4 * (l >> 5) + j) * nin + n) * 4u : kPast);
    return v;
  });
  build_image<GO * kHT * 64, kThreads>(&w2img[0][0][0], [&](int i) {
    const int l = i & 63, t = (i >> 6) % kHT, g = (i >> 6) / kHT, k = 8 * g + 4 * (l >> 5);
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      v[j] = load1(rw2, k + j < nout ? (uint32_t)((k + j) * kHid + kT * t + (l & 31)) * 4u : kPast);
    return v;
  });
  __syncthreads();

  const int64_t step = (int64_t)gridDim.x * (kThreads / 64);
  int64_t tile = (int64_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kThreads / 64) + threadIdx.x / 64));
  f32x4 dv[GO], dn[GO], av[kHT][4];
  const RowLoad<GO> rl(nout, c, h);
  const uint32_t arow = (uint32_t)(c * kHid + 4 * h) * 4u;
  auto rows_of = [&](int64_t t) { return t < tiles ? min<int64_t>(kT, rows - t * kT) : (int64_t)0; };
  auto load_dy = [&](int64_t t) {
    const int64_t nr = rows_of(t);
    rl.load(rows_rsrc(dy + (nr > 0 ? t * kT * nout : 0), nr * nout * 4), dn);
  };
  auto load_a = [&](int64_t t, int u) {
    const int64_t nr = rows_of(t);
    const __amdgpu_buffer_rsrc_t ra = rows_rsrc(a + (nr > 0 ? t * kT * kHid : 0), nr * kHid * 4);
#pragma unroll
    for (int q = 0; q < 4; ++q) av[u][q] = load4(ra, arow + (uint32_t)(kT * u + 8 * q) * 4u);
  };
  load_dy(tile);
#pragma unroll
  for (int u = 0; u < kHT; ++u) load_a(tile, u);
  for (; tile < tiles; tile += step) {
    rl.settle(dn);
#pragma unroll
    for (int g = 0; g < GO; ++g) dv[g] = dn[g];
    __builtin_amdgcn_sched_barrier(0);
    load_dy(tile + step);  // in flight until the next row tile
    __builtin_amdgcn_sched_barrier(0);
    f32x16 out[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) out[ct] = f32x16{};
    // one hidden tile after the other, so that one of them is live
#pragma unroll
    for (int t = 0; t < kHT; ++t) {
      f32x16 dh = f32x16{};
#pragma unroll
      for (int g = 0; g < GO; ++g) {
        const f32x4 w = w2img[g][t][lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) dh = mma(w[j], dv[g][j], dh);
      }
      // torch's threshold_backward: 0 where relu(a) <= 0
#pragma unroll
      for (int r = 0; r < 16; ++r) dh[r] = av[t][r / 4][r % 4] <= 0.0f ? 0.0f : dh[r];
      __builtin_amdgcn_sched_barrier(0);
      load_a(tile + step, t);  // in flight until the next row tile
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        f32x4 w[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) w[ct] = w1img[4 * t + p][ct][lane];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
          for (int ct = 0; ct < CT; ++ct) out[ct] = mma(w[ct][j], dh[4 * p + j], out[ct]);
        }
      }
    }
    const int64_t r0 = tile * kT, nr = min<int64_t>(kT, rows - r0);
    const __amdgpu_buffer_rsrc_t rz = rows_rsrc(dz + r0 * nin, nr * nin * 4);
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) store_row(rz, nin, kT * ct, c, h, out[ct]);
  }
}

// -------------------------------------------------------- weight gradients

// Waves per SIMD of the weight gradients: as many as their sums in registers
// leave room for.
constexpr int weight_grad_waves(int ct, int go) { return ct > 3 ? 1 : ct > 2 || go > 3 ? 2 : 3; }

// Workgroup = one chunk of rows; wave t the hidden units 32 t .. 32 t + 31.
// The four waves share each row tile's z and dy, staged in LDS as they lie in
// memory (the tile's rows are one contiguous piece of each), the next tile's
// loaded under this one's products; read straight from memory by every wave,
// a tile's operands took more registers than two waves a SIMD have.  The
// chunk's partial sums: dW1 (128 x nin), db1 (128), dW2 (nout x 128), db2
// (nout), in that order.
template <int CT, int GO>
__global__ __launch_bounds__(kMlpThreads, weight_grad_waves(CT, GO)) void k_mlp_weight_grad(
    const float* __restrict__ z, const float* __restrict__ a, const float* __restrict__ dy,
    const float* __restrict__ w2, float* __restrict__ part, int64_t rows, int nin, int nout, int64_t chunk_rows) {
  constexpr int OT = (GO + 3) / 4;
  constexpr int kZ4 = kT * kT * CT / 4, kD4 = kT * 8 * GO / 4;        // 16-byte pieces of a tile's z and dy
  constexpr int kLZ = (kZ4 + kMlpThreads - 1) / kMlpThreads;          // pieces a thread stages
  constexpr int kLD = (kD4 + kMlpThreads - 1) / kMlpThreads;
  static_assert(kMlpWaves == kHT, "one hidden band a wave");
  // operand reads of columns past a row's end fall into the next row, and for
  // the last row into the padding: their results are not kept
  __shared__ f32x4 zs[2][kZ4 + kT / 4], ds[2][kD4 + OT * kT / 4];
  // dW2, whose rows relu(a) >= 0 do not cancel: every kFold tiles its sums
  // move to LDS (each thread its own words), so that no chain of roundings is
  // longer than kFold * kT rows (10^6 rows, 83 -> 128 -> 19: error against
  // 64 bits 4.8e-7 with a chain a chunk, 3.8e-7 so)
  constexpr int kFold = 8;
  __shared__ float fold[OT][16][kMlpThreads];
#pragma unroll
  for (int o = 0; o < OT; ++o) {
#pragma unroll
    for (int r = 0; r < 16; ++r) fold[o][r][threadIdx.x] = 0.0f;
  }
  const int lane = threadIdx.x & 63, c = lane & 31, h = lane >> 5;
  const int band = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64) * kT;
  const int64_t r0 = (int64_t)blockIdx.x * chunk_rows, nr = min<int64_t>(chunk_rows, rows - r0);

  f32x4 wv[GO];  // W2[8 g + 4 h + j][band + c]
#pragma unroll
  for (int g = 0; g < GO; ++g) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = 8 * g + 4 * h + j;
      wv[g][j] = k < nout ? w2[(int64_t)k * kHid + band + c] : 0.0f;
    }
  }
  const uint32_t ac = (uint32_t)(4 * h * kHid + band + c) * 4u;
  f32x16 acc1[CT], acc2[OT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) acc1[ct] = f32x16{};
#pragma unroll
  for (int o = 0; o < OT; ++o) acc2[o] = f32x16{};
  float sb1 = 0.0f, sb2[OT] = {};

  // a row past the chunk loads zeros: it adds nothing
  f32x4 zst[kLZ], dst[kLD];
  float av[16];
  auto rsrc = [&](const float* base, int width, int64_t t0) {
    const int64_t left = t0 < nr ? nr - t0 : 0;
    return rows_rsrc(base + (r0 + (left > 0 ? t0 : 0)) * width, left * width * 4);
  };
  auto load = [&](int64_t t0) {
    const __amdgpu_buffer_rsrc_t rz = rsrc(z, nin, t0), rd = rsrc(dy, nout, t0), ra = rsrc(a, kHid, t0);
#pragma unroll
    for (int u = 0; u < kLZ; ++u) {
      const int i = u * kMlpThreads + (int)threadIdx.x;
      zst[u] = load4(rz, i < 8 * nin ? (uint32_t)i * 16u : kPast);  // a tile's z is 8 nin pieces
    }
#pragma unroll
    for (int u = 0; u < kLD; ++u) {
      const int i = u * kMlpThreads + (int)threadIdx.x;
      dst[u] = load4(rd, i < 8 * nout ? (uint32_t)i * 16u : kPast);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) av[r] = load1(ra, ac + (uint32_t)((8 * (r / 4) + r % 4) * kHid) * 4u);
  };
  load(0);
  int buf = 0;
  for (int64_t t0 = 0; t0 < nr; t0 += kT, buf ^= 1) {
    if (t0 > 0 && t0 % (kFold * kT) == 0) {
#pragma unroll
      for (int o = 0; o < OT; ++o) {
#pragma unroll
        for (int r = 0; r < 16; ++r) fold[o][r][threadIdx.x] += acc2[o][r];
        acc2[o] = f32x16{};
      }
    }
#pragma unroll
    for (int u = 0; u < kLZ; ++u) {
      const int i = u * kMlpThreads + (int)threadIdx.x;
      if (i < kZ4) zs[buf][i] = zst[u];
    }
#pragma unroll
    for (int u = 0; u < kLD; ++u) {
      const int i = u * kMlpThreads + (int)threadIdx.x;
      if (i < kD4) ds[buf][i] = dst[u];
    }
    // one barrier a tile: a wave writes a buffer again only after the next
    // barrier, which every wave reaches after its reads of this one
    __syncthreads();
    float am[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) am[r] = av[r];
    __builtin_amdgcn_sched_barrier(0);
    load(t0 + kT);  // the next tile's, in flight under this one's products
    __builtin_amdgcn_sched_barrier(0);
    const float* __restrict__ zt = reinterpret_cast<const float*>(zs[buf]);
    const float* __restrict__ dt = reinterpret_cast<const float*>(ds[buf]);
    f32x16 dh = f32x16{};
#pragma unroll
    for (int g = 0; g < GO; ++g) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 8 * g + 4 * h + j;
        float v = dt[c * nout + k];
        if (g == GO - 1) v = k < nout ? v : 0.0f;
        dh = mma(v, wv[g][j], dh);
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      dh[r] = am[r] <= 0.0f ? 0.0f : dh[r];
      sb1 += dh[r];
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 8 * (r / 4) + 4 * h + r % 4;
#pragma unroll
      for (int o = 0; o < OT; ++o) {
        const float v = dt[row * nout + kT * o + c];
        sb2[o] += v;
        acc2[o] = mma(v, relu(am[r]), acc2[o]);
      }
#pragma unroll
      for (int ct = 0; ct < CT; ++ct) acc1[ct] = mma(dh[r], zt[row * nin + kT * ct + c], acc1[ct]);
    }
  }

  const int64_t n1 = (int64_t)kHid * nin, n2 = (int64_t)nout * kHid;
  float* __restrict__ p = part + (int64_t)blockIdx.x * (n1 + kHid + n2 + nout);
#pragma unroll
  for (int ct = 0; ct < CT; ++ct) {
    const int col = kT * ct + c;
    if (col < nin) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        p[(int64_t)(band + 8 * (r / 4) + 4 * h + r % 4) * nin + col] = acc1[ct][r];
    }
  }
  sb1 += __shfl_xor(sb1, 32);
  if (h == 0) p[n1 + band + c] = sb1;
#pragma unroll
  for (int o = 0; o < OT; ++o) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = kT * o + 8 * (r / 4) + 4 * h + r % 4;
      if (m < nout) p[n1 + kHid + (int64_t)m * kHid + band + c] = fold[o][r][threadIdx.x] + acc2[o][r];
    }
    const float s = sb2[o] + __shfl_xor(sb2[o], 32);
    if (band == 0 && h == 0 && kT * o + c < nout) p[n1 + kHid + n2 + kT * o + c] = s;
  }
}

// out[e] = sum over chunks of part[chunk * n + e] in a fixed order: wave q of
// the workgroup keeps eight running sums over chunks q + 16 (8 s + k), adds
// them k = 0..7, and wave 0 adds the 16 waves' sums.  Element e goes to dW1,
// db1, dW2 or db2 (any of them may be null).
constexpr int kSumWaves = 16;
__global__ __launch_bounds__(64 * kSumWaves) void k_mlp_chunk_sum(const float* __restrict__ part,
                                                                  float* __restrict__ dw1, float* __restrict__ db1,
                                                                  float* __restrict__ dw2, float* __restrict__ db2,
                                                                  int n1, int n2, int n, int64_t chunks) {
  __shared__ float red[kSumWaves][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int e = (int)blockIdx.x * 64 + lane;
  float s[8] = {};
  if (e < n) {
    int64_t c = q;
    for (; c + 7 * kSumWaves < chunks; c += 8 * kSumWaves) {
#pragma unroll
      for (int k = 0; k < 8; ++k) s[k] += part[(c + k * kSumWaves) * n + e];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (c + k * kSumWaves < chunks) s[k] += part[(c + k * kSumWaves) * n + e];
  }
  float total = 0.0f;
#pragma unroll
  for (int k = 0; k < 8; ++k) total += s[k];
  red[q][lane] = total;
  __syncthreads();
  if (q != 0 || e >= n) return;
  float t = 0.0f;
#pragma unroll
  for (int k = 0; k < kSumWaves; ++k) t += red[k][lane];
  if (e < n1) {
    if (dw1 != nullptr) dw1[e] = t;
  } else if (e < n1 + kHid) {
    if (db1 != nullptr) db1[e - n1] = t;
  } else if (e < n1 + kHid + n2) {
    if (dw2 != nullptr) dw2[e - n1 - kHid] = t;
  } else if (db2 != nullptr) {
    db2[e - n1 - kHid - n2] = t;
  }
}

// Workgroups of the tile kernels: two waves a SIMD over the 256 CUs (what
// registers allow), fewer for fewer tiles.
inline dim3 tile_grid(int64_t tiles, int threads) {
  const int waves = threads / 64;
  return dim3((uint32_t)std::min<int64_t>(2048 / waves, (tiles + waves - 1) / waves));
}

// Rows per chunk of the weight gradients: a chunk (of four waves) for every
// workgroup the chip holds at once, two where that is two a CU (shorter chains
// of roundings: dW1), at least two row tiles and at most kMaxChunkRows, which
// bounds the chains of dW1 and db1 for any number of rows (from 4.2 or 8.4
// million rows on).
int64_t weight_chunk_rows(int64_t rows, int nin, int nout) {
  const int waves = weight_grad_waves((nin + kT - 1) / kT, (nout + 7) / 8);
  const int64_t want = 256 * (waves == 2 ? 4 : std::max(2, waves));
  const int64_t c = (rows + want - 1) / want;
  return std::min<int64_t>(kMaxChunkRows, std::max<int64_t>(64, (c + kT - 1) / kT * kT));
}
int64_t weight_chunks(int64_t rows, int nin, int nout) {
  const int64_t c = weight_chunk_rows(rows, nin, nout);
  return rows > 0 ? (rows + c - 1) / c : 0;
}

// f(integral_constant n) for a run-time 1 <= n <= N.
template <int N, class F>
void with_groups(int n, F&& f) {
  if constexpr (N > 1) {
    if (n < N) return with_groups<N - 1>(n, std::forward<F>(f));
  }
  f(std::integral_constant<int, N>{});
}

}  // namespace

bool mlp_fits(int64_t rows, int nin, int hidden, int nout) {
  return hidden == kHid && nin >= 4 && nin <= kMaxMlpIn && nout >= 4 && nout <= kMaxMlpOut && rows >= 0 &&
         rows <= kMaxMlpRows;
}

int64_t mlp_weight_grad_floats(int64_t rows, int nin, int nout) {
  return weight_chunks(rows, nin, nout) * ((int64_t)kHid * nin + kHid + (int64_t)nout * kHid + nout);
}

void run_mlp_forward(const float* z, const float* w1, const float* b1, const float* w2, const float* b2, float* a,
                     float* y, int64_t rows, int nin, int nout, hipStream_t st) {
  if (rows == 0) return;
  const int64_t tiles = (rows + kT - 1) / kT;
  with_groups<kMaxMlpIn / 8>((nin + 7) / 8, [&](auto gc) {
    constexpr int G = decltype(gc)::value;
    auto launch = [&](auto ot, auto threads) {
      constexpr int T = decltype(threads)::value;
      hipLaunchKernelGGL((k_mlp_forward<G, decltype(ot)::value, T>), tile_grid(tiles, T), dim3(T), 0, st, z, w1, b1,
                         w2, b2, a, y, rows, nin, nout, tiles);
    };
    with_groups<2>(nout <= kT ? 1 : 2, [&](auto ot) {
      if constexpr (forward_threads(G, kMaxMlpRows) == 512) {
        if (forward_threads(G, tiles) == 512) return launch(ot, std::integral_constant<int, 512>{});
      }
      launch(ot, std::integral_constant<int, 256>{});
    });
  });
  SPHOPS_LAUNCHED();
}

namespace {
// f(column tiles, output groups) for the backward kernels
template <class F>
void with_tiles(int nin, int nout, F&& f) {
  constexpr int kMaxCT = (kMaxMlpIn + kT - 1) / kT;
  with_groups<kMaxCT>((nin + kT - 1) / kT, [&](auto ct) {
    with_groups<kMaxMlpOut / 8>((nout + 7) / 8, [&](auto go) { f(ct, go); });
  });
}
}  // namespace

void run_mlp_input_grad(const float* dy, const float* w1, const float* w2, const float* a, float* dz, int64_t rows,
                        int nin, int nout, hipStream_t st) {
  if (rows == 0) return;
  const int64_t tiles = (rows + kT - 1) / kT;
  with_tiles(nin, nout, [&](auto ct, auto go) {
    constexpr int CT = decltype(ct)::value, T = kMlpThreads;
    hipLaunchKernelGGL((k_mlp_input_grad<CT, decltype(go)::value>), tile_grid(tiles, T), dim3(T), 0, st, dy, w1, w2,
                       a, dz, rows, nin, nout, tiles);
  });
  SPHOPS_LAUNCHED();
}

void run_mlp_weight_grad(const float* z, const float* a, const float* dy, const float* w2, float* dw1, float* db1,
                         float* dw2, float* db2, int64_t rows, int nin, int nout, float* work, hipStream_t st) {
  const int64_t chunks = weight_chunks(rows, nin, nout);
  if (chunks > 0) {
    with_tiles(nin, nout, [&](auto ct, auto go) {
      hipLaunchKernelGGL((k_mlp_weight_grad<decltype(ct)::value, decltype(go)::value>), dim3((uint32_t)chunks),
                         dim3(kMlpThreads), 0, st, z, a, dy, w2, work, rows, nin, nout,
                         weight_chunk_rows(rows, nin, nout));
    });
    SPHOPS_LAUNCHED();
  }
  const int n1 = kHid * nin, n2 = nout * kHid, n = n1 + kHid + n2 + nout;
  hipLaunchKernelGGL(k_mlp_chunk_sum, dim3((uint32_t)((n + 63) / 64)), dim3(64 * kSumWaves), 0, st, work, dw1, db1,
                     dw2, db2, n1, n2, n, chunks);
  SPHOPS_LAUNCHED();
}

}  // namespace sphops
