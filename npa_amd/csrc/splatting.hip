// Differentiable 2D Gaussian splatting of particles into images
// (utils/splatting.py:6-117 of the reference), forward and backward, for
// gfx950.
//
// The reference evaluates a (2r+1)^2 patch of Gaussian weights around each
// particle's pixel, optionally normalises them to sum to K over the patch,
// and scatter-adds w and w * rgb into the image with float atomics
// (torch.scatter_add_), so its sums come in no fixed order.  Here:
//  * forward: a per-particle pass writes each particle's patch centre,
//    offset and normalised colour (32 bytes); then one workgroup per 16 x 16
//    pixel tile gathers: its waves list the particles whose patch overlaps
//    the tile and multiply their separable weights on the matrix cores.
//    Every pixel's sum runs in a fixed order: deterministic, no atomics, no
//    zero-fill pass (each tile writes all of its pixels);
//  * backward: the same lists per tile, dL/dimage of the tile times the
//    weights on the matrix cores, one record per particle and tile, and a
//    pass that adds a particle's records in a fixed order; or, for patches
//    or images where that does not pay, one wave per particle that sweeps
//    its own patch.  The patch normalisation's sum and its derivative are
//    separable (a product of two 1D sums), which costs 4(2r+1) exponentials
//    per particle instead of (2r+1)^2.
#include "sphops_internal.hpp"

namespace sphops {

namespace {

constexpr int kTile = 16;               // pixels per tile side; one thread per pixel
constexpr int kTileThreads = kTile * kTile;
constexpr int kWavesPerTile = kTileThreads / 64;
constexpr int kBwdWaves = 4;            // particles per backward workgroup

// pos = (x - lo) / (hi - lo) * (img_size - 1) per axis; with y_up, pos_y =
// (img_size - 1) - pos_y (utils/splatting.py:33-37).  Each step is in fp32
// as torch evaluates it; torch divides a tensor by a Python scalar as a
// product with the scalar's fp32 reciprocal, and so does this code.
// Returns false for particles whose patch cannot reach the image (and for
// NaN positions); otherwise the patch centre pixel (bx, by) = floor(pos) and
// the fractional offset (fx, fy) = pos - floor(pos).
__device__ __forceinline__ bool particle_setup(const SplatParams& sp, float x0, float x1, int& bx, int& by, float& fx,
                                               float& fy) {
  const float px = (x0 - sp.lo) * sp.inv_span * sp.scale;
  float py = (x1 - sp.lo) * sp.inv_span * sp.scale;
  if (sp.y_up) py = sp.scale - py;
  const float lim_lo = -(float)sp.r - 1.0f, lim_hi = (float)(sp.H + sp.r);
  if (!(px >= lim_lo && px < lim_hi && py >= lim_lo && py < lim_hi)) return false;
  const float fbx = floorf(px), fby = floorf(py);
  bx = (int)fbx;
  by = (int)fby;
  fx = px - fbx;
  fy = py - fby;
  return true;
}

// exp(-(a^2 + b^2) / (2 sigma^2)).  The argument is never below -25 (a patch
// corner: |offset|^2 <= 2 r^2, r = ceil(5 sigma)), where the hardware 2^x on
// x log2(e) is within 1e-6 relative of expf.
__device__ __forceinline__ float gauss(float a, float b, float inv_two_s2) {
  return __expf(-(a * a + b * b) * inv_two_s2);
}

__device__ __forceinline__ uint32_t rank_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Orders a wave's LDS writes before its own later reads (its LDS operations
// complete in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Per particle, once: the patch centre pixel (kNoPatch where the patch cannot
// reach the image), the fractional offset and the colour scaled by the
// normalisation, (k r, k g, k b, k), k = K / (1e-8 + S) (1 without it): three
// arrays, 32 bytes a particle, so that the tiles' search for their particles
// reads 8 bytes of each.
constexpr int kNoPatch = -(1 << 30);

// Share of an image's tiles that have to do the work for the tile by tile
// backward (measurements with its other limits, below).
constexpr float kTilesMinShare = 0.5f;

struct SplatRecords {
  float4* __restrict__ col;
  int2* __restrict__ centre;
  float2* __restrict__ frac;
  SplatRecords(void* work, int64_t n)
      : col(static_cast<float4*>(work)), centre(reinterpret_cast<int2*>(col + n)),
        frac(reinterpret_cast<float2*>(centre + n)) {}
};

__device__ __forceinline__ void prepare_particle(const SplatParams& sp, const float* __restrict__ x,
                                                 const float* __restrict__ color, int64_t i,
                                                 const SplatRecords& rec) {
  int bx = 0, by = 0;
  float fx = 0.0f, fy = 0.0f;
  const bool live = particle_setup(sp, x[2 * i], x[2 * i + 1], bx, by, fx, fy);
  float k = 1.0f;
  if (live && sp.normalize) {
    float sx = 0.0f, sy = 0.0f;
    for (int d = -sp.r; d <= sp.r; ++d) {
      sx += gauss((float)d - fx, 0.0f, sp.inv_two_s2);
      sy += gauss((float)d - fy, 0.0f, sp.inv_two_s2);
    }
    k = sp.K / (1e-8f + sx * sy);
  }
  const float* c = color + i * sp.ncolor + (sp.ncolor - 3);
  rec.centre[i] = make_int2(live ? bx : kNoPatch, by);
  rec.frac[i] = make_float2(fx, fy);
  rec.col[i] = make_float4(c[0] * k, c[1] * k, c[2] * k, k);
}

__global__ __launch_bounds__(256) void k_splat_prep(SplatParams sp, const float* __restrict__ x,
                                                    const float* __restrict__ color, int64_t n, SplatRecords rec) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) prepare_particle(sp, x, color, i, rec);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma_16x16x4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Calls use(count) with the indices of the particles p0 .. p1 - 1 whose patch
// reaches the tile at (tx0, ty0) in `list` (kListSlots slots of LDS, this
// wave's), in ascending order, a list at a time; this wave takes every
// `waves`-th turn of 64 particles, four turns' centres loaded together.
constexpr int kListSlots = 512;
constexpr int kTurns = 4;

template <class Use>
__device__ __forceinline__ void for_tile_particles(const SplatRecords& rec, int r, int p0, int p1, int tx0, int ty0,
                                                   int wave, int waves, int* list, Use use) {
  const int lane = threadIdx.x % 64;
  int count = 0;
  for (int64_t c0 = p0 + 64 * (int64_t)wave; c0 < p1; c0 += (int64_t)64 * kTurns * waves) {
    int2 at[kTurns];
#pragma unroll
    for (int u = 0; u < kTurns; ++u) {
      const int64_t i = c0 + (int64_t)64 * waves * u + lane;
      at[u] = i < p1 ? rec.centre[i] : make_int2(kNoPatch, 0);
    }
#pragma unroll
    for (int u = 0; u < kTurns; ++u) {
      const bool hit = at[u].x + r >= tx0 && at[u].x - r < tx0 + kTile && at[u].y + r >= ty0 &&
                       at[u].y - r < ty0 + kTile;
      const uint64_t m = __ballot(hit);
      if (hit) list[count + (int)rank_below(m)] = (int)(c0 + (int64_t)64 * waves * u + lane);
      count += (int)__popcll(m);
    }
    if (count > kListSlots - 64 * kTurns) {
      wave_lds_fence();
      use(count);
      wave_lds_fence();
      count = 0;
    }
  }
  wave_lds_fence();
  if (count > 0) use(count);
}

// A tile's image is a product over its particles: pixel (row i, column j) of
// channel c is sum_p gy[p][i] * (gx[p][j] col[p][c]), the Gaussian being the
// product of its two axes.  So the weights cost 32 exponentials a particle
// and tile instead of 256, and the sums run on the fp32 matrix cores
// (v_mfma_f32_16x16x4_f32: a 16 x 16 tile, four particles an instruction, one
// instruction a channel): lane l supplies A[m = l % 16][k = l / 16] = gy of
// particle k at row m and B[k][n = l % 16] = gx col at column n, both computed
// in place, 0 outside the patch; result register r of lane l is row 4 (l / 16)
// + r, column l % 16.  Each of the workgroup's four waves lists its share of
// the image's particles that reach the tile, then multiplies them four at a
// time, the next four's records in flight; the four waves' sums are added in
// a fixed order.  A particle whose colour is not finite would turn the zeros
// outside its patch into NaN: a group with one is added pixel by pixel.
// 8 images of 256^2 with 4096 particles of radius 20 px: 92 us with one
// exponential and five multiply-adds a pixel and particle, 39 so (72 at eight
// waves a SIMD, which spills); what is left is the lists' latency and the
// weights' vector instructions.
__global__ __launch_bounds__(kTileThreads, 6) void k_splat_forward(SplatParams sp, SplatRecords rec,
                                                                   const int32_t* __restrict__ starts,
                                                                   float* __restrict__ out) {
  // the waves' lists, then their sums
  __shared__ __align__(16) float red[kWavesPerTile][4][kTile * kTile];
  static_assert(kWavesPerTile * kListSlots * sizeof(int) <= sizeof(red), "the lists fit where the sums go");
  const int b = blockIdx.z;
  const int tx0 = blockIdx.x * kTile, ty0 = blockIdx.y * kTile;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, kq = lane >> 4, ij = lane & 15;
  int* list = reinterpret_cast<int*>(red) + wave * kListSlots;
  const int r = sp.r;
  f32x4 acc[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) acc[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  auto multiply = [&](int count) {
    int p = list[min(kq, count - 1)];
    int2 at = rec.centre[p];
    float2 f = rec.frac[p];
    float4 c = rec.col[p];
    for (int e = 0; e < count; e += 4) {
      const int dx = ij + tx0 - at.x, dy = ij + ty0 - at.y;
      const float2 q = f;
      float4 w = c;
      const bool live = e + kq < count;
      if (e + 4 < count) {
        p = list[min(e + 4 + kq, count - 1)];
        at = rec.centre[p];
        f = rec.frac[p];
        c = rec.col[p];
      }
      const bool odd = live && !(isfinite(w.x) && isfinite(w.y) && isfinite(w.z) && isfinite(w.w));
      if (__ballot(odd) == 0) {
        float gx = gauss((float)dx - q.x, 0.0f, sp.inv_two_s2);
        float gy = gauss((float)dy - q.y, 0.0f, sp.inv_two_s2);
        gx = live && dx >= -r && dx <= r ? gx : 0.0f;
        gy = dy >= -r && dy <= r ? gy : 0.0f;
        if (!live) w = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        acc[0] = mfma_16x16x4(gy, gx * w.x, acc[0]);
        acc[1] = mfma_16x16x4(gy, gx * w.y, acc[1]);
        acc[2] = mfma_16x16x4(gy, gx * w.z, acc[2]);
        acc[3] = mfma_16x16x4(gy, gx * w.w, acc[3]);
        continue;
      }
      for (int u = e; u < min(e + 4, count); ++u) {  // uniform
        const int pu = list[u];
        const int2 au = rec.centre[pu];
        const float2 fu = rec.frac[pu];
        const float4 cu = rec.col[pu];
        const int ux = ij + tx0 - au.x;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int uy = 4 * kq + v + ty0 - au.y;
          if (ux >= -r && ux <= r && uy >= -r && uy <= r) {
            const float t = gauss((float)ux - fu.x, (float)uy - fu.y, sp.inv_two_s2);
            acc[0][v] += cu.x * t;
            acc[1][v] += cu.y * t;
            acc[2][v] += cu.z * t;
            acc[3][v] += cu.w * t;
          }
        }
      }
    }
  };
  for_tile_particles(rec, r, starts[b], starts[b + 1], tx0, ty0, wave, kWavesPerTile, list, multiply);
  __syncthreads();  // every wave is done with its list

#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave][c][(4 * kq + v) * kTile + ij] = acc[c][v];
  }
  __syncthreads();
  float o[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    o[c] = red[0][c][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kWavesPerTile; ++w) o[c] += red[w][c][threadIdx.x];
  }
  const int px = tx0 + (int)(threadIdx.x % kTile), py = ty0 + (int)(threadIdx.x / kTile);
  if (px < sp.H && py < sp.H)
    reinterpret_cast<float4*>(out)[((int64_t)b * sp.H + py) * sp.H + px] = make_float4(o[0], o[1], o[2], o[3]);
}

// The image a particle belongs to: the last b with starts[b] <= i.
__device__ __forceinline__ int image_of(const int32_t* starts, int images, int i) {
  int lo = 0, hi = images - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (starts[mid] <= i) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// Per particle, with g_q the patch weights, w_q = g_q K / n (n = 1e-8 + S,
// S = sum of g over the whole patch; w = g and n = 1 without normalisation),
// d_q = dL/dimage at pixel q (r, g, b, density) and G_q = rgb . d_q.rgb +
// d_q.density = dL/dw_q, over the pixels q of the patch inside the image:
//   dL/drgb = sum_q w_q d_q.rgb,
//   dL/dg_q = G_q K / n  (q inside) - (K / n^2) sum_p G_p g_p  (every q),
//   dg_q/dfx = g_q * 2 (q_x - fx) / (2 sigma^2), the same for y,
// and dL/dx = dL/dfx * (img_size - 1) / (hi - lo) (floor has no gradient), the y term
// negated with y_up.  Only the colour row's last three channels get a
// gradient.
struct PatchSums {
  float dr = 0.0f, dg = 0.0f, db = 0.0f;     // sum g d.rgb
  float gg = 0.0f, ggx = 0.0f, ggy = 0.0f;   // sum G g, G g (qx - fx), G g (qy - fy)
};
// sum g and sum g (q - f) over the whole patch, per axis: the normaliser
struct AxisSums {
  float sx = 0.0f, sy = 0.0f, sxa = 0.0f, sya = 0.0f;
};

// Lane `lane` of `lanes`' share of a particle's axis sums.
__device__ __forceinline__ AxisSums axis_sums(const SplatParams& sp, float fx, float fy, int lane, int lanes) {
  AxisSums a;
  for (int d = lane - sp.r; d <= sp.r; d += lanes) {
    const float ax = (float)d - fx, ay = (float)d - fy;
    const float gx = gauss(ax, 0.0f, sp.inv_two_s2), gy = gauss(ay, 0.0f, sp.inv_two_s2);
    a.sx += gx;
    a.sy += gy;
    a.sxa += gx * ax;
    a.sya += gy * ay;
  }
  return a;
}

// The gradients of particle i from its sums, by `lanes` lanes that all hold
// them.
__device__ __forceinline__ void store_gradients(const SplatParams& sp, int64_t i, bool live, const PatchSums& t,
                                                const AxisSums& a, int lane, int lanes, float* __restrict__ d_x,
                                                float* __restrict__ d_color) {
  float dfx = 0.0f, dfy = 0.0f, dr = 0.0f, dg = 0.0f, db = 0.0f;
  if (live) {
    const float k2 = 2.0f * sp.inv_two_s2;
    if (sp.normalize) {
      const float nrm = 1e-8f + a.sx * a.sy;
      const float kn = sp.K / nrm;
      const float dnrm = -kn / nrm * t.gg;  // dL/dn, times dn/dg_q = 1 for every q
      dr = kn * t.dr;
      dg = kn * t.dg;
      db = kn * t.db;
      dfx = k2 * (kn * t.ggx + dnrm * a.sxa * a.sy);
      dfy = k2 * (kn * t.ggy + dnrm * a.sx * a.sya);
    } else {
      dr = t.dr;
      dg = t.dg;
      db = t.db;
      dfx = k2 * t.ggx;
      dfy = k2 * t.ggy;
    }
    if (sp.y_up) dfy = -dfy;
  }
  const float jac = sp.inv_span * sp.scale;
  if (lane == 0) {
    d_x[2 * i] = dfx * jac;
    d_x[2 * i + 1] = dfy * jac;
  }
  for (int j = lane; j < sp.ncolor; j += lanes) {
    const int k = j - (sp.ncolor - 3);
    d_color[i * sp.ncolor + j] = k == 0 ? dr : k == 1 ? dg : k == 2 ? db : 0.0f;
  }
}

// A particle's sums over its patch, by a whole wave.
__device__ __forceinline__ PatchSums sweep_patch(const SplatParams& sp, int bx, int by, float fx, float fy, float cr,
                                                 float cg, float cb, const float4* __restrict__ dimg, int lane) {
  const int r = sp.r, P = 2 * r + 1, H = sp.H;
  PatchSums t;
  for (int q = lane; q < P * P; q += 64) {
    const int qy = q / P, qx = q - qy * P;
    const int ix = bx + qx - r, iy = by + qy - r;
    if (ix >= 0 && ix < H && iy >= 0 && iy < H) {
      const float ax = (float)(qx - r) - fx, ay = (float)(qy - r) - fy;
      const float g = gauss(ax, ay, sp.inv_two_s2);
      const float4 d = dimg[(int64_t)iy * H + ix];
      const float G = cr * d.x + cg * d.y + cb * d.z + d.w;
      t.dr += g * d.x;
      t.dg += g * d.y;
      t.db += g * d.z;
      t.gg += G * g;
      t.ggx += G * g * ax;
      t.ggy += G * g * ay;
    }
  }
  t.dr = wave_sum(t.dr);
  t.dg = wave_sum(t.dg);
  t.db = wave_sum(t.db);
  t.gg = wave_sum(t.gg);
  t.ggx = wave_sum(t.ggx);
  t.ggy = wave_sum(t.ggy);
  return t;
}

__global__ __launch_bounds__(64 * kBwdWaves) void k_splat_backward(SplatParams sp, const float* __restrict__ x,
                                                                   const float* __restrict__ color,
                                                                   const int32_t* __restrict__ starts, int images,
                                                                   int64_t n, const float* __restrict__ d_img,
                                                                   float* __restrict__ d_x,
                                                                   float* __restrict__ d_color) {
  const int64_t i = (int64_t)blockIdx.x * kBwdWaves + threadIdx.x / 64;
  const int lane = threadIdx.x % 64;
  if (i >= n) return;
  int bx = 0, by = 0;
  float fx = 0.0f, fy = 0.0f;
  const bool live = particle_setup(sp, x[2 * i], x[2 * i + 1], bx, by, fx, fy);
  const float* c = color + i * sp.ncolor + (sp.ncolor - 3);
  PatchSums t;
  AxisSums a;
  if (live) {  // wave-uniform
    const int b = image_of(starts, images, (int)i);
    t = sweep_patch(sp, bx, by, fx, fy, c[0], c[1], c[2],
                    reinterpret_cast<const float4*>(d_img) + (int64_t)b * sp.H * sp.H, lane);
    if (sp.normalize) a = axis_sums(sp, fx, fy, lane, 64);
  }
  if (live && sp.normalize) {  // wave-uniform
    a.sx = wave_sum(a.sx);
    a.sy = wave_sum(a.sy);
    a.sxa = wave_sum(a.sxa);
    a.sya = wave_sum(a.sya);
  }
  store_gradients(sp, i, live, t, a, lane, 64, d_x, d_color);
}

__device__ __forceinline__ int first_tile(int c, int r) { return max(0, c - r) / kTile; }
__device__ __forceinline__ int last_tile(int c, int r, int H) { return c + r < 0 ? -1 : min(H - 1, c + r) / kTile; }

// The records for the backward, and for each image whether its particles
// crowd in few tiles (crowded[its first particle]; the first `images`
// workgroups).  With h_t the particles that reach tile t, (sum h)^2 / sum h^2
// is the number of tiles that do the work; sum h is a mean over particles of
// the tiles that one reaches, sum h^2 one over pairs of the tiles that both
// reach, taken here from 256 particles, evenly spaced in the image's order,
// and 32 partners each.
constexpr int kLookPairs = 32;

__global__ __launch_bounds__(256) void k_splat_backward_prep(SplatParams sp, const float* __restrict__ x,
                                                             const float* __restrict__ color,
                                                             const int32_t* __restrict__ starts, int images,
                                                             int64_t n, SplatRecords rec, int* __restrict__ crowded) {
  if ((int)blockIdx.x >= images) {
    const int64_t i = (int64_t)(blockIdx.x - images) * 256 + threadIdx.x;
    if (i < n) prepare_particle(sp, x, color, i, rec);
    return;
  }
  __shared__ int4 reach[256];  // first and last tile, x and y
  __shared__ int sums[2][4];
  const int p0 = starts[blockIdx.x], size = starts[blockIdx.x + 1] - p0, m = min(size, 256), t = threadIdx.x;
  if (m <= 0) return;
  auto shared_tiles = [](int4 u, int4 v) {
    return max(0, min(u.y, v.y) - max(u.x, v.x) + 1) * max(0, min(u.w, v.w) - max(u.z, v.z) + 1);
  };
  int4 mine = make_int4(1, 0, 1, 0);
  if (t < m) {
    const int64_t i = p0 + (int64_t)t * size / m;
    int bx, by;
    float fx, fy;
    if (particle_setup(sp, x[2 * i], x[2 * i + 1], bx, by, fx, fy))
      mine = make_int4(first_tile(bx, sp.r), last_tile(bx, sp.r, sp.H), first_tile(by, sp.r),
                       last_tile(by, sp.r, sp.H));
    reach[t] = mine;
  }
  __syncthreads();
  int one = shared_tiles(mine, mine), both = 0;
  if (t < m && m > 1) {
    for (int j = 0; j < kLookPairs; ++j) both += shared_tiles(mine, reach[(t + 1 + j * (m - 1) / kLookPairs) % m]);
  }
  one = wave_sum(one);
  both = wave_sum(both);
  if (t % 64 == 0) {
    sums[0][t / 64] = one;
    sums[1][t / 64] = both;
  }
  __syncthreads();
  if (t == 0) {
    const float k = (float)(sums[0][0] + sums[0][1] + sums[0][2] + sums[0][3]) / (float)m;
    const float k2 = (float)(sums[1][0] + sums[1][1] + sums[1][2] + sums[1][3]) / (float)(m * kLookPairs);
    const float tiles = (float)((sp.H + kTile - 1) / kTile);
    crowded[p0] = k * k < kTilesMinShare * tiles * tiles * k2 ? 1 : 0;
  }
}

// The same sums tile by tile.  With d_c the tile's 16 x 16 pixels of channel c
// of dL/dimage, T_c[j] = sum_i d_c[i][j] gy[i] and Y_c[j] = sum_i d_c[i][j]
// gy[i] (i - fy) of 16 particles are two products on the fp32 matrix cores a
// channel: lane l supplies A[m = l % 16][k = l / 16] = d_c at column m of row
// k (of four; kept in registers) and B[k][n = l % 16] = gy of particle n at
// that row, and holds in result register v column 4 (l / 16) + v of particle
// l % 16.  So the lane weighs four columns of one particle with gx and two
// exchanges add the others: no pixel is read again for each particle that
// covers it.  A particle's sums over a tile go to the slot of that tile among
// the side * side that its patch can reach.  A wave takes every `waves`-th
// turn of 64 of the image's particles; blockIdx.z is the image and the part
// of the waves.  Non-finite colours or pixels, which zero weights do not
// silence, are summed pixel by pixel; crowded images are left out.  8 images of 256^2, 4096 particles of
// radius 20 px: 83 us a wave per particle (880 MB of pixels from the L2), 54
// so and 11 for the records and their sum; storing a group's sums a group
// later changes nothing.
__global__ __launch_bounds__(kTileThreads, 4) void k_splat_backward_tiles(SplatParams sp, SplatRecords rec,
                                                                          const int32_t* __restrict__ starts,
                                                                          int parts, int side,
                                                                          const float* __restrict__ d_img,
                                                                          const int* __restrict__ crowded,
                                                                          float4* __restrict__ slots) {
  __shared__ int lists[kWavesPerTile][kListSlots];
  const int b = blockIdx.z / parts, part = blockIdx.z % parts;
  if (starts[b] == starts[b + 1] || crowded[starts[b]]) return;
  const int tx0 = blockIdx.x * kTile, ty0 = blockIdx.y * kTile;
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, kq = lane >> 4, ij = lane & 15;
  int* list = lists[wave];
  const int r = sp.r, H = sp.H;
  const float4* dimg = reinterpret_cast<const float4*>(d_img) + (int64_t)b * H * H;
  float d[4][4];  // [row block][channel]
  bool odd_pixel = false;
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    const int iy = ty0 + 4 * kb + kq, ix = tx0 + ij;
    const float4 q = iy < H && ix < H ? dimg[(int64_t)iy * H + ix] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    d[kb][0] = q.x;
    d[kb][1] = q.y;
    d[kb][2] = q.z;
    d[kb][3] = q.w;
    odd_pixel = odd_pixel || !(isfinite(q.x) && isfinite(q.y) && isfinite(q.z) && isfinite(q.w));
  }
  const bool odd_tile = __ballot(odd_pixel) != 0;

  auto slot_of = [&](int p, int2 at) {
    const int sx = (int)blockIdx.x - first_tile(at.x, r), sy = (int)blockIdx.y - first_tile(at.y, r);
    return ((int64_t)p * (side * side) + sy * side + sx) * 2;
  };
  auto multiply = [&](int count) {
    int np = list[min(ij, count - 1)];  // the next group's, in flight
    int2 nat = rec.centre[np];
    float2 nf = rec.frac[np];
    float4 nc = rec.col[np];
    for (int e = 0; e < count; e += 16) {
      const bool live = e + ij < count;
      const int p = np;
      const int2 at = nat;
      const float2 f = nf;
      const float4 c = nc;
      if (e + 16 < count) {
        np = list[min(e + 16 + ij, count - 1)];
        nat = rec.centre[np];
        nf = rec.frac[np];
        nc = rec.col[np];
      }
      const bool odd = live && !(isfinite(c.x) && isfinite(c.y) && isfinite(c.z));
      if (odd_tile || __ballot(odd) != 0) {
        for (int u = e; u < min(e + 16, count); ++u) {  // uniform
          const int pu = list[u];
          const int2 au = rec.centre[pu];
          const float2 fu = rec.frac[pu];
          const float4 cu = rec.col[pu];
          PatchSums t;
#pragma unroll
          for (int kb = 0; kb < 4; ++kb) {
            const int iy = ty0 + 4 * kb + kq, ix = tx0 + ij, qy = iy - au.y, qx = ix - au.x;
            if (iy < H && ix < H && qx >= -r && qx <= r && qy >= -r && qy <= r) {
              const float ax = (float)qx - fu.x, ay = (float)qy - fu.y;
              const float g = gauss(ax, ay, sp.inv_two_s2);
              const float G = cu.x * d[kb][0] + cu.y * d[kb][1] + cu.z * d[kb][2] + d[kb][3];
              t.dr += g * d[kb][0];
              t.dg += g * d[kb][1];
              t.db += g * d[kb][2];
              t.gg += G * g;
              t.ggx += G * g * ax;
              t.ggy += G * g * ay;
            }
          }
          t.dr = wave_sum(t.dr);
          t.dg = wave_sum(t.dg);
          t.db = wave_sum(t.db);
          t.gg = wave_sum(t.gg);
          t.ggx = wave_sum(t.ggx);
          t.ggy = wave_sum(t.ggy);
          if (lane == 0) {
            float4* o = slots + slot_of(pu, au);
            o[0] = make_float4(t.dr, t.dg, t.db, t.gg);
            o[1] = make_float4(t.ggx, t.ggy, 0.0f, 0.0f);
          }
        }
        continue;
      }
      f32x4 T[4], Y[4];
#pragma unroll
      for (int ch = 0; ch < 4; ++ch) T[ch] = Y[ch] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const int qy = ty0 + 4 * kb + kq - at.y;
        const float ay = (float)qy - f.y;
        const float w = gauss(ay, 0.0f, sp.inv_two_s2);
        const float gy = qy >= -r && qy <= r ? w : 0.0f;
        const float gya = gy * ay;
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) {
          T[ch] = mfma_16x16x4(d[kb][ch], gy, T[ch]);
          Y[ch] = mfma_16x16x4(d[kb][ch], gya, Y[ch]);
        }
      }
      PatchSums t;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int qx = tx0 + 4 * kq + v - at.x;
        // not a zero weight: a column outside the patch may overflow
        if (qx < -r || qx > r) continue;
        const float ax = (float)qx - f.x;
        const float gx = gauss(ax, 0.0f, sp.inv_two_s2);
        const float U = c.x * T[0][v] + c.y * T[1][v] + c.z * T[2][v] + T[3][v];
        const float V = c.x * Y[0][v] + c.y * Y[1][v] + c.z * Y[2][v] + Y[3][v];
        t.dr += gx * T[0][v];
        t.dg += gx * T[1][v];
        t.db += gx * T[2][v];
        t.gg += gx * U;
        t.ggx += gx * ax * U;
        t.ggy += gx * V;
      }
      float* s[6] = {&t.dr, &t.dg, &t.db, &t.gg, &t.ggx, &t.ggy};
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        *s[k] += __shfl_xor(*s[k], 16, 64);
        *s[k] += __shfl_xor(*s[k], 32, 64);
      }
      if (live && kq < 2)
        slots[slot_of(p, at) + kq] =
            kq == 0 ? make_float4(t.dr, t.dg, t.db, t.gg) : make_float4(t.ggx, t.ggy, 0.0f, 0.0f);
    }
  };
  for_tile_particles(rec, r, starts[b], starts[b + 1], tx0, ty0, part * kWavesPerTile + wave, parts * kWavesPerTile,
                     list, multiply);
}

// Adds a particle's records (L lanes a particle, lane l the slots l, l + L,
// ... of the tiles its patch reaches) and turns them into gradients.  In
// crowded images, which the tiles left out, the wave sweeps the patches of its
// 64 / L particles instead, one after the other.
template <int L>
__global__ __launch_bounds__(256) void k_splat_backward_sum(SplatParams sp, SplatRecords rec,
                                                            const int32_t* __restrict__ starts, int images, int64_t n,
                                                            int side, const float* __restrict__ d_img,
                                                            const int* __restrict__ crowded,
                                                            const float4* __restrict__ slots,
                                                            float* __restrict__ d_x, float* __restrict__ d_color) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) / L;
  const int lane = threadIdx.x % L, group = threadIdx.x % 64 / L;
  const int2 at = i < n ? rec.centre[i] : make_int2(kNoPatch, 0);
  const float2 f = i < n ? rec.frac[i] : make_float2(0.0f, 0.0f);
  const bool live = at.x != kNoPatch;
  const int image = live ? image_of(starts, images, (int)i) : 0;
  const bool sweep = live && crowded[starts[image]] != 0;
  PatchSums t;
  AxisSums a;
  if (live && !sweep) {
    const int fx = first_tile(at.x, sp.r), fy = first_tile(at.y, sp.r);
    const int nx = last_tile(at.x, sp.r, sp.H) - fx + 1, ny = last_tile(at.y, sp.r, sp.H) - fy + 1;
    for (int k = lane; k < side * side; k += L) {
      if (k % side < nx && k / side < ny) {
        const float4* o = slots + (i * side * side + k) * 2;
        const float4 u = o[0], v = o[1];
        t.dr += u.x;
        t.dg += u.y;
        t.db += u.z;
        t.gg += u.w;
        t.ggx += v.x;
        t.ggy += v.y;
      }
    }
  }
  if (live && sp.normalize) a = axis_sums(sp, f.x, f.y, lane, L);
  const uint64_t sweeps = __ballot(sweep);
  for (int u = 0; u < 64 / L; ++u) {
    if (((sweeps >> (L * u)) & 1ull) == 0) continue;  // wave-uniform
    const int64_t iu = i - group + u;
    const int2 au = rec.centre[iu];
    const float2 fu = rec.frac[iu];
    const float4 cu = rec.col[iu];
    const int bu = __shfl(image, L * u, 64);
    const PatchSums w = sweep_patch(sp, au.x, au.y, fu.x, fu.y, cu.x, cu.y, cu.z,
                                    reinterpret_cast<const float4*>(d_img) + (int64_t)bu * sp.H * sp.H,
                                    threadIdx.x % 64);
    if (group == u && lane == 0) t = w;  // the group adds its lanes' below
  }
  float* s[10] = {&t.dr, &t.dg, &t.db, &t.gg, &t.ggx, &t.ggy, &a.sx, &a.sy, &a.sxa, &a.sya};
#pragma unroll
  for (int k = 0; k < 10; ++k) {
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) *s[k] += __shfl_xor(*s[k], o, L);
  }
  if (i < n) store_gradients(sp, i, live, t, a, lane, L, d_x, d_color);
}

// The tile by tile backward serves patches up to kTilesMaxRadius whose pixels
// outweigh the search (every tile looks at every particle of its image) and
// with kTilesMinPixels of them in all its two further launches, with at most
// kTilesMaxBytes of records.  Measured (us of the whole call, tiles against a
// wave a particle; 4096 particles an image): 8 x 256^2 at radius 10 (14 M
// pixels, search above) 41 and 39, at 16 (36 M) 58 and 59, at 20 (55 M) 63 and
// 76, at 32 (138 M) 91 and 163; 8 x 128^2 at 20 59 and 71; 1 x 512^2 at 32 (17
// M) 45 and 37.
// Of those images it takes the ones at least kTilesMinShare of whose tiles do
// the work (k_splat_backward_prep): in the others most of the chip waits for
// the few tiles' waves.  Tiles against waves, shares .48-.56: 103-113 and
// 148-156 (radius 32, 128^2); .45: 108 and 70 (10, 64^2); .33: 80 and 65 (20,
// 128^2); .16: 110 and 65 (20, 256^2); .04: 397 and 156 (32, 512^2); .06: 203
// and 70 (10, 128^2, 100 000 particles), now 83.  An image that is left to the
// waves pays the look and the empty launch, 8 to 12 us up to 32 768 particles.
constexpr int kTilesMaxRadius = 32;
constexpr int64_t kTilesMinPixels = (int64_t)1 << 25;
constexpr int64_t kTilesMaxBytes = (int64_t)1 << 30;
constexpr uint64_t kTilesBlocks = 4096;

// Tiles an axis that a patch can reach.
int tile_side(int r) { return (2 * r + kTile - 1) / kTile + 1; }

}  // namespace

int64_t splat_tiles_bytes(const SplatParams& sp, int64_t n) {
  const int64_t tiles = (sp.H + kTile - 1) / kTile, side = tile_side(sp.r), patch = 2 * sp.r + 1;
  const int64_t bytes = n * (32 * (1 + side * side) + 4);
  return sp.r <= kTilesMaxRadius && n * patch * patch >= kTilesMinPixels && 2 * tiles * tiles <= patch * patch &&
                 bytes <= kTilesMaxBytes
             ? bytes
             : 0;
}

void run_splat_forward(const SplatParams& sp, const float* x, const float* color, const int32_t* starts, int images,
                       int64_t n, void* work, float* out, hipStream_t st) {
  if (images == 0 || sp.H == 0) return;
  const SplatRecords rec(work, n);
  if (n > 0) {
    hipLaunchKernelGGL(k_splat_prep, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, sp, x, color, n, rec);
    SPHOPS_LAUNCHED();
  }
  const dim3 grid((uint32_t)((sp.H + kTile - 1) / kTile), (uint32_t)((sp.H + kTile - 1) / kTile), (uint32_t)images);
  hipLaunchKernelGGL(k_splat_forward, grid, dim3(kTileThreads), 0, st, sp, rec, starts, out);
  SPHOPS_LAUNCHED();
}

void run_splat_backward(const SplatParams& sp, const float* x, const float* color, const int32_t* starts, int images,
                        int64_t n, const float* d_img, float* d_x, float* d_color, void* work, hipStream_t st) {
  if (n == 0) return;
  if (work == nullptr || splat_tiles_bytes(sp, n) == 0) {
    const dim3 grid((uint32_t)((n + kBwdWaves - 1) / kBwdWaves));
    hipLaunchKernelGGL(k_splat_backward, grid, dim3(64 * kBwdWaves), 0, st, sp, x, color, starts, images, n, d_img,
                       d_x, d_color);
    SPHOPS_LAUNCHED();
    return;
  }
  SplatParams raw = sp;
  raw.normalize = 0;  // the colours themselves
  const SplatRecords rec(work, n);
  float4* slots = static_cast<float4*>(work) + 2 * n;
  const uint32_t tiles = (uint32_t)((sp.H + kTile - 1) / kTile);
  const int side = tile_side(sp.r);
  int* crowded = reinterpret_cast<int*>(slots + 2 * n * side * side);
  hipLaunchKernelGGL(k_splat_backward_prep, dim3((uint32_t)((n + 255) / 256 + images)), dim3(256), 0, st, raw, x,
                     color, starts, images, n, rec, crowded);
  SPHOPS_LAUNCHED();
  const uint64_t blocks = (uint64_t)tiles * tiles * (uint64_t)images;
  // enough parts to fill the chip, each wave with two turns or more
  const uint64_t most = std::max<uint64_t>(1, (uint64_t)n / (uint64_t)images / (64 * 2 * kWavesPerTile));
  const int parts = (int)std::min<uint64_t>({most, std::max<uint64_t>(1, kTilesBlocks / blocks),
                                             65535ull / (uint64_t)images});
  hipLaunchKernelGGL(k_splat_backward_tiles, dim3(tiles, tiles, (uint32_t)(images * parts)), dim3(kTileThreads), 0,
                     st, sp, rec, starts, parts, side, d_img, crowded, slots);
  SPHOPS_LAUNCHED();
  // few particles: more waves for a crowded image's sweeps (16 x 1024 of radius
  // 32, 256^2, in the same tiles: 101 us with 16 lanes a particle, 89 with 64,
  // where an even cloud's sum takes 7 longer; 32 between them)
#define SPHOPS_SPLAT_SUM(L)                                                                                       \
  hipLaunchKernelGGL(k_splat_backward_sum<L>, dim3((uint32_t)((n * L + 255) / 256)), dim3(256), 0, st, sp, rec,  \
                     starts, images, n, side, d_img, crowded, slots, d_x, d_color)
  if (n <= 1 << 14) SPHOPS_SPLAT_SUM(32);
  else SPHOPS_SPLAT_SUM(16);
#undef SPHOPS_SPLAT_SUM
  SPHOPS_LAUNCHED();
}

}  // namespace sphops
