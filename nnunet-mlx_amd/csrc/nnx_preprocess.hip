// Raw-case preprocessing on the device: nonzero crop bounds, crop + transpose + per-channel
// normalisation, and the spline resampling of image data to the plans' spacing.
//
// Replaces the host steps of preprocess_raw_case (src/nnunet_mlx/data/preprocessing.py:63-163):
// the crop bounds of crop_to_nonzero (:166-214; no mask, as CT normalisation uses none),
// the CTNormalization branch of _normalize_channel (:274-285), and the data resize of
// resample_probabilities_or_data for spline plans (src/nnunet_mlx/data/resampling.py:87-172,
// 268-306, 379-442, 476-501), which the reference delegates to scikit-image's
// resize(order, mode="edge", anti_aliasing=False): scipy.ndimage.zoom in grid mode with
// edge extension, then a clip to the input's [min, max].
//
// Spline arithmetic (float64 throughout, no contraction):
//   * every resized axis extended by 12 edge samples, then reflected about the padded ends
//     (SciPy pads this way before building coefficients for edge extension);
//   * order 3: per axis in turn, per line: gain (1 - z)(1 - 1/z), causal recursion c[i] += z c[i-1],
//     anticausal recursion c[i] = z (c[i+1] - c[i]), pole z = sqrt(3) - 2, each started where what
//     lies before it is below float64 resolution;
//   * evaluation one axis at a time: output index o samples the padded coordinate
//     cc = (o + 0.5) * n_in / n_out - 0.5 + 12 with the cardinal cubic B-spline weights of
//     t = cc - floor(cc) at floor(cc) - 1 .. floor(cc) + 2 (order 1: 1 - t, t at floor(cc),
//     floor(cc) + 1), summed from 0 in tap order;
//   * whole volume: cast to float32, clip to the channel's input [min, max]; separate axis:
//     the other two axes resized per plane (float64, clipped to the plane's [min, max]),
//     then the separate axis by half-pixel nearest indices floor(old/new (o + 0.5) - 0.5 +
//     0.5) clamped, cast to float32 once.
// Roofline: HBM — order 3 reads and writes each axis's float64 volume once (order 1 also an edge
// copy); the crop/normalise pass reads and writes 4 B per kept voxel.  A CT of 120 x 512 x 512 to
// 300 x 534 x 534 by order 3 with a separate axis: 2.68 -> 0.86 ms per case; prefilter and
// interpolation 1.54 -> 0.42 ms with the plane copies included (strided pass 0.27 ms, contiguous
// pass 0.15 ms at 4 TB/s), bounds 0.20 -> 0.04, crop 0.13 -> 0.04.

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>

#include "nnx_internal.h"

namespace nnx {
namespace {

constexpr int kSplinePad = 12;
constexpr int kMinmaxParts = 16;  // blocks per plane of the min/max reduction

// ---- nonzero bounds -------------------------------------------------------------------

__global__ void bbox_init_kernel(int* bbox) {
  if (threadIdx.x < 3) {
    bbox[2 * threadIdx.x] = INT_MAX;
    bbox[2 * threadIdx.x + 1] = -1;
  }
}

// bbox[2a] / bbox[2a + 1] = smallest / largest index along axis a of a voxel where any
// channel is nonzero.  One wave per (x, y) row at a time, its lanes along z (coalesced), eight
// loads in flight: of a row, or of as many rows where 64 lanes hold one.  The bounds along z stay
// in the lanes until the end; block minima and maxima reach memory by one vector atomic each.
// Bound by latency: 8 M voxels in rows of 3, 8, 40, 160 and 512: 250, 100, 32, 37 and 32 us (367,
// 212, 195, 192 and 94 with a load in flight and an atomic of every block; 850, 307, 71, 38 and 32
// while eight loads went to a row however short it is).
__global__ __launch_bounds__(256) void bbox_kernel(const float* __restrict__ x, int C, int64_t X,
                                                   int64_t Y, int64_t Z, int* bbox) {
  __shared__ int red[6][4];
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {-1, -1, -1};
  const int64_t n = X * Y * Z, rows = X * Y;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int64_t waves = (int64_t)gridDim.x * 4;
  const int64_t first = blockIdx.x * (int64_t)4 + wave;
  auto row_found = [&](int64_t r) {  // uniform over the wave
    const int rx = (int)(r / Y), ry = (int)(r - rx * Y);
    lo[0] = min(lo[0], rx);
    hi[0] = max(hi[0], rx);
    lo[1] = min(lo[1], ry);
    hi[1] = max(hi[1], ry);
  };
  if (Z <= 64) {
    const bool in = lane < Z;
    for (int64_t r = first; r < rows; r += 8 * waves) {
      bool nz[8] = {};
      for (int c = 0; c < C; ++c) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          v[j] = x[c * n + min(r + j * waves, rows - 1) * Z + (in ? lane : 0)];
#pragma unroll
        for (int j = 0; j < 8; ++j) nz[j] |= v[j] != 0.f;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const bool found = in && nz[j];
        if (r + j * waves < rows && __any(found)) row_found(r + j * waves);
        // (past the last row it is the last row again)
        if (found) {
          lo[2] = min(lo[2], lane);
          hi[2] = max(hi[2], lane);
        }
      }
    }
  } else {
    for (int64_t r = first; r < rows; r += waves) {
      const float* row = x + r * Z;
      bool any = false;
      for (int64_t z0 = lane; z0 < Z; z0 += 8 * 64) {
        bool nz[8] = {};
        for (int c = 0; c < C; ++c) {
          float v[8];
#pragma unroll
          for (int j = 0; j < 8; ++j)
            v[j] = row[(int64_t)c * n + (z0 + j * 64 < Z ? z0 + j * 64 : z0)];
#pragma unroll
          for (int j = 0; j < 8; ++j) nz[j] |= v[j] != 0.f;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (nz[j] && z0 + j * 64 < Z) {
            lo[2] = min(lo[2], (int)(z0 + j * 64));
            hi[2] = max(hi[2], (int)(z0 + j * 64));
            any = true;
          }
      }
      if (__any(any)) row_found(r);
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    lo[2] = min(lo[2], __shfl_xor(lo[2], o));
    hi[2] = max(hi[2], __shfl_xor(hi[2], o));
  }
  if (lane == 0)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      red[2 * a][wave] = lo[a];
      red[2 * a + 1][wave] = hi[a];
    }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int k = threadIdx.x;
    int v = red[k][0];
    for (int w = 1; w < 4; ++w) v = (k & 1) ? max(v, red[k][w]) : min(v, red[k][w]);
    // Only a bound that moves the box goes to memory (a stale read costs an atomic, never a
    // bound): the six addresses serialise, and 8192 blocks' atomics took 195 us of which the
    // reads of 120 x 512 x 512 floats need 25.
    const int now = __hip_atomic_load(&bbox[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (k & 1) {
      if (v > now) atomicMax(&bbox[k], v);
    } else if (v < now) {
      atomicMin(&bbox[k], v);
    }
  }
}

// ---- crop + transpose + normalise -------------------------------------------------------

constexpr int kMaxNormChannels = 16;

struct ChannelNorms {
  int scheme[kMaxNormChannels];  // NNX_NORM_*
  float mean[kMaxNormChannels], std[kMaxNormChannels];  // std already max(std, 1e-8)
  float lower[kMaxNormChannels], upper[kMaxNormChannels];
};

// ---- filled nonzero mask ----------------------------------------------------------------
// Cells of the crop box (E0, E1, E2) of the raw volume: 2 = some channel nonzero, 1 =
// background reached from the box border through background (6-connected), 0 = background
// not reached yet.  After the sweeps converge the filled mask is cell != 1.

__global__ __launch_bounds__(256) void mask_init_kernel(const float* __restrict__ x, int C,
                                                        int64_t X, int64_t Y, int64_t Z,
                                                        int64_t b0, int64_t b1, int64_t b2,
                                                        int64_t E0, int64_t E1, int64_t E2,
                                                        uint8_t* __restrict__ cell) {
  const int64_t n = X * Y * Z, total = E0 * E1 * E2;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i2 = e % E2, i1 = (e / E2) % E1, i0 = e / (E1 * E2);
    const int64_t src = ((b0 + i0) * Y + (b1 + i1)) * Z + (b2 + i2);
    bool nz = false;
    for (int c = 0; c < C; ++c) nz |= x[(int64_t)c * n + src] != 0.f;
    const bool border = i0 == 0 || i1 == 0 || i2 == 0 || i0 == E0 - 1 || i1 == E1 - 1 ||
                        i2 == E2 - 1;
    cell[e] = nz ? 2 : (border ? 1 : 0);
  }
}

// Propagate "reached" along every line of `axis` in both directions (one thread per line;
// for axes 0 and 1 neighbouring threads hold neighbouring lines).  *changed = 1 when a
// cell changed.
__global__ __launch_bounds__(256) void mask_sweep_kernel(uint8_t* __restrict__ cell, int64_t E0,
                                                         int64_t E1, int64_t E2, int axis,
                                                         int* __restrict__ changed) {
  const int64_t dims[3] = {E0, E1, E2};
  const int64_t strides[3] = {E1 * E2, E2, 1};
  const int64_t len = dims[axis], stride = strides[axis];
  const int64_t lines = E0 * E1 * E2 / len;
  const int64_t line = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (line >= lines) return;
  int64_t base;
  if (axis == 2) base = line * E2;
  else if (axis == 1) base = (line / E2) * E1 * E2 + line % E2;
  else base = line;
  bool any = false, carry = false;
  for (int64_t i = 0; i < len; ++i) {
    uint8_t& v = cell[base + i * stride];
    if (v == 2) carry = false;
    else if (v == 1) carry = true;
    else if (carry) { v = 1; any = true; }
  }
  carry = false;
  for (int64_t i = len - 1; i >= 0; --i) {
    uint8_t& v = cell[base + i * stride];
    if (v == 2) carry = false;
    else if (v == 1) carry = true;
    else if (carry) { v = 1; any = true; }
  }
  if (any) *changed = 1;
}

__global__ void flag_clear_kernel(int* flag) { *flag = 0; }

__global__ __launch_bounds__(256) void mask_finish_kernel(uint8_t* __restrict__ cell, int64_t n) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x)
    cell[e] = cell[e] != 1;
}

// ---- channel extrema over the crop box ----------------------------------------------------

__global__ __launch_bounds__(256) void box_minmax_partial_kernel(
    const float* __restrict__ xc, int64_t Y, int64_t Z, int64_t b0, int64_t b1, int64_t b2,
    int64_t E0, int64_t E1, int64_t E2, float2* __restrict__ partial) {
  __shared__ float smin[4], smax[4];
  const int64_t total = E0 * E1 * E2;
  float lo = INFINITY, hi = -INFINITY;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i2 = e % E2, i1 = (e / E2) % E1, i0 = e / (E1 * E2);
    const float v = xc[((b0 + i0) * Y + (b1 + i1)) * Z + (b2 + i2)];
    lo = fminf(lo, v);
    hi = fmaxf(hi, v);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, o));
    hi = fmaxf(hi, __shfl_xor(hi, o));
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    smin[wave] = lo;
    smax[wave] = hi;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    partial[blockIdx.x] = make_float2(fminf(fminf(smin[0], smin[1]), fminf(smin[2], smin[3])),
                                      fmaxf(fmaxf(smax[0], smax[1]), fmaxf(smax[2], smax[3])));
}

__global__ __launch_bounds__(64) void box_minmax_final_kernel(const float2* __restrict__ partial,
                                                             int parts, float* __restrict__ out) {
  float lo = INFINITY, hi = -INFINITY;
  for (int i = threadIdx.x; i < parts; i += 64) {
    lo = fminf(lo, partial[i].x);
    hi = fmaxf(hi, partial[i].y);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, o));
    hi = fmaxf(hi, __shfl_xor(hi, o));
  }
  if (threadIdx.x == 0) {
    out[0] = lo;
    out[1] = hi;
  }
}

// ---- z-score statistics -----------------------------------------------------------------
// Per block: float64 sums over the crop box of channel c (mask cells only when `mask`),
// pass 0: (sum x, count), pass 1: (sum (x - mean32)^2, count) with mean32 = stats[2c].

constexpr int kStatBlocks = 1024;

__global__ __launch_bounds__(256) void zscore_partial_kernel(
    const float* __restrict__ xc, int64_t Y, int64_t Z, int64_t b0, int64_t b1, int64_t b2,
    int64_t E0, int64_t E1, int64_t E2, const uint8_t* __restrict__ mask, int pass,
    const float* __restrict__ stats, double2* __restrict__ partial) {
  __shared__ double ssum[4], scnt[4];
  const int64_t total = E0 * E1 * E2;
  const double mean = pass ? (double)stats[0] : 0.0;
  double acc = 0.0, cnt = 0.0;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    if (mask && !mask[e]) continue;
    const int64_t i2 = e % E2, i1 = (e / E2) % E1, i0 = e / (E1 * E2);
    const double v = (double)xc[((b0 + i0) * Y + (b1 + i1)) * Z + (b2 + i2)];
    acc += pass ? (v - mean) * (v - mean) : v;
    cnt += 1.0;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    acc += __shfl_xor(acc, o);
    cnt += __shfl_xor(cnt, o);
  }
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    ssum[wave] = acc;
    scnt[wave] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    partial[blockIdx.x] = make_double2(ssum[0] + ssum[1] + ssum[2] + ssum[3],
                                       scnt[0] + scnt[1] + scnt[2] + scnt[3]);
}

// stats[0] = float(sum / n) (pass 0) or stats[1] = float(sqrt(sum / n)) (pass 1); a fixed
// summation order over the partials, so the result is deterministic
__global__ __launch_bounds__(64) void zscore_final_kernel(const double2* __restrict__ partial,
                                                         int parts, int pass,
                                                         float* __restrict__ stats) {
  double acc = 0.0, cnt = 0.0;
  for (int i = threadIdx.x; i < parts; i += 64) {
    acc += partial[i].x;
    cnt += partial[i].y;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    acc += __shfl_xor(acc, o);
    cnt += __shfl_xor(cnt, o);
  }
  if (threadIdx.x == 0) {
    const double m = cnt > 0 ? acc / cnt : NAN;
    if (pass == 0) stats[0] = (float)m;
    else stats[1] = (float)sqrt(m);
  }
}

// A channel's normalisation.  `inside` (whether the filled mask is set at the value) is asked for by
// the masked scheme only.
struct ChannelNorm {
  int scheme;
  float mean, std, lower, upper;
  __device__ ChannelNorm(const ChannelNorms& n, int c)
      : scheme(n.scheme[c]), mean(n.mean[c]), std(n.std[c]), lower(n.lower[c]), upper(n.upper[c]) {}
  template <class F>
  __device__ __forceinline__ float operator()(float v, F&& inside) const {
    if (scheme == NNX_NORM_CT) {
      v = fminf(fmaxf(v, lower), upper);
      v = __fdiv_rn(__fsub_rn(v, mean), std);
    } else if (scheme == NNX_NORM_ZSCORE || (scheme == NNX_NORM_ZSCORE_MASKED && inside())) {
      v = __fdiv_rn(__fsub_rn(v, mean), std);
    }
    return v;
  }
};

// out[c][o0][o1][o2] = norm_c(x[c][r0][r1][r2]) with r[t_k] = s_k + o_k: out axis k is input
// axis t_k, cropped to start s_k.  NNX_NORM_ZSCORE_MASKED normalises only where the filled
// mask (a box of the raw axes) is set.  `in` and `mask` point at the window's first voxel of
// channel 0; strides by out axis.
struct CropArgs {
  const float* in;
  const uint8_t* mask;
  float* out;
  int channels;
  int64_t in_channel;
  int64_t n[3], in_stride[3], mask_stride[3];
  ChannelNorms norms;
};

// A thread a voxel, for short rows: in 8 M voxels 34 us whatever their length (the index
// arithmetic bounds it), where a wave a row takes 377 us at 8 voxels, 37 at 64, 35 at 72, 31 at
// 80, 22 at 128 and 12 at 512 (5.2 TB/s).
__global__ __launch_bounds__(256) void crop_normalize_kernel(CropArgs a) {
  const int64_t per = a.n[0] * a.n[1] * a.n[2];
  const int64_t total = per * a.channels;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int c = (int)(e / per);
    const int64_t p = e - c * per;
    const int64_t o2 = p % a.n[2], o1 = (p / a.n[2]) % a.n[1], o0 = p / (a.n[1] * a.n[2]);
    const float v = a.in[c * a.in_channel + o0 * a.in_stride[0] + o1 * a.in_stride[1] + o2 * a.in_stride[2]];
    a.out[e] = ChannelNorm(a.norms, c)(v, [&] {
      return a.mask[o0 * a.mask_stride[0] + o1 * a.mask_stride[1] + o2 * a.mask_stride[2]] != 0;
    });
  }
}

// Rows of kRowForm voxels and more that are contiguous on both sides, a wave a row at a time: the
// index arithmetic is per row, and eight loads of a lane are in flight.
constexpr int64_t kRowForm = 80;

__global__ __launch_bounds__(256) void crop_normalize_rows_kernel(CropArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t n2 = a.n[2], rows = a.n[0] * a.n[1] * a.channels;
  for (int64_t r = blockIdx.x * (int64_t)4 + (threadIdx.x >> 6); r < rows;
       r += (int64_t)gridDim.x * 4) {
    const int64_t o1 = r % a.n[1], rest = r / a.n[1];
    const int64_t o0 = rest % a.n[0];
    const int c = (int)(rest / a.n[0]);
    const float* src = a.in + c * a.in_channel + o0 * a.in_stride[0] + o1 * a.in_stride[1];
    const uint8_t* msrc = a.mask + o0 * a.mask_stride[0] + o1 * a.mask_stride[1];
    float* dst = a.out + r * n2;
    const ChannelNorm norm(a.norms, c);
    for (int64_t o = lane; o < n2; o += 8 * 64) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = src[o + j * 64 < n2 ? o + j * 64 : o];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int64_t oj = o + j * 64;
        if (oj >= n2) break;
        dst[oj] = norm(v[j], [&] { return msrc[oj] != 0; });
      }
    }
  }
}

// Transposed rows: the raw rows are out axis A (0 or 1).  A workgroup moves tiles of TA voxels of it
// by 64 of out axis 2 through LDS, read along the one and written along the other (TA = 64, or
// the next power of two from 16 on that holds a short axis).  Bound by HBM: 160 x 512 x 512 with
// its axes in reverse 74 us (4.5 TB/s), where reads that stride over the raw rows took 212 us (a
// thread a voxel) and 468 (a wave a row), both at the mercy of the caches; 40 x 512 x 512 likewise
// 24, 54 and 163 us.  Out rows below kTileForm voxels fill too little of a tile's 64: 700 x 16 x
// 700 to rows of 16, 40 us against 35 a thread a voxel, of 20, 40 against 43.
constexpr int64_t kTileForm = 20;

template <int A, int TA>
__global__ __launch_bounds__(256) void crop_normalize_tiles_kernel(CropArgs a) {
  constexpr int B = 1 - A, kPer = TA * 64 / 256;
  __shared__ float tile[64][TA + 1];
  const int64_t na = a.n[A], nb = a.n[B], n2 = a.n[2];
  const int64_t ta = (na + TA - 1) / TA, t2 = (n2 + 63) / 64, total = ta * t2 * nb * a.channels;
  const int64_t out_stride[2] = {a.n[1] * n2, n2};
  for (int64_t t = blockIdx.x; t < total; t += gridDim.x) {
    const int64_t a0 = t % ta * TA, rest = t / ta;
    const int64_t j0 = rest % t2 * 64, plane = rest / t2;
    const int64_t b = plane % nb;
    const int c = (int)(plane / nb);
    const float* src = a.in + c * a.in_channel + b * a.in_stride[B];
    const uint8_t* msrc = a.mask + b * a.mask_stride[B];
    const ChannelNorm norm(a.norms, c);
    float v[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int l = i * 256 + (int)threadIdx.x;
      v[i] = src[min(a0 + l % TA, na - 1) + min(j0 + l / TA, n2 - 1) * a.in_stride[2]];
    }
    __syncthreads();  // the last tile is read
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int l = i * 256 + (int)threadIdx.x;
      tile[l / TA][l % TA] = norm(v[i], [&] {
        return msrc[min(a0 + l % TA, na - 1) + min(j0 + l / TA, n2 - 1) * a.mask_stride[2]] != 0;
      });
    }
    __syncthreads();
    float* dst = a.out + c * (a.n[0] * a.n[1] * n2) + b * out_stride[B];
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int la = i * 4 + (int)(threadIdx.x >> 6);
      if (a0 + la < na && j0 + lane < n2)
        dst[(a0 + la) * out_stride[A] + j0 + lane] = tile[lane][la];
    }
  }
}

// ---- spline resampling -----------------------------------------------------------------

// out (P0, P1, P2) float64 = in (n0, n1, n2) float32 edge-extended by p_a on each side of
// axis a.
__global__ __launch_bounds__(256) void pad_edge_kernel(const float* __restrict__ in, int64_t n0,
                                                       int64_t n1, int64_t n2, int p0, int p1,
                                                       int p2, double* __restrict__ out) {
  const int64_t P0 = n0 + 2 * p0, P1 = n1 + 2 * p1, P2 = n2 + 2 * p2;
  const int64_t total = P0 * P1 * P2;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i2 = e % P2, i1 = (e / P2) % P1, i0 = e / (P1 * P2);
    const int64_t j0 = min(max(i0 - p0, (int64_t)0), n0 - 1);
    const int64_t j1 = min(max(i1 - p1, (int64_t)0), n1 - 1);
    const int64_t j2 = min(max(i2 - p2, (int64_t)0), n2 - 1);
    out[e] = (double)in[(j0 * n1 + j1) * n2 + j2];
  }
}

// ---- order 3: one axis in one pass -------------------------------------------------------
//
// The cubic coefficients of a line are the two-sided exponential filter of its extension
// (pole z = sqrt(3) - 2, |z| = 0.27): padded by 12 edge samples, then reflected about the
// padded ends, as the initial values of the recursions over the padded line assume.  |z|^32 is
// 5e-19, below float64 resolution, so the recursions may start 32 samples outside any piece
// of a line: a wave takes a segment of kSeg source intervals of 64 lines, runs the causal
// recursion over it from 32 samples before, the anticausal one from 32 samples behind, and
// forms the outputs whose four taps lie in the segment as the coefficients come by.  So an axis
// costs one read and one write of the volume and every line is cut into independent pieces,
// where the padded copy, the two sweeps over it and the interpolation moved it eight times
// and ran whole lines serially.  Neither the padding nor the coefficients are stored.
// Roofline: HBM for the volumes; the recursions are a serial chain of two float64 operations a
// sample, which the number of waves has to cover (LDS allows 4 and 3 a CU; segments of 64
// would need a third less recomputation but 2 or 3 waves).
constexpr int kSeg = 32;                     // source intervals [f, f + 1) of a segment
constexpr int kWarm = 32;                    // samples a recursion starts outside
constexpr int kSweep = kSeg + 2 * kWarm + 3;  // samples of the causal recursion
constexpr int kKept = kSeg + kWarm + 3;       // causal values that the anticausal one reads

// Taps of output o of an axis: coefficients f - 1 .. f + 2 of the unpadded line.
struct SplineTap {
  double w[4];
  int64_t f;
};

__device__ __forceinline__ double spline_coord(int64_t o, double ratio) {
  return ((double)o + 0.5) * ratio - 0.5 + (double)kSplinePad;
}

__device__ __forceinline__ int64_t nearest_source(int64_t o, double ratio, int64_t n) {
  const double coord = ratio * ((double)o + 0.5) - 0.5;
  return min(max((int64_t)floor(coord + 0.5), (int64_t)0), n - 1);
}

__global__ __launch_bounds__(256) void spline_taps_kernel(int64_t N, double ratio,
                                                          SplineTap* __restrict__ taps) {
  const int64_t o = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (o >= N) return;
  const double cc = spline_coord(o, ratio);
  const double f = floor(cc);
  const double t = cc - f, u = 1.0 - t;
  SplineTap r;
  r.w[0] = u * u * u / 6.0;
  r.w[1] = 2.0 / 3.0 - t * t + t * t * t / 2.0;
  r.w[2] = 2.0 / 3.0 - u * u + u * u * u / 2.0;
  r.w[3] = t * t * t / 6.0;
  r.f = (int64_t)f - kSplinePad;
  taps[o] = r;
}

// the first output o of [0, N] with taps[o].f >= f (the coordinates ascend)
__device__ __forceinline__ int64_t first_with(const SplineTap* taps, int64_t N, double ratio,
                                              int64_t f) {
  int64_t o = (int64_t)fmin(fmax(((double)f + 0.5) / ratio - 1.5, 0.0), (double)N);
  while (o > 0 && taps[o - 1].f >= f) --o;
  while (o < N && taps[o].f < f) ++o;
  return o;
}

// the first output of [0, N] whose nearest source plane is >= k
__device__ __forceinline__ int64_t first_nearest(int64_t N, double ratio, int64_t n, int64_t k) {
  int64_t o = (int64_t)fmin(fmax((double)k / ratio - 1.5, 0.0), (double)N);
  while (o > 0 && nearest_source(o - 1, ratio, n) >= k) --o;
  while (o < N && nearest_source(o, ratio, n) < k) ++o;
  return o;
}

// index of sample p of the extended line
__device__ __forceinline__ int64_t extended(int64_t p, int64_t n) {
  while (p < -kSplinePad || p > n + kSplinePad - 1)
    p = p < -kSplinePad ? -2 * kSplinePad - 1 - p : 2 * (n + kSplinePad) - 1 - p;
  return min(max(p, (int64_t)0), n - 1);
}

struct SplineConst {
  double z, gain, start, turn;  // gain / (1 - z), z / (z - 1)
};

// Value of lane `l` (uniform) in every lane.
__device__ __forceinline__ int from_lane(int v, int l) { return __builtin_amdgcn_readlane(v, l); }
__device__ __forceinline__ double from_lane(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// The outputs [beg, end) of a segment from `s` on, last first, as a wave meets them: 64 taps at
// a time in the lanes' registers (a tap read from memory where it is used would put a load's
// latency behind every coefficient).
struct TapWalk {
  const SplineTap* taps;
  int64_t s, beg, at, base;  // next output; lane l holds output base + l
  int f;                     // its f - s
  double w[4];
  __device__ void load(int lane) {
    base = max(beg, at - 63);
    const SplineTap& t = taps[min(base + lane, at)];
    f = (int)(t.f - s);
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = t.w[e];
  }
  __device__ TapWalk(const SplineTap* t, int64_t seg, int64_t b, int64_t e, int lane)
      : taps(t), s(seg), beg(b), at(e - 1) {
    load(lane);
  }
  // emit(output, value) for every output whose coefficients are c0 .. c3 = s - 1 + q .. s + 2 + q
  template <class F>
  __device__ void step(int q, double c0, double c1, double c2, double c3, int lane, F&& emit) {
    while (at >= beg) {
      const int l = __builtin_amdgcn_readfirstlane((int)(at - base));
      if (from_lane(f, l) != q) return;
      double sum = 0.0 + c0 * from_lane(w[0], l);
      sum = sum + c1 * from_lane(w[1], l);
      sum = sum + c2 * from_lane(w[2], l);
      sum = sum + c3 * from_lane(w[3], l);
      emit(at, sum);
      --at;
      if (at >= beg && at < base) load(lane);
    }
  }
};

// Axis 0 or 1: in (outer, n, inner) -> out (outer, N, inner) float64, a lane a line, 64
// neighbouring lines a wave (coalesced).  Grid (inner / 64, segments, outer).  sep_n > 0: the
// outer index is the separate axis, and its planes that no output plane takes are left out.
template <class T>
__global__ __launch_bounds__(64) void spline_strided_kernel(
    const T* __restrict__ in, int64_t n, int64_t inner, const SplineTap* __restrict__ taps,
    int64_t N, double ratio, SplineConst k, int64_t outer, int64_t sep_n, int64_t sep_N,
    double sep_ratio, double* __restrict__ out) {
  __shared__ double kept[kKept][64];
  const int lane = threadIdx.x;
  const int64_t i = blockIdx.x * (int64_t)64 + lane;
  for (int64_t s = -1 + (int64_t)blockIdx.y * kSeg; s < n; s += (int64_t)gridDim.y * kSeg) {
    const int64_t o_beg = first_with(taps, N, ratio, s);
    const int64_t o_end = first_with(taps, N, ratio, s + kSeg);
    if (o_beg >= o_end) continue;
    // rows of the sweep's samples relative to its first row in the volume, held by the lanes
    const int64_t row0 = max(s - 1 - kWarm, (int64_t)0);
    const int rel0 = (int)(extended(s - 1 - kWarm + lane, n) - row0);
    const int rel1 = (int)(extended(s - 1 - kWarm + 64 + lane, n) - row0);
    for (int64_t ou = blockIdx.z; ou < outer; ou += gridDim.z) {
      if (sep_n > 0) {
        const int64_t first = first_nearest(sep_N, sep_ratio, sep_n, ou);
        if (first >= sep_N || nearest_source(first, sep_ratio, sep_n) != ou) continue;
      }
      const T* line = in + (ou * n + row0) * inner + (i < inner ? i : inner - 1);
      auto sample = [&](int q) {
        const int rel = q < 64 ? from_lane(rel0, q) : from_lane(rel1, q - 64);
        return line[rel * inner];
      };
      // the sweep in groups of samples, the next group's loads in flight
      constexpr int kGroup = 14, kGroups = (kSweep - 1) / kGroup;
      static_assert((kSweep - 1) % kGroup == 0, "the sweep is whole groups");
      double prev = (double)sample(0) * k.start;
      T v[2][kGroup];
#pragma unroll
      for (int g = 0; g < kGroup; ++g) v[0][g] = sample(1 + g);
#pragma unroll
      for (int j = 0; j < kGroups; ++j) {
        if (j + 1 < kGroups) {
#pragma unroll
          for (int g = 0; g < kGroup; ++g) v[(j + 1) & 1][g] = sample(1 + (j + 1) * kGroup + g);
        }
#pragma unroll
        for (int g = 0; g < kGroup; ++g) {
          const int q = 1 + j * kGroup + g;
          prev = (double)v[j & 1][g] * k.gain + k.z * prev;
          if (q >= kWarm) kept[q - kWarm][lane] = prev;
        }
      }
      double next = prev * k.turn;
#pragma unroll 10
      for (int q = kKept - 2; q > kSeg + 2; --q) next = k.z * (next - kept[q][lane]);
      // c0 .. c3 = coefficients s - 1 + q .. s + 2 + q, which the outputs with f = s + q take
      double c0 = 0.0, c1 = 0.0, c2 = 0.0, c3 = 0.0;
      TapWalk walk(taps, s, o_beg, o_end, lane);
      double* dst = out + ou * N * inner + i;
#pragma unroll 7
      for (int q = kSeg + 2; q >= 0; --q) {
        next = k.z * (next - kept[q][lane]);
        c3 = c2;
        c2 = c1;
        c1 = c0;
        c0 = next;
        walk.step(q, c0, c1, c2, c3, lane, [&](int64_t o, double sum) {
          if (i < inner) dst[o * inner] = sum;
        });
      }
    }
  }
}

// One order-1 interpolation pass along `axis`: in (I0, I1, I2) -> out with that axis n_out long.
// The axis holds n_in source samples padded by `pad` on each side.
__global__ __launch_bounds__(256) void interp_axis_kernel(const double* __restrict__ in,
                                                          int64_t I0, int64_t I1, int64_t I2,
                                                          int axis, int64_t n_out, double ratio,
                                                          int pad, double* __restrict__ out) {
  int64_t dims[3] = {I0, I1, I2};
  const int64_t in_stride = axis == 0 ? I1 * I2 : axis == 1 ? I2 : 1;
  dims[axis] = n_out;
  const int64_t total = dims[0] * dims[1] * dims[2];
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q2 = e % dims[2], q1 = (e / dims[2]) % dims[1], q0 = e / (dims[1] * dims[2]);
    const int64_t o = axis == 0 ? q0 : axis == 1 ? q1 : q2;
    // source element of tap 0 with the axis coordinate set to 0
    const int64_t row = axis == 0 ? q1 * I2 + q2 : axis == 1 ? q0 * I1 * I2 + q2
                                                             : (q0 * I1 + q1) * I2;
    const double cc = ((double)o + 0.5) * ratio - 0.5 + (double)pad;
    const double f = floor(cc);
    const double t = cc - f;
    double sum = 0.0;
    const int64_t start = (int64_t)f;
    sum = sum + in[row + start * in_stride] * (1.0 - t);
    sum = sum + in[row + (start + 1) * in_stride] * t;
    out[e] = sum;
  }
}

// Bounds of a set of samples without its NaN (+inf, -inf of an empty one), and whether it holds
// an infinity or a NaN.
struct Extrema {
  float lo, hi;
  int nonfinite;
};

// The bounds that resampled values are clipped to.  Order 3 (`spread`): the recursions carry an
// infinity or a NaN over its line, every line that crosses it and so on, so one of either makes
// every value of the resized axes NaN, of which the clip makes the lower bound.  The
// pieces that lines are cut into would end that at their ends: both bounds take its place.
__device__ __forceinline__ float2 clip_bounds(const Extrema& e, bool spread) {
  if (!spread || !e.nonfinite) return make_float2(e.lo, e.hi);
  const float v = fminf(e.lo, e.hi);
  return make_float2(v, v);
}

// part[k * parts + j] = bounds of part j of plane k along `axis` of a (n0, n1, n2)
// float32 channel; grid (planes, parts).
__global__ __launch_bounds__(256) void plane_minmax_kernel(const float* __restrict__ in,
                                                           int64_t n0, int64_t n1, int64_t n2,
                                                           int axis, Extrema* __restrict__ part) {
  __shared__ float smin[4], smax[4];
  __shared__ int sbad[4];
  const int64_t k = blockIdx.x;
  const int parts = gridDim.y, j = blockIdx.y;
  const int64_t dims[3] = {n0, n1, n2};
  const int a1 = axis == 0 ? 1 : 0, a2 = axis == 2 ? 1 : 2;
  const int64_t strides[3] = {n1 * n2, n2, 1};
  const int64_t m = dims[a1] * dims[a2];
  float lo = INFINITY, hi = -INFINITY;
  bool bad = false;
  for (int64_t i = j * (int64_t)blockDim.x + threadIdx.x; i < m; i += (int64_t)parts * blockDim.x) {
    const float v = in[k * strides[axis] + (i / dims[a2]) * strides[a1] + (i % dims[a2]) * strides[a2]];
    lo = fminf(lo, v);
    hi = fmaxf(hi, v);
    bad |= !isfinite(v);
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, o));
    hi = fmaxf(hi, __shfl_xor(hi, o));
  }
  const int wave = threadIdx.x >> 6;
  const bool any = __any(bad);
  if ((threadIdx.x & 63) == 0) {
    smin[wave] = lo;
    smax[wave] = hi;
    sbad[wave] = any;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) {
      lo = fminf(lo, smin[w]);
      hi = fmaxf(hi, smax[w]);
    }
    part[k * parts + j] = Extrema{lo, hi, sbad[0] | sbad[1] | sbad[2] | sbad[3]};
  }
}

// all[k] = bounds over part[k * parts .. k * parts + parts) and mm[k] = what plane k is clipped
// to, one thread per plane
__global__ __launch_bounds__(256) void plane_parts_kernel(const Extrema* __restrict__ part,
                                                          int64_t planes, int parts, bool spread,
                                                          Extrema* __restrict__ all,
                                                          float2* __restrict__ mm) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= planes) return;
  Extrema e{INFINITY, -INFINITY, 0};
  for (int j = 0; j < parts; ++j) {
    const Extrema& p = part[k * parts + j];
    e.lo = fminf(e.lo, p.lo);
    e.hi = fmaxf(e.hi, p.hi);
    e.nonfinite |= p.nonfinite;
  }
  all[k] = e;
  mm[k] = clip_bounds(e, spread);
}

// *mm = what the volume is clipped to, from the n planes' bounds
__global__ __launch_bounds__(64) void reduce_minmax_kernel(const Extrema* __restrict__ all,
                                                           int64_t n, bool spread, float2* mm) {
  float lo = INFINITY, hi = -INFINITY;
  bool bad = false;
  for (int64_t i = threadIdx.x; i < n; i += 64) {
    lo = fminf(lo, all[i].lo);
    hi = fmaxf(hi, all[i].hi);
    bad |= all[i].nonfinite != 0;
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, o));
    hi = fmaxf(hi, __shfl_xor(hi, o));
  }
  const bool any = __any(bad);
  if (threadIdx.x == 0) *mm = clip_bounds(Extrema{lo, hi, any}, spread);
}

// One rounding of a float64 result: to float32, or to float16 (nearest even) when HALF,
// returned as float32.
template <bool HALF>
__device__ inline float round_result(double v) {
  if constexpr (HALF) return (float)(_Float16)v;  // correctly rounded (integer sequence)
  else return (float)v;
}

// whole-volume resize: out = clip(round(v), min, max); the bounds are values of the input,
// so clipping before or after the monotone rounding gives the same result
template <bool HALF>
__global__ __launch_bounds__(256) void cast_clip_kernel(const double* __restrict__ in, int64_t n,
                                                        const float2* __restrict__ mm,
                                                        float* __restrict__ out) {
  const float2 b = *mm;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x)
    out[e] = fminf(fmaxf(round_result<HALF>(in[e]), b.x), b.y);
}

// separate axis: out[.. o ..] = round(clip_k(inter[.. k ..])), k = nearest source plane of o
template <bool HALF>
__global__ __launch_bounds__(256) void plane_clip_nearest_kernel(
    const double* __restrict__ inter, int64_t d0, int64_t d1, int64_t d2, int axis,
    int64_t n_new, double ratio, const float2* __restrict__ mm, float* __restrict__ out) {
  int64_t dims[3] = {d0, d1, d2};
  const int64_t n_old = dims[axis];
  const int64_t in_stride = axis == 0 ? d1 * d2 : axis == 1 ? d2 : 1;
  dims[axis] = n_new;
  const int64_t total = dims[0] * dims[1] * dims[2];
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t q2 = e % dims[2], q1 = (e / dims[2]) % dims[1], q0 = e / (dims[1] * dims[2]);
    const int64_t o = axis == 0 ? q0 : axis == 1 ? q1 : q2;
    const int64_t row = axis == 0 ? q1 * d2 + q2 : axis == 1 ? q0 * d1 * d2 + q2
                                                             : (q0 * d1 + q1) * d2;
    const double coord = ratio * ((double)o + 0.5) - 0.5;
    int64_t k = (int64_t)floor(coord + 0.5);
    k = min(max(k, (int64_t)0), n_old - 1);
    const float2 b = mm[k];
    const double v = fmin(fmax(inter[row + k * in_stride], (double)b.x), (double)b.y);
    out[e] = round_result<HALF>(v);
  }
}

// Axis 2, the last pass: rows of n float64 samples -> clipped and rounded rows of N floats.
// A wave takes a tile of a row, kLane consecutive samples a lane: each lane runs the recursions
// over its own samples from zero, and what its neighbours carry in is added afterwards
// (z^kLane times smaller per lane of distance: three lanes reach below float64 resolution).  So
// a row's chain is kLane steps instead of n, loads and stores are whole rows, and the LDS of a
// wave is its coefficients only.  Tiles overlap by kEdge samples on either side, where the
// values carried in from outside are not known.  With a separate axis (sep_n > 0), rows are
// (outer, k, mid) with k its source plane: the row is written to every output plane that takes
// plane k (planes[k] = first output, number), clipped to that plane's [min, max]; otherwise *mm
// bounds all.
constexpr int kLane = 10, kTile = 64 * kLane, kEdge = 4 * kLane;
constexpr int kTileF = kTile - 2 * kEdge - 4;  // values of f whose taps lie in a tile
constexpr int kRowsPerWave = 2;                // rows that share a read of the taps

struct SplinePowers {
  double z[kLane + 1];  // z^0 .. z^kLane
};

__global__ __launch_bounds__(256) void spline_planes_kernel(int64_t n, int64_t N, double ratio,
                                                            longlong2* __restrict__ planes) {
  const int64_t k = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (k >= n) return;
  const int64_t first = first_nearest(N, ratio, n, k);
  planes[k] = make_longlong2(first, first_nearest(N, ratio, n, k + 1) - first);
}

template <bool HALF>
__global__ __launch_bounds__(64) void spline_contig_kernel(
    const double* __restrict__ in, int64_t rows, int64_t n, const SplineTap* __restrict__ taps,
    int64_t N, double ratio, SplineConst k, SplinePowers pw, int64_t sep_n, int64_t sep_N,
    int64_t mid, const longlong2* __restrict__ planes, const float2* __restrict__ mm,
    float* __restrict__ out) {
  __shared__ __align__(16) double coef[kRowsPerWave][kTile];
  const int lane = threadIdx.x;
  for (int64_t t0 = -1 + (int64_t)blockIdx.y * kTileF; t0 < n; t0 += (int64_t)gridDim.y * kTileF) {
    const int64_t o_beg = first_with(taps, N, ratio, t0);
    const int64_t o_end = first_with(taps, N, ratio, t0 + kTileF);
    if (o_beg >= o_end) continue;
    const int64_t start = t0 - 1 - kEdge;  // position of the tile's first sample
    int64_t at[kLane];
#pragma unroll
    for (int j = 0; j < kLane; ++j) at[j] = extended(start + j * 64 + lane, n);
    for (int64_t r0 = blockIdx.x * (int64_t)kRowsPerWave; r0 < rows;
         r0 += (int64_t)gridDim.x * kRowsPerWave) {
      float2 bounds[kRowsPerWave];
      int64_t base[kRowsPerWave], copies[kRowsPerWave];
      bool any = false;
#pragma unroll
      for (int rr = 0; rr < kRowsPerWave; ++rr) {
        const int64_t r = min(r0 + rr, rows - 1);
        base[rr] = r * N;
        copies[rr] = 1;
        int64_t plane = 0;
        if (sep_n > 0) {
          // 32-bit divisions where the rows allow them
          int64_t km, m, ou;
          if (rows < (int64_t)1 << 31) {
            km = (unsigned)r / (unsigned)mid;
            ou = (unsigned)km / (unsigned)sep_n;
          } else {
            km = r / mid;
            ou = km / sep_n;
          }
          m = r - km * mid;
          plane = km - ou * sep_n;
          const longlong2 pl = planes[plane];
          base[rr] = ((ou * sep_N + pl.x) * mid + m) * N;
          copies[rr] = pl.y;
        }
        if (r0 + rr >= rows) copies[rr] = 0;
        any |= copies[rr] > 0;
        bounds[rr] = mm[plane];
      }
      if (!any) continue;  // uniform
      double x[kRowsPerWave][kLane];
#pragma unroll
      for (int rr = 0; rr < kRowsPerWave; ++rr) {
        const double* row = in + min(r0 + rr, rows - 1) * n;
#pragma unroll
        for (int j = 0; j < kLane; ++j) x[rr][j] = row[at[j]];
      }
      __syncthreads();  // the previous rows' coefficients are read
#pragma unroll
      for (int rr = 0; rr < kRowsPerWave; ++rr)
#pragma unroll
        for (int j = 0; j < kLane; ++j) coef[rr][j * 64 + lane] = x[rr][j];
      __syncthreads();
#pragma unroll
      for (int rr = 0; rr < kRowsPerWave; ++rr) {
        double c[kLane];
#pragma unroll
        for (int i = 0; i < kLane; ++i) c[i] = coef[rr][lane * kLane + i];
        const double before = c[0] * k.start;  // lane 0: as if constant before the tile
        c[0] = c[0] * k.gain;
#pragma unroll
        for (int i = 1; i < kLane; ++i) c[i] = c[i] * k.gain + k.z * c[i - 1];
        const double zs = pw.z[kLane];
        double e1 = __shfl_up(c[kLane - 1], 1), e2 = __shfl_up(c[kLane - 1], 2),
               e3 = __shfl_up(c[kLane - 1], 3);
        if (lane < 1) e1 = before;
        if (lane < 2) e2 = 0.0;
        if (lane < 3) e3 = 0.0;
        const double carry = e1 + zs * (e2 + zs * e3);
#pragma unroll
        for (int i = 0; i < kLane; ++i) c[i] = c[i] + pw.z[i + 1] * carry;
        const double behind = c[kLane - 1] * k.turn;  // lane 63: as if constant behind
        c[kLane - 1] = -k.z * c[kLane - 1];
#pragma unroll
        for (int i = kLane - 2; i >= 0; --i) c[i] = k.z * (c[i + 1] - c[i]);
        double d1 = __shfl_down(c[0], 1), d2 = __shfl_down(c[0], 2), d3 = __shfl_down(c[0], 3);
        if (lane > 62) d1 = behind;
        if (lane > 61) d2 = 0.0;
        if (lane > 60) d3 = 0.0;
        const double back = d1 + zs * (d2 + zs * d3);
#pragma unroll
        for (int i = 0; i < kLane; ++i)
          coef[rr][lane * kLane + i] = c[i] + pw.z[kLane - i] * back;
      }
      __syncthreads();
      const int64_t plane_out = mid * N;
      for (int64_t o = o_beg + lane; o < o_end; o += 64) {
        const SplineTap tp = taps[o];
        const int q = (int)(tp.f - 1 - start);
#pragma unroll
        for (int rr = 0; rr < kRowsPerWave; ++rr) {
          double sum = 0.0 + coef[rr][q] * tp.w[0];
          sum = sum + coef[rr][q + 1] * tp.w[1];
          sum = sum + coef[rr][q + 2] * tp.w[2];
          sum = sum + coef[rr][q + 3] * tp.w[3];
          sum = fmin(fmax(sum, (double)bounds[rr].x), (double)bounds[rr].y);
          const float value = round_result<HALF>(sum);
          float* to = out + base[rr] + o;
          for (int64_t c = 0; c < copies[rr]; ++c) to[c * plane_out] = value;
        }
      }
    }
  }
}

int blocks_for(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 256), 1 << 20)); }

struct SplinePlan {
  int64_t n[3], N[3];
  int pad[3];
  int axes[3], naxes;  // resized axes, in order
  int64_t a_elems, b_elems, mm_elems;
  int64_t extrema;  // of the planes, then of their parts
};

SplinePlan spline_plan(const int64_t* size, const int64_t* new_size, int separate_axis) {
  SplinePlan p{};
  p.naxes = 0;
  for (int a = 0; a < 3; ++a) {
    p.n[a] = size[a];
    p.N[a] = new_size[a];
    const bool resized = a != separate_axis;
    p.pad[a] = resized ? kSplinePad : 0;
    if (resized) p.axes[p.naxes++] = a;
  }
  // ping-pong: A holds the padded copy, B the first pass, A the second, B the third
  int64_t d[3] = {p.n[0] + 2 * p.pad[0], p.n[1] + 2 * p.pad[1], p.n[2] + 2 * p.pad[2]};
  int64_t sizes[4];
  sizes[0] = d[0] * d[1] * d[2];
  for (int k = 0; k < p.naxes; ++k) {
    d[p.axes[k]] = p.N[p.axes[k]];
    sizes[k + 1] = d[0] * d[1] * d[2];
  }
  p.a_elems = p.b_elems = 0;
  for (int k = 0; k <= p.naxes; ++k) {
    int64_t& slot = (k % 2 == 0) ? p.a_elems : p.b_elems;
    slot = std::max(slot, sizes[k]);
  }
  // per-plane bounds + the whole-volume entry
  const int64_t planes = separate_axis >= 0 ? p.n[separate_axis] : p.n[0];
  p.mm_elems = planes + 1;
  p.extrema = planes * (1 + kMinmaxParts);
  return p;
}

// Bytes of the two volumes, up to the alignment of what follows.
int64_t volume_bytes(const SplinePlan& p) {
  return ceil_div((p.a_elems + p.b_elems) * (int64_t)sizeof(double), 256) * 256;
}

// Bytes of the bounds and the extrema behind them, up to the tables' alignment.
int64_t bounds_bytes(const SplinePlan& p) {
  return ceil_div(p.mm_elems * (int64_t)sizeof(float2) + p.extrema * (int64_t)sizeof(Extrema), 256) * 256;
}

// entries of the tap tables (order 3): the outputs of every resized axis
int64_t tap_count(const SplinePlan& p) {
  int64_t taps = 0;
  for (int k = 0; k < p.naxes; ++k) taps += p.N[p.axes[k]];
  return taps;
}

// Order 3 of one channel: the resized axes in order, each one pass; A and B hold the float64
// volumes between them (spline_plan's slots, which are sized for padded ones).
void spline_cubic(const float* x, const int64_t* size, const int64_t* new_size, int separate_axis,
                  double* A, double* B, const SplineTap* taps, const longlong2* planes,
                  const float2* mm, float* out, hipStream_t st, bool round_half) {
  const double z = std::sqrt(3.0) - 2.0;
  SplineConst k;
  k.z = z;
  k.gain = (1.0 - z) * (1.0 - 1.0 / z);
  k.start = k.gain / (1.0 - z);
  k.turn = z / (z - 1.0);
  int64_t d[3] = {size[0], size[1], size[2]};
  const double sep_ratio =
      separate_axis < 0 ? 1.0 : (double)size[separate_axis] / (double)new_size[separate_axis];
  const void* src = x;
  double* dst = B;
  for (int a = 0; a < 3; ++a) {
    if (a == separate_axis) continue;
    const int64_t n = size[a], N = new_size[a];
    const double ratio = (double)size[a] / (double)new_size[a];
    const unsigned segs = (unsigned)std::min<int64_t>(ceil_div(n + 1, kSeg), 65535);
    const double moved = 8.0 * (double)(d[0] * d[1] * d[2]) / (double)n;
    if (a < 2) {
      const int64_t inner = a == 0 ? d[1] * d[2] : d[2], outer = a == 0 ? 1 : d[0];
      const bool skip = a == 1 && separate_axis == 0;
      const dim3 grid((unsigned)ceil_div(inner, 64), segs, (unsigned)std::min<int64_t>(outer, 65535));
      ProfScope prof("spline_strided", 0.0, moved * ((src == x ? 0.5 : 1.0) * (double)n + (double)N), st);
      if (src == x)
        hipLaunchKernelGGL(spline_strided_kernel<float>, grid, dim3(64), 0, st, x, n, inner, taps, N,
                           ratio, k, outer, skip ? size[0] : 0, skip ? new_size[0] : 0, sep_ratio, dst);
      else
        hipLaunchKernelGGL(spline_strided_kernel<double>, grid, dim3(64), 0, st,
                           static_cast<const double*>(src), n, inner, taps, N, ratio, k, outer,
                           skip ? size[0] : 0, skip ? new_size[0] : 0, sep_ratio, dst);
      d[a] = N;
      taps += N;
      src = dst;
      dst = dst == B ? A : B;
      continue;
    }
    const int64_t rows = d[0] * d[1];
    const int64_t mid = separate_axis == 0 ? d[1] : 1;
    const int64_t sep_n = separate_axis < 0 ? 0 : size[separate_axis];
    const int64_t sep_N = separate_axis < 0 ? 0 : new_size[separate_axis];
    const float2* bounds = separate_axis < 0 ? mm + size[0] : mm;
    // enough waves for the chip several times over; each takes its rows in turn
    const dim3 grid((unsigned)std::min<int64_t>(ceil_div(rows, kRowsPerWave), 16384),
                    (unsigned)std::min<int64_t>(ceil_div(n + 1, kTileF), 65535));
    SplinePowers pw;
    pw.z[0] = 1.0;
    for (int i = 1; i <= kLane; ++i) pw.z[i] = pw.z[i - 1] * z;
    ProfScope prof("spline_contig", 0.0,
                   moved * (double)n + 4.0 * (double)new_size[0] * (double)new_size[1] * (double)N, st);
    auto kernel = round_half ? spline_contig_kernel<true> : spline_contig_kernel<false>;
    hipLaunchKernelGGL(kernel, grid, dim3(64), 0, st, static_cast<const double*>(src), rows, n, taps,
                       N, ratio, k, pw, sep_n, sep_N, mid, planes, bounds, out);
  }
  if (separate_axis == 2) {
    const int64_t out_vox = new_size[0] * new_size[1] * new_size[2];
    ProfScope prof("spline_finish", 0.0, 8.0 * (double)(d[0] * d[1] * d[2]) + 4.0 * (double)out_vox,
                   st);
    auto kernel = round_half ? plane_clip_nearest_kernel<true> : plane_clip_nearest_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3(blocks_for(out_vox)), dim3(256), 0, st,
                       static_cast<const double*>(src), d[0], d[1], d[2], 2, new_size[2], sep_ratio,
                       mm, out);
  }
}

}  // namespace

void nonzero_bbox(const float* x, int channels, const int64_t* size, int* bbox, hipStream_t st) {
  require(x && bbox && size, "bounding-box pointers must not be null");
  require(channels >= 1 && size[0] >= 1 && size[1] >= 1 && size[2] >= 1, "invalid volume shape");
  const int64_t n = size[0] * size[1] * size[2];
  require(size[0] < INT_MAX && size[1] < INT_MAX && size[2] < INT_MAX, "volume axis too long");
  ProfScope prof("preprocess_bbox", 0.0, 4.0 * (double)n * channels, st);
  hipLaunchKernelGGL(bbox_init_kernel, dim3(1), dim3(64), 0, st, bbox);
  hipLaunchKernelGGL(bbox_kernel,
                     dim3((unsigned)std::min<int64_t>(ceil_div(size[0] * size[1], 4), 2048)),
                     dim3(256), 0, st, x, channels, size[0], size[1], size[2], bbox);
  launch_check("nonzero_bbox");
}

int nonzero_mask_filled(const float* x, int channels, const int64_t* size, const int64_t* start,
                        const int64_t* extent, uint8_t* mask, void* work, hipStream_t st) {
  require(x && size && start && extent && mask && work, "mask pointers must not be null");
  require(channels >= 1, "mask needs at least one channel");
  for (int a = 0; a < 3; ++a)
    require(extent[a] >= 1 && start[a] >= 0 && start[a] <= size[a] &&
                extent[a] <= size[a] - start[a],
            "mask box outside the volume");
  const int64_t total = extent[0] * extent[1] * extent[2];
  int* flag = static_cast<int*>(work);
  ProfScope prof("preprocess_fill_holes", 0.0, 4.0 * (double)total * channels, st);
  hipLaunchKernelGGL(mask_init_kernel, dim3(blocks_for(total)), dim3(256), 0, st, x, channels,
                     size[0], size[1], size[2], start[0], start[1], start[2], extent[0],
                     extent[1], extent[2], mask);
  // every round with a change reaches at least one more cell, so at most `total` rounds
  int rounds = 0;
  for (int64_t r = 0; r <= total; ++r) {
    hipLaunchKernelGGL(flag_clear_kernel, dim3(1), dim3(1), 0, st, flag);
    for (int axis = 2; axis >= 0; --axis) {
      const int64_t lines = total / extent[axis];
      hipLaunchKernelGGL(mask_sweep_kernel, dim3((unsigned)ceil_div(lines, 256)), dim3(256), 0,
                         st, mask, extent[0], extent[1], extent[2], axis, flag);
    }
    int changed = 0;
    hip_check(hipMemcpyAsync(&changed, flag, sizeof(int), hipMemcpyDeviceToHost, st),
              "mask flag copy");
    hip_check(hipStreamSynchronize(st), "mask flag sync");
    ++rounds;
    if (!changed) break;
  }
  hipLaunchKernelGGL(mask_finish_kernel, dim3(blocks_for(total)), dim3(256), 0, st, mask, total);
  launch_check("nonzero_mask_filled");
  return rounds;
}

size_t zscore_stats_workspace() { return kStatBlocks * sizeof(double2); }

void zscore_stats(const float* x, int channels, const int64_t* size, int channel,
                  const int64_t* start, const int64_t* extent, const uint8_t* mask, float* stats,
                  void* work, hipStream_t st) {
  require(x && size && start && extent && stats && work, "z-score pointers must not be null");
  require(channel >= 0 && channel < channels, "z-score channel out of range");
  for (int a = 0; a < 3; ++a)
    require(extent[a] >= 1 && start[a] >= 0 && start[a] <= size[a] &&
                extent[a] <= size[a] - start[a],
            "z-score box outside the volume");
  const int64_t total = extent[0] * extent[1] * extent[2];
  const float* xc = x + (int64_t)channel * size[0] * size[1] * size[2];
  double2* partial = static_cast<double2*>(work);
  const int blocks = (int)std::min<int64_t>(kStatBlocks, ceil_div(total, 256));
  ProfScope prof("preprocess_zscore_stats", 0.0, 8.0 * (double)total, st);
  for (int pass = 0; pass < 2; ++pass) {
    hipLaunchKernelGGL(zscore_partial_kernel, dim3(blocks), dim3(256), 0, st, xc, size[1],
                       size[2], start[0], start[1], start[2], extent[0], extent[1], extent[2],
                       mask, pass, stats, partial);
    hipLaunchKernelGGL(zscore_final_kernel, dim3(1), dim3(64), 0, st, partial, blocks, pass,
                       stats);
  }
  launch_check("zscore_stats");
}

void box_minmax(const float* x, int channels, const int64_t* size, int channel,
                const int64_t* start, const int64_t* extent, float* minmax, void* work,
                hipStream_t st) {
  require(x && size && start && extent && minmax && work, "extrema pointers must not be null");
  require(channel >= 0 && channel < channels, "extrema channel out of range");
  for (int a = 0; a < 3; ++a)
    require(extent[a] >= 1 && start[a] >= 0 && start[a] <= size[a] &&
                extent[a] <= size[a] - start[a],
            "extrema box outside the volume");
  const int64_t total = extent[0] * extent[1] * extent[2];
  const float* xc = x + (int64_t)channel * size[0] * size[1] * size[2];
  float2* partial = static_cast<float2*>(work);  // zscore_stats_workspace() bytes suffice
  const int blocks = (int)std::min<int64_t>(kStatBlocks, ceil_div(total, 256));
  ProfScope prof("preprocess_minmax", 0.0, 4.0 * (double)total, st);
  hipLaunchKernelGGL(box_minmax_partial_kernel, dim3(blocks), dim3(256), 0, st, xc, size[1],
                     size[2], start[0], start[1], start[2], extent[0], extent[1], extent[2],
                     partial);
  hipLaunchKernelGGL(box_minmax_final_kernel, dim3(1), dim3(64), 0, st, partial, blocks, minmax);
  launch_check("box_minmax");
}

void crop_normalize(const float* x, int channels, const int64_t* size, const int* transpose,
                    const int64_t* start, const int64_t* out_size, const int* schemes,
                    const float* norm, float* out, hipStream_t st) {
  crop_normalize_masked(x, channels, size, transpose, start, out_size, schemes, norm, nullptr,
                        nullptr, nullptr, out, st);
}

void crop_normalize_masked(const float* x, int channels, const int64_t* size,
                           const int* transpose, const int64_t* start, const int64_t* out_size,
                           const int* schemes, const float* norm, const uint8_t* mask,
                           const int64_t* mask_start, const int64_t* mask_extent, float* out,
                           hipStream_t st) {
  require(x && out && size && transpose && start && out_size && schemes,
          "crop/normalise pointers must not be null");
  require(channels >= 1 && channels <= kMaxNormChannels,
          "device normalisation supports 1..16 channels");
  bool seen[3] = {false, false, false};
  for (int k = 0; k < 3; ++k) {
    require(transpose[k] >= 0 && transpose[k] < 3 && !seen[transpose[k]],
            "transpose must be a permutation of the three spatial axes");
    seen[transpose[k]] = true;
  }
  for (int k = 0; k < 3; ++k) {
    const int64_t n = size[transpose[k]];
    require(out_size[k] >= 1 && start[k] >= 0 && start[k] <= n &&
                out_size[k] <= n - start[k],
            "crop window outside the volume");
  }
  ChannelNorms cn{};
  bool masked = false;
  for (int c = 0; c < channels; ++c) {
    require(schemes[c] >= NNX_NORM_NONE && schemes[c] <= NNX_NORM_ZSCORE_MASKED,
            "device normalisation supports NoNormalization, CTNormalization and "
            "ZScoreNormalization");
    cn.scheme[c] = schemes[c];
    if (schemes[c] == NNX_NORM_ZSCORE || schemes[c] == NNX_NORM_ZSCORE_MASKED) {
      require(norm != nullptr, "z-score normalisation needs its statistics");
      const float* p = norm + 4 * c;
      require(std::isfinite(p[0]) && std::isfinite(p[1]) && p[1] >= 0.f,
              "z-score statistics must be finite with a non-negative std");
      cn.mean[c] = p[0];
      cn.std[c] = std::max(p[1], 1e-8f);
      masked |= schemes[c] == NNX_NORM_ZSCORE_MASKED;
    }
    if (schemes[c] == NNX_NORM_CT) {
      require(norm != nullptr, "CT normalisation needs its statistics");
      const float* p = norm + 4 * c;
      require(std::isfinite(p[0]) && std::isfinite(p[1]) && p[1] > 0.f && std::isfinite(p[2]) &&
                  std::isfinite(p[3]) && p[2] <= p[3],
              "CT statistics must be finite, std positive and the percentiles ordered");
      cn.mean[c] = p[0];
      cn.std[c] = std::max(p[1], 1e-8f);
      cn.lower[c] = p[2];
      cn.upper[c] = p[3];
    }
  }
  int64_t ms[3] = {0, 0, 0}, me[3] = {1, 1, 1};
  if (masked) {
    require(mask && mask_start && mask_extent, "masked z-score normalisation needs the mask");
    // every cropped voxel (raw axis transpose[k] from start[k]) must lie in the mask box
    for (int k = 0; k < 3; ++k) {
      const int a = transpose[k];
      require(mask_extent[a] >= 1 && start[k] >= mask_start[a] &&
                  start[k] + out_size[k] <= mask_start[a] + mask_extent[a],
              "crop window outside the mask box");
    }
    for (int a = 0; a < 3; ++a) {
      ms[a] = mask_start[a];
      me[a] = mask_extent[a];
    }
  }
  const int64_t total = out_size[0] * out_size[1] * out_size[2] * channels;
  ProfScope prof("preprocess_crop_normalize", 0.0, 8.0 * (double)total, st);
  CropArgs a{};
  a.out = out;
  a.channels = channels;
  a.in_channel = size[0] * size[1] * size[2];
  a.norms = cn;
  const int64_t in_strides[3] = {size[1] * size[2], size[2], 1};
  const int64_t mask_strides[3] = {me[1] * me[2], me[2], 1};
  int64_t first = 0, mask_first = 0;
  for (int k = 0; k < 3; ++k) {
    a.n[k] = out_size[k];
    a.in_stride[k] = in_strides[transpose[k]];
    a.mask_stride[k] = mask_strides[transpose[k]];
    first += start[k] * a.in_stride[k];
    mask_first += (start[k] - ms[transpose[k]]) * a.mask_stride[k];
  }
  a.in = x + first;
  a.mask = masked ? mask + mask_first : nullptr;
  if (transpose[2] != 2 && out_size[2] >= kTileForm) {
    const int along = transpose[0] == 2 ? 0 : 1;
    const int64_t n = a.n[along];
    const int tile = n > 32 ? 64 : n > 16 ? 32 : 16;
    const int64_t tiles = ceil_div(n, tile) * ceil_div(a.n[2], 64) * a.n[1 - along] * channels;
    auto kernel = along == 0 ? (tile == 64 ? crop_normalize_tiles_kernel<0, 64>
                                : tile == 32 ? crop_normalize_tiles_kernel<0, 32>
                                             : crop_normalize_tiles_kernel<0, 16>)
                             : (tile == 64 ? crop_normalize_tiles_kernel<1, 64>
                                : tile == 32 ? crop_normalize_tiles_kernel<1, 32>
                                             : crop_normalize_tiles_kernel<1, 16>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)std::min<int64_t>(tiles, 1 << 20)), dim3(256), 0, st, a);
  } else if (transpose[2] == 2 && out_size[2] >= kRowForm) {
    hipLaunchKernelGGL(crop_normalize_rows_kernel, dim3(blocks_for(64 * (total / out_size[2]))),
                       dim3(256), 0, st, a);
  } else {
    hipLaunchKernelGGL(crop_normalize_kernel, dim3(blocks_for(total)), dim3(256), 0, st, a);
  }
  launch_check("crop_normalize");
}

size_t resample_spline_workspace(const int64_t* size, const int64_t* new_size, int separate_axis) {
  const SplinePlan p = spline_plan(size, new_size, separate_axis);
  const int64_t planes = separate_axis >= 0 ? p.n[separate_axis] : 0;
  return (size_t)volume_bytes(p) + (size_t)bounds_bytes(p) +
         (size_t)tap_count(p) * sizeof(SplineTap) + (size_t)planes * sizeof(longlong2) + 1024;
}

void resample_spline(const float* x, int channels, const int64_t* size, const int64_t* new_size,
                     int order, int separate_axis, int order_z, void* work, size_t work_bytes,
                     float* out, hipStream_t st, bool round_half) {
  require(x && out && size && new_size, "resampling pointers must not be null");
  require(channels >= 1, "resampling needs at least one channel");
  for (int a = 0; a < 3; ++a)
    require(size[a] >= 1 && new_size[a] >= 1, "resampling shapes must be positive");
  require(order == 1 || order == 3, "device spline resampling supports orders 1 and 3");
  require(separate_axis >= -1 && separate_axis < 3, "separate axis must be -1, 0, 1 or 2");
  require(separate_axis < 0 || order_z == 0,
          "device separate-axis resampling supports order_z 0 (nearest)");
  const SplinePlan p = spline_plan(size, new_size, separate_axis);
  require(work && work_bytes >= resample_spline_workspace(size, new_size, separate_axis),
          "resampling workspace too small");
  double* A = static_cast<double*>(work);
  double* B = A + p.a_elems;
  // (the tables behind hold 16-byte values, and the volumes may be an odd number of doubles)
  float2* mm = reinterpret_cast<float2*>(static_cast<char*>(work) + volume_bytes(p));
  const int64_t in_vox = size[0] * size[1] * size[2];
  const int64_t out_vox = new_size[0] * new_size[1] * new_size[2];
  Extrema* extrema = reinterpret_cast<Extrema*>(mm + p.mm_elems);
  SplineTap* taps = reinterpret_cast<SplineTap*>(reinterpret_cast<char*>(mm) + bounds_bytes(p));
  longlong2* sep_planes = reinterpret_cast<longlong2*>(
      reinterpret_cast<char*>(taps) + ceil_div(tap_count(p) * (int64_t)sizeof(SplineTap), 256) * 256);
  if (order == 3) {
    // the taps of the resized axes, one table after the other
    int64_t at = 0;
    for (int k = 0; k < p.naxes; ++k) {
      const int a = p.axes[k];
      hipLaunchKernelGGL(spline_taps_kernel, dim3((unsigned)ceil_div(new_size[a], 256)), dim3(256),
                         0, st, new_size[a], (double)size[a] / (double)new_size[a], taps + at);
      at += new_size[a];
    }
    if (separate_axis >= 0)
      hipLaunchKernelGGL(spline_planes_kernel, dim3((unsigned)ceil_div(size[separate_axis], 256)),
                         dim3(256), 0, st, size[separate_axis], new_size[separate_axis],
                         (double)size[separate_axis] / (double)new_size[separate_axis], sep_planes);
  }
  const int mm_axis = separate_axis >= 0 ? separate_axis : 0;
  for (int c = 0; c < channels; ++c) {
    const float* xc = x + (int64_t)c * in_vox;
    const int64_t planes = size[mm_axis];
    Extrema* part = extrema + planes;
    const bool spread = order == 3;
    {
      ProfScope prof("spline_minmax", 0.0, 4.0 * (double)in_vox, st);
      hipLaunchKernelGGL(plane_minmax_kernel, dim3((unsigned)planes, kMinmaxParts), dim3(256), 0,
                         st, xc, size[0], size[1], size[2], mm_axis, part);
      hipLaunchKernelGGL(plane_parts_kernel, dim3((unsigned)ceil_div(planes, 256)), dim3(256), 0,
                         st, part, planes, kMinmaxParts, spread, extrema, mm);
      if (separate_axis < 0)
        hipLaunchKernelGGL(reduce_minmax_kernel, dim3(1), dim3(64), 0, st, extrema, planes, spread,
                           mm + planes);
    }
    float* oc = out + (int64_t)c * out_vox;
    if (order == 3) {
      spline_cubic(xc, size, new_size, separate_axis, A, B, taps, sep_planes, mm, oc, st,
                   round_half);
      continue;
    }
    int64_t d[3] = {size[0] + 2 * p.pad[0], size[1] + 2 * p.pad[1], size[2] + 2 * p.pad[2]};
    {
      const int64_t padded = d[0] * d[1] * d[2];
      ProfScope prof("spline_pad", 0.0, 4.0 * (double)in_vox + 8.0 * (double)padded, st);
      hipLaunchKernelGGL(pad_edge_kernel, dim3(blocks_for(padded)), dim3(256), 0, st, xc, size[0],
                         size[1], size[2], p.pad[0], p.pad[1], p.pad[2], A);
    }
    double* src = A;
    double* dst = B;
    for (int k = 0; k < p.naxes; ++k) {
      const int a = p.axes[k];
      int64_t od[3] = {d[0], d[1], d[2]};
      od[a] = new_size[a];
      const double ratio = (double)size[a] / (double)new_size[a];
      const int64_t total = od[0] * od[1] * od[2];
      ProfScope prof("spline_interp", 0.0, 8.0 * (double)(d[0] * d[1] * d[2] + total), st);
      hipLaunchKernelGGL(interp_axis_kernel, dim3(blocks_for(total)), dim3(256), 0, st, src, d[0],
                         d[1], d[2], a, new_size[a], ratio, p.pad[a], dst);
      d[a] = new_size[a];
      std::swap(src, dst);
    }
    ProfScope prof("spline_finish", 0.0, 8.0 * (double)(d[0] * d[1] * d[2]) + 4.0 * (double)out_vox,
                   st);
    if (separate_axis < 0) {
      auto kernel = round_half ? cast_clip_kernel<true> : cast_clip_kernel<false>;
      hipLaunchKernelGGL(kernel, dim3(blocks_for(out_vox)), dim3(256), 0, st, src, out_vox,
                         mm + size[0], oc);
    } else {
      const int a = separate_axis;
      auto kernel = round_half ? plane_clip_nearest_kernel<true> : plane_clip_nearest_kernel<false>;
      hipLaunchKernelGGL(kernel, dim3(blocks_for(out_vox)), dim3(256), 0, st, src, d[0], d[1],
                         d[2], a, new_size[a], (double)size[a] / (double)new_size[a], mm, oc);
    }
  }
  launch_check("resample_spline");
}

}  // namespace nnx
