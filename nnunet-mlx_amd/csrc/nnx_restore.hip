// Fused class-logit restoration: half-pixel trilinear resampling (edge-clamped) of
// channels-last logits to the original grid, in float64, and the first-maximum argmax.
//
// Replaces the reference's fused Metal restoration
// (src/nnunet_mlx/kernels/metal_restore.py:69-137 kernel, :401-427 launch, :464-489 axis
// metadata).  The reference emulates float64 with double-single arithmetic because the
// host resampler it must agree with interpolates in float64; gfx950 has native float64,
// so every coordinate, weight, product and sum here is an IEEE float64 operation in the
// same order as the oracle's numpy restatement (no contraction: -ffp-contract=off).
//
// One thread per output voxel (grid-stride).  Per axis: c = (i + 0.5) * (S / T) - 0.5
// clipped to [0, S - 1], lower = floor(c), upper = min(lower + 1, S - 1), weights
// 1 - (c - lower) and c - lower.  Per class: the eight corners in the order
// 000, 001, 010, 011, 100, 101, 110, 111 (z, y, x bits), each term ((v * w_z) * w_y) * w_x,
// summed left to right from 0; the sum rounded to float32 (or to float16, nearest even,
// for float16 logits) is compared with strict ">" so ties keep the earliest class.
// Roofline: HBM — reads the source logits (8 corners per voxel, reused through the
// caches) and writes 2 bytes per output voxel; float64 VALU work ~(24 + 32 K) operations
// per output voxel.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "nnx_internal.h"

namespace nnx {
namespace {

struct AxisCoord {
  int lo, hi;
  double wlo, whi;
};

__device__ __forceinline__ AxisCoord axis_coord(int i, double ratio, int source) {
  double c = ((double)i + 0.5) * ratio - 0.5;
  c = fmin(fmax(c, 0.0), (double)(source - 1));
  AxisCoord a;
  a.lo = (int)floor(c);
  a.hi = a.lo + 1 < source ? a.lo + 1 : source - 1;
  a.whi = c - (double)a.lo;
  a.wlo = 1.0 - a.whi;
  return a;
}

template <bool HALF>
__device__ __forceinline__ double load_logit(const void* logits, int64_t i) {
  if constexpr (HALF)
    return (double)static_cast<const _Float16*>(logits)[i];
  else
    return (double)static_cast<const float*>(logits)[i];
}

template <bool HALF>
__global__ __launch_bounds__(256) void restore_argmax_kernel(const void* __restrict__ logits,
                                                             int classes, int sz, int sy, int sx,
                                                             int tz, int ty, int tx, double rz,
                                                             double ry, double rx,
                                                             uint16_t* __restrict__ labels) {
  const int64_t total = (int64_t)tz * ty * tx;
  const int64_t plane = (int64_t)sy * sx;
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total;
       e += (int64_t)gridDim.x * blockDim.x) {
    const int x = (int)(e % tx);
    const int64_t rest = e / tx;
    const int y = (int)(rest % ty);
    const int z = (int)(rest / ty);
    const AxisCoord cz = axis_coord(z, rz, sz);
    const AxisCoord cy = axis_coord(y, ry, sy);
    const AxisCoord cx = axis_coord(x, rx, sx);
    const int zs[2] = {cz.lo, cz.hi}, ys[2] = {cy.lo, cy.hi}, xs[2] = {cx.lo, cx.hi};
    const double wz[2] = {cz.wlo, cz.whi}, wy[2] = {cy.wlo, cy.whi}, wx[2] = {cx.wlo, cx.whi};
    int64_t base[8];
#pragma unroll
    for (int c = 0; c < 8; ++c)
      base[c] = ((int64_t)zs[c >> 2] * plane + (int64_t)ys[(c >> 1) & 1] * sx + xs[c & 1]) * classes;
    float best = -INFINITY;
    int label = 0;
    for (int k = 0; k < classes; ++k) {
      double sum = 0.0;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const double v = load_logit<HALF>(logits, base[c] + k);
        sum = sum + ((v * wz[c >> 2]) * wy[(c >> 1) & 1]) * wx[c & 1];
      }
      const float value = HALF ? (float)(_Float16)sum : (float)sum;
      if (value > best) {
        best = value;
        label = k;
      }
    }
    labels[e] = (uint16_t)label;
  }
}

// ---- restoration along an order-1 spline plan, every class of a voxel in one pass -------
//
// The spline resampler's order-1 arithmetic (nnx_preprocess.hip: axes in ascending order, the
// separate axis skipped; per axis 0.0 + v[f] (1 - t) + v[f + 1] t at the padded coordinate
// cc = (o + 0.5) n_in / n_out - 0.5 + 12, f = floor(cc), t = cc - f, edge samples repeated) from
// the four or eight logits that a voxel needs, instead of a float64 copy of the padded volume
// and of every axis pass per class: an interpolation between two values is formed at each
// place where the axis-by-axis form reads it.  The resampler's clip to the plane's [min, max]
// cannot change a finite result: it lies within a few float64 ulps of the bounds, which are
// float32 (or float16) values, so the rounding to that type already returns them.  Only a NaN
// (infinite or NaN logits) is replaced, by what the clip makes of one: the plane's minimum, or
// -inf where the plane holds NaN only (the bounds of an empty reduction).  A first pass that
// met a NaN raises a flag, and the two kernels behind it, which otherwise return at once, form
// these values and redo the voxels.
//
// Roofline: HBM — the logits of the source planes that the nearest indices pick, once, and 2 B a
// voxel.  300 x 534 x 534 x 3 float16 -> 120 x 512 x 512: 4.90 ms as 30 launches
// through float64 volumes, 0.25 ms in one pass (0.27 GB of it needed: 1.1 TB/s).
constexpr int kSplinePad = 12;

struct LinTap {
  int lo, hi;
  double t;
};

__device__ __forceinline__ LinTap lin_tap(int o, double ratio, int n) {
  const double cc = ((double)o + 0.5) * ratio - 0.5 + (double)kSplinePad;
  const double f = floor(cc);
  LinTap r;
  r.t = cc - f;
  const int start = (int)f - kSplinePad;
  r.lo = min(max(start, 0), n - 1);
  r.hi = min(max(start + 1, 0), n - 1);
  return r;
}

// nearest source plane of output o along the separate axis
__device__ __forceinline__ int nearest_plane(int o, double ratio, int n) {
  const double coord = ratio * ((double)o + 0.5) - 0.5;
  return min(max((int)floor(coord + 0.5), 0), n - 1);
}

struct LinArgs {
  const void* logits;
  int classes;
  int n[3], N[3];
  double ratio[3];
  uint16_t* labels;
  int* flag;
  // redo pass: classes [c0, c1), clipped NaN [plane * (c1 - c0) + class - c0], running winners
  int c0, c1;
  const float* clipped;
  float* best;
};

// Block (64 x, 4 y) of output voxels, z over gridDim.z.  SEP: the separate axis, -1 for none.
template <bool HALF, int SEP, bool REDO>
__global__ __launch_bounds__(256) void restore_linear_kernel(LinArgs a) {
  if constexpr (REDO) {
    if (*a.flag == 0) return;
  }
  const int x = blockIdx.x * 64 + (threadIdx.x & 63);
  if (x >= a.N[2]) return;
  LinTap taps[3];
  auto tap = [&](int axis, int o) {
    if (axis != SEP) return lin_tap(o, a.ratio[axis], a.n[axis]);
    const int k = nearest_plane(o, a.ratio[axis], a.n[axis]);
    return LinTap{k, k, 0.0};
  };
  taps[2] = tap(2, x);
  bool nan = false;
  for (int y = blockIdx.y * 4 + (threadIdx.x >> 6); y < a.N[1]; y += gridDim.y * 4) {
    taps[1] = tap(1, y);
    for (int z = blockIdx.z; z < a.N[0]; z += gridDim.z) {
      taps[0] = tap(0, z);
      constexpr int c0n = SEP == 0 ? 1 : 2, c1n = SEP == 1 ? 1 : 2, c2n = SEP == 2 ? 1 : 2;
      int64_t base[2][2][2];
#pragma unroll
      for (int i = 0; i < c0n; ++i)
#pragma unroll
        for (int j = 0; j < c1n; ++j)
#pragma unroll
          for (int k = 0; k < c2n; ++k)
            base[i][j][k] = (((int64_t)(i ? taps[0].hi : taps[0].lo) * a.n[1] +
                              (j ? taps[1].hi : taps[1].lo)) * a.n[2] +
                             (k ? taps[2].hi : taps[2].lo)) * a.classes;
      const int64_t e = ((int64_t)z * a.N[1] + y) * a.N[2] + x;
      float best = 0.f;
      int label = 0;
      if constexpr (REDO) {
        if (a.c0 > 0) {
          best = a.best[e];
          label = a.labels[e];
        }
      }
      auto mix = [](double u, double v, double t) { return (0.0 + u * (1.0 - t)) + v * t; };
      const int cbeg = REDO ? a.c0 : 0, cend = REDO ? a.c1 : a.classes;
#pragma unroll 4
      for (int c = cbeg; c < cend; ++c) {
        auto at = [&](int i, int j, int k) { return load_logit<HALF>(a.logits, base[i][j][k] + c); };
        // along axis 0 at each corner of the others, then axis 1, then axis 2
        auto along0 = [&](int j, int k) {
          if constexpr (SEP == 0) return at(0, j, k);
          else return mix(at(0, j, k), at(1, j, k), taps[0].t);
        };
        auto along1 = [&](int k) {
          if constexpr (SEP == 1) return along0(0, k);
          else return mix(along0(0, k), along0(1, k), taps[1].t);
        };
        double v;
        if constexpr (SEP == 2) v = along1(0);
        else v = mix(along1(0), along1(1), taps[2].t);
        if constexpr (REDO) {
          if (v != v) {
            const int plane = SEP == 0 ? taps[0].lo : SEP == 1 ? taps[1].lo : SEP == 2 ? taps[2].lo : 0;
            v = (double)a.clipped[(int64_t)plane * (a.c1 - a.c0) + c - a.c0];
          }
        } else {
          nan |= v != v;
        }
        const float value = HALF ? (float)(_Float16)v : (float)v;
        if (c == 0 || value > best) {
          best = value;
          label = c;
        }
      }
      if constexpr (REDO) a.best[e] = best;
      a.labels[e] = (uint16_t)label;
    }
  }
  if constexpr (!REDO) {
    if (nan) *a.flag = 1;
  }
}

__global__ void restore_flag_clear_kernel(int* flag) { *flag = 0; }

// clipped[plane * (c1 - c0) + class - c0] = min(max(NaN, lo), hi) with the bounds lo, hi of the
// source plane (sep < 0: the volume) of each class, formed without its NaN; one workgroup a
// plane.  Returns at once unless the flag is raised.
template <bool HALF>
__global__ __launch_bounds__(1024) void restore_clipped_kernel(LinArgs a, int sep, float* clipped) {
  __shared__ float low[16], high[16];
  if (*a.flag == 0) return;
  const int64_t m = sep < 0 ? (int64_t)a.n[0] * a.n[1] * a.n[2]
                            : (int64_t)a.n[0] * a.n[1] * a.n[2] / a.n[sep];
  const int64_t inner = sep == 0 || sep < 0 ? m : sep == 1 ? a.n[2] : 1;
  for (int c = a.c0; c < a.c1; ++c) {
    float lo = INFINITY, hi = -INFINITY;
    for (int64_t i = threadIdx.x; i < m; i += 1024) {
      const int64_t v = sep < 0 ? i : (i / inner * a.n[sep] + blockIdx.x) * inner + i % inner;
      const float x = (float)load_logit<HALF>(a.logits, v * a.classes + c);
      lo = fminf(lo, x);
      hi = fmaxf(hi, x);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      lo = fminf(lo, __shfl_xor(lo, o));
      hi = fmaxf(hi, __shfl_xor(hi, o));
    }
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
      low[threadIdx.x >> 6] = lo;
      high[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < 16; ++w) {
        lo = fminf(lo, low[w]);
        hi = fmaxf(hi, high[w]);
      }
      clipped[(int64_t)blockIdx.x * (a.c1 - a.c0) + c - a.c0] = fminf(lo, hi);
    }
  }
}

// out[v] = class c of channels-last logits (n voxels, `classes` per voxel) as float32
template <bool HALF>
__global__ __launch_bounds__(256) void extract_class_kernel(const void* __restrict__ logits,
                                                            int classes, int c, int64_t n,
                                                            float* __restrict__ out) {
  for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = v * classes + c;
    if constexpr (HALF) out[v] = __half2float(static_cast<const __half*>(logits)[i]);
    else out[v] = static_cast<const float*>(logits)[i];
  }
}

// running first-maximum argmax: class 0 initialises, later classes win only when strictly
// greater (ties keep the earliest class)
__global__ __launch_bounds__(256) void argmax_update_kernel(const float* __restrict__ value,
                                                            int64_t n, int c,
                                                            float* __restrict__ best,
                                                            uint16_t* __restrict__ labels) {
  for (int64_t v = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x) {
    const float x = value[v];
    if (c == 0) {
      best[v] = x;
      labels[v] = 0;
    } else if (x > best[v]) {
      best[v] = x;
      labels[v] = (uint16_t)c;
    }
  }
}

int grid_for(int64_t n) { return (int)std::max<int64_t>(1, std::min<int64_t>(ceil_div(n, 256), 1 << 20)); }

int64_t align256(int64_t bytes) { return ceil_div(bytes, 256) * 256; }

template <bool HALF, int SEP>
void launch_linear(LinArgs a, int planes, float* clipped, int64_t room, hipStream_t st) {
  const dim3 grid((unsigned)ceil_div(a.N[2], 64),
                  (unsigned)std::min<int64_t>(ceil_div(a.N[1], 4), 65535),
                  (unsigned)std::min(a.N[0], 65535));
  hipLaunchKernelGGL(restore_flag_clear_kernel, dim3(1), dim3(1), 0, st, a.flag);
  hipLaunchKernelGGL((restore_linear_kernel<HALF, SEP, false>), grid, dim3(256), 0, st, a);
  // as many classes a round as the clipped values have room for (all of them, as a rule)
  const int round = (int)std::min<int64_t>(a.classes, std::max<int64_t>(1, room / planes));
  for (a.c0 = 0; a.c0 < a.classes; a.c0 = a.c1) {
    a.c1 = std::min(a.classes, a.c0 + round);
    a.clipped = clipped;
    hipLaunchKernelGGL(restore_clipped_kernel<HALF>, dim3((unsigned)planes), dim3(1024), 0, st, a,
                       SEP, clipped);
    // a small grid (it loops): nearly always every workgroup returns at once, and the full
    // grid took 52 us to do so
    hipLaunchKernelGGL((restore_linear_kernel<HALF, SEP, true>),
                       dim3(grid.x, std::min(grid.y, 16u), std::min(grid.z, 16u)), dim3(256), 0, st, a);
  }
}

// `work`: its first 256 bytes hold the flag, then a float per source voxel, then one per output
// voxel
void restore_linear(const void* logits, bool half, int classes, const int* src, const int* dst,
                    int separate_axis, char* work, uint16_t* labels, hipStream_t st) {
  LinArgs a{};
  a.logits = logits;
  a.classes = classes;
  int64_t n_src = 1, n_dst = 1;
  for (int i = 0; i < 3; ++i) {
    a.n[i] = src[i];
    a.N[i] = dst[i];
    a.ratio[i] = (double)src[i] / (double)dst[i];
    n_src *= src[i];
    n_dst *= dst[i];
  }
  a.labels = labels;
  a.flag = reinterpret_cast<int*>(work);
  float* clipped = reinterpret_cast<float*>(work + 256);
  a.best = reinterpret_cast<float*>(work + 256 + align256(4 * n_src));
  const int planes = separate_axis < 0 ? 1 : src[separate_axis];
  ProfScope prof("restore_linear", 0.0, (half ? 2.0 : 4.0) * classes * n_src + 2.0 * n_dst, st);
  auto launch = [&](auto h) {
    constexpr bool H = decltype(h)::value;
    if (separate_axis < 0) launch_linear<H, -1>(a, planes, clipped, n_src, st);
    else if (separate_axis == 0) launch_linear<H, 0>(a, planes, clipped, n_src, st);
    else if (separate_axis == 1) launch_linear<H, 1>(a, planes, clipped, n_src, st);
    else launch_linear<H, 2>(a, planes, clipped, n_src, st);
  };
  if (half) launch(std::true_type{});
  else launch(std::false_type{});
  launch_check("restore_labels_spline");
}

}  // namespace

// Order 1: the flag, the clipped values and the running winners of the redo pass; order 3: a class's
// logits and values, the winners and the resampler's workspace.
size_t restore_labels_spline_workspace(const int* src, const int* dst, int order, int separate_axis) {
  const int64_t s[3] = {src[0], src[1], src[2]}, d[3] = {dst[0], dst[1], dst[2]};
  const int64_t n_src = s[0] * s[1] * s[2], n_dst = d[0] * d[1] * d[2];
  if (order == 1) return (size_t)(256 + align256(4 * n_src) + align256(4 * n_dst));
  return (size_t)(align256(4 * n_src) + 2 * align256(4 * n_dst)) +
         resample_spline_workspace(s, d, separate_axis);
}

void restore_labels_spline(const void* logits, bool half, int classes, const int* src,
                           const int* dst, int order, int separate_axis, void* work,
                           size_t work_bytes, uint16_t* labels, hipStream_t st) {
  require(logits && labels && src && dst && work, "restoration pointers must not be null");
  require(classes >= 1 && classes <= 65536, "restoration supports 1..65536 classes");
  for (int i = 0; i < 3; ++i)
    require(src[i] >= 1 && dst[i] >= 1, "restoration shapes must be positive");
  require(separate_axis >= -1 && separate_axis < 3, "separate axis must be -1, 0, 1 or 2");
  require(work_bytes >= restore_labels_spline_workspace(src, dst, order, separate_axis),
          "restoration workspace too small");
  const int64_t s[3] = {src[0], src[1], src[2]}, d[3] = {dst[0], dst[1], dst[2]};
  const int64_t n_src = s[0] * s[1] * s[2], n_dst = d[0] * d[1] * d[2];
  char* base = static_cast<char*>(work);
  if (order == 1) {
    restore_linear(logits, half, classes, src, dst, separate_axis, base, labels, st);
    return;
  }
  float* channel = reinterpret_cast<float*>(base);
  float* value = reinterpret_cast<float*>(base + align256(4 * n_src));
  float* best = reinterpret_cast<float*>(base + align256(4 * n_src) + align256(4 * n_dst));
  void* spline_work = base + align256(4 * n_src) + 2 * align256(4 * n_dst);
  const size_t spline_bytes = work_bytes - (size_t)(align256(4 * n_src) + 2 * align256(4 * n_dst));
  for (int c = 0; c < classes; ++c) {
    {
      ProfScope prof("restore_extract", 0.0, (half ? 2.0 : 4.0) * classes * n_src + 4.0 * n_src, st);
      if (half)
        hipLaunchKernelGGL(extract_class_kernel<true>, dim3(grid_for(n_src)), dim3(256), 0, st,
                           logits, classes, c, n_src, channel);
      else
        hipLaunchKernelGGL(extract_class_kernel<false>, dim3(grid_for(n_src)), dim3(256), 0, st,
                           logits, classes, c, n_src, channel);
    }
    resample_spline(channel, 1, s, d, order, separate_axis, 0, spline_work, spline_bytes, value,
                    st, half);
    ProfScope prof("restore_argmax_update", 0.0, 4.0 * n_dst + (c ? 8.0 : 6.0) * n_dst, st);
    hipLaunchKernelGGL(argmax_update_kernel, dim3(grid_for(n_dst)), dim3(256), 0, st, value,
                       n_dst, c, best, labels);
  }
  launch_check("restore_labels_spline");
}

void restore_labels(const void* logits, bool half, int classes, const int* src, const int* dst,
                    uint16_t* labels, hipStream_t st) {
  require(logits && labels && src && dst, "restoration pointers must not be null");
  require(classes >= 1 && classes <= 65536, "restoration supports 1..65536 classes");
  for (int i = 0; i < 3; ++i)
    require(src[i] >= 1 && dst[i] >= 1, "restoration shapes must be positive");
  const int64_t total = (int64_t)dst[0] * dst[1] * dst[2];
  const double rz = (double)src[0] / dst[0], ry = (double)src[1] / dst[1],
               rx = (double)src[2] / dst[2];
  const int64_t in_bytes = (int64_t)src[0] * src[1] * src[2] * classes * (half ? 2 : 4);
  ProfScope prof("restore_argmax", 0.0, (double)in_bytes + 2.0 * (double)total, st);
  const int blocks = (int)std::min<int64_t>(ceil_div(total, 256), 1 << 20);
  if (half)
    hipLaunchKernelGGL(restore_argmax_kernel<true>, dim3(blocks), dim3(256), 0, st, logits,
                       classes, src[0], src[1], src[2], dst[0], dst[1], dst[2], rz, ry, rx,
                       labels);
  else
    hipLaunchKernelGGL(restore_argmax_kernel<false>, dim3(blocks), dim3(256), 0, st, logits,
                       classes, src[0], src[1], src[2], dst[0], dst[1], dst[2], rz, ry, rx,
                       labels);
  launch_check("restore_labels");
}

}  // namespace nnx
