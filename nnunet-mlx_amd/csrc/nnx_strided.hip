// Strided 3x3x3 convolutions (strides (1 or 2, 2, 2), padding 1) with split-fp16 products (hi*hi +
// hi*lo + lo*hi) on v_mfma_f32_32x32x16_f16, or bf16 operands and one product, float32
// accumulation.
//
// Workgroup: 4 waves, an output box of 2 x 4 x 8 voxels and 64 output channels, two workgroups a
// CU, so that one converts while the other multiplies (one workgroup of 8 waves and 4 planes a
// box ran the two phases in turn: 1.32 ms on the first shape below).  One MFMA's K = 16 is two taps of 8
// channels, so the packed words of the other split kernels serve here too.  Wave (h, cb)
// accumulates both z planes (32 voxels each) and the 32 channels of block cb over the channels of
// half h of every 16-channel chunk; the halves are added through LDS at the end.  So a weight
// word, which each wave takes from L2 seven steps ahead, meets two planes and all three products.
// A operands are read from LDS a step ahead.
//
// Per chunk the halo (stride 2: 5 x 9 x 17 voxels) is loaded to registers during the previous
// chunk, a line a step between the weights, normalised (the input's pending InstanceNorm +
// LeakyReLU), split and written to LDS between two barriers.  16 channels are 64 bytes of a
// voxel's row: the 8-channel chunks of the implicit GEMM ask for every 128-byte line four times.
// Voxels are stored by the parity of their row and column, so that the 32 output voxels of a tap
// read 32 different 16-byte bank groups.  Persistent: two workgroups a CU loop over boxes (XCDs take
// contiguous ranges, column group slowest), a box's last chunk loading the next box's first.
//
// Bound by issue: the conversion's VALU work and the products take about as long, and each
// SIMD's two waves overlap them in part.  Against the implicit GEMM: 32 -> 64 on 128^3 x 8, stride 2,
// 1.42 -> 1.14 ms (203 TFLOP/s), 64 -> 128 on 37 x 61 x 43 x 2 66 -> 57 us, 256 -> 320 on 16^3 98 -> 50 us;
// error against float64 2.5e-7 relative (3.3e-7).
#include <cmath>
#include <type_traits>

#include "nnx_internal.h"

namespace nnx {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

constexpr int kSThreads = 256;
constexpr int kWaves = kSThreads / 64;
constexpr int kSChunk = 16;          // input channels per chunk
constexpr int kSMaxChannels = 1024;  // c1 + c2 (pending-norm parameters in LDS)
constexpr int kBZ = 2, kBY = 4, kBX = 8;      // output box
constexpr int kHY = 2 * kBY + 1, kHX = 2 * kBX + 1;
constexpr int kYPitch = 145, kYPar = 72, kXPar = 36;  // 16-byte slots; four a voxel
constexpr int kPlaneSlots = 4 * kYPitch + kYPar;      // halo plane: rows 0 .. 8
constexpr int kPairs = 14;           // of taps (tap 27 has zero weights)
constexpr int kRing = 7;
static_assert(kPairs % kRing == 0, "ring slots are the same in every chunk");

__host__ __device__ constexpr int voxel_slot(int hy, int hx) {
  return (hy >> 1) * kYPitch + (hy & 1) * kYPar + (hx & 1) * kXPar + (hx >> 1) * 4;
}

template <int SZ>
struct StridedGeom {
  static constexpr int hz = (kBZ - 1) * SZ + 3;
  static constexpr int lines = hz * kHY * kHX * 4;
  static constexpr int rounds = (lines + kSThreads - 1) / kSThreads;
  static constexpr int epilogue = (2 * kWaves * 1024 + 2 * kWaves * 32) / 4;
  static constexpr int slots = hz * kPlaneSlots > epilogue ? hz * kPlaneSlots : epilogue;
  static_assert(slots * 16 + 3 * kSMaxChannels * 4 <= 80 * 1024, "LDS");
};

struct StridedArgs {
  const float* x0;
  const float* x1;
  int c0, c1, chunks0, chunks;
  const uint4* w;
  int nblk16;  // 16-column blocks of the packing
  const float* bias;
  float* y;
  int id, ih, iw, od, oh, ow;
  int cout, nblk;  // 32-column blocks
  int nbz, nby, nbx;
  int nbox, nvirt;
  int cper;
  int64_t split_stride;
  float out_scale;
  float4* stats;
  const float4* nrm0;
  const float4* nrm1;
  int act0, act1;
  float slope;
};

__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct StridedBox {
  int ng, b, bzi, byi, bxi;
};

__device__ __forceinline__ StridedBox strided_box(const StridedArgs& a, int v) {
  StridedBox r;
  r.ng = v / a.nbox;
  int box = v - r.ng * a.nbox;
  r.bxi = box % a.nbx;
  box /= a.nbx;
  r.byi = box % a.nby;
  box /= a.nby;
  r.bzi = box % a.nbz;
  r.b = box / a.nbz;
  return r;
}

__device__ __forceinline__ float add_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int AR>
__device__ __forceinline__ f16v mfma(uint4 a, uint4 b, f16v c) {
  if constexpr (AR == kArithBf16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a),
                                                   __builtin_bit_cast(bf8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a),
                                                  __builtin_bit_cast(h8, b), c, 0, 0, 0);
}

template <int SZ, int AR>
__global__ __launch_bounds__(kSThreads, 2) void conv_strided_kernel(StridedArgs a) {
  using G = StridedGeom<SZ>;
  constexpr int kR = G::rounds, kParts = AR == kArithBf16 ? 1 : 2;
  __shared__ __align__(16) uint4 s_a[G::slots];
  __shared__ __align__(16) float s_prm[3 * kSMaxChannels];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, stride = gridDim.x >> 3;
  const int vq = a.nvirt >> 3, vr = a.nvirt & 7;
  const int vbeg = xcd < vr ? xcd * (vq + 1) : vr * (vq + 1) + (xcd - vr) * vq;
  const int vend = vbeg + vq + (xcd < vr ? 1 : 0);
  int v = vbeg + (int)(blockIdx.x >> 3);
  if (v >= vend) return;  // uniform over the workgroup, before any barrier
  const int cbeg = blockIdx.y * a.cper, cend = min(cbeg + a.cper, a.chunks);
  __builtin_assume(cend > cbeg);
  const int h = wave & 1, cb = wave >> 1;

  // voxel of line r of this thread (round r: line r * 256 + tid, its quad tid % 4)
  auto line_voxel = [&](int tid, int r, int& hz, int& hy, int& hx) {
    const int vox = r * (kSThreads / 4) + (tid >> 2);
    hz = vox / (kHY * kHX);
    const int rem = vox - hz * (kHY * kHX);
    hy = rem / kHX;
    hx = rem - hy * kHX;
  };
  auto box_lines = [&](int tid, const StridedBox& bx, int (&at)[kR]) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < kR; ++r) {
      int hz, hy, hx;
      line_voxel(tid, r, hz, hy, hx);
      const int z = bx.bzi * kBZ * SZ - 1 + hz, yy = bx.byi * kBY * 2 - 1 + hy,
                xx = bx.bxi * kBX * 2 - 1 + hx;
      at[r] = hz < G::hz && (unsigned)z < (unsigned)a.id && (unsigned)yy < (unsigned)a.ih &&
                      (unsigned)xx < (unsigned)a.iw
                  ? (z * a.ih + yy) * a.iw + xx : -1;
    }
  };
  struct Source {
    const float* base;  // channel chunk of the item
    int C;
  };
  auto source = [&](const StridedBox& bx, int chunk) __attribute__((always_inline)) {
    const bool first = chunk < a.chunks0;
    Source r;
    r.C = first ? a.c0 : a.c1;
    r.base = (first ? a.x0 : a.x1) + (int64_t)bx.b * a.id * a.ih * a.iw * r.C +
             (first ? chunk : chunk - a.chunks0) * kSChunk;
    return r;
  };
  // line r of the halo; outside the volume the item's first line, zeroed when it is written
  auto load_line = [&](const Source& src, const int (&at)[kR], int r) __attribute__((always_inline)) {
    return *reinterpret_cast<const f4*>(src.base + (int64_t)max(at[r], 0) * src.C +
                                        (threadIdx.x & 3) * 4);
  };
  auto load_prm = [&](int tid, int b) __attribute__((always_inline)) {
    if (!a.nrm0 && !a.nrm1) return;
    for (int c = tid; c < a.c0 + a.c1; c += kSThreads) {
      const float4* pp4 = c < a.c0 ? a.nrm0 : a.nrm1;
      const int C = c < a.c0 ? a.c0 : a.c1;
      const int cc = c < a.c0 ? c : c - a.c0;
      float4 pv = make_float4(0.f, 1.f, 0.f, 0.f);
      if (pp4) pv = pp4[(int64_t)b * C + cc];
      s_prm[c] = pv.x;
      s_prm[kSMaxChannels + c] = pv.y;
      s_prm[2 * kSMaxChannels + c] = pv.z;
    }
  };
  // The pending norm (the apply pass's operations), the split or rounding, and the write.  A
  // voxel's slots: hi of channels 0-7 and 8-15, then lo.
  int slot[kR];  // of each line, in 8 bytes
#pragma unroll
  for (int r = 0; r < kR; ++r) {
    int hz, hy, hx;
    line_voxel(threadIdx.x, r, hz, hy, hx);
    slot[r] = hz < G::hz ? 2 * (hz * kPlaneSlots + voxel_slot(hy, hx)) + ((int)threadIdx.x & 3) : -1;
  }
  auto convert = [&](const f4 (&hl)[kR], const int (&at)[kR], int chunk) __attribute__((always_inline)) {
    const bool first = chunk < a.chunks0;
    const bool norm = (first ? a.nrm0 : a.nrm1) != nullptr;
    const float s = (first ? a.act0 : a.act1) != 0 ? a.slope : 1.f;
    const int q = threadIdx.x & 3;
    f4 mean = {}, scale = {}, beta = {};
    if (norm) {
      const float* prm = s_prm + chunk * kSChunk + q * 4;
      mean = *reinterpret_cast<const f4*>(prm);
      scale = *reinterpret_cast<const f4*>(prm + kSMaxChannels);
      beta = *reinterpret_cast<const f4*>(prm + 2 * kSMaxChannels);
    }
#pragma unroll
    for (int r = 0; r < kR; ++r) {
      if ((r + 1) * kSThreads > G::lines && slot[r] < 0) continue;  // past the halo
      f4 x = hl[r];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (norm) {
          const float t = fmaf(x[e] - mean[e], scale[e], beta[e]);
          x[e] = fmaxf(s * t, t);
        }
        x[e] = at[r] >= 0 ? x[e] : 0.f;
      }
      uint2* dst = reinterpret_cast<uint2*>(s_a) + slot[r];
      if constexpr (AR == kArithBf16) {
        bf4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (__bf16)x[e];
        dst[0] = __builtin_bit_cast(uint2, o);
      } else {
        h4 hv, lv;
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          // hi = fp16(x), lo = fp16(x - hi): one rounding of an exact difference
          const h2 hi = __builtin_convertvector((f2{x[e], x[e + 1]}), h2);
          h2 lo;
          asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(lo) : "v"(hi), "v"(x[e]));
          asm("v_fma_mixhi_f16 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
              : "+v"(lo) : "v"(hi), "v"(x[e + 1]));
          hv[e] = hi[0];
          hv[e + 1] = hi[1];
          lv[e] = lo[0];
          lv[e + 1] = lo[1];
        }
        dst[0] = __builtin_bit_cast(uint2, hv);
        dst[4] = __builtin_bit_cast(uint2, lv);
      }
    }
  };
  // Packed words (16x16x32 fragments): [8-channel chunk][group of 4 taps][16-column block][hi |
  // lo][slot of the group * 16 + column].  Pair p is slots 2 (p % 2) and + 1 of group p / 2; a
  // lane's slot follows its K half, its block and column its MFMA column.
  auto waddr = [&](int lane, int ng, int chunk) {
    const int blk = min(ng * 2 + cb, a.nblk - 1);
    return a.w + (((int64_t)(2 * chunk + h) * 7) * a.nblk16 + blk * 2 + ((lane >> 4) & 1)) * 128 +
           (lane >> 5) * 16 + (lane & 15);
  };
  uint4 ub[kRing][kParts];
  // (in the global address space: a flat load counts as an LDS read too, and every A operand would
  // wait for the weights)
  using Words = const __attribute__((address_space(1))) v4u*;
  const int64_t group = (int64_t)a.nblk16 * 128;
  // pair p at the words of its group; leaves them at the next pair's group (a running address:
  // fourteen of them would fill the scalar registers)
  auto load_w = [&](Words& words, int p) __attribute__((always_inline)) {
#pragma unroll
    for (int part = 0; part < kParts; ++part)
      ub[p % kRing][part] = __builtin_bit_cast(uint4, words[part * 64 + (p & 1) * 32]);
    if (p & 1) {
      words += group;
      asm volatile("" : "+v"(words));
    }
  };

  int at[kR];
  f4 hl[kR];
  {
    const int tid = threadIdx.x;
    const StridedBox first = strided_box(a, v);
    box_lines(tid, first, at);
    const Source src = source(first, cbeg);
#pragma unroll
    for (int r = 0; r < kR; ++r) hl[r] = load_line(src, at, r);
    Words wp = (Words)waddr(tid & 63, first.ng, cbeg);
#pragma unroll
    for (int p = 0; p < kRing; ++p) load_w(wp, p);
    load_prm(tid, first.b);
    lds_barrier();  // the parameters
  }

  for (;;) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const StridedBox cur = strided_box(a, v);
    const int vnext = v + stride;
    const bool more = vnext < vend;
    const StridedBox nxt = more ? strided_box(a, vnext) : cur;
    const int t = lane & 31, g8 = lane >> 5;
    const int blk = cur.ng * 2 + cb;
    const bool live = blk < a.nblk;
    const float bias = a.bias && live ? a.bias[blk * 32 + t] : 0.f;
    // the lane's output voxel (t / 8, t % 8) at tap 0 of the first plane, this half
    const int lane_slot = (t >> 3) * kYPitch + (t & 7) * 4 + h;

    f16v acc[2];
#pragma unroll
    for (int z = 0; z < 2; ++z)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[z][r] = 0.f;

    for (int chunk = cbeg; chunk < cend; ++chunk) {
      const bool last = chunk + 1 == cend;
      convert(hl, at, chunk);
      lds_barrier();
      const int nchunk = last ? cbeg : chunk + 1;
      if (last && more) {
        int tid_n = tid;
        asm volatile("" : "+v"(tid_n));
        box_lines(tid_n, nxt, at);
      }
      const Source src = source(last ? nxt : cur, nchunk);
      Words words = (Words)waddr(lane, cur.ng, chunk) + (kRing >> 1) * group;
      uint4 av[2][2][kParts];
      // the lane's tap of the pair, by its K half (the 28th tap reads the 27th's voxel)
      auto load_a = [&](int p) __attribute__((always_inline)) {
        const int t0 = 2 * p, t1 = min(2 * p + 1, 26);
        const int o0 = t0 / 9 * kPlaneSlots + voxel_slot(t0 / 3 % 3, t0 % 3);
        const int o1 = t1 / 9 * kPlaneSlots + voxel_slot(t1 / 3 % 3, t1 % 3);
        const uint4* src_a = s_a + lane_slot + (g8 ? o1 : o0);
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
          for (int part = 0; part < kParts; ++part)
            av[p & 1][z][part] = src_a[z * SZ * kPlaneSlots + part * 2];
      };
      load_a(0);
#pragma unroll
      for (int p = 0; p < kPairs; ++p) {
        if (p + 1 < kPairs) load_a(p + 1);
        if (p < kR) hl[p] = load_line(src, at, p);
        __builtin_amdgcn_sched_barrier(0);  // a pair's operands are read before the last pair's products
#pragma unroll
        for (int product = 0; product < (kParts == 2 ? 3 : 1); ++product)
#pragma unroll
          for (int z = 0; z < 2; ++z)
            acc[z] = mfma<AR>(av[p & 1][z][product == 2 ? 1 : 0], ub[p % kRing][product == 1 ? 1 : 0], acc[z]);
        if (p + kRing == kPairs) words = (Words)waddr(lane, last ? nxt.ng : cur.ng, nchunk);
        load_w(words, (p + kRing) % kPairs);
      }
      lds_barrier();  // the halo is read
    }

    // ---- epilogue, in the halo's LDS
    float* stage = reinterpret_cast<float*>(s_a) + wave * 1024;
    float* exch = reinterpret_cast<float*>(s_a) + kWaves * 1024;
    float* red = reinterpret_cast<float*>(s_a) + 2 * kWaves * 1024;
    // the two halves of the channels: wave h keeps plane h
    auto swap_halves = [&](const f16v& keep, const f16v& send) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) exch[wave * 1024 + r * 64 + lane] = send[r];
      lds_barrier();
      f16v o;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        o[r] = (keep[r] + exch[(wave ^ 1) * 1024 + r * 64 + lane]) * a.out_scale + bias;
      return o;
    };
    const f16v val = h == 0 ? swap_halves(acc[0], acc[1]) : swap_halves(acc[1], acc[0]);
    const int z = cur.bzi * kBZ + h, y0 = cur.byi * kBY, x0 = cur.bxi * kBX;
    if (a.stats) {
      // accumulator r of a lane: voxel (r / 4, 4 g8 + r % 4) of its column
      auto valid = [&](int r) {
        return z < a.od && y0 + (r >> 2) < a.oh && x0 + 4 * g8 + (r & 3) < a.ow;
      };
      const int nz = min(kBZ, a.od - cur.bzi * kBZ), ny = min(kBY, a.oh - y0);
      const int nx = min(kBX, a.ow - x0);
      const float cnt = (float)(nz * ny * nx);
      float sm = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (valid(r)) sm += val[r];
      sm = add_halves(sm);
      if (lane < 32) red[wave * 32 + t] = sm;
      lds_barrier();
      const float mean = (red[cb * 64 + t] + red[cb * 64 + 32 + t]) / cnt;
      float m2 = 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (valid(r)) {
          const float d = val[r] - mean;
          m2 = fmaf(d, d, m2);
        }
      m2 = add_halves(m2);
      if (lane < 32) red[kWaves * 32 + wave * 32 + t] = m2;
      lds_barrier();
      if (h == 0 && lane < 32 && live) {
        const float tm = red[(kWaves + cb * 2) * 32 + t] + red[(kWaves + cb * 2 + 1) * 32 + t];
        const int tiles = a.nbz * a.nby * a.nbx;
        const int tile = (cur.bzi * a.nby + cur.byi) * a.nbx + cur.bxi;
        a.stats[((int64_t)cur.b * tiles + tile) * a.cout + blk * 32 + t] =
            make_float4(mean, tm, cnt, 0.f);
      }
    }
    // 16-byte channel runs: voxel i of the plane at row (i / 8) * 8 + (i % 4) * 2 + (i / 4) % 2 of the
    // tile, so that a lane's voxels and those 4 further write different banks
    const int quad = lane & 7;
#pragma unroll
    for (int r = 0; r < 16; ++r) stage[((r >> 2) * 8 + (r & 3) * 2 + g8) * 32 + t] = val[r];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rho = i * 8 + (lane >> 3);
      const int yy = y0 + i, xx = x0 + 4 * (rho & 1) + ((rho >> 1) & 3);
      const f4 o = *reinterpret_cast<const f4*>(stage + rho * 32 + quad * 4);
      if (live && z < a.od && yy < a.oh && xx < a.ow)
        *reinterpret_cast<f4*>(a.y + blockIdx.y * a.split_stride +
                               ((((int64_t)cur.b * a.od + z) * a.oh + yy) * a.ow + xx) * a.cout +
                               blk * 32 + quad * 4) = o;
    }
    if (!more) break;
    if (nxt.b != cur.b) load_prm(tid, nxt.b);  // (the last convert lies before a barrier)
    lds_barrier();  // the tiles are read and the parameters there: the next halo may be written
    v = vnext;
  }
}

}  // namespace

int conv_strided_stats_tiles(const ConvGeom& g) {
  return (int)(ceil_div(g.out[0], kBZ) * ceil_div(g.out[1], kBY) * ceil_div(g.out[2], kBX));
}

// Wide layers that fill the chip many times over stay with the implicit GEMM, whose 128 columns share
// a staged halo (us, here against there: 128 -> 256 on 32^3 x 8, 2048 workgroups, 215 against 208;
// 64 -> 128 on 64^3 x 8, 8192, 491 against 486; with stride 1 in z 64 -> 128 on
// 37 x 61 x 43 x 2, 1824, 103 against 100; below: 64 -> 128 on 64^3, 1024, 64 against 73;
// 256 -> 320 on 16^3 x 8, 320, 88 against 106; 320 -> 320 on 8^3 58 against 88).
// So do outputs that leave boxes of 2 x 4 x 8 voxels half empty, where the GEMM's fitted ones come
// to three a CU for four here, or in bf16, where this kernel's boxes are the cheaper, to three for
// five (64 -> 128 to 82 x 32 x 4 x 2, 1312 boxes for 672, 79 against 48, in bf16 48 against 36;
// 128 -> 320 to 30 x 16 x 4 x 2, 600 for 320, 65 against 53, but in bf16 it is 38 against 34 there
// and 28 against 32 on 64 -> 64 to 36 x 32 x 10 x 2, 576 for 432).  While the resident workgroups
// take all boxes in one round this kernel is ahead at any fill (128 -> 128 to 20 x 32 x 4 x 2, 320
// for 160, 45 against 54; in bf16 64 -> 320 to 20 x 16 x 4 x 2, 400 for 200, 17 against 19), but
// for split layers of one to four chunks only up to a box a CU (that layer, 27 against 23).
bool conv_strided_supported(const ConvGeom& g, int c1, int c2, int cout, int arith) {
  if (!conv_strided_layer(g, c1, c2, cout)) return false;
  const int64_t cus = compute_units(), groups = ceil_div(cout, 64);
  const int64_t boxes = (int64_t)g.batch * conv_strided_stats_tiles(g) * groups;
  if (cout > 64 && boxes >= 6 * cus) return false;
  const int64_t resident = arith == kArithSplit3 && c1 + c2 <= 64 ? cus : 2 * cus;
  return boxes <= resident ||
         3 * ceil_div(boxes, cus) <
             (arith == kArithSplit3 ? 4 : 5) * ceil_div(conv_x3_boxes(g) * groups, cus);
}

bool conv_strided_layer(const ConvGeom& g, int c1, int c2, int cout) {
  for (int i = 0; i < 3; ++i)
    if (g.k[i] != 3) return false;
  return (g.s[0] == 1 || g.s[0] == 2) && g.s[1] == 2 && g.s[2] == 2 && c1 > 0 && c1 % kSChunk == 0 &&
         c2 % kSChunk == 0 && c1 + c2 <= kSMaxChannels && cout % 32 == 0 &&
         (int64_t)g.in[0] * g.in[1] * g.in[2] < (1LL << 31);
}

// As the register-staged kernel's: chunks over the idle CUs, at least two a workgroup.
int conv_strided_splits(const ConvGeom& g, int c1, int c2, int cout) {
  const int64_t boxes = (int64_t)g.batch * conv_strided_stats_tiles(g) * ceil_div(cout, 64);
  const int chunks = (c1 + c2) / kSChunk;
  const int64_t spatial = (int64_t)g.out[0] * g.out[1] * g.out[2];
  const int64_t most = std::min<int64_t>(2 * compute_units() / boxes, chunks / 2);
  if (most < 2 || !split_sum_supported(spatial, cout)) return 1;
  if (split_sum_parts(spatial) > 1 && chunks < 8) return 1;
  return (int)ceil_div(chunks, ceil_div(chunks, most));
}

void conv3d_strided(const float* x1, int c1, const float* x2, int c2, const void* packed,
                    int nblk16, float scale, const float* bias, float* y, const ConvGeom& g,
                    int cout, hipStream_t st, float4* stats, const PendingNorm& n1,
                    const PendingNorm& n2, int arith, int splits) {
  StridedArgs a{};
  a.x0 = x1;
  a.x1 = x2;
  a.c0 = c1;
  a.c1 = c2;
  a.chunks0 = c1 / kSChunk;
  a.chunks = a.chunks0 + c2 / kSChunk;
  a.w = reinterpret_cast<const uint4*>(packed);
  a.nblk16 = nblk16;
  a.bias = bias;
  a.y = y;
  a.id = g.in[0];
  a.ih = g.in[1];
  a.iw = g.in[2];
  a.od = g.out[0];
  a.oh = g.out[1];
  a.ow = g.out[2];
  a.cout = cout;
  a.nblk = cout / 32;
  a.nbz = (int)ceil_div(g.out[0], kBZ);
  a.nby = (int)ceil_div(g.out[1], kBY);
  a.nbx = (int)ceil_div(g.out[2], kBX);
  const int64_t nwg = (int64_t)g.batch * a.nbz * a.nby * a.nbx * ceil_div(a.nblk, 2);
  require(nwg < (1LL << 31), "convolution grid too large");
  a.nvirt = (int)nwg;
  a.nbox = a.nvirt / (int)ceil_div(a.nblk, 2);
  a.cper = (int)ceil_div(a.chunks, splits);
  a.split_stride = (int64_t)g.batch * g.out[0] * g.out[1] * g.out[2] * cout;
  a.out_scale = 1.0f / scale;
  a.stats = stats;
  a.nrm0 = n1.params;
  a.nrm1 = n2.params;
  a.act0 = n1.act ? 1 : 0;
  a.act1 = n2.act ? 1 : 0;
  a.slope = n1.params ? n1.slope : n2.slope;
  const double out_vox = (double)g.batch * g.out[0] * g.out[1] * g.out[2];
  ProfScope prof(arith == kArithBf16 ? "conv3d_x3_bf16_strided" : "conv3d_x3_strided",
                 2.0 * (c1 + c2) * cout * 27.0 * out_vox,
                 4.0 * ((double)g.batch * g.in[0] * g.in[1] * g.in[2] * (c1 + c2) + out_vox * cout),
                 st);
  const dim3 grid((unsigned)std::min<int64_t>(2 * compute_units(), ceil_div(nwg, 8) * 8),
                  (unsigned)ceil_div(a.chunks, a.cper)), block(kSThreads);
  if (arith == kArithBf16) {
    if (g.s[0] == 2)
      hipLaunchKernelGGL((conv_strided_kernel<2, kArithBf16>), grid, block, 0, st, a);
    else
      hipLaunchKernelGGL((conv_strided_kernel<1, kArithBf16>), grid, block, 0, st, a);
  } else if (g.s[0] == 2) {
    hipLaunchKernelGGL((conv_strided_kernel<2, kArithSplit3>), grid, block, 0, st, a);
  } else {
    hipLaunchKernelGGL((conv_strided_kernel<1, kArithSplit3>), grid, block, 0, st, a);
  }
  launch_check("conv3d_strided");
}

}  // namespace nnx
