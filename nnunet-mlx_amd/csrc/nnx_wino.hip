// Convolution of the stride-1, padding-1 3x3x3 layers: Winograd F(2x2, 3x3) in the (y, x)
// plane, the three z taps summed directly, with split-fp16 products (hi*hi + hi*lo + lo*hi,
// float32 accumulation) on v_mfma_f32_32x32x16_f16.
//
// For each z plane a 2x2 output tile is Y = A^T [ sum_kz U[kz] (.) V[z + kz - 1] ] A, with
// V = B^T d B the transform of the tile's 4x4 input patch and U[kz] = G w[kz] G^T the
// transform of the filter's kz slice (F(2,3): B^T = [1 0 -1 0; 0 1 1 0; 0 -1 1 0; 0 1 0 -1],
// G = [1 0 0; .5 .5 .5; .5 -.5 .5; 0 0 1], A^T = [1 1 1 0; 0 1 -1 -1]).  Summed over input
// channels and z taps, each of the 16 transform positions xi = (xy, xx) is an independent
// GEMM.  Against F(2x2x2) in all three axes this issues 12 products an output instead of 8,
// but transforms and splits 4 values an output instead of 8, keeps 4 accumulators an output
// instead of 8 (so the register file holds a box of twice the voxels) and reads each
// transformed plane for three output planes; the three-axis form was bound by the VALU work
// of the transform and split and by the fixed cost of its small boxes, with the matrix cores
// 15 % busy.  The transforms are exact additions of float32 values (and the 1/2 of G, exact),
// so the arithmetic stays float32-class; U is formed in float64 and rounded once, V in
// float32, each then split into fp16 halves.  V adds up to 4 inputs.
//
// Workgroup: 8 waves (two a SIMD), an output box of ZB z planes x 32 tiles (4 x 8 tiles =
// 8 x 16 voxels; 8 x 4 tiles, or 4 x 4 in two slabs of planes, where that wastes less) and 32
// output channels.  Wave
// w = 2 xy + h owns the positions (xy, xx = 0, 1) for h = 0 and (xy, xx = 3, 2) for h = 1: its
// accumulators are 2 x ZB blocks of 32 x 32 floats (128 registers a lane at ZB = 4), which
// leaves room for a second wave on the SIMD to issue while one waits.  Per chunk of 16 input
// channels:
//   1. the raw halo, (ZB + 2) planes, was fetched by global_load_lds_dwordx4 into one of two
//      LDS buffers during the previous chunk, its slots laid out so that the 32 tiles of a
//      half-wave read 32 different 16-byte bank groups;
//   2. each thread applies the input's pending InstanceNorm (+ LeakyReLU) in place to the
//      lines that it fetched itself (so it waits for its own loads only); one barrier, behind
//      which it waits for U too;
//   3. the next chunk's halo DMA is issued, into the other buffer;
//   4. per input plane each wave reads the two rows and three columns of its positions'
//      patches, forms V, splits it in registers and issues the products with the packed U of
//      every z tap that reaches an output plane of the box (up to 18 MFMAs).  U (2 positions x
//      3 taps, 48 registers) is reloaded from L2 tap by tap as the chunk's last product with it
//      is issued, so its latency is covered by the planes that follow.
//
// Sums: an accumulator rounds once a product, and that is most of the error: squared and
// relative it measures 1.5e-15 a rounding, in accumulators that hold three z taps and three
// products a chunk.  From four chunks on two of the taps are therefore summed from zero, their
// small products first, and added as one (4 roundings a chunk instead of 9) in half the output
// planes, from six chunks in all; it takes the last plane's V in registers and 16 additions for
// six products.
// Epilogue, a z plane at a time: each wave applies its share of the x-output transform and
// writes its two partials to LDS, and a thread sums the eight waves' partials of one tile
// column for four output channels (y-output transform), scales back, adds the bias and stores
// 16 bytes; the InstanceNorm partials of the box are reduced from the same registers.
//
// The kernel is persistent: one workgroup a CU loops over boxes.  The eight XCDs take contiguous
// ranges of the (column block, box) pairs, column block slowest, so an XCD's L2 holds one
// column block's packed weights and neighbouring boxes' halos.  The last chunk of a box
// issues the next box's first halo DMA and U loads; the epilogue exchanges through the raw
// buffer that this DMA does not target.
//
// Bound by power and issue together: the matrix cores are 33 % busy in 32 + 32 -> 32 on 128^3 x 8
// and 36 % in 128 -> 128 on 32^3 x 8 (23 % in the 32-channel layers of a network, two chunks a
// box), a wave issues VALU work in 25 to 27 % of its cycles and waits in 27 to 30 %.  With plain
// sums, leaving out any one part of 128 -> 128 (products 38 %, halo DMA 21 %, transform and split
// 18 %, epilogue 11 %, patch reads 9 %, U loads 7 %) took its share off the time, and the clock
// rose from 1.9 to 2.4 GHz without the products.  The kernels of 4-plane boxes are at the register
// limit of 256: those with half the sums apart spill one (8 bytes a lane), and all of them 56 to 61
// scalar registers to vector lanes.
// Measured, three-axis form / plain sums / now, us and relative error against float64:
//   32 + 32 -> 32 on 128^3 x 8       4300 / 3615 / 3730   2.62 / 2.79 / 2.52e-7  (498 TFLOP/s of
//                                                          the direct convolution's work)
//   128 -> 128 on 32^3 x 8            464 /  402 /  411   3.06 / 3.54 / 2.61e-7  (564)
//   64 -> 64 on 37 x 61 x 43 x 4      245 /  219 /  219   2.61 / 2.78 / 2.52e-7  (392)
//   256 + 256 -> 256 on 16^3 x 8      415 /  366 /  382   5.18 / 6.65 / 4.44e-7
//   320 -> 320 on 5 x 6 x 7          65.4 / 60.2 / 61.6   4.19 / 5.20 / 3.56e-7 (on 12 x 13 x 11)
//   32 -> 192 on 6 x 9 x 8 x 8       12.7 / 13.4 / 12.6   2.40 / 2.24 / 2.24e-7
#include <cmath>
#include <string>
#include <type_traits>

#include "nnx_internal.h"

namespace nnx {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

constexpr int kWThreads = 512;    // 8 waves, two a SIMD
constexpr int kWChunk = 16;       // input channels per chunk (one MFMA K)
constexpr int kMaxChannels = 1024;  // c1 + c2 (pending-norm parameters in LDS)
constexpr int kPlane = 768;       // 16-byte slots of a raw halo plane: 1.5 rounds of the workgroup
constexpr int kPositions = 16;    // transform positions (xy, xx)
constexpr int kTapWords = 128;    // packed words of one (position, z tap): hi, lo x 64 lanes
constexpr int kPartSlots = 8 * 2 * 32 * 8;  // epilogue partials: wave, ox, tile, 4 columns
constexpr int kRedSlots = 2 * 8 * 8;        // InstanceNorm partials: pass, wave, 4 columns

// Box shapes: tiles of a z plane side by side (wide, tall), or two slabs of ZB planes with 4 x 4
// tiles each (cube), the MFMA rows 16-31 taking the upper slab.
enum WinoShape { kWide, kTall, kCube };

// Box geometry.  A raw halo plane is stored as [y / 2][y % 2][x % 2][x / 2] (tile rows and
// columns are every second row and column) with q = channel quad fastest: slot = yi * py +
// jump * (yi / 4) + yp * pyp + xp * pxp + xi * 4 + q.  For a fixed (row, column, quad) of the
// patch the 32 tiles then fall on 32 different slots modulo 32 (ds_read_b128 serves 32 lanes
// a pass from 32 16-byte groups); the cube's plane stride puts its two slabs 16 slots apart.
template <int ZB, WinoShape S>
struct WinoBoxGeom {
  static constexpr int slabs = S == kCube ? 2 : 1;
  static constexpr int ty = S == kTall ? 8 : 4, tx = S == kWide ? 8 : 4;  // tiles
  static constexpr int by = 2 * ty, bx = 2 * tx, bz = ZB * slabs;  // output voxels
  static constexpr int hz = bz + 2, hy = by + 2, hx = bx + 2;       // halo
  static constexpr int pxp = (tx + 1) * 4, pyp = 2 * pxp, py = 2 * pyp + 1;
  static constexpr int jump = S == kTall ? 12 : 0;
  static constexpr int plane = S == kCube ? 408 : kPlane;
  static constexpr int rounds = (hz * plane + kWThreads - 1) / kWThreads;
  // in-plane patterns of a thread's rounds: three for plane pairs of 1.5 rounds each, else one
  // voxel a round
  static constexpr int lines = S == kCube ? rounds : 3;
  static constexpr int slots = rounds * kWThreads;
  // the epilogue's partials and reductions use one raw buffer
  static constexpr int buf = slots > kPartSlots + kRedSlots ? slots : kPartSlots + kRedSlots;
  static_assert(py * ty + jump * (ty / 4) + 2 * pyp <= plane, "a halo plane fits its slots");
  static_assert(S == kCube || hz % 2 == 0, "plane pairs are three rounds of the workgroup");
  static_assert(S != kCube || ZB * plane % 32 == 16, "the slabs' tiles interleave");
  static_assert(2 * buf * 16 + 3 * kMaxChannels * 4 + 128 <= 160 * 1024, "LDS");
};

struct WinoArgs {
  const float* x0;
  const float* x1;
  int c0, c1, chunks0, chunks;
  const uint4* u;  // packed transformed weights
  const float* bias;
  float* y;
  int D, H, W;
  int cout;
  int nbz, nby, nbx;
  int nbox;   // batch * nbz * nby * nbx (boxes of one column block)
  int nvirt;  // nbox * cout / 32: (column block, box) pairs, column block slowest
  int cper;   // chunks of a workgroup: blockIdx.y takes chunks [cper blockIdx.y, + cper)
  int64_t split_stride;  // elements between the outputs of two blockIdx.y
  float out_scale;
  float4* stats;
  const float4* nrm0;
  const float4* nrm1;
  int act0, act1;
  float slope;
  unsigned rbox, rz, ry, rx;  // reciprocals of nbox, nbz, nby, nbx
};

// n / d by d's reciprocal floor((2^32 - 1) / d): the product is the quotient or one less, as n is
// below 2^32.  (A box takes twelve of them before its first load: as divisions they were 0.4 us of
// every launch.)
inline unsigned reciprocal(int d) { return 0xffffffffu / (unsigned)d; }
__device__ __forceinline__ int divide(int n, int d, unsigned r) {
  const int q = (int)__umulhi((unsigned)n, r);
  return n - q * d >= d ? q + 1 : q;
}

// 16 zero bytes: halo lines outside the volume are fetched from here.
__device__ __align__(16) float g_wino_zero[4];

__device__ __forceinline__ f16v mfma32(h8 a, h8 b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// hi = fp16(v) (nearest even), lo = fp16(v - hi).  v - hi is exact in float32, so the
// single rounding of v_fma_mix{lo,hi}_f16 (fma(-hi, 1, v) formed exactly, rounded once to
// fp16) gives the same lo as converting hi back, subtracting and converting: one
// instruction per element instead of three.
__device__ __forceinline__ void split8(const float (&v)[8], h8& hi, h8& lo) {
#pragma unroll
  for (int q = 0; q < 8; q += 2) {
    const h2 h = __builtin_convertvector((f2{v[q], v[q + 1]}), h2);
    h2 l;
    asm("v_fma_mixlo_f16 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(l) : "v"(h), "v"(v[q]));
    asm("v_fma_mixhi_f16 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "+v"(l) : "v"(h), "v"(v[q + 1]));
    hi[q] = h[0];
    hi[q + 1] = h[1];
    lo[q] = l[0];
    lo[q + 1] = l[1];
  }
}

// Six patch points (two rows x columns P, Q, R; 8 channels each, two 16-byte reads) at LDS byte
// addresses ad[row * 3 + column] + OFFSET, with the wait for them.  Written as
// one asm block so that the compiler's wait-count pass does not see LDS reads here: it
// would otherwise order them behind the halo DMA in flight to the other buffer (it cannot
// tell the two apart) and wait for that DMA first.
template <int OFFSET>
__device__ __forceinline__ void read_patch(const unsigned (&ad)[6], f4 (&v)[12]) {
  asm volatile(
      "ds_read_b128 %0, %12 offset:%18\n\tds_read_b128 %1, %12 offset:%19\n\t"
      "ds_read_b128 %6, %15 offset:%18\n\tds_read_b128 %7, %15 offset:%19\n\t"
      "ds_read_b128 %2, %13 offset:%18\n\tds_read_b128 %3, %13 offset:%19\n\t"
      "ds_read_b128 %8, %16 offset:%18\n\tds_read_b128 %9, %16 offset:%19\n\t"
      "ds_read_b128 %4, %14 offset:%18\n\tds_read_b128 %5, %14 offset:%19\n\t"
      "ds_read_b128 %10, %17 offset:%18\n\tds_read_b128 %11, %17 offset:%19\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
        "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11])
      : "v"(ad[0]), "v"(ad[1]), "v"(ad[2]), "v"(ad[3]), "v"(ad[4]), "v"(ad[5]),
        "n"(OFFSET), "n"(OFFSET + 16)
      : "memory");
}

// The same by columns, two (P and Q) and one (R).
template <int OFFSET>
__device__ __forceinline__ void read_column(unsigned a0, unsigned a1, f4 (&v)[4]) {
  asm volatile(
      "ds_read_b128 %0, %4 offset:%6\n\tds_read_b128 %1, %4 offset:%7\n\t"
      "ds_read_b128 %2, %5 offset:%6\n\tds_read_b128 %3, %5 offset:%7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
      : "v"(a0), "v"(a1), "n"(OFFSET), "n"(OFFSET + 16)
      : "memory");
}

template <int OFFSET>
__device__ __forceinline__ void read_columns(unsigned a0, unsigned a1, unsigned b0, unsigned b1,
                                             f4 (&v)[4], f4 (&w)[4]) {
  asm volatile(
      "ds_read_b128 %0, %8 offset:%12\n\tds_read_b128 %1, %8 offset:%13\n\t"
      "ds_read_b128 %2, %9 offset:%12\n\tds_read_b128 %3, %9 offset:%13\n\t"
      "ds_read_b128 %4, %10 offset:%12\n\tds_read_b128 %5, %10 offset:%13\n\t"
      "ds_read_b128 %6, %11 offset:%12\n\tds_read_b128 %7, %11 offset:%13\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(w[0]), "=&v"(w[1]),
        "=&v"(w[2]), "=&v"(w[3])
      : "v"(a0), "v"(a1), "v"(b0), "v"(b1), "n"(OFFSET), "n"(OFFSET + 16)
      : "memory");
}

// x summed over the eight lanes of a wave that share lane % 8, in every lane: a rotation by
// 8 within rows of 16, then v_permlane16_swap and v_permlane32_swap (each leaves a pair's two
// values in every lane of the pair).
__device__ __forceinline__ float sum_stride8(float x) {
  x += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0x128, 0xf, 0xf, false));
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

__device__ __forceinline__ f4 sum_stride8(f4 v) {
  f4 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) r[e] = sum_stride8(v[e]);
  return r;
}

// Barrier that waits for this wave's LDS accesses only (not __syncthreads(), whose release
// fence would also wait for the halo DMA and the stores in flight).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct WinoBox {
  int nt, b, bzi, byi, bxi;
};

__device__ __forceinline__ WinoBox wino_box(const WinoArgs& a, int v) {
  WinoBox r;
  r.nt = divide(v, a.nbox, a.rbox);
  int box = v - r.nt * a.nbox;
  int q = divide(box, a.nbx, a.rx);
  r.bxi = box - q * a.nbx;
  box = q;
  q = divide(box, a.nby, a.ry);
  r.byi = box - q * a.nby;
  r.b = divide(q, a.nbz, a.rz);
  r.bzi = q - r.b * a.nbz;
  return r;
}

// CH: output planes of a slab whose first two z taps are summed apart.
template <int ZB, WinoShape S, int CH>
__global__ __launch_bounds__(kWThreads, 1) void wino_yx_kernel(WinoArgs a) {
  using G = WinoBoxGeom<ZB, S>;
  __shared__ __align__(16) f4 s_raw[2 * G::buf];             // two raw halo buffers
  __shared__ __align__(16) float s_prm[3 * kMaxChannels];    // mean, scale, beta by channel
  __shared__ __align__(16) float s_bias[32];                 // of the current column block
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  // this workgroup's (column block, box) pairs: XCD blockIdx % 8 takes a contiguous range,
  // its workgroups interleave over it (the grid is a multiple of 8)
  const int xcd = blockIdx.x & 7, stride = gridDim.x >> 3;
  const int vq = a.nvirt >> 3, vr = a.nvirt & 7;
  const int vbeg = xcd < vr ? xcd * (vq + 1) : vr * (vq + 1) + (xcd - vr) * vq;
  const int vend = vbeg + vq + (xcd < vr ? 1 : 0);
  int v = vbeg + (int)(blockIdx.x >> 3);
  if (v >= vend) return;  // uniform over the workgroup, before any barrier
  const int cbeg = blockIdx.y * a.cper, cend = min(cbeg + a.cper, a.chunks);
  __builtin_assume(cend > cbeg);
  const int64_t plane_vox = (int64_t)a.H * a.W;
  constexpr int kRounds = G::rounds, kL = G::lines;
  uint64_t zero = (uint64_t)g_wino_zero;
  asm volatile("" : "+s"(zero));  // held, not loaded from the GOT at every use

  // ---- raw halo lines.  Wide and tall: round 3 k + j of this thread is slot j * 512 + tid of the
  // plane pair 2 k, 2 k + 1: three in-plane patterns j, the plane uniform over a wave; `at` is
  // their in-plane voxel.  Cube: round r is slot r * 512 + tid of all planes, `at` its voxel in
  // the item.  -1 outside the volume or on a padding slot; `quads`: two bits a pattern.
  auto round_plane = [&](int k, int j) { return 2 * k + ((j == 2 || (j == 1 && wave >= 4)) ? 1 : 0); };
  auto box_lines = [&](int tid, const WinoBox& bx, int (&at)[kL], int& quads)
      __attribute__((always_inline)) {
    quads = 0;
#pragma unroll
    for (int j = 0; j < kL; ++j) {
      int s, hz = 0;
      if constexpr (S == kCube) {
        hz = (j * kWThreads + tid) / G::plane;
        s = j * kWThreads + tid - hz * G::plane;
      } else {
        s = j == 0 ? tid : j == 1 ? (tid < 256 ? 512 + tid : tid - 256) : 256 + tid;
      }
      int t = s;
      if constexpr (S == kTall) t = s < G::py * 4 + G::jump ? s : s < G::py * 8 + 2 * G::jump ? s - G::jump
                                                                                             : s - 2 * G::jump;
      const int yi = t / G::py, rem = t - yi * G::py;
      const int yp = rem / G::pyp, rx = rem - yp * G::pyp;
      const int xp = rx / G::pxp, rq = rx - xp * G::pxp;
      const int hy = 2 * yi + yp, hx = 2 * (rq >> 2) + xp;
      const int yy = bx.byi * G::by - 1 + hy, xx = bx.bxi * G::bx - 1 + hx;
      const int zz = bx.bzi * G::bz - 1 + hz;
      bool line = s - t == G::jump * (yi >> 2) && rem < 2 * G::pyp && hy < G::hy && hx < G::hx &&
                  (unsigned)yy < (unsigned)a.H && (unsigned)xx < (unsigned)a.W;
      if constexpr (S == kCube) line = line && hz < G::hz && (unsigned)zz < (unsigned)a.D;
      at[j] = line ? (S == kCube ? zz * a.H + yy : yy) * a.W + xx : -1;
      quads |= (rq & 3) << (2 * j);
    }
  };
  // A chunk of a box's halo into buffer `buf`, during the previous chunk's products.  The address of
  // a pattern is formed once for its planes (formed for each round and spread over the planes,
  // 128 -> 128 on 32^3 x 8 took 449 us instead of 436).
  struct Source {
    uint64_t base;         // channel chunk of the halo's first plane (may lie outside the volume;
                           // cube: of the item)
    int64_t plane_bytes;
    int C, z0;
  };
  auto source = [&](const WinoBox& bx, int chunk) __attribute__((always_inline)) {
    const bool first = chunk < a.chunks0;
    Source r;
    r.C = first ? a.c0 : a.c1;
    r.plane_bytes = plane_vox * r.C * 4;
    r.z0 = S == kCube ? 0 : bx.bzi * G::bz - 1;
    r.base = (uint64_t)(first ? a.x0 : a.x1) + ((int64_t)bx.b * a.D + r.z0) * r.plane_bytes +
             (first ? chunk : chunk - a.chunks0) * kWChunk * 4;
    return r;
  };
  auto fetch = [&](const Source& src, const int (&at)[kL], int quads, int buf) __attribute__((always_inline)) {
    f4* dst = s_raw + buf * G::buf + wave * 64;
#pragma unroll
    for (int j = 0; j < kL; ++j) {
      // this thread's line of the pattern in plane 0 (cube: the line)
      const uint64_t line = src.base + ((int64_t)at[j] * src.C + ((quads >> (2 * j)) & 3) * 4) * 4;
      constexpr int kPer = S == kCube ? 1 : G::hz / 2;
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int r = S == kCube ? j : 3 * k + j;
        const int p = S == kCube ? 0 : round_plane(k, j);
        const bool in = at[j] >= 0 && (unsigned)(src.z0 + p) < (unsigned)a.D;
        const uint64_t g = in ? line + p * src.plane_bytes : zero;
        __builtin_amdgcn_global_load_lds(
            (const void*)g, (__attribute__((address_space(3))) void*)(dst + r * kWThreads), 16, 0, 0);
      }
    }
  };
  // pending-norm parameters of every input channel (both inputs, in chunk order) of item b
  auto load_prm = [&](int tid, int b) __attribute__((always_inline)) {
    if (!a.nrm0 && !a.nrm1) return;
    for (int c = tid; c < a.c0 + a.c1; c += kWThreads) {
      const float4* pp = c < a.c0 ? a.nrm0 : a.nrm1;
      const int C = c < a.c0 ? a.c0 : a.c1;
      const int cc = c < a.c0 ? c : c - a.c0;
      float4 pv = make_float4(0.f, 1.f, 0.f, 0.f);
      if (pp) pv = pp[(int64_t)b * C + cc];
      s_prm[c] = pv.x;
      s_prm[kMaxChannels + c] = pv.y;
      s_prm[2 * kMaxChannels + c] = pv.z;
    }
  };
  // The input's pending InstanceNorm on this thread's lines of the chunk, in place (the apply
  // pass's operations: t = fma(x - mean, scale, beta), then max(s * t, t) with s = the
  // LeakyReLU slope under the activation and s = 1, the identity, without it).  Lines outside
  // the volume stay zero.
  auto normalise = [&](const WinoBox& bx, const int (&at)[kL], int quads, int chunk, int buf)
      __attribute__((always_inline)) {
    const bool first = chunk < a.chunks0;
    if ((first ? a.nrm0 : a.nrm1) == nullptr) return;
    const float s = (first ? a.act0 : a.act1) != 0 ? a.slope : 1.f;
    f4* lines = s_raw + buf * G::buf + threadIdx.x;
    constexpr int kPer = S == kCube ? 1 : G::hz / 2;  // rounds of a pattern
#pragma unroll
    for (int j = 0; j < kL; ++j) {
      if (at[j] < 0) continue;
      const float* prm = s_prm + chunk * kWChunk + ((quads >> (2 * j)) & 3) * 4;
      const f4 mean = *reinterpret_cast<const f4*>(prm);
      const f4 scale = *reinterpret_cast<const f4*>(prm + kMaxChannels);
      const f4 beta = *reinterpret_cast<const f4*>(prm + 2 * kMaxChannels);
      f4 d[kPer];
#pragma unroll
      for (int k = 0; k < kPer; ++k) d[k] = lines[(kPer == 1 ? j : 3 * k + j) * kWThreads];
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        if constexpr (S != kCube) {
          const int z = bx.bzi * G::bz - 1 + round_plane(k, j);
          if ((unsigned)z >= (unsigned)a.D) continue;  // uniform over the wave
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float t = fmaf(d[k][e] - mean[e], scale[e], beta[e]);
          d[k][e] = fmaxf(s * t, t);
        }
        lines[(kPer == 1 ? j : 3 * k + j) * kWThreads] = d[k];
      }
    }
  };

  // ---- this wave's positions: row pair (a, b) and sign of xy, columns P, Q, R and sign of xx.
  // Q0 = d[a] + sy d[b]; the first position is P - Q (xx = 0, or minus xx = 3, a sign that
  // the output transform undoes), the second R + sx Q (xx = 1 or 2).
  const int xy = wave >> 1, h = wave & 1;
  const int ra = xy == 0 ? 0 : xy == 2 ? 2 : 1, rb = xy == 2 ? 1 : xy == 3 ? 3 : 2;
  const float sy = xy == 1 ? 1.f : -1.f;
  const int cp = h ? 3 : 0, cq = h ? 1 : 2, cr = h ? 2 : 1;
  const float sx = h ? -1.f : 1.f;
  // packed U: [nt][chunk][position in wave order][z tap][hi | lo][64 lanes] x 16 bytes
  auto uaddr = [&](int lane, int nt, int chunk) {
    return a.u + (((int64_t)nt * a.chunks + chunk) * kPositions + 2 * wave) * 3 * kTapWords + lane;
  };
  uint4 ub[2][3][2];  // [position][z tap][hi | lo]
  auto load_u = [&](const uint4* base, int kz) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int part = 0; part < 2; ++part)
        ub[p][kz][part] = base[(p * 3 + kz) * kTapWords + part * 64];
  };

  // loop-carried: the lines of the box whose first chunk is in flight, its U, the raw buffer
  int yx[kL], quads, buf = 0;
  {
    const int tid = threadIdx.x;
    const WinoBox first = wino_box(a, v);
    box_lines(tid, first, yx, quads);
    fetch(source(first, cbeg), yx, quads, 0);
    const uint4* up = uaddr(tid & 63, first.nt, cbeg);
#pragma unroll
    for (int kz = 0; kz < 3; ++kz) load_u(up, kz);
    load_prm(tid, first.b);  // (behind the halo, whose latency theirs hides in)
    if (tid < 32) s_bias[tid] = a.bias ? a.bias[first.nt * 32 + tid] : 0.f;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();  // the parameters and the bias
  }

  for (;;) {
    // per-lane values rebuilt from an opaque copy each box, so that nothing derived from
    // them is hoisted out of the box loop and held through it
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const WinoBox cur = wino_box(a, v);
    const int vnext = v + stride;
    const bool more = vnext < vend;
    const WinoBox nxt = more ? wino_box(a, vnext) : cur;

    // LDS byte addresses of this lane's six patch points in plane 0 of buffer 0
    unsigned ad[6];
    {
      const int t = lane & 31, g8 = lane >> 5;
      const int tyl = S == kWide ? t >> 3 : S == kTall ? t >> 2 : (t >> 2) & 3;
      const int txl = S == kWide ? t & 7 : t & 3;
      const int slab = S == kCube ? (t >> 4) * ZB * G::plane : 0;
      const unsigned raw0 = (unsigned)(uintptr_t)((__attribute__((address_space(3))) f4*)s_raw);
      auto point = [&](int r, int c) {
        const int yi = tyl + (r >> 1);
        return raw0 + 16u * (unsigned)(slab + yi * G::py + G::jump * (yi >> 2) + (r & 1) * G::pyp +
                                       (c & 1) * G::pxp + (txl + (c >> 1)) * 4 + 2 * g8);
      };
      ad[0] = point(ra, cp);
      ad[1] = point(ra, cq);
      ad[2] = point(ra, cr);
      ad[3] = point(rb, cp);
      ad[4] = point(rb, cq);
      ad[5] = point(rb, cr);
    }
    {
      const unsigned o = buf ? (unsigned)(G::buf * 16) : 0u;
#pragma unroll
      for (int i = 0; i < 6; ++i) ad[i] += o;
    }

    f16v acc[2][ZB];
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int z = 0; z < ZB; ++z)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[p][z][r] = 0.f;

    // Input plane Z of the halo: V of both positions, then its products.  z tap 2 of an output plane
    // is added to its accumulator, tap 0 and 1 too from plane CH on; below it they are summed
    // from zero, the small products first, once both planes' V are there, and then added.
    h8 vh[2][2], vl[2][2];  // V of this plane and the last, split: [plane & 1][position]
    auto plane = [&](auto zc) __attribute__((always_inline)) {
      constexpr int Z = decltype(zc)::value, kAt = Z * G::plane * 16, now = Z & 1;
      constexpr bool chain = Z >= 1 && Z - 1 < CH;
      if constexpr (chain && ZB == 4) {
        // (two columns, then one: the last plane's V is held too, and the registers are full)
        float vq[8];
        {
          f4 dp[4], dq[4];
          read_columns<kAt>(ad[0], ad[3], ad[1], ad[4], dp, dq);
          float va[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            vq[e] = fmaf(sy, dq[2 + (e >> 2)][e & 3], dq[e >> 2][e & 3]);
            va[e] = fmaf(sy, dp[2 + (e >> 2)][e & 3], dp[e >> 2][e & 3]) - vq[e];
          }
          split8(va, vh[now][0], vl[now][0]);
        }
        __builtin_amdgcn_sched_barrier(0);
        f4 dr[4];
        read_column<kAt>(ad[2], ad[5], dr);
        float vb[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          vb[e] = fmaf(sx, vq[e], fmaf(sy, dr[2 + (e >> 2)][e & 3], dr[e >> 2][e & 3]));
        split8(vb, vh[now][1], vl[now][1]);
        __builtin_amdgcn_sched_barrier(0);
      } else {
        f4 d[12];
        read_patch<kAt>(ad, d);
        float va[8], vb[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float vp = fmaf(sy, d[6 + (e >> 2)][e & 3], d[e >> 2][e & 3]);
          const float vq = fmaf(sy, d[8 + (e >> 2)][e & 3], d[2 + (e >> 2)][e & 3]);
          const float vr = fmaf(sy, d[10 + (e >> 2)][e & 3], d[4 + (e >> 2)][e & 3]);
          va[e] = vp - vq;
          vb[e] = fmaf(sx, vq, vr);
        }
        split8(va, vh[now][0], vl[now][0]);
        split8(vb, vh[now][1], vl[now][1]);
      }
      // product 0: lo * hi, 1: hi * lo, 2: hi * hi
      auto product = [&](int which, int v, int p, int kz, f16v c) __attribute__((always_inline)) {
        return mfma32(which == 0 ? vl[v][p] : vh[v][p],
                      *reinterpret_cast<const h8*>(&ub[p][kz][which == 1 ? 1 : 0]), c);
      };
      if constexpr (chain) {
        if constexpr (ZB == 2) {
          f16v t[2]{};
#pragma unroll
          for (int i = 0; i < 6; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) t[p] = product(i >> 1, (Z - 1 + (i & 1)) & 1, p, i & 1, t[p]);
          if constexpr (Z >= 2) {
#pragma unroll
            for (int i = 0; i < 6; ++i)
              acc[i & 1][Z - 2] = product(2 - (i >> 1), now, i & 1, 2, acc[i & 1][Z - 2]);
          }
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            acc[p][Z - 1] += t[p];
            asm volatile("" : "+v"(acc[p][Z - 1]));  // added here, not where it is used next
          }
        } else {
          // (one position after the other: the registers hold one sum.  The third tap's products
          // of both positions cover the wait for the first)
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            f16v t{};
#pragma unroll
            for (int i = 0; i < 6; ++i) t = product(i >> 1, (Z - 1 + (i & 1)) & 1, p, i & 1, t);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (Z >= 2) {
#pragma unroll
              for (int i = 0; i < 6; ++i)
                if (p == 0) acc[i & 1][Z - 2] = product(2 - (i >> 1), now, i & 1, 2, acc[i & 1][Z - 2]);
              __builtin_amdgcn_sched_barrier(0);
            }
            acc[p][Z - 1] += t;
            asm volatile("" : "+v"(acc[p][Z - 1]));  // added here: left to its next use, t is held till then
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
#pragma unroll
      for (int which = 2; which >= 0; --which)
#pragma unroll
        for (int kz = 0; kz < 3; ++kz) {
          const int o = Z - kz;
          if (o < 0 || o >= ZB || (kz < 2 && o < CH) || (kz == 2 && chain)) continue;
#pragma unroll
          for (int p = 0; p < 2; ++p) acc[p][o] = product(which, now, p, kz, acc[p][o]);
        }
      if constexpr (CH > 0) __builtin_amdgcn_sched_barrier(0);
    };

    for (int chunk = cbeg; chunk < cend; ++chunk) {
      // This thread's halo lines have landed: vector-memory operations complete in order, and the
      // twelve loads of U follow the halo's, as may stores of the last box.  U is waited for behind
      // the barrier (320 -> 320 on 5 x 6 x 7 64.2 to 61.3 us, 128 -> 128 on 32^3 x 8 430 to 424), but
      // before the next halo's loads, which the compiler would wait for with it.
      asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
      normalise(cur, yx, quads, chunk, buf);
      lds_barrier();  // every thread's lines; the other buffer is free
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
      const bool last = chunk + 1 == cend;
      // the next chunk's halo; after the box's last chunk the next box's first, if there is one
      if (last && more) {
        int tid_n = tid;
        asm volatile("" : "+v"(tid_n));  // computed here, not hoisted and held
        box_lines(tid_n, nxt, yx, quads);
      }
      const Source src = source(last ? nxt : cur, last ? cbeg : chunk + 1);
      if (!last || more) fetch(src, yx, quads, buf ^ 1);
      const uint4* un = uaddr(lane, last ? nxt.nt : cur.nt, last ? cbeg : chunk + 1);
      plane(std::integral_constant<int, 0>{});
      plane(std::integral_constant<int, 1>{});
      if constexpr (ZB == 4) {
        plane(std::integral_constant<int, 2>{});
        plane(std::integral_constant<int, 3>{});
      }
      if constexpr (CH < ZB) load_u(un, 0);
      plane(std::integral_constant<int, ZB>{});
      if constexpr (CH == ZB) load_u(un, 0);
      load_u(un, 1);
      plane(std::integral_constant<int, ZB + 1>{});
      load_u(un, 2);
      const unsigned flip = buf ? 0u - (unsigned)(G::buf * 16) : (unsigned)(G::buf * 16);
#pragma unroll
      for (int i = 0; i < 6; ++i) ad[i] += flip;
      buf ^= 1;
    }

    // ---- epilogue, in the raw buffer of the box's last chunk
    lds_barrier();  // every wave is past its last read of it
    f4* red = s_raw + (buf ^ 1) * G::buf + kPartSlots;
    if (nxt.b != cur.b) load_prm(tid, nxt.b);  // visible after the barriers below
    const int quad = tid & 7, rho = (tid >> 3) & 31, ox = tid >> 8;
    const f4 bias = *reinterpret_cast<const f4*>(s_bias + 4 * quad);
    f4 yo[ZB][2];  // [z][oy]
#pragma unroll
    for (int z = 0; z < ZB; ++z) {
      // partials [wave][ox][tile][column]; tile row r sits at rho(r) = (r / 8) * 8 + (r % 4) * 2 +
      // (r / 4) % 2, so that a wave's two row groups (r and r + 4) write different banks
      float* part = reinterpret_cast<float*>(s_raw + (more || (z & 1) == 0 ? buf ^ 1 : buf) * G::buf);
      float* pw = part + wave * 2048 + (lane >> 5) * 32 + (lane & 31);
      auto write_parts = [&](auto hc) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float ma = acc[0][z][r], mb = acc[1][z][r];
          float x0, x1;
          if constexpr (decltype(hc)::value == 0) {
            x0 = ma + mb;  // xx 0, 1
            x1 = mb;
          } else {
            x0 = mb;       // xx 2 and minus xx 3
            x1 = ma - mb;
          }
          const int at = ((r >> 2) * 8 + (r & 3) * 2) * 32;
          pw[at] = x0;
          pw[1024 + at] = x1;
        }
      };
      if (h == 0)
        write_parts(std::integral_constant<int, 0>{});
      else
        write_parts(std::integral_constant<int, 1>{});
      lds_barrier();
      if (z == 0 && nxt.nt != cur.nt && tid < 32)
        s_bias[tid] = a.bias ? a.bias[nxt.nt * 32 + tid] : 0.f;  // every thread has read its own
      const float* pr = part + ox * 1024 + rho * 32 + 4 * quad;
      f4 m[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        m[i] = *reinterpret_cast<const f4*>(pr + (2 * i) * 2048) +
               *reinterpret_cast<const f4*>(pr + (2 * i + 1) * 2048);
      yo[z][0] = ((m[0] + m[1]) + m[2]) * a.out_scale + bias;
      yo[z][1] = ((m[1] - m[2]) - m[3]) * a.out_scale + bias;
      if (more) lds_barrier();  // (the last box's planes take the two buffers in turn)
    }
    const int row = 8 * (rho >> 3) + 4 * (rho & 1) + ((rho >> 1) & 3);
    const int yy = cur.byi * G::by + 2 * (S == kWide ? row >> 3 : S == kTall ? row >> 2 : (row >> 2) & 3);
    const int xx = cur.bxi * G::bx + 2 * (S == kWide ? row & 7 : row & 3) + ox;
    const int z0 = cur.bzi * G::bz + (S == kCube ? (row >> 4) * ZB : 0);
    const bool xin = xx < a.W;
    auto valid = [&](int z, int oy) { return xin && yy + oy < a.H && z0 + z < a.D; };
    if (a.stats) {
      const int nz = min(G::bz, a.D - cur.bzi * G::bz), ny = min(G::by, a.H - cur.byi * G::by);
      const int nx = min(G::bx, a.W - cur.bxi * G::bx);
      const float cnt = (float)(nz * ny * nx);
      f4 sm = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int z = 0; z < ZB; ++z)
#pragma unroll
        for (int oy = 0; oy < 2; ++oy)
          if (valid(z, oy)) sm += yo[z][oy];
      sm = sum_stride8(sm);
      if (lane < 8) red[wave * 8 + quad] = sm;
      lds_barrier();
      f4 mean = red[quad];
#pragma unroll
      for (int w = 1; w < 8; ++w) mean += red[w * 8 + quad];
      mean = mean / cnt;
      f4 m2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int z = 0; z < ZB; ++z)
#pragma unroll
        for (int oy = 0; oy < 2; ++oy)
          if (valid(z, oy)) {
            const f4 d = yo[z][oy] - mean;
#pragma unroll
            for (int e = 0; e < 4; ++e) m2[e] = fmaf(d[e], d[e], m2[e]);
          }
      m2 = sum_stride8(m2);
      if (lane < 8) red[64 + wave * 8 + quad] = m2;
      lds_barrier();
      if (tid < 8) {
        f4 t = red[64 + quad];
#pragma unroll
        for (int w = 1; w < 8; ++w) t += red[64 + w * 8 + quad];
        const int tiles = a.nbz * a.nby * a.nbx;
        const int tile = (cur.bzi * a.nby + cur.byi) * a.nbx + cur.bxi;
        float4* out = a.stats + ((int64_t)cur.b * tiles + tile) * a.cout + cur.nt * 32 + 4 * quad;
#pragma unroll
        for (int e = 0; e < 4; ++e) out[e] = make_float4(mean[e], t[e], cnt, 0.f);
      }
    }
    float* out = a.y + blockIdx.y * a.split_stride + (((int64_t)cur.b * a.D + z0) * plane_vox + (int64_t)yy * a.W + xx) * a.cout +
                 cur.nt * 32 + 4 * quad;
#pragma unroll
    for (int z = 0; z < ZB; ++z)
#pragma unroll
      for (int oy = 0; oy < 2; ++oy)
        if (valid(z, oy))
          *reinterpret_cast<f4*>(out + (z * plane_vox + (int64_t)oy * a.W) * a.cout) = yo[z][oy];
    if (!more) break;
    v = vnext;
  }
}

// U[cout][cin][kz][xi] = sum_{b,e} G[xy][b] G[xx][e] w[cout][kz][b][e][cin] in float64, times
// `scale`, rounded to float32, split into fp16 halves.  Word layout:
// packed[((((nt * chunks + chunk) * 16 + pos) * 3 + kz) * 2 + part) * 64 + lane], pos = 2 * wave + i
// in the kernel's order (xy = wave / 2; xx = 0, 1 for an even wave, 3, 2 for an odd one), lane =
// column (cout = nt * 32 + lane % 32) and k slot (cin = chunk channel 8 * (lane / 32) + q).
__global__ void pack_wino_weight_kernel(const float* __restrict__ w, uint4* __restrict__ out,
                                        int cout, int c1, int c2, int chunks0, int chunks,
                                        int ntn, float scale) {
  const double G[4][3] = {{1.0, 0.0, 0.0}, {0.5, 0.5, 0.5}, {0.5, -0.5, 0.5}, {0.0, 0.0, 1.0}};
  const int cin_total = c1 + c2;
  const int64_t total = (int64_t)ntn * chunks * kPositions * 3 * 64;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(i & 63);
    int64_t rest = i >> 6;
    const int kz = (int)(rest % 3);
    rest /= 3;
    const int pos = (int)(rest % kPositions);
    rest /= kPositions;
    const int chunk = (int)(rest % chunks);
    const int nt = (int)(rest / chunks);
    const int xy = pos >> 2, odd = (pos >> 1) & 1, second = pos & 1;
    const int xx = odd ? 3 - second : second;
    const int n = nt * 32 + (lane & 31);
    h8 hv, lv;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int k = 8 * (lane >> 5) + q;
      int wc = -1;
      if (chunk < chunks0) {
        const int cc = chunk * kWChunk + k;
        if (cc < c1) wc = cc;
      } else {
        const int cc = (chunk - chunks0) * kWChunk + k;
        if (cc < c2) wc = c1 + cc;
      }
      float v = 0.f;
      if (n < cout && wc >= 0) {
        double u = 0.0;
        for (int ay = 0; ay < 3; ++ay)
          for (int ax = 0; ax < 3; ++ax) {
            const double gw = G[xy][ay] * G[xx][ax];
            if (gw != 0.0)
              u += gw * (double)w[((((int64_t)n * 3 + kz) * 3 + ay) * 3 + ax) * cin_total + wc];
          }
        v = (float)(u * (double)scale);
      }
      const _Float16 hh = (_Float16)v;
      hv[q] = hh;
      lv[q] = (_Float16)(v - (float)hh);
    }
    const int64_t word = (i >> 6) * kTapWords + lane;
    out[word] = *reinterpret_cast<const uint4*>(&hv);
    out[word + 64] = *reinterpret_cast<const uint4*>(&lv);
  }
}

// The box of a layer: its z planes and shape, and the boxes per axis of an item.
struct WinoPlan {
  int zb;
  WinoShape shape;
  int nbz, nby, nbx;
};

// Every box: planes of a slab, shape, voxels a side and cost.
template <class F>
void wino_boxes(F&& f) {
  f(4, kWide, 4, 8, 16, 10);
  f(4, kTall, 4, 16, 8, 10);
  f(2, kWide, 2, 8, 16, 6);
  f(2, kTall, 2, 16, 8, 6);
  f(2, kCube, 4, 8, 8, 6);
}

// The shape that needs the least time by rounds of boxes over the CUs: a box of four planes
// takes 1 of it, one of two planes 0.6 (320 -> 320: 4.8 and 2.9 us a 16-channel chunk), so the
// small boxes win where they fill CUs that would stand idle: 320 -> 320 on 8^3 x 8 95.6 us in
// boxes of 4 x 8 x 16 (half of each outside the volume), 63.9 us in boxes of 4 x 8 x 8 (the three-axis
// form: 67 to 69).
WinoPlan wino_plan(const ConvGeom& g, int cout) {
  const int64_t cus = compute_units();
  const int64_t columns = (int64_t)g.batch * ceil_div(cout, 32);
  WinoPlan best{};
  int64_t best_cost = -1;
  auto consider = [&](int zb, WinoShape shape, int bz, int by, int bx, int64_t cost) {
    const int64_t nbz = ceil_div(g.out[0], bz), nby = ceil_div(g.out[1], by), nbx = ceil_div(g.out[2], bx);
    const int64_t total = ceil_div(columns * nbz * nby * nbx, cus) * cost;
    if (best_cost >= 0 && total >= best_cost) return;
    best_cost = total;
    best = WinoPlan{zb, shape, (int)nbz, (int)nby, (int)nbx};
  };
  wino_boxes(consider);
  return best;
}

}  // namespace

// Compute units of the current device, rounded down to a multiple of the 8 XCDs (the
// persistent kernel's grid: one workgroup a CU).
int compute_units() {
  static int cached[64] = {0};
  int dev = 0;
  hip_check(hipGetDevice(&dev), "hipGetDevice");
  if (dev < 0 || dev >= 64) dev = 0;
  if (cached[dev] == 0) {
    int n = 0;
    hip_check(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev),
              "hipDeviceGetAttribute");
    cached[dev] = n >= 8 ? n / 8 * 8 : 8;
  }
  return cached[dev];
}

// Layers outside this set take the direct split kernel (the route is chosen with it).
bool conv_wino_supported(const ConvGeom& g, int c1, int c2, int cout) {
  for (int i = 0; i < 3; ++i)
    if (g.k[i] != 3 || g.s[i] != 1) return false;
  return cout % 32 == 0 && c1 % kWChunk == 0 && c2 % kWChunk == 0 && c1 > 0 && c2 >= 0 &&
         c1 + c2 <= kMaxChannels;
}

// Layers with less than half a box a CU stand on a chain of chunks (2.9 us each) in a few
// workgroups: their chunks are split over the idle CUs, at least two a workgroup, and summed
// behind.
int conv_wino_splits(const ConvGeom& g, int c1, int c2, int cout) {
  const WinoPlan p = wino_plan(g, cout);
  const int64_t boxes = (int64_t)g.batch * p.nbz * p.nby * p.nbx * (cout / 32);
  const int chunks = (c1 + c2) / kWChunk;
  const int64_t spatial = (int64_t)g.out[0] * g.out[1] * g.out[2];
  const int64_t most = std::min<int64_t>(compute_units() / boxes, chunks / 2);
  if (most < 2 || !split_sum_supported(spatial, cout)) return 1;
  // where the sum is a launch more (6 us) it takes eight chunks to gain by it
  if (split_sum_parts(spatial) > 1 && chunks < 8) return 1;
  return (int)ceil_div(chunks, ceil_div(chunks, most));
}

int conv_wino_stats_tiles(const ConvGeom& g, int cout) {
  const WinoPlan p = wino_plan(g, cout);
  return p.nbz * p.nby * p.nbx;
}

int conv_wino_stats_room(const ConvGeom& g) {
  int64_t room = 0;
  wino_boxes([&](int, WinoShape, int bz, int by, int bx, int64_t) {
    room = std::max(room, ceil_div(g.out[0], bz) * ceil_div(g.out[1], by) * ceil_div(g.out[2], bx));
  });
  return (int)room;
}

float wino_weight_scale(float max_abs) {
  // |U| <= (1.5)^2 max |w|: the scale keeps every split high half below 2^15, with the room of
  // a third factor 1.5 (the bound in float32, or in float64 where the float32 product would
  // overflow)
  require(std::isfinite(max_abs) && max_abs >= 0.f, "weight magnitude must be finite");
  const float bound = 3.375f * max_abs;
  return split_weight_scale(std::isfinite(bound) ? (double)bound : 3.375 * (double)max_abs);
}

int64_t conv_wino_packed_bytes(int cout, int c1, int c2) {
  const int64_t chunks = ceil_div(c1, kWChunk) + ceil_div(c2, kWChunk);
  return ceil_div(cout, 32) * chunks * kPositions * 3 * kTapWords * 16;
}

void conv_wino_pack_weight(const float* d_w, int cout, int c1, int c2, float scale,
                           void* d_packed, hipStream_t st) {
  require(d_w && d_packed, "Winograd packing pointers must not be null");
  require(cout >= 1 && c1 >= 1 && c2 >= 0, "invalid Winograd convolution channel counts");
  require(scale > 0.f && std::isfinite(scale), "weight scale must be positive");
  const int chunks0 = (int)ceil_div(c1, kWChunk);
  const int chunks = chunks0 + (int)ceil_div(c2, kWChunk);
  const int ntn = (int)ceil_div(cout, 32);
  const int64_t total = (int64_t)ntn * chunks * kPositions * 3 * 64;
  const int blocks = (int)std::min<int64_t>(ceil_div(total, 256), 65536);
  hipLaunchKernelGGL(pack_wino_weight_kernel, dim3(blocks), dim3(256), 0, st, d_w,
                     reinterpret_cast<uint4*>(d_packed), cout, c1, c2, chunks0, chunks, ntn,
                     scale);
  launch_check("conv3d_winograd_pack_weight");
}

void conv3d_wino(const float* x1, int c1, const float* x2, int c2, const void* packed,
                 float scale, const float* bias, float* y, const ConvGeom& g, int cout,
                 hipStream_t st, float4* stats, const PendingNorm& n1, const PendingNorm& n2,
                 int splits) {
  require(x1 && y && packed, "convolution pointers must not be null");
  require(c2 == 0 || x2, "invalid convolution inputs");
  require(splits == 1 || (!stats && !bias), "a split convolution is finished by its sum");
  require(conv_wino_supported(g, c1, c2, cout),
          "the Winograd convolution takes stride-1 3x3x3 layers with C_out % 32 == 0 and input "
          "channel counts that are multiples of 16, at most 1024 input channels in all");
  require(scale > 0.f && std::isfinite(scale), "weight scale must be positive");
  require(!(n1.params && n2.params) || n1.slope == n2.slope,
          "pending normalisations of one convolution must share the LeakyReLU slope");
  require(reinterpret_cast<uintptr_t>(y) % 16 == 0 && reinterpret_cast<uintptr_t>(x1) % 16 == 0 &&
              reinterpret_cast<uintptr_t>(x2) % 16 == 0,
          "Winograd convolution tensors must be 16-byte aligned");
  WinoArgs a{};
  a.x0 = x1;
  a.x1 = x2;
  a.c0 = c1;
  a.c1 = c2;
  a.chunks0 = c1 / kWChunk;
  a.chunks = a.chunks0 + c2 / kWChunk;
  a.u = reinterpret_cast<const uint4*>(packed);
  a.bias = bias;
  a.y = y;
  a.D = g.in[0];
  a.H = g.in[1];
  a.W = g.in[2];
  a.cout = cout;
  const WinoPlan p = wino_plan(g, cout);
  a.nbz = p.nbz;
  a.nby = p.nby;
  a.nbx = p.nbx;
  const int64_t nwg = (int64_t)g.batch * a.nbz * a.nby * a.nbx * (cout / 32);
  require(nwg < (1LL << 31), "convolution grid too large");
  a.nvirt = (int)nwg;
  a.nbox = a.nvirt / (cout / 32);
  a.rbox = reciprocal(a.nbox);
  a.rz = reciprocal(a.nbz);
  a.ry = reciprocal(a.nby);
  a.rx = reciprocal(a.nbx);
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
  const double flops = 2.0 * (c1 + c2) * cout * 27.0 * out_vox;
  const double bytes = 4.0 * ((double)g.batch * g.in[0] * g.in[1] * g.in[2] * (c1 + c2) +
                              out_vox * cout);
  ProfScope prof("conv3d_wino", flops, bytes, st);
  const dim3 grid((unsigned)std::min<int64_t>(compute_units(), ceil_div(nwg, 8) * 8),
                  (unsigned)ceil_div(a.chunks, a.cper)), block(kWThreads);
  auto launch = [&](auto chained) {
    constexpr int C = decltype(chained)::value;
    auto kernel = p.zb == 4 ? (p.shape == kWide ? wino_yx_kernel<4, kWide, C> : wino_yx_kernel<4, kTall, C>)
                  : p.shape == kWide ? wino_yx_kernel<2, kWide, C / 2>
                  : p.shape == kTall ? wino_yx_kernel<2, kTall, C / 2>
                                     : wino_yx_kernel<2, kCube, C / 2>;
    hipLaunchKernelGGL(kernel, grid, block, 0, st, a);
  };
  // The error must not exceed the three-axis form's: up to three chunks a workgroup it does not
  // with plain sums, up to five with half the planes' apart (see the head of the file).
  if (a.cper <= 3)
    launch(std::integral_constant<int, 0>{});
  else if (a.cper <= 5)
    launch(std::integral_constant<int, 2>{});
  else
    launch(std::integral_constant<int, 4>{});
  launch_check("conv3d_winograd");
}

}  // namespace nnx
