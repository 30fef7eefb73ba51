// Direct bf16 convolution of the stride-1, padding-1 3x3x3 layers on
// v_mfma_f32_32x32x16_bf16: operands rounded to bf16 (nearest even), one product a term,
// float32 accumulation.
//
// Workgroup: 8 waves (two a SIMD), an output box of 4 x 8 x 16 voxels and 32 NC output
// channels (NC = 2, or 1 where C_out is 32; of 96 or 160 channels the last group computes 32 for
// nothing, a quarter and a sixth of the products).  A wave owns one of the four
// 4 x 8 patches of the (y, x) plane as its MFMA rows, 32 channels as its columns, and all four
// z planes (NC = 2) or two of them (NC = 1) as separate accumulators, so the A operand of an
// input plane and a (ky, kx) tap, read from LDS once, serves every kz that reaches an output
// plane of the box: 6 reads for 12 products.  B operands come from L2 (the four waves of a
// column block read the same words) in a ring of three (ky, kx) steps.
//
// Per chunk of 16 input channels the (ZB + 2) x 10 x 18 halo is loaded to registers during the
// previous chunk, a line a step between the B operands, so that a B operand's wait never
// stands behind a load younger than three steps (vector-memory loads return in order); at the
// chunk's end each thread applies the pending InstanceNorm (+ LeakyReLU) to its lines, rounds
// them and writes them to the other of two LDS buffers.  Voxel rows are laid out so that the 32
// voxels of a patch read 32 different 16-byte bank groups.  One barrier a chunk.  Persistent:
// one workgroup a CU loops over boxes (XCDs take contiguous ranges, column group slowest), a
// box's last chunk loading the next box's first halo and B operands.  Each wave finishes its
// own outputs: scale, bias, InstanceNorm partials, and 16-byte channel runs through a
// wave-private LDS tile.
//
// Bound by latency and issue (matrix cores about 40 % busy).  Against the weight-staged 16x16x32
// kernel: 64 -> 64 on 64 x 80 x 80 x 4 0.753 -> 0.443 ms (818 TFLOP/s), 256 -> 256 on 16^3 x 8
// 0.246 -> 0.109 ms (1065), 320 -> 320 on 8^3 0.140 -> 0.107 ms.
#include <cmath>
#include <type_traits>

#include "nnx_internal.h"

namespace nnx {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf4 __attribute__((ext_vector_type(4)));

constexpr int kBThreads = 512;
constexpr int kBChunk = 16;          // input channels per chunk (one MFMA K)
constexpr int kBMaxChannels = 1024;  // c1 + c2 (pending-norm parameters in LDS)
constexpr int kZB = 4, kBY = 8, kBX = 16;
constexpr int kHZ = kZB + 2, kHY = kBY + 2, kHX = kBX + 2;
constexpr int kRawPlane = 768;   // 16-byte lines of a halo plane: 1.5 rounds of the workgroup
constexpr int kLines = kHZ / 2 * 3;  // lines (rounds) per thread
constexpr int kPlaneSlots = 400;     // 16-byte slots of a bf16 halo plane
constexpr int kBufSlots = kHZ * kPlaneSlots;
constexpr int kSteps = 9;            // (ky, kx)
constexpr int kRing = 3;
constexpr int kStageFloats = 32 * 32;  // a wave's output tile (one plane)
static_assert(kHY * kHX * 4 <= kRawPlane, "a halo plane fits its rounds");
static_assert(kLines == kSteps, "a halo line a step");
static_assert(kSteps % kRing == 0, "ring slots are the same in every chunk");
static_assert(8 * kStageFloats + 2 * 8 * 32 <= kBufSlots * 4, "epilogue fits one buffer");

// slot of halo row hy: four consecutive rows of 8 voxels (2 slots each) fall on different slots
// modulo 32
__device__ __forceinline__ int row_slot(int hy) {
  const int t = hy & 3;
  return (hy >> 2) * 160 + t * 37 + (t >= 2 ? 6 : 0);
}

struct Bf16Args {
  const float* x0;
  const float* x1;
  int c0, c1, chunks0, chunks;
  const uint4* u;
  const float* bias;
  float* y;
  int D, H, W;
  int cout, nblk;  // 32-column blocks
  int nbz, nby, nbx;
  int nbox, nvirt;
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

struct Bf16Box {
  int ng, b, bzi, byi, bxi;
};

__device__ __forceinline__ Bf16Box bf16_box(const Bf16Args& a, int v) {
  Bf16Box r;
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

template <int NC>
__global__ __launch_bounds__(kBThreads, 1) void conv_bf16_kernel(Bf16Args a) {
  constexpr int PZ = NC == 2 ? 4 : 2;  // output planes of a wave
  __shared__ __align__(16) uint4 s_a[2 * kBufSlots];
  __shared__ __align__(16) float s_prm[3 * kBMaxChannels];
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int xcd = blockIdx.x & 7, stride = gridDim.x >> 3;
  const int vq = a.nvirt >> 3, vr = a.nvirt & 7;
  const int vbeg = xcd < vr ? xcd * (vq + 1) : vr * (vq + 1) + (xcd - vr) * vq;
  const int vend = vbeg + vq + (xcd < vr ? 1 : 0);
  int v = vbeg + (int)(blockIdx.x >> 3);
  if (v >= vend) return;  // uniform over the workgroup, before any barrier
  __builtin_assume(a.chunks > 0);
  const int64_t plane_vox = (int64_t)a.H * a.W;
  const int patch = wave & 3, py = patch >> 1, px = patch & 1, upper = wave >> 2;
  const int pz0 = NC == 2 ? 0 : 2 * upper;  // the wave's first output plane

  auto round_plane = [&](int r) {
    const int k = r / 3, j = r % 3;
    return 2 * k + ((j == 2 || (j == 1 && wave >= 4)) ? 1 : 0);
  };
  // in-plane voxel of this thread's three line patterns (-1 outside the volume)
  auto box_lines = [&](int tid, const Bf16Box& bx, int (&yx)[3]) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int s = j == 0 ? tid : j == 1 ? (tid < 256 ? 512 + tid : tid - 256) : 256 + tid;
      const int vox = s >> 2, hy = vox / kHX, hx = vox - hy * kHX;
      const int yy = bx.byi * kBY - 1 + hy, xx = bx.bxi * kBX - 1 + hx;
      yx[j] = hy < kHY && (unsigned)yy < (unsigned)a.H && (unsigned)xx < (unsigned)a.W
                  ? yy * a.W + xx : -1;
    }
  };
  struct Source {
    const float* base;  // channel chunk of the item
    int64_t plane;      // elements
    int C, z0;
  };
  auto source = [&](const Bf16Box& bx, int chunk) __attribute__((always_inline)) {
    const bool first = chunk < a.chunks0;
    Source r;
    r.C = first ? a.c0 : a.c1;
    r.plane = plane_vox * r.C;
    r.z0 = bx.bzi * kZB - 1;
    r.base = (first ? a.x0 : a.x1) + (int64_t)bx.b * a.D * r.plane +
             (first ? chunk : chunk - a.chunks0) * kBChunk;
    return r;
  };
  // line r of the halo; outside the volume the item's first line, zeroed when it is written
  auto load_line = [&](const Source& src, const int (&yx)[3], int r) __attribute__((always_inline)) {
    const int j = r % 3;
    const int z = src.z0 + round_plane(r);
    const float* p = src.base + min(max(z, 0), a.D - 1) * src.plane +
                     (int64_t)max(yx[j], 0) * src.C + (threadIdx.x & 3) * 4;
    return *reinterpret_cast<const f4*>(p);
  };
  auto load_prm = [&](int tid, int b) __attribute__((always_inline)) {
    if (!a.nrm0 && !a.nrm1) return;
    for (int c = tid; c < a.c0 + a.c1; c += kBThreads) {
      const float4* pp = c < a.c0 ? a.nrm0 : a.nrm1;
      const int C = c < a.c0 ? a.c0 : a.c1;
      const int cc = c < a.c0 ? c : c - a.c0;
      float4 pv = make_float4(0.f, 1.f, 0.f, 0.f);
      if (pp) pv = pp[(int64_t)b * C + cc];
      s_prm[c] = pv.x;
      s_prm[kBMaxChannels + c] = pv.y;
      s_prm[2 * kBMaxChannels + c] = pv.z;
    }
  };
  // The pending norm (the apply pass's operations), rounding, and the write to buffer `buf`.
  auto convert = [&](const f4 (&hl)[kLines], const int (&yx)[3], int z0, int chunk, int buf)
      __attribute__((always_inline)) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // the slots are computed here, not held through the chunk
    const bool first = chunk < a.chunks0;
    const bool norm = (first ? a.nrm0 : a.nrm1) != nullptr;
    const float s = (first ? a.act0 : a.act1) != 0 ? a.slope : 1.f;
    f4 mean = {}, scale = {}, beta = {};
    if (norm) {
      const float* prm = s_prm + chunk * kBChunk + (tid & 3) * 4;
      mean = *reinterpret_cast<const f4*>(prm);
      scale = *reinterpret_cast<const f4*>(prm + kBMaxChannels);
      beta = *reinterpret_cast<const f4*>(prm + 2 * kBMaxChannels);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int sl = j == 0 ? tid : j == 1 ? (tid < 256 ? 512 + tid : tid - 256) : 256 + tid;
      const int vox = sl >> 2, hy = vox / kHX, hx = vox - hy * kHX;
      if (hy >= kHY) continue;  // a padding line
      uint2* dst = reinterpret_cast<uint2*>(s_a + buf * kBufSlots + row_slot(hy) + hx * 2) + (tid & 3);
#pragma unroll
      for (int k = 0; k < kHZ / 2; ++k) {
        const int r = 3 * k + j, p = round_plane(r);
        const bool inside = yx[j] >= 0 && (unsigned)(z0 + p) < (unsigned)a.D;
        bf4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float x = hl[r][e];
          if (norm) {
            const float t = fmaf(x - mean[e], scale[e], beta[e]);
            x = fmaxf(s * t, t);
          }
          o[e] = (__bf16)(inside ? x : 0.f);
        }
        dst[p * kPlaneSlots * 2] = __builtin_bit_cast(uint2, o);
      }
    }
  };
  // packed words of this wave's column block: [block][chunk][tap] x 64 lanes, 2 KB apart
  auto uaddr = [&](int lane, int ng, int chunk) {
    const int blk = min(NC == 2 ? ng * 2 + upper : ng, a.nblk - 1);
    return a.u + (((int64_t)blk * a.chunks + chunk) * 27 * 2 + 1) * 64 + lane;
  };
  uint4 ub[kRing][3];
  auto load_u = [&](const uint4* base, int step) __attribute__((always_inline)) {
#pragma unroll
    for (int kz = 0; kz < 3; ++kz) ub[step % kRing][kz] = base[(kz * kSteps + step) * 128];
  };

  int yx[3], buf = 0;
  {
    const int tid = threadIdx.x;
    const Bf16Box first = bf16_box(a, v);
    box_lines(tid, first, yx);
    const Source src = source(first, 0);
    f4 hl[kLines];
#pragma unroll
    for (int r = 0; r < kLines; ++r) hl[r] = load_line(src, yx, r);
    const uint4* up = uaddr(tid & 63, first.ng, 0);
#pragma unroll
    for (int s = 0; s < kRing; ++s) load_u(up, s);
    load_prm(tid, first.b);
    lds_barrier();  // the parameters
    convert(hl, yx, src.z0, 0, 0);
    lds_barrier();
  }

  for (;;) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const Bf16Box cur = bf16_box(a, v);
    const int vnext = v + stride;
    const bool more = vnext < vend;
    const Bf16Box nxt = bf16_box(a, more ? vnext : v);
    const int t = lane & 31, g8 = lane >> 5;
    const int blk = NC == 2 ? cur.ng * 2 + upper : cur.ng;
    const bool live = blk < a.nblk;
    const float bias = a.bias && live ? a.bias[blk * 32 + t] : 0.f;
    int row[3];  // slots of the lane's voxel at (ky, kx = 0) in the wave's first input plane
#pragma unroll
    for (int ky = 0; ky < 3; ++ky)
      row[ky] = pz0 * kPlaneSlots + row_slot(py * 4 + (t >> 3) + ky) + (px * 8 + (t & 7)) * 2 + g8;

    f16v acc[PZ];
#pragma unroll
    for (int z = 0; z < PZ; ++z)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[z][r] = 0.f;

    for (int chunk = 0; chunk < a.chunks; ++chunk) {
      const bool last = chunk + 1 == a.chunks;
      const bool item = last && nxt.b != cur.b;  // the next halo takes another item's parameters
      if (last) {
        int tid_n = tid;
        asm volatile("" : "+v"(tid_n));
        box_lines(tid_n, nxt, yx);
        if (item) load_prm(tid_n, nxt.b);
      }
      const int nchunk = last ? 0 : chunk + 1;
      const Source src = source(last ? nxt : cur, nchunk);
      const uint4* uc = uaddr(lane, cur.ng, chunk);
      const uint4* un = uaddr(lane, last ? nxt.ng : cur.ng, nchunk);
      const uint4* tile = s_a + buf * kBufSlots;
      f4 hl[kLines];
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        uint4 av[PZ + 2];
#pragma unroll
        for (int p = 0; p < PZ + 2; ++p) av[p] = tile[row[s / 3] + p * kPlaneSlots + (s % 3) * 2];
        hl[s] = load_line(src, yx, s);
#pragma unroll
        for (int kz = 0; kz < 3; ++kz)
#pragma unroll
          for (int z = 0; z < PZ; ++z)
            acc[z] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                __builtin_bit_cast(bf8, av[z + kz]), __builtin_bit_cast(bf8, ub[s % kRing][kz]),
                acc[z], 0, 0, 0);
        if (s + kRing < kSteps) load_u(uc, s + kRing);
        else load_u(un, s + kRing - kSteps);
      }
      if (item) lds_barrier();  // its parameters
      convert(hl, yx, src.z0, nchunk, buf ^ 1);
      lds_barrier();  // the next chunk's tile; this one is free
      buf ^= 1;
    }

    // ---- epilogue, in the buffer of the box's last chunk
    float* stage = reinterpret_cast<float*>(s_a + (buf ^ 1) * kBufSlots);
    float* red = stage + 8 * kStageFloats;
    stage += wave * kStageFloats;
    const int z0 = cur.bzi * kZB + pz0, y0 = cur.byi * kBY + py * 4, x0 = cur.bxi * kBX + px * 8;
#pragma unroll
    for (int z = 0; z < PZ; ++z)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[z][r] = acc[z][r] * a.out_scale + bias;
    if (a.stats) {
      // accumulator r of a lane: patch voxel (r / 4, 4 g8 + r % 4) of its column
      auto valid = [&](int z, int r) {
        return z0 + z < a.D && y0 + (r >> 2) < a.H && x0 + 4 * g8 + (r & 3) < a.W;
      };
      const int nz = min(kZB, a.D - cur.bzi * kZB), ny = min(kBY, a.H - cur.byi * kBY);
      const int nx = min(kBX, a.W - cur.bxi * kBX);
      const float cnt = (float)(nz * ny * nx);
      // the waves of this column block: four (NC = 2) or eight
      const int w0 = NC == 2 ? upper * 4 : 0;
      constexpr int kW = NC == 2 ? 4 : 8;
      float sm = 0.f;
#pragma unroll
      for (int z = 0; z < PZ; ++z)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (valid(z, r)) sm += acc[z][r];
      sm = add_halves(sm);
      if (lane < 32) red[wave * 32 + t] = sm;
      lds_barrier();
      float tot = 0.f;
#pragma unroll
      for (int w = 0; w < kW; ++w) tot += red[(w0 + w) * 32 + t];
      const float mean = tot / cnt;
      float m2 = 0.f;
#pragma unroll
      for (int z = 0; z < PZ; ++z)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (valid(z, r)) {
            const float d = acc[z][r] - mean;
            m2 = fmaf(d, d, m2);
          }
      m2 = add_halves(m2);
      if (lane < 32) red[256 + wave * 32 + t] = m2;
      lds_barrier();
      if (wave == w0 && lane < 32 && live) {
        float tm = 0.f;
#pragma unroll
        for (int w = 0; w < kW; ++w) tm += red[256 + (w0 + w) * 32 + t];
        const int tiles = a.nbz * a.nby * a.nbx;
        const int tile = (cur.bzi * a.nby + cur.byi) * a.nbx + cur.bxi;
        a.stats[((int64_t)cur.b * tiles + tile) * a.cout + blk * 32 + t] =
            make_float4(mean, tm, cnt, 0.f);
      }
    }
    // 16-byte channel runs: voxel i of the patch at row rho(i) = (i / 8) * 8 + (i % 4) * 2 + (i / 4) % 2
    // of the tile, so that a lane's voxels and those 4 further write different banks
    const int quad = lane & 7;
#pragma unroll
    for (int z = 0; z < PZ; ++z) {
#pragma unroll
      for (int r = 0; r < 16; ++r) stage[((r >> 2) * 8 + (r & 3) * 2 + g8) * 32 + t] = acc[z][r];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int rho = i * 8 + (lane >> 3);
        const int yy = y0 + i, xx = x0 + 4 * (rho & 1) + ((rho >> 1) & 3);
        const f4 val = *reinterpret_cast<const f4*>(stage + rho * 32 + quad * 4);
        if (live && z0 + z < a.D && yy < a.H && xx < a.W)
          *reinterpret_cast<f4*>(a.y + ((((int64_t)cur.b * a.D + z0 + z) * a.H + yy) * a.W + xx) * a.cout +
                                 blk * 32 + quad * 4) = val;
      }
    }
    if (!more) break;
    lds_barrier();  // every wave's tile is read: the next chunk's halo may take the buffer
    v = vnext;
  }
}

// words[(2 j + 1) * 64 + lane], j = (block * chunks + chunk) * 27 + tap: bf16(scale * W[n][tap][c]),
// n = block * 32 + lane % 32, c = channel 8 * (lane / 32) + q of the chunk
__global__ void pack_bf16_weight_kernel(const float* __restrict__ w, uint4* __restrict__ out,
                                        int chunks, int cin, float scale, int64_t total) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int lane = (int)(i & 63);
    const int64_t j = i >> 6;
    const int tap = (int)(j % 27);
    const int chunk = (int)(j / 27 % chunks);
    const int64_t n = j / 27 / chunks * 32 + (lane & 31);
    bf8 o;
#pragma unroll
    for (int q = 0; q < 8; ++q)
      o[q] = (__bf16)(w[(n * 27 + tap) * cin + chunk * kBChunk + 8 * (lane >> 5) + q] * scale);
    out[(2 * j + 1) * 64 + lane] = __builtin_bit_cast(uint4, o);
  }
}

}  // namespace

bool conv_bf16_direct_packed(const int* ksize, int c1, int c2, int cout) {
  return ksize[0] == 3 && ksize[1] == 3 && ksize[2] == 3 && c1 > 0 && c1 % kBChunk == 0 &&
         c2 % kBChunk == 0 && c1 + c2 <= kBMaxChannels && cout % 32 == 0;
}

int conv_bf16_direct_stats_tiles(const ConvGeom& g) {
  return (int)(ceil_div(g.out[0], kZB) * ceil_div(g.out[1], kBY) * ceil_div(g.out[2], kBX));
}

// With one or two chunks and less than a box a CU, the first halo's latency is most of a box, and
// the weight-staged kernel's smaller tiles are ahead (32 -> 192 on 6 x 9 x 8 x 8: 16.6 against
// 18.1 us); from there on this kernel is (20.1 us both on 32 -> 96, 12 x 30 x 40 x 2; 67 against
// 52 us on 128 -> 128, 32^3).  A full round of it, a box of 4 x 8 x 16 voxels and 64 channels a CU,
// takes about 2/3 of that kernel's, three a CU of 256 voxels, fitted, and 32 channels; narrow
// volumes, whose boxes here are mostly padding, need more rounds than that wins (us, here against
// there: 128 -> 128 on 70 x 2 x 70 x 4, three rounds against one, 136 and 75; 76 x 32 x 8 x 2, two
// against one, 97 and 71; 256 -> 320 on 16 x 32 x 20 x 2, two and two, 186 and 239; 128 -> 128 on
// 70 x 9 x 70 x 2, three and three, 151 and 201).
bool conv_bf16_direct_supported(const ConvGeom& g, int c1, int c2, int cout) {
  if (!conv_bf16_direct_packed(g.k, c1, c2, cout) || g.s[0] != 1 || g.s[1] != 1 || g.s[2] != 1)
    return false;
  const int64_t boxes = (int64_t)g.batch * conv_bf16_direct_stats_tiles(g) *
                        ceil_div(cout / 32, cout == 32 ? 1 : 2);
  if (c1 + c2 <= 2 * kBChunk && boxes < compute_units()) return false;
  const int64_t cus = compute_units();
  return 2 * ceil_div(boxes, cus) <= 3 * ceil_div(conv_x3_boxes(g) * (cout / 32), 3 * cus);
}

void conv_bf16_direct_pack(const float* d_w, int cout, int c1, int c2, float scale, void* d_packed,
                           hipStream_t st) {
  const int chunks = (c1 + c2) / kBChunk;
  const int64_t total = (int64_t)(cout / 32) * chunks * 27 * 64;
  hipLaunchKernelGGL(pack_bf16_weight_kernel,
                     dim3((unsigned)std::min<int64_t>(ceil_div(total, 256), 65536)), dim3(256), 0, st,
                     d_w, reinterpret_cast<uint4*>(d_packed), chunks, c1 + c2, scale, total);
  launch_check("conv3d_bf16_pack_weight");
}

void conv3d_bf16_direct(const float* x1, int c1, const float* x2, int c2, const void* packed,
                        float scale, const float* bias, float* y, const ConvGeom& g, int cout,
                        hipStream_t st, float4* stats, const PendingNorm& n1,
                        const PendingNorm& n2) {
  Bf16Args a{};
  a.x0 = x1;
  a.x1 = x2;
  a.c0 = c1;
  a.c1 = c2;
  a.chunks0 = c1 / kBChunk;
  a.chunks = a.chunks0 + c2 / kBChunk;
  a.u = reinterpret_cast<const uint4*>(packed);
  a.bias = bias;
  a.y = y;
  a.D = g.in[0];
  a.H = g.in[1];
  a.W = g.in[2];
  a.cout = cout;
  a.nblk = cout / 32;
  a.nbz = (int)ceil_div(g.out[0], kZB);
  a.nby = (int)ceil_div(g.out[1], kBY);
  a.nbx = (int)ceil_div(g.out[2], kBX);
  const int nc = cout == 32 ? 1 : 2;
  const int64_t nwg = (int64_t)g.batch * a.nbz * a.nby * a.nbx * ceil_div(a.nblk, nc);
  require(nwg < (1LL << 31), "convolution grid too large");
  a.nvirt = (int)nwg;
  a.nbox = a.nvirt / (int)ceil_div(a.nblk, nc);
  a.out_scale = 1.0f / scale;
  a.stats = stats;
  a.nrm0 = n1.params;
  a.nrm1 = n2.params;
  a.act0 = n1.act ? 1 : 0;
  a.act1 = n2.act ? 1 : 0;
  a.slope = n1.params ? n1.slope : n2.slope;
  const double out_vox = (double)g.batch * g.out[0] * g.out[1] * g.out[2];
  ProfScope prof("conv3d_x3s_bf16_m512n64", 2.0 * (c1 + c2) * cout * 27.0 * out_vox,
                 4.0 * ((double)g.batch * g.in[0] * g.in[1] * g.in[2] * (c1 + c2) + out_vox * cout),
                 st);
  const dim3 grid((unsigned)std::min<int64_t>(compute_units(), ceil_div(nwg, 8) * 8));
  if (nc == 2)
    hipLaunchKernelGGL(conv_bf16_kernel<2>, grid, dim3(kBThreads), 0, st, a);
  else
    hipLaunchKernelGGL(conv_bf16_kernel<1>, grid, dim3(kBThreads), 0, st, a);
  launch_check("conv3d_bf16");
}

}  // namespace nnx
