// Kernels of the learned coarse-grid correction: a small 3D convolutional
// network on node grids (no counterpart in topoptlab).  Activations are fp32,
// channel-major a[c][z][x][y]; convolution weights are fp16 w[cout][cin][27]
// (tap t = (dz+1)*9 + (dx+1)*3 + (dy+1)) with fp32 accumulation; the fp32
// master weights live with the optimiser.  Stride-2 convolutions map 2m+1
// nodes to m+1 (node-aligned, like the multigrid levels); upsampling is the
// trilinear node interpolation (the multigrid prolongation) and its
// transpose.  All reductions are fixed-order (no atomics).
#include "tl_internal.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace tl {
namespace {

constexpr int BS = 256;

__device__ inline int tap_dz(int t) { return t / 9 - 1; }
__device__ inline int tap_dx(int t) { return (t / 3) % 3 - 1; }
__device__ inline int tap_dy(int t) { return t % 3 - 1; }

// Forward convolution and its data gradient as an implicit product on the
// FP32 matrix cores (v_mfma_f32_16x16x4f32: fp32 inputs, fp32 sums):
//   forward  y[co][o] = relu?(b[co] + sum_t sum_ci w[co][ci][t] a[ci][stride*o + off_t])
//   BWD      ga[ci][n] (+)= sum_t sum_co w[co][ci][t] gy[co][o], stride*o + off_t = n
// rows = 16 channels of the result (blockIdx.y), columns = 16 consecutive nodes
// of the result grid, inner dimension = 4 source channels of one tap.  A lane
// loads one source value per product, 16 lanes a run of y.  A wave takes a node
// tile, or on small grids (SPLIT) the waves of a workgroup share one, taps in
// turn, and add their sums through LDS; the workgroup's weights are staged once
// in LDS (fp16, [t][k][16 rows]) for all its node tiles.
//
// The grids are small (4,225 nodes for a 48x24x24 design), so the split is
// over channels and taps as well as nodes.  One thread per node and 8 result
// channels, looping over all taps and source channels, left most of the chip
// idle: 186 us (forward) and 148 us (gradient) per layer on average at that
// size against 25 and 12 now (a design of 192x96x96: forward pass 2.5 -> 0.63
// ms, forward and backward 26.2 -> 12.3 ms).
//
// A tap that has no source node for a result node is a product with 0 there,
// which an infinite or NaN weight (an fp16 overflow) would turn into a NaN.
// The staging looks for such weights; a workgroup that holds one skips those
// terms on scalar FMAs instead, in the same order of sums.
typedef float nn_f4 __attribute__((ext_vector_type(4)));
// NG: channel groups of 4, at least kc / 4; a power of two, so that every load
// of a tap is issued before its first product.
constexpr int CT = 512, CW = CT / 64;  // threads and waves of a workgroup
template <bool BWD, bool SPLIT, int NG, int TB>
__global__ __launch_bounds__(CT) void conv_kernel(int kc, int mc, int rz, int rx, int ry, int sz,
                                                  int sx, int sy, int stride, int relu,
                                                  int accumulate, int ntiles,
                                                  const float* __restrict__ src,
                                                  const _Float16* __restrict__ w,
                                                  const float* __restrict__ bias,
                                                  float* __restrict__ out) {
  constexpr int TP = 4 * NG * 16 + 2;  // tap pitch: staging writes of 27 taps in 27 banks
  __shared__ _Float16 wl[27 * TP];     // [27][kp][16]
  constexpr int kp = 4 * NG;
  const int m0 = int(blockIdx.y) * 16;
  // weights in their memory order ([rows][k][t], BWD [k][rows][t]), a batch of
  // loads in flight
  constexpr int NW = 27 * kp * 16, NB = 9;
  uint32_t top = 0;  // largest exponent and fraction among the staged weights
  for (int i0 = threadIdx.x; i0 < NW; i0 += CT * NB) {
    _Float16 r[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int i = i0 + b * CT;
      const int k = BWD ? i / (27 * 16) : i / 27 % kp, m = BWD ? i / 27 % 16 : i / (27 * kp);
      const bool in = i < NW && k < kc && m0 + m < mc;
      const int64_t at = (BWD ? int64_t(k) * mc + m0 + m : int64_t(m0 + m) * kc + k) * 27 + i % 27;
      r[b] = w[in ? at : 0];
      r[b] = in ? r[b] : _Float16(0);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int i = i0 + b * CT;
      const int k = BWD ? i / (27 * 16) : i / 27 % kp, m = BWD ? i / 27 % 16 : i / (27 * kp);
      top = max(top, __builtin_bit_cast(uint16_t, r[b]) & 0x7fffu);
      if (i < NW) wl[i % 27 * TP + k * 16 + m] = r[b];
    }
  }
  const bool special = __syncthreads_or(top >= 0x7c00u);  // one is infinite or NaN
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, j = l & 15, g = l >> 4;
  const int64_t nres = int64_t(rz) * rx * ry, nsrc = int64_t(sz) * sx * sy;
  // Source node of the lane's result node for each offset of an axis (as an
  // offset in memory) and, in bits of `ok`, whether there is one: axis z 0..2, x
  // 3..5, y 6..8.  (Formed per tap, index arithmetic was most of a narrow layer:
  // 6 to 3 channels on 49x97x49 nodes 43.9 us, 35.8 now.)
  int64_t oz[3], ox[3], oy[3];
  uint32_t ok;
  auto node = [&](int64_t o) {
    o = o < nres ? o : nres - 1;
    int X, Y, Z;
    if (nres < (int64_t(1) << 31)) {  // 32-bit divisions
      const uint32_t u = uint32_t(o), line = u / uint32_t(ry);
      Y = int(u - line * uint32_t(ry));
      Z = int(line / uint32_t(rx));
      X = int(line - uint32_t(Z) * uint32_t(rx));
    } else {
      Y = int(o % ry); X = int((o / ry) % rx); Z = int(o / (int64_t(ry) * rx));
    }
    ok = 0;
    auto axis = [&](int a, int r, int n, int64_t step, int64_t (&off)[3]) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const int at = BWD ? r - (d - 1) : stride * r + d - 1;
        const int s = BWD && stride == 2 ? at >> 1 : at;
        const bool in = at >= 0 && s < n && !(BWD && stride == 2 && (at & 1));
        off[d] = s * step;
        ok |= uint32_t(in) << (3 * a + d);
      }
    };
    axis(0, Z, sz, int64_t(sx) * sy, oz);
    axis(1, X, sx, sy, ox);
    axis(2, Y, sy, 1, oy);
  };
  auto pick = [](const int64_t (&v)[3], int d) { return d == 0 ? v[0] : (d == 1 ? v[1] : v[2]); };
  // tap t's source node; false where there is none
  auto source = [&](int t, const float*& p) {
    const int a = t / 9, b = t / 3 % 3, c = t % 3;
    const uint32_t m = (1u << a) | (8u << b) | (64u << c);
    const bool in = (ok & m) == m;
    const int64_t off = pick(oz, a) + pick(ox, b) + pick(oy, c);
    p = src + (in ? off : 0);
    return in;
  };
  // source values of tap t for the lane's node (0 where the tap has none)
  auto load = [&](int t, float (&v)[NG]) {
    const float* p;
    const bool in = source(t, p);
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      const int c = 4 * q + g;
      v[q] = p[int64_t(c < kc ? c : 0) * nsrc];
      v[q] = in && c < kc ? v[q] : 0.f;
    }
  };
  auto product = [&](int t, const float (&v)[NG], nn_f4& acc) {
    const _Float16* wt = wl + t * TP + g * 16 + j;
#pragma unroll
    for (int q = 0; q < NG; ++q)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(float(wt[q * 64]), v[q], acc, 0, 0, 0);
  };
  // the same sums of the lane's four results without the terms that have no source
  auto skip_product = [&](int t, nn_f4& acc) {
    const float* p;
    if (!source(t, p)) return;
    const _Float16* wt = wl + t * TP + 4 * g;
    for (int c = 0; c < kc; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        acc[i] = fmaf(float(wt[c * 16 + i]), p[int64_t(c) * nsrc], acc[i]);
  };
  auto store = [&](int m, int64_t o, float v) {
    if (m >= mc || o >= nres) return;
    float* dst = out + int64_t(m) * nres + o;
    if constexpr (BWD) {
      *dst = accumulate ? *dst + v : v;
    } else {
      v += bias[m];
      *dst = relu ? fmaxf(v, 0.f) : v;
    }
  };
  if (special) {
    for (int tile = int(blockIdx.x) * CW + wave; tile < ntiles; tile += int(gridDim.x) * CW) {
      const int64_t o = int64_t(tile) * 16 + j;
      node(o);
      nn_f4 acc{0.f, 0.f, 0.f, 0.f};
      for (int t = 0; t < 27; ++t) skip_product(t, acc);
#pragma unroll
      for (int i = 0; i < 4; ++i) store(m0 + 4 * g + i, o, acc[i]);
    }
    return;
  }
  if constexpr (!SPLIT) {
    // a wave per node tile, all taps in order: the sum of every output keeps
    // the order of a loop over taps and source channels
    for (int tile = int(blockIdx.x) * CW + wave; tile < ntiles; tile += int(gridDim.x) * CW) {
      const int64_t o = int64_t(tile) * 16 + j;
      node(o);
      nn_f4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll NG <= 4 ? 27 / TB : 1
      for (int t = 0; t < 27; t += TB) {
        float v[TB][NG];
#pragma unroll
        for (int q = 0; q < TB; ++q) load(t + q, v[q]);
#pragma unroll
        for (int q = 0; q < TB; ++q) product(t + q, v[q], acc);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) store(m0 + 4 * g + i, o, acc[i]);
    }
  } else {
    // the waves share a node tile, taps in turn, sums added through LDS
    __shared__ float red[CW][16][16];
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
      node(int64_t(tile) * 16 + j);
      nn_f4 acc{0.f, 0.f, 0.f, 0.f};
      for (int t = wave; t < 27; t += CW) {
        float v[NG];
        load(t, v);
        product(t, v, acc);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave][4 * g + i][j] = acc[i];
      __syncthreads();
      const int m = threadIdx.x >> 4, n = threadIdx.x & 15;
      if (threadIdx.x < 256) {
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < CW; ++q) v += red[q][m][n];
        store(m0 + m, int64_t(tile) * 16 + n, v);
      }
      __syncthreads();
    }
  }
}

// One source channel on a large grid: a thread per node and 8 result channels,
// taps in order (a tap without a source node is skipped).  The matrix tile would
// have three of its four source channels empty and most of its 16 rows.
constexpr int NR = 8;
template <bool BWD>
__global__ __launch_bounds__(BS) void conv_one_kernel(int mc, int rz, int rx, int ry, int sz, int sx,
                                                      int sy, int stride, int relu, int accumulate,
                                                      const float* __restrict__ src,
                                                      const _Float16* __restrict__ w,
                                                      const float* __restrict__ bias,
                                                      float* __restrict__ out) {
  __shared__ float wl[27][NR];
  const int m0 = int(blockIdx.y) * NR;
  for (int i = threadIdx.x; i < 27 * NR; i += BS)
    wl[i % 27][i / 27] = m0 + i / 27 < mc ? float(w[int64_t(m0) * 27 + i]) : 0.f;
  __syncthreads();
  const int64_t nres = int64_t(rz) * rx * ry;
  const int64_t o = int64_t(blockIdx.x) * BS + threadIdx.x;
  if (o >= nres) return;
  const int Y = int(o % ry), X = int((o / ry) % rx), Z = int(o / (int64_t(ry) * rx));
  float acc[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) acc[k] = 0.f;
#pragma unroll
  for (int t = 0; t < 27; ++t) {
    int z, x, y;
    if constexpr (BWD) {
      const int pz = Z - tap_dz(t), px = X - tap_dx(t), py = Y - tap_dy(t);
      if (stride == 2 && ((pz | px | py) & 1)) continue;
      z = stride == 2 ? pz >> 1 : pz; x = stride == 2 ? px >> 1 : px; y = stride == 2 ? py >> 1 : py;
    } else {
      z = stride * Z + tap_dz(t); x = stride * X + tap_dx(t); y = stride * Y + tap_dy(t);
    }
    if (z < 0 || z >= sz || x < 0 || x >= sx || y < 0 || y >= sy) continue;
    const float v = src[(int64_t(z) * sx + x) * sy + y];
#pragma unroll
    for (int k = 0; k < NR; ++k) acc[k] = fmaf(wl[t][k], v, acc[k]);
  }
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    if (m0 + k >= mc) break;
    float* dst = out + int64_t(m0 + k) * nres + o;
    if constexpr (BWD) {
      *dst = accumulate ? *dst + acc[k] : acc[k];
    } else {
      const float v = acc[k] + bias[m0 + k];
      *dst = relu ? fmaxf(v, 0.f) : v;
    }
  }
}

// Workgroups per 16 result channels: a workgroup stages up to 55 KB of weights
// before its first tile, so beyond two rounds of the chip (two workgroups of
// that size per CU) a workgroup takes several tiles.
constexpr int64_t kConvGroups = 1024;
// The data gradient's waves share a node tile while there are fewer (node,
// channel) tiles than about half the SIMDs, and with more source channels a
// little longer, which take a wave of its own more time (16 source channels:
// 265 tiles 10.6 us shared, 14.3 a wave each, 977 tiles 17.3 and 12.5; 64 source
// channels: 530 tiles 33.2 and 39.1, 977 tiles 42.8 and 38.9).  Shared on every
// grid it took 92 us for 6 source and 3 result channels on 49x97x49 nodes, 35
// now.
constexpr int64_t conv_split(int kc) { return kc > 16 ? 768 : 512; }
// Node tiles from which one source channel takes a thread per node (1 result
// channel forward: 4,424 tiles 11.4 us on the matrix cores; 14,557 tiles 22.4 and
// 8.2).
constexpr int64_t kConvOne = 4096;

template <bool BWD>
int conv_launch(int kc, int mc, int rz, int rx, int ry, int sz, int sx, int sy, int stride,
                int relu, int accumulate, const float* src, const uint16_t* w16,
                const float* bias, float* out, void* stream) {
  const int64_t ntiles = (int64_t(rz) * rx * ry + 15) / 16, mt = (mc + 15) / 16;
  TL_ARG(ntiles < (int64_t(1) << 31) && mt < 65536, "grid too large for the convolution");
  if (kc == 1 && mc <= 64 && ntiles >= kConvOne) {
    const dim3 grid(unsigned((int64_t(rz) * rx * ry + BS - 1) / BS), unsigned((mc + NR - 1) / NR));
    hipLaunchKernelGGL(conv_one_kernel<BWD>, grid, dim3(BS), 0, static_cast<hipStream_t>(stream), mc,
                       rz, rx, ry, sz, sx, sy, stride, relu, accumulate, src,
                       reinterpret_cast<const _Float16*>(w16), bias, out);
    TL_CHECK_LAUNCH();
    return TL_OK;
  }
  const bool split = BWD && ntiles * mt < conv_split(kc);
  const int64_t groups = split ? ntiles : (ntiles + CW - 1) / CW;
  const int64_t gx = std::min<int64_t>(groups, kConvGroups / std::min<int64_t>(mt, 4));
  auto launch = [&](auto sp, auto ng) {
    constexpr int NG = decltype(ng)::value;
    hipLaunchKernelGGL((conv_kernel<BWD, decltype(sp)::value, NG, NG <= 4 ? 9 : 3>),
                       dim3(unsigned(gx), unsigned(mt)), dim3(CT), 0,
                       static_cast<hipStream_t>(stream), kc, mc, rz, rx, ry, sz, sx, sy, stride, relu,
                       accumulate, int(ntiles), src, reinterpret_cast<const _Float16*>(w16), bias, out);
  };
  auto go = [&](auto ng) {
    if constexpr (BWD)
      if (split) return launch(std::true_type{}, ng);
    launch(std::false_type{}, ng);
  };
  if (kc <= 4) go(std::integral_constant<int, 1>{});
  else if (kc <= 8) go(std::integral_constant<int, 2>{});
  else if (kc <= 16) go(std::integral_constant<int, 4>{});
  else if (kc <= 32) go(std::integral_constant<int, 8>{});
  else go(std::integral_constant<int, 16>{});  // the entry points admit at most 64
  TL_CHECK_LAUNCH();
  return TL_OK;
}

// gw[co][ci][t] = sum_o gy[co][o] * a[ci][stride*o + off_t]; gb[co] = sum_o gy[co][o],
// products and sums in FP64 on the matrix cores (v_mfma_f64_16x16x4f64, whose
// operands are exact): rows = 16 output channels, columns = 16 input channels
// of one tap (blockIdx.x = tap, .y = channel tile), inner dimension = 4 nodes.
// The 16 waves of a workgroup take runs of 16 nodes in turn (so that the
// nodes a lane reads in one channel lie in one line), and their sums are
// added through LDS in a fixed order.  Tap 13 (the centre) also sums gy.
// One workgroup per channel pair with 28 FP64 sums per thread: 62 us per
// layer on average for a 48x24x24 design, 23 now.
typedef double nn_d4 __attribute__((ext_vector_type(4)));
constexpr int WG_WAVES = 16;
__global__ __launch_bounds__(64 * WG_WAVES) void conv_bwd_weight_kernel(
    int cin, int cout, int nz, int nx, int ny, int oz, int ox, int oy, int stride,
    const float* __restrict__ a, const float* __restrict__ gy, float* __restrict__ gw,
    float* __restrict__ gb) {
  __shared__ double red[WG_WAVES][16][17];
  const int t = int(blockIdx.x), cit = (cin + 15) / 16;
  const int co0 = int(blockIdx.y) / cit * 16, ci0 = int(blockIdx.y) % cit * 16;
  const int dz = tap_dz(t), dx = tap_dx(t), dy = tap_dy(t);
  const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, j = l & 15, g = l >> 4;
  const int64_t nout = int64_t(oz) * ox * oy, plane = int64_t(nz) * nx * ny;
  const bool cok = co0 + j < cout, iok = ci0 + j < cin;
  const float* gp = gy + int64_t(cok ? co0 + j : 0) * nout;
  const float* ap = a + int64_t(iok ? ci0 + j : 0) * plane;
  nn_d4 acc{0.0, 0.0, 0.0, 0.0};
  double gs = 0.0;
  // lane (j, g): nodes base + 4 g + k of channel row/column j, slice k = 0..3
  for (int64_t base = int64_t(wave) * 16; base < nout; base += 16 * WG_WAVES) {
    const int64_t o0 = base + 4 * g;
    int y = int(o0 % oy), x = int((o0 / oy) % ox), z = int(o0 / (int64_t(oy) * ox));
    float gv[4], av[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool in = o0 + k < nout;
      const int Z = stride * z + dz, X = stride * x + dx, Y = stride * y + dy;
      const bool ok = in && Z >= 0 && Z < nz && X >= 0 && X < nx && Y >= 0 && Y < ny;
      const float gq = gp[in ? o0 + k : 0];
      const float aq = ap[ok ? (int64_t(Z) * nx + X) * ny + Y : 0];
      gv[k] = in && cok ? gq : 0.f;
      gs += double(gv[k]);
      gv[k] = ok ? gv[k] : 0.f;  // both operands: a skipped term stays out whatever it holds
      av[k] = ok && iok ? aq : 0.f;
      if (++y == oy) { y = 0; if (++x == ox) { x = 0; ++z; } }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(double(gv[k]), double(av[k]), acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][g + 4 * i][j] = acc[i];
  __syncthreads();
  if (threadIdx.x < 256) {
    const int m = threadIdx.x >> 4, n = threadIdx.x & 15;
    double s = 0.0;
    for (int q = 0; q < WG_WAVES; ++q) s += red[q][m][n];
    if (co0 + m < cout && ci0 + n < cin)
      gw[(int64_t(co0 + m) * cin + ci0 + n) * 27 + t] = float(s);
  }
  if (t != 13 || ci0 != 0) return;
  __syncthreads();
  red[wave][g][j] = gs;
  __syncthreads();
  if (threadIdx.x < 16 && co0 + int(threadIdx.x) < cout) {
    double s = 0.0;
    for (int q = 0; q < WG_WAVES; ++q)
      for (int r = 0; r < 4; ++r) s += red[q][r][threadIdx.x];
    gb[co0 + threadIdx.x] = float(s);
  }
}

// g *= (y > 0)
__global__ void relu_mask_kernel(int64_t n, const float* __restrict__ y, float* __restrict__ g) {
  for (int64_t i = blockIdx.x * int64_t(BS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * BS)
    if (!(y[i] > 0.f)) g[i] = 0.f;
}

__device__ inline float lin_w(int d) { return d == 0 ? 1.f : 0.5f; }

// fine[c][Z][X][Y] (+)= sum of the coarse neighbours with weights 1 or 1/2 per axis
__global__ void upsample_kernel(int c, int cz, int cx, int cy, const float* __restrict__ in,
                                float* __restrict__ out, int accumulate) {
  const int fz = 2 * cz - 1, fx = 2 * cx - 1, fy = 2 * cy - 1;
  const int64_t nf = int64_t(fz) * fx * fy, nc = int64_t(cz) * cx * cy;
  for (int64_t i = blockIdx.x * int64_t(BS) + threadIdx.x; i < nf * c; i += int64_t(gridDim.x) * BS) {
    const int ch = int(i / nf);
    const int64_t f = i % nf;
    const int Y = int(f % fy), X = int((f / fy) % fx), Z = int(f / (int64_t(fy) * fx));
    float s = 0.f;
    for (int az = Z >> 1; az <= (Z + 1) >> 1; ++az)
      for (int ax = X >> 1; ax <= (X + 1) >> 1; ++ax)
        for (int ay = Y >> 1; ay <= (Y + 1) >> 1; ++ay)
          s += lin_w(Z - 2 * az) * lin_w(X - 2 * ax) * lin_w(Y - 2 * ay) *
               in[int64_t(ch) * nc + (int64_t(az) * cx + ax) * cy + ay];
    out[i] = accumulate ? out[i] + s : s;
  }
}

// coarse[c][z][x][y] (+)= transpose of upsample applied to the fine gradient
__global__ void upsample_t_kernel(int c, int cz, int cx, int cy, const float* __restrict__ gf,
                                  float* __restrict__ gc, int accumulate) {
  const int fz = 2 * cz - 1, fx = 2 * cx - 1, fy = 2 * cy - 1;
  const int64_t nf = int64_t(fz) * fx * fy, nc = int64_t(cz) * cx * cy;
  for (int64_t i = blockIdx.x * int64_t(BS) + threadIdx.x; i < nc * c; i += int64_t(gridDim.x) * BS) {
    const int ch = int(i / nc);
    const int64_t k = i % nc;
    const int y = int(k % cy), x = int((k / cy) % cx), z = int(k / (int64_t(cy) * cx));
    float s = 0.f;
    for (int dz = -1; dz <= 1; ++dz)
      for (int dx = -1; dx <= 1; ++dx)
        for (int dy = -1; dy <= 1; ++dy) {
          const int Z = 2 * z + dz, X = 2 * x + dx, Y = 2 * y + dy;
          if (Z < 0 || Z >= fz || X < 0 || X >= fx || Y < 0 || Y >= fy) continue;
          s += lin_w(dz) * lin_w(dx) * lin_w(dy) * gf[int64_t(ch) * nf + (int64_t(Z) * fx + X) * fy + Y];
        }
    gc[i] = accumulate ? gc[i] + s : s;
  }
}

// grad = 2 (p - t) / n; per-block partial sums of (p - t)^2
__global__ __launch_bounds__(BS) void mse_kernel(int64_t n, const float* __restrict__ p,
                                                 const float* __restrict__ t,
                                                 float* __restrict__ grad,
                                                 double* __restrict__ partials) {
  __shared__ double sh[BS / 64 + 2];
  double acc = 0.0;
  for (int64_t i = blockIdx.x * int64_t(BS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * BS) {
    const float d = p[i] - t[i];
    grad[i] = 2.f * d / float(n);
    acc += double(d) * double(d);
  }
  double v[1] = {acc};
  block_sum<1>(v, sh);
  if (threadIdx.x == 0) partials[blockIdx.x] = v[0];
}

__global__ __launch_bounds__(BS) void sum_kernel(const double* __restrict__ partials, int nb,
                                                 double scale, double* __restrict__ out) {
  __shared__ double sh[BS / 64 + 2];
  double v[1] = {0.0};
  for (int i = threadIdx.x; i < nb; i += BS) v[0] += partials[i];
  block_sum<1>(v, sh);
  if (threadIdx.x == 0) *out = v[0] * scale;
}

// Adam (Kingma & Ba 2015, Algorithm 1) on fp32 master weights; fp16 copy for the kernels
__global__ void adam_kernel(int64_t n, float* __restrict__ w, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v,
                            _Float16* __restrict__ w16, float lr, float b1, float b2, float eps,
                            float c1, float c2) {
  for (int64_t i = blockIdx.x * int64_t(BS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * BS) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    if (w16) w16[i] = _Float16(wi);
  }
}

// Network inputs on the level-1 node grid (fine node (2i, 2j, 2k)) of a 3D
// grid: [0] mean density of the fine elements at the node, [1..3] the load
// restricted by full weighting (the transpose of the trilinear
// prolongation) times fscale, [4] 1 where a DOF of the node is fixed, [5] 1.
__global__ void features_kernel(int nelx, int nely, int nelz, const double* __restrict__ xe,
                                const double* __restrict__ f, const uint8_t* __restrict__ mask,
                                double fscale, float* __restrict__ out) {
  const int nx = nelx + 1, ny = nely + 1, nz = nelz + 1;
  const int cx = nelx / 2 + 1, cy = nely / 2 + 1, cz = nelz / 2 + 1;
  const int64_t nc = int64_t(cx) * cy * cz;
  for (int64_t k = blockIdx.x * int64_t(BS) + threadIdx.x; k < nc; k += int64_t(gridDim.x) * BS) {
    const int y = int(k % cy), x = int((k / cy) % cx), z = int(k / (int64_t(cy) * cx));
    const int X = 2 * x, Y = 2 * y, Z = 2 * z;
    double xs = 0.0;
    int ne = 0;
    for (int ez = Z - 1; ez <= Z; ++ez)
      for (int ex = X - 1; ex <= X; ++ex)
        for (int ey = Y - 1; ey <= Y; ++ey) {
          if (ex < 0 || ex >= nelx || ey < 0 || ey >= nely || ez < 0 || ez >= nelz) continue;
          xs += xe[(int64_t(ez) * nelx + ex) * nely + ey];
          ++ne;
        }
    double fr[3] = {0.0, 0.0, 0.0};
    for (int dz = -1; dz <= 1; ++dz)
      for (int dx = -1; dx <= 1; ++dx)
        for (int dy = -1; dy <= 1; ++dy) {
          const int FZ = Z + dz, FX = X + dx, FY = Y + dy;
          if (FZ < 0 || FZ >= nz || FX < 0 || FX >= nx || FY < 0 || FY >= ny) continue;
          const double wgt = (dz ? 0.5 : 1.0) * (dx ? 0.5 : 1.0) * (dy ? 0.5 : 1.0);
          const int64_t fn = (int64_t(FZ) * nx + FX) * ny + FY;
          for (int c = 0; c < 3; ++c) fr[c] += wgt * f[fn * 3 + c];
        }
    const int64_t fn0 = (int64_t(Z) * nx + X) * ny + Y;
    out[k] = float(ne ? xs / ne : 0.0);
    for (int c = 0; c < 3; ++c) out[(1 + c) * nc + k] = float(fr[c] * fscale);
    out[4 * nc + k] = mask[fn0] ? 1.f : 0.f;
    out[5 * nc + k] = 1.f;
  }
}

// out[c][k] = scale * u[fine node (2i, 2j, 2k)][c]  (injection)
__global__ void inject_kernel(int nelx, int nely, int nelz, const double* __restrict__ u,
                              double scale, float* __restrict__ out) {
  const int nx = nelx + 1, ny = nely + 1;
  const int cx = nelx / 2 + 1, cy = nely / 2 + 1, cz = nelz / 2 + 1;
  const int64_t nc = int64_t(cx) * cy * cz;
  for (int64_t k = blockIdx.x * int64_t(BS) + threadIdx.x; k < nc; k += int64_t(gridDim.x) * BS) {
    const int y = int(k % cy), x = int((k / cy) % cx), z = int(k / (int64_t(cy) * cx));
    const int64_t fn = (int64_t(2 * z) * nx + 2 * x) * ny + 2 * y;
    for (int c = 0; c < 3; ++c) out[c * nc + k] = float(u[fn * 3 + c] * scale);
  }
}

// x[fine DOF] = trilinear interpolation of the channel-major level-1 field y
// (zero on fixed DOFs)
__global__ void prolong3_kernel(int nelx, int nely, int nelz, const float* __restrict__ yc,
                                const uint8_t* __restrict__ mask, double* __restrict__ x) {
  const int nx = nelx + 1, ny = nely + 1, nz = nelz + 1;
  const int cx = nelx / 2 + 1, cy = nely / 2 + 1, cz = nelz / 2 + 1;
  const int64_t nc = int64_t(cx) * cy * cz, nf = int64_t(nx) * ny * nz;
  for (int64_t n = blockIdx.x * int64_t(BS) + threadIdx.x; n < nf; n += int64_t(gridDim.x) * BS) {
    const int Y = int(n % ny), X = int((n / ny) % nx), Z = int(n / (int64_t(ny) * nx));
    double s[3] = {0.0, 0.0, 0.0};
    for (int az = Z >> 1; az <= (Z + 1) >> 1; ++az)
      for (int ax = X >> 1; ax <= (X + 1) >> 1; ++ax)
        for (int ay = Y >> 1; ay <= (Y + 1) >> 1; ++ay) {
          const double wgt = double(lin_w(Z - 2 * az)) * lin_w(X - 2 * ax) * lin_w(Y - 2 * ay);
          const int64_t k = (int64_t(az) * cx + ax) * cy + ay;
          for (int c = 0; c < 3; ++c) s[c] += wgt * double(yc[c * nc + k]);
        }
    const uint8_t mk = mask[n];
    for (int c = 0; c < 3; ++c) x[n * 3 + c] = ((mk >> c) & 1) ? 0.0 : s[c];
  }
}

// partial sums of (a.b, c.d)
__global__ __launch_bounds__(BS) void dot2_kernel(int64_t n, const double* __restrict__ a,
                                                  const double* __restrict__ b,
                                                  const double* __restrict__ c,
                                                  const double* __restrict__ d,
                                                  double* __restrict__ partials) {
  __shared__ double sh[2 * (BS / 64) + 2];
  double v[2] = {0.0, 0.0};
  for (int64_t i = blockIdx.x * int64_t(BS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * BS) {
    v[0] += a[i] * b[i];
    v[1] += c[i] * d[i];
  }
  block_sum<2>(v, sh);
  if (threadIdx.x == 0) {
    partials[blockIdx.x] = v[0];
    partials[1024 + blockIdx.x] = v[1];
  }
}

__global__ __launch_bounds__(BS) void scale_by_ratio_kernel(int64_t n, const double* __restrict__ partials,
                                                            int nb, double* __restrict__ x,
                                                            double* __restrict__ alpha) {
  // every block folds the partials in the same fixed order (identical result)
  __shared__ double sh[2 * (BS / 64) + 2];
  double v[2] = {0.0, 0.0};
  for (int i = threadIdx.x; i < nb; i += BS) {
    v[0] += partials[i];
    v[1] += partials[1024 + i];
  }
  block_sum<2>(v, sh);
  const double a = v[1] > 0.0 ? v[0] / v[1] : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) *alpha = a;
  for (int64_t i = blockIdx.x * int64_t(BS) + threadIdx.x; i < n; i += int64_t(gridDim.x) * BS)
    x[i] *= a;
}

unsigned grid1(int64_t n) { return unsigned(std::min<int64_t>((n + BS - 1) / BS, 4096)); }

int out_dim(int n, int stride) { return stride == 1 ? n : (n - 1) / 2 + 1; }

}  // namespace
}  // namespace tl

using namespace tl;

extern "C" {

int tl_nn_conv3d(int32_t cin, int32_t cout, int32_t nz, int32_t nx, int32_t ny, int32_t stride,
                 int32_t relu, const float* in, const uint16_t* w16, const float* bias, float* out,
                 void* stream) {
  TL_ARG(in && w16 && bias && out, "null argument");
  TL_ARG(cin >= 1 && cin <= 64 && cout >= 1 && nz >= 1 && nx >= 1 && ny >= 1,
         "bad shape (1 <= cin <= 64)");
  TL_ARG(stride == 1 || (stride == 2 && nz % 2 == 1 && nx % 2 == 1 && ny % 2 == 1),
         "stride must be 1, or 2 on odd node counts");
  const int oz = out_dim(nz, stride), ox = out_dim(nx, stride), oy = out_dim(ny, stride);
  return conv_launch<false>(cin, cout, oz, ox, oy, nz, nx, ny, stride, relu, 0, in, w16, bias, out,
                            stream);
}

int tl_nn_conv3d_bwd_data(int32_t cin, int32_t cout, int32_t nz, int32_t nx, int32_t ny,
                          int32_t stride, const float* gout, const uint16_t* w16, float* gin,
                          int32_t accumulate, void* stream) {
  TL_ARG(gout && w16 && gin, "null argument");
  TL_ARG(cin >= 1 && cout >= 1 && cout <= 64 && nz >= 1 && nx >= 1 && ny >= 1,
         "bad shape (1 <= cout <= 64)");
  TL_ARG(stride == 1 || (stride == 2 && nz % 2 == 1 && nx % 2 == 1 && ny % 2 == 1),
         "stride must be 1, or 2 on odd node counts");
  const int oz = out_dim(nz, stride), ox = out_dim(nx, stride), oy = out_dim(ny, stride);
  return conv_launch<true>(cout, cin, nz, nx, ny, oz, ox, oy, stride, 0, accumulate, gout, w16,
                           nullptr, gin, stream);
}

int tl_nn_conv3d_bwd_weight(int32_t cin, int32_t cout, int32_t nz, int32_t nx, int32_t ny,
                            int32_t stride, const float* in, const float* gout, float* gw,
                            float* gb, void* stream) {
  TL_ARG(in && gout && gw && gb, "null argument");
  TL_ARG(cin >= 1 && cout >= 1 && nz >= 1 && nx >= 1 && ny >= 1, "bad shape");
  TL_ARG(stride == 1 || (stride == 2 && nz % 2 == 1 && nx % 2 == 1 && ny % 2 == 1),
         "stride must be 1, or 2 on odd node counts");
  const int oz = out_dim(nz, stride), ox = out_dim(nx, stride), oy = out_dim(ny, stride);
  const int64_t tiles = int64_t((cout + 15) / 16) * ((cin + 15) / 16);
  TL_ARG(tiles < 65536, "too many channels for the weight gradient");
  hipLaunchKernelGGL(conv_bwd_weight_kernel, dim3(27, unsigned(tiles)), dim3(64 * WG_WAVES), 0,
                     static_cast<hipStream_t>(stream), cin, cout, nz, nx, ny, oz, ox, oy, stride,
                     in, gout, gw, gb);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_nn_relu_mask(int64_t n, const float* y, float* g, void* stream) {
  TL_ARG(y && g && n >= 0, "bad argument");
  if (n == 0) return TL_OK;
  hipLaunchKernelGGL(relu_mask_kernel, dim3(grid1(n)), dim3(BS), 0,
                     static_cast<hipStream_t>(stream), n, y, g);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_nn_upsample(int32_t c, int32_t cz, int32_t cx, int32_t cy, const float* coarse,
                   float* fine, int32_t accumulate, void* stream) {
  TL_ARG(coarse && fine && c >= 1 && cz >= 2 && cx >= 2 && cy >= 2, "bad argument");
  const int64_t n = int64_t(c) * (2 * cz - 1) * (2 * cx - 1) * (2 * cy - 1);
  hipLaunchKernelGGL(upsample_kernel, dim3(grid1(n)), dim3(BS), 0,
                     static_cast<hipStream_t>(stream), c, cz, cx, cy, coarse, fine, accumulate);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_nn_upsample_t(int32_t c, int32_t cz, int32_t cx, int32_t cy, const float* gfine,
                     float* gcoarse, int32_t accumulate, void* stream) {
  TL_ARG(gfine && gcoarse && c >= 1 && cz >= 2 && cx >= 2 && cy >= 2, "bad argument");
  const int64_t n = int64_t(c) * cz * cx * cy;
  hipLaunchKernelGGL(upsample_t_kernel, dim3(grid1(n)), dim3(BS), 0,
                     static_cast<hipStream_t>(stream), c, cz, cx, cy, gfine, gcoarse, accumulate);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_nn_mse(int64_t n, const float* pred, const float* target, float* grad, double* partials,
              double* loss, void* stream) {
  TL_ARG(pred && target && grad && partials && loss && n > 0, "bad argument");
  const unsigned nb = std::min<unsigned>(grid1(n), 1024u);
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(mse_kernel, dim3(nb), dim3(BS), 0, s, n, pred, target, grad, partials);
  TL_CHECK_LAUNCH();
  hipLaunchKernelGGL(sum_kernel, dim3(1), dim3(BS), 0, s, partials, int(nb), 1.0 / double(n), loss);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_nn_adam(int64_t n, float* w, const float* g, float* m, float* v, uint16_t* w16,
               int32_t step, float lr, void* stream) {
  TL_ARG(w && g && m && v && n > 0 && step >= 1, "bad argument");
  const float b1 = 0.9f, b2 = 0.999f;
  const float c1 = float(1.0 - std::pow(0.9, step)), c2 = float(1.0 - std::pow(0.999, step));
  hipLaunchKernelGGL(adam_kernel, dim3(grid1(n)), dim3(BS), 0, static_cast<hipStream_t>(stream),
                     n, w, g, m, v, reinterpret_cast<_Float16*>(w16), lr, b1, b2, 1e-8f, c1, c2);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_nn_features(tl_problem* p, const double* xPhys, const double* f, double fscale,
                   float* out) {
  TL_ARG(p && xPhys && f && out, "null argument");
  const Grid& g = p->g;
  TL_ARG(g.dim == 3 && p->ndpn == 3 && g.nelx % 2 == 0 && g.nely % 2 == 0 && g.nelz % 2 == 0,
         "network features: 3D H8 elasticity with even element counts");
  const int64_t nc = int64_t(g.nelx / 2 + 1) * (g.nely / 2 + 1) * (g.nelz / 2 + 1);
  hipLaunchKernelGGL(features_kernel, dim3(grid1(nc)), dim3(BS), 0, p->stream, g.nelx, g.nely,
                     g.nelz, xPhys, f, p->op.mask.as<uint8_t>(), fscale, out);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_nn_inject(tl_problem* p, const double* u, double scale, float* out) {
  TL_ARG(p && u && out, "null argument");
  const Grid& g = p->g;
  TL_ARG(g.dim == 3 && p->ndpn == 3 && g.nelx % 2 == 0 && g.nely % 2 == 0 && g.nelz % 2 == 0,
         "network targets: 3D H8 elasticity with even element counts");
  const int64_t nc = int64_t(g.nelx / 2 + 1) * (g.nely / 2 + 1) * (g.nelz / 2 + 1);
  hipLaunchKernelGGL(inject_kernel, dim3(grid1(nc)), dim3(BS), 0, p->stream, g.nelx, g.nely,
                     g.nelz, u, scale, out);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_nn_prolong(tl_problem* p, const float* y, double* x) {
  TL_ARG(p && y && x, "null argument");
  const Grid& g = p->g;
  TL_ARG(g.dim == 3 && p->ndpn == 3 && g.nelx % 2 == 0 && g.nely % 2 == 0 && g.nelz % 2 == 0,
         "network output: 3D H8 elasticity with even element counts");
  hipLaunchKernelGGL(prolong3_kernel, dim3(grid1(g.nnodes)), dim3(BS), 0, p->stream, g.nelx,
                     g.nely, g.nelz, y, p->op.mask.as<uint8_t>(), x);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

int tl_energy_scale(tl_problem* p, const double* f, double* x, double* work, double* alpha) {
  TL_ARG(p && f && x && work && alpha, "null argument");
  TL_TRY(tl_apply_K(p, x, work, TL_PREC_FP64));
  TL_TRY(p->partials.alloc(sizeof(double) * 2048));
  const unsigned nb = std::min<unsigned>(grid1(p->ndof), 1024u);
  double* part = p->partials.as<double>();
  hipLaunchKernelGGL(dot2_kernel, dim3(nb), dim3(BS), 0, p->stream, p->ndof, f, x, x, work, part);
  TL_CHECK_LAUNCH();
  TL_TRY(p->t.alloc(sizeof(double) * 2));
  hipLaunchKernelGGL(scale_by_ratio_kernel, dim3(grid1(p->ndof)), dim3(BS), 0, p->stream,
                     p->ndof, part, int(nb), x, p->t.as<double>());
  TL_CHECK_LAUNCH();
  TL_HIP(hipMemcpyAsync(alpha, p->t.ptr, sizeof(double), hipMemcpyDeviceToHost, p->stream));
  TL_HIP(hipStreamSynchronize(p->stream));
  return TL_OK;
}

}  // extern "C"
