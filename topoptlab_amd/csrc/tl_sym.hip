// 3D operators in the reflection-symmetric form of the H8 element matrix: the
// fine grid's K.u and the first coarse level's Galerkin operator, both
// matrix-free (the products of topoptlab/topology_optimization.py:429-451 and
// multigrid.py:142-168).
//
// The unit-cell element matrix of an isotropic material commutes with the
// reflections of the cell.  With H the 8-point Hadamard transform of each
// displacement component over the element's corners, KE = H^T B H, and B
// couples only within one parity class: 45 nonzeros instead of 576.  An
// element then costs about 160 instead of 600 operations: transform the two
// node planes (each plane's in-plane part is shared by the layers below and
// above it), 45 multiply-adds, transform back.
//
// The Galerkin matrix of a level-1 element is linear in its 8 children's
// scales, and in the same basis sum_m t_m B_m with t the Hadamard transform of
// the child scales and B_m constant: 279 nonzeros together.  Applying it from
// the densities reads about 25 MB at 192x96x96 in FP64 where the stored
// half-stencil reads 252 MB.  Its arithmetic is FP64 in the FP32 cycles too
// (vectors in FP32): the coefficients of a stored FP32 stencil are FP64 sums
// rounded once, and formed in FP32 from FP32 scales they had up to a tenth more
// error on rough fields (white noise, scales over nine decades: stored 8.4e-8,
// FP32 9.1e-8, FP64 2.6e-8 with the output's rounding; on nearly constant fields
// 1e-5, 2e-6 and 2.5e-8).  It costs a third: at 192x96x96 residual 12.6 -> 16.3
// us, sweep 11.6 -> 15.9, sweep with the correction 15.9 -> 23.2.
//
// A workgroup owns a 16x16 tile of element columns (thread (tx, ty): element
// column (X0 + tx - 1, Y0 + ty - 1), y fastest) and walks a range of element
// layers in z; it produces the 15x15 nodes all of whose elements it holds.  A
// node plane (17x17 nodes) is staged in LDS once, a layer ahead, through
// registers.  The four columns around a node are summed by a DPP row shift in
// y and through LDS in x; one barrier per layer covers both the staged plane
// and that exchange.
#include "tl_internal.hpp"
#include "sym_pattern.hpp"

#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

namespace tl {
namespace {

constexpr int BS = 256;
constexpr int TE = 16;       // element columns per tile side
constexpr int TN = TE - 1;   // nodes produced per tile side
constexpr int TS = TE + 1;   // nodes staged per tile side
static_assert(TE * TE == BS, "one element column per thread");

constexpr int TC = 10;  // coarse nodes per tile side that 17 staged nodes interpolate from
constexpr int CR = 4;   // coarse tiles kept in LDS

// Arithmetic of an operator with vectors of type T.
template <typename T, bool CG>
using sym_arith = std::conditional_t<CG, double, T>;

// T: vectors, A: arithmetic
template <typename T, typename A>
struct SymArgs {
  const T* u;          // input; SRC_P: z
  const T* pin;        // SRC_P: previous search direction
  T* pout;             // SRC_P: new search direction
  const double* beta;  // SRC_P: device scalar, or the partials of rho
  FoldIn rho;
  FoldIn rr;           // SRC_SEED: partials of r.r of the iteration before, or none
  const T* xc;         // SRC_*CORR: the coarse level's correction
  int cnx, cny, cnz;   // and its node counts
  const A* sp;         // zero-bordered scales of the fine grid
  const uint8_t* mask;
  const void* b;       // KU_RESID / KU_JACOBI*: right-hand side
  const T* dinv;
  T omega;
  void* y;
  double* partials;
  const int* done;
  int nelx, nely, nelz, nx, ny, nz;  // the operator's own grid
  int fnelx, fnely;                  // CG: the fine grid below it
  int ncy;                           // tile columns along y
  unsigned ncol;                     // tile columns
  unsigned nseg;                     // equal z ranges per column, or 0 (see sym_segments)
  A kv[16];                          // group values of the pattern
  A kt;                              // products: stiffness against a translation
};

template <int NDPN, bool CG>
__host__ __device__ constexpr int sym_tab(int i) {
  if constexpr (NDPN == 3) return CG ? kTabSymC_elast[i] : kTabSym_elast[i];
  else return CG ? kTabSymC_poisson[i] : kTabSym_poisson[i];
}

// parity class of basis function (mode m, component c)
template <int NDPN>
__host__ __device__ constexpr int sym_class(int m, int c) {
  return NDPN == 3 ? m ^ (1 << c) : m;
}
// mode of component c in class x
template <int NDPN>
__host__ __device__ constexpr int sym_mode(int x, int c) {
  return NDPN == 3 ? x ^ (1 << c) : x;
}

__device__ __forceinline__ float sym_fma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double sym_fma(double a, double b, double c) { return __builtin_fma(a, b, c); }

// value of the next lane in the caller's row of 16 (0 past its end)
__device__ __forceinline__ float next_lane(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
                                       0, __builtin_bit_cast(int, v), 0x101 /* row_shl:1 */, 0xf, 0xf, true));
}
__device__ __forceinline__ double next_lane(double v) {
  int2 w = __builtin_bit_cast(int2, v);
  w.x = __builtin_amdgcn_update_dpp(0, w.x, 0x101, 0xf, 0xf, true);
  w.y = __builtin_amdgcn_update_dpp(0, w.y, 0x101, 0xf, 0xf, true);
  return __builtin_bit_cast(double, w);
}

// 8-point Hadamard transform, index m = mx + 2 my + 4 mz from cz 4 + cx 2 + cy
template <typename T>
__device__ __forceinline__ void child_modes(T (&t)[8]) {
  T s[8];
#pragma unroll
  for (int c = 0; c < 4; ++c) {  // z
    s[c] = t[c] + t[4 + c];
    s[4 + c] = t[c] - t[4 + c];
  }
#pragma unroll
  for (int h = 0; h < 8; h += 4) {  // (cx, cy) -> mx + 2 my
    const T a = s[h] + s[h + 1], b = s[h] - s[h + 1];          // cx = 0: y sum, difference
    const T c = s[h + 2] + s[h + 3], d = s[h + 2] - s[h + 3];  // cx = 1
    t[h] = a + c;
    t[h + 1] = a - c;
    t[h + 2] = b + d;
    t[h + 3] = b - d;
  }
}

// Element scales of the thread's column in one layer: the element's own
// (fine) or its children's modes (CG).
template <typename A, bool CG>
struct Scales {
  A s[CG ? 8 : 1];
  template <typename T>
  __device__ __forceinline__ void load(const SymArgs<T, A>& a, int ix, int iy, int ez) {
    if constexpr (CG) {
      // element (ix - 1, iy - 1, ez); zero outside the grid
      const bool in = ix >= 1 && ix <= a.nelx && iy >= 1 && iy <= a.nely && ez >= 0 && ez < a.nelz;
      const int cx = min(max(ix, 1), a.nelx), cy = min(max(iy, 1), a.nely),
                cz = min(max(ez, 0), a.nelz - 1);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int64_t i = (int64_t(2 * cz + (k >> 2) + 1) * (a.fnelx + 2) + 2 * cx - 1 + (k >> 1 & 1)) *
                              (a.fnely + 2) + 2 * cy - 1 + (k & 1);
        const A v = a.sp[i];
        s[k] = in ? v : A(0);
      }
    } else {
      // the border of the padded array holds zeros
      const int px = min(ix, a.nelx + 1), py = min(iy, a.nely + 1);
      s[0] = a.sp[(int64_t(ez + 1) * (a.nelx + 2) + px) * (a.nely + 2) + py];
    }
  }
  __device__ __forceinline__ void modes() {
    if constexpr (CG) child_modes(s);
  }
};

// Element contraction of one layer: lower and upper plane's in-plane modes
// flo, fhi (index mode * NDPN + component, mode = mx + 2 my); adds the lower
// plane's contribution to tot and returns the upper plane's in up.
//
// TR (the products that define the system, not the preconditioner's): the
// translations' entry of B, which is 0 but for the rounding of the caller's
// matrix (about 1e-17 of it), is applied as well.  On stiff islands held by
// void elements of 1e-9 of their stiffness it decides the ninth digit of the
// solution: without it a 120x20x12 solve differs by 9e-9 from one with the
// matrix as given.  12 operations per element: 95x61x47 product 15.6 -> 16.1 us,
// 192x96x96 solve 28.3 -> 28.0 ms.
template <int NDPN, typename T, typename A, bool CG, bool TR>
__device__ __forceinline__ void sym_layer(const SymArgs<T, A>& a, const Scales<A, CG>& S,
                                          const A (&flo)[4 * NDPN], const A (&fhi)[4 * NDPN],
                                          A (&tot)[4 * NDPN], A (&up)[4 * NDPN]) {
  constexpr int ND = 8 * NDPN;
  A U[ND];
#pragma unroll
  for (int i = 0; i < 4 * NDPN; ++i) {
    U[i] = flo[i] + fhi[i];
    U[4 * NDPN + i] = flo[i] - fhi[i];
  }
  A ks[16];  // fine: the group values times the element's scale
  if constexpr (!CG) {
#pragma unroll
    for (int g = 0; g < (NDPN == 3 ? kGroupsSym_elast : kGroupsSym_poisson); ++g) ks[g] = S.s[0] * a.kv[g];
  }
#pragma unroll
  for (int i = 0; i < 4 * NDPN; ++i) {
    A y[2];
    bool any[2] = {false, false};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int m = 4 * h + i / NDPN, c = i % NDPN, r = m * NDPN + c;
      y[h] = A(0);
      if (TR && m == 0) {
        y[h] = S.s[0] * a.kt * U[r];
        any[h] = true;
      }
      if constexpr (!CG) {
#pragma unroll
        for (int k = 0; k < NDPN; ++k) {
          const int col = sym_mode<NDPN>(sym_class<NDPN>(m, c), k) * NDPN + k;
          const int p = sym_tab<NDPN, false>(r * ND + col);
          if (p == 0) continue;
          const A v = ks[(p > 0 ? p : -p) - 1];
          if (!any[h]) y[h] = p > 0 ? v * U[col] : -v * U[col];
          else y[h] = sym_fma(p > 0 ? v : -v, U[col], y[h]);
          any[h] = true;
        }
      } else {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          A t = A(0);
          bool anyq = false;
#pragma unroll
          for (int k = 0; k < NDPN; ++k) {
            const int col = sym_mode<NDPN>(sym_class<NDPN>(m, c) ^ q, k) * NDPN + k;
            const int p = sym_tab<NDPN, true>((q * ND + r) * ND + col);
            if (p == 0) continue;
            const A v = a.kv[(p > 0 ? p : -p) - 1];
            if (!anyq) t = p > 0 ? v * U[col] : -v * U[col];
            else t = sym_fma(p > 0 ? v : -v, U[col], t);
            anyq = true;
          }
          if (!anyq) continue;
          y[h] = any[h] ? sym_fma(S.s[q], t, y[h]) : S.s[q] * t;
          any[h] = true;
        }
      }
    }
    if (any[0] && any[1]) {
      tot[i] += y[0] + y[1];
      up[i] = y[0] - y[1];
    } else if (any[0]) {
      tot[i] += y[0];
      up[i] = y[0];
    } else {
      tot[i] += y[1];
      up[i] = -y[1];
    }
  }
}

// Staging of one node plane: the thread's entries of the 17x17x NDPN tile,
// loaded into registers and stored to LDS later.  With a coarse correction the
// stored value adds the in-plane interpolation of the coarse tile of its plane
// (`ring`, plane z at z % CR, already interpolated in z): in a direction with
// an even coordinate both neighbours are the coinciding coarse node, so one
// average serves every case.
template <int NDPN, typename T, typename A, typename TB, int SRC>
struct Stage {
  static constexpr int N = TS * TS * NDPN, NR = (N + BS - 1) / BS;
  static constexpr bool kTwo = SRC == SRC_P || src_seed(SRC), kCorr = src_corr(SRC);
  using V = std::conditional_t<src_seed(SRC), TB, T>;
  uint32_t off[NR];  // entry offsets within a plane (clamped to the grid)
  int co[kCorr ? NR : 1];      // coarse tile entry, + 1024 if y is odd, + 2048 if x is odd
  struct Vals {  // a plane's values in flight
    V v[NR];
    T w[kTwo ? NR : 1];
    uint8_t mk[kCorr ? NR : 1];  // masks of the entries' nodes
    int z;                       // the plane asked for (past the grid: the last one is held)
  };
  __device__ __forceinline__ bool has(int k) const { return k + 1 < NR || int(threadIdx.x) + k * BS < N; }
  __device__ __forceinline__ void init(const SymArgs<T, A>& a, int x0, int y0) {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int e = int(threadIdx.x) + k * BS;
      const int row = e / (TS * NDPN), rem = e % (TS * NDPN);
      const int x = min(max(x0 - 1 + row, 0), a.nx - 1), y = min(max(y0 - 1 + rem / NDPN, 0), a.ny - 1);
      off[k] = uint32_t((x * a.ny + y) * NDPN + rem % NDPN);
      if constexpr (kCorr)
        co[k] = (((x >> 1) - coarse_base(x0)) * TC + (y >> 1) - coarse_base(y0)) * NDPN + rem % NDPN +
                (y & 1) * 1024 + (x & 1) * 2048;
    }
  }
  __device__ __forceinline__ static int coarse_base(int x0) { return max(x0 - 1, 0) >> 1; }
  __device__ __forceinline__ void load(const SymArgs<T, A>& a, int z, Vals& q) const {
    q.z = z;
    const int64_t base = int64_t(min(max(z, 0), a.nz - 1)) * a.nx * a.ny * NDPN;
    const V* p = (src_seed(SRC) ? static_cast<const V*>(a.b) : reinterpret_cast<const V*>(a.u)) + base;
#pragma unroll
    for (int k = 0; k < NR; ++k)
      if (has(k)) q.v[k] = p[off[k]];
    if constexpr (kTwo) {
      const T* p2 = (src_seed(SRC) ? a.dinv : a.pin) + base;
#pragma unroll
      for (int k = 0; k < NR; ++k)
        if (has(k)) q.w[k] = p2[off[k]];
    }
    if constexpr (kCorr) {
      const uint8_t* m = a.mask + int64_t(min(max(z, 0), a.nz - 1)) * a.nx * a.ny;
#pragma unroll
      for (int k = 0; k < NR; ++k)
        if (has(k)) q.mk[k] = m[off[k] / NDPN];
    }
  }
  __device__ __forceinline__ T value(const SymArgs<T, A>& a, int k, const Vals& q, T beta) const {
    if constexpr (SRC == SRC_P) return T(q.v[k]) + beta * q.w[k];
    else if constexpr (src_seed(SRC)) return zero_guess_sweep<T, TB>(a.omega, q.w[k], q.v[k]);
    else return q.v[k];
  }
  __device__ __forceinline__ void store(const SymArgs<T, A>& a, T* lds, const T* ring, T beta,
                                        const Vals& q) const {
#pragma unroll
    for (int k = 0; k < NR; ++k)
      if (has(k)) {
        T r = value(a, k, q, beta);
        if constexpr (kCorr) {
          const int e = co[k] & 1023, dy = (co[k] & 1024) ? NDPN : 0, dx = (co[k] & 2048) ? TC * NDPN : 0;
          const T* c = ring + (q.z % CR) * (TC * TC * NDPN) + e;
          const T s = T(0.25) * ((c[0] + c[dy]) + (c[dx] + c[dx + dy]));
          if (!((q.mk[k] >> (off[k] % NDPN)) & 1)) r += s;
        }
        lds[threadIdx.x + k * BS] = r;
      }
  }
};

// The thread's entries of the coarse 10x10 tiles (clamped to the grid).  Fine
// plane z interpolates from coarse planes z/2 and (z+1)/2; `next` holds the
// latter of the plane prepared last.
template <int NDPN, typename T, typename A>
struct CoarseStage {
  static constexpr int N = TC * TC * NDPN, NR = (N + BS - 1) / BS;
  uint32_t off[NR];
  T cur[NR], next[NR];
  __device__ __forceinline__ bool has(int k) const { return int(threadIdx.x) + k * BS < N; }
  __device__ __forceinline__ void load(const SymArgs<T, A>& a, int c, T (&v)[NR]) const {
    const T* p = a.xc + int64_t(min(c, a.cnz - 1)) * a.cnx * a.cny * NDPN;
#pragma unroll
    for (int k = 0; k < NR; ++k)
      if (has(k)) v[k] = p[off[k]];
  }
  // Tiles of planes z0 - 1 (if any) to z0 + 2.
  __device__ __forceinline__ void begin(const SymArgs<T, A>& a, int x0, int y0, int z0, T* ring) {
#pragma unroll
    for (int k = 0; k < NR; ++k) {
      const int e = int(threadIdx.x) + k * BS;
      const int x = min((max(x0 - 1, 0) >> 1) + e / (TC * NDPN), a.cnx - 1);
      const int y = min((max(y0 - 1, 0) >> 1) + e % (TC * NDPN) / NDPN, a.cny - 1);
      off[k] = uint32_t((x * a.cny + y) * NDPN + e % NDPN);
    }
    const int z = max(z0 - 1, 0);
    T v[NR];
    load(a, z >> 1, cur);
    load(a, (z + 1) >> 1, next);
    load(a, (z + 2) >> 1, v);
    put(ring, z, cur, next);
    put(ring, z + 1, next, v);
    load(a, (z + 3) >> 1, cur);
    put(ring, z + 2, v, cur);
    if (z0 > 0) {
      load(a, (z + 4) >> 1, next);
      put(ring, z + 3, cur, next);
    } else {
#pragma unroll
      for (int k = 0; k < NR; ++k) next[k] = cur[k];
    }
  }
  __device__ __forceinline__ void put(T* ring, int z, const T (&lo)[NR], const T (&hi)[NR]) const {
#pragma unroll
    for (int k = 0; k < NR; ++k)
      if (has(k)) ring[(z % CR) * N + threadIdx.x + k * BS] = T(0.5) * (lo[k] + hi[k]);
  }
  // Start of the step that prepares plane z, and its end.
  __device__ __forceinline__ void advance(const SymArgs<T, A>& a, int z) {
#pragma unroll
    for (int k = 0; k < NR; ++k) cur[k] = next[k];
    if (z & 1) load(a, (z + 1) >> 1, next);
  }
  __device__ __forceinline__ void finish(T* ring, int z) const { put(ring, z, cur, next); }
};

// In-plane modes of the thread's element from the staged plane, and the value
// of its own output node (the element's corner (1, 1)).
template <int NDPN, typename T, typename A>
__device__ __forceinline__ void plane_modes(const T* lds, int tx, int ty, A (&f)[4 * NDPN],
                                            T (&uc)[NDPN]) {
  const T* p = lds + (tx * TS + ty) * NDPN;
#pragma unroll
  for (int c = 0; c < NDPN; ++c) {
    const A v00 = p[c], v01 = p[NDPN + c], v10 = p[TS * NDPN + c], v11 = p[(TS + 1) * NDPN + c];
    const A a = v00 + v01, b = v00 - v01, d = v10 + v11, e = v10 - v11;
    f[c] = a + d;
    f[NDPN + c] = a - d;
    f[2 * NDPN + c] = b + e;
    f[3 * NDPN + c] = b - e;
    uc[c] = T(v11);
  }
}

// Node planes z0 .. z1-1 of tile column col.
template <int NDPN, typename T, typename A, int MODE, typename TB, typename TO, int SRC, bool CG>
__device__ __forceinline__ void sym_segment(const SymArgs<T, A>& a, T (*plane)[TS * TS * NDPN],
                                            A (*xch)[NDPN * BS], T* ring, unsigned col, int z0,
                                            int z1, T beta, double& dot) {
  constexpr bool CORR = src_corr(SRC), kTrans = MODE == KU_STORE || MODE == KU_STORE_DOT;
  const int tid = int(threadIdx.x), tx = tid >> 4, ty = tid & 15;
  const int x0 = int(col / unsigned(a.ncy)) * TN, y0 = int(col % unsigned(a.ncy)) * TN;
  const int ix = x0 + tx, iy = y0 + ty;
  const bool active = tx < TN && ty < TN && ix < a.nx && iy < a.ny;
  const int64_t node0 = active ? int64_t(ix) * a.ny + iy : 0;
  const int64_t nplane = int64_t(a.nx) * a.ny;
  Stage<NDPN, T, A, TB, SRC> st;
  CoarseStage<NDPN, T, A> cs;
  Scales<A, CG> S, Sn;
  A flo[4 * NDPN], carry[4 * NDPN];
  T uc[NDPN];
  // (planes z0 - 1, z0 and z0 + 1 requested together: product and residual 3 us
  // slower at 192x96x96)
  typename Stage<NDPN, T, A, TB, SRC>::Vals in;
  st.init(a, x0, y0);
  st.load(a, z0, in);
  S.load(a, ix, iy, z0);
  __syncthreads();  // the LDS of the previous segment is free
  if constexpr (CORR) {
    cs.begin(a, x0, y0, z0, ring);
    __syncthreads();
  }
  st.store(a, plane[z0 & 1], ring, beta, in);
#pragma unroll
  for (int i = 0; i < 4 * NDPN; ++i) carry[i] = A(0);
  if (z0 > 0) {  // the layer below gives plane z0's lower part
    Scales<A, CG> Sb;
    st.load(a, z0 - 1, in);
    Sb.load(a, ix, iy, z0 - 1);
    st.store(a, plane[(z0 + 1) & 1], ring, beta, in);
    st.load(a, z0 + 1, in);
    __syncthreads();
    A fb[4 * NDPN], unused[4 * NDPN];
    T ub[NDPN];
    plane_modes<NDPN, T, A>(plane[(z0 + 1) & 1], tx, ty, fb, ub);
    plane_modes<NDPN, T, A>(plane[z0 & 1], tx, ty, flo, uc);
#pragma unroll
    for (int i = 0; i < 4 * NDPN; ++i) unused[i] = A(0);
    Sb.modes();
    sym_layer<NDPN, T, A, CG, kTrans>(a, Sb, fb, flo, unused, carry);
  } else {
    st.load(a, z0 + 1, in);
    __syncthreads();
    plane_modes<NDPN, T, A>(plane[z0 & 1], tx, ty, flo, uc);
  }
  if (z0 > 0) __syncthreads();  // plane z0 - 1 has been read
  st.store(a, plane[(z0 + 1) & 1], ring, beta, in);
  __syncthreads();
  for (int z = z0; z < z1; ++z) {
    const bool more = z + 1 < z1;  // uniform
    if (more) {
      st.load(a, z + 2, in);
      Sn.load(a, ix, iy, z + 1);
      if constexpr (CORR) cs.advance(a, z + 3);  // plane z + 3 is staged in the next step
    }
    // epilogue inputs of the node of plane z
    const int64_t node = int64_t(z) * nplane + node0;
    const uint8_t mk = a.mask[node];
    TB bv[NDPN];
    T dv[NDPN];
#pragma unroll
    for (int c = 0; c < NDPN; ++c) {
      if constexpr (MODE == KU_RESID || MODE == KU_JACOBI || MODE == KU_JACOBI_DOT)
        bv[c] = static_cast<const TB*>(a.b)[node * NDPN + c];
      if constexpr (MODE == KU_JACOBI || MODE == KU_JACOBI_DOT) dv[c] = a.dinv[node * NDPN + c];
    }
    A fhi[4 * NDPN], up[4 * NDPN];
    T un[NDPN];
    plane_modes<NDPN, T, A>(plane[(z + 1) & 1], tx, ty, fhi, un);
    S.modes();
    sym_layer<NDPN, T, A, CG, kTrans>(a, S, flo, fhi, carry, up);
    // carry now holds plane z's in-plane modes from both layers: corner values,
    // summed over the element columns in y (DPP) and x (LDS)
    A acc[NDPN];
    A* xo = xch[z & 1];
#pragma unroll
    for (int c = 0; c < NDPN; ++c) {
      const A p = carry[c] + carry[2 * NDPN + c], q = carry[c] - carry[2 * NDPN + c];
      const A r = carry[NDPN + c] + carry[3 * NDPN + c], s = carry[NDPN + c] - carry[3 * NDPN + c];
      xo[c * BS + tid] = (q + s) + next_lane(p + r);
      acc[c] = (q - s) + next_lane(p - r);
    }
    if (more) {
      st.store(a, plane[z & 1], ring, beta, in);
      if constexpr (CORR) cs.finish(ring, z + 3);
    }
    __syncthreads();
    if (active) {
#pragma unroll
      for (int c = 0; c < NDPN; ++c) {
        acc[c] += xo[c * BS + tid + TE];
        const int64_t g = node * NDPN + c;
        const bool fixed = (mk >> c) & 1;
        TO* y = static_cast<TO*>(a.y);
        if constexpr (SRC == SRC_P) a.pout[g] = uc[c];
        if constexpr (MODE == KU_STORE || MODE == KU_STORE_DOT) {
          const T v = fixed ? T(0) : T(acc[c]);
          y[g] = TO(v);
          if constexpr (MODE == KU_STORE_DOT) dot += double(uc[c]) * double(v);
        } else if constexpr (MODE == KU_RESID) {
          y[g] = TO(fixed ? T(0) : T(A(T(bv[c])) - acc[c]));
        } else {
          const T bb = T(bv[c]);
          const T v = fixed ? T(0) : uc[c] + a.omega * dv[c] * T(A(bb) - acc[c]);
          y[g] = TO(v);
          if constexpr (MODE == KU_JACOBI_DOT) dot += double(bb) * double(v);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 4 * NDPN; ++i) {
      flo[i] = fhi[i];
      carry[i] = up[i];
    }
#pragma unroll
    for (int c = 0; c < NDPN; ++c) uc[c] = un[c];
    S = Sn;
  }
}

template <int NDPN, int SRC, bool CG>
constexpr int sym_waves() {
  return NDPN == 3 && CG && src_corr(SRC) ? 1 : 2;
}

// Split: every column into the same nseg z ranges, a workgroup each, numbered
// range by range, so that the workgroups of an XCD walk the same planes side by
// side and find their neighbours' halo lines in its L2; or, where that leaves
// too many workgroups idle (sym_segments), the ncol * nz (tile column, node
// plane) units evenly over the workgroups, in column order.  A
// segment costs one extra element layer (the one below its first plane).  Two
// waves per SIMD: 170-184 VGPRs in FP64 (256 for the level-1 form); a bound of
// three spills (192x96x96, FP64: residual 40.2 instead of 39.9 us, level-1
// sweep 45.6 instead of 17.2).
//
// Measured at 192x96x96 (kernel times, against the general kernels): FP64
// residual 52.1 -> 39.9 us (146.7 MB; 3.7 TB/s of the 5.1 a copy reaches), last
// smoothing sweep 53.7 -> 45.7, product with the search-direction update
// 19.4 + 52.9 -> 54; level-1 residual and sweep 59.4 and 54.4 (stored
// stencil, 252 MB) -> 17.3 and 17.2.  Inside V(1,1) cycles: residual from the
// seed 45, last sweep from the seed and the coarse correction 57.5 (45.7 and a
// prolongation of 33 before), level-1 sweep with the correction 24 (17.2 + 7),
// and 9 us less in the PCG update, which no longer writes the seed.
// Side by side instead of evenly: 95x61x47 product 16.1 -> 14.0 us; at 192x96x96
// plain product 34.3 -> 32.7 (L2 misses 121 -> 66 MB), level-1 residual and sweep
// 18.7 and 26.0 -> 17.5 and 24.7, the fine kernels with two staged inputs
// unchanged within 1% (61.4, 51.9 and 63.2 us).
// Measured and not kept: two layers per loop turn without the register moves
// (the sweep spills, the rest is unchanged: the moves are not what bounds it).
template <int NDPN, typename T, int MODE, typename TB, typename TO, int SRC, bool CG>
__global__ __launch_bounds__(BS, (sym_waves<NDPN, SRC, CG>())) void sym_kernel(
    SymArgs<T, sym_arith<T, CG>> a) {
  using A = sym_arith<T, CG>;
  __shared__ double sh[BS / 64 + 2];
  if (op_ended<SRC == SRC_SEED>(a.rr, a.done, blockIdx.x == 0 && threadIdx.x == 0, sh)) return;
  __shared__ T plane[2][TS * TS * NDPN];
  __shared__ A xch[2][NDPN * BS];
  __shared__ T ring[src_corr(SRC) ? CR * TC * TC * NDPN : 1];
  // workgroups go round-robin over the 8 XCDs: give each a contiguous range
  const unsigned nb = gridDim.x, hw = blockIdx.x;
  const unsigned xcd = hw & 7u, q = nb >> 3, r = nb & 7u;
  const unsigned w = xcd * q + min(xcd, r) + (hw >> 3);
  const unsigned units = a.ncol * unsigned(a.nz);  // units * (nb + 1) < 2^32 (launcher)
  unsigned u0, u1;
  if (a.nseg) {
    const unsigned seg = w / a.ncol, first = (w - seg * a.ncol) * unsigned(a.nz);
    u0 = first + unsigned(a.nz) * seg / a.nseg;
    u1 = first + unsigned(a.nz) * (seg + 1) / a.nseg;
  } else {
    u0 = units * w / nb;
    u1 = units * (w + 1) / nb;
  }
  u0 = __builtin_amdgcn_readfirstlane(u0);
  u1 = __builtin_amdgcn_readfirstlane(u1);
  T beta = T(0);
  if constexpr (SRC == SRC_P)
    beta = T(fold_in_beta(a.rho, a.beta, blockIdx.x == 0 && threadIdx.x == 0, sh));
  double dot = 0.0;
  while (u0 < u1) {
    const unsigned col = u0 / unsigned(a.nz);
    const int z0 = int(u0 - col * unsigned(a.nz));
    const int z1 = min(a.nz, z0 + int(u1 - u0));
    sym_segment<NDPN, T, A, MODE, TB, TO, SRC, CG>(a, plane, xch, ring, col, z0, z1, beta, dot);
    u0 += unsigned(z1 - z0);
  }
  if constexpr (MODE == KU_STORE_DOT || MODE == KU_JACOBI_DOT) {
    double v[1] = {dot};
    block_sum<1>(v, sh);
    store_partials<1>(v, a.partials);
  }
}

// workgroups the device holds at once (cached per device and kernel)
int sym_slots(const void* kernel, int64_t& slots) {
  static std::mutex mu;
  static std::map<std::pair<int, const void*>, int64_t> cache;
  int dev = 0;
  TL_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(mu);
  auto it = cache.find({dev, kernel});
  if (it == cache.end()) {
    int ncu = 0, per = 0;
    TL_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
    TL_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, BS, 0));
    it = cache.emplace(std::make_pair(dev, kernel), int64_t(std::max(ncu, 1)) * std::max(per, 1)).first;
  }
  slots = it->second;
  return TL_OK;
}

int64_t tile_cols(const Grid& g) {
  return int64_t((g.nx + TN - 1) / TN) * ((g.ny + TN - 1) / TN);
}

// z ranges per column of the side-by-side split, 0 for the even one: taken where
// its longest walk (with the layer below) is no longer than the even split's,
// whose workgroups start a second column on the way.
unsigned sym_segments(int64_t ncol, int64_t nz, int64_t slots) {
  const int64_t nseg = std::min(slots / ncol, nz);
  if (nseg < 1) return 0;
  const int64_t even = (ncol * nz + slots - 1) / slots + 2;
  return (nz + nseg - 1) / nseg + 1 <= even ? unsigned(nseg) : 0;
}

template <int NDPN, typename T, int MODE, typename TB, typename TO, int SRC, bool CG>
int sym_launch(hipStream_t s, const Grid& g, SymArgs<T, sym_arith<T, CG>> a, unsigned* nblocks) {
  auto* kern = sym_kernel<NDPN, T, MODE, TB, TO, SRC, CG>;
  a.nelx = g.nelx; a.nely = g.nely; a.nelz = g.nelz;
  a.nx = g.nx; a.ny = g.ny; a.nz = g.nz;
  a.ncy = (g.ny + TN - 1) / TN;
  a.ncol = unsigned(tile_cols(g));
  int64_t slots = 0;
  TL_TRY(sym_slots(reinterpret_cast<const void*>(kern), slots));
  const int64_t units = int64_t(a.ncol) * g.nz;
  slots = std::max<int64_t>(1, std::min(slots, int64_t(kMaxRedBlocks)));
  a.nseg = sym_segments(a.ncol, g.nz, slots);
  const int64_t nwg = a.nseg ? int64_t(a.ncol) * a.nseg : std::min(slots, units);
  TL_ARG(units * (nwg + 1) < (int64_t(1) << 32), "internal: grid too large for the tiled operator");
  if (nblocks) *nblocks = unsigned(nwg);
  hipLaunchKernelGGL(kern, dim3(unsigned(nwg)), dim3(BS), 0, s, a);
  TL_CHECK_LAUNCH();
  return TL_OK;
}

// 24x24 (8x8) matrix in the Hadamard basis, B = H K H^T / 64
template <typename R>
void to_modes(int ndpn, const double* K, R* B) {
  const int nd = 8 * ndpn;
  auto sign = [](int m, int k) {
    return ((m & 1) * loc_dx(k) + (m >> 1 & 1) * loc_dy(k) + (m >> 2) * loc_dz(k)) & 1 ? -1.0 : 1.0;
  };
  std::vector<R> t(size_t(nd) * nd);
  for (int m = 0; m < 8; ++m)
    for (int c = 0; c < ndpn; ++c)
      for (int j = 0; j < nd; ++j) {
        R s = 0;
        for (int k = 0; k < 8; ++k) s += sign(m, k) * K[size_t(k * ndpn + c) * nd + j];
        t[size_t(m * ndpn + c) * nd + j] = s;
      }
  for (int i = 0; i < nd; ++i)
    for (int m = 0; m < 8; ++m)
      for (int c = 0; c < ndpn; ++c) {
        R s = 0;
        for (int k = 0; k < 8; ++k) s += sign(m, k) * t[size_t(i) * nd + k * ndpn + c];
        B[size_t(i) * nd + m * ndpn + c] = s / 64;
      }
}

// Group values of `n` entries against their pattern; false when an entry
// differs by more than 1e-13 of the largest.
bool match(const double* v, size_t n, const signed char* tab, const int* first, int ng, double* kv) {
  double mx = 0.0;
  for (size_t i = 0; i < n; ++i) mx = std::max(mx, std::fabs(v[i]));
  for (int g = 0; g < ng; ++g) kv[g] = v[first[g]];
  for (size_t i = 0; i < n; ++i) {
    const int p = tab[i];
    const double want = p == 0 ? 0.0 : (p > 0 ? kv[p - 1] : -kv[-p - 1]);
    if (!(std::fabs(want - v[i]) <= 1e-13 * mx)) return false;
  }
  return true;
}

// Group values that fit all entries of K best: the means of its B, formed with
// more digits.  They are those of a product for the caller (tl_apply_K).  A
// group's first entry, out of a K that repeats first entries itself, carries the
// rounding of a few entries of the caller's matrix: error of the FP64 product on
// white noise 2.14e-16, 1.35e-16 with the means; 3.09 and 2.04e-16 with scales
// over nine decades; the general operator 1.35 and 2.36e-16.  A solve keeps the
// first entries: its solution is no nearer to the exact one with the means, but
// 1e-16 in the operator moves a slender design (60x28x12) by up to 4e-6, where
// the design update takes the square root of a sensitivity that is rounding.
void mean_values(int ndpn, const double* K, const signed char* tab, int ng, double* kv) {
  const size_t n2 = size_t(64) * ndpn * ndpn;
  std::vector<long double> B(n2), sum(ng, 0.0L);
  std::vector<int> cnt(ng, 0);
  to_modes(ndpn, K, B.data());
  for (size_t i = 0; i < n2; ++i) {
    const int p = tab[i];
    if (p == 0) continue;
    sum[(p > 0 ? p : -p) - 1] += p > 0 ? B[i] : -B[i];
    ++cnt[(p > 0 ? p : -p) - 1];
  }
  for (int g = 0; g < ng; ++g) kv[g] = double(sum[g] / cnt[g]);
}

}  // namespace

// Whether KE (its pattern's values repeated where it matches one) has the
// reflection-symmetric pattern; fills the group values of the fine operator, those
// of a product for the caller from the matrix `given`, and kt, the entry for
// translations.
bool sym_detect(int ndpn, const double* KE, const double* given, double (&kv)[16],
                double (&kv_product)[16], double& kt) {
  const int nd = 8 * ndpn;
  long double t = 0.0L;  // a sum of cancelling entries: what is left is their rounding
  for (int k = 0; k < 8; ++k)
    for (int l = 0; l < 8; ++l) t += KE[size_t(k * ndpn) * nd + l * ndpn];
  kt = double(t / 64.0L);
  std::vector<double> B(size_t(nd) * nd);
  to_modes(ndpn, KE, B.data());
  if (ndpn == 3) {
    if (!match(B.data(), B.size(), kTabSym_elast, kFirstSym_elast, kGroupsSym_elast, kv)) return false;
    mean_values(ndpn, given, kTabSym_elast, kGroupsSym_elast, kv_product);
    return true;
  }
  if (ndpn == 1) {
    if (!match(B.data(), B.size(), kTabSym_poisson, kFirstSym_poisson, kGroupsSym_poisson, kv))
      return false;
    mean_values(ndpn, given, kTabSym_poisson, kGroupsSym_poisson, kv_product);
    return true;
  }
  return false;
}

// Group values of the level-1 Galerkin operator (G: the 8 child matrices, child
// (cz 2 + cx) 2 + cy).
bool sym_detect_coarse(int ndpn, const double* G, double (&kv)[16]) {
  if (ndpn != 1 && ndpn != 3) return false;
  const int nd = 8 * ndpn;
  const size_t n2 = size_t(nd) * nd;
  std::vector<double> B(8 * n2), K(n2);
  for (int m = 0; m < 8; ++m) {
    for (size_t i = 0; i < n2; ++i) {
      double s = 0.0;
      for (int c = 0; c < 8; ++c) {
        const int cy = c & 1, cx = c >> 1 & 1, cz = c >> 2;
        const bool neg = ((m & 1) * cx + (m >> 1 & 1) * cy + (m >> 2) * cz) & 1;
        s += neg ? -G[size_t(c) * n2 + i] : G[size_t(c) * n2 + i];
      }
      K[i] = s / 8.0;
    }
    to_modes(ndpn, K.data(), B.data() + m * n2);
  }
  if (ndpn == 3)
    return match(B.data(), B.size(), kTabSymC_elast, kFirstSymC_elast, kGroupsSymC_elast, kv);
  return match(B.data(), B.size(), kTabSymC_poisson, kFirstSymC_poisson, kGroupsSymC_poisson, kv);
}

// The tiled operators take a 3D grid whose launch arithmetic and in-plane
// offsets fit 32 bits.
bool sym_fits(const Grid& g, int ndpn) {
  if (g.dim != 3 || (ndpn != 1 && ndpn != 3)) return false;
  const int64_t units = tile_cols(g) * g.nz;
  return units * (kMaxRedBlocks + 1) < (int64_t(1) << 32) &&
         int64_t(g.nx) * g.ny * ndpn < (int64_t(1) << 31);
}

template <int NDPN, typename T>
static int fine_mode(tl_problem* P, const SymArgs<T, T>& a, int mode, bool b64, int src, unsigned* nb) {
  hipStream_t s = P->stream;
  const Grid& g = P->g;
  switch (mode) {
    case KU_STORE:
      if constexpr (std::is_same<T, double>::value)
        return sym_launch<NDPN, T, KU_STORE, T, T, SRC_U, false>(s, g, a, nb);
      break;
    case KU_STORE_DOT:
      if constexpr (std::is_same<T, double>::value)
        if (src == SRC_P) return sym_launch<NDPN, T, KU_STORE_DOT, T, T, SRC_P, false>(s, g, a, nb);
      break;
    case KU_RESID:
      if (src == SRC_SEED) return sym_launch<NDPN, T, KU_RESID, double, T, SRC_SEED, false>(s, g, a, nb);
      if (b64) return sym_launch<NDPN, T, KU_RESID, double, T, SRC_U, false>(s, g, a, nb);
      break;
    case KU_JACOBI:
      if (b64) return sym_launch<NDPN, T, KU_JACOBI, double, T, SRC_U, false>(s, g, a, nb);
      break;
    case KU_JACOBI_DOT:
      if (src == SRC_SEED_CORR)
        return sym_launch<NDPN, T, KU_JACOBI_DOT, double, double, SRC_SEED_CORR, false>(s, g, a, nb);
      if (b64) return sym_launch<NDPN, T, KU_JACOBI_DOT, double, double, SRC_U, false>(s, g, a, nb);
      break;
  }
  set_error("internal: unsupported mode of the tiled operator");
  return TL_EINVAL;
}

template <int NDPN, typename T>
static int fine_call(tl_problem* P, const void* u, void* y, int mode, const void* b, bool b64,
                     const void* dinv, double omega, const void* pin, void* pout,
                     const double* beta, const FoldIn& rho, const FoldIn& rr, double* partials,
                     const int* done, unsigned* nb) {
  SymArgs<T, T> a{};
  a.u = static_cast<const T*>(u);
  a.pin = static_cast<const T*>(pin);
  a.pout = static_cast<T*>(pout);
  a.beta = beta;
  a.rho = rho;
  a.rr = rr;
  a.sp = sizeof(T) == 8 ? reinterpret_cast<const T*>(P->op.sp64.ptr)
                        : reinterpret_cast<const T*>(P->op.sp32.ptr);
  a.mask = P->op.mask.as<uint8_t>();
  a.b = b;
  a.dinv = static_cast<const T*>(dinv);
  a.omega = T(omega);
  a.y = y;
  a.partials = partials;
  a.done = done;
  for (int g = 0; g < 16; ++g) a.kv[g] = T(mode == KU_APPLY ? P->op.symkvp[g] : P->op.symkv[g]);
  if (mode == KU_APPLY) mode = KU_STORE;
  a.kt = T(P->op.symkt);
  int src = pin ? SRC_P : SRC_U;
  if (!u) {  // the V-cycle's first sweep on the fly, with the coarse correction in the last one
    src = mode == KU_RESID ? SRC_SEED : SRC_SEED_CORR;
    a.dinv = reinterpret_cast<const T*>(sizeof(T) == 8 ? P->op.dinv64.ptr : P->op.dinv32.ptr);
    a.omega = T(P->mg.omega);
    if (mode != KU_RESID) {
      const Level& C = P->mg.lv[1];
      a.xc = static_cast<const T*>(C.vx.ptr);
      a.cnx = C.g.nx; a.cny = C.g.ny; a.cnz = C.g.nz;
    }
  }
  return fine_mode<NDPN, T>(P, a, mode, b64, src, nb);
}

int sym_fine_apply(tl_problem* P, const void* u, void* y, int prec, int mode, const void* b,
                   bool b64, const void* dinv, double omega, const void* pin, void* pout,
                   const double* beta, const FoldIn& rho, const FoldIn& rr, double* partials,
                   const int* done, unsigned* nb) {
  auto go = [&](auto ndpn, auto t) {
    return fine_call<decltype(ndpn)::value, decltype(t)>(P, u, y, mode, b, b64, dinv, omega, pin, pout,
                                                         beta, rho, rr, partials, done, nb);
  };
  using N1 = std::integral_constant<int, 1>;
  using N3 = std::integral_constant<int, 3>;
  const bool f64 = prec == TL_PREC_FP64;
  if (P->ndpn == 3) return f64 ? go(N3{}, double{}) : go(N3{}, float{});
  return f64 ? go(N1{}, double{}) : go(N1{}, float{});
}

template <int NDPN, typename T>
static int coarse_call(tl_problem* P, int mode, const T* x, const T* xc, const T* b, T* y,
                       const int* done) {
  const Level& L = P->mg.lv[1];
  SymArgs<T, double> a{};
  a.u = x;
  a.xc = xc;
  a.sp = P->op.sp64.as<double>();
  a.mask = L.mask.as<uint8_t>();
  a.b = b;
  a.dinv = reinterpret_cast<const T*>(sizeof(T) == 8 ? L.dinv64.ptr : L.dinv32.ptr);
  a.omega = T(P->mg.omega);
  a.y = y;
  a.done = done;
  a.fnelx = P->g.nelx;
  a.fnely = P->g.nely;
  for (int g = 0; g < 16; ++g) a.kv[g] = P->mg.symkv[g];
  hipStream_t s = P->stream;
  if (mode == 0) return sym_launch<NDPN, T, KU_RESID, T, T, SRC_U, true>(s, L.g, a, nullptr);
  if (!xc) return sym_launch<NDPN, T, KU_JACOBI, T, T, SRC_U, true>(s, L.g, a, nullptr);
  const Grid& gc = P->mg.lv[2].g;
  a.cnx = gc.nx; a.cny = gc.ny; a.cnz = gc.nz;
  return sym_launch<NDPN, T, KU_JACOBI, T, T, SRC_CORR, true>(s, L.g, a, nullptr);
}

// Level 1: y = b - A x (mode 0) or y = x' + omega D^-1 (b - A x') (mode 1), x' = x
// or, with xc, x plus the coarse correction.
int sym_coarse_apply(tl_problem* P, bool f64, int mode, const void* x, const void* xc,
                     const void* b, void* y, const int* done) {
  auto go = [&](auto ndpn, auto t) {
    using T = decltype(t);
    return coarse_call<decltype(ndpn)::value, T>(P, mode, static_cast<const T*>(x),
                                                 static_cast<const T*>(xc),
                                                 static_cast<const T*>(b), static_cast<T*>(y), done);
  };
  using N1 = std::integral_constant<int, 1>;
  using N3 = std::integral_constant<int, 3>;
  if (P->ndpn == 3) return f64 ? go(N3{}, double{}) : go(N3{}, float{});
  return f64 ? go(N1{}, double{}) : go(N1{}, float{});
}

}  // namespace tl
