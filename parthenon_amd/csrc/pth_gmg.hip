// Geometric-multigrid Poisson solver on the GPU (the reference's poisson_gmg MGSolver,
// src/solvers/mg_solver.hpp:37-521, with the PoissonEquation operator of
// example/poisson_gmg/poisson_equation.hpp:41-205), for uniform N^3 cell-centred grids on
// [0, 1]^3 with FixedFace-0 boundaries (boundary_conditions_generic.hpp:174-255).
//
// Mixed precision by iterative refinement:
//   outer (FP64):  r = b - A u  (with u <- u + e fused in),  ||r|| / ||b|| stop test
//   inner (T):     one V-cycle on A e = r from e = 0: weighted Jacobi pre-smoothing,
//                  residual + average restriction, coarser levels, linear prolongation of the
//                  correction, post-smoothing; the coarsest level only smooths
// T = float is the mixed solver, T = double the plain FP64 solver: same kernels.
//
// Levels are single arrays of n^3 cells (the blocks of the reference's GMG grids are a
// distribution artefact: on one GPU every level fits whole), so no level needs a ghost
// exchange; the Dirichlet ghost (2 * 0 - mirror) is formed on the fly at the domain faces.
// Levels of at most 16 cells per side run inside one workgroup (BottomKernel).
//
// Every kernel is batched: its grid covers a table of entries, one per (problem, level), so
// the same V-cycle stage of several concurrent solves is one launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <vector>

#include "pth_device.hpp"
#include "pth_gmg.hpp"

namespace pth {
namespace {

constexpr int kWG = 256;

// a / d for many a: the products with the rounded reciprocal y = 1 / d, corrected by the
// remainder until the quotient is the correctly rounded one (Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", 1990: one step from a quotient
// that is within one unit in the last place). The first step makes it that for any d. Infinite
// products pass through, so an overflow gives what a division gives.
__device__ __forceinline__ double DivBy(double a, double d, double y) {
  double q = a * y;
  const bool big = __builtin_isinf(q);
  const double q0 = q;
  q = __builtin_fma(__builtin_fma(-q, d, a), y, q);
  q = __builtin_fma(__builtin_fma(-q, d, a), y, q);
  return big ? q0 : q;
}
__device__ __forceinline__ float DivBy(float a, float d, float) { return a / d; }

template <typename T>
__device__ __forceinline__ T Diagonal(T dx) {  // SetDiagonal (poisson_equation.hpp:86-125)
  const T D = T(1), alpha = T(0);
  T d = -(D + D) / (dx * dx) - alpha;
  d -= (D + D) / (dx * dx);
  d -= (D + D) / (dx * dx);
  return d;
}

// Per-level constants. With n a power of two (mul) every factor of the operator, the
// restriction and the prolongation is a power of two, which commutes with rounding: the
// factors are gathered into one product per cell, with the reference's bits. FP32 levels take
// the same form for every n, since there the inner cycle only has to reduce the error.
template <typename T>
struct Lv {
  T dx, rdx, idx2, D, rD, tv;
  bool mul;
};
template <typename T>
__device__ __forceinline__ Lv<T> MakeLv(int n) {
  Lv<T> o;
  o.dx = T(1) / T(n);
  o.mul = sizeof(T) == 4 || (n & (n - 1)) == 0;
  o.idx2 = T(n) * T(n);
  if (o.mul) {
    o.D = T(-6) * o.idx2;
    o.rdx = T(n);
  } else {
    o.D = Diagonal(o.dx);
    o.rdx = T(1) / o.dx;
  }
  o.rD = T(1) / o.D;
  const T vol = o.dx * o.dx * o.dx;
  o.tv = ((vol + vol) + (vol + vol)) + ((vol + vol) + (vol + vol));
  return o;
}

// 7-point operator at one cell in the reference's flux form (D = 1, alpha = 0); neighbours
// across a domain face are the FixedFace-0 ghost -u.
template <typename T>
__device__ __forceinline__ T ApplyA(T u, T xm, T xp, T ym, T yp, T zm, T zp, const Lv<T> &o) {
  if (o.mul)
    return ((((xm - u) + (xp - u)) + ((ym - u) + (yp - u))) + ((zm - u) + (zp - u))) * o.idx2;
  const T dx = o.dx;
  auto div = [&](T a) { return DivBy(a, dx, o.rdx); };
  T out = div(o.rdx * (xm - u) - o.rdx * (u - xp));  // D / dx is the rounded 1 / dx
  out += div(div(ym - u) - div(u - yp));
  out += div(div(zm - u) - div(u - zp));
  return out;
}

struct Cell {
  int i, j, k;
};
__device__ __forceinline__ Cell Decode(int c, int n) {
  Cell q;
  if ((n & (n - 1)) == 0) {  // power of two: shifts and masks (n is uniform per workgroup)
    const int sh = __builtin_ctz(static_cast<unsigned>(n));
    q.i = c & (n - 1);
    q.j = (c >> sh) & (n - 1);
    q.k = c >> (2 * sh);
    return q;
  }
  q.i = c % n;
  const int r = c / n;
  q.j = r % n;
  q.k = r / n;
  return q;
}

// the 6 neighbours of cell c of an n^3 array with the Dirichlet ghost
template <typename T>
struct Nbrs {
  T u, xm, xp, ym, yp, zm, zp;
};
// Those of an array in global memory, every load unconditional: a neighbour outside the
// array reads the cell itself and the ghost value -u replaces it afterwards. (gfx9 counts
// loads and stores on one in-order counter; loads under a per-lane branch make the compiler
// wait for each before the next.)
template <typename T>
__device__ __forceinline__ Nbrs<T> LoadG(const T *x0, int c, const Cell &q, int n) {
  const auto *x = Glob(x0);
  const int s1 = n, s2 = n * n;
  const T u = x[c];
  const T xm = x[q.i > 0 ? c - 1 : c], xp = x[q.i < n - 1 ? c + 1 : c];
  const T ym = x[q.j > 0 ? c - s1 : c], yp = x[q.j < n - 1 ? c + s1 : c];
  const T zm = x[q.k > 0 ? c - s2 : c], zp = x[q.k < n - 1 ? c + s2 : c];
  Nbrs<T> v;
  v.u = u;
  v.xm = q.i > 0 ? xm : -u;
  v.xp = q.i < n - 1 ? xp : -u;
  v.ym = q.j > 0 ? ym : -u;
  v.yp = q.j < n - 1 ? yp : -u;
  v.zm = q.k > 0 ? zm : -u;
  v.zp = q.k < n - 1 ? zp : -u;
  return v;
}

// One weighted Jacobi update: w (b - (A u - D u)) / D + (1 - w) u. In FP32 the off-diagonal part
// is the sum of the neighbours itself (the terms in u cancel), in fused operations: 5 sums and
// 3 products for 24 operations, with fewer roundings.
template <typename T>
__device__ __forceinline__ T JacobiPoint(const Nbrs<T> &v, T b, const Lv<T> &o, T w) {
  if constexpr (sizeof(T) == 4) {
    const T sum = ((v.xm + v.xp) + (v.ym + v.yp)) + (v.zm + v.zp);
    return __builtin_fmaf(w * o.rD, __builtin_fmaf(-o.idx2, sum, b), (T(1) - w) * v.u);
  } else {
    const T off = ApplyA(v.u, v.xm, v.xp, v.ym, v.yp, v.zm, v.zp, o) - o.D * v.u;
    return w * DivBy(b - off, o.D, o.rD) + (T(1) - w) * v.u;
  }
}

// The first Jacobi sweep from x = 0: JacobiPoint with zero neighbours, whose operator part
// vanishes.
template <typename T>
__device__ __forceinline__ T JacobiZero(T b, const Lv<T> &o, T w) {
  if constexpr (sizeof(T) == 4) return w * o.rD * b;
  return w * DivBy(b, o.D, o.rD);
}

// Entry q of a launch. Inline entries are selected with constant indices only, so the kernel
// arguments are read in place (a runtime index into them would copy them to scratch).
template <typename T>
__device__ __forceinline__ GmgEntry<T> At(const GmgArgs<T> &A, int q) {
  if (A.dev) return A.dev[q];
  GmgEntry<T> e = A.e[0];
#pragma unroll
  for (int i = 1; i < kGmgInline; ++i)
    if (i == q) e = A.e[i];
  return e;
}

// The entry whose workgroup range holds this workgroup: entries sorted by wg_begin, the last
// one ends at gridDim.x. The logical workgroup id is XCD-remapped, so each XCD walks
// contiguous rows and planes of a level and finds the y and z neighbours of its rows in its
// own L2.
template <typename T>
__device__ __forceinline__ GmgEntry<T> Find(const GmgArgs<T> &A, int &local) {
  const int w = static_cast<int>(XcdRemap(blockIdx.x, gridDim.x));
  GmgEntry<T> e;
  if (A.dev) {  // binary search over the staged entries
    int lo = 0, hi = A.ne - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) / 2;
      if (A.dev[mid].wg_begin <= w)
        lo = mid;
      else
        hi = mid - 1;
    }
    e = A.dev[lo];
  } else {
    e = A.e[0];
#pragma unroll
    for (int i = 1; i < kGmgInline; ++i)
      if (i < A.ne && A.e[i].wg_begin <= w) e = A.e[i];
  }
  local = w - e.wg_begin;
  return e;
}

// ---- kernels --------------------------------------------------------------------------

// FP64 outer step: u = u_old + e (e may be null), r = b - A u, r stored in T as the inner
// right-hand side, per-workgroup partial sums of r^2. A workgroup marches through nz planes of
// 64 x 13 cells and the ring of one cell around them, 986 columns for 2 x 512 threads; u of a
// column stays in registers for the z neighbours, the plane is left in LDS for the others, so a
// cell's u, e and b are loaded once (1.19 times with the ring). nz depends on the entry's size
// alone, so an entry's sum is the same alone and in a batch. What bounds it is memory: 32 bytes
// a cell in the mixed solver, 40 in FP64. 256^3: 148 -> 117 us and 217 -> 141 against a thread
// per cell with 15 loads, and 1280 partial sums instead of 65536 (their sum 20 -> 4 us).
constexpr int kOuterX = 64, kOuterY = 13, kOuterWG = 512;
template <typename T, bool CORR, bool MUL>
__device__ __forceinline__ double OuterBody(const GmgEntry<T> &e, int local, double *lds) {
  constexpr int PX = kOuterX + 2, PY = kOuterY + 2, NC = PX * PY - 4;
  constexpr int SL = (NC + kOuterWG - 1) / kOuterWG, PAD = PX + 1, LP = PX * PY + 2 * PAD;
  const int n = e.n, s2 = n * n, nz = e.nz;
  const int tx = (n + kOuterX - 1) / kOuterX, ty = (n + kOuterY - 1) / kOuterY;
  const int x0 = local % tx * kOuterX, y0 = local / tx % ty * kOuterY;
  const int k0 = local / (tx * ty) * nz, k1 = min(k0 + nz, n);
  Lv<double> o = MakeLv<double>(n);
  o.mul = MUL;  // known when compiling
  const auto *gu = Glob(static_cast<const double *>(e.u_old));
  const auto *gb = Glob(e.b64);
  const auto *ge = Glob(static_cast<const T *>(e.x));
  auto *gn = Glob(e.u_new);
  auto *gr = Glob(e.b);
  unsigned col[SL];
  int li[SL];
  bool xl[SL], xr[SL], yl[SL], yr[SL], in[SL];
#pragma unroll
  for (int q = 0; q < SL; ++q) {
    const int id = threadIdx.x + q * kOuterWG;
    int m = min(id, NC - 1) + 1;  // the four corners are not needed
    if (m >= PX - 1) ++m;
    if (m >= (PY - 1) * PX) ++m;
    const int lx = m % PX, ly = m / PX, gi = x0 + lx - 1, gj = y0 + ly - 1;
    li[q] = m + PAD;
    in[q] = id < NC && lx >= 1 && lx < PX - 1 && ly >= 1 && ly < PY - 1 && gi < n && gj < n;
    const int i = min(max(gi, 0), n - 1), j = min(max(gj, 0), n - 1);
    xl[q] = i > 0;
    xr[q] = i < n - 1;
    yl[q] = j > 0;
    yr[q] = j < n - 1;
    col[q] = static_cast<unsigned>(j * n + i);
  }
  double un[SL], bn[SL], b[SL], a[SL], c[SL], rr = 0.0;
  T en[SL];
  auto load = [&](int p, int q) {
    const std::int64_t at = static_cast<std::int64_t>(min(max(p, 0), n - 1)) * s2;
    un[q] = (gu + at)[col[q]];
    if (CORR) en[q] = (ge + at)[col[q]];
    bn[q] = (gb + at)[col[q]];
  };
#pragma unroll
  for (int q = 0; q < SL; ++q) {
    load(k0 - 1, q);
    a[q] = c[q] = b[q] = 0.0;
  }
  for (int p = k0 - 1; p <= k1; ++p) {
    double v[SL], bp[SL];
#pragma unroll
    for (int q = 0; q < SL; ++q) {
      v[q] = CORR ? un[q] + static_cast<double>(en[q]) : un[q];
      bp[q] = bn[q];
    }
    if (p < k1) {
#pragma unroll
      for (int q = 0; q < SL; ++q) load(p + 1, q);
    }
#pragma unroll
    for (int q = 0; q < SL; ++q) lds[(p & 1) * LP + li[q]] = v[q];
    if (CORR && p >= k0 && p < k1) {
      auto *out = gn + static_cast<std::int64_t>(p) * s2;
#pragma unroll
      for (int q = 0; q < SL; ++q)
        if (in[q]) out[col[q]] = v[q];
    }
    const int k = p - 1;
    if (k >= k0) {
      const double *L = lds + (k & 1) * LP;
      auto *out = gr + static_cast<std::int64_t>(k) * s2;
#pragma unroll
      for (int q = 0; q < SL; ++q) {
        const double u = c[q];
        const double xm = L[li[q] - 1], xp = L[li[q] + 1], ym = L[li[q] - PX], yp = L[li[q] + PX];
        const double r = b[q] - ApplyA(u, xl[q] ? xm : -u, xr[q] ? xp : -u, yl[q] ? ym : -u,
                                       yr[q] ? yp : -u, k > 0 ? a[q] : -u,
                                       k < n - 1 ? v[q] : -u, o);
        if (in[q]) {
          out[col[q]] = static_cast<T>(r);
          rr += r * r;
        }
      }
    }
#pragma unroll
    for (int q = 0; q < SL; ++q) {
      a[q] = c[q];
      c[q] = v[q];
      b[q] = bp[q];
    }
    __syncthreads();
  }
  return rr;
}

template <typename T>
__global__ void __launch_bounds__(kOuterWG) OuterKernel(const GmgArgs<T> A) {
  constexpr int PX = kOuterX + 2, PY = kOuterY + 2;
  __shared__ double lds[2 * (PX * PY + 2 * (PX + 1))];
  __shared__ double wsum[kOuterWG / 64];
  int local;
  const GmgEntry<T> e = Find(A, local);
  const bool mul = (e.n & (e.n - 1)) == 0;
  double rr = e.x ? (mul ? OuterBody<T, true, true>(e, local, lds)
                         : OuterBody<T, true, false>(e, local, lds))
                  : (mul ? OuterBody<T, false, true>(e, local, lds)
                         : OuterBody<T, false, false>(e, local, lds));
  for (int off = 32; off > 0; off >>= 1) rr += __shfl_xor(rr, off, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = rr;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0.0;
    for (int w = 0; w < kOuterWG / 64; ++w) s += wsum[w];
    e.partial[local] = s;
  }
}

// per-entry sum of the partials of OuterKernel (or of the rhs norm): one workgroup of kNormWG
// threads per entry, each thread adding four interleaved streams of partials into separate
// sums (independent loads in flight), then the workgroup tree. The order is fixed, so an
// entry's norm is the same alone and in a batch. out is pinned host memory: the value that the
// host waits for takes no copy after the kernel (a V-cycle and step of 64^3 in FP64 81.1 -> 78.6 us).
constexpr int kNormWG = 1024;
template <typename T>
__global__ void __launch_bounds__(kNormWG)
    NormKernel(const GmgArgs<T> A, double *__restrict__ out) {
  __shared__ double wsum[kNormWG / 64];
  const GmgEntry<T> e = At(A, blockIdx.x);
  const int np = e.np;
  const double *pa = e.partial;
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  for (int p = threadIdx.x; p < np; p += 4 * kNormWG) {
    s0 += pa[p];
    if (p + kNormWG < np) s1 += pa[p + kNormWG];
    if (p + 2 * kNormWG < np) s2 += pa[p + 2 * kNormWG];
    if (p + 3 * kNormWG < np) s3 += pa[p + 3 * kNormWG];
  }
  double s = (s0 + s1) + (s2 + s3);
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kNormWG / 64; ++w) t += wsum[w];
    out[blockIdx.x] = t;
  }
}

// partial sums of b^2 (the stop test's denominator), kRhsCells cells per workgroup
constexpr int kRhsCells = 16 * kWG;
template <typename T>
__global__ void __launch_bounds__(kWG) RhsNormKernel(const GmgArgs<T> A) {
  __shared__ double wsum[kWG / 64];
  int local;
  const GmgEntry<T> e = Find(A, local);
  const int cells = e.n * e.n * e.n;
  double s = 0.0;
#pragma unroll
  for (int q = 0; q < kRhsCells / kWG; ++q) {
    const std::int64_t c =
        static_cast<std::int64_t>(local) * kRhsCells + q * kWG + threadIdx.x;
    const double v = Glob(e.b64)[c < cells ? c : cells - 1];
    if (c < cells) s += v * v;
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kWG / 64; ++w) t += wsum[w];
    e.partial[local] = t;
  }
}

// Pre-smoothing from x = 0: one sweep (PRE2 = false) or two sweeps fused, the first sweep's
// values at the 7 points being formed from b where they are needed (the same operations as
// two separate sweeps, so the same bits).
template <typename T, bool PRE2>
__global__ void __launch_bounds__(kWG)
    PreZeroKernel(const GmgArgs<T> A, T w) {
  int local;
  const GmgEntry<T> e = Find(A, local);
  const int n = e.n, c = local * kWG + threadIdx.x;
  if (c >= n * n * n) return;
  const Cell q = Decode(c, n);
  const Lv<T> o = MakeLv<T>(n);
  const T *b = e.b;
  if (!PRE2) {
    Glob(e.x)[c] = JacobiZero(static_cast<T>(Glob(b)[c]), o, w);
    return;
  }
  const Nbrs<T> bb = LoadG(b, c, q, n);
  Nbrs<T> x1;
  x1.u = JacobiZero(bb.u, o, w);
  x1.xm = q.i > 0 ? JacobiZero(bb.xm, o, w) : -x1.u;
  x1.xp = q.i < n - 1 ? JacobiZero(bb.xp, o, w) : -x1.u;
  x1.ym = q.j > 0 ? JacobiZero(bb.ym, o, w) : -x1.u;
  x1.yp = q.j < n - 1 ? JacobiZero(bb.yp, o, w) : -x1.u;
  x1.zm = q.k > 0 ? JacobiZero(bb.zm, o, w) : -x1.u;
  x1.zp = q.k < n - 1 ? JacobiZero(bb.zp, o, w) : -x1.u;
  Glob(e.x)[c] = JacobiPoint(x1, bb.u, o, w);
}

template <typename T>
__global__ void __launch_bounds__(kWG) ZeroKernel(const GmgArgs<T> A) {
  int local;
  const GmgEntry<T> e = Find(A, local);
  const int c = local * kWG + threadIdx.x;
  if (c < e.n * e.n * e.n) Glob(e.x)[c] = T(0);
}

// one Jacobi sweep x -> t (the caller swaps x and t)
template <typename T>
__global__ void __launch_bounds__(kWG)
    JacobiKernel(const GmgArgs<T> A, T w) {
  int local;
  const GmgEntry<T> e = Find(A, local);
  const int n = e.n, c = local * kWG + threadIdx.x;
  if (c >= n * n * n) return;
  const Cell q = Decode(c, n);
  const Lv<T> o = MakeLv<T>(n);
  Glob(e.t)[c] = JacobiPoint(LoadG(static_cast<const T *>(e.x), c, q, n), Glob(e.b)[c], o, w);
}

// RestrictAverage of the 8 children's residuals, t[z][y][x]: the reference's sum of volume times
// residual over the total volume.
template <typename T>
__device__ __forceinline__ T Restrict8(const T t[2][2][2], const Lv<T> &o) {
  const T vol = o.mul ? T(1) : o.dx * o.dx * o.dx;
  auto v = [&](int a, int b, int c) { return o.mul ? t[a][b][c] : vol * t[a][b][c]; };
  const T sum = ((v(0, 0, 0) + v(0, 1, 0)) + (v(0, 0, 1) + v(0, 1, 1))) +
                ((v(1, 0, 0) + v(1, 1, 0)) + (v(1, 0, 1) + v(1, 1, 1)));
  return o.mul ? sum * T(0.125) : sum / o.tv;
}

// residual of the 8 children of one coarse cell and their average (RestrictAverage) into the
// coarser level's rhs; one thread per coarse cell
template <typename T>
__global__ void __launch_bounds__(kWG)
    ResidualRestrictKernel(const GmgArgs<T> A) {
  int local;
  const GmgEntry<T> e = Find(A, local);
  const int nc = e.nc, n = e.n, cc = local * kWG + threadIdx.x;
  if (cc >= nc * nc * nc) return;
  const Cell p = Decode(cc, nc);
  const Lv<T> o = MakeLv<T>(n);
  T t[2][2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int bb = 0; bb < 2; ++bb)
#pragma unroll
      for (int c2 = 0; c2 < 2; ++c2) {
        const Cell q = {2 * p.i + c2, 2 * p.j + bb, 2 * p.k + a};
        const int c = (q.k * n + q.j) * n + q.i;
        const Nbrs<T> v = LoadG(static_cast<const T *>(e.x), c, q, n);
        const T r = Glob(e.b)[c] - ApplyA(v.u, v.xm, v.xp, v.ym, v.yp, v.zm, v.zp, o);
        t[a][bb][c2] = r;
      }
  Glob(e.bc)[cc] = Restrict8(t, o);
}

// ProlongateSharedLinear (pr_ops.hpp:166-289) from a coarse cell fc and its neighbours f1, f2,
// f3 (x, y, z) on the fine cell's side, the Dirichlet ghost where there is none. The reference
// adds +/- (gradient x offset), grouped as +/- (x +/- y +/- z) with signs of the child's
// offsets; the signs cancel against those of the one-sided gradients, and for power-of-two
// spacings gradient x offset is a quarter of the difference.
template <typename T>
__device__ __forceinline__ T ProlongPoint(T fc, T f1, T f2, T f3, int oi, int oj, int ok,
                                          const Lv<T> &oc) {
  if (oc.mul) return fc + T(0.25) * (((f1 - fc) + (f2 - fc)) + (f3 - fc));
  const T hc = oc.dx, df = T(0.25) * hc;
  auto grad = [&](T diff) { return DivBy(diff, hc, oc.rdx); };
  const T g1 = grad(oi ? f1 - fc : fc - f1);
  const T g2 = grad(oj ? f2 - fc : fc - f2);
  const T g3 = grad(ok ? f3 - fc : fc - f3);
  const T so = oi ? T(1) : T(-1);
  const T sb = oi == oj ? T(1) : T(-1);
  const T sc = oi == ok ? T(1) : T(-1);
  return fc + so * ((g1 * df + sb * (g2 * df)) + sc * (g3 * df));
}

// The same at fine cell q of an n^3 level. Every load is unconditional: a coarse neighbour
// outside the level reads the cell itself and the ghost value replaces it.
template <typename T, typename P>
__device__ __forceinline__ T ProlongValue(const P *xc, int nc, const Cell &q, const Lv<T> &oc) {
  const Cell p = {q.i >> 1, q.j >> 1, q.k >> 1};
  const int oi = q.i & 1, oj = q.j & 1, ok = q.k & 1;
  const int cc = (p.k * nc + p.j) * nc + p.i;
  const T fc = xc[cc];
  const bool in1 = oi ? p.i < nc - 1 : p.i > 0;
  const bool in2 = oj ? p.j < nc - 1 : p.j > 0;
  const bool in3 = ok ? p.k < nc - 1 : p.k > 0;
  const T l1 = xc[in1 ? cc + (oi ? 1 : -1) : cc];
  const T l2 = xc[in2 ? cc + (oj ? nc : -nc) : cc];
  const T l3 = xc[in3 ? cc + (ok ? nc * nc : -nc * nc) : cc];
  return ProlongPoint(fc, in1 ? l1 : -fc, in2 ? l2 : -fc, in3 ? l3 : -fc, oi, oj, ok, oc);
}

// x += ProlongateSharedLinear(coarse x); one thread per fine cell
template <typename T>
__global__ void __launch_bounds__(kWG) ProlongKernel(const GmgArgs<T> A) {
  int local;
  const GmgEntry<T> e = Find(A, local);
  const int n = e.n, c = local * kWG + threadIdx.x;
  if (c >= n * n * n) return;
  const Cell q = Decode(c, n);
  const T v = ProlongValue<T>(Glob(static_cast<const T *>(e.xc)), e.nc, q, MakeLv<T>(e.nc));
  Glob(e.x)[c] += v;
}

// ---- one pass over a level ------------------------------------------------------------
// Source values, up to two Jacobi sweeps and the restriction of the residual in one kernel:
//   kFromZero: the first sweep from x = 0, formed from b alone (writes x)
//   kFromX:    the level's x (writes t)
//   kFromBelow: x + P xc, the correction of the coarser level (writes t)
// then NS sweeps, then (RES) the residual and its restriction into the coarser right-hand side.
// A workgroup covers TX x TY cells of nz planes and marches in z. With H = NS + RES it holds
// the tile and H cells around it: each thread owns SL columns of that area, keeps two planes of
// every stage of them in registers for the z neighbours and leaves the newest in LDS for the x
// and y neighbours of the next stage, which runs one plane behind; planes of LDS alternate, so
// a plane takes one barrier. A cell's values come from the operations of the one-stage kernels
// in the same order, so the results are the same bits.
// Traffic per cell of a 2 + 2 cycle: 5.25 values (b; x, b and xc) against 17 (FP64) and 13
// (FP32, prolongation inside the first sweep) with a launch per stage, and 2 launches a level
// instead of 5 and 4; what bounds a large level now is the instructions of the overlapped area
// (1.5 times the cells at H = 2), what bounds a small one the march. Per V-cycle, outer step and
// bottom included (2 + 2, FP32 with 2 cycles a step, FP64 with 1): 64^3 103 -> 58 and 131 -> 81 us,
// 128^3 156 -> 98 and 220 -> 145, 256^3 440 -> 262 and 953 -> 533.
enum { kFromZero = 0, kFromX = 1, kFromBelow = 2 };

template <int TX_, int TY_, int WG_>
struct PassTile {
  static constexpr int TX = TX_, TY = TY_, WG = WG_;
};
using PassLarge = PassTile<64, 16, 512>;
using PassSmall = PassTile<32, 8, 512>;

template <typename T, int SRC, int NS, bool RES, typename F>
struct PassShape {
  static constexpr int H = NS + (RES ? 1 : 0), PX = F::TX + 2 * H, PY = F::TY + 2 * H;
  static constexpr int NC = PX * PY - 4;  // no stage reads the four corners
  static constexpr int SL = (NC + F::WG - 1) / F::WG;
  static constexpr int PAD = PX + 1, LP = PX * PY + 2 * PAD;  // one plane, neighbours in range
  static constexpr int LDS = H * 2 * LP + (RES ? 2 * F::TX * F::TY : 0);
};

template <typename T, int SRC, int NS, bool RES, typename F, bool MUL>
__device__ __forceinline__ void PassBody(const GmgEntry<T> &e, int local, int nz, T w, T *lds) {
  using P = PassShape<T, SRC, NS, RES, F>;
  constexpr int H = P::H, PX = P::PX, SL = P::SL, LP = P::LP;
  const int n = e.n, nc = e.nc, s2 = n * n, c2 = nc * nc;
  const int tx = (n + F::TX - 1) / F::TX, ty = (n + F::TY - 1) / F::TY;
  const int x0 = local % tx * F::TX, y0 = local / tx % ty * F::TY, k0 = local / (tx * ty) * nz;
  const int k1 = min(k0 + nz, n);
  Lv<T> o = MakeLv<T>(n), oc = MakeLv<T>(nc);
  o.mul = oc.mul = MUL;  // known when compiling
  const T vol = o.dx * o.dx * o.dx;
  const auto *gx = Glob(static_cast<const T *>(e.x));
  const auto *gb = Glob(static_cast<const T *>(e.b));
  const auto *gc = Glob(static_cast<const T *>(e.xc));
  auto *go = Glob(SRC == kFromZero ? e.x : e.t);

  // this thread's columns (cells past the level's edge: clamped positions whose values nobody
  // reads; threads past the area repeat its last column)
  unsigned col[SL], cc[SL];
  int li[SL], ri[SL], d1[SL], d2[SL];
  bool xl[SL], xr[SL], yl[SL], yr[SL], in[SL], in1[SL], in2[SL], oi[SL], oj[SL];
#pragma unroll
  for (int q = 0; q < SL; ++q) {
    int m = min(static_cast<int>(threadIdx.x) + q * F::WG, P::NC - 1) + 1;
    if (m >= PX - 1) ++m;
    if (m >= (P::PY - 1) * PX) ++m;
    const int lx = m % PX, ly = m / PX;
    li[q] = m + P::PAD;
    ri[q] = (ly - H) * F::TX + (lx - H);
    const int gi = x0 + lx - H, gj = y0 + ly - H;
    in[q] = lx >= H && lx < PX - H && ly >= H && ly < P::PY - H && gi < n && gj < n;
    const int i = min(max(gi, 0), n - 1), j = min(max(gj, 0), n - 1);
    xl[q] = i > 0;
    xr[q] = i < n - 1;
    yl[q] = j > 0;
    yr[q] = j < n - 1;
    col[q] = static_cast<unsigned>(j * n + i);
    if (SRC == kFromBelow) {
      const int pi = i >> 1, pj = j >> 1;
      oi[q] = (i & 1) != 0;
      oj[q] = (j & 1) != 0;
      in1[q] = oi[q] ? pi < nc - 1 : pi > 0;
      in2[q] = oj[q] ? pj < nc - 1 : pj > 0;
      cc[q] = static_cast<unsigned>(pj * nc + pi);
      d1[q] = in1[q] ? (oi[q] ? 1 : -1) : 0;
      d2[q] = in2[q] ? (oj[q] ? nc : -nc) : 0;
    }
  }

  T B[SL][H + 1], bn[SL];           // b of planes p, p - 1, .. and the next one
  T X[SL], xn[SL];                  // source x of plane p and the next one
  T a[NS + 1][SL], c[NS + 1][SL];   // stage s at planes p - s - 2 and p - s - 1
  T lo[SL], mid[SL], hi[SL], l1[SL], l2[SL], hn[SL], l1n[SL], l2n[SL];  // coarse column
  T half = T(0);                    // restriction: sum over the pair's lower plane
  auto plane = [&](int k) { return min(max(k, 0), n - 1); };
  const int p0 = k0 - H, p1 = k1 + H;
#pragma unroll
  for (int q = 0; q < SL; ++q) {
    const auto *b = gb + static_cast<std::int64_t>(plane(p0)) * s2;
    B[q][0] = b[col[q]];
#pragma unroll
    for (int h = 1; h <= H; ++h) B[q][h] = T(0);
    if (SRC != kFromZero) X[q] = (gx + static_cast<std::int64_t>(plane(p0)) * s2)[col[q]];
    if (SRC == kFromBelow) {
      const int K = plane(p0) >> 1;
      lo[q] = (gc + static_cast<std::int64_t>(max(K - 1, 0)) * c2)[cc[q]];
      mid[q] = (gc + static_cast<std::int64_t>(K) * c2)[cc[q]];
      hi[q] = (gc + static_cast<std::int64_t>(min(K + 1, nc - 1)) * c2)[cc[q]];
      l1[q] = (gc + static_cast<std::int64_t>(K) * c2)[cc[q] + d1[q]];
      l2[q] = (gc + static_cast<std::int64_t>(K) * c2)[cc[q] + d2[q]];
    }
#pragma unroll
    for (int s = 0; s <= NS; ++s) a[s][q] = c[s][q] = T(0);
  }

  for (int p = p0; p < p1; ++p) {
    const int pn = plane(p + 1);
    const bool nextK = SRC == kFromBelow && (pn >> 1) != (plane(p) >> 1);
    {  // the next plane's loads
      const auto *b = gb + static_cast<std::int64_t>(pn) * s2;
      const auto *x = gx + static_cast<std::int64_t>(pn) * s2;
#pragma unroll
      for (int q = 0; q < SL; ++q) {
        bn[q] = b[col[q]];
        if (SRC != kFromZero) xn[q] = x[col[q]];
      }
      if (nextK) {
        const int K = pn >> 1;
        const auto *m = gc + static_cast<std::int64_t>(K) * c2;
        const auto *h = gc + static_cast<std::int64_t>(min(K + 1, nc - 1)) * c2;
#pragma unroll
        for (int q = 0; q < SL; ++q) {
          hn[q] = h[cc[q]];
          l1n[q] = m[cc[q] + d1[q]];
          l2n[q] = m[cc[q] + d2[q]];
        }
      }
    }
    if (RES && p - H - 1 >= k0) {  // restriction of the plane before
      const int r = p - H - 1;
      if (threadIdx.x < F::TX / 2 * (F::TY / 2)) {
        const int ci = threadIdx.x % (F::TX / 2), cj = threadIdx.x / (F::TX / 2);
        const T *R = lds + H * 2 * LP + (r & 1) * F::TX * F::TY + 2 * cj * F::TX + 2 * ci;
        const T sum = (R[0] + R[F::TX]) + (R[1] + R[F::TX + 1]);
        if (r & 1) {
          const T all = half + sum;
          const int gi = x0 / 2 + ci, gj = y0 / 2 + cj;
          if (gi < nc && gj < nc)
            Glob(e.bc)[(r / 2 * nc + gj) * nc + gi] = MUL ? all * T(0.125) : all / o.tv;
        }
        half = sum;
      }
    }
    T v[SL];  // the newest values of the stage before
#pragma unroll
    for (int q = 0; q < SL; ++q) {
      if (SRC == kFromZero)
        v[q] = JacobiZero(B[q][0], o, w);
      else if (SRC == kFromX)
        v[q] = X[q];
      else {  // ProlongValue at plane p
        const int k = plane(p), ok = k & 1, K = k >> 1;
        const T fc = mid[q];
        const T f3 = ok ? (K < nc - 1 ? hi[q] : -fc) : (K > 0 ? lo[q] : -fc);
        v[q] = X[q] + ProlongPoint(fc, in1[q] ? l1[q] : -fc, in2[q] ? l2[q] : -fc, f3, oi[q],
                                   oj[q], ok, oc);
      }
      if (H > 0) lds[(p & 1) * LP + li[q]] = v[q];
    }
    if (nextK) {
#pragma unroll
      for (int q = 0; q < SL; ++q) {
        lo[q] = mid[q];
        mid[q] = hi[q];
        hi[q] = hn[q];
        l1[q] = l1n[q];
        l2[q] = l2n[q];
      }
    }
#pragma unroll
    for (int s = 0; s < H; ++s) {  // stage s + 1 at plane k = p - s - 1
      const int k = p - s - 1;
      const T *L = lds + (2 * s + (k & 1)) * LP;
      T *M = lds + (2 * (s + 1) + (k & 1)) * LP;
#pragma unroll
      for (int q = 0; q < SL; ++q) {
        Nbrs<T> u;
        u.u = c[s][q];
        const T xm = L[li[q] - 1], xp = L[li[q] + 1], ym = L[li[q] - PX], yp = L[li[q] + PX];
        u.xm = xl[q] ? xm : -u.u;
        u.xp = xr[q] ? xp : -u.u;
        u.ym = yl[q] ? ym : -u.u;
        u.yp = yr[q] ? yp : -u.u;
        u.zm = k > 0 ? a[s][q] : -u.u;
        u.zp = k < n - 1 ? v[q] : -u.u;
        a[s][q] = c[s][q];
        c[s][q] = v[q];
        if (s < NS) {
          v[q] = JacobiPoint(u, B[q][s + 1], o, w);
          if (s + 1 < H) M[li[q]] = v[q];
        } else {
          const T r = B[q][s + 1] - ApplyA(u.u, u.xm, u.xp, u.ym, u.yp, u.zm, u.zp, o);
          if (in[q]) lds[H * 2 * LP + (k & 1) * F::TX * F::TY + ri[q]] = MUL ? r : vol * r;
        }
      }
      if (s + 1 == NS && k >= k0 && k < k1) {
        auto *out = go + static_cast<std::int64_t>(k) * s2;
#pragma unroll
        for (int q = 0; q < SL; ++q)
          if (in[q]) out[col[q]] = v[q];
      }
    }
#pragma unroll
    for (int q = 0; q < SL; ++q) {
#pragma unroll
      for (int h = H; h > 0; --h) B[q][h] = B[q][h - 1];
      B[q][0] = bn[q];
      if (SRC != kFromZero) X[q] = xn[q];
    }
    __syncthreads();
  }
  if (RES) {  // the last plane
    const int r = k1 - 1;
    if (threadIdx.x < F::TX / 2 * (F::TY / 2)) {
      const int ci = threadIdx.x % (F::TX / 2), cj = threadIdx.x / (F::TX / 2);
      const T *R = lds + H * 2 * LP + (r & 1) * F::TX * F::TY + 2 * cj * F::TX + 2 * ci;
      const T all = half + ((R[0] + R[F::TX]) + (R[1] + R[F::TX + 1]));
      const int gi = x0 / 2 + ci, gj = y0 / 2 + cj;
      if (gi < nc && gj < nc)
        Glob(e.bc)[(r / 2 * nc + gj) * nc + gi] = MUL ? all * T(0.125) : all / o.tv;
    }
  }
}

// FP32: at most 128 registers, so a CU holds two workgroups and one computes while the other
// waits at its barrier (256^3, prolongation and two sweeps: 89 us with the compiler's 130
// registers, 64 with 124). FP64 needs up to 210 and keeps one.
template <typename T, int SRC, int NS, bool RES, typename F>
__global__ void __launch_bounds__(F::WG, sizeof(T) == 4 ? 4 : 1) PassKernel(const GmgArgs<T> A, int nz, T w) {
  __shared__ T lds[PassShape<T, SRC, NS, RES, F>::LDS];
  int local;
  const GmgEntry<T> e = Find(A, local);
  if (sizeof(T) == 4 || (e.n & (e.n - 1)) == 0)
    PassBody<T, SRC, NS, RES, F, true>(e, local, nz, w, lds);
  else
    PassBody<T, SRC, NS, RES, F, false>(e, local, nz, w, lds);
}

// ---- bottom of the V-cycle in one workgroup (levels of at most NB cells per side) --------
// One workgroup per entry: the V-cycle from this entry's level (rhs e.b, result in e.x) down
// to the coarsest level. What bounds it is latency, a chain of about seven dependent steps a
// level, so a thread keeps the x and b of its cells in registers at every level and LDS only
// carries a level's x (or its residual) to the neighbours: 1024 threads as 256 columns by 4
// groups of planes for levels of 5 to 16 cells per side, and one wavefront, which needs no
// barrier, for those of at most 4. Measured between events 13.7 us from 16^3 in FP32 (38.7 with a
// launch-wide loop over cells and a copy per sweep) and 19.6 from 16^3 in FP64, where 8^3 took
// 27.5; the kernels alone, from a trace, 12.1 and 17.6.
constexpr int kBottomWG = 1024;
// cells of the levels above l (l = 31: of all)
__host__ __device__ constexpr int BottomCells(int NB, int l) {
  int s = 0;
  for (int q = 0; q < l; ++q) s += (NB >> q) * (NB >> q) * (NB >> q);
  return s;
}

template <typename T, int NB, bool MUL>
struct Bottom {
  T *lds;
  T w;
  int pre, post;

  // Level l holds at most M = NB >> l cells per side, in an LDS array of M^3; a thread has SL
  // consecutive planes of one column.
  static constexpr int Side(int l) { return NB >> l; }
  static constexpr int Slots(int l) { return Side(l) > 4 ? Side(l) / 4 : 1; }
  template <int l>
  struct Own {
    static constexpr int M = Side(l), SL = Slots(l), S2 = M * M;
    int n, i, j, k;  // first cell
    int c, xm, xp, ym, yp, zm, zp;  // LDS positions: it, and its column's neighbours (clamped)
    bool in, xl, xr, yl, yr;
    __device__ __forceinline__ explicit Own(int n_) : n(n_) {
      if (M <= 4) {
        const int r = threadIdx.x / n;
        i = threadIdx.x - r * n;
        k = r / n;
        j = r - k * n;
        in = k < n && threadIdx.x < 64;
      } else {
        const int col = threadIdx.x % 256;
        j = col / n;
        i = col - j * n;
        k = __builtin_amdgcn_readfirstlane(threadIdx.x / 256) * SL;
        in = j < n && k < n;
      }
      xl = i > 0;
      xr = i < n - 1;
      yl = j > 0;
      yr = j < n - 1;
      c = (k * M + j) * M + i;
      xm = xl ? c - 1 : c;
      xp = xr ? c + 1 : c;
      ym = yl ? c - M : c;
      yp = yr ? c + M : c;
      zm = k > 0 ? c - S2 : c;
      zp = k + SL < n ? c + SL * S2 : c;
    }
    __device__ __forceinline__ bool has(int q) const { return in && k + q < n; }
    __device__ __forceinline__ int cell(int q) const { return ((k + q) * n + j) * n + i; }
  };
  // order LDS accesses: of the workgroup, or of the one wavefront that works on a small level
  template <int l>
  static __device__ __forceinline__ void Sync() {
    if (Side(l) > 4) {
      __syncthreads();
    } else {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }

  template <int l>
  __device__ __forceinline__ void Put(T *X, const T (&u)[Slots(l)], const Own<l> &o) const {
#pragma unroll
    for (int q = 0; q < Slots(l); ++q)
      if (o.has(q)) X[o.c + q * o.S2] = u[q];
    Sync<l>();
  }
  // fn(slot, neighbours) for this thread's cells, X holding the level's values and u this
  // thread's. The loads are unconditional, at positions clamped into the level, so they are in
  // flight together; a slot without a cell gets values that nobody uses.
  template <int l, typename Fn>
  __device__ __forceinline__ void Each(const T *X, const T (&u)[Slots(l)], const Own<l> &o,
                                       Fn fn) const {
    constexpr int SL = Slots(l);
    Nbrs<T> v[SL];
    if (o.in) {
      const T zm = X[o.zm], zp = X[o.zp];
#pragma unroll
      for (int q = 0; q < SL; ++q) {
        const T xm = X[o.xm + q * o.S2], xp = X[o.xp + q * o.S2];
        const T ym = X[o.ym + q * o.S2], yp = X[o.yp + q * o.S2];
        v[q] = {u[q],
                o.xl ? xm : -u[q],
                o.xr ? xp : -u[q],
                o.yl ? ym : -u[q],
                o.yr ? yp : -u[q],
                o.k + q > 0 ? (q > 0 ? u[q > 0 ? q - 1 : 0] : zm) : -u[q],
                o.k + q < o.n - 1 ? (q + 1 < SL ? u[q + 1 < SL ? q + 1 : 0] : zp) : -u[q]};
      }
    }
    Sync<l>();  // everybody has read: X may be written again
    if (o.in) {
#pragma unroll
      for (int q = 0; q < SL; ++q) fn(q, v[q]);
    }
  }

  template <int l>
  __device__ __forceinline__ void Sweeps(T *X, T (&u)[Slots(l)], const T (&b)[Slots(l)],
                                         const Own<l> &o, const Lv<T> &lv, int count) const {
    for (int s = 0; s < count; ++s) {
      Put<l>(X, u, o);
      Each<l>(X, u, o, [&](int q, const Nbrs<T> &v) { u[q] = JacobiPoint(v, b[q], lv, w); });
    }
  }

  // The cycle on level l of n cells per side; b: right-hand side, u: start (from_x) and result.
  template <int l>
  __device__ __forceinline__ void Level(int n, T (&u)[Slots(l)], const T (&b)[Slots(l)],
                                        bool from_x) const {
    constexpr int M = Side(l), SL = Slots(l), S2 = M * M;
    if (M <= 4 && threadIdx.x >= 64) return;
    T *X = lds + BottomCells(NB, l);
    const Own<l> o(n);
    Lv<T> lv = MakeLv<T>(n);
    lv.mul = MUL;  // known when compiling
    if (!from_x) {
#pragma unroll
      for (int q = 0; q < SL; ++q) u[q] = pre > 0 ? JacobiZero(b[q], lv, w) : T(0);
    }
    Sweeps<l>(X, u, b, o, lv, pre - (from_x ? 0 : 1));
    if constexpr (M > 1) {
      if (n % 2 == 0) {
        constexpr int SC = Slots(l + 1), MC = Side(l + 1);
        const int nc = n / 2;
        T r[SL], uc[SC], bc[SC];
        Put<l>(X, u, o);
        Each<l>(X, u, o, [&](int q, const Nbrs<T> &v) {
          r[q] = b[q] - ApplyA(v.u, v.xm, v.xp, v.ym, v.yp, v.zm, v.zp, lv);
        });
        Put<l>(X, r, o);
        const Own<l + 1> oc(nc);
#pragma unroll
        for (int q = 0; q < SC; ++q) uc[q] = bc[q] = T(0);
        if (oc.in) {
#pragma unroll
          for (int q = 0; q < SC; ++q) {
            const T *R = X + (2 * min(oc.k + q, nc - 1) * M + 2 * oc.j) * M + 2 * oc.i;
            T t[2][2][2];
#pragma unroll
            for (int a = 0; a < 8; ++a)
              t[a / 4][a / 2 % 2][a % 2] = R[a / 4 * S2 + a / 2 % 2 * M + a % 2];
            bc[q] = Restrict8(t, lv);
          }
        }
        Level<l + 1>(nc, uc, bc, false);
        // the coarse level's x for everybody
        T *XC = lds + BottomCells(NB, l + 1);
#pragma unroll
        for (int q = 0; q < SC; ++q)
          if (oc.has(q)) XC[oc.c + q * MC * MC] = uc[q];
        Sync<l>();
        Lv<T> lc = MakeLv<T>(nc);
        lc.mul = MUL;
        if (o.in) {  // u += P xc: the coarse column's planes and its x and y neighbours
          const int pi = o.i >> 1, pj = o.j >> 1, oi = o.i & 1, oj = o.j & 1, K = o.k >> 1;
          const bool in1 = oi ? pi < nc - 1 : pi > 0, in2 = oj ? pj < nc - 1 : pj > 0;
          const int c = pj * MC + pi;
          const int c1 = in1 ? (oi ? c + 1 : c - 1) : c, c2 = in2 ? (oj ? c + MC : c - MC) : c;
          constexpr int P = (SL + 1) / 2;
          T f[P + 2], f1[P], f2[P];
#pragma unroll
          for (int p = 0; p < P + 2; ++p) f[p] = XC[min(max(K + p - 1, 0), nc - 1) * MC * MC + c];
#pragma unroll
          for (int p = 0; p < P; ++p) {
            f1[p] = XC[min(K + p, nc - 1) * MC * MC + c1];
            f2[p] = XC[min(K + p, nc - 1) * MC * MC + c2];
          }
#pragma unroll
          for (int q = 0; q < SL; ++q) {
            const int p = q / 2, ok = (o.k + q) & 1;
            const T fc = f[p + 1];
            const T f3 = ok ? (K + p < nc - 1 ? f[p + 2] : -fc) : (K + p > 0 ? f[p] : -fc);
            u[q] += ProlongPoint(fc, in1 ? f1[p] : -fc, in2 ? f2[p] : -fc, f3, oi, oj, ok, lc);
          }
        }
        Sweeps<l>(X, u, b, o, lv, post);
      }
    }
  }
};

template <typename T, int NB, bool MUL>
__device__ __forceinline__ void BottomBody(const GmgEntry<T> &e, T *lds, T w, int pre, int post) {
  using B = Bottom<T, NB, MUL>;
  constexpr int SL = B::Slots(0);
  const bool warm = e.warm != 0;
  const typename B::template Own<0> o(e.n);
  T u[SL], b[SL];
#pragma unroll
  for (int q = 0; q < SL; ++q) {
    u[q] = b[q] = T(0);
    if (!o.has(q)) continue;
    b[q] = Glob(e.b)[o.cell(q)];
    if (warm) u[q] = Glob(e.x)[o.cell(q)];
  }
  const B body = {lds, w, pre, post};
  body.template Level<0>(e.n, u, b, warm);
#pragma unroll
  for (int q = 0; q < SL; ++q)
    if (o.has(q)) Glob(e.x)[o.cell(q)] = u[q];
}

template <typename T, int NB>
__global__ void __launch_bounds__(kBottomWG)
    BottomKernel(const GmgArgs<T> A, T w, int pre, int post) {
  __shared__ T lds[BottomCells(NB, 31)];
  const GmgEntry<T> e = At(A, blockIdx.x);
  if (sizeof(T) == 4 || (e.n & (e.n - 1)) == 0)
    BottomBody<T, NB, true>(e, lds, w, pre, post);
  else
    BottomBody<T, NB, false>(e, lds, w, pre, post);
}

// Right-hand side: 16 seeded Gaussian blobs at cell centres (FP64)
struct BlobParams {
  double v[80];  // per blob: cx, cy, cz, width, sign
};
__global__ void __launch_bounds__(kWG) BlobKernel(double *__restrict__ b, int n, BlobParams P) {
  const double *blob = P.v;
  const int c = blockIdx.x * kWG + threadIdx.x;
  if (c >= n * n * n) return;
  const Cell q = Decode(c, n);
  const double h = 1.0 / n;
  const double x = (q.i + 0.5) * h, y = (q.j + 0.5) * h, z = (q.k + 0.5) * h;
  double v = 0.0;
  for (int m = 0; m < 16; ++m) {
    const double *p = blob + 5 * m;
    const double dx = x - p[0], dy = y - p[1], dz = z - p[2];
    v += p[4] * exp(-(dx * dx + dy * dy + dz * dz) / (p[3] * p[3]));
  }
  b[c] = v;
}

__global__ void __launch_bounds__(kWG) FillKernel(double *__restrict__ a, std::int64_t n) {
  const std::int64_t c = static_cast<std::int64_t>(blockIdx.x) * kWG + threadIdx.x;
  if (c < n) a[c] = 0.0;
}

// Planes a workgroup of a pass marches through, for `planes` tile planes in the launch: as many
// workgroups as fill the chip twice (each plane past the tile's own costs 2 H planes of
// overlap), even, for the restriction, and from 2, where a short march beats the overlap: 32^3
// V-cycles in FP64 take 83 / 91 / 103 / 131 us with at least 2 / 4 / 8 / 16 planes, 128^3 in FP32
// 147 / 149 / 151 / 186. At most `most` planes: 32 for the passes, where 256^3 in FP32 takes
// 270 us with 32 and 272 with 16 (192^3 158 and 180).
int PassPlanes(std::int64_t planes, int most) {
  const int nz = static_cast<int>(std::min<std::int64_t>((planes + 511) / 512, most));
  return std::max((nz + 1) / 2 * 2, 2);
}

// Planes a workgroup of the outer step marches through, at most 16: it is bound by memory and
// its registers let three workgroups share a CU, which the 1280 of 256^3 fill (64 / 32 / 24 / 16 / 8
// planes: 152 / 131 / 128 / 117 / 120 us). The workgroups are never more than the partial sums a
// problem has room for.
int OuterTiles(int n) {
  return ((n + kOuterX - 1) / kOuterX) * ((n + kOuterY - 1) / kOuterY);
}
int OuterPlanes(int n) {
  const std::int64_t room = (static_cast<std::int64_t>(n) * n * n + kWG - 1) / kWG;
  int nz = PassPlanes(static_cast<std::int64_t>(OuterTiles(n)) * n, 16);
  while (static_cast<std::int64_t>(OuterTiles(n)) * ((n + nz - 1) / nz) > room) nz += 2;
  return nz;
}

constexpr std::int64_t kPassLarge = std::int64_t(1) << 22;

int Blocks(std::int64_t cells) { return static_cast<int>((cells + kWG - 1) / kWG); }


}  // namespace

// ---- host side -------------------------------------------------------------------------

void GmgBlobs(std::uint64_t seed, double out[80]) {
  std::uint64_t st = seed;
  auto next = [&]() {
    std::uint64_t z = (st += 0x9E3779B97F4A7C15ULL);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return static_cast<double>((z ^ (z >> 31)) >> 11) * 0x1.0p-53;
  };
  for (int m = 0; m < 16; ++m) {
    for (int d = 0; d < 3; ++d) out[5 * m + d] = 0.1 + 0.8 * next();
    out[5 * m + 3] = 0.02 + 0.06 * next();
    out[5 * m + 4] = next() < 0.5 ? -1.0 : 1.0;
  }
}

std::vector<int> GmgLevelSizes(int N) {
  std::vector<int> s;
  for (int n = N;; n /= 2) {
    s.push_back(n);
    if (n % 2 != 0 || n == 1) break;
  }
  return s;
}

template <typename T>
std::int64_t GmgProblem<T>::Bytes(int N) {
  std::int64_t b = 0;
  for (int n : GmgLevelSizes(N)) b += 3 * static_cast<std::int64_t>(n) * n * n * sizeof(T);
  const std::int64_t c = static_cast<std::int64_t>(N) * N * N;
  return b + 3 * c * 8 + ((c + kWG - 1) / kWG) * 8;
}

template <typename T>
pth_status GmgProblem<T>::Allocate(int N_) {
  constexpr int bottom = GmgBottom<T>::kN;
  N = N_;
  sizes = GmgLevelSizes(N);
  nbottom = 0;
  while (nbottom < static_cast<int>(sizes.size()) && sizes[nbottom] > bottom) ++nbottom;
  if (sizes.back() > GmgBottom<T>::kCoarsest) {
    SetError("GMG: the coarsest level is larger than the in-LDS bottom solver");
    return PTH_FAIL;
  }
  const std::int64_t c = static_cast<std::int64_t>(N) * N * N;
  if (c >= (std::int64_t(1) << 31)) {
    SetError("GMG: grid too large");
    return PTH_FAIL;
  }
  std::int64_t total = 0;
  for (int n : sizes) total += 3 * static_cast<std::int64_t>(n) * n * n;
  PTH_HIP(hipMalloc(&levels, sizeof(T) * total));
  PTH_HIP(hipMemset(levels, 0, sizeof(T) * total));
  PTH_HIP(hipMalloc(&u[0], sizeof(double) * c));
  PTH_HIP(hipMalloc(&u[1], sizeof(double) * c));
  PTH_HIP(hipMalloc(&b64, sizeof(double) * c));
  PTH_HIP(hipMalloc(&partial, sizeof(double) * ((c + kWG - 1) / kWG)));
  PTH_HIP(hipMemset(u[0], 0, sizeof(double) * c));
  PTH_HIP(hipMemset(u[1], 0, sizeof(double) * c));
  PTH_HIP(hipMemset(b64, 0, sizeof(double) * c));
  PTH_HIP(hipDeviceSynchronize());  // the clears above are ordered before any stream's work
  lv.clear();
  std::int64_t o = 0;
  for (int n : sizes) {
    const std::int64_t s = static_cast<std::int64_t>(n) * n * n;
    lv.push_back({levels + o, levels + o + s, levels + o + 2 * s});
    o += 3 * s;
  }
  cur = 0;
  return PTH_COMPLETE;
}

template <typename T>
void GmgProblem<T>::Free() {
  if (levels) PTH_DROP(hipFree(levels));
  for (double *&p : u)
    if (p) PTH_DROP(hipFree(p));
  if (b64) PTH_DROP(hipFree(b64));
  if (partial) PTH_DROP(hipFree(partial));
  levels = nullptr;
  u[0] = u[1] = b64 = partial = nullptr;
}

template <typename T>
GmgEntry<T> GmgProblem<T>::Entry(int l) const {
  GmgEntry<T> e;
  std::memset(&e, 0, sizeof(e));
  e.x = lv[l].x;
  e.t = lv[l].t;
  e.b = lv[l].b;
  if (l + 1 < static_cast<int>(lv.size())) {
    e.xc = lv[l + 1].x;
    e.bc = lv[l + 1].b;
    e.nc = sizes[l + 1];
  }
  e.n = sizes[l];
  e.u_old = u[cur];
  e.u_new = u[1 - cur];
  e.b64 = b64;
  e.partial = partial;
  return e;
}

template <typename T>
pth_status GmgBatch<T>::Stage(const std::vector<GmgEntry<T>> &es, bool coarse_cells,
                              GmgArgs<T> *args, int *nwg) {
  std::vector<GmgEntry<T>> v = es;
  int wg = 0;
  for (auto &e : v) {
    e.wg_begin = wg;
    const std::int64_t n = coarse_cells ? e.nc : e.n;
    wg += static_cast<int>((n * n * n + kWG - 1) / kWG);
  }
  *nwg = wg;
  return Put(v, args);
}

// The same for a pass: workgroups of tx x ty cells and *nz planes.
template <typename T>
pth_status GmgBatch<T>::StagePass(const std::vector<GmgEntry<T>> &es, int tx, int ty,
                                  GmgArgs<T> *args, int *nwg, int *nz) {
  std::int64_t planes = 0;
  auto tiles = [&](int n) { return ((n + tx - 1) / tx) * ((n + ty - 1) / ty); };
  for (const auto &e : es) planes += static_cast<std::int64_t>(tiles(e.n)) * e.n;
  *nz = PassPlanes(planes, 32);
  std::vector<GmgEntry<T>> v = es;
  int wg = 0;
  for (auto &e : v) {
    e.wg_begin = wg;
    wg += tiles(e.n) * ((e.n + *nz - 1) / *nz);
  }
  *nwg = wg;
  return Put(v, args);
}

// The entries of a launch into its arguments.
template <typename T>
pth_status GmgBatch<T>::Put(const std::vector<GmgEntry<T>> &v, GmgArgs<T> *args) {
  std::memset(args, 0, sizeof(*args));
  args->ne = static_cast<int>(v.size());
  if (static_cast<int>(v.size()) <= kGmgInline) {  // in the kernel arguments
    std::copy(v.begin(), v.end(), args->e);
    return PTH_COMPLETE;
  }
  // larger batches: written to a host staging ring and copied once per stage
  if (static_cast<int>(v.size()) > kStageCap) {
    SetError("GMG: too many batched entries in one launch");
    return PTH_FAIL;
  }
  if (stage_used + static_cast<int>(v.size()) > kStageCap) {
    // the ring is full: the copies queued from it must have run before it is rewritten
    PTH_HIP(hipStreamSynchronize(stream));
    stage_used = 0;
  }
  GmgEntry<T> *h = stage_host + stage_used, *d = stage_dev + stage_used;
  std::copy(v.begin(), v.end(), h);
  PTH_HIP(hipMemcpyAsync(d, h, sizeof(GmgEntry<T>) * v.size(), hipMemcpyHostToDevice, stream));
  stage_used += static_cast<int>(v.size());
  args->dev = d;
  return PTH_COMPLETE;
}

template <typename T>
pth_status GmgBatch<T>::Init(hipStream_t s) {
  stream = s;
  if (!stage_host) {
    PTH_HIP(hipHostMalloc(&stage_host, sizeof(GmgEntry<T>) * kStageCap));
    PTH_HIP(hipMalloc(&stage_dev, sizeof(GmgEntry<T>) * kStageCap));
    PTH_HIP(hipHostMalloc(&norms, sizeof(double) * kMaxProblems));
  }
  return PTH_COMPLETE;
}

template <typename T>
void GmgBatch<T>::Free() {
  if (stage_host) PTH_DROP(hipHostFree(stage_host));
  if (stage_dev) PTH_DROP(hipFree(stage_dev));
  if (norms) PTH_DROP(hipHostFree(norms));
  stage_host = nullptr;
  stage_dev = nullptr;
  norms = nullptr;
}

template <typename T>
pth_status GmgBatch<T>::RhsNorms(const std::vector<GmgProblem<T> *> &ps, double *out) {
  std::vector<GmgEntry<T>> es;
  for (auto *p : ps) es.push_back(p->Entry(0));
  int nwg = 0;
  for (auto &e : es) {
    e.wg_begin = nwg;
    e.np = static_cast<int>((static_cast<std::int64_t>(e.n) * e.n * e.n + kRhsCells - 1) /
                            kRhsCells);
    nwg += e.np;
  }
  GmgArgs<T> a;
  if (Put(es, &a) != PTH_COMPLETE) return PTH_FAIL;
  const int ne = a.ne;
  PTH_LAUNCH(RhsNormKernel<T>, dim3(nwg), dim3(kWG), 0, stream, a);
  PTH_LAUNCH(NormKernel<T>, dim3(ne), dim3(kNormWG), 0, stream, a, norms);
  PTH_HIP(hipStreamSynchronize(stream));
  stage_used = 0;  // every queued copy has run
  for (int q = 0; q < ne; ++q) out[q] = std::sqrt(norms[q]);
  return PTH_COMPLETE;
}

// Outer FP64 step for every problem in ps: apply the pending correction (when correct[q]),
// form r = b - A u as the inner right-hand side, and return ||r|| in out[] (synchronizes).
template <typename T>
pth_status GmgBatch<T>::Residual(const std::vector<GmgProblem<T> *> &ps,
                                 const std::vector<char> &correct, double *out) {
  std::vector<GmgEntry<T>> es;
  int nwg = 0;
  for (size_t q = 0; q < ps.size(); ++q) {
    GmgEntry<T> e = ps[q]->Entry(0);
    if (!correct[q]) e.x = nullptr;
    e.nz = OuterPlanes(e.n);
    e.np = OuterTiles(e.n) * ((e.n + e.nz - 1) / e.nz);
    e.wg_begin = nwg;
    nwg += e.np;
    es.push_back(e);
  }
  GmgArgs<T> a;
  if (Put(es, &a) != PTH_COMPLETE) return PTH_FAIL;
  const int ne = a.ne;
  {
    ProfScope prof("gmg_outer", stream);
    PTH_LAUNCH(OuterKernel<T>, dim3(nwg), dim3(kOuterWG), 0, stream, a);
  }
  PTH_LAUNCH(NormKernel<T>, dim3(ne), dim3(kNormWG), 0, stream, a, norms);
  PTH_HIP(hipStreamSynchronize(stream));
  stage_used = 0;  // every queued copy has run
  for (size_t q = 0; q < ps.size(); ++q) {
    if (correct[q]) ps[q]->cur = 1 - ps[q]->cur;
    out[q] = std::sqrt(norms[q]);
  }
  return PTH_COMPLETE;
}

// One V-cycle on A e = r from e = 0 for every problem in ps, level by level: the same stage of
// every problem is one launch. The level arrays' x / t roles follow the Jacobi ping-pong.
template <typename T>
pth_status GmgBatch<T>::Cycle(const std::vector<GmgProblem<T> *> &ps, double omega, int pre,
                              int post, bool warm) {
  const T w = static_cast<T>(omega);
  int L = 0;
  for (auto *p : ps) L = std::max(L, p->nbottom);
  auto entries = [&](int l) {
    std::vector<GmgEntry<T>> es;
    for (auto *p : ps)
      if (l < p->nbottom) es.push_back(p->Entry(l));
    return es;
  };
  auto swap = [&](int l) {  // a sweep from x left its result in t
    for (auto *p : ps)
      if (l < p->nbottom) std::swap(p->lv[l].x, p->lv[l].t);
  };
  // a one-stage kernel, one thread per cell of the level (or of the next coarser one)
  auto cells = [&](int l, bool coarse, const char *name, auto kernel, auto... arg) -> pth_status {
    GmgArgs<T> a;
    int nwg;
    if (Stage(entries(l), coarse, &a, &nwg) != PTH_COMPLETE) return PTH_FAIL;
    ProfScope prof(name, stream);
    PTH_LAUNCH(kernel, dim3(nwg), dim3(kWG), 0, stream, a, arg...);
    return PTH_COMPLETE;
  };
  auto pass = [&](int l, const char *name, auto src, auto ns, auto res) -> pth_status {
    const std::vector<GmgEntry<T>> es = entries(l);
    std::int64_t total = 0;
    for (const auto &e : es) total += static_cast<std::int64_t>(e.n) * e.n * e.n;
    GmgArgs<T> a;
    int nwg, nz;
    auto run = [&](auto f) -> pth_status {
      using F = decltype(f);
      if (StagePass(es, F::TX, F::TY, &a, &nwg, &nz) != PTH_COMPLETE) return PTH_FAIL;
      ProfScope prof(name, stream);
      PTH_LAUNCH((PassKernel<T, decltype(src)::value, decltype(ns)::value,
                             decltype(res)::value, F>),
                 dim3(nwg), dim3(F::WG), 0, stream, a, nz, w);
      return PTH_COMPLETE;
    };
    // below kPassLarge cells the smaller tile: more workgroups and shorter planes against less
    // overlap (V-cycles with small / large tiles: 64^3 FP32 95 / 103 us, 128^3 FP64 196 / 208,
    // 192^3 FP32 267 / 254, 192^3 FP64 683 / 590)
    if ((total < kPassLarge ? run(PassSmall()) : run(PassLarge())) != PTH_COMPLETE)
      return PTH_FAIL;
    if (decltype(src)::value != kFromZero) swap(l);
    return PTH_COMPLETE;
  };
  using std::integral_constant;
  integral_constant<int, kFromZero> zero;
  integral_constant<int, kFromX> from_x;
  integral_constant<int, kFromBelow> below;
  integral_constant<int, 1> one;
  integral_constant<int, 2> two;
  std::true_type res;
  std::false_type nores;
  const bool fused = jacobi_columns > 0;
  auto jacobi = [&](int l) -> pth_status {
    if (cells(l, false, l == 0 ? "gmg_jacobi_l0" : "gmg_jacobi", JacobiKernel<T>, w) !=
        PTH_COMPLETE)
      return PTH_FAIL;
    swap(l);
    return PTH_COMPLETE;
  };
  auto sweeps = [&](int l, int k) -> pth_status {
    const char *name = l == 0 ? "gmg_jacobi_l0" : "gmg_jacobi";
    while (k > 0) {
      const int m = fused && k >= 2 ? 2 : 1;
      if ((m == 2   ? pass(l, name, from_x, two, nores)
           : fused  ? pass(l, name, from_x, one, nores)
                    : jacobi(l)) != PTH_COMPLETE)
        return PTH_FAIL;
      k -= m;
    }
    return PTH_COMPLETE;
  };
  for (int l = 0; l < L; ++l) {
    const bool top = warm && l == 0;
    const char *pname = l == 0 ? "gmg_pre_l0" : "gmg_pre";
    const char *rname = l == 0 ? "gmg_restrict_l0" : "gmg_restrict";
    const char *fname = l == 0 ? "gmg_pre_restrict_l0" : "gmg_pre_restrict";
    int k = pre;  // sweeps still to do
    if (fused && !top && pre == 2) {
      if (pass(l, fname, zero, one, res) != PTH_COMPLETE) return PTH_FAIL;
      continue;
    }
    if (!top) {
      if (pre == 0) {
        if (cells(l, false, pname, ZeroKernel<T>) != PTH_COMPLETE) return PTH_FAIL;
      } else if (pre >= 2 && !(fused && pre == 3)) {
        if (cells(l, false, pname, PreZeroKernel<T, true>, w) != PTH_COMPLETE) return PTH_FAIL;
        k -= 2;
      } else {
        if (cells(l, false, pname, PreZeroKernel<T, false>, w) != PTH_COMPLETE) return PTH_FAIL;
        k -= 1;
      }
    }
    if (fused && k > 0) {
      const int last = sizeof(T) == 4 && k % 2 == 0 ? 2 : 1;
      if (sweeps(l, k - last) != PTH_COMPLETE) return PTH_FAIL;
      if constexpr (sizeof(T) == 4) {
        if (last == 2) {
          if (pass(l, fname, from_x, two, res) != PTH_COMPLETE) return PTH_FAIL;
          continue;
        }
      }
      if (pass(l, fname, from_x, one, res) != PTH_COMPLETE) return PTH_FAIL;
      continue;
    }
    if (sweeps(l, k) != PTH_COMPLETE) return PTH_FAIL;
    if (cells(l, true, rname, ResidualRestrictKernel<T>) != PTH_COMPLETE) return PTH_FAIL;
  }
  {
    std::vector<GmgEntry<T>> es;
    for (auto *p : ps) {
      es.push_back(p->Entry(p->nbottom));
      es.back().warm = warm && p->nbottom == 0;
    }
    GmgArgs<T> a;
    int nwg;
    if (Stage(es, false, &a, &nwg) != PTH_COMPLETE) return PTH_FAIL;
    ProfScope prof("gmg_bottom", stream);
    PTH_LAUNCH((BottomKernel<T, GmgBottom<T>::kN>), dim3(a.ne), dim3(kBottomWG), 0,
               stream, a, w, pre, post);
  }
  for (int l = L - 1; l >= 0; --l) {
    const char *name = l == 0 ? "gmg_prolong_jacobi_l0" : "gmg_prolong_jacobi";
    const int in = fused ? std::min(post, 2) : 0;
    if ((in == 2   ? pass(l, name, below, two, nores)
         : in == 1 ? pass(l, name, below, one, nores)
                   : cells(l, false, l == 0 ? "gmg_prolong_l0" : "gmg_prolong",
                           ProlongKernel<T>)) != PTH_COMPLETE)
      return PTH_FAIL;
    if (sweeps(l, post - in) != PTH_COMPLETE) return PTH_FAIL;
  }
  return PTH_COMPLETE;
}

template <typename T>
pth_status GmgBatch<T>::SetBlobs(GmgProblem<T> &p, std::uint64_t seed) {
  BlobParams P;
  GmgBlobs(seed, P.v);
  PTH_LAUNCH(BlobKernel, dim3(Blocks(static_cast<std::int64_t>(p.N) * p.N * p.N)),
             dim3(kWG), 0, stream, p.b64, p.N, P);
  return PTH_COMPLETE;
}

// u = 0 on the finest level (the solve's initial guess)
template <typename T>
pth_status GmgBatch<T>::Reset(GmgProblem<T> &p) {
  const std::int64_t c = static_cast<std::int64_t>(p.N) * p.N * p.N;
  PTH_LAUNCH(FillKernel, dim3(Blocks(c)), dim3(kWG), 0, stream, p.u[0], c);
  p.cur = 0;
  return PTH_COMPLETE;
}

template struct GmgProblem<float>;
template struct GmgProblem<double>;
template struct GmgBatch<float>;
template struct GmgBatch<double>;

}  // namespace pth
