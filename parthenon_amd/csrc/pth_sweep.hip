// Block-sweep form of the Burgers stage for gfx950, FP64: one launch per stage does the
// reconstruction, HLL fluxes, flux divergence, RK update, derived field and CFL minimum
// (benchmarks/burgers/burgers_package.cpp:143-200, 236-401; src/interface/update.cpp:63-84,
// update.hpp:43-90), plus the direct flux-correction send of the same stage.
//
// This file is built with FMA contraction (-ffp-contract=fast), as a CUDA build of the
// reference is by default (--fmad=true): a multiply feeding an add becomes one fused
// instruction, which takes a quarter of the FP64 instructions out of this issue-bound kernel.
// Its results therefore agree with an IEEE CPU evaluation to rounding (about 1e-15 relative
// after several cycles) rather than bit for bit; the task and plane-tiled forms in
// pth_burgers.hip are built without contraction and stay bit-exact. The flux-correction send
// of this form is here too, so the fine fluxes it restricts are the same bits as the ones the
// sweep applies to the fine blocks.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <map>
#include <type_traits>

#include "pth_burgers.hpp"
#include "pth_device.hpp"
#include "pth_stencil.hpp"

namespace pth {

namespace {

// HllGen with the scalar components multiplied by the reciprocal the velocity components
// already use (burgers_package.cpp:307-401 divides them by the same denominator).
template <int V, class LS, class RS>
__device__ __forceinline__ void SweepHll(LS l, RS r, int d, double *F) {
  const double upl = l(d), upr = r(d);
  const double sl = DMin(DMin(upl, upr), 0.0);
  const double sr = DMax(DMax(upl, upr), 0.0);
  const double islsr = 1.0 / (sr - sl + (sl * sr == 0.0));
#pragma unroll
  for (int n = 0; n < 3; ++n) {
    const double ul = l(n), ur = r(n);
    F[n] = 0.5 * (sr * ul * upl - sl * ur * upr + sl * sr * (ur - ul)) * islsr;
  }
#pragma unroll
  for (int n = 3; n < V; ++n) {
    const double ql = l(n), qr = r(n);
    F[n] = (sr * upl * ql - sl * upr * qr + sl * sr * (qr - ql)) * islsr;
  }
}

// ---- helpers of the tile sweep ---------------------------------------------------------
//
// Reciprocal by v_rcp_f64 and one third-order step r <- r (1 + e + e^2), e = 1 - x r: the
// hardware estimate is good to about 25 bits, so the step's e^3 is far below an ulp. Four
// instructions; an IEEE divide takes ten. The callers' arguments are positive normal numbers
// (sums of weights, or HLL denominators that are >= 1 whenever the speeds' product underflows).
__device__ __forceinline__ double Recip(double x) {
  const double r = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// WENO5Z of recon.hpp:28-99 for the block sweeps in about 100 instructions, where the
// reference's order of operations with the same reciprocals takes 130: the sweep is bound by
// FP64 issue, so everything is formed from the four differences d_k and the three second
// differences a_k.
//   * weights w_k = g_k h_k times be0 be1 be2: h_k = tau5 be_i be_j + (1 + eps / g_k) be0 be1
//     be2 needs no reciprocal; one reciprocal per side normalises them to sum w = 1;
//   * results relative to q2: g_k (p_k - q2) of a candidate polynomial is two multiply-adds;
//   * then al = 3 w0 w1 w2 / D + eps with D = g2 w0 w1 + g1 w0 w2 + g0 w1 w2 = g0 g1 g2 E,
//     E = h0 h1 + h0 h2 + h1 h2, so al = 3 u / E with u = h0 h1 h2 + eps E / 3 and the
//     harmonic mean 2 al ar / (al + ar) is 6 ul ur / (ul Er + ur El): the third reciprocal.
// Measured with both reciprocal steps and min / max as single instructions: 960-block refined
// cycle 1.83 -> 1.75 ms, 64-block cycle 146 -> 132 us.
// The values are the reference's to rounding. Range: h is of the size of be^3 and stays finite
// below a jump in q of about 1e50; beside a jump j the smallest normalised h is ~eps / j^2 and
// the harmonic mean's denominator ~eps^3 / j^4, normal to 1e60.
__device__ __forceinline__ void Weno5ZFast(double q0, double q1, double q2, double q3,
                                           double q4, double &ql, double &qr) {
  const double g0 = 0.1, g1 = 0.6, g2 = 0.3;
  const double eps = 10.0 * DBL_EPSILON;  // robust::EPS (src/utils/robust.hpp:38-41)
  const double t13 = 13.0 / 3.0;
  const double d0 = q1 - q0, d1 = q2 - q1, d2 = q3 - q2, d3 = q4 - q3;
  const double a0 = d1 - d0, a1 = d2 - d1, a2 = d3 - d2;
  const double b0 = fma(2.0, d1, a0), b1 = d1 + d2, b2 = fma(-2.0, d2, a2);
  const double be0 = fma(t13 * a0, a0, fma(b0, b0, eps));
  const double be1 = fma(t13 * a1, a1, fma(b1, b1, eps));
  const double be2 = fma(t13 * a2, a2, fma(b2, b2, eps));
  const double tau5 = fabs(be2 - be0);
  const double p12 = be1 * be2, p02 = be0 * be2, p01 = be0 * be1, p = be0 * p12;
  const double t0 = tau5 * p12, t1 = tau5 * p02, t2 = tau5 * p01;
  double l0 = fma(1.0 + eps / g0, p, t0), l1 = fma(1.0 + eps / g1, p, t1),
         l2 = fma(1.0 + eps / g2, p, t2);
  double r0 = fma(1.0 + eps / g0, p, t2), r1 = l1, r2 = fma(1.0 + eps / g2, p, t0);
  const double w1 = g1 * l1;
  const double il = Recip(fma(g0, l0, fma(g2, l2, w1)));
  const double ir = Recip(fma(g0, r0, fma(g2, r2, w1)));
  l0 *= il, l1 *= il, l2 *= il;
  r0 *= ir, r1 *= ir, r2 *= ir;
  // sums of w_k (p_k - q2)
  const double s1 = (g1 / 2) * d1;
  const double vl = fma(l0, fma(g0 / 3, a0, (g0 / 2) * d1),
                        fma(l1, fma(g1 / 3, a1, s1), l2 * fma(-g2 / 6, a2, (g2 / 2) * d2)));
  const double vr = fma(r0, fma(g0 / 3, a2, (-g0 / 2) * d2),
                        -fma(r1, fma(g1 / 6, a1, s1), r2 * fma(g2 / 6, a0, (g2 / 2) * d1)));
  const double ml = l1 * l2, mr = r1 * r2;
  const double El = fma(l0, l1 + l2, ml), Er = fma(r0, r1 + r2, mr);
  const double ul = fma(l0, ml, (eps / 3) * El), ur = fma(r0, mr, (eps / 3) * Er);
  const double alin = 6.0 * ul * ur * Recip(fma(ul, Er, ur * El));
  // half the MC-limited difference
  double dq = fmin(fmin(fabs(d1), fabs(d2)), 0.25 * fabs(b1));
  dq = copysign(d1 * d2 > 0.0 ? dq : 0.0, b1);
  ql = q2 + fma(alin, vl - dq, dq);
  qr = q2 + fma(alin, vr + dq, -dq);
}

__device__ __forceinline__ void FastStates(int recon, double q0, double q1, double q2, double q3,
                                           double q4, double &ql, double &qr) {
  if (recon == 0)
    Weno5ZFast(q0, q1, q2, q3, q4, ql, qr);
  else
    LinearRecon(q1, q2, q3, ql, qr);
}

// CellStates with the sweep's WENO5Z (the 8^3 block sweep and its flux-correction send).
__device__ __forceinline__ void SweepStates(const double *q, unsigned c, unsigned st, int recon,
                                            double &ql, double &qr) {
  if (recon == 0)
    Weno5ZFast(LoadAt(q, c - 2 * st), LoadAt(q, c - st), LoadAt(q, c), LoadAt(q, c + st),
               LoadAt(q, c + 2 * st), ql, qr);
  else
    LinearRecon(LoadAt(q, c - st), LoadAt(q, c), LoadAt(q, c + st), ql, qr);
}

// HLL of burgers_package.cpp:307-401 (lr_to_flux, burgers_package.hpp:33-43) as two
// coefficients per face: with sl, sr the signal speeds and islsr = 1 / (sr - sl + (sl sr ==
// 0)), the scalar flux (sr upl ql - sl upr qr + sl sr (qr - ql)) islsr equals a ql + b qr with
// a = islsr sr (upl - sl), b = islsr sl (sr - upr), and the velocity flux is half of the same
// combination of ul, ur. So the coupling of the components goes through (a, b) only.
__device__ __forceinline__ void HllCoef(double upl, double upr, double &a, double &b) {
  const double sl = fmin(fmin(upl, upr), 0.0);
  const double sr = fmax(fmax(upl, upr), 0.0);
  const double is = Recip(sr - sl + (sl * sr == 0.0));
  a = (is * sr) * (upl - sl);
  b = (is * sl) * (sr - upr);
}

// flux of component n from the face coefficients and its left / right states
__device__ __forceinline__ double HllFluxN(int n, double a, double b, double l, double r) {
  if (n < 3) return fma(0.5 * a, l, (0.5 * b) * r);
  return fma(a, l, b * r);
}

// v, as a value the compiler knows nothing about
__device__ __forceinline__ int Opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

__device__ __forceinline__ int DMinI(int a, int b) { return b < a ? b : a; }

// value of lane - 1 / lane + 1 within each 16-lane DPP row; the row's first / last lane gets
// its own `edge`
__device__ __forceinline__ double FromLeft16(double v, double edge) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), 0x111, 0xF,
                                             0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), 0x111, 0xF,
                                             0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double FromRight16(double v, double edge) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(edge), __double2loint(v), 0x101, 0xF,
                                             0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(edge), __double2hiint(v), 0x101, 0xF,
                                             0xF, false);
  return __hiloint2double(hi, lo);
}

// flxcor_send of the block-sweep stage: four adjacent threads per coarse face cell of a patch,
// one per fine face (p, q), evaluate the HLL flux of their face straight from the fine block's
// state (the left state of face f is ql of cell f - 1, the right state qr of cell f, as
// CalculateFluxes stores them); the first of the four gathers the other three by lane
// shuffles and writes their restriction to the correction store.
template <int V, bool RING>
__global__ void __launch_bounds__(64)
    FlxcorDirectKernel(const FluxPatch *__restrict__ patches, const double *__restrict__ U,
                       double *__restrict__ store, Geo G, int recon) {
  const FluxPatch &P = patches[blockIdx.x];
  const int t = blockIdx.y * 64 + threadIdx.x;
  const int cell = t >> 2, sub = t & 3, p = sub & 1, q = sub >> 1;
  const bool live = cell < P.n[0] * P.n[1];
  const int a = live ? cell % P.n[0] : 0, c = live ? cell / P.n[0] : 0;
  const std::int64_t cs = G.cells;
  const double *Ub = U + static_cast<std::int64_t>(P.fine) * V * cs;
  const unsigned st = 8u * static_cast<unsigned>(P.d == 0 ? 1 : P.d == 1 ? G.e0 : G.e0 * G.e1);
  double F[V];
#pragma unroll
  for (int n = 0; n < V; ++n) F[n] = 0.0;
  if (live && p < P.step[0] && q < P.step[1]) {
    const unsigned o = 8u * static_cast<unsigned>(PatchFineCell(P, G, a, c, p, q));
    double l[V], r[V];
    if (RING) {
      // the expressions of TileSweepKernel: FastStates and the face coefficients
#pragma unroll
      for (int n = 0; n < V; ++n) {
        const double *q = Ub + n * cs;
        double x, y;
        FastStates(recon, LoadAt(q, o - 3 * st), LoadAt(q, o - 2 * st), LoadAt(q, o - st),
                   LoadAt(q, o), LoadAt(q, o + st), l[n], x);
        FastStates(recon, LoadAt(q, o - 2 * st), LoadAt(q, o - st), LoadAt(q, o),
                   LoadAt(q, o + st), LoadAt(q, o + 2 * st), y, r[n]);
      }
      double a, bb;
      HllCoef(l[P.d], r[P.d], a, bb);
#pragma unroll
      for (int n = 0; n < V; ++n) F[n] = HllFluxN(n, a, bb, l[n], r[n]);
    } else {
#pragma unroll
      for (int n = 0; n < V; ++n) {
        double x, y;
        SweepStates(Ub + n * cs, o - st, st, recon, l[n], x);
        SweepStates(Ub + n * cs, o, st, recon, y, r[n]);
      }
      SweepHll<V>([&](int n) { return l[n]; }, [&](int n) { return r[n]; }, P.d, F);
    }
  }
  const int lane0 = static_cast<int>(threadIdx.x) & ~3;
  const std::int64_t dst = P.dst + a + static_cast<std::int64_t>(c) * P.rows;
#pragma unroll
  for (int n = 0; n < V; ++n) {
    const double f00 = __shfl(F[n], lane0, 64), f01 = __shfl(F[n], lane0 + 1, 64);
    const double f10 = __shfl(F[n], lane0 + 2, 64), f11 = __shfl(F[n], lane0 + 3, 64);
    if (live && sub == 0)
      store[dst + static_cast<std::int64_t>(n) * P.comp] =
          RestrictFace(P.d, P.area, f00, f01, f10, f11, P.step[0], P.step[1]);
  }
}

// ---- block sweep: reconstruction, HLL, flux divergence and RK update in one launch ----------
//
// One thread per (i, j) column of a cubic block of N cells per side, marching k over interior
// planes. Per plane: the x states of the plane's rows (extended by one cell each way) go to
// LDS, the HLL flux of every x face of the plane is evaluated once into LDS (each thread the
// high face of its cell, the first N threads the low face of one row each), and each thread
// forms its cell's x difference; then the same for y; then the z states of the plane above,
// whose qr closes the high z face (the low z face of plane k is the high z face of plane
// k - 1, carried in registers). The flux divergence sums x, y, z in the order of
// FluxDivHelper (update.hpp:43-57), then the RK averaging and update, the derived field and
// the CFL minimum follow as in FluxUpdateKernel. Every face flux is the same expression as in
// the other forms up to FMA contraction and the folded divides, so the stage output agrees
// with theirs to rounding, and no flux or face state reaches HBM. On
// multilevel meshes, faces with a finer neighbour take the restricted fine fluxes from the
// correction store (fover gives the face's image in fcor, or -1).
// The grid is persistent: workgroup g takes planes [g T / G, (g + 1) T / G) of the
// T = nblocks * N planes in block order, so every workgroup does the same number of planes
// (a segment that starts inside a block first rebuilds the z state below its first plane).
// partial[g] is the workgroup's CFL minimum.

template <int N, int NG, int V, int MINW>
__global__ void __launch_bounds__(N * N, MINW)
    BlockSweepKernel(const double *__restrict__ U, const double *base, double *out,
                     double *__restrict__ derived, double *__restrict__ partial,
                     const BlockCoefs *__restrict__ coef, int nblocks, double beta,
                     const double *__restrict__ dtvar, int recon, const int *__restrict__ fover,
                     const double *__restrict__ fcor, const int *__restrict__ push) {
  static_assert(N >= 2 * NG, "a cell lies in at most one boundary strip per dimension");
  constexpr int E = N + 2 * NG;
  constexpr int NT = N * N;
  constexpr int R = N + 2;  // states per row: ext cells lo - 1 .. hi + 1
  constexpr int P = R * N;  // states of one plane per component
  constexpr int FP = (N + 1) * N;  // faces of one plane per component and direction
  __shared__ double sl[V * P], sr[V * P];
  __shared__ double fx[V * FP];  // x (then y) face fluxes of the plane, each face once
  __shared__ double wmin[(NT + 63) / 64];
  const int tx = threadIdx.x % N, ty = threadIdx.x / N;
  constexpr std::int64_t cs = static_cast<std::int64_t>(E) * E * E;
  const double bdt = beta * dtvar[0];
  const double w2 = 1.0 - beta;
  constexpr int comp = N * N;  // correction-store stride between components
  constexpr unsigned sx = 8u, sy = 8u * E, sz = 8u * E * E;
  double m = DBL_MAX;
  const std::int64_t T = static_cast<std::int64_t>(nblocks) * N;
  std::int64_t pnext = T * blockIdx.x / gridDim.x;
  const std::int64_t pend = T * (blockIdx.x + 1) / gridDim.x;
  while (pnext < pend) {
    const int b = static_cast<int>(pnext / N);
    const int k0 = static_cast<int>(pnext % N);
    const int k1 = static_cast<int>(pend - pnext < N - k0 ? k0 + (pend - pnext) : N);
    pnext += k1 - k0;
    const double *Ub = U + static_cast<std::int64_t>(b) * V * cs;
    const BlockCoefs &C = coef[b];
    const int ox0 = fover ? fover[6 * b + 0] : -1, ox1 = fover ? fover[6 * b + 1] : -1;
    const int oy0 = fover ? fover[6 * b + 2] : -1, oy1 = fover ? fover[6 * b + 3] : -1;
    const int oz0 = fover ? fover[6 * b + 4] : -1, oz1 = fover ? fover[6 * b + 5] : -1;
    // z states of one plane of cells kc for every column, [n][j][i] (a flat loop like x and y)
    auto zstates = [&](int kc) {
      for (int t = threadIdx.x; t < V * NT; t += NT) {
        const int n = t / NT, u = t % NT;
        const unsigned c = 8u * static_cast<unsigned>((kc * E + NG + u / N) * E + NG + u % N);
        SweepStates(Ub + n * cs, c, sz, recon, sl[n * P + u], sr[n * P + u]);
      }
    };
    // z faces: zl = ql of the cell below the current plane, zf = flux on the current low z face
    double zl[V], zf[V];
    __syncthreads();  // the previous segment's states have been read
    zstates(NG + k0 - 1);
    __syncthreads();
#pragma unroll
    for (int n = 0; n < V; ++n) zl[n] = sl[n * P + threadIdx.x];
    __syncthreads();
    zstates(NG + k0);
    __syncthreads();
    SweepHll<V>([&](int n) { return zl[n]; }, [&](int n) { return sr[n * P + threadIdx.x]; }, 2, zf);
    if (k0 == 0 && oz0 >= 0)
#pragma unroll
      for (int n = 0; n < V; ++n) zf[n] = fcor[oz0 + tx + ty * N + n * comp];
#pragma unroll
    for (int n = 0; n < V; ++n) zl[n] = sl[n * P + threadIdx.x];
    for (int k = k0; k < k1; ++k) {
      const int kk = NG + k;
      double du[V];
      // ---- x: states of ext cells lo - 1 .. hi + 1 of every row of the plane, [n][row][a]
      __syncthreads();  // the previous states have been read
      for (int t = threadIdx.x; t < V * P; t += NT) {
        const int n = t / P, u = t % P;
        const int a = u % R, row = u / R;
        const unsigned c = 8u * static_cast<unsigned>((kk * E + NG + row) * E + NG - 1 + a);
        SweepStates(Ub + n * cs, c, sx, recon, sl[t], sr[t]);
      }
      __syncthreads();
      {
        // every x face once: each thread the high face of its cell, threads 0 .. N - 1 also
        // the low face of row threadIdx.x; fluxes to LDS as [n][row][face]
        double F[V];
        const double *L = sl + ty * R + tx, *Rr = sr + ty * R + tx;
        SweepHll<V>([&](int n) { return L[n * P + 1]; }, [&](int n) { return Rr[n * P + 2]; }, 0,
                  F);
        if (tx == N - 1 && ox1 >= 0)
#pragma unroll
          for (int n = 0; n < V; ++n) F[n] = fcor[ox1 + ty + k * N + n * comp];
#pragma unroll
        for (int n = 0; n < V; ++n) fx[n * FP + ty * (N + 1) + tx + 1] = F[n];
        if (static_cast<int>(threadIdx.x) < N) {
          const int row = threadIdx.x;
          SweepHll<V>([&](int n) { return sl[n * P + row * R]; },
                    [&](int n) { return sr[n * P + row * R + 1]; }, 0, F);
          if (ox0 >= 0)
#pragma unroll
            for (int n = 0; n < V; ++n) F[n] = fcor[ox0 + row + k * N + n * comp];
#pragma unroll
          for (int n = 0; n < V; ++n) fx[n * FP + row * (N + 1)] = F[n];
        }
      }
      __syncthreads();  // the x fluxes are in LDS and the x states have been read
      {
        // du = A F(hi) - A F(lo)
        const double A = C.area[0];
        const double *f = fx + ty * (N + 1) + tx;
#pragma unroll
        for (int n = 0; n < V; ++n) du[n] = (A * f[n * FP + 1] - A * f[n * FP]);
      }
      // ---- y: states of ext cells lo - 1 .. hi + 1 of every column, [n][a][i]
      for (int t = threadIdx.x; t < V * P; t += NT) {
        const int n = t / P, u = t % P;
        const int i = u % N, a = u / N;
        const unsigned c = 8u * static_cast<unsigned>((kk * E + NG - 1 + a) * E + NG + i);
        SweepStates(Ub + n * cs, c, sy, recon, sl[t], sr[t]);
      }
      __syncthreads();  // also: every thread has read its x fluxes
      {
        // every y face once, as [n][face][i]
        double F[V];
        const double *L = sl + ty * N + tx, *Rr = sr + ty * N + tx;
        SweepHll<V>([&](int n) { return L[n * P + N]; }, [&](int n) { return Rr[n * P + 2 * N]; },
                  1, F);
        if (ty == N - 1 && oy1 >= 0)
#pragma unroll
          for (int n = 0; n < V; ++n) F[n] = fcor[oy1 + tx + k * N + n * comp];
#pragma unroll
        for (int n = 0; n < V; ++n) fx[n * FP + (ty + 1) * N + tx] = F[n];
        if (static_cast<int>(threadIdx.x) < N) {
          const int col = threadIdx.x;
          SweepHll<V>([&](int n) { return sl[n * P + col]; },
                    [&](int n) { return sr[n * P + N + col]; }, 1, F);
          if (oy0 >= 0)
#pragma unroll
            for (int n = 0; n < V; ++n) F[n] = fcor[oy0 + col + k * N + n * comp];
#pragma unroll
          for (int n = 0; n < V; ++n) fx[n * FP + col] = F[n];
        }
      }
      __syncthreads();  // the y fluxes are in LDS and the y states have been read
      {
        const double A = C.area[1];
        const double *f = fx + ty * N + tx;
#pragma unroll
        for (int n = 0; n < V; ++n) du[n] = du[n] + (A * f[n * FP + N] - A * f[n * FP]);
      }
      // ---- z: qr of the cell above this plane gives the high z face; its ql moves down
      zstates(kk + 1);
      __syncthreads();  // also: every thread has read its y fluxes
      {
        double Fhi[V];
        SweepHll<V>([&](int n) { return zl[n]; }, [&](int n) { return sr[n * P + threadIdx.x]; }, 2,
                  Fhi);
        if (k == N - 1 && oz1 >= 0)
#pragma unroll
          for (int n = 0; n < V; ++n) Fhi[n] = fcor[oz1 + tx + ty * N + n * comp];
        const double A = C.area[2];
#pragma unroll
        for (int n = 0; n < V; ++n) {
          du[n] = du[n] + (A * Fhi[n] - A * zf[n]);
          zf[n] = Fhi[n];
          zl[n] = sl[n * P + threadIdx.x];
        }
      }
      // ---- divergence, RK averaging and update, derived field, CFL
      const std::int64_t cell = (static_cast<std::int64_t>(kk) * E + NG + ty) * E + NG + tx;
      const std::int64_t c0 = static_cast<std::int64_t>(b) * V * cs + cell;
      double u1[V];
#pragma unroll
      for (int n = 0; n < V; ++n) {
        const double dudt = -du[n] / C.vol;
        const double avg = beta * U[c0 + n * cs] + w2 * base[c0 + n * cs];
        u1[n] = 1.0 * avg + bdt * dudt;
        out[c0 + n * cs] = u1[n];
      }
      if (push) {
        // the exchange's same-level copies: a cell within NG of a face is a ghost cell of the
        // same-level neighbours across that face, edge or corner (push[27 b + direction]),
        // at its index shifted by N along each crossed dimension
        const int lx = tx < NG ? -1 : (tx >= N - NG ? 1 : 0);
        const int ly = ty < NG ? -1 : (ty >= N - NG ? 1 : 0);
        const int lz = k < NG ? -1 : (k >= N - NG ? 1 : 0);
        for (int az = 0; az < (lz ? 2 : 1); ++az)
          for (int ay = 0; ay < (ly ? 2 : 1); ++ay)
            for (int ax = 0; ax < (lx ? 2 : 1); ++ax) {
              const int dx = ax ? lx : 0, dy = ay ? ly : 0, dz = az ? lz : 0;
              if (!(dx | dy | dz)) continue;
              const int g = push[27 * b + (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)];
              if (g < 0) continue;
              const std::int64_t d0 =
                  static_cast<std::int64_t>(g) * V * cs +
                  (static_cast<std::int64_t>(kk - dz * N) * E + NG + ty - dy * N) * E + NG + tx -
                  dx * N;
#pragma unroll
              for (int n = 0; n < V; ++n) out[d0 + n * cs] = u1[n];
            }
      }
      if (derived)
        derived[static_cast<std::int64_t>(b) * cs + cell] =
            0.5 * u1[3] * (u1[0] * u1[0] + u1[1] * u1[1] + u1[2] * u1[2]);
      double sp = fabs(u1[0]) / C.dx[0];
      sp = sp + fabs(u1[1]) / C.dx[1];
      sp = sp + fabs(u1[2]) / C.dx[2];
      m = DMin(m, 1.0 / sp);
    }
  }
  if (!partial) return;
  m = WaveMin(m);
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = wmin[0];
#pragma unroll
    for (int w = 1; w < (NT + 63) / 64; ++w) v = DMin(v, wmin[w]);
    partial[blockIdx.x] = v;
  }
}

// ---- block sweep for 16^3 blocks of at most 7 components ------------------------------------
//
// One workgroup of 256 threads marches the z planes of a block; thread (tx, ty) owns column
// (i, j) = (tx, ty). Per plane kk:
//   * the plane's U (all components, with 3-cell x and y halos) is staged in LDS; its interior
//     comes from the thread's register ring, the halos from HBM;
//   * x: each thread reconstructs its own cell (stencil read from LDS); the neighbouring
//     cells' states come by DPP row shifts (a row of 16 cells is a 16-lane DPP row), those of
//     the cells beyond the row ends from a small pass over all components; the face
//     coefficients (a, b) of HllCoef follow from the x velocity's states, then every
//     component's two face fluxes are two multiply-adds each;
//   * y: the same with the thread mapping transposed (thread (tx, ty) takes cell i = ty,
//     j = tx, so a column is a DPP row); the y differences reach the owning thread through
//     LDS;
//   * z: each thread keeps U of its column at planes kk - 1, kk + 1, kk + 2, kk + 3 in
//     registers (kk itself is in LDS), so the z stencil of the cell above needs no load; the
//     high z face's flux becomes the next plane's low face flux; the load of plane kk + 4 is
//     issued a whole plane ahead of its use.
// The divergence adds x, y and z in the order of FluxDivHelper (update.hpp:43-57); the RK
// averaging and update, derived field, CFL minimum, flux-correction faces and same-level push
// are those of BlockSweepKernel. Each U element is read from HBM once per workgroup (plus
// the halos and the segment's first planes), and face states and fluxes never leave the CU.
template <int V, int MINW, int RECON>
__global__ void __launch_bounds__(256, MINW)
    BlockSweep16Kernel(const double *__restrict__ U, const double *base, double *out,
                       double *__restrict__ derived, double *__restrict__ partial,
                       const BlockCoefs *__restrict__ coef, int nblocks, double beta,
                       const double *__restrict__ dtvar, const int *__restrict__ fover,
                       const double *__restrict__ fcor, const int *__restrict__ push,
                       const int *__restrict__ list) {
  constexpr int N = 16, NG = 4, E = N + 2 * NG, NT = N * N;
  constexpr int H = 3;             // halo of the staged plane
  constexpr int PW = N + 2 * H;    // staged rows / columns
  constexpr int PP = PW + 1;       // row pitch (odd, fewer bank conflicts on column reads)
  constexpr int PS = PW * PP;      // one component of the staged plane
  constexpr int SP = N + 1;        // pitch of the difference tile
  constexpr int NX = V * N * 2;    // beyond-the-row states of one direction
  constexpr int NH = V * 12 * N;   // halo cells of one staged plane (all components)
  constexpr int QH = (NH + NT - 1) / NT;  // halo cells per thread
  constexpr std::int64_t cs = static_cast<std::int64_t>(E) * E * E;
  constexpr std::int64_t sz = static_cast<std::int64_t>(E) * E;
  constexpr int comp = N * N;      // correction-store stride between components
  __shared__ double pl[V * PS];      // [n][j + H][i + H]
  __shared__ double ext[2 * NX];     // [dir][n][line][side]: side 0 ql of cell -1, 1 qr of cell N
  __shared__ double sd[V * N * SP];  // x + y differences [n][j][i], then the new state
  __shared__ double zs[2 * V * NT];  // this thread's z state: [0][n] ql of its cell, [1][n] flux
                                     // of its low z face (own slots, no barriers)
  __shared__ double fxy[2 * V * 2 * N];  // corrected x / y face fluxes of the plane,
                                          // [dir][n][side][line] (blocks with such faces)
  __shared__ double wmin[NT / 64];
  const int tx = threadIdx.x % N, ty = threadIdx.x / N;
  const double bdt = beta * dtvar[0];
  const double w2 = 1.0 - beta;
  const bool same_base = base == U;
  double m = DBL_MAX;
  const std::int64_t T = static_cast<std::int64_t>(nblocks) * N;
  std::int64_t pnext = T * blockIdx.x / gridDim.x;
  const std::int64_t pend = T * (blockIdx.x + 1) / gridDim.x;
  const double *own_pl = pl + (ty + H) * PP + tx + H;  // own cell, component 0
  const int own_sd = ty * SP + tx;                      // own cell in the difference tile
  // halo cell q of this thread (q < QH): its component, offset within a plane of the brick
  // and place in the staged plane; cells past the last share its address (loads are
  // unconditional, so the compiler can count them in its memory waits)
  auto halo = [&](int q, std::int64_t &goff, int &loff) {
    const int t = DMinI(static_cast<int>(threadIdx.x) + q * NT, NH - 1);
    const int n = t / (12 * N), r = t % (12 * N);
    int i, j;
    if (r < 6 * N) {  // y strips: rows -3 .. -1 and N .. N + 2, all interior columns
      const int yy = r / N;
      i = r % N;
      j = yy < 3 ? yy - 3 : N + yy - 3;
    } else {          // x strips: all interior rows, columns -3 .. -1 and N .. N + 2
      const int qq = r - 6 * N;
      j = qq / 6;
      const int c = qq % 6;
      i = c < 3 ? c - 3 : N + c - 3;
    }
    goff = n * cs + static_cast<std::int64_t>(NG + j) * E + NG + i;
    loff = n * PS + (j + H) * PP + i + H;
  };
  // the new state of plane kk (in the thread's own slots of sd) to out, the same-level
  // neighbours' ghosts, the derived field and the CFL minimum
  auto flush = [&](int b, int k) {
    const int kk = NG + k;
    const std::int64_t cell = static_cast<std::int64_t>(kk) * sz + (NG + ty) * E + NG + tx;
    const std::int64_t c0 = static_cast<std::int64_t>(b) * V * cs + cell;
    double u1[V];
#pragma unroll
    for (int n = 0; n < V; ++n) {
      u1[n] = sd[n * N * SP + own_sd];
      out[c0 + n * cs] = u1[n];
    }
    if (push) {
      // same-level ghost copies: a cell within NG of a face is a ghost cell of the
      // same-level neighbours across that face, edge or corner (push[27 b + direction]), at
      // its index shifted by N along each crossed dimension
      const int lx = tx < NG ? -1 : (tx >= N - NG ? 1 : 0);
      const int ly = ty < NG ? -1 : (ty >= N - NG ? 1 : 0);
      const int lz = k < NG ? -1 : (k >= N - NG ? 1 : 0);
      for (int az_ = 0; az_ < (lz ? 2 : 1); ++az_)
        for (int ay = 0; ay < (ly ? 2 : 1); ++ay)
          for (int ax = 0; ax < (lx ? 2 : 1); ++ax) {
            const int dx = ax ? lx : 0, dy = ay ? ly : 0, dz = az_ ? lz : 0;
            if (!(dx | dy | dz)) continue;
            const int g = push[27 * b + (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1)];
            if (g < 0) continue;
            const std::int64_t d0 =
                static_cast<std::int64_t>(g) * V * cs +
                (static_cast<std::int64_t>(kk - dz * N) * E + NG + ty - dy * N) * E + NG + tx -
                dx * N;
#pragma unroll
            for (int n = 0; n < V; ++n) out[d0 + n * cs] = u1[n];
          }
    }
    if (derived)
      derived[static_cast<std::int64_t>(b) * cs + cell] =
          0.5 * u1[3] * (u1[0] * u1[0] + u1[1] * u1[1] + u1[2] * u1[2]);
    const BlockCoefs &Cb = coef[b];
    double sp = fabs(u1[0]) / Cb.dx[0];
    sp = sp + fabs(u1[1]) / Cb.dx[1];
    sp = sp + fabs(u1[2]) / Cb.dx[2];
    m = DMin(m, 1.0 / sp);
  };
  while (pnext < pend) {
    // the planes of the launch run over its blocks in order: all blocks, or the listed ones
    const int b = list ? list[pnext / N] : static_cast<int>(pnext / N);
    const int k0 = static_cast<int>(pnext % N);
    const int k1 = static_cast<int>(pend - pnext < N - k0 ? k0 + (pend - pnext) : N);
    pnext += k1 - k0;
    const double *Ub = U + static_cast<std::int64_t>(b) * V * cs;
    const BlockCoefs &C = coef[b];
    const double ivol = 1.0 / C.vol;
    const int ox0 = fover ? fover[6 * b + 0] : -1, ox1 = fover ? fover[6 * b + 1] : -1;
    const int oy0 = fover ? fover[6 * b + 2] : -1, oy1 = fover ? fover[6 * b + 3] : -1;
    const int oz0 = fover ? fover[6 * b + 4] : -1, oz1 = fover ? fover[6 * b + 5] : -1;
    const std::int64_t col = static_cast<std::int64_t>(NG + ty) * E + NG + tx;  // in a plane
    const double *Uc = Ub + col;  // this thread's column, component 0, plane 0
    const int kk0 = NG + k0;
    // halo of the first plane
    double hv[QH];
#pragma unroll
    for (int q = 0; q < QH; ++q) {
      std::int64_t go;
      int lo;
      halo(q, go, lo);
      hv[q] = Ub[go + kk0 * sz];
    }
    // ---- z state at the segment's first plane kk0: ql of cell kk0 (zl) and the flux of face
    // kk0 - 1/2 (flo); the z velocity first gives the face coefficients. The per-component
    // part runs as a loop through LDS (once per segment, kept out of the unrolled code).
    double az, bz;
    {
      const double *q = Uc + 2 * cs + static_cast<std::int64_t>(kk0 - 3) * sz;
      double qm, qx, ql, qr;
      FastStates(RECON, q[0], q[sz], q[2 * sz], q[3 * sz], q[4 * sz], qm, qx);
      FastStates(RECON, q[sz], q[2 * sz], q[3 * sz], q[4 * sz], q[5 * sz], ql, qr);
      HllCoef(qm, qr, az, bz);
    }
#pragma unroll 1
    for (int n = 0; n < V; ++n) {
      const double *q = Uc + n * cs + static_cast<std::int64_t>(kk0 - 3) * sz;
      double qm, qx, ql, qr;
      FastStates(RECON, q[0], q[sz], q[2 * sz], q[3 * sz], q[4 * sz], qm, qx);
      FastStates(RECON, q[sz], q[2 * sz], q[3 * sz], q[4 * sz], q[5 * sz], ql, qr);
      double f = HllFluxN(n, az, bz, qm, qr);
      if (k0 == 0 && oz0 >= 0) f = fcor[oz0 + tx + ty * N + n * comp];
      zs[(V + n) * NT + threadIdx.x] = f;
      zs[n * NT + threadIdx.x] = ql;
    }
    double r0[V], r1[V], r2[V], r3[V], r4[V];
#pragma unroll
    for (int n = 0; n < V; ++n) {
      const double *q = Uc + n * cs + static_cast<std::int64_t>(kk0 - 1) * sz;
      r0[n] = q[0];
      r1[n] = q[sz];
      r2[n] = q[2 * sz];
      r3[n] = q[3 * sz];
      r4[n] = q[4 * sz];
    }
    for (int k = k0; k < k1; ++k) {
      const int kk = NG + k;
      __syncthreads();  // the previous plane's (or the segment start's) LDS has been read
      // ---- stage plane kk: interior from the ring, halos from the prefetch
#pragma unroll
      for (int n = 0; n < V; ++n) pl[n * PS + (ty + H) * PP + tx + H] = r1[n];
#pragma unroll
      for (int q = 0; q < QH; ++q) {
        std::int64_t go;
        int lo;
        halo(q, go, lo);
        pl[lo] = hv[q];
      }
      // corrected fluxes of this plane's x and y faces (only blocks next to finer ones):
      // staged here, so the loops below read LDS and issue no conditional load
      if (ox0 >= 0 || ox1 >= 0 || oy0 >= 0 || oy1 >= 0) {
        for (int t = threadIdx.x; t < 2 * V * 2 * N; t += NT) {
          const int dir = t / (2 * V * N), r = t % (2 * V * N);
          const int n = r / (2 * N), side = (r / N) & 1, line = r % N;
          const int o = dir == 0 ? (side ? ox1 : ox0) : (side ? oy1 : oy0);
          fxy[t] = o >= 0 ? fcor[o + line + k * N + n * comp] : 0.0;
        }
      }
      // the previous plane's results leave now, well before the next wait on a load; then the
      // ring's top plane (kk + 3) for this plane's z stencils, issued after those stores so
      // that the wait for it counts only loads
      if (k > k0) {
        flush(b, k - 1);
#pragma unroll
        for (int n = 0; n < V; ++n) r4[n] = Uc[n * cs + static_cast<std::int64_t>(kk + 3) * sz];
      }
      __syncthreads();
      // ---- states of the cells just beyond each row (x) and column (y), every component
      for (int t = threadIdx.x; t < 2 * NX; t += NT) {
        const int dir = t / NX, r = t % NX;
        const int n = r / (2 * N), q = r % (2 * N);
        const int line = q >> 1, side = q & 1;
        const int cell = side ? N : -1;
        const int st = dir ? PP : 1;
        const double *c = pl + n * PS + (dir ? (cell + H) * PP + line + H
                                             : (line + H) * PP + cell + H);
        double ql, qr;
        FastStates(RECON, c[-2 * st], c[-st], c[0], c[st], c[2 * st], ql, qr);
        ext[t] = side ? qr : ql;
      }
      __syncthreads();
      // ---- x: own cell (tx, ty); differences to sd[n][ty][tx]
      {
        const double A = C.area[0];
        double ql0, qr0;
        FastStates(RECON, own_pl[-2], own_pl[-1], own_pl[0], own_pl[1], own_pl[2], ql0, qr0);
        double qlm = FromLeft16(ql0, 0.0), qrp = FromRight16(qr0, 0.0);
        if (tx == 0) qlm = ext[ty * 2];
        if (tx == N - 1) qrp = ext[ty * 2 + 1];
        double alo, blo, ahi, bhi;
        HllCoef(qlm, qr0, alo, blo);
        HllCoef(ql0, qrp, ahi, bhi);
#pragma unroll 2
        for (int n = 0; n < V; ++n) {
          double ql = ql0, qr = qr0;
          if (n > 0) {
            const double *cn = own_pl + n * PS;
            FastStates(RECON, cn[-2], cn[-1], cn[0], cn[1], cn[2], ql, qr);
          }
          double lm = FromLeft16(ql, 0.0), rp = FromRight16(qr, 0.0);
          if (tx == 0) lm = ext[(n * N + ty) * 2];
          if (tx == N - 1) rp = ext[(n * N + ty) * 2 + 1];
          double fl = HllFluxN(n, alo, blo, lm, qr);
          double fh = HllFluxN(n, ahi, bhi, ql, rp);
          if (tx == 0 && ox0 >= 0) fl = fxy[(n * 2 + 0) * N + ty];
          if (tx == N - 1 && ox1 >= 0) fh = fxy[(n * 2 + 1) * N + ty];
          sd[n * N * SP + own_sd] = A * fh - A * fl;
        }
      }
      __syncthreads();  // the x differences are in the tile
      // ---- y: cell i = ty, j = tx (a column per DPP row); adds to sd[n][j][i]
      {
        const double A = C.area[1];
        const double *c = pl + (tx + H) * PP + ty + H;
        double ql1, qr1;
        FastStates(RECON, c[PS - 2 * PP], c[PS - PP], c[PS], c[PS + PP], c[PS + 2 * PP], ql1,
                   qr1);
        double qlm = FromLeft16(ql1, 0.0), qrp = FromRight16(qr1, 0.0);
        if (tx == 0) qlm = ext[NX + (N + ty) * 2];
        if (tx == N - 1) qrp = ext[NX + (N + ty) * 2 + 1];
        double alo, blo, ahi, bhi;
        HllCoef(qlm, qr1, alo, blo);
        HllCoef(ql1, qrp, ahi, bhi);
#pragma unroll 2
        for (int n = 0; n < V; ++n) {
          double ql = ql1, qr = qr1;
          if (n != 1) {
            const double *cn = c + n * PS;
            FastStates(RECON, cn[-2 * PP], cn[-PP], cn[0], cn[PP], cn[2 * PP], ql, qr);
          }
          double lm = FromLeft16(ql, 0.0), rp = FromRight16(qr, 0.0);
          if (tx == 0) lm = ext[NX + (n * N + ty) * 2];
          if (tx == N - 1) rp = ext[NX + (n * N + ty) * 2 + 1];
          double fl = HllFluxN(n, alo, blo, lm, qr);
          double fh = HllFluxN(n, ahi, bhi, ql, rp);
          if (tx == 0 && oy0 >= 0) fl = fxy[((V + n) * 2 + 0) * N + ty];
          if (tx == N - 1 && oy1 >= 0) fh = fxy[((V + n) * 2 + 1) * N + ty];
          double &slot = sd[n * N * SP + tx * SP + ty];
          slot = slot + (A * fh - A * fl);
        }
      }
      __syncthreads();  // x + y differences complete
      // the base state of this plane (second stage), then the next plane's halo; both are
      // issued before this plane's results are stored, so no wait drains a store
      const std::int64_t c0 = static_cast<std::int64_t>(b) * V * cs +
                              static_cast<std::int64_t>(kk) * sz + col;
      double bv[V];
#pragma unroll
      for (int n = 0; n < V; ++n) bv[n] = same_base ? 0.0 : base[c0 + n * cs];
      if (k + 1 < k1) {
#pragma unroll
        for (int q = 0; q < QH; ++q) {
          std::int64_t go;
          int lo;
          halo(q, go, lo);
          hv[q] = Ub[go + (kk + 1) * sz];
        }
      }
      // ---- z: the cell above (kk + 1) from the ring; its low face closes this cell
      const double A = C.area[2];
      {
        double ql2, qr2;
        FastStates(RECON, r0[2], own_pl[2 * PS], r2[2], r3[2], r4[2], ql2, qr2);
        HllCoef(zs[2 * NT + threadIdx.x], qr2, az, bz);
      }
      // the z loop in two copies: the top plane of a block whose upper z face takes the
      // correction store's fluxes loads them; no other plane has a load in this loop
      auto zloop = [&](auto top_tag) {
        constexpr bool TOP = decltype(top_tag)::value;
  #pragma unroll
        for (int n = 0; n < V; ++n) {
          const double uo = own_pl[n * PS];
          double ql, qr;
          FastStates(RECON, r0[n], uo, r2[n], r3[n], r4[n], ql, qr);
          double &zl = zs[n * NT + threadIdx.x], &flo = zs[(V + n) * NT + threadIdx.x];
          double fh = HllFluxN(n, az, bz, zl, qr);
          if (TOP) fh = fcor[oz1 + tx + ty * N + n * comp];
          double &slot = sd[n * N * SP + own_sd];
          const double du = slot + (A * fh - A * flo);
          flo = fh;
          zl = ql;
          const double dudt = -du * ivol;
          const double avg = beta * uo + w2 * (same_base ? uo : bv[n]);
          slot = 1.0 * avg + bdt * dudt;  // the new state waits here until the next plane
          r0[n] = uo;  // the ring moves up one plane
          r1[n] = r2[n];
          r2[n] = r3[n];
          r3[n] = r4[n];
          // one component at a time: interleaving the seven reconstructions needs more
          // registers than the budget holds
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (k == N - 1 && oz1 >= 0)
        zloop(std::true_type());
      else
        zloop(std::false_type());
    }
    flush(b, k1 - 1);  // the segment's last plane (own slots only: no barrier needed)
  }
  if (!partial) return;
  m = WaveMin(m);
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = wmin[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) v = DMin(v, wmin[w]);
    partial[blockIdx.x] = v;
  }
}
// ---- tile sweep: blocks whose x and y sizes are multiples of 16 ----------------------------
//
// One workgroup of G groups of 256 threads (4 wavefronts each) marches the z planes of a 16 x 16
// column tile of a block: group g owns components g, g + G, g + 2 G, ..., and thread (tx, ty) of
// a group the tile's column (i, j) = (tx, ty). Three steps a plane, a barrier after each:
//   1. the last plane's update: flux divergence, RK averaging and update, the output and the
//      same-level ghost copies; then the normal velocities' states in the plane's cells (u along
//      x, v along y, w of the cell above) and those of the cells beyond the tile's rows and
//      columns, every component, from the plane staged in LDS;
//   2. the face coefficients (a, b) of HllCoef of the three directions, every x and y face
//      once; the last plane's derived field and CFL maximum;
//   3. the fluxes, a group's components one after another. x: own cell's stencil from LDS, the
//      neighbouring cells' states by DPP row shifts (a row of 16 cells is a 16-lane DPP row),
//      flux = a ql + b qr; y: the same with the thread mapping transposed (thread (tx, ty)
//      takes cell i = ty, j = tx, so a column is a row too); both differences to LDS. z: each
//      thread keeps U of its column at planes kk - 1, kk + 1, kk + 2 and kk + 3 in registers (kk
//      itself is in LDS), so the z stencil of the cell above needs no load; the high z
//      face's flux becomes the next plane's low face flux. Before them the next plane is
//      staged in the other LDS buffer (the tile's own cells from the rings, 3-cell x and y
//      halos from HBM) and the loads that the next plane needs are issued.
// The divergence adds x, y and z in the order of FluxDivHelper (update.hpp:43-57). A velocity's
// flux carries a factor 1/2 against the scalars': it is applied to the face area (an exact
// product), and corrected fluxes of velocities are doubled where they are read. Each U element
// is read from HBM once per workgroup (plus the halos and the segment's first planes), and face
// states and fluxes never leave the CU.
//
// Bound: FP64 issue, at 59% of it (176 M wave64 instructions in a launch of 488 us, 11
// components, at 4 cycles each and 2.4 GHz; 2 wavefronts per SIMD from one workgroup a CU; the
// barriers and the memory waits of the staging show). Two groups a tile, since one thread per
// column with 8 components and more needs over 256 VGPRs: spilled registers cost most here, as
// each reload waits for every load and store in flight. (Four groups of 128 VGPRs spill and took
// 1105 us for the cycle below.) Measured, cycles of 128^3 cells in 32^3 blocks: 980 us with 11
// components (fluxes, update and exchange as launches of their own: 2365), 653 us with 7
// (1538); 16^3 blocks with 11 components: 186 us on 64 blocks, 238 by one thread per column.
struct TileShape {
  int n0, n1, n2;     // interior cells of a block
  int e0;             // brick row pitch
  int sz, cs;         // brick plane and component strides
  int tx, tiles;      // tiles per block along x, and in all
};

template <int V, int RECON>
__global__ void __launch_bounds__(512, 2)
    TileSweepKernel(const double *__restrict__ U, const double *base, double *out,
                    double *__restrict__ derived, double *__restrict__ partial,
                    const BlockCoefs *__restrict__ coef, TileShape S, int nblocks, double beta,
                    const double *__restrict__ dtvar, const int *__restrict__ fover,
                    const double *__restrict__ fcor, const int *__restrict__ push,
                    const int *__restrict__ list) {
  constexpr int N = 16, NG = 4, G = 2, NT = 256 * G, NC = (V + G - 1) / G;
  constexpr int H = 3;             // halo of the staged plane
  constexpr int PW = N + 2 * H;    // staged rows / columns
  constexpr int PP = PW + 1;       // row pitch (odd, fewer bank conflicts on column reads)
  constexpr int PS = PW * PP;      // one component of the staged plane
  constexpr int SP = N + 1;        // pitch of the difference tiles and of the face rows
  constexpr int NX = V * N * 2;    // beyond-the-row states of one direction
  constexpr int NH = V * 12 * N;   // halo cells of one staged plane (all components)
  constexpr int QH = (NH + NT - 1) / NT;  // halo cells per thread
  // a y difference tile of its own where the LDS (160 KiB) holds it beside the two staged
  // planes, up to 11 components; without it the y pass waits for the x differences and adds
  constexpr int kLds = 2 * V * PS + 2 * NX + V * N * SP + 6 * N * SP + 4 * V * N + 16;
  static_assert(8 * kLds <= 160 * 1024);
  constexpr bool SY = 8 * (kLds + V * N * SP) <= 160 * 1024;
  constexpr int gW = 0, mW = 1;  // the z velocity's group and place in it
  constexpr int gD = 1;          // the group of the derived field and CFL
  __shared__ double pl[2 * V * PS];  // [plane parity][n][j + H][i + H]
  __shared__ double ext[2 * NX];     // [dir][n][line][side]: side 0 ql of cell -1, 1 qr of cell N
  __shared__ double sd[(SY ? 2 : 1) * V * N * SP];  // x (+ y) differences [n][j][i], then the new
                                                    // state; the y differences
  __shared__ double ca[3][N * SP], cb[3][N * SP];  // face coefficients [dir][line][face]
  __shared__ double fxy[2 * V * 2 * N];  // corrected x / y face fluxes of the plane,
                                         // [dir][n][side][line] (tiles with such faces)
  __shared__ double wmax[NT / 64];
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int grp = wave >> 2, wrow = wave & 3;  // uniform: a wavefront takes rows 4 wrow .. + 3
  const int tx = threadIdx.x % N, ty = (threadIdx.x / N) % N;
  const bool last = (NC - 1) * G + grp < V;  // the group has a component at m = NC - 1
  const int nc = last ? NC : NC - 1;
  const double bdt = beta * dtvar[0];
  const double w2 = 1.0 - beta;
  const bool same_base = base == U;
  const int n0 = S.n0, n1 = S.n1, n2 = S.n2, e0 = S.e0, tilesx = S.tx, tiles = S.tiles;
  const std::int64_t cs = S.cs, sz = S.sz;
  const unsigned col = 8u * static_cast<unsigned>((NG + ty) * e0 + NG + tx);  // byte offset
  const int own = (ty + H) * PP + tx + H;  // own cell in the staged plane
  const int osd = ty * SP + tx;            // own cell in the difference tile
  // halo cell q of this thread (q < QH): byte offset from the tile's plane in the brick (the
  // component's included) and place in the staged plane; cells past the last repeat it (loads
  // are unconditional, so the compiler can count them in its memory waits)
  unsigned hoff[QH];
  int hloc[QH];
#pragma unroll
  for (int q = 0; q < QH; ++q) {
    const int t = DMinI(static_cast<int>(threadIdx.x) + q * NT, NH - 1);
    const int n = t / (12 * N), r = t % (12 * N);
    int i, j;
    if (r < 6 * N) {  // y strips: rows -3 .. -1 and N .. N + 2, all interior columns
      const int yy = r / N;
      i = r % N;
      j = yy < 3 ? yy - 3 : N + yy - 3;
    } else {          // x strips: all interior rows, columns -3 .. -1 and N .. N + 2
      const int qq = r - 6 * N;
      j = qq / 6;
      const int c = qq % 6;
      i = c < 3 ? c - 3 : N + c - 3;
    }
    hoff[q] = 8u * static_cast<unsigned>(n * static_cast<int>(cs) + (NG + j) * e0 + NG + i);
    hloc[q] = n * PS + (j + H) * PP + i + H;
  }
  double smax = 0.0;  // largest sum of |u| / dx of the new states
  const std::int64_t T = static_cast<std::int64_t>(nblocks) * tiles * n2;
  std::int64_t pnext = T * blockIdx.x / gridDim.x;
  const std::int64_t pend = T * (blockIdx.x + 1) / gridDim.x;
  while (pnext < pend) {
    // the planes of the launch run over its blocks' tiles in order: all blocks, or the listed
    const int unit = static_cast<int>(pnext / n2);
    const int k0 = static_cast<int>(pnext - static_cast<std::int64_t>(unit) * n2);
    const int k1 = static_cast<int>(pend - pnext < n2 - k0 ? k0 + (pend - pnext) : n2);
    pnext += k1 - k0;
    const int bi = unit / tiles, tile = unit - bi * tiles;
    const int b = list ? list[bi] : bi;
    const int tj = tile / tilesx, ti = tile - tj * tilesx;
    const bool lox = ti == 0, hix = ti == tilesx - 1, loy = tj == 0, hiy = (tj + 1) * N == n1;
    const int toff = tj * N * e0 + ti * N;  // the tile within a plane
    const std::int64_t at = static_cast<std::int64_t>(b) * V * cs + toff;
    const BlockCoefs &C = coef[b];
    const double ivol = 1.0 / C.vol;
    const double ax = C.area[0], ay = C.area[1], az = C.area[2];
    const double ix = 1.0 / C.dx[0], iy = 1.0 / C.dx[1], iz = 1.0 / C.dx[2];
    // the block's same-level neighbours, one per lane, read by readlane: a load in the middle
    // of a plane would be waited for
    const int nbr = push ? push[27 * b + DMinI(static_cast<int>(threadIdx.x) % 64, 26)] : -1;
    // the block's face images of corrected fluxes, where the tile touches the face
    const int *fo = fover ? fover + 6 * b : nullptr;
    const int ox0 = fo && lox ? fo[0] : -1, ox1 = fo && hix ? fo[1] : -1;
    const int oy0 = fo && loy ? fo[2] : -1, oy1 = fo && hiy ? fo[3] : -1;
    const int oz0 = fo ? fo[4] : -1, oz1 = fo ? fo[5] : -1;
    const bool fixed = ox0 >= 0 || ox1 >= 0 || oy0 >= 0 || oy1 >= 0;
    const int zimg = ti * N + tx + (tj * N + ty) * n0;  // this column in a z face's image
    const int kk0 = NG + k0;
    auto plane = [=](auto *f, int n, int kk) __attribute__((always_inline)) {
      return Glob(f) + (at + n * cs + kk * sz);  // the tile's plane kk of component n
    };
    auto load = [=](const __attribute__((address_space(1))) double *p, unsigned off)
        __attribute__((always_inline)) {
      return *reinterpret_cast<const __attribute__((address_space(1))) double *>(
          reinterpret_cast<const __attribute__((address_space(1))) char *>(p) + off);
    };
    auto store = [=](__attribute__((address_space(1))) double *p, unsigned off, double v)
        __attribute__((always_inline)) {
      *reinterpret_cast<__attribute__((address_space(1))) double *>(
          reinterpret_cast<__attribute__((address_space(1))) char *>(p) + off) = v;
    };
    // copies of value m of v, plane k, into the same-level neighbours' ghosts: a cell within NG
    // of a face of the block is a ghost cell of the neighbours across that face, edge or
    // corner (push[27 b + direction]), at its index shifted by the block size along each
    // crossed dimension. Every strip that a cell can lie in is uniform in the wavefront but for
    // the x one, so each neighbour's copies are stores at one base address.
    auto copies = [=](const double (&v)[NC], int k, int tx, unsigned col)
        __attribute__((always_inline)) {
      const int ly = loy && wrow == 0 ? -1 : hiy && wrow == 3 ? 1 : 0;
      const int lz = k < NG ? -1 : k >= n2 - NG ? 1 : 0;
      for (int sz_ = 0; sz_ <= (lz ? 1 : 0); ++sz_)
        for (int sy = 0; sy <= (ly ? 1 : 0); ++sy)
          for (int dx = lox ? -1 : 0; dx <= (hix ? 1 : 0); ++dx) {
            const int dy = sy ? ly : 0, dz = sz_ ? lz : 0;
            if (!(dx | dy | dz)) continue;
            const int g = __builtin_amdgcn_readlane(nbr, (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1));
            if (g < 0) continue;
            const std::int64_t to = static_cast<std::int64_t>(g - b) * V * cs - dz * n2 * sz -
                                    dy * n1 * e0 - dx * n0;
            if (dx == 0 || (dx < 0 ? tx < NG : tx >= N - NG)) {
#pragma unroll
              for (int m = 0; m < NC; ++m) {
                if (m == NC - 1 && !last) break;
                store(plane(out, G * m + grp, NG + k) + to, col, v[m]);
              }
            }
          }
    };
    // CFL maximum and derived field of plane k from the new states in sd (group gD)
    auto gather = [=](int k, double s, int osd, unsigned col) __attribute__((always_inline)) {
      const double v0 = sd[osd], v1 = sd[N * SP + osd], v2 = sd[2 * N * SP + osd],
                   v3 = sd[3 * N * SP + osd];
      const double sp = fabs(v0) * ix + fabs(v1) * iy + fabs(v2) * iz;
      if (derived)
        store(Glob(derived) + (static_cast<std::int64_t>(b) * cs + toff + (NG + k) * sz), col,
              0.5 * v3 * (v0 * v0 + v1 * v1 + v2 * v2));
      return DMax(s, sp);
    };
    // corrected fluxes of plane k's x and y faces (only tiles next to finer blocks), staged in
    // LDS so that the loops below issue no conditional load
    auto corrected = [=](int k, int tid) __attribute__((always_inline)) {
      for (int t = tid; t < 2 * V * 2 * N; t += NT) {
        const int dir = t / (2 * V * N), r = t % (2 * V * N);
        const int n = r / (2 * N), side = (r / N) & 1, line = r % N;
        const int o = dir == 0 ? (side ? ox1 : ox0) : (side ? oy1 : oy0);
        const int rows = dir == 0 ? n1 : n0;
        const int a = (dir == 0 ? tj : ti) * N + line;
        fxy[t] = o >= 0 ? (n < 3 ? 2.0 : 1.0) * fcor[o + a + (k + n * n2) * rows] : 0.0;
      }
    };
    // ---- the segment's first plane kk0, staged; the rings
    double hv[QH], r0[NC], r2[NC], r3[NC], r4[NC];
    {
      double *const to = pl + (k0 & 1) * V * PS;
#pragma unroll
      for (int q = 0; q < QH; ++q) hv[q] = load(plane(U, 0, kk0), hoff[q]);
      double own_u[NC];
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        if (m == NC - 1 && !last) break;
        const int n = G * m + grp;
        r0[m] = load(plane(U, n, kk0 - 1), col);
        own_u[m] = load(plane(U, n, kk0), col);
        r2[m] = load(plane(U, n, kk0 + 1), col);
        r3[m] = load(plane(U, n, kk0 + 2), col);
        r4[m] = load(plane(U, n, kk0 + 3), col);
      }
#pragma unroll
      for (int q = 0; q < QH; ++q) to[hloc[q]] = hv[q];
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        if (m == NC - 1 && !last) break;
        to[(G * m + grp) * PS + own] = own_u[m];
      }
    }
#pragma unroll
    for (int q = 0; q < QH; ++q) hv[q] = load(plane(U, 0, kk0 + 1), hoff[q]);
    // ---- z state at plane kk0: ql of cell kk0 (zl) and the flux of face kk0 - 1/2 (zf); the
    // z velocity gives the face coefficients
    double zl[NC], zf[NC];
    {
      auto ends = [=](int n, double &below, double &qr, double &ql)
          __attribute__((always_inline)) {
        double x;
        double q[6];
#pragma unroll
        for (int s = 0; s < 6; ++s) q[s] = load(plane(U, n, kk0 - 3 + s), col);
        FastStates(RECON, q[0], q[1], q[2], q[3], q[4], below, x);
        FastStates(RECON, q[1], q[2], q[3], q[4], q[5], ql, qr);
      };
      double wb, wr, wl, za, zb;  // the z velocity's
      ends(2, wb, wr, wl);
      HllCoef(wb, wr, za, zb);
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        if (m == NC - 1 && !last) break;
        const int n = G * m + grp;
        double qb = wb, qr = wr, ql = wl;
        if (n != 2) ends(n, qb, qr, ql);
        double f = fma(za, qb, zb * qr);
        if (k0 == 0 && oz0 >= 0)
          f = (n < 3 ? 2.0 : 1.0) * fcor[oz0 + zimg + n * n0 * n1];
        zf[m] = f;
        zl[m] = ql;
        // one component at a time, as in the z fluxes
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    double bv[NC], dz[NC];  // of the plane in hand: base state, z difference
    // the update of plane k, whose differences are complete
    auto finish = [&](int k, int tx, int osd, unsigned col) __attribute__((always_inline)) {
      double v[NC];
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        if (m == NC - 1 && !last) break;
        const int n = G * m + grp;
        double &slot = sd[n * N * SP + osd];
        double du = slot;
        if (SY) du = du + sd[V * N * SP + n * N * SP + osd];
        du = du + dz[m];
        const double dudt = -du * ivol;
        const double avg = beta * r0[m] + w2 * (same_base ? r0[m] : bv[m]);
        v[m] = 1.0 * avg + bdt * dudt;
        if (n < 4) slot = v[m];  // for the derived field and the CFL
        store(plane(out, n, NG + k), col, v[m]);
      }
      if (push) copies(v, k, tx, col);
    };
    __syncthreads();
    for (int k = k0; k < k1; ++k) {
      const int kk = NG + k;
      // the thread's place, formed anew for each plane: addresses derived from it would
      // otherwise be hoisted out of the loop and take the registers of the stencils (a
      // spilled register costs more than its reload: every reload waits for all the loads
      // and stores in flight)
      const int tid = Opaque(static_cast<int>(threadIdx.x));
      const int tx = tid % N, ty = (tid / N) % N;
      const int own = (ty + H) * PP + tx + H, osd = ty * SP + tx;
      const unsigned col = 8u * static_cast<unsigned>((NG + ty) * e0 + NG + tx);
      const double *const P = pl + (k & 1) * V * PS;
      const double *const crow = P + own;                     // own cell
      const double *const ccol = P + (tx + H) * PP + ty + H;  // cell i = ty, j = tx
      // ---- 1.
      // the next plane into the other buffer first (also past the block's last plane: ghost
      // planes): every load in flight is waited for here, before the stores below, since a
      // later wait would count these too
      // (as a lambda, which the compiler schedules better: the same lines in place cost 0.7% of
      // the cycle below)
      auto stage = [&](double *to) __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < NC; ++m) {
          if (m == NC - 1 && !last) break;
          to[(G * m + grp) * PS + own] = r2[m];
        }
#pragma unroll
        for (int q = 0; q < QH; ++q) to[hloc[q]] = hv[q];
      };
      stage(pl + ((k + 1) & 1) * V * PS);
      if (k > k0) finish(k - 1, tx, osd, col);
      if (fixed) corrected(k, tid);
      double vl, vr, wl = 0.0, wr = 0.0;
      {
        const double *c = grp == 0 ? crow : ccol + PS;
        const int st = grp == 0 ? 1 : PP;
        FastStates(RECON, c[-2 * st], c[-st], c[0], c[st], c[2 * st], vl, vr);
      }
      if (grp == gW)
        FastStates(RECON, r0[mW], crow[2 * PS], r2[mW], r3[mW], r4[mW], wl, wr);
      for (int t = tid ^ (NT / 2); t < 2 * NX; t += NT) {
        const int dir = t / NX, r = t % NX;
        const int n = r / (2 * N), q = r % (2 * N);
        const int line = q >> 1, side = q & 1;
        const int cell = side ? N : -1;
        const int st = dir ? PP : 1;
        const double *c = P + n * PS + (dir ? (cell + H) * PP + line + H
                                            : (line + H) * PP + cell + H);
        double ql, qr;
        FastStates(RECON, c[-2 * st], c[-st], c[0], c[st], c[2 * st], ql, qr);
        ext[t] = side ? qr : ql;
      }
      __syncthreads();
      // ---- 2. [line][face]: the low face of every cell and the high face of the last
      {
        const double *e = ext + grp * (NX + 2 * N) + ty * 2;
        const double lm = FromLeft16(vl, e[0]);
        double a, bb;
        HllCoef(lm, vr, a, bb);
        ca[grp][osd] = a;
        cb[grp][osd] = bb;
        if (tx == N - 1) {
          HllCoef(vl, e[1], a, bb);
          ca[grp][osd + 1] = a;
          cb[grp][osd + 1] = bb;
        }
      }
      if (grp == gW) {
        double a, bb;
        HllCoef(zl[mW], wr, a, bb);
        ca[2][osd] = a;
        cb[2][osd] = bb;
      }
      if (k > k0 && grp == gD) smax = gather(k - 1, smax, osd, col);
      __syncthreads();
      // ---- 3.
      // x: own cell (tx, ty), differences to sd[n][ty][tx]
      {
#pragma unroll 1
        for (int m = 0; m < nc; ++m) {
          const int n = G * m + grp;
          double ql = vl, qr = vr;
          if (n != 0) {
            const double *c = crow + n * PS;
            FastStates(RECON, c[-2], c[-1], c[0], c[1], c[2], ql, qr);
          }
          const double e = ext[(n * N + ty) * 2 + (tx == N - 1)];
          double fl = fma(ca[0][osd], FromLeft16(ql, e), cb[0][osd] * qr);
          double fh = fma(ca[0][osd + 1], ql, cb[0][osd + 1] * FromRight16(qr, e));
          if (fixed) {
            if (tx == 0 && ox0 >= 0) fl = fxy[(n * 2 + 0) * N + ty];
            if (tx == N - 1 && ox1 >= 0) fh = fxy[(n * 2 + 1) * N + ty];
          }
          const double A = n < 3 ? 0.5 * ax : ax;
          sd[n * N * SP + osd] = A * fh - A * fl;
        }
      }
      if (!SY) __syncthreads();  // the x differences are in the tile
      // the loads that the next plane needs (indices in range also past the block's last
      // plane: ghost planes); before the x fluxes they would take registers from them
#pragma unroll
      for (int q = 0; q < QH; ++q) hv[q] = load(plane(U, 0, kk + 2), hoff[q]);
      double r5[NC];
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        if (m == NC - 1 && !last) break;
        r5[m] = load(plane(U, G * m + grp, kk + 4), col);
      }
      // y: cell i = ty, j = tx, differences to the y tile or added to sd[n][j][i]
      {
#pragma unroll 1
        for (int m = 0; m < nc; ++m) {
          const int n = G * m + grp;
          double ql = vl, qr = vr;
          if (n != 1) {
            const double *c = ccol + n * PS;
            FastStates(RECON, c[-2 * PP], c[-PP], c[0], c[PP], c[2 * PP], ql, qr);
          }
          const double e = ext[NX + (n * N + ty) * 2 + (tx == N - 1)];
          double fl = fma(ca[1][osd], FromLeft16(ql, e), cb[1][osd] * qr);
          double fh = fma(ca[1][osd + 1], ql, cb[1][osd + 1] * FromRight16(qr, e));
          if (fixed) {
            if (tx == 0 && oy0 >= 0) fl = fxy[((V + n) * 2 + 0) * N + ty];
            if (tx == N - 1 && oy1 >= 0) fh = fxy[((V + n) * 2 + 1) * N + ty];
          }
          const double A = n < 3 ? 0.5 * ay : ay;
          const int at_y = n * N * SP + tx * SP + ty;
          if (SY)
            sd[V * N * SP + at_y] = A * fh - A * fl;
          else
            sd[at_y] = sd[at_y] + (A * fh - A * fl);
        }
      }
#pragma unroll
      for (int m = 0; m < NC; ++m) {
        if (m == NC - 1 && !last) break;
        bv[m] = same_base ? 0.0 : load(plane(base, G * m + grp, kk), col);
      }
      // z: the cell above (kk + 1) from the ring; its low face closes this cell
      {
        const double za = ca[2][osd], zb = cb[2][osd];
        const bool top = k == n2 - 1 && oz1 >= 0;
        const int zimg = ti * N + tx + (tj * N + ty) * n0;
#pragma unroll
        for (int m = 0; m < NC; ++m) {
          if (m == NC - 1 && !last) break;
          const int n = G * m + grp;
          const double uo = crow[n * PS];
          double ql = wl, qr = wr;
          if (n != 2) FastStates(RECON, r0[m], uo, r2[m], r3[m], r4[m], ql, qr);
          double fh = fma(za, zl[m], zb * qr);
          if (top) {  // only here a load: waited for inside the branch
            fh = (n < 3 ? 2.0 : 1.0) * fcor[oz1 + zimg + n * n0 * n1];
            asm volatile("" : "+v"(fh));
          }
          const double A = n < 3 ? 0.5 * az : az;
          dz[m] = A * fh - A * zf[m];
          zf[m] = fh;
          zl[m] = ql;
          // one component at a time: interleaving the reconstructions needs more registers
          // than the budget holds
          __builtin_amdgcn_sched_barrier(0);
          r0[m] = uo;  // the ring moves up one plane
          r2[m] = r3[m];
          r3[m] = r4[m];
          r4[m] = r5[m];
        }
      }
      __syncthreads();
    }
    finish(k1 - 1, tx, osd, col);
    __syncthreads();
    if (grp == gD) smax = gather(k1 - 1, smax, osd, col);
    __syncthreads();  // sd and the staged planes are free for the next segment
  }
  if (!partial) return;
  for (int off = 32; off > 0; off >>= 1) smax = DMax(smax, __shfl_xor(smax, off, 64));
  if ((threadIdx.x & 63) == 0) wmax[wave] = smax;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = wmax[0];
#pragma unroll
    for (int w = 1; w < NT / 64; ++w) v = DMax(v, wmax[w]);
    partial[blockIdx.x] = DMin(DBL_MAX, 1.0 / v);
  }
}
}  // namespace

// 16^3 blocks of at most 7 components: one thread per column, of which two workgroups fit a
// CU's LDS and registers; from 8 on only one fits and the tile form is the faster. Cycles by this form
// and by the tile form, WENO5: 7 components 61 / 69 us on 8 blocks, 86 / 117 on 27, 135 / 144 on 64, 396 /
// 363 on 216, 729 / 982 on 512, 1723 / 1916 on 960 refined ones; 4 components 46 / 47, 60 / 76, 86 / 95, 215 /
// 234, 446 / 534, 1013 / 1121. The linear reconstruction gains more (7 components, 64 blocks 83 / 106).
static bool RingSweep(const Topology &t, int V) {
  const Extent &f = t.fine;
  return f.n[0] == 16 && f.n[1] == 16 && f.n[2] == 16 && V <= 7;
}

// Blocks of the tile sweep: x and y sizes in whole 16-cell tiles, z any size whose low and
// high ghost strips do not meet, 4 ghosts; a block's components within 32-bit byte offsets.
bool BurgersTileSweep(const Topology &t, int V) {
  const Extent &f = t.fine;
  return t.ndim == 3 && f.n[0] % 16 == 0 && f.n[1] % 16 == 0 && f.n[2] >= 8 && f.g[0] == 4 &&
         f.g[1] == 4 && f.g[2] == 4 && V >= 4 && V <= 13 &&
         f.cells() * V < (std::int64_t(1) << 29);
}

std::int64_t BurgersTilePlanes(const Topology &t) {
  const Extent &f = t.fine;
  return static_cast<std::int64_t>(t.blocks.size()) * (f.n[0] / 16) * (f.n[1] / 16) * f.n[2];
}

bool BurgersSweepTuned(const Topology &t, int V) {
  return !BurgersTileSweep(t, V) || RingSweep(t, V);
}

bool BurgersSweepSupported(const Topology &t, int V) {
  return BurgersTileSweep(t, V) || (ReconFluxSupported(t, V) && t.fine.n[0] == 8);
}

// Workgroups of a kernel resident on the whole device at once (occupancy x compute units).
int ResidentGroups(const void *kernel, int threads) {
  static std::map<const void *, int> cache;
  auto it = cache.find(kernel);
  if (it != cache.end()) return it->second;
  int dev = 0, cus = 0, per = 0;
  if (Failed(hipGetDevice(&dev)) ||
      Failed(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev)) ||
      Failed(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, threads, 0)) ||
      per < 1 || cus < 1)
    return -1;
  cache[kernel] = per * cus;
  return per * cus;
}

pth_status BurgersSweep(const Topology &t, int V, const double *U, const double *base,
                        double *out, double *derived, double *partial, int max_partials,
                        const BlockCoefs *coef, double beta, const double *dtvar, int recon,
                        const FluxCorrection *fc, int waves, int spread, const int *push,
                        int *groups, hipStream_t s, const int *list, int nlist) {
  if (!BurgersSweepSupported(t, V) || waves < 2 || waves > 4 || spread < 1 || spread > 3) {
    SetError("block sweep: unsupported block shape or component count");
    return PTH_FAIL;
  }
  const bool tiled = BurgersTileSweep(t, V);
  if (list && !(tiled && nlist > 0)) {
    SetError("block sweep: block lists need blocks of the tile sweep");
    return PTH_FAIL;
  }
  ProfScope prof("block_sweep", s);
  const int nb = list ? nlist : static_cast<int>(t.blocks.size());
  const int *fover = fc ? fc->dev_face : nullptr;
  const double *fcor = fc ? fc->store : nullptr;
  int grid = 0;
  // a launch takes the resident workgroups divided by spread, at most one plane each
  auto groups_of = [&](const void *kernel, int threads, std::int64_t planes) {
    const int r = ResidentGroups(kernel, threads);
    if (r < 1) SetError("block sweep: occupancy query failed");
    grid = r < 1 ? 0
                 : static_cast<int>(std::min<std::int64_t>(
                       std::min(std::max(r / spread, 1), max_partials), planes));
    return grid > 0;
  };
  if (RingSweep(t, V)) {
    // built for 2 or 3 waves per SIMD
    auto run = [&](auto kernel) {
      if (!groups_of(reinterpret_cast<const void *>(kernel), 256,
                     static_cast<std::int64_t>(nb) * 16))
        return PTH_FAIL;
      PTH_LAUNCH(kernel, dim3(grid), dim3(256), 0, s, U, base, out, derived, partial,
                 coef, nb, beta, dtvar, fover, fcor, push, list);
      return PTH_COMPLETE;
    };
    auto pick = [&](auto v) {
      constexpr int NV = decltype(v)::value;
      if (waves >= 3)
        return recon == 0 ? run(BlockSweep16Kernel<NV, 3, 0>) : run(BlockSweep16Kernel<NV, 3, 1>);
      return recon == 0 ? run(BlockSweep16Kernel<NV, 2, 0>) : run(BlockSweep16Kernel<NV, 2, 1>);
    };
    const pth_status st = V == 4   ? pick(std::integral_constant<int, 4>())
                          : V == 5 ? pick(std::integral_constant<int, 5>())
                          : V == 6 ? pick(std::integral_constant<int, 6>())
                                   : pick(std::integral_constant<int, 7>());
    if (st != PTH_COMPLETE) return PTH_FAIL;
    if (groups) *groups = grid;
    return PTH_COMPLETE;
  }
  if (tiled) {
    TileShape S;
    S.n0 = t.fine.n[0];
    S.n1 = t.fine.n[1];
    S.n2 = t.fine.n[2];
    S.e0 = t.fine.ent(0);
    S.sz = S.e0 * t.fine.ent(1);
    S.cs = S.sz * t.fine.ent(2);
    S.tx = S.n0 / 16;
    S.tiles = S.tx * (S.n1 / 16);
    const std::int64_t planes = static_cast<std::int64_t>(nb) * S.tiles * S.n2;
    auto run = [&](auto kernel, int threads) {
      if (!groups_of(reinterpret_cast<const void *>(kernel), threads, planes)) return PTH_FAIL;
      PTH_LAUNCH(kernel, dim3(grid), dim3(threads), 0, s, U, base, out, derived, partial,
                 coef, S, nb, beta, dtvar, fover, fcor, push, list);
      return PTH_COMPLETE;
    };
    auto pick = [&](auto v) {
      constexpr int NV = decltype(v)::value;
      return recon == 0 ? run(TileSweepKernel<NV, 0>, 512) : run(TileSweepKernel<NV, 1>, 512);
    };
    pth_status st = PTH_FAIL;
#define PTH_TS_CASE(NV)                          \
  case NV:                                       \
    st = pick(std::integral_constant<int, NV>()); \
    break;
    switch (V) {
      PTH_TS_CASE(4)
      PTH_TS_CASE(5)
      PTH_TS_CASE(6)
      PTH_TS_CASE(7)
      PTH_TS_CASE(8)
      PTH_TS_CASE(9)
      PTH_TS_CASE(10)
      PTH_TS_CASE(11)
      PTH_TS_CASE(12)
      PTH_TS_CASE(13)
    }
#undef PTH_TS_CASE
    if (st != PTH_COMPLETE) return PTH_FAIL;
    if (groups) *groups = grid;
    return PTH_COMPLETE;
  }
  if (waves == 2) waves = 3;
#define PTH_SW_LAUNCH_W(NV, W)                                                                \
  {                                                                                           \
    if (!groups_of(reinterpret_cast<const void *>(&BlockSweepKernel<8, 4, NV, W>), 64,         \
                   static_cast<std::int64_t>(nb) * 8))                                        \
      return PTH_FAIL;                                                                        \
    PTH_LAUNCH((BlockSweepKernel<8, 4, NV, W>), dim3(grid), dim3(64), 0, s, U, base,   \
               out, derived, partial, coef, nb, beta, dtvar, recon, fover, fcor, push); \
  }
#define PTH_SW_CASE(NV)                        \
  case NV:                                     \
    if (waves == 4)                            \
      PTH_SW_LAUNCH_W(NV, (NV <= 8 ? 4 : 2))   \
    else                                       \
      PTH_SW_LAUNCH_W(NV, (NV <= 8 ? 3 : 2))   \
    break;
  switch (V) {
    PTH_SW_CASE(4)
    PTH_SW_CASE(5)
    PTH_SW_CASE(6)
    PTH_SW_CASE(7)
    PTH_SW_CASE(8)
    PTH_SW_CASE(9)
    PTH_SW_CASE(10)
    PTH_SW_CASE(11)
    PTH_SW_CASE(12)
    PTH_SW_CASE(13)
  }
#undef PTH_SW_CASE
#undef PTH_SW_LAUNCH_W
  if (groups) *groups = grid;
  return PTH_COMPLETE;
}

pth_status FlxcorDirect(const Topology &t, int V, const FluxCorrection &fc, const double *U,
                        int recon, hipStream_t s) {
  if (fc.host.empty()) return PTH_COMPLETE;
  if (V < 4 || V > 16) {
    SetError("flux correction supports 4 to 16 components");
    return PTH_FAIL;
  }
  ProfScope prof("flxcor_direct", s);
  const Geo G = MakeGeo(t, V);
  const dim3 grid(static_cast<unsigned>(fc.host.size()), (4 * fc.max_cells + 63) / 64);
  const bool ring = BurgersTileSweep(t, V);
#define PTH_FD_CASE(NV)                                                                       \
  case NV:                                                                                    \
    if (ring)                                                                                 \
      PTH_LAUNCH((FlxcorDirectKernel<NV, true>), grid, dim3(64), 0, s, fc.dev, U,     \
                 fc.store, G, recon);                                                 \
    else                                                                                      \
      PTH_LAUNCH((FlxcorDirectKernel<NV, false>), grid, dim3(64), 0, s, fc.dev, U,    \
                 fc.store, G, recon);                                                 \
    break;
  switch (V) {
    PTH_FD_CASE(4)
    PTH_FD_CASE(5)
    PTH_FD_CASE(6)
    PTH_FD_CASE(7)
    PTH_FD_CASE(8)
    PTH_FD_CASE(9)
    PTH_FD_CASE(10)
    PTH_FD_CASE(11)
    PTH_FD_CASE(12)
    PTH_FD_CASE(13)
    PTH_FD_CASE(14)
    PTH_FD_CASE(15)
    PTH_FD_CASE(16)
  }
#undef PTH_FD_CASE
  return PTH_COMPLETE;
}

}  // namespace pth
