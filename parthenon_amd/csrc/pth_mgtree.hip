// Multigrid Poisson solver over MeshData on meshes of any static refinement, any dimension
// and any mix of FixedFace / periodic faces: the general form of MGSolver<u, rhs,
// PoissonEquation> (src/solvers/mg_solver.hpp:73-520) on a hierarchy of block meshes.
//
// Hierarchy (the levels of src/mesh/mesh-gmg.cpp:103-154, finest first):
//   * the leaf mesh itself;
//   * the mesh capped at each coarser refinement level down to the base grid: every block of
//     the capped level whose children exist becomes one block (its children restrict into
//     it, the reference's gmg_restrict_send to gmg_coarser_neighbors), every other block is
//     the same block on both levels (the reference shares those MeshBlocks between its grids:
//     gmg_leaf_neighbors, same_to_same buffers, bvals_utils.hpp:49-63);
//   * below the base grid, the tree levels of the forest (2^d base blocks merge into one, as
//     many times as the forest's root level, forest.cpp:64-105), then levels whose blocks keep
//     their positions and halve their cells (the reference's negative logical levels) while
//     every block size is even, down to one cell per block (one ghost layer on these levels)
//     and two cells per dimension for the level (where the reference's single-tree forest
//     ends with one cell).
// Every level is a full tiling of the domain, so each level's boundary exchange is the leaf
// exchange of that level's mesh (same-level copies, restriction into coarse buffers and
// linear prolongation at fine-coarse faces, FixedFace conditions). The reference's grids
// instead hold only the level's blocks and the coarser leaves beside them
// (two_level_composite, tree.cpp:163-230) and smooth only those; here the unrefined part of
// each level is smoothed as well. The fixed point is the same: the solve stops on the RMS
// residual of the leaf problem, measured with the leaf exchange and PoissonEquation::Ax as in
// AddTasks (mg_solver.hpp:131-158).
//
// Cycle (correction scheme; the reference cycles the full solution, FAS, which gives the same
// iterates for this linear operator in exact arithmetic): on each level, pre-smoothing,
// residual r = b - A x, restriction of r (RestrictAverage) into the coarser level's b with a
// zero initial x there, the coarser cycle, prolongation of its x (ProlongateSharedLinear from
// the coarse cells and their face neighbours, the reference's gmg_prolongate_recv with
// ProResInfo::GetInteriorProlongate, bnd_info.cpp:371-385) added to x, post-smoothing; the
// coarsest level only pre-smooths (mg_solver.hpp:441-448). The smoother is the reference's
// SRJ (stages 1-3 with the Yang & Mittal weights of mg_solver.hpp:312-345), or weighted Jacobi
// with explicit weight and sweep counts. One Jacobi stage (mg_solver.hpp:222-297, 299-311):
// exchange x, t = w (b - (A x - diag x)) / diag + (1 - w) x with the unigrid diagonal of
// PoissonEquation::SetDiagonal (poisson_equation.hpp:86-125), x = t.
//
// Launches. The coarse levels are a few microseconds of work each, so a V-cycle costs what its
// launches cost. A stencil reads a neighbour in another block of the same level from that
// block's interior (a table of face neighbours) and a FixedFace ghost as -u, so a level whose
// blocks all have one size needs no exchange: a smoothing stage is one launch from x to its
// second array, the residual goes straight into the coarser level's b, a correction straight
// from the coarser x. Levels with blocks of different sizes first run the part of the
// exchange that their stencils read: the channels between levels, and the same-level ghosts of
// blocks that restrict them for their coarse neighbours. On the mesh of 568 16^3 blocks (one
// refined level, 8 levels) a V-cycle with its residual norm takes 468 us as a replayed graph;
// with exchange, stage and copy back as launches of their own, 160 of them, it took 1224 us
// and the norm 120. FP64 throughout.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "pth_burgers.hpp"
#include "pth_device.hpp"
#include "pth_internal.hpp"
#include "pth_mgtree.hpp"

namespace pth {
namespace {

constexpr int kWG = 256;
enum { kX = 0, kT = 1, kB = 2, kD = 3 };  // level fields: solution/correction, its second array
                                          // (levels of one block size), right-hand side, face
                                          // field D (3 components)

// A level's blocks for the kernels. face[6 b + 2 d + side]: the same-level block across that
// face, or kFixed (FixedFace-0 boundary), or kGhost (a block of another level: the ghost cell
// holds the exchanged value).
constexpr int kFixed = -1, kGhost = -2;
struct LevelView {
  int n0, n1, n2;     // interior cells of a block
  int e0, p;          // brick row pitch, plane stride
  int first;          // brick offset of the first interior cell
  int per, chunks;    // interior cells of a block, and workgroups over them
  int ndim;
  long long cells;    // brick cells
  const int *face;
};

// 1 / dx^2 per dimension and, for a constant D, 1 / diagonal of a block
struct StageCoef {
  double i2[3], rdiag;
};

struct Local {
  int i, j, k, c;  // cell of a block and its brick offset
};
__device__ __forceinline__ Local At(const LevelView &V, unsigned t) {
  Local q;
  const unsigned r = t / static_cast<unsigned>(V.n0);
  q.i = static_cast<int>(t - r * static_cast<unsigned>(V.n0));
  q.k = static_cast<int>(r / static_cast<unsigned>(V.n1));
  q.j = static_cast<int>(r - static_cast<unsigned>(q.k) * static_cast<unsigned>(V.n1));
  q.c = V.first + q.k * V.p + q.j * V.e0 + q.i;
  return q;
}

// A cell's value and its neighbours' along the active dimensions, [d][low, high]; every load
// unconditional (a FixedFace neighbour reads the cell itself and becomes its negative)
struct Near {
  double u, v[3][2];
};
__device__ __forceinline__ Near LoadNear(const double *__restrict__ x, const LevelView &V, int b,
                                         const Local &q) {
  const double *xb = x + b * V.cells;
  const int *f = V.face + 6 * b;
  Near o;
  o.u = xb[q.c];
  auto side = [&](int at, int n, int st, int lo, int hi, double (&v)[2]) {
    const bool in0 = at > 0, in1 = at < n - 1;
    const long long a0 = in0 || lo == kGhost ? q.c - st
                         : lo >= 0           ? q.c + st * (n - 1) + (lo - b) * V.cells
                                             : q.c;
    const long long a1 = in1 || hi == kGhost ? q.c + st
                         : hi >= 0           ? q.c - st * (n - 1) + (hi - b) * V.cells
                                             : q.c;
    const double x0 = xb[a0], x1 = xb[a1];
    v[0] = !in0 && lo == kFixed ? 0.0 - o.u : x0;
    v[1] = !in1 && hi == kFixed ? 0.0 - o.u : x1;
  };
  side(q.i, V.n0, 1, f[0], f[1], o.v[0]);
  if (V.ndim > 1) side(q.j, V.n1, V.e0, f[2], f[3], o.v[1]);
  if (V.ndim > 2) side(q.k, V.n2, V.p, f[4], f[5], o.v[2]);
  return o;
}

// A x at a cell, D on the cell's faces from the face field Df (the block's 3-component brick,
// component d = D on the lower face along d) or the constant D; *diag is the operator's
// diagonal (SetDiagonal). Inverse squares of the cell widths in place of divisions: the values
// are the reference's to rounding.
__device__ __forceinline__ double ApplyA(const Near &o, const LevelView &V, const StageCoef &S,
                                         double D, const double *Df, int c, double alpha,
                                         double *diag) {
  double ax = -alpha * o.u, dg = -alpha;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    if (d >= V.ndim) break;
    const int st = d == 0 ? 1 : d == 1 ? V.e0 : V.p;
    const double Dl = Df ? Df[d * V.cells + c] : D, Dh = Df ? Df[d * V.cells + c + st] : D;
    ax += (Dl * (o.v[d][0] - o.u) - Dh * (o.u - o.v[d][1])) * S.i2[d];
    dg -= (Dl + Dh) * S.i2[d];
  }
  *diag = dg;
  return ax;
}

// The same in the operation order of CalculateFluxes + FluxMultiplyMatrix
// (poisson_equation.hpp:131-205), for the residual that the solve reports and stops on.
__device__ __forceinline__ double ApplyExact(const Near &o, const LevelView &V,
                                             const BlockCoefs &C, double D, const double *Df,
                                             int c, double alpha) {
  double ax = -alpha * o.u;
  const double f1l = (Df ? Df[c] : D) / C.dx[0] * (o.v[0][0] - o.u);
  const double f1r = (Df ? Df[c + 1] : D) / C.dx[0] * (o.u - o.v[0][1]);
  ax += (f1l - f1r) / C.dx[0];
  if (V.ndim > 1) {
    const double f2l = (Df ? Df[V.cells + c] : D) * (o.v[1][0] - o.u) / C.dx[1];
    const double f2r = (Df ? Df[V.cells + c + V.e0] : D) * (o.u - o.v[1][1]) / C.dx[1];
    ax += (f2l - f2r) / C.dx[1];
  }
  if (V.ndim > 2) {
    const double f3l = (Df ? Df[2 * V.cells + c] : D) * (o.v[2][0] - o.u) / C.dx[2];
    const double f3r = (Df ? Df[2 * V.cells + c + V.p] : D) * (o.u - o.v[2][1]) / C.dx[2];
    ax += (f3l - f3r) / C.dx[2];
  }
  return ax;
}

// One Jacobi stage out = x + w (b - A x) / diag; ZERO: from x = 0, which is not read.
template <bool ZERO>
__global__ void __launch_bounds__(kWG)
    StageKernel(const double *__restrict__ x, const double *__restrict__ b,
                double *__restrict__ out, LevelView V, const StageCoef *__restrict__ coef,
                double D, const double *__restrict__ Df, double alpha, double w) {
  const unsigned L = XcdRemap(blockIdx.x, gridDim.x);
  const int blk = static_cast<int>(L / static_cast<unsigned>(V.chunks));
  const int t = static_cast<int>(L % static_cast<unsigned>(V.chunks)) * kWG +
                static_cast<int>(threadIdx.x);
  if (t >= V.per) return;
  const Local q = At(V, t);
  const StageCoef &S = coef[blk];
  const double *Db = Df ? Df + blk * 3 * V.cells : nullptr;
  const long long c = blk * V.cells + q.c;
  Near o{};
  if (!ZERO) o = LoadNear(x, V, blk, q);
  double diag;
  const double r = b[c] - ApplyA(o, V, S, D, Db, q.c, alpha, &diag);
  out[c] = o.u + w * (Df ? r / diag : r * S.rdiag);
}

// Residual of a level into the coarser level's right-hand side. The first nchild records are
// blocks whose residual is averaged over 2^ndim cells (RestrictAverage) into octant o of block
// cb; the others are the same block on both levels.
struct Xfer {
  int fb, cb;
  int o[3];
  int child;
};
__global__ void __launch_bounds__(kWG)
    ResidualDownKernel(const double *__restrict__ x, const double *__restrict__ b, LevelView V,
                       const StageCoef *__restrict__ coef, double D,
                       const double *__restrict__ Df, double alpha, double *__restrict__ bc,
                       LevelView C, const Xfer *__restrict__ recs, int nchild, int cchunks) {
  const unsigned L = XcdRemap(blockIdx.x, gridDim.x);
  const bool child = L < static_cast<unsigned>(nchild * cchunks);
  const unsigned M = child ? L : L - static_cast<unsigned>(nchild * cchunks);
  const unsigned ch = static_cast<unsigned>(child ? cchunks : V.chunks);
  const Xfer R = recs[M / ch + (child ? 0u : static_cast<unsigned>(nchild))];
  const int t = static_cast<int>(M % ch) * kWG + static_cast<int>(threadIdx.x);
  const StageCoef &S = coef[R.fb];
  const double *Db = Df ? Df + R.fb * 3 * V.cells : nullptr;
  const double *bb = b + R.fb * V.cells;
  double diag;
  if (!child) {
    if (t >= V.per) return;
    const Local q = At(V, t);
    bc[R.cb * C.cells + C.first + q.k * C.p + q.j * C.e0 + q.i] =
        bb[q.c] - ApplyA(LoadNear(x, V, R.fb, q), V, S, D, Db, q.c, alpha, &diag);
    return;
  }
  const int s1 = V.ndim > 1 ? 2 : 1, s2 = V.ndim > 2 ? 2 : 1;
  const int m0 = V.n0 / 2, m1 = V.n1 / s1, m2 = V.n2 / s2;
  if (t >= m0 * m1 * m2) return;
  const int I = t % m0, J = t / m0 % m1, K = t / m0 / m1;
  double sum = 0.0;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      if (a >= s2 || e >= s1) continue;
      double pair[2];
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        Local q;
        q.i = 2 * I + f;
        q.j = s1 * J + e;
        q.k = s2 * K + a;
        q.c = V.first + q.k * V.p + q.j * V.e0 + q.i;
        pair[f] = bb[q.c] - ApplyA(LoadNear(x, V, R.fb, q), V, S, D, Db, q.c, alpha, &diag);
      }
      sum += pair[0] + pair[1];
    }
  bc[R.cb * C.cells + C.first + (R.o[2] * m2 + K) * C.p + (R.o[1] * m1 + J) * C.e0 +
     R.o[0] * m0 + I] = sum * (V.ndim == 3 ? 0.125 : V.ndim == 2 ? 0.25 : 0.5);
}

// The coarser level's x added to a level's: prolongated (ProlongateSharedLinear: from the coarse
// cell and its neighbour on the fine cell's side along each dimension, the terms grouped like
// pr_ops.hpp:261-283) into child blocks, as it is into blocks that are the same on both.
__global__ void __launch_bounds__(kWG)
    ProlongAddKernel(double *__restrict__ x, LevelView V, const double *__restrict__ xc,
                     LevelView C, const Xfer *__restrict__ recs) {
  const unsigned L = XcdRemap(blockIdx.x, gridDim.x);
  const Xfer R = recs[L / static_cast<unsigned>(V.chunks)];
  const int t = static_cast<int>(L % static_cast<unsigned>(V.chunks)) * kWG +
                static_cast<int>(threadIdx.x);
  if (t >= V.per) return;
  const Local q = At(V, t);
  double *xf = x + R.fb * V.cells + q.c;
  if (!R.child) {
    *xf = *xf + xc[R.cb * C.cells + C.first + q.k * C.p + q.j * C.e0 + q.i];
    return;
  }
  const int fi[3] = {q.i, q.j, q.k}, n[3] = {V.n0, V.n1, V.n2};
  int at[3], odd[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const bool on = d < V.ndim;
    odd[d] = on ? fi[d] & 1 : 0;
    at[d] = on ? R.o[d] * (n[d] / 2) + (fi[d] >> 1) : fi[d];
  }
  Local cq;
  cq.i = at[0];
  cq.j = at[1];
  cq.k = at[2];
  cq.c = C.first + cq.k * C.p + cq.j * C.e0 + cq.i;
  const Near o = LoadNear(xc, C, R.cb, cq);
  double g[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int d = 0; d < 3; ++d)
    if (d < V.ndim) g[d] = 0.25 * (odd[d] ? o.v[d][1] - o.u : o.u - o.v[d][0]);
  const double s0 = odd[0] ? 1.0 : -1.0;
  const double s1 = odd[0] == odd[1] ? 1.0 : -1.0, s2 = odd[0] == odd[2] ? 1.0 : -1.0;
  *xf = *xf + (o.u + s0 * ((g[0] + s1 * g[1]) + s2 * g[2]));
}

template <int WG>
__device__ __forceinline__ double GroupSum(double v) {
  __shared__ double w[WG / 64];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int q = 0; q < WG / 64; ++q) s += w[q];
  return s;
}

// Per-workgroup sums of the squared residual of every cell (fixed order, so every call gives
// the same bits), then their sum.
__global__ void __launch_bounds__(kWG)
    ResidualNormKernel(const double *__restrict__ x, const double *__restrict__ b, LevelView V,
                       const BlockCoefs *__restrict__ coef, double D,
                       const double *__restrict__ Df, double alpha,
                       double *__restrict__ partial) {
  const unsigned L = XcdRemap(blockIdx.x, gridDim.x);
  const int blk = static_cast<int>(L / static_cast<unsigned>(V.chunks));
  const int t = static_cast<int>(L % static_cast<unsigned>(V.chunks)) * kWG +
                static_cast<int>(threadIdx.x);
  double r = 0.0;
  if (t < V.per) {
    const Local q = At(V, t);
    r = 1.0 * b[blk * V.cells + q.c] +
        (-1.0) * ApplyExact(LoadNear(x, V, blk, q), V, coef[blk], D,
                            Df ? Df + blk * 3 * V.cells : nullptr, q.c, alpha);
  }
  const double s = GroupSum<kWG>(r * r);
  if (threadIdx.x == 0) partial[L] = s;
}

constexpr int kSumWG = 1024;
__global__ void __launch_bounds__(kSumWG)
    SumKernel(const double *__restrict__ partial, int n, double *__restrict__ out) {
  double v = 0.0;
  for (int p = threadIdx.x; p < n; p += kSumWG) v += partial[p];
  const double s = GroupSum<kSumWG>(v);
  if (threadIdx.x == 0) *out = s;
}

// Face-field restriction (RestrictAverage on faces) from a block into its coarser-level
// counterpart: coarse face (I, J, K) along direction d, with I in [0, nc_d] and the transverse
// indices in [0, nc), is the mean of the fine faces it covers (2 x 2 in 3-D, 2 in 2-D, one in
// 1-D), fine face index 2 I along d.
struct FaceXfer {
  const double *f;  // the fine block's D brick, component 0
  double *c;        // the coarse block's D brick, component 0
  int o[3];         // octant of the fine block in the coarse one
  int pad;
};
struct FaceGeom {
  int fe0, fe1, ce0, ce1;
  long long fcells, ccells;
  int fg[3], cg[3], nc[3], act[3];
  int ndim;
};

__global__ void __launch_bounds__(kWG)
    FaceRestrictKernel(const FaceXfer *__restrict__ recs, FaceGeom G, long long per_rec,
                       long long total) {
  const long long t = static_cast<long long>(blockIdx.x) * kWG + threadIdx.x;
  if (t >= total) return;
  const FaceXfer R = recs[t / per_rec];
  long long q = t % per_rec;
  int P[3];
  for (int e = 0; e < 3; ++e) P[e] = G.act[e] ? G.nc[e] + 1 : 1;
  const long long per_d = static_cast<long long>(P[0]) * P[1] * P[2];
  const int d = static_cast<int>(q / per_d);
  q %= per_d;
  int I[3];
  I[0] = static_cast<int>(q % P[0]);
  I[1] = static_cast<int>((q / P[0]) % P[1]);
  I[2] = static_cast<int>(q / (static_cast<long long>(P[0]) * P[1]));
  for (int e = 0; e < 3; ++e)
    if (e != d && G.act[e] && I[e] >= G.nc[e]) return;  // padding of a transverse range
  int f[3], n2[3];
  for (int e = 0; e < 3; ++e) {
    f[e] = G.act[e] ? G.fg[e] + 2 * I[e] : 0;
    n2[e] = (e != d && G.act[e]) ? 2 : 1;
  }
  double sum = 0.0;
  for (int kk = 0; kk < n2[2]; ++kk)
    for (int jj = 0; jj < n2[1]; ++jj)
      for (int ii = 0; ii < n2[0]; ++ii)
        sum += R.f[d * G.fcells + (static_cast<long long>(f[2] + kk) * G.fe1 + (f[1] + jj)) *
                                      G.fe0 +
                   (f[0] + ii)];
  const int cnt = n2[0] * n2[1] * n2[2];
  int C[3];
  for (int e = 0; e < 3; ++e) C[e] = G.act[e] ? G.cg[e] + R.o[e] * G.nc[e] + I[e] : 0;
  R.c[d * G.ccells + (static_cast<long long>(C[2]) * G.ce1 + C[1]) * G.ce0 + C[0]] =
      sum / cnt;
}

__global__ void __launch_bounds__(kWG) ZeroKernel(double *__restrict__ x, LevelView V) {
  const int blk = static_cast<int>(blockIdx.x) / V.chunks;
  const int t = (static_cast<int>(blockIdx.x) % V.chunks) * kWG + static_cast<int>(threadIdx.x);
  if (t < V.per) x[blk * V.cells + At(V, t).c] = 0.0;
}

unsigned Grid(long long n) { return static_cast<unsigned>((n + kWG - 1) / kWG); }

// SRJ weights of mg_solver.hpp:312-345 (Yang & Mittal 2017), by dimension and stage count
constexpr double kSrj2[3][2] = {{0.8723, 0.5395}, {1.3895, 0.5617}, {1.7319, 0.5695}};
constexpr double kSrj3[3][3] = {
    {0.9372, 0.6667, 0.5173}, {1.6653, 0.8000, 0.5264}, {2.2473, 0.8571, 0.5296}};

Box Whole(const Extent &e) {
  Box b;
  for (int d = 0; d < 3; ++d) {
    b.lo[d] = 0;
    b.hi[d] = e.ent(d) - 1;
  }
  return b;
}

Region Rec(double *a, double *b, const Box &box, int gid, const Extent &ea, const Extent *eb,
           int nc = 1) {
  Region r{};
  r.a = a;
  r.b = b;
  r.nc = nc;
  r.gid = gid;
  for (int d = 0; d < 3; ++d) {
    r.lo[d] = box.lo[d];
    r.n[d] = box.hi[d] - box.lo[d] + 1;
    r.magic[d] = Magic(r.n[d]);
  }
  r.astride[0] = ea.ent(0);
  r.astride[1] = ea.ent(0) * ea.ent(1);
  r.astride[2] = static_cast<int>(ea.cells());
  if (eb) {
    r.bstride[0] = eb->ent(0);
    r.bstride[1] = eb->ent(0) * eb->ent(1);
    r.bstride[2] = static_cast<int>(eb->cells());
  }
  return r;
}

Lattice UpOne(const Lattice &a, const bool *active) {
  Lattice p;
  p.level = a.level - 1;
  for (int d = 0; d < 3; ++d) p.x[d] = active[d] ? a.x[d] / 2 : a.x[d];
  return p;
}

}  // namespace

// How the blocks of a level relate to the next coarser level's.
enum class Coarsen {
  kCap,    // blocks of the finest refinement level restrict into their parents; others are
           // the same blocks
  kMerge,  // every base block restricts into its parent of the next tree level
  kShrink  // every block keeps its position and halves its cells
};

struct TreeLevel {
  std::unique_ptr<Mesh> mesh;
  // a smoothing stage goes from x[cur] to x[1 - cur]: two containers on a level with blocks of
  // different sizes (each with its exchange tables), fields x and t of one container elsewhere
  MeshData *md = nullptr, *other = nullptr;
  double *x[2] = {nullptr, nullptr};
  int cur = 0;
  LevelView view{};
  StageCoef *coef = nullptr;
  int *face = nullptr;
  Coarsen to_coarser = Coarsen::kCap;
  Xfer *xfer = nullptr;  // to the next coarser level, child blocks first
  int nxfer = 0, nchild = 0, cchunks = 1;
  // what a stencil's exchange needs, per container: region pairs of the channels between
  // levels and of the same-level ghosts that a block restricts for its coarse neighbours, and
  // the coarse-buffer conditions of blocks that prolongate
  struct Cross {
    Table send, recv;
    BcTable bc;
  } cross[2];
  // the face field D to the next coarser level: same blocks copied, the others face-averaged
  Table copy_D;
  std::vector<FaceXfer> face_host;
  FaceXfer *face_D = nullptr;
  FaceGeom face_geom{};
  long long cells = 0;  // interior cells of all blocks
  ~TreeLevel() {
    for (Cross &q : cross) {
      q.send.Free();
      q.recv.Free();
      q.bc.Free();
    }
    copy_D.Free();
    for (void *q : {static_cast<void *>(face_D), static_cast<void *>(coef),
                    static_cast<void *>(face), static_cast<void *>(xfer)})
      if (q) PTH_DROP(hipFree(q));
  }
};

class MgTree {
 public:
  Mesh *user = nullptr;
  int fu = -1, frhs = -1, fD = -1;
  pth_mg_params P{};
  double D = 1.0, alpha = 0.0;
  std::vector<std::unique_ptr<TreeLevel>> lv;  // finest (a copy of the user's mesh) first
  std::vector<double> w_pre, w_post;           // Jacobi weight of each smoothing stage
  // a V-cycle is ~6 launches per level, each a few microseconds of work on the coarse levels:
  // the second V-cycle, with the residual norm after it, is captured and later ones replay it
  bool use_graph = true, warmed = false;
  double *partial = nullptr, *norm_host = nullptr;  // residual norm: partials and their sum
  int npartial = 0;
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  hipStream_t capture_stream = nullptr;

  ~MgTree() {
    if (partial) PTH_DROP(hipFree(partial));  // waits for the device: nothing runs past here
    if (graph_exec) PTH_DROP(hipGraphExecDestroy(graph_exec));
    if (graph) PTH_DROP(hipGraphDestroy(graph));
    if (capture_stream) PTH_DROP(hipStreamDestroy(capture_stream));
    if (norm_host) PTH_DROP(hipHostFree(norm_host));
  }
  pth_status Build();
  pth_status Setup(MeshData &md);
  pth_status Solve(MeshData &md, int *iters, std::vector<double> *history);

 private:
  pth_status Iterate(double *rms);
  pth_status NewLevel(const Topology &t, int x_prolong);
  pth_status BuildTransfers(int l);
  pth_status BuildCross(TreeLevel &L, MeshData &md, TreeLevel::Cross &q);
  pth_status Exchange(int l);
  pth_status Smooth(int l, const std::vector<double> &w, bool zero);
  pth_status Cycle(int l);
  pth_status Norm();
  pth_status Rms(double *rms);
  double *Data(int l, int f) { return lv[l]->md->store[f].data; }
  const double *Df(int l) { return fD >= 0 ? Data(l, kD) : nullptr; }
  hipStream_t Stream(int l) { return lv[l]->mesh->stream; }
};

pth_status MgTree::NewLevel(const Topology &t, int x_prolong) {
  std::unique_ptr<TreeLevel> L(new TreeLevel());
  L->mesh.reset(new Mesh());
  Mesh &m = *L->mesh;
  m.topo = t;
  m.stream = user->stream;
  m.fields.push_back(FieldSpec{"x", 1, PTH_FILL_GHOST | PTH_INDEPENDENT, x_prolong});
  m.fields.push_back(FieldSpec{"t", 1, PTH_ONE_COPY, PTH_PROLONG_LINEAR});
  m.fields.push_back(FieldSpec{"b", 1, PTH_ONE_COPY, PTH_PROLONG_LINEAR});
  m.fields.push_back(FieldSpec{"D", 3, PTH_ONE_COPY, PTH_PROLONG_LINEAR});
  if (m.Finalize() != PTH_COMPLETE) return PTH_FAIL;
  L->md = m.Get("base");
  if (!L->md) return PTH_FAIL;
  const Topology &mt = m.topo;
  const Extent &e = mt.fine;
  const int nb = static_cast<int>(mt.blocks.size());
  L->cells = static_cast<long long>(nb) * e.n[0] * e.n[1] * e.n[2];
  L->x[0] = L->md->store[kX].data;
  L->x[1] = L->md->store[kT].data;
  if (mt.multilevel) {
    L->other = m.Get("other");
    if (!L->other) return PTH_FAIL;
    L->x[1] = L->other->store[kX].data;
    if (BuildCross(*L, *L->md, L->cross[0]) != PTH_COMPLETE ||
        BuildCross(*L, *L->other, L->cross[1]) != PTH_COMPLETE)
      return PTH_FAIL;
  }
  LevelView &V = L->view;
  V.n0 = e.n[0], V.n1 = e.n[1], V.n2 = e.n[2];
  V.e0 = e.ent(0);
  V.p = e.ent(0) * e.ent(1);
  V.first = e.g[2] * V.p + e.g[1] * V.e0 + e.g[0];
  V.per = e.n[0] * e.n[1] * e.n[2];
  V.chunks = (V.per + kWG - 1) / kWG;
  V.ndim = mt.ndim;
  V.cells = e.cells();
  std::vector<int> face(6 * static_cast<size_t>(nb), kGhost);
  std::vector<StageCoef> coef(nb);
  for (int b = 0; b < nb; ++b) {
    const Block &B = mt.blocks[b];
    double diag = -alpha;
    for (int d = 0; d < 3; ++d) {
      coef[b].i2[d] = 1.0 / (B.dx[d] * B.dx[d]);
      if (!mt.active[d]) continue;
      diag -= (D + D) * coef[b].i2[d];
      const double tol = 1e-12 * (mt.xmax[d] - mt.xmin[d]);
      if (!mt.periodic[d]) {
        if (std::fabs(B.xmin[d] - mt.xmin[d]) <= tol) face[6 * b + 2 * d] = kFixed;
        if (std::fabs(B.xmax[d] - mt.xmax[d]) <= tol) face[6 * b + 2 * d + 1] = kFixed;
      }
    }
    coef[b].rdiag = 1.0 / diag;
    for (const Link &l : B.links) {
      int d = -1, faces = 0;
      for (int q = 0; q < 3; ++q)
        if (l.off[q]) d = q, ++faces;
      if (faces == 1 && l.level == B.at.level) face[6 * b + 2 * d + (l.off[d] > 0)] = l.gid;
    }
    // on a level of one block size every face has its block or the domain's condition
    for (int f = 0; f < 2 * mt.ndim; ++f)
      if (!mt.multilevel && face[6 * b + f] == kGhost) {
        SetError("MGSolver hierarchy: a block face without a neighbour");
        return PTH_FAIL;
      }
  }
  PTH_HIP(hipMalloc(&L->face, sizeof(int) * face.size()));
  PTH_HIP(hipMemcpy(L->face, face.data(), sizeof(int) * face.size(), hipMemcpyHostToDevice));
  PTH_HIP(hipMalloc(&L->coef, sizeof(StageCoef) * nb));
  PTH_HIP(hipMemcpy(L->coef, coef.data(), sizeof(StageCoef) * nb, hipMemcpyHostToDevice));
  V.face = L->face;
  lv.push_back(std::move(L));
  return PTH_COMPLETE;
}

// The exchange of x in md cut to what a stencil reads (see the head of this file).
pth_status MgTree::BuildCross(TreeLevel &L, MeshData &md, TreeLevel::Cross &q) {
  Mesh &m = *L.mesh;
  if (m.BuildCache(md, PTH_BT_ANY) != PTH_COMPLETE) return PTH_FAIL;
  BoundCache &c = md.cache[PTH_BT_ANY];
  if (!CanExchangeDirect(c.pack, c.unpack)) {
    SetError("MGSolver hierarchy: exchange tables do not pair up");
    return PTH_FAIL;
  }
  const FieldStore &x = md.store[kX];
  const std::int64_t cells = m.topo.fine.cells(), ccells = m.topo.coarse.cells();
  const size_t nb = m.topo.blocks.size();
  std::vector<char> restricts(nb, 0), prolongs(nb, 0);
  for (const Region &r : c.restrict_set.host) restricts[(r.a - x.data) / cells] = 1;
  for (const Table *t : {&c.prolong, &c.prolong_linear})
    for (const Region &r : t->host) prolongs[(r.a - x.data) / cells] = 1;
  auto fine = [&](const double *a) { return a >= x.data && a < x.data + x.ndata; };
  for (size_t i = 0; i < c.pack.host.size(); ++i) {
    const Region &s = c.pack.host[i], &r = c.unpack.host[i];
    if (s.b != r.b) {
      SetError("internal: send and receive regions do not pair up");
      return PTH_FAIL;
    }
    if (fine(s.a) && fine(r.a) && !restricts[(r.a - x.data) / cells]) continue;
    q.send.host.push_back(s);
    q.recv.host.push_back(r);
  }
  for (const BcBox &b : c.bc[1].host)
    if (prolongs[(b.slab - x.coarse) / ccells]) q.bc.host.push_back(b);
  if (q.send.Upload() != PTH_COMPLETE || q.recv.Upload() != PTH_COMPLETE) return PTH_FAIL;
  return q.bc.Upload();
}

pth_status MgTree::Build() {
  const Topology &ut = user->topo;
  // the level weights
  const int nd = std::max(ut.ndim, 1) - 1;
  if (P.smoother == 0) {
    w_pre.assign(P.pre_sweeps, P.omega);
    w_post.assign(P.post_sweeps, P.omega);
  } else {
    std::vector<double> w;
    if (P.smoother == 1) w = {1.0};
    if (P.smoother == 2) w = {kSrj2[nd][0], kSrj2[nd][1]};
    if (P.smoother == 3) w = {kSrj3[nd][0], kSrj3[nd][1], kSrj3[nd][2]};
    w_pre = w_post = w;
  }
  int top = 0;
  for (const auto &a : ut.leaf) top = std::max(top, a.level);
  // refined levels: the leaf mesh capped at level L = top .. 0
  for (int L = top; L >= 0; --L) {
    Topology t = ut;
    t.leaf.clear();
    t.inner.clear();
    for (const auto &a : ut.leaf)
      if (a.level <= L) t.leaf.insert(a);
    for (const auto &a : ut.inner) {
      if (a.level < L) t.inner.insert(a);
      if (a.level == L) t.leaf.insert(a);
    }
    t.multilevel = !t.inner.empty();
    const int xp = L == top ? user->fields[fu].prolong : PTH_PROLONG_LINEAR;
    if (NewLevel(t, xp) != PTH_COMPLETE) return PTH_FAIL;
    lv.back()->to_coarser = Coarsen::kCap;
  }
  // below the base grid: the forest's tree levels (root_level merges of 2^d base blocks,
  // forest.cpp:64-105), then levels that halve every block's cells as many times as the block
  // size has trailing binary zeros (mesh-gmg.cpp:106-118), with one ghost layer
  int nx[3], bnx[3], ng = ut.ng;
  for (int d = 0; d < 3; ++d) {
    nx[d] = ut.nx[d];
    bnx[d] = ut.bnx[d];
  }
  int merges = ut.RootLevel(), shrinks = 1 << 30;
  for (int d = 0; d < 3; ++d) {
    if (!ut.active[d]) continue;
    int z = 0;
    while (((bnx[d] >> z) & 1) == 0) ++z;
    shrinks = std::min(shrinks, z);
  }
  if (shrinks == (1 << 30)) shrinks = 0;
  for (int q = 0; q < merges + shrinks; ++q) {
    const bool merge = q < merges;
    // a level keeps at least two cells along every active dimension (a mesh of one cell
    // along a dimension is a mesh without that dimension here)
    bool fits = true;
    for (int d = 0; d < 3; ++d) fits = fits && (!ut.active[d] || nx[d] / 2 >= 2);
    if (!fits) break;
    lv.back()->to_coarser = merge ? Coarsen::kMerge : Coarsen::kShrink;
    for (int d = 0; d < 3; ++d) {
      if (!ut.active[d]) continue;
      nx[d] /= 2;
      if (!merge) bnx[d] /= 2;
    }
    if (!merge) ng = 1;
    Topology t;
    const int per[3] = {ut.periodic[0], ut.periodic[1], ut.periodic[2]};
    const std::string err = t.Init(nx, bnx, ng, ut.xmin, ut.xmax, per);
    if (!err.empty()) {
      SetError("MGSolver hierarchy: " + err);
      return PTH_FAIL;
    }
    for (int f = 0; f < 6; ++f) t.bc[f] = ut.bc[f];
    if (NewLevel(t, PTH_PROLONG_LINEAR) != PTH_COMPLETE) return PTH_FAIL;
  }
  for (int l = 0; l + 1 < static_cast<int>(lv.size()); ++l)
    if (BuildTransfers(l) != PTH_COMPLETE) return PTH_FAIL;
  npartial = static_cast<int>(lv[0]->mesh->topo.blocks.size()) * lv[0]->view.chunks;
  PTH_HIP(hipMalloc(&partial, sizeof(double) * (npartial + 1)));
  PTH_HIP(hipHostMalloc(&norm_host, sizeof(double)));
  return PTH_COMPLETE;
}

pth_status MgTree::BuildTransfers(int l) {
  TreeLevel &F = *lv[l], &C = *lv[l + 1];
  const Topology &ft = F.mesh->topo, &ct = C.mesh->topo;
  const Extent &fe = ft.fine, &Ce = ct.fine;
  int top = 0;
  for (const auto &a : ft.leaf) top = std::max(top, a.level);
  std::vector<Xfer> kids, same;
  for (int fb = 0; fb < static_cast<int>(ft.blocks.size()); ++fb) {
    const Lattice &a = ft.blocks[fb].at;
    bool child = false;
    Lattice target = a;
    int o[3] = {0, 0, 0};
    if (F.to_coarser == Coarsen::kCap) {
      child = a.level == top && a.level > 0;
      if (child) target = UpOne(a, ft.active);
    } else if (F.to_coarser == Coarsen::kMerge) {
      child = true;
      target = a;
      for (int d = 0; d < 3; ++d) target.x[d] = ft.active[d] ? a.x[d] / 2 : a.x[d];
    }
    if (child)
      for (int d = 0; d < 3; ++d)
        o[d] = ft.active[d] ? static_cast<int>(a.x[d] - 2 * target.x[d]) : 0;
    auto it = ct.id.find(target);
    if (it == ct.id.end()) {
      SetError("MGSolver hierarchy: a block has no counterpart on the coarser level");
      return PTH_FAIL;
    }
    const int cbk = it->second;
    if (F.to_coarser == Coarsen::kCap && !child) {  // the same block on both levels
      if (fe.n[0] != Ce.n[0] || fe.n[1] != Ce.n[1] || fe.n[2] != Ce.n[2]) {
        SetError("MGSolver hierarchy: block shapes differ between levels");
        return PTH_FAIL;
      }
      same.push_back(Xfer{fb, cbk, {0, 0, 0}, 0});
      F.copy_D.host.push_back(Rec(F.md->store[kD].data + fb * 3 * fe.cells(),
                                  C.md->store[kD].data + cbk * 3 * Ce.cells(), Whole(fe), fb,
                                  fe, &Ce, 3));
      continue;
    }
    for (int d = 0; d < 3; ++d)
      if (ft.active[d] && (fe.n[d] % 2 || (o[d] + 1) * (fe.n[d] / 2) > Ce.n[d])) {
        SetError("MGSolver hierarchy: a block does not fit its coarser block");
        return PTH_FAIL;
      }
    F.face_host.push_back(FaceXfer{F.md->store[kD].data + fb * 3 * fe.cells(),
                                   C.md->store[kD].data + cbk * 3 * Ce.cells(),
                                   {o[0], o[1], o[2]}, 0});
    kids.push_back(Xfer{fb, cbk, {o[0], o[1], o[2]}, 1});
  }
  F.nchild = static_cast<int>(kids.size());
  kids.insert(kids.end(), same.begin(), same.end());
  F.nxfer = static_cast<int>(kids.size());
  F.cchunks = (F.view.per / (1 << ft.ndim) + kWG - 1) / kWG;
  PTH_HIP(hipMalloc(&F.xfer, sizeof(Xfer) * kids.size()));
  PTH_HIP(hipMemcpy(F.xfer, kids.data(), sizeof(Xfer) * kids.size(), hipMemcpyHostToDevice));
  if (F.copy_D.Upload() != PTH_COMPLETE) return PTH_FAIL;
  FaceGeom &G = F.face_geom;
  G.fe0 = fe.ent(0), G.fe1 = fe.ent(1), G.ce0 = Ce.ent(0), G.ce1 = Ce.ent(1);
  G.fcells = fe.cells(), G.ccells = Ce.cells();
  for (int d = 0; d < 3; ++d) {
    G.fg[d] = fe.g[d], G.cg[d] = Ce.g[d];
    G.nc[d] = ft.active[d] ? fe.n[d] / 2 : fe.n[d];
    G.act[d] = ft.active[d] ? 1 : 0;
    // the upper face of the last cell lies in the first ghost cell on both levels
    if (ft.active[d] && (fe.g[d] < 1 || Ce.g[d] < 1)) {
      SetError("MGSolver hierarchy: the face field needs one ghost layer");
      return PTH_FAIL;
    }
  }
  G.ndim = ft.ndim;
  if (!F.face_host.empty()) {
    PTH_HIP(hipMalloc(&F.face_D, sizeof(FaceXfer) * F.face_host.size()));
    PTH_HIP(hipMemcpy(F.face_D, F.face_host.data(), sizeof(FaceXfer) * F.face_host.size(),
                      hipMemcpyHostToDevice));
  }
  return PTH_COMPLETE;
}

// x's ghost cells that the level's stencils read (none on a level of one block size)
pth_status MgTree::Exchange(int l) {
  TreeLevel &L = *lv[l];
  if (!L.other) return PTH_COMPLETE;
  Mesh &m = *L.mesh;
  BoundCache &c = (L.cur ? L.other : L.md)->cache[PTH_BT_ANY];
  TreeLevel::Cross &q = L.cross[L.cur];
  if (LaunchRestrictT(c.restrict_send, m.topo, m.geom, m.stream) != PTH_COMPLETE ||
      LaunchExchangeDirect(q.send, q.recv, m.stream) != PTH_COMPLETE ||
      LaunchRestrictT(c.restrict_set, m.topo, m.geom, m.stream) != PTH_COMPLETE ||
      LaunchBoundaryConditions(q.bc, m.stream) != PTH_COMPLETE ||
      LaunchProlongT(c.prolong, m.topo, m.geom, m.stream, true) != PTH_COMPLETE)
    return PTH_FAIL;
  return LaunchProlongT(c.prolong_linear, m.topo, m.geom, m.stream, false);
}

// Smoothing stages with weights w; zero: the first starts from x = 0 (which is not stored)
pth_status MgTree::Smooth(int l, const std::vector<double> &w, bool zero) {
  TreeLevel &L = *lv[l];
  const dim3 grid(static_cast<unsigned>(L.mesh->topo.blocks.size()) * L.view.chunks);
  if (zero) L.cur = 0;
  if (zero && w.empty()) {
    PTH_LAUNCH(ZeroKernel, grid, dim3(kWG), 0, Stream(l), L.x[0], L.view);
  }
  for (size_t q = 0; q < w.size(); ++q) {
    if (zero && q == 0) {
      ProfScope prof("mg_level_jacobi", Stream(l));
      PTH_LAUNCH(StageKernel<true>, grid, dim3(kWG), 0, Stream(l), nullptr,
                 Data(l, kB), L.x[0], L.view, L.coef, D, Df(l), alpha, w[q]);
    } else {
      if (Exchange(l) != PTH_COMPLETE) return PTH_FAIL;
      ProfScope prof("mg_level_jacobi", Stream(l));
      PTH_LAUNCH(StageKernel<false>, grid, dim3(kWG), 0, Stream(l), L.x[L.cur],
                 Data(l, kB), L.x[1 - L.cur], L.view, L.coef, D, Df(l), alpha, w[q]);
      L.cur = 1 - L.cur;
    }
  }
  return PTH_COMPLETE;
}

pth_status MgTree::Cycle(int l) {
  const int last = static_cast<int>(lv.size()) - 1;
  if (Smooth(l, w_pre, l > 0) != PTH_COMPLETE) return PTH_FAIL;
  TreeLevel &F = *lv[l];
  if (l < last) {
    TreeLevel &C = *lv[l + 1];
    // residual, restricted into the coarser level's right-hand side
    if (Exchange(l) != PTH_COMPLETE) return PTH_FAIL;
    {
      ProfScope prof("mg_level_residual", Stream(l));
      const unsigned grid = static_cast<unsigned>(F.nchild * F.cchunks +
                                                  (F.nxfer - F.nchild) * F.view.chunks);
      PTH_LAUNCH(ResidualDownKernel, dim3(grid), dim3(kWG), 0, Stream(l), F.x[F.cur],
                 Data(l, kB), F.view, F.coef, D, Df(l), alpha, Data(l + 1, kB), C.view,
                 F.xfer, F.nchild, F.cchunks);
    }
    if (Cycle(l + 1) != PTH_COMPLETE) return PTH_FAIL;
    // the coarser correction, prolongated and added
    if (Exchange(l + 1) != PTH_COMPLETE) return PTH_FAIL;
    {
      ProfScope prof("mg_level_prolong", Stream(l));
      PTH_LAUNCH(ProlongAddKernel,
                 dim3(static_cast<unsigned>(F.nxfer) * F.view.chunks), dim3(kWG), 0,
                 Stream(l), F.x[F.cur], F.view, C.x[C.cur], C.view, F.xfer);
    }
    if (Smooth(l, w_post, false) != PTH_COMPLETE) return PTH_FAIL;
  }
  if (l == 0 && F.cur == 1) {  // an odd number of stages: back to the first array
    PTH_HIP(hipMemcpyAsync(F.x[0], F.x[1], sizeof(double) * F.md->store[kX].ndata,
                           hipMemcpyDeviceToDevice, Stream(0)));
    F.cur = 0;
  }
  return PTH_COMPLETE;
}

// sum of squares of the leaf level's residual into partial[npartial]
pth_status MgTree::Norm() {
  TreeLevel &L = *lv[0];
  if (Exchange(0) != PTH_COMPLETE) return PTH_FAIL;
  ProfScope prof("mg_residual_norm", Stream(0));
  PTH_LAUNCH(ResidualNormKernel, dim3(npartial), dim3(kWG), 0, Stream(0), L.x[0],
             Data(0, kB), L.view, L.mesh->coef, D, Df(0), alpha, partial);
  PTH_LAUNCH(SumKernel, dim3(1), dim3(kSumWG), 0, Stream(0), partial, npartial,
             partial + npartial);
  return PTH_COMPLETE;
}

// one V-cycle and the RMS residual after it
pth_status MgTree::Iterate(double *rms) {
  auto both = [&]() -> pth_status {
    if (Cycle(0) != PTH_COMPLETE) return PTH_FAIL;
    return Norm();
  };
  if (!use_graph || !warmed) {
    warmed = true;
    if (both() != PTH_COMPLETE) return PTH_FAIL;
    return Rms(rms);
  }
  hipStream_t s = Stream(0);
  if (!graph_exec) {
    // the caller's stream may be the null stream, which cannot be captured: the levels launch
    // on a stream of the solver's own while the V-cycle is captured
    if (!capture_stream)
      PTH_HIP(hipStreamCreateWithFlags(&capture_stream, hipStreamNonBlocking));
    for (auto &L : lv) L->mesh->stream = capture_stream;
    const bool prof = Prof().on;
    Prof().on = false;  // no event records inside the captured V-cycle
    hipError_t e = hipStreamBeginCapture(capture_stream, hipStreamCaptureModeThreadLocal);
    const bool began = !Failed(e);
    pth_status st = PTH_FAIL;
    hipGraph_t g = nullptr;
    if (began) {
      st = both();
      e = hipStreamEndCapture(capture_stream, &g);
      (void)Failed(e);
    }
    Prof().on = prof;
    for (auto &L : lv) L->mesh->stream = s;
    if (e != hipSuccess && (!began || st == PTH_COMPLETE))
      SetError(std::string("MGSolver: V-cycle capture: ") + hipGetErrorString(e));
    if (st != PTH_COMPLETE || e != hipSuccess) {
      if (g) PTH_DROP(hipGraphDestroy(g));
      return PTH_FAIL;
    }
    graph = g;
    PTH_HIP(hipGraphInstantiate(&graph_exec, g, nullptr, nullptr, 0));
  }
  {
    ProfScope prof("mg_vcycle_graph", s);
    PTH_HIP(hipGraphLaunch(graph_exec, s));
  }
  return Rms(rms);
}

// the RMS residual from the sum that Norm left (waits for it)
pth_status MgTree::Rms(double *rms) {
  PTH_HIP(hipMemcpyAsync(norm_host, partial + npartial, sizeof(double), hipMemcpyDeviceToHost,
                         Stream(0)));
  PTH_HIP(hipStreamSynchronize(Stream(0)));
  *rms = std::sqrt(*norm_host / static_cast<double>(lv[0]->cells));
  return PTH_COMPLETE;
}

pth_status MgTree::Setup(MeshData &md) {
  // the leaf level is a copy of the user's mesh: same blocks in the same order
  Mesh &m0 = *lv[0]->mesh;
  const Topology &ut = user->topo;
  if (ut.blocks.size() != m0.topo.blocks.size()) {
    SetError("MGSolver: the mesh changed since the solver was created");
    return PTH_FAIL;
  }
  for (size_t b = 0; b < ut.blocks.size(); ++b)
    if (!(ut.blocks[b].at == m0.topo.blocks[b].at)) {
      SetError("MGSolver: the mesh changed since the solver was created");
      return PTH_FAIL;
    }
  lv[0]->cur = 0;
  const size_t n = sizeof(double) * md.store[fu].ndata;
  PTH_HIP(hipMemcpyAsync(Data(0, kX), md.store[fu].data, n, hipMemcpyDeviceToDevice, m0.stream));
  PTH_HIP(hipMemcpyAsync(Data(0, kB), md.store[frhs].data, n, hipMemcpyDeviceToDevice,
                         m0.stream));
  if (fD < 0) return PTH_COMPLETE;
  // AddSetupTasks: the face field D (GMGRestrict) down the levels
  PTH_HIP(hipMemcpyAsync(Data(0, kD), md.store[fD].data, sizeof(double) * md.store[fD].ndata,
                         hipMemcpyDeviceToDevice, m0.stream));
  for (int l = 0; l + 1 < static_cast<int>(lv.size()); ++l) {
    TreeLevel &F = *lv[l];
    if (LaunchCopy(F.copy_D, F.mesh->stream) != PTH_COMPLETE) return PTH_FAIL;
    if (F.face_host.empty()) continue;
    const FaceGeom &G = F.face_geom;
    long long per_rec = G.ndim;
    for (int d = 0; d < 3; ++d) per_rec *= G.act[d] ? G.nc[d] + 1 : 1;
    const long long total = per_rec * static_cast<long long>(F.face_host.size());
    PTH_LAUNCH(FaceRestrictKernel, dim3(Grid(total)), dim3(kWG), 0, F.mesh->stream,
               F.face_D, G, per_rec, total);
  }
  return PTH_COMPLETE;
}

pth_status MgTree::Solve(MeshData &md, int *iters, std::vector<double> *history) {
  history->clear();
  double rms = 0.0;
  if (Norm() != PTH_COMPLETE || Rms(&rms) != PTH_COMPLETE) return PTH_FAIL;
  history->push_back(rms);
  int it = 0;
  do {
    if (Iterate(&rms) != PTH_COMPLETE) return PTH_FAIL;
    ++it;
    history->push_back(rms);
  } while (rms > P.residual_tolerance && it < P.max_iters);
  *iters = it;
  Mesh &m0 = *lv[0]->mesh;
  PTH_HIP(hipMemcpyAsync(md.store[fu].data, Data(0, kX), sizeof(double) * md.store[fu].ndata,
                         hipMemcpyDeviceToDevice, m0.stream));
  return PTH_COMPLETE;
}

MgTree *MgTreeCreate(Mesh *m, int fu, int frhs, int fD, const pth_mg_params &p, double D,
                     double alpha) {
  std::unique_ptr<MgTree> t(new MgTree());
  t->user = m;
  t->fu = fu;
  t->frhs = frhs;
  t->fD = fD;
  t->P = p;
  t->D = D;
  t->alpha = alpha;
  if (t->Build() != PTH_COMPLETE) return nullptr;
  return t.release();
}

void MgTreeDestroy(MgTree *t) { delete t; }

int MgTreeLevels(const MgTree *t) { return static_cast<int>(t->lv.size()); }

void MgTreeSetGraph(MgTree *t, bool on) { t->use_graph = on; }

pth_status MgTreeSetup(MgTree *t, MeshData &md) { return t->Setup(md); }

pth_status MgTreeSolve(MgTree *t, MeshData &md, int *iters, std::vector<double> *history) {
  return t->Solve(md, iters, history);
}

}  // namespace pth
