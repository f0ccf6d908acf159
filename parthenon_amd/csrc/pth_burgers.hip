// Burgers benchmark (Parthenon-VIBE) stage kernels for gfx950, FP64.
//
// Task-level kernels, one launch per reference task over every block of the MeshData:
//   FluxTaskKernel   burgers_package::CalculateFluxes: reconstruction
//                    (benchmarks/burgers/burgers_package.cpp:236-303, recon.hpp:28-99) and HLL
//                    (burgers_package.cpp:307-401, burgers_package.hpp:33-43)
//   FluxDivKernel    Update::FluxDivergence (src/interface/update.cpp:63-84, update.hpp:43-57)
//   WsumKernel       Update::WeightedSumData (src/interface/update.hpp:71-90)
//   DerivedKernel    burgers_package::CalculateDerived (burgers_package.cpp:143-167)
//   DtKernel         burgers_package::EstimateTimestepMesh (burgers_package.cpp:170-200):
//                    per-workgroup min via 64-lane wavefront shuffles, then one final pass
// Expression order matches the reference operator by operator and this file is built with
// -ffp-contract=off, so results are reproducible bit for bit by an IEEE CPU evaluation (the
// block-sweep form, in pth_sweep.hip, is built with contraction instead).
// Arrays are [block][comp][k][j][i] bricks of (n+2g)^3 with i fastest; consecutive lanes
// take consecutive i, so every load and store is a coalesced run along x.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <type_traits>

#include "pth_burgers.hpp"
#include "pth_device.hpp"
#include "pth_stencil.hpp"

namespace pth {

namespace {

constexpr int kWG = 256;

// HLL flux of component n at one face from its left and right states and those of the normal
// velocity (burgers_package.cpp:307-401 with lr_to_flux, burgers_package.hpp:33-43).
__device__ __forceinline__ double HllOne(int n, double upl, double upr, double l, double r) {
  const double sl = DMin(DMin(upl, upr), 0.0);
  const double sr = DMax(DMax(upl, upr), 0.0);
  const double den = sr - sl + (sl * sr == 0.0);
  if (n < 3) {
    const double islsr = 1.0 / den;
    return 0.5 * (sr * l * upl - sl * r * upr + sl * sr * (r - l)) * islsr;
  }
  return (sr * upl * l - sl * upr * r + sl * sr * (r - l)) / den;
}

// How FluxTaskKernel splits the work: units of `pack` consecutive blocks, `chunks` groups of
// `comps` components (one of all, by segments); per unit and group workgroups of each direction, in `stripes`; y and z by rows
// or by segments of `seg` faces.
constexpr int kSegFaces = 9;
struct FluxSplit {
  int wgs[3], seg[3];
  int pack, chunks, comps, stripes, rows;
};

// CalculateFluxes of any block shape in one launch, from U to the fluxes [3][block][comp][k][j][i]
// (x-face i - 1/2 at index i): the face states stay on chip. One workgroup takes a piece of one
// block (of several, where one would leave most of its lanes idle) in one direction and goes
// through its components one after another, the normal velocity first (its face states give every
// component's signal speeds), so any number of components fits.
//   rows (x; y and z where the mesh is small): a wavefront takes 64 consecutive cells of the rows
//      along the direction, extended by one cell on each side; a lane reconstructs its cell and
//      gets the left state of its low face from the lane below (the first lane of a wavefront
//      repeats the last one's cell of the wavefront before; the first cell of a row, and so of a
//      block, has no low face);
//   segments (y, z): a thread marches a column segment of at most kSegFaces faces with the stencil
//      in a register window, lanes along x; the normal velocity's states wait in LDS, each thread
//      in its own slots (no barriers).
// A cell is reconstructed once, but for two cells a row or one a segment or wavefront. The
// operations are those of the reference in its order, without contraction. Bound: FP64 issue
// (about 300 instructions a reconstruction with its flux, 8 IEEE divides among them). On the
// 960-block mesh with 7 components the reconstruction and HLL as two launches, with the states in
// HBM between them, took 1341 + 1043 us; this kernel takes 1070. One block of 128^3: 1417 us with
// the directions one after another, which leaves XCDs with long workgroups alone, 509 in stripes.
// WIDE: 64-bit cell offsets, for components of 4 GB and more. ROWS: y and z by rows too.
template <int RECON, bool WIDE, bool ROWS>
__global__ void __launch_bounds__(kWG)
    FluxTaskKernel(const double *__restrict__ U, double *__restrict__ flux, Geo G, int nblocks,
                   FluxSplit S) {
  using I = std::conditional_t<WIDE, std::int64_t, int>;       // cells
  using O = std::conditional_t<WIDE, std::int64_t, unsigned>;  // byte offsets
  // one unit's workgroups are adjacent and run on one XCD: the three directions read the
  // same cells
  const unsigned L = XcdRemap(blockIdx.x, gridDim.x);
  const unsigned per = S.wgs[0] + S.wgs[1] + S.wgs[2];
  const int chunk = ROWS ? static_cast<int>(L / per) % S.chunks : 0;
  const int b0 = static_cast<int>(L / per) / (ROWS ? S.chunks : 1) * S.pack;
  const int nb = nblocks - b0 < S.pack ? nblocks - b0 : S.pack;  // blocks of this unit
  const int na = ROWS ? chunk * S.comps : 0;
  const int nz = ROWS && na + S.comps < G.V ? na + S.comps : G.V;
  // the unit's stripes, each with its share of the x, the y and the z workgroups
  auto from = [&](int d, std::uint64_t s) { return static_cast<int>(s * S.wgs[d] / S.stripes); };
  auto start = [&](std::uint64_t s) { return from(0, s) + from(1, s) + from(2, s); };
  int r = static_cast<int>(L % per), d = 0;
  std::uint64_t s = static_cast<std::uint64_t>(r) * S.stripes / per;
  while (start(s) > r) --s;
  while (start(s + 1) <= r) ++s;
  r -= start(s);
  while (r >= from(d, s + 1) - from(d, s)) r -= from(d, s + 1) - from(d, s), ++d;
  r += from(d, s);
  // the normal velocity is one of this chunk's components
  const bool own = !ROWS || (d >= na && d < nz);
  const int n0 = G.hi0 - G.lo0 + 1, n1 = G.hi1 - G.lo1 + 1, n2 = G.hi2 - G.lo2 + 1;
  const double *Ub = U + static_cast<std::int64_t>(b0) * G.V * G.cells;
  double *Fb = flux + (static_cast<std::int64_t>(d) * nblocks + b0) * G.V * G.cells;
  const int tid = static_cast<int>(threadIdx.x);
  const int nd = d == 0 ? n0 : d == 1 ? n1 : n2;
  const O st = O(8) * static_cast<O>(d == 0 ? 1 : d == 1 ? G.e0 : G.e0 * G.e1);
  if (ROWS || d == 0) {
    const int m = nd + 2, across = d == 0 ? n1 : n0;
    const I cells = static_cast<I>(m) * across * (d == 2 ? n1 : n2), all = cells * nb;
    const I e0 = static_cast<I>(63) * (r * (kWG / 64) + (tid >> 6)) + (tid & 63);
    I e = e0 < all ? e0 : all - 1, at = 0;
    if (S.pack > 1) {
      const I lb = e / cells;
      e -= lb * cells;
      at = lb * static_cast<I>(G.V) * static_cast<I>(G.cells);
    }
    const int a = static_cast<int>(e % m), row = static_cast<int>(e / m);
    const int p = row % across, o = row / across;  // the other two directions, in order
    const int i = d == 0 ? a - 1 : p, j = d == 0 ? p : d == 1 ? a - 1 : o, k = d == 2 ? a - 1 : o;
    const O c = O(8) * static_cast<O>(at + (static_cast<I>(G.lo2 + k) * G.e1 + G.lo1 + j) * G.e0 +
                                      G.lo0 + i);
    const bool face = a > 0 && e0 < all && (tid & 63) > 0;
    auto fluxes = [&](auto step) {  // x's step as a constant: it goes into the loads' offsets
      double upl = 0.0, upr = 0.0;
      for (int q = na - 1; q < nz; ++q) {
        const int n = q < na ? d : q;
        if (q >= na && n == d) continue;  // the normal velocity came first
        double ql, qr;
        CellStates(Ub + n * G.cells, c, static_cast<O>(step), RECON, ql, qr);
        const double l = __shfl_up(ql, 1, 64);
        if (q < na) {
          upl = l;
          upr = qr;
          if (!own) continue;
        }
        if (face) StoreAt(Fb + n * G.cells, c, HllOne(n, upl, upr, l, qr));
      }
    };
    if (d == 0)
      fluxes(std::integral_constant<O, 8>());
    else
      fluxes(st);
    return;
  }
  __shared__ double up[2][kSegFaces][kWG];
  const int len = S.seg[d];
  const I cols = static_cast<I>(n0) * (d == 1 ? n2 : n1), all = cols * S.pack;
  I t = static_cast<I>(r) * kWG + tid, at = 0;
  const int f0 = static_cast<int>(t / all) * len, f1 = f0 + len < nd + 1 ? f0 + len : nd + 1;
  if (f0 > nd) return;
  t %= all;
  if (S.pack > 1) {
    const I lb = t / cols;
    if (lb >= nb) return;
    t -= lb * cols;
    at = lb * static_cast<I>(G.V) * static_cast<I>(G.cells);
  }
  const int o = static_cast<int>(t / n0);
  // first face's high cell: face f of the column lies below cell f
  const O c0 = O(8) * static_cast<O>(at + (static_cast<I>(G.lo2 + (d == 1 ? o : f0)) * G.e1 +
                                           G.lo1 + (d == 1 ? f0 : o)) * G.e0 + G.lo0 + t % n0);
  for (int q = na - 1; q < nz; ++q) {
    const int n = q < na ? d : q;
    if (q >= na && n == d) continue;
    const double *u = Ub + n * G.cells;
    // window of the cell below the first face
    constexpr int H = RECON == 0 ? 2 : 1;
    double w[2 * H + 1], below = 0.0;
#pragma unroll
    for (int x = 0; x < 2 * H; ++x) w[x] = LoadAt(u, c0 + st * static_cast<O>(x - 1 - H));
    O c = c0 - st;
    double next = LoadAt(u, c + H * st);
    for (int f = f0 - 1; f < f1; ++f, c += st) {
      w[2 * H] = next;
      if (f + 1 < f1) next = LoadAt(u, c + (H + 1) * st);
      double ql, qr;
      if constexpr (RECON == 0)
        Weno5Z(w[0], w[1], w[2], w[3], w[4], ql, qr);
      else
        LinearRecon(w[0], w[1], w[2], ql, qr);
      if (f >= f0) {
        if (q < na) {
          up[0][f - f0][tid] = below;
          up[1][f - f0][tid] = qr;
        }
        StoreAt(Fb + n * G.cells, c, HllOne(n, up[0][f - f0][tid], up[1][f - f0][tid], below, qr));
      }
      below = ql;
#pragma unroll
      for (int x = 0; x < 2 * H; ++x) w[x] = w[x + 1];
    }
  }
}

// FluxDivKernel's workgroups: kChunk consecutive interior cells of one brick (a block's component),
// kCells a thread, 256 apart. The brick and the chunk's first plane are the workgroup's (scalar),
// a thread divides 32-bit numbers below a plane's cells. SMALL: bricks of
// fewer than kChunk / 4 cells, of which a workgroup takes several, one after another (1024 blocks of
// 8^2, 7 components: 9.9 us alone, 5.7; 512 of 8^3 20.0 alone, 20.8).
constexpr int kCells = 4, kChunk = kCells * kWG;
template <bool SMALL>
struct Chunk {
  std::int64_t brick, t0, per, end;
  int n0, plane, k0;
  std::uint32_t x0;
  __device__ __forceinline__ Chunk(const Geo &G, int nblocks) {
    n0 = G.hi0 - G.lo0 + 1;
    plane = n0 * (G.hi1 - G.lo1 + 1);
    per = static_cast<std::int64_t>(plane) * (G.hi2 - G.lo2 + 1);
    if (SMALL) {
      t0 = static_cast<std::int64_t>(blockIdx.x) * kChunk;
      end = per * G.V * nblocks;
      brick = t0 / per;
      x0 = static_cast<std::uint32_t>(t0 - brick * per);
      k0 = 0;
      return;
    }
    const std::uint32_t chunks = static_cast<std::uint32_t>((per + kChunk - 1) / kChunk);
    brick = blockIdx.x / chunks;
    t0 = static_cast<std::int64_t>(blockIdx.x % chunks) * kChunk;
    end = per;
    k0 = static_cast<int>(t0 / plane);
    x0 = static_cast<std::uint32_t>(t0 % plane);
  }
  // slot u has a cell (the workgroup's last slots may be past the end)
  __device__ __forceinline__ bool has(int u) const { return t0 + u * kWG < end; }
  // offset from the first brick of this thread's cell u, and that brick's number past the first;
  // past the end those of the last cell
  __device__ __forceinline__ std::int64_t cell(const Geo &G, int u, int *past) const {
    const int o = u * kWG + static_cast<int>(threadIdx.x);
    std::uint32_t x = x0 + static_cast<std::uint32_t>(t0 + o < end ? o : end - 1 - t0);
    *past = 0;
    if (SMALL) {
      *past = static_cast<int>(x / static_cast<std::uint32_t>(per));
      x -= static_cast<std::uint32_t>(*past) * static_cast<std::uint32_t>(per);
    }
    const int dk = static_cast<int>(x / static_cast<std::uint32_t>(plane));
    const std::uint32_t y = x - static_cast<std::uint32_t>(dk) * plane;
    const int j = static_cast<int>(y / static_cast<std::uint32_t>(n0));
    const int i = static_cast<int>(y) - j * n0;
    return (SMALL ? *past * G.cells : 0) +
           (static_cast<std::int64_t>(k0 + dk + G.lo2) * G.e1 + (j + G.lo1)) * G.e0 + i + G.lo0;
  }
};
std::int64_t BrickCells(const Topology &t) {
  return static_cast<std::int64_t>(t.fine.n[0]) * t.fine.n[1] * t.fine.n[2];
}
bool SmallBricks(const Topology &t) { return BrickCells(t) * 4 < kChunk; }
unsigned ChunkGrid(const Topology &t, std::int64_t bricks) {
  const std::int64_t per = BrickCells(t);
  return static_cast<unsigned>(SmallBricks(t) ? (bricks * per + kChunk - 1) / kChunk
                                              : bricks * ((per + kChunk - 1) / kChunk));
}

// Bound by memory: a cell takes two values of each face array, which share lines along x, and
// writes one. 7 components in 16^3 blocks of a 64^3 mesh refined in a sphere: 402 -> 365 us
// against four 64-bit divisions a cell and one cell at a time; 12 x 20 x 24 blocks 29 -> 22.
template <bool SMALL>
__global__ void __launch_bounds__(kWG)
    FluxDivKernel(const double *__restrict__ flux, double *__restrict__ dudt,
                  const BlockCoefs *__restrict__ coef, Geo G, int nblocks) {
  const Chunk<SMALL> K(G, nblocks);
  const std::int64_t slab = G.cells * G.V * nblocks;
  const std::int64_t sj = G.e0, sk = static_cast<std::int64_t>(G.e0) * G.e1;
  const double *f = flux + K.brick * G.cells;
  double x0[kCells], x1[kCells], y0[kCells], y1[kCells], z0[kCells], z1[kCells];
  std::int64_t c[kCells];
  int past[kCells];
#pragma unroll
  for (int u = 0; u < kCells; ++u) {
    if (!K.has(u)) break;
    c[u] = K.cell(G, u, &past[u]);
    const double *fx = f + c[u];
    x0[u] = fx[0];
    x1[u] = fx[1];
    y0[u] = G.ndim >= 2 ? fx[slab] : 0.0;
    y1[u] = G.ndim >= 2 ? fx[slab + sj] : 0.0;
    z0[u] = G.ndim == 3 ? fx[2 * slab] : 0.0;
    z1[u] = G.ndim == 3 ? fx[2 * slab + sk] : 0.0;
  }
  double *out = dudt + K.brick * G.cells;
#pragma unroll
  for (int u = 0; u < kCells; ++u) {
    if (!K.has(u)) break;
    const BlockCoefs &C = coef[(K.brick + past[u]) / G.V];
    double du = (C.area[0] * x1[u] - C.area[0] * x0[u]);
    if (G.ndim >= 2) du += (C.area[1] * y1[u] - C.area[1] * y0[u]);
    if (G.ndim == 3) du += (C.area[2] * z1[u] - C.area[2] * z0[u]);
    out[c[u]] = -du / C.vol;  // past the end: the last cell's value once more
  }
}

__global__ void __launch_bounds__(kWG)
    WsumKernel(const double *__restrict__ x, const double *__restrict__ y, double w1, double w2,
               double *__restrict__ z, std::int64_t n) {
  for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * kWG + threadIdx.x; t < n;
       t += static_cast<std::int64_t>(gridDim.x) * kWG)
    z[t] = w1 * x[t] + w2 * y[t];
}

__global__ void __launch_bounds__(kWG)
    DerivedKernel(const double *__restrict__ U, double *__restrict__ out, Geo G, int nblocks) {
  const int n0 = G.hi0 - G.lo0 + 1, n1 = G.hi1 - G.lo1 + 1, n2 = G.hi2 - G.lo2 + 1;
  const std::int64_t total = static_cast<std::int64_t>(n0) * n1 * n2 * nblocks;
  for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * kWG + threadIdx.x; t < total;
       t += static_cast<std::int64_t>(gridDim.x) * kWG) {
    std::int64_t r = t;
    const int i = static_cast<int>(r % n0) + G.lo0;
    r /= n0;
    const int j = static_cast<int>(r % n1) + G.lo1;
    r /= n1;
    const int k = static_cast<int>(r % n2) + G.lo2;
    r /= n2;
    const std::int64_t c = (static_cast<std::int64_t>(k) * G.e1 + j) * G.e0 + i;
    const double *u = U + r * G.V * G.cells + c;
    const double u1 = u[0], u2 = u[G.cells], u3 = u[2 * G.cells], d = u[3 * G.cells];
    out[r * G.cells + c] = 0.5 * d * (u1 * u1 + u2 * u2 + u3 * u3);
  }
}

// Per-workgroup minimum of the CFL time step over interior cells; partial[blockIdx.x].
__global__ void __launch_bounds__(kWG)
    DtKernel(const double *__restrict__ U, const BlockCoefs *__restrict__ coef, Geo G,
             int nblocks, double *__restrict__ partial) {
  __shared__ double wmin[kWG / 64];
  const int n0 = G.hi0 - G.lo0 + 1, n1 = G.hi1 - G.lo1 + 1, n2 = G.hi2 - G.lo2 + 1;
  const std::int64_t total = static_cast<std::int64_t>(n0) * n1 * n2 * nblocks;
  double m = DBL_MAX;
  for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * kWG + threadIdx.x; t < total;
       t += static_cast<std::int64_t>(gridDim.x) * kWG) {
    std::int64_t r = t;
    const int i = static_cast<int>(r % n0) + G.lo0;
    r /= n0;
    const int j = static_cast<int>(r % n1) + G.lo1;
    r /= n1;
    const int k = static_cast<int>(r % n2) + G.lo2;
    r /= n2;
    const BlockCoefs &C = coef[r];
    const double *u = U + r * G.V * G.cells + (static_cast<std::int64_t>(k) * G.e1 + j) * G.e0 + i;
    double s = fabs(u[0]) / C.dx[0];
    if (G.ndim > 1) s = s + fabs(u[G.cells]) / C.dx[1];
    if (G.ndim > 2) s = s + fabs(u[2 * G.cells]) / C.dx[2];
    m = DMin(m, 1.0 / s);
  }
  m = WaveMin(m);
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = wmin[0];
#pragma unroll
    for (int w = 1; w < kWG / 64; ++w) v = DMin(v, wmin[w]);
    partial[blockIdx.x] = v;
  }
}

__global__ void __launch_bounds__(64) MinFinalKernel(const double *__restrict__ partial, int n,
                                                     double *__restrict__ out) {
  double m = DBL_MAX;
  for (int t = threadIdx.x; t < n; t += 64) m = DMin(m, partial[t]);
  m = WaveMin(m);
  if (threadIdx.x == 0) out[0] = m;
}

// cfl times the minimum of the partials, into out[0] (the product the host forms after
// MinFinalKernel in the synchronous form, so the two give the same bits)
__global__ void __launch_bounds__(64) MinScaleKernel(const double *__restrict__ partial, int n,
                                                     double cfl, double *__restrict__ out) {
  double m = DBL_MAX;
  for (int t = threadIdx.x; t < n; t += 64) m = DMin(m, partial[t]);
  m = WaveMin(m);
  if (threadIdx.x == 0) out[0] = cfl * m;
}

// ---- fused stage path ----------------------------------------------------------------

// HllGen over state arrays: L, R point at component 0 of the face; component stride cs.
template <int V>
__device__ __forceinline__ void HllFace(const double *__restrict__ L, const double *__restrict__ R,
                                        std::int64_t cs, int d, double *F) {
  HllGen<V>([&](int n) { return L[n * cs]; }, [&](int n) { return R[n * cs]; }, d, F);
}

constexpr int kMaxV = 16;  // components handled by the update kernel

// ---- plane-tiled reconstruction + HLL (cubic blocks of N <= 16 cells per side) ----------
//
// ReconFluxKernel: one workgroup = PPW consecutive planes of one block for one direction. For
// each plane the WENO5Z (or linear) states of the plane's cells, extended by one cell along the
// direction, go to LDS; then the HLL flux of every face of the plane goes to the flux array
// [3][block][comp][brick] (x-face i at index i). The operations are those of FluxTaskKernel,
// so the fluxes are the same bits; this form also splits off the faces that read no ghost. PPW
// (planes per workgroup) changes only the work split and is picked by timing.
// PART selects the cells and faces of each plane row along the direction (ext index a of the
// N + 2 cells lo - 1 .. hi + 1; face f between ext cells f and f + 1):
//   0: every cell and face;
//   1: the cells whose WENO stencil reads no ghost cell (a in [3, N - 2]) and the faces
//      between two of them (f in [3, N - 3]): no dependence on the boundary exchange;
//   2: the rest (a in [0, 3] and [N - 2, N + 1], f in [0, 2] and [N - 2, N]); the cells 3 and
//      N - 2 are evaluated in both parts.
// The LDS holds the part's cells only: local cell q of a row is ext cell Cell(q), and face q
// lies between local cells Left(q) and Left(q) + 1.
template <int N, int PART>
struct PlaneSet {
  static constexpr int kCells = PART == 0 ? N + 2 : PART == 1 ? N - 4 : 8;
  static constexpr int kFaces = PART == 0 ? N + 1 : PART == 1 ? N - 5 : 6;
  __device__ static int Cell(int q) {
    return PART == 0 ? q : PART == 1 ? 3 + q : (q < 4 ? q : N - 6 + q);
  }
  __device__ static int Face(int q) {
    return PART == 0 ? q : PART == 1 ? 3 + q : (q < 3 ? q : N - 5 + q);
  }
  __device__ static int Left(int q) { return PART == 2 && q >= 3 ? q + 1 : q; }
};

template <int N, int NG, int V, int PART, int PPW>
__global__ void __launch_bounds__(kWG)
    ReconFluxKernel(const double *__restrict__ U, double *__restrict__ flux, int nblocks,
                    int recon) {
  constexpr int E = N + 2 * NG;  // brick extent
  using S = PlaneSet<N, PART>;
  constexpr int P = S::kCells * N;  // states of one plane per component
  constexpr int G = N / PPW;        // plane groups per (block, direction)
  __shared__ double sl[V * P], sr[V * P];
  // logical workgroup = (block * 3 + direction) * G + group; one block's planes are adjacent
  // and stay on one XCD
  const unsigned L = XcdRemap(blockIdx.x, gridDim.x);
  const int b = static_cast<int>(L / (3 * G)), r = static_cast<int>(L % (3 * G));
  const int d = r / G, plane0 = (r % G) * PPW;
  constexpr std::int64_t cs = static_cast<std::int64_t>(E) * E * E;
  const std::int64_t slab = cs * V * nblocks;
  const double *Ub = U + static_cast<std::int64_t>(b) * V * cs;
  const unsigned st = 8u * static_cast<unsigned>(d == 0 ? 1 : d == 1 ? E : E * E);
  for (int pp = 0; pp < PPW; ++pp) {
    const int plane = plane0 + pp;
    if (pp > 0) __syncthreads();  // the previous plane's faces have read the states
    // plane index of (local cell q along the direction, transverse tv): rows of kCells along
    // x for d = 0, else rows of N along x; consecutive threads take consecutive x
    for (int t = threadIdx.x; t < V * P; t += kWG) {
      const int n = t / P, u = t % P;
      int q, tv;
      if (d == 0) {
        q = u % S::kCells;
        tv = u / S::kCells;
      } else {
        tv = u % N;
        q = u / N;
      }
      const int a = S::Cell(q);
      int i, j, k;
      if (d == 0) {
        i = NG - 1 + a;
        j = NG + tv;
        k = NG + plane;
      } else if (d == 1) {
        i = NG + tv;
        j = NG - 1 + a;
        k = NG + plane;
      } else {
        i = NG + tv;
        j = NG + plane;
        k = NG - 1 + a;
      }
      const unsigned c = 8u * static_cast<unsigned>((k * E + j) * E + i);
      const double *qv = Ub + n * cs;
      double ql, qr;
      if (recon == 0)
        Weno5Z(LoadAt(qv, c - 2 * st), LoadAt(qv, c - st), LoadAt(qv, c), LoadAt(qv, c + st),
               LoadAt(qv, c + 2 * st), ql, qr);
      else
        LinearRecon(LoadAt(qv, c - st), LoadAt(qv, c), LoadAt(qv, c + st), ql, qr);
      sl[t] = ql;  // t = n * P + u and u is the plane index
      sr[t] = qr;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < S::kFaces * N; t += kWG) {
      int q, tv;
      if (d == 0) {
        q = t % S::kFaces;
        tv = t / S::kFaces;
      } else {
        tv = t % N;
        q = t / N;
      }
      const int f = S::Face(q), lq = S::Left(q);
      int pl, pr, i, j, k;
      if (d == 0) {  // face between ext cells f and f + 1 of row tv
        pl = tv * S::kCells + lq;
        pr = pl + 1;
        i = NG + f;
        j = NG + tv;
        k = NG + plane;
      } else {  // face between ext rows f and f + 1
        pl = lq * N + tv;
        pr = pl + N;
        i = NG + tv;
        j = d == 1 ? NG + f : NG + plane;
        k = d == 1 ? NG + plane : NG + f;
      }
      double Fv[V];
      HllFace<V>(sl + pl, sr + pr, P, d, Fv);
      double *fo = flux + d * slab + static_cast<std::int64_t>(b) * V * cs + (k * E + j) * E + i;
#pragma unroll
      for (int n = 0; n < V; ++n) fo[n * cs] = Fv[n];
    }
  }
}

// FluxUpdateKernel: one thread = one interior cell. Flux divergence (update.hpp:43-57) from
// the stored face fluxes, the RK averaging and update in the WeightedSumData form
// (update.hpp:71-90, 122-137), the derived field and the per-workgroup CFL minimum of the
// updated state.
template <int V>
__global__ void __launch_bounds__(kWG)
    FluxUpdateKernel(const double *__restrict__ flux, const double *U0, const double *base,
                     double *out, double *__restrict__ derived, double *__restrict__ partial,
                     const BlockCoefs *__restrict__ coef, Geo G, int nblocks, double beta,
                     const double *__restrict__ dtvar) {
  __shared__ double wmin[kWG / 64];
  const int n0 = G.hi0 - G.lo0 + 1, n1 = G.hi1 - G.lo1 + 1, n2 = G.hi2 - G.lo2 + 1;
  const unsigned L = XcdRemap(blockIdx.x, gridDim.x);  // = block * tiles + tile
  const int tiles = (n0 * n1 * n2 + kWG - 1) / kWG;
  const int b = static_cast<int>(L / tiles);
  const int t = static_cast<int>(L % tiles) * kWG + threadIdx.x;
  double m = DBL_MAX;
  if (t < n0 * n1 * n2) {
    const int i = t % n0 + G.lo0;
    const int r = t / n0;
    const int j = r % n1 + G.lo1;
    const int k = r / n1 + G.lo2;
    const std::int64_t slab = G.cells * V * nblocks;
    const std::int64_t cs = G.cells;
    const std::int64_t c0 = static_cast<std::int64_t>(b) * V * cs + (k * G.e1 + j) * G.e0 + i;
    const BlockCoefs &C = coef[b];
    const std::int64_t st[3] = {1, G.e0, static_cast<std::int64_t>(G.e0) * G.e1};
    double du[V];
    for (int d = 0; d < G.ndim; ++d) {
      const double *Fd = flux + d * slab + c0;
      const double A = C.area[d];
#pragma unroll
      for (int n = 0; n < V; ++n) {
        const double term = (A * Fd[n * cs + st[d]] - A * Fd[n * cs]);
        du[n] = d == 0 ? term : du[n] + term;
      }
    }
    const double bdt = beta * dtvar[0];
    const double w2 = 1.0 - beta;
    double u1[V];
#pragma unroll
    for (int n = 0; n < V; ++n) {
      const double dudt = -du[n] / C.vol;
      const double avg = beta * U0[c0 + n * cs] + w2 * base[c0 + n * cs];
      u1[n] = 1.0 * avg + bdt * dudt;
      out[c0 + n * cs] = u1[n];
    }
    if (derived)
      derived[static_cast<std::int64_t>(b) * cs + (k * G.e1 + j) * G.e0 + i] =
          0.5 * u1[3] * (u1[0] * u1[0] + u1[1] * u1[1] + u1[2] * u1[2]);
    double sp = fabs(u1[0]) / C.dx[0];
    if (G.ndim > 1) sp = sp + fabs(u1[1]) / C.dx[1];
    if (G.ndim > 2) sp = sp + fabs(u1[2]) / C.dx[2];
    m = 1.0 / sp;
  }
  if (!partial) return;
  m = WaveMin(m);
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    double v = wmin[0];
#pragma unroll
    for (int w = 1; w < kWG / 64; ++w) v = DMin(v, wmin[w]);
    partial[L] = v;
  }
}

// SendBoundBufs<flxcor_send> over stored face fluxes [dir][block][comp][brick].
__global__ void __launch_bounds__(64)
    FlxcorSendKernel(const FluxPatch *__restrict__ patches, const double *__restrict__ flux,
                     double *__restrict__ store, Geo G, int nblocks, int nc) {
  const FluxPatch &P = patches[blockIdx.x];
  const int t = blockIdx.y * 64 + threadIdx.x;
  if (t >= P.n[0] * P.n[1]) return;
  const int a = t % P.n[0], c = t / P.n[0];
  const std::int64_t cs = G.cells, slab = G.cells * nc * nblocks;
  const double *F = flux + P.d * slab + static_cast<std::int64_t>(P.fine) * nc * cs;
  const std::int64_t o00 = PatchFineCell(P, G, a, c, 0, 0);
  const std::int64_t o01 = P.step[0] > 1 ? PatchFineCell(P, G, a, c, 1, 0) : o00;
  const std::int64_t o10 = P.step[1] > 1 ? PatchFineCell(P, G, a, c, 0, 1) : o00;
  const std::int64_t o11 =
      P.step[0] > 1 && P.step[1] > 1 ? PatchFineCell(P, G, a, c, 1, 1) : o00;
  const std::int64_t dst = P.dst + a + static_cast<std::int64_t>(c) * P.rows;
  for (int n = 0; n < nc; ++n) {
    const double *Fn = F + n * cs;
    store[dst + static_cast<std::int64_t>(n) * P.comp] =
        RestrictFace(P.d, P.area, Fn[o00], Fn[o01], Fn[o10], Fn[o11], P.step[0], P.step[1]);
  }
}

// SetBounds<flxcor_recv>: the coarse block's stored fluxes on the patch's part of its face.
__global__ void __launch_bounds__(64)
    FlxcorSetKernel(const FluxPatch *__restrict__ patches, const double *__restrict__ store,
                    double *__restrict__ flux, Geo G, int nblocks, int nc) {
  const FluxPatch &P = patches[blockIdx.x];
  const int t = blockIdx.y * 64 + threadIdx.x;
  if (t >= P.n[0] * P.n[1]) return;
  const int a = t % P.n[0], c = t / P.n[0];
  const std::int64_t cs = G.cells, slab = G.cells * nc * nblocks;
  double *F = flux + P.d * slab + static_cast<std::int64_t>(P.coarse) * nc * cs +
              PatchCoarseCell(P, G, a, c);
  const std::int64_t src = P.dst + a + static_cast<std::int64_t>(c) * P.rows;
  for (int n = 0; n < nc; ++n) F[n * cs] = store[src + static_cast<std::int64_t>(n) * P.comp];
}

// burgers_package::MassHistory (benchmarks/burgers/burgers_package.cpp:406-439) for the 8
// octants of the mesh at once: sum over interior cells and components of mask * q * q * w,
// w = cell volume / (mesh volume + 1e-20), mask from the inclusive cell-centre test.
// Per-workgroup partials [workgroup][8]; the order of the sum is this build's own (the
// reference's Kokkos::Sum order is not fixed either).
struct Octants {
  double lo[8][3], hi[8][3];
};
__global__ void __launch_bounds__(kWG)
    MassHistoryKernel(const double *__restrict__ U, const DeviceBlockGeom *__restrict__ geom,
                      const BlockCoefs *__restrict__ coef, Geo G, int nblocks, Octants O,
                      double mesh_vol, double *__restrict__ partial) {
  __shared__ double acc[kWG / 64][8];
  const int n0 = G.hi0 - G.lo0 + 1, n1 = G.hi1 - G.lo1 + 1, n2 = G.hi2 - G.lo2 + 1;
  const std::int64_t per = static_cast<std::int64_t>(n0) * n1 * n2;
  const std::int64_t total = per * G.V * nblocks;
  double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (std::int64_t t = static_cast<std::int64_t>(blockIdx.x) * kWG + threadIdx.x; t < total;
       t += static_cast<std::int64_t>(gridDim.x) * kWG) {
    std::int64_t r = t;
    const int i = static_cast<int>(r % n0) + G.lo0;
    r /= n0;
    const int j = static_cast<int>(r % n1) + G.lo1;
    r /= n1;
    const int k = static_cast<int>(r % n2) + G.lo2;
    r /= n2;  // block * V + comp
    const int b = static_cast<int>(r / G.V);
    const DeviceBlockGeom &g = geom[b];
    const double w = coef[b].vol / (mesh_vol + 1e-20);
    const double x1 = g.x0[0] + (i + 0.5) * g.dx[0];
    const double x2 = g.x0[1] + (j + 0.5) * g.dx[1];
    const double x3 = g.x0[2] + (k + 0.5) * g.dx[2];
    const double q = U[r * G.cells + (static_cast<std::int64_t>(k) * G.e1 + j) * G.e0 + i];
#pragma unroll
    for (int o = 0; o < 8; ++o) {
      const double mask = (O.lo[o][0] <= x1) && (x1 <= O.hi[o][0]) && (O.lo[o][1] <= x2) &&
                          (x2 <= O.hi[o][1]) && (O.lo[o][2] <= x3) && (x3 <= O.hi[o][2]);
      s[o] += mask * q * q * w;
    }
  }
#pragma unroll
  for (int o = 0; o < 8; ++o) {
    double v = s[o];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0) acc[threadIdx.x >> 6][o] = v;
  }
  __syncthreads();
  if (threadIdx.x < 8) {
    double v = 0.0;
    for (int w2 = 0; w2 < kWG / 64; ++w2) v += acc[w2][threadIdx.x];
    partial[8 * blockIdx.x + threadIdx.x] = v;
  }
}

__global__ void __launch_bounds__(64)
    SumPartials8Kernel(const double *__restrict__ partial, int n, double *__restrict__ out) {
  if (threadIdx.x >= 8) return;
  double v = 0.0;
  for (int q = 0; q < n; ++q) v += partial[8 * q + threadIdx.x];
  out[threadIdx.x] = v;
}

// Final CFL minimum and EvolutionDriver::SetGlobalTimeStep on device (driver.cpp:210-269,
// dt_factor 2), with SimTime::KeepGoing's stop at tlim (basic_types.hpp:241).
// dtvar = {dt of the next cycle, time, estimate, dt of the last cycle, tm.dt}.
// advance 0 (start, ncycle 0): tm.dt is still the initial maximum and dt_init applies;
// advance 1 (end of a cycle): time += dt and the cycle's dt is kept before the rule;
// advance 2 (after a remesh): the estimate of the new blocks replaces the old one and the rule
// starts again from the dt of the last cycle.
// The loop of EvolutionDriver::Execute ends once time >= tlim. A cycle queued after that runs
// with dt = 0 (slot 0), which leaves the state, the time and the clock unchanged, so a host
// loop may queue cycles without reading the clock; slot 4 keeps the reference's tm.dt.
// One workgroup of kClockWG threads: strided partial minima, wavefront shuffles, then LDS.
constexpr int kClockWG = 1024;
__global__ void __launch_bounds__(kClockWG)
    ClockKernel(const double *__restrict__ partial, int n, double cfl, double *dtvar,
                int advance, ClockLimits L) {
  __shared__ double wmin[kClockWG / 64];
  double m = DBL_MAX;
  for (int t = threadIdx.x; t < n; t += kClockWG) m = DMin(m, partial[t]);
  m = WaveMin(m);
  if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    m = wmin[0];
    for (int w = 1; w < kClockWG / 64; ++w) m = DMin(m, wmin[w]);
    const double est = cfl * m;
    double time = dtvar[1];
    if (advance == 1) {
      if (!(time < L.tlim)) return;  // a cycle after the end: nothing moved
      time = time + dtvar[0];
      dtvar[1] = time;
      dtvar[3] = dtvar[0];
    }
    double dt = advance == 0 ? dtvar[4] : dtvar[3];
    if (L.dt_force > 0.0) {
      dt = L.dt_force;
    } else if (advance == 0 && L.dt_init_force && L.dt_init > 0.0) {
      dt = L.dt_init;
    } else {
      if (dt < 0.1 * DBL_MAX) dt *= 2.0;
      if (advance == 0) dt = DMin(dt, L.dt_init);
      dt = DMin(dt, est);
      dt = DMin(dt, L.dt_user);
      dt = DMax(L.dt_floor, DMin(dt, L.dt_ceil));
    }
    if (time < L.tlim && (L.tlim - time) < dt) dt = L.tlim - time;
    dtvar[4] = dt;
    dtvar[0] = time < L.tlim ? dt : 0.0;
    dtvar[2] = est;
  }
}

int Grid(std::int64_t total) {
  const std::int64_t want = (total + kWG - 1) / kWG;
  return static_cast<int>(want < 8192 ? want : 8192);
}

}  // namespace

// The split for nb blocks, by rows or by column segments: the one for which these two, squared and
// added, are least:
//   * the reconstructions of all wavefronts over the chip's SIMDs, those of y and z rows counted 1.1
//     times, more on long rows (their loads are strided, and fewer rows meet in a CU's cache);
//     segments share evenly among the XCDs, which take equal numbers of workgroups in their
//     order, only if the stripes divide by them or are many;
//   * 2.2 times the longest chain of a thread, which small meshes end with.
// Rows win until a mesh fills the chip many times over, and on blocks of up to 32. Measured, segments /
// rows: 8 blocks of 24^3 with 4 components 44.5 / 26.5 us, 64 blocks of 16^3 with 7 149 / 72, 960
// 1012 / 1065, 512 of 12^3 392 / 231, one of 128^3 526 / 743. Small meshes take their components in
// groups (the normal velocity repeated: 8 blocks of 8^3, 7 components 12.7 us in one, 9.8 in four), small
// blocks share workgroups (1024 blocks of 8^2: 43 us alone, 24 in units of 8).
static FluxSplit SplitFluxes(const Geo &G, const int n[3], int nb) {
  constexpr double kSimds = 1024.0, kWaves = kWG / 64, kStripe = 192.0;
  auto up = [](double a, double b) { return std::ceil(a / b); };
  FluxSplit best{};
  double least = 0.0;
  for (int pack = 1; pack <= 32 && pack <= std::max(nb, 1); pack *= 2) {
    // a packed unit's offsets are 32-bit
    if (pack > 1 && pack * G.V * G.cells >= std::int64_t(1) << 29) break;
    for (bool rows : {false, true}) {
      FluxSplit S{};
      S.pack = pack;
      S.rows = rows;
      double steps = 0.0, longest = 1.0, wgs = 0.0;
      for (int d = 0; d < G.ndim; ++d) {
        const double cols = static_cast<double>(n[d == 0 ? 1 : 0]) * n[d == 2 ? 1 : 2];
        double w;
        if (rows || d == 0) {
          w = up(up((n[d] + 2.0) * cols * pack - 1.0, 63.0), kWaves);
          steps += w * (d == 0 ? 1.0 : 1.1 + 0.006 * std::max(n[d] - 16, 0));
        } else {
          const double segs = up(n[d] + 1.0, kSegFaces);
          S.seg[d] = static_cast<int>(up(n[d] + 1.0, segs));
          w = up(cols * segs * pack, kWG);
          steps += w * (S.seg[d] + 1.0);
          longest = std::max(longest, S.seg[d] + 1.0);
        }
        S.wgs[d] = static_cast<int>(w);
        wgs += w;
      }
      S.stripes = rows ? 1 : std::max(1, static_cast<int>(wgs / kStripe));
      for (int groups : {1, 2, 4}) {
        if (groups > G.V || (groups > 1 && !rows)) continue;
        S.comps = (G.V + groups - 1) / groups;
        S.chunks = (G.V + S.comps - 1) / S.comps;
        const double comps = S.comps + (S.chunks > 1), units = up(nb, pack) * S.chunks;
        const double parts = units * S.stripes;
        const double uneven = rows ? 1.0 : up(parts, kXcds) * kXcds / parts;
        const double cost =
            comps * std::hypot(steps * kWaves * units / kSimds * uneven, 2.2 * longest);
        // by rows, blocks share workgroups only for a gain: the order suits the caches less (27
        // blocks of 32^3 228 us alone, 265 in units of 8)
        if (least > 0.0 && cost >= least * (rows && pack > best.pack ? 0.97 : 1.0)) continue;
        least = cost;
        best = S;
      }
    }
  }
  return best;
}

pth_status BurgersFluxes(const Topology &t, int V, const double *U, double *flux, int recon,
                         hipStream_t s) {
  ProfScope prof("fluxes", s);
  const Geo G = MakeGeo(t, V);
  const int nb = static_cast<int>(t.blocks.size());
  const int n[3] = {t.fine.n[0], t.fine.n[1], t.fine.n[2]};
  const FluxSplit S = SplitFluxes(G, n, nb);
  const dim3 grid(static_cast<unsigned>(S.wgs[0] + S.wgs[1] + S.wgs[2]) *
                  static_cast<unsigned>(S.chunks * ((nb + S.pack - 1) / S.pack)));
  const bool wide = G.cells >= std::int64_t(1) << 29;
  auto run = [&](auto kernel) -> pth_status {
    PTH_LAUNCH(kernel, grid, dim3(kWG), 0, s, U, flux, G, nb, S);
    return PTH_COMPLETE;
  };
  auto form = [&](auto rows) -> pth_status {
    constexpr bool ROWS = decltype(rows)::value;
    if (recon == 0)
      return wide ? run(FluxTaskKernel<0, true, ROWS>) : run(FluxTaskKernel<0, false, ROWS>);
    return wide ? run(FluxTaskKernel<1, true, ROWS>) : run(FluxTaskKernel<1, false, ROWS>);
  };
  return S.rows ? form(std::true_type()) : form(std::false_type());
}

pth_status FluxDivergence(const Topology &t, int V, const double *flux, double *dudt,
                          const BlockCoefs *coef, hipStream_t s) {
  ProfScope prof("flux_div", s);
  const Geo G = MakeGeo(t, V);
  const int nb = static_cast<int>(t.blocks.size());
  const dim3 grid(ChunkGrid(t, static_cast<std::int64_t>(V) * nb));
  if (grid.x == 0) return PTH_COMPLETE;
  auto *kernel = SmallBricks(t) ? FluxDivKernel<true> : FluxDivKernel<false>;
  PTH_LAUNCH(kernel, grid, dim3(kWG), 0, s, flux, dudt, coef, G, nb);
  return PTH_COMPLETE;
}

pth_status WeightedSum(const double *x, const double *y, double w1, double w2, double *z,
                       std::int64_t n, hipStream_t s) {
  if (n == 0) return PTH_COMPLETE;
  ProfScope prof("weighted_sum", s);
  PTH_LAUNCH(WsumKernel, dim3(Grid(n)), dim3(kWG), 0, s, x, y, w1, w2, z, n);
  return PTH_COMPLETE;
}

pth_status BurgersDerived(const Topology &t, int V, const double *U, double *out,
                          hipStream_t s) {
  ProfScope prof("derived", s);
  const Geo G = MakeGeo(t, V);
  const int nb = static_cast<int>(t.blocks.size());
  const std::int64_t total =
      static_cast<std::int64_t>(t.fine.n[0]) * t.fine.n[1] * t.fine.n[2] * nb;
  PTH_LAUNCH(DerivedKernel, dim3(Grid(total)), dim3(kWG), 0, s, U, out, G, nb);
  return PTH_COMPLETE;
}

int FusedUpdatePartials(const Topology &t) {
  const int cells = t.fine.n[0] * t.fine.n[1] * t.fine.n[2];
  return ((cells + kWG - 1) / kWG) * static_cast<int>(t.blocks.size());
}

pth_status FlxcorSend(const Topology &t, const FluxCorrection &fc, const double *flux,
                      hipStream_t s) {
  if (fc.host.empty()) return PTH_COMPLETE;
  ProfScope prof("flxcor_send", s);
  const Geo G = MakeGeo(t, fc.ncomp);
  const int nb = static_cast<int>(t.blocks.size());
  const dim3 grid(static_cast<unsigned>(fc.host.size()), (fc.max_cells + 63) / 64);
  PTH_LAUNCH(FlxcorSendKernel, grid, dim3(64), 0, s, fc.dev, flux, fc.store, G, nb,
             fc.ncomp);
  return PTH_COMPLETE;
}

pth_status FlxcorSet(const Topology &t, const FluxCorrection &fc, double *flux, hipStream_t s) {
  if (fc.host.empty()) return PTH_COMPLETE;
  ProfScope prof("flxcor_set", s);
  const Geo G = MakeGeo(t, fc.ncomp);
  const int nb = static_cast<int>(t.blocks.size());
  const dim3 grid(static_cast<unsigned>(fc.host.size()), (fc.max_cells + 63) / 64);
  PTH_LAUNCH(FlxcorSetKernel, grid, dim3(64), 0, s, fc.dev, fc.store, flux, G, nb,
             fc.ncomp);
  return PTH_COMPLETE;
}

bool ReconFluxSupported(const Topology &t, int V) {
  const Extent &f = t.fine;
  const bool cubic = t.ndim == 3 && f.n[0] == f.n[1] && f.n[1] == f.n[2] &&
                     f.g[0] == f.g[1] && f.g[1] == f.g[2];
  return cubic && (f.n[0] == 16 || f.n[0] == 8) && f.g[0] == 4 && V >= 4 && V <= 13;
}

pth_status BurgersReconFlux(const Topology &t, int V, const double *U, double *flux, int recon,
                            int part, int ppw, hipStream_t s) {
  if (!ReconFluxSupported(t, V) || part < 0 || part > 2 || (ppw != 1 && ppw != 2 && ppw != 4)) {
    SetError("plane-tiled reconstruction: unsupported block shape, component count or split");
    return PTH_FAIL;
  }
  ProfScope prof(part == 0 ? "recon_flux" : part == 1 ? "recon_flux_inner" : "recon_flux_outer",
                 s);
  const int nb = static_cast<int>(t.blocks.size());
  const int N = t.fine.n[0];
  const dim3 grid(static_cast<unsigned>(3 * (N / ppw) * nb));
#define PTH_RF_LAUNCH(NN, NV, PT, PW)                                                         \
  PTH_LAUNCH((ReconFluxKernel<NN, 4, NV, PT, PW>), grid, dim3(kWG), 0, s, U, flux, nb, \
             recon)
#define PTH_RF_PPW(NN, NV, PT)                                                                \
  if (ppw == 1)                                                                               \
    PTH_RF_LAUNCH(NN, NV, PT, 1);                                                             \
  else if (ppw == 2)                                                                          \
    PTH_RF_LAUNCH(NN, NV, PT, 2);                                                             \
  else                                                                                        \
    PTH_RF_LAUNCH(NN, NV, PT, 4);
#define PTH_RF_PARTS(NN, NV)                                                                  \
  if (part == 0) {                                                                            \
    PTH_RF_PPW(NN, NV, 0)                                                                     \
  } else if (part == 1) {                                                                     \
    PTH_RF_PPW(NN, NV, 1)                                                                     \
  } else {                                                                                    \
    PTH_RF_PPW(NN, NV, 2)                                                                     \
  }
#define PTH_RF_CASE(NV)                                                                       \
  case NV:                                                                                    \
    if (N == 16) {                                                                            \
      PTH_RF_PARTS(16, NV)                                                                    \
    } else {                                                                                  \
      PTH_RF_PARTS(8, NV)                                                                     \
    }                                                                                         \
    break;
  switch (V) {
    PTH_RF_CASE(4)
    PTH_RF_CASE(5)
    PTH_RF_CASE(6)
    PTH_RF_CASE(7)
    PTH_RF_CASE(8)
    PTH_RF_CASE(9)
    PTH_RF_CASE(10)
    PTH_RF_CASE(11)
    PTH_RF_CASE(12)
    PTH_RF_CASE(13)
  }
#undef PTH_RF_CASE
#undef PTH_RF_PARTS
#undef PTH_RF_PPW
#undef PTH_RF_LAUNCH
  return PTH_COMPLETE;
}

pth_status BurgersFluxUpdate(const Topology &t, int V, const double *flux, const double *U0,
                             const double *base, double *out, double *derived, double *partial,
                             const BlockCoefs *coef, double beta, const double *dtvar,
                             hipStream_t s) {
  if (V > kMaxV || V < 4) {
    SetError("flux update supports 4 to 16 components");
    return PTH_FAIL;
  }
  ProfScope prof("flux_update", s);
  const Geo G = MakeGeo(t, V);
  const int nb = static_cast<int>(t.blocks.size());
  const int cells = t.fine.n[0] * t.fine.n[1] * t.fine.n[2];
  const dim3 grid(((cells + kWG - 1) / kWG) * nb);
#define PTH_FU_CASE(NV)                                                                       \
  case NV:                                                                                    \
    PTH_LAUNCH(FluxUpdateKernel<NV>, grid, dim3(kWG), 0, s, flux, U0, base, out,      \
               derived, partial, coef, G, nb, beta, dtvar);                           \
    break;
  switch (V) {
    PTH_FU_CASE(4)
    PTH_FU_CASE(5)
    PTH_FU_CASE(6)
    PTH_FU_CASE(7)
    PTH_FU_CASE(8)
    PTH_FU_CASE(9)
    PTH_FU_CASE(10)
    PTH_FU_CASE(11)
    PTH_FU_CASE(12)
    PTH_FU_CASE(13)
    PTH_FU_CASE(14)
    PTH_FU_CASE(15)
    PTH_FU_CASE(16)
  }
#undef PTH_FU_CASE
  return PTH_COMPLETE;
}

pth_status BurgersMassHistory(const Topology &t, int V, const double *U,
                              const DeviceBlockGeom *geom, const BlockCoefs *coef,
                              const double mesh_lo[3], const double mesh_hi[3], double *scratch,
                              int nscratch, double *out, hipStream_t s) {
  ProfScope prof("mass_history", s);
  // octants in the reference order (burgers_package.cpp:104-119): x outer, then y, then z
  Octants O;
  double mid[3], vol = 1.0;
  for (int d = 0; d < 3; ++d) {
    vol *= (mesh_hi[d] - mesh_lo[d]);
    mid[d] = 0.5 * (mesh_lo[d] + mesh_hi[d]);
  }
  int o = 0;
  for (int s1 = 0; s1 < 2; ++s1)
    for (int s2 = 0; s2 < 2; ++s2)
      for (int s3 = 0; s3 < 2; ++s3, ++o) {
        const int side[3] = {s1, s2, s3};
        for (int d = 0; d < 3; ++d) {
          O.lo[o][d] = side[d] ? mid[d] : mesh_lo[d];
          O.hi[o][d] = side[d] ? mesh_hi[d] : mid[d];
        }
      }
  const Geo G = MakeGeo(t, V);
  const int nb = static_cast<int>(t.blocks.size());
  const std::int64_t total =
      static_cast<std::int64_t>(t.fine.n[0]) * t.fine.n[1] * t.fine.n[2] * V * nb;
  int grid = Grid(total);
  if (grid > nscratch / 8) grid = nscratch / 8;
  PTH_LAUNCH(MassHistoryKernel, dim3(grid), dim3(kWG), 0, s, U, geom, coef, G, nb, O,
             vol, scratch);
  PTH_LAUNCH(SumPartials8Kernel, dim3(1), dim3(64), 0, s, scratch, grid, out);
  return PTH_COMPLETE;
}

pth_status BurgersClock(const double *partial, int n, double cfl, double *dtvar, int advance,
                        const ClockLimits &lim, hipStream_t s) {
  ProfScope prof("clock", s);
  PTH_LAUNCH(ClockKernel, dim3(1), dim3(kClockWG), 0, s, partial, n, cfl, dtvar,
             advance, lim);
  return PTH_COMPLETE;
}

int BurgersDtPartials(const Topology &t) {
  return Grid(static_cast<std::int64_t>(t.fine.n[0]) * t.fine.n[1] * t.fine.n[2] *
              static_cast<std::int64_t>(t.blocks.size()));
}

pth_status BurgersDtToDevice(const Topology &t, int V, const double *U, const BlockCoefs *coef,
                             double *partial, int npartial, double cfl, double *out,
                             hipStream_t s) {
  ProfScope prof("dt_reduce", s);
  const Geo G = MakeGeo(t, V);
  const int nb = static_cast<int>(t.blocks.size());
  const int grid = BurgersDtPartials(t);
  if (grid > npartial) {
    SetError("CFL reduction: more partials than the scratch holds");
    return PTH_FAIL;
  }
  PTH_LAUNCH(DtKernel, dim3(grid), dim3(kWG), 0, s, U, coef, G, nb, partial);
  PTH_LAUNCH(MinScaleKernel, dim3(1), dim3(64), 0, s, partial, grid, cfl, out);
  return PTH_COMPLETE;
}

pth_status BurgersDtMin(const Topology &t, int V, const double *U, const BlockCoefs *coef,
                        double *partial, int npartial, double *out, hipStream_t s) {
  ProfScope prof("dt_reduce", s);
  const Geo G = MakeGeo(t, V);
  const int nb = static_cast<int>(t.blocks.size());
  const std::int64_t total =
      static_cast<std::int64_t>(t.fine.n[0]) * t.fine.n[1] * t.fine.n[2] * nb;
  int grid = Grid(total);
  if (grid > npartial) grid = npartial;
  PTH_LAUNCH(DtKernel, dim3(grid), dim3(kWG), 0, s, U, coef, G, nb, partial);
  PTH_LAUNCH(MinFinalKernel, dim3(1), dim3(64), 0, s, partial, grid, out);
  return PTH_COMPLETE;
}

}  // namespace pth
