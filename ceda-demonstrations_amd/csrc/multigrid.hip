// Geometric-multigrid preconditioner for the implicit path on gfx950: one
// V-cycle per application for A = I - gamma J (J the 5-point stencil of the
// RHS face tables), with the settings of the reference's hypre PFMG
// preconditioner (preconditioner_hypre.cpp:51-102, 142-160;
// diffusion_2D.hpp:187-193): zero initial guess, one cycle, red/black
// Gauss-Seidel smoothing, by default symmetric (PFMG relax type 2) with 2 pre
// and 2 post sweeps; relax type 3 (nonsymmetric: red then black both before
// and after the coarse correction) and the sweep count are the reference's
// --pfmg_relax / --pfmg_nrelax options (diffusion_2D.cpp:137-151).
//
// Hierarchy (Dirichlet, the manufactured problem): vertex-centred coarsening
// n -> n/2 (coarse node I on fine node 2I+1) until a side would drop below 3;
// coarse operators rediscretised from the fine face tables (coarse face I on
// fine node 2I: (f[2I] + f[2I+1]) / 8).  Periodic (the reference's problem,
// even sides only): coarse node I on fine node 2I, coarse face I spanning
// fine faces 2I-1 and 2I ((f[2I-1] + f[2I]) / 8, f[-1] = f[n-1]), coarsening
// while the coarse sides stay even and at least 4, every neighbour, transfer
// and sweep wrapping around (red/black colours stay consistent across the
// wrap because every side is even);
// full-weighting restriction = P^T/4 of the bilinear prolongation; red then
// black sweeps before the coarse correction, black then red after (the
// adjoint), 4 symmetric pairs on the coarsest grid.  The cycle is therefore
// symmetric and usable inside PCG.
//
// Every operation is element-wise or in-place red/black with a fixed
// expression order and no FMA contraction, so the V-cycle equals the CPU
// oracle's bit for bit (but for values below 1e-270, see mg_quot).
//
// Execution: two launches per level (k_mg_tile), on tiles held in registers:
// down (zero guess, all pre-sweeps, residual, restriction) reads b and writes
// x and the coarse b; up (prolongation, all post-sweeps) reads x, b and the
// coarse x and writes x.  The trailing levels of at most kMGCoarseCells cells
// run in one workgroup (k_mg_coarse).  The finest level works on the caller's
// vectors directly; gamma lives in device memory and the other levels'
// launches are captured as one HIP graph.  With more than kMGTileRelax
// sweep pairs (the tiles' halos would outgrow them), and on hierarchies that
// end in a grid too large for one workgroup, every sweep is a launch of its
// own (vcycle), captured as one graph; it clears with a fill kernel, not a
// memset.
//
// One cycle at 2048^2: the per-sweep launches moved about 290 bytes per fine
// cell and took 0.62 ms; the tiles move about 55 and take 0.16 ms (finest
// level 29 + 35 us).
#include <cstring>
#include <type_traits>

#include "diffusion_internal.hpp"

using namespace ceda;

struct MGLevel {
  int64_t nx = 0, ny = 0;
  double *fx = nullptr, *fy = nullptr;  // face tables, nx+1 / ny+1
  double *x = nullptr, *b = nullptr, *r = nullptr;
};

// a level as the kernels see it
struct MGLevelD {
  int64_t nx, ny;
  const double *fx, *fy;
  double *x, *b, *r;
};

struct MGHierarchy {
  int nl = 0;
  MGLevel L[24];
  int per = 0;              // periodic grid
  double* gamma = nullptr;  // device scalar
  double* h_gamma = nullptr;
  hipGraphExec_t graph = nullptr;
  int relax = 2, nrelax = 2;  // the options the graph was captured with
  long cycles = 0;            // V-cycles applied (MGPSolve calls)
  int lc = 0;                 // first level of the single-workgroup coarse cycle
  size_t lc_lds = 0;          // its LDS bytes
  double* ctab = nullptr;     // the face tables of its levels, one after another
};

namespace {

constexpr int kMGMaxL = 24;
constexpr int kCoarse = 4;
constexpr int64_t kMGCoarseCells = 1024;  // levels this small run in one workgroup (k_mg_coarse)

unsigned grid_of(int64_t n)
{
  int64_t g = (n + kBlock - 1) / kBlock;
  if (g < 1) g = 1;
  if (g > 65536) g = 65536;
  return (unsigned)g;
}

__device__ inline void mg_row(int64_t nx, int64_t ny, const double* __restrict__ fx,
                              const double* __restrict__ fy, double g, const double* x, int64_t i,
                              int64_t j, int per, double& off, double& d)
{
  const int64_t k = j * nx + i;
  double xw, xe, xs, xn;
  if (per) {
    xw = x[j * nx + (i > 0 ? i - 1 : nx - 1)];
    xe = x[j * nx + (i < nx - 1 ? i + 1 : 0)];
    xs = x[(j > 0 ? j - 1 : ny - 1) * nx + i];
    xn = x[(j < ny - 1 ? j + 1 : 0) * nx + i];
  } else {
    xw = i > 0 ? x[k - 1] : 0.0;
    xe = i < nx - 1 ? x[k + 1] : 0.0;
    xs = j > 0 ? x[k - nx] : 0.0;
    xn = j < ny - 1 ? x[k + nx] : 0.0;
  }
  off = ((fx[i] * xw + fx[i + 1] * xe) + fy[j] * xs) + fy[j + 1] * xn;
  d = 1.0 + g * ((fx[i] + fx[i + 1]) + (fy[j] + fy[j + 1]));
}

// ---- per-point operations, shared by the per-level kernels and the
// single-workgroup coarse cycle (same arithmetic, same order)

// q-th point of one colour of a red/black Gauss-Seidel sweep (red: i + j
// even), in place
__device__ inline void pt_sweep(const MGLevelD& L, double g, int color, int per, int64_t q)
{
  const int64_t half = (L.nx + 1) / 2;
  const int64_t j = q / half;
  const int64_t i = 2 * (q - j * half) + ((j + color) & 1);
  if (i >= L.nx) return;
  double off, d;
  mg_row(L.nx, L.ny, L.fx, L.fy, g, L.x, i, j, per, off, d);
  L.x[j * L.nx + i] = (L.b[j * L.nx + i] + g * off) / d;
}

__device__ inline void pt_resid(const MGLevelD& L, double g, int per, int64_t k)
{
  const int64_t j = k / L.nx, i = k - j * L.nx;
  double off, d;
  mg_row(L.nx, L.ny, L.fx, L.fy, g, L.x, i, j, per, off, d);
  double t = d * L.x[k];
  t = t - g * off;
  L.r[k] = L.b[k] - t;
}

// full weighting of F's residual onto coarse node q of C: (I, J) = fine node
// (2I+1, 2J+1), or (2I, 2J) with wrap-around on a periodic grid
__device__ inline void pt_restrict(const MGLevelD& F, const MGLevelD& C, int per, int64_t q)
{
  const int64_t nx = F.nx, ny = F.ny;
  const double* __restrict__ r = F.r;
  const int64_t J = q / C.nx, I = q - J * C.nx;
  const int64_t i = per ? 2 * I : 2 * I + 1, j = per ? 2 * J : 2 * J + 1;
  auto R = [&](int64_t a, int64_t c) -> double {
    if (per) return r[((c + ny) % ny) * nx + ((a + nx) % nx)];
    return (a < nx && c < ny) ? r[c * nx + a] : 0.0;
  };
  double t = 4.0 * R(i, j);
  t = t + 2.0 * ((R(i - 1, j) + R(i + 1, j)) + (R(i, j - 1) + R(i, j + 1)));
  t = t + ((R(i - 1, j - 1) + R(i + 1, j - 1)) + (R(i - 1, j + 1) + R(i + 1, j + 1)));
  C.b[q] = t * 0.0625;
}

// bilinear prolongation of C's correction onto fine point k of F, added: a
// fine index coincides with coarse index I (Dirichlet: odd i, I = i/2;
// periodic: even i, I = i/2) or lies between I and I+1 (Dirichlet:
// I = i/2 - 1, zero outside; periodic: I = i/2, wrapping)
__device__ inline void pt_prolong(const MGLevelD& F, const MGLevelD& C, int per, int64_t k)
{
  const int64_t cx = C.nx, cy = C.ny;
  const double* __restrict__ xc = C.x;
  const int64_t j = k / F.nx, i = k - j * F.nx;
  auto XC = [&](int64_t a, int64_t c) -> double {
    if (per) return xc[((c + cy) % cy) * cx + ((a + cx) % cx)];
    return (a >= 0 && a < cx && c >= 0 && c < cy) ? xc[c * cx + a] : 0.0;
  };
  const bool cxo = per ? !(i & 1) : (i & 1), cyo = per ? !(j & 1) : (j & 1);
  const int64_t I = (per || cxo) ? i / 2 : i / 2 - 1;
  const int64_t J = (per || cyo) ? j / 2 : j / 2 - 1;
  double v;
  if (cxo && cyo) v = XC(I, J);
  else if (cyo) v = 0.5 * (XC(I, J) + XC(I + 1, J));
  else if (cxo) v = 0.5 * (XC(I, J) + XC(I, J + 1));
  else v = 0.25 * ((XC(I, J) + XC(I + 1, J)) + (XC(I, J + 1) + XC(I + 1, J + 1)));
  F.x[k] = F.x[k] + v;
}

#define CEDA_MG_GRID_STRIDE(q, n) \
  for (int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x; q < (n); q += (int64_t)gridDim.x * kBlock)

__global__ __launch_bounds__(kBlock) void k_mg_fill0(int64_t n, double* __restrict__ x)
{
  CEDA_MG_GRID_STRIDE(k, n) x[k] = 0.0;
}

__global__ __launch_bounds__(kBlock) void k_mg_sweep(const MGLevelD L, const double* __restrict__ gp, int color,
                                                     int per)
{
  const double g = *gp;
  CEDA_MG_GRID_STRIDE(q, (L.nx + 1) / 2 * L.ny) pt_sweep(L, g, color, per, q);
}

__global__ __launch_bounds__(kBlock) void k_mg_resid(const MGLevelD L, const double* __restrict__ gp, int per)
{
  const double g = *gp;
  CEDA_MG_GRID_STRIDE(k, L.nx * L.ny) pt_resid(L, g, per, k);
}

__global__ __launch_bounds__(kBlock) void k_mg_restrict(const MGLevelD F, const MGLevelD C, int per)
{
  CEDA_MG_GRID_STRIDE(q, C.nx * C.ny) pt_restrict(F, C, per, q);
}

__global__ __launch_bounds__(kBlock) void k_mg_prolong(const MGLevelD F, const MGLevelD C, int per)
{
  CEDA_MG_GRID_STRIDE(k, F.nx * F.ny) pt_prolong(F, C, per, k);
}

// n / d for many n and one d: the correctly rounded quotient from the
// correctly rounded reciprocal y = 1 / d (two exact-residual corrections;
// Markstein, IBM J. Res. Dev. 34 (1990)) and, for zeros of either sign,
// infinities and NaN, the division's own fix-up: 6 instructions instead of
// the 13 of a division.  The bits are the division's while d, the diagonal of
// I - gamma J, is from 1 to 2^50 and n zero, not finite or at least 2^-900;
// below, where a residual may underflow, the last bits may differ.  (A test for
// such n at every quotient, or once per pass with the least |n| kept, made a
// cycle at 2048^2 185 us long instead of 166.)
__device__ inline double mg_quot(double n, double d, double y)  // n / d, y = 1 / d
{
  double q = n * y;
  q = __builtin_fma(__builtin_fma(-d, q, n), y, q);
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-d, q, n), y, q), d, n);
}

// The V-cycle from level l0 down to the coarsest and back, in one workgroup:
// the same operations in the same order as the per-level launches.  Every
// array of these levels (x, b, r and the face tables) is in LDS; b of level l0
// comes in from global memory (the restriction of the level above, or the
// preconditioner's input) and x of level l0 goes back (for the prolongation to
// the level above, or as the result).  Used for the trailing levels whose
// arrays fit in a workgroup's LDS (mg_coarse_lds).
//
// The cycle is a chain of about 55 phases (half-sweeps, residuals, transfers)
// of 0.4 to 0.6 us each: an LDS round trip, the update's dependent operations
// and a barrier.  Every operation's code stands once, in one loop over the
// levels, and nothing is unrolled (4 KB: a version that kept the cells'
// coefficients in registers, 77 KB of instructions that each run once or
// twice, took 71 us at 64^2).  Threads map to a level as 32 x 32, so that no
// index is divided, LDS is addressed by words from one base, Dirichlet ghosts
// read a zero word, and the diagonals are divided once.  A cycle from 64^2
// took 83 us through generic pointers and index divisions; from 32^2, where
// it starts now, 30 us, and the 64^2 level 11 us on tiles (46 us in here).
constexpr int kCoarseThreads = 1024, kCoarseRows = kCoarseThreads / 32;
constexpr int kCoarseMaxL = 16;
struct MGCoarseLevel {
  int nx, ny;
  int fx, fy, x, b, r, d, y;  // LDS words of the level's arrays (y = 1 / d)
  int pad;
};
struct MGCoarse {
  int nl, tab;                  // levels; words of their face tables, which start at word 1
  const double* tables;         // the face tables, in the order of the levels
  const double* b;              // level l0: input and result
  double* x;
  MGCoarseLevel lev[kCoarseMaxL];
};
__global__ __launch_bounds__(kCoarseThreads) void k_mg_coarse(const MGCoarse G, const double* __restrict__ gp,
                                                               int relax, int nrelax, int per)
{
  extern __shared__ double lds[];
  const double g = *gp;
  const int p0 = (relax == 2) ? 1 : 0;
  const int tid = threadIdx.x, tx = tid & 31, ty = tid >> 5;
  MGCoarseLevel L = G.lev[0];
  if (tid == 0) lds[0] = 0.0;
  for (int q = tid; q < G.tab; q += kCoarseThreads) lds[1 + q] = G.tables[q];
  for (int q = tid; q < L.nx * L.ny; q += kCoarseThreads) lds[L.b + q] = G.b[q];
  __syncthreads();
  // every level's diagonal and its reciprocal
#pragma unroll 1
  for (int l = 0; l < G.nl; l++) {
    const MGCoarseLevel M = G.lev[l];
#pragma unroll 1
    for (int j = ty; j < M.ny; j += kCoarseRows)
#pragma unroll 1
      for (int i = tx; i < M.nx; i += 32) {
        const double d = 1.0 + g * ((lds[M.fx + i] + lds[M.fx + i + 1]) + (lds[M.fy + j] + lds[M.fy + j + 1]));
        lds[M.d + j * M.nx + i] = d;
        lds[M.y + j * M.nx + i] = 1.0 / d;
      }
  }
  __syncthreads();
  // the off-diagonal sum at cell (i, j) of level L
  auto row = [&](int i, int j) {
    const int k = L.x + j * L.nx + i;
    const double f0 = lds[L.fx + i], f1 = lds[L.fx + i + 1], h0 = lds[L.fy + j], h1 = lds[L.fy + j + 1];
    const int w = i > 0 ? k - 1 : (per ? k + L.nx - 1 : 0), e = i < L.nx - 1 ? k + 1 : (per ? k - L.nx + 1 : 0);
    const int s = j > 0 ? k - L.nx : (per ? k + (L.ny - 1) * L.nx : 0), n = j < L.ny - 1 ? k + L.nx : (per ? L.x + i : 0);
    return ((f0 * lds[w] + f1 * lds[e]) + h0 * lds[s]) + h1 * lds[n];
  };
  int l = 0;
  bool up = false;
  for (;;) {
    // sweeps: red then black before the coarse correction, p0 first after it;
    // both on the coarsest level.  The first one starts from x = 0 (and black
    // reads red cells only, so nothing need be cleared before it).
    const bool last = l == G.nl - 1;
    const int nsw = last ? 4 * kCoarse : 2 * nrelax, half = (L.nx + 1) / 2;
    if (!up && nsw == 0) {
      for (int q = tid; q < L.nx * L.ny; q += kCoarseThreads) lds[L.x + q] = 0.0;
      __syncthreads();
    }
#pragma unroll 1
    for (int k = 0; k < nsw; k++) {
      const int color = (k & 1) ^ ((up || (last && k >= 2 * kCoarse)) ? p0 : 0);
#pragma unroll 1
      for (int j = ty; j < L.ny; j += kCoarseRows)
#pragma unroll 1
        for (int q = tx; q < half; q += 32) {
          const int i = 2 * q + ((j + color) & 1);
          if (i >= L.nx) continue;
          const int c = j * L.nx + i;
          const double off = (up || k > 0) ? row(i, j) : 0.0;
          lds[L.x + c] = mg_quot(lds[L.b + c] + g * off, lds[L.d + c], lds[L.y + c]);
        }
      __syncthreads();
    }
    if (!up && !last) {
#pragma unroll 1
      for (int j = ty; j < L.ny; j += kCoarseRows)
#pragma unroll 1
        for (int i = tx; i < L.nx; i += 32) {
          const int k = j * L.nx + i;
          double t = lds[L.d + k] * lds[L.x + k];
          t = t - g * row(i, j);
          lds[L.r + k] = lds[L.b + k] - t;
        }
      __syncthreads();
      const MGCoarseLevel C = G.lev[++l];
#pragma unroll 1
      for (int J = ty; J < C.ny; J += kCoarseRows)
#pragma unroll 1
        for (int I = tx; I < C.nx; I += 32) {
          const int i = per ? 2 * I : 2 * I + 1, j = per ? 2 * J : 2 * J + 1;
          const int iw = i > 0 ? i - 1 : L.nx - 1, ie = i + 1, js = j > 0 ? j - 1 : L.ny - 1, jn = j + 1;
          // (an even periodic side never ends on a coarse node)
          auto R = [&](int a, int c) { return lds[(a < L.nx && c < L.ny) ? L.r + c * L.nx + a : 0]; };
          double t = 4.0 * R(i, j);
          t = t + 2.0 * ((R(iw, j) + R(ie, j)) + (R(i, js) + R(i, jn)));
          t = t + ((R(iw, js) + R(ie, js)) + (R(iw, jn) + R(ie, jn)));
          lds[C.b + J * C.nx + I] = t * 0.0625;
        }
      __syncthreads();
      L = C;
      continue;
    }
    up = true;
    if (l == 0) break;
    const MGCoarseLevel C = L;
    L = G.lev[--l];
#pragma unroll 1
    for (int j = ty; j < L.ny; j += kCoarseRows)
#pragma unroll 1
      for (int i = tx; i < L.nx; i += 32) {
        const bool cxo = per ? !(i & 1) : (i & 1), cyo = per ? !(j & 1) : (j & 1);
        const int I = (per || cxo) ? i / 2 : i / 2 - 1, J = (per || cyo) ? j / 2 : j / 2 - 1;
        auto XC = [&](int a, int c) {
          if (per) {
            a -= a >= C.nx ? C.nx : 0;
            c -= c >= C.ny ? C.ny : 0;
          }
          return lds[(a >= 0 && a < C.nx && c >= 0 && c < C.ny) ? C.x + c * C.nx + a : 0];
        };
        const double a00 = XC(I, J), a10 = XC(I + 1, J), a01 = XC(I, J + 1), a11 = XC(I + 1, J + 1);
        double v = 0.25 * ((a00 + a10) + (a01 + a11));
        if (cyo) v = 0.5 * (a00 + a10);
        if (cxo) v = cyo ? a00 : 0.5 * (a00 + a01);
        const int k = L.x + j * L.nx + i;
        lds[k] = lds[k] + v;
      }
    __syncthreads();
  }
  for (int q = tid; q < L.nx * L.ny; q += kCoarseThreads) G.x[q] = lds[L.x + q];
}

// LDS bytes k_mg_coarse needs for levels l0..nl-1
size_t mg_coarse_lds(const MGLevel* L, int l0, int nl)
{
  size_t words = 1;
  for (int l = l0; l < nl; l++) words += (size_t)(L[l].nx + 1) + (size_t)(L[l].ny + 1) + 5 * (size_t)(L[l].nx * L[l].ny);
  return words * sizeof(double);
}

MGLevelD dev_level(const MGLevel& L) { return MGLevelD{L.nx, L.ny, L.fx, L.fy, L.x, L.b, L.r}; }

void sweep(MGHierarchy* H, int l, int color, hipStream_t s)
{
  const MGLevel& L = H->L[l];
  hipLaunchKernelGGL(k_mg_sweep, dim3(grid_of((L.nx + 1) / 2 * L.ny)), dim3(kBlock), 0, s, dev_level(L),
                     H->gamma, color, H->per);
}

// levels lc.. in one workgroup, from b to x of level lc
void coarse_cycle(MGHierarchy* H, const double* b, double* x, hipStream_t s)
{
  MGCoarse G{};
  G.nl = H->nl - H->lc;
  G.tables = H->ctab;
  G.b = b;
  G.x = x;
  int at = 1;
  for (int l = 0; l < G.nl; l++) {
    MGCoarseLevel& C = G.lev[l];
    C.nx = (int)H->L[H->lc + l].nx;
    C.ny = (int)H->L[H->lc + l].ny;
    C.fx = at;
    C.fy = C.fx + C.nx + 1;
    at = C.fy + C.ny + 1;
  }
  G.tab = at - 1;
  for (int l = 0; l < G.nl; l++) {
    MGCoarseLevel& C = G.lev[l];
    C.x = at;
    C.b = C.x + C.nx * C.ny;
    C.r = C.b + C.nx * C.ny;
    C.d = C.r + C.nx * C.ny;
    C.y = C.d + C.nx * C.ny;
    at = C.y + C.nx * C.ny;
  }
  hipLaunchKernelGGL(k_mg_coarse, dim3(1), dim3(kCoarseThreads), H->lc_lds, s, G, H->gamma, H->relax, H->nrelax, H->per);
}

void vcycle(MGHierarchy* H, int l, hipStream_t s)
{
  if (l >= H->lc) {  // the rest of the cycle in one workgroup
    coarse_cycle(H, H->L[l].b, H->L[l].x, s);
    return;
  }
  const MGLevel& L = H->L[l];
  hipLaunchKernelGGL(k_mg_fill0, dim3(grid_of(L.nx * L.ny)), dim3(kBlock), 0, s, L.nx * L.ny, L.x);
  // post-smoothing order: black then red (the adjoint of the pre-smoother,
  // relax type 2) or red then black again (relax type 3)
  const int p0 = (H->relax == 2) ? 1 : 0;
  if (l == H->nl - 1) {
    for (int k = 0; k < kCoarse; k++) {
      sweep(H, l, 0, s);
      sweep(H, l, 1, s);
    }
    for (int k = 0; k < kCoarse; k++) {
      sweep(H, l, p0, s);
      sweep(H, l, 1 - p0, s);
    }
    return;
  }
  for (int k = 0; k < H->nrelax; k++) {
    sweep(H, l, 0, s);
    sweep(H, l, 1, s);
  }
  const MGLevel& C = H->L[l + 1];
  hipLaunchKernelGGL(k_mg_resid, dim3(grid_of(L.nx * L.ny)), dim3(kBlock), 0, s, dev_level(L), H->gamma,
                     H->per);
  hipLaunchKernelGGL(k_mg_restrict, dim3(grid_of(C.nx * C.ny)), dim3(kBlock), 0, s, dev_level(L),
                     dev_level(C), H->per);
  vcycle(H, l + 1, s);
  hipLaunchKernelGGL(k_mg_prolong, dim3(grid_of(L.nx * L.ny)), dim3(kBlock), 0, s, dev_level(L),
                     dev_level(C), H->per);
  for (int k = 0; k < H->nrelax; k++) {
    sweep(H, l, p0, s);
    sweep(H, l, 1 - p0, s);
  }
}

// ------------------------------------------------ one level on register tiles
// A workgroup of nw wavefronts holds nw*R rows x 128 columns of a level: x, b,
// the diagonal d and its reciprocal in registers, two adjacent columns per
// lane, R rows per wavefront (the layout of the super-time-stepping tiles).
// Half of the cells change in a half-sweep: of a lane's two cells the one whose
// colour it is, known at compile time because tiles start at even rows and
// columns.  Neighbours in x come from the adjacent lanes, in y from the
// wavefront's own rows or, at its rim, through LDS (double-buffered, one
// barrier per half-sweep).  Each half-sweep, the residual and the restriction
// take one cell off the valid rim; wavefronts past it skip.
//
// Down: x = 0, nr sweep pairs, the residual and its restriction: 8 bytes per
// cell read (with the halo: 1.36 times that at nr = 2 and 64 rows), 8 + 2
// written.  Up: prolongation and nr sweep pairs, 16 + 2 read (1.23 times) and 8
// written.  Both are bound by these bytes on large levels and by the launch
// and their 5 to 7 barriers on small ones.
//
struct MGTile {
  int64_t nx, ny, cnx, cny;
  const double *fx, *fy, *b, *xin, *xc;  // up: x before the correction and the coarse x
  double *xout, *bc;                     // down: also the coarse b
  const double* gp;
  int strips, hl, own, y0, nr;
  int vec;  // 16-byte accesses: even rows, aligned vectors
};

__device__ inline double mg_west(double x)  // lane i receives lane i-1, the first zero
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ inline double mg_east(double x)  // lane i receives lane i+1, the last zero
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

constexpr int kMGTileWaves = 16;
constexpr int kMGTileRelax = 4;  // sweep pairs up to which a level runs on tiles

// C0: the first colour of a sweep pair
template <int R, bool PER, bool UP, int C0>
__global__ __launch_bounds__(kMGTileWaves* kWave) void k_mg_tile(const MGTile a)
{
  static_assert(R % 2 == 0, "a wavefront's rows start at an even row");
  __shared__ double2 rim[2][kMGTileWaves][2][kWave];
  typedef __attribute__((address_space(4))) const double ccdouble;
  const unsigned nb = gridDim.x, bi = blockIdx.x;
  const unsigned bq = nb >> 3, br = nb & 7u, xcd = bi & 7u, loc = bi >> 3;
  const unsigned tile = xcd * bq + (xcd < br ? xcd : br) + loc;  // XCD-aware order
  const int strip = (int)(tile % (unsigned)a.strips), rb = (int)(tile / (unsigned)a.strips);
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int nw = (int)(blockDim.x / kWave);
  const int nx = (int)a.nx, ny = (int)a.ny;
  const double g = *(ccdouble*)a.gp;
  const int c = strip * (kWave - 2 * a.hl) * 2 + 2 * (lane - a.hl);
  const int jown = rb * a.own, jend = min(jown + a.own, ny);
  const int j0 = jown + a.y0 + wave * R;
  int c0 = c;
  if (PER) {  // even sides: a lane's two columns wrap together
    while (c0 < 0) c0 += nx;
    while (c0 >= nx) c0 -= nx;
  }
  const bool in0 = PER || (c0 >= 0 && c0 < nx), in1 = PER || (c0 + 1 >= 0 && c0 + 1 < nx);
  const double f0 = in0 ? a.fx[c0] : 0.0, f1 = (in0 || in1) ? a.fx[c0 + 1] : 0.0, f2 = in1 ? a.fx[c0 + 2] : 0.0;
  ccdouble* fy = (ccdouble*)a.fy;
  int jr[R];
  double h0[R], h1[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    int j = j0 + r;
    if (PER) {
      while (j < 0) j += ny;
      while (j >= ny) j -= ny;
    }
    jr[r] = j;
    const bool ok = PER || (j >= 0 && j < ny);
    h0[r] = ok ? fy[j] : 0.0;
    h1[r] = ok ? fy[j + 1] : 0.0;
  }
  double x[R][2], b[R][2], d[R][2], y[R][2];
  auto ld = [&](const double* __restrict__ p, double (&v)[R][2]) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      v[r][0] = v[r][1] = 0.0;
      if (!PER && (jr[r] < 0 || jr[r] >= ny)) continue;
      const double* q = p + (int64_t)jr[r] * nx + c0;
      if (a.vec) {
        if (in0) {
          const double2 t = *reinterpret_cast<const double2*>(q);
          v[r][0] = t.x;
          v[r][1] = t.y;
        }
      } else {
        if (in0) v[r][0] = q[0];
        if (in1) v[r][1] = q[1];
      }
    }
  };
  ld(a.b, b);
  if (UP) ld(a.xin, x);
#pragma unroll
  for (int r = 0; r < R; r++) {
    if (!UP) x[r][0] = x[r][1] = 0.0;
    d[r][0] = 1.0 + g * ((f0 + f1) + (h0[r] + h1[r]));
    d[r][1] = 1.0 + g * ((f1 + f2) + (h0[r] + h1[r]));
    y[r][0] = 1.0 / d[r][0];
    y[r][1] = 1.0 / d[r][1];
  }
  if (UP) {
    // bilinear correction.  Coarse columns a lane needs: I - 1 and I
    // (Dirichlet: column c lies between them, column c + 1 on I) or I and
    // I + 1 (periodic: column c on I, column c + 1 between), I = c0 / 2
    const int cnx = (int)a.cnx, cny = (int)a.cny;
    const int I = c0 >> 1;
    auto XC = [&](int i, int j) -> double {
      if (PER) {
        i -= i >= cnx ? cnx : 0;
        j -= j >= cny ? cny : 0;
      }
      return (i >= 0 && i < cnx && j >= 0 && j < cny) ? a.xc[(int64_t)j * cnx + i] : 0.0;
    };
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (!PER && (jr[r] < 0 || jr[r] >= ny)) continue;
      // row parity r: the row starts are even
      const bool on = PER ? !(r & 1) : (r & 1);  // the row lies on a coarse row
      const int J = (PER || on) ? jr[r] / 2 : jr[r] / 2 - 1;
      double v0, v1;  // columns c and c + 1
      if (PER) {
        if (on) {
          const double p = XC(I, J);
          v0 = p;
          v1 = 0.5 * (p + XC(I + 1, J));
        } else {
          const double p = XC(I, J), q = XC(I, J + 1);
          v0 = 0.5 * (p + q);
          v1 = 0.25 * ((p + XC(I + 1, J)) + (q + XC(I + 1, J + 1)));
        }
      } else {
        if (on) {
          const double p = XC(I, J);
          v0 = 0.5 * (XC(I - 1, J) + p);
          v1 = p;
        } else {
          const double p = XC(I, J), q = XC(I, J + 1);
          v0 = 0.25 * ((XC(I - 1, J) + p) + (XC(I - 1, J + 1) + q));
          v1 = 0.5 * (p + q);
        }
      }
      if (in0) x[r][0] = x[r][0] + v0;
      if (in1) x[r][1] = x[r][1] + v1;
    }
  }

  auto publish = [&](int k, const double (&v)[R][2]) {
    rim[k][wave][0][lane] = make_double2(v[0][0], v[0][1]);
    rim[k][wave][1][lane] = make_double2(v[R - 1][0], v[R - 1][1]);
  };
  const double2 zero2 = make_double2(0.0, 0.0);
  auto south = [&](int k) { return wave > 0 ? rim[k][wave > 0 ? wave - 1 : 0][1][lane] : zero2; };
  auto north = [&](int k) { return wave < nw - 1 ? rim[k][wave + 1][0][lane] : zero2; };
  publish(0, x);
  // wavefronts of ghost rows only never compute: their rows are zero for good
  const bool ghosts = !PER && (j0 + R <= 0 || j0 >= ny);
  if (ghosts) publish(1, x);
  const int L = UP ? 2 * a.nr : 2 * a.nr + 2;  // rim cells the tile loses in all
  auto needed = [&](int m) {                   // after m operations
    const int lo = jown - (L - m), hi = jend + (L - m);
    return j0 + R > (PER ? lo : max(lo, 0)) && j0 < (PER ? hi : min(hi, ny));
  };
  // one half-sweep of colour CLR: rows of even parity their column c + CLR,
  // rows of odd parity the other one
  auto half = [&](auto clr, int m) {
    constexpr int CLR = decltype(clr)::value;
    __syncthreads();
    if (!needed(m + 1)) return;
    const double2 S2 = south(m & 1), N2 = north(m & 1);
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (!PER && (j0 + r < 0 || j0 + r >= ny)) continue;  // wavefront-uniform
      const int k = (r + CLR) & 1;
      const double W = k ? x[r][0] : mg_west(x[r][1]), E = k ? mg_east(x[r][0]) : x[r][1];
      const double S = r > 0 ? x[r > 0 ? r - 1 : 0][k] : (k ? S2.y : S2.x);
      const double N = r < R - 1 ? x[r < R - 1 ? r + 1 : 0][k] : (k ? N2.y : N2.x);
      const double off = (((k ? f1 : f0) * W + (k ? f2 : f1) * E) + h0[r] * S) + h1[r] * N;
      const double v = mg_quot(b[r][k] + g * off, d[r][k], y[r][k]);
      x[r][k] = (PER || (k ? in1 : in0)) ? v : 0.0;
    }
    publish((m + 1) & 1, x);
  };
  int m = 0;
  for (int k = 0; k < a.nr; k++) {
    half(std::integral_constant<int, C0>(), m++);
    half(std::integral_constant<int, 1 - C0>(), m++);
  }
  const bool ownl = lane >= a.hl && lane < kWave - a.hl;
  if (ownl) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int j = j0 + r;
      if (j < jown || j >= jend) continue;
      double* q = a.xout + (int64_t)j * nx + c;
      if (a.vec) {
        if (c < nx) *reinterpret_cast<double2*>(q) = make_double2(x[r][0], x[r][1]);
      } else {
        if (c < nx) q[0] = x[r][0];
        if (c + 1 < nx) q[1] = x[r][1];
      }
    }
  }
  if (UP) return;
  // residual (zero outside the domain), over b
  __syncthreads();
  if (needed(m + 1)) {
    const double2 S2 = south(m & 1), N2 = north(m & 1);
#pragma unroll
    for (int r = 0; r < R; r++) {
      if (!PER && (j0 + r < 0 || j0 + r >= ny)) continue;
      const double W = mg_west(x[r][1]), E = mg_east(x[r][0]);
      const double S0 = r > 0 ? x[r > 0 ? r - 1 : 0][0] : S2.x, S1 = r > 0 ? x[r > 0 ? r - 1 : 0][1] : S2.y;
      const double N0 = r < R - 1 ? x[r < R - 1 ? r + 1 : 0][0] : N2.x;
      const double N1 = r < R - 1 ? x[r < R - 1 ? r + 1 : 0][1] : N2.y;
      const double o0 = ((f0 * W + f1 * x[r][1]) + h0[r] * S0) + h1[r] * N0;
      const double o1 = ((f1 * x[r][0] + f2 * E) + h0[r] * S1) + h1[r] * N1;
      const double t0 = d[r][0] * x[r][0] - g * o0, t1 = d[r][1] * x[r][1] - g * o1;
      b[r][0] = (PER || in0) ? b[r][0] - t0 : 0.0;
      b[r][1] = (PER || in1) ? b[r][1] - t1 : 0.0;
    }
    publish((m + 1) & 1, b);
  }
  __syncthreads();
  m++;
  if (!needed(L)) return;
  // full weighting onto the coarse nodes of the tile's own cells: fine node
  // (2I+1, 2J+1), or (2I, 2J) on a periodic grid
  constexpr int K = PER ? 0 : 1;  // the coarse node's column and row parity
  const double2 S2 = south(m & 1), N2 = north(m & 1);
  auto rowv = [&](int r, double& w, double& ce, double& e) {  // west, centre, east of row r (-1 .. R)
    const double v0 = r < 0 ? S2.x : (r >= R ? N2.x : b[r < 0 ? 0 : (r >= R ? R - 1 : r)][0]);
    const double v1 = r < 0 ? S2.y : (r >= R ? N2.y : b[r < 0 ? 0 : (r >= R ? R - 1 : r)][1]);
    if (K) {
      w = v0;
      ce = v1;
      e = mg_east(v0);
    } else {
      w = mg_west(v1);
      ce = v0;
      e = v1;
    }
  };
#pragma unroll
  for (int r = K; r < R; r += 2) {
    const int j = j0 + r;
    double w0, c1, e0, w1, cc, e1, w2, c2, e2;
    rowv(r - 1, w0, c1, e0);
    rowv(r, w1, cc, e1);
    rowv(r + 1, w2, c2, e2);
    if (j < jown || j >= jend || !ownl || c + K >= nx) continue;
    double t = 4.0 * cc;
    t = t + 2.0 * ((w1 + e1) + (c1 + c2));
    t = t + ((w0 + e0) + (w2 + e2));
    a.bc[(int64_t)(j >> 1) * a.cnx + (c >> 1)] = t * 0.0625;
  }
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// one level's down (xc null) or up pass; rows per wavefront: 4, or 2 where
// tiles of 4 would leave most of the 256 CUs without one
void tile_level(MGHierarchy* H, int l, const double* b, const double* xin, const double* xc, double* xout,
                hipStream_t s)
{
  const MGLevel& L = H->L[l];
  const MGLevel& C = H->L[l + 1];
  const bool up = xc != nullptr;
  MGTile a{};
  a.nx = L.nx;
  a.ny = L.ny;
  a.cnx = C.nx;
  a.cny = C.ny;
  a.fx = L.fx;
  a.fy = L.fy;
  a.b = b;
  a.xin = xin;
  a.xc = xc;
  a.xout = xout;
  a.bc = C.b;
  a.gp = H->gamma;
  a.nr = H->nrelax;
  a.vec = L.nx % 2 == 0 && aligned16(b) && aligned16(xout) && (!up || aligned16(xin));
  const int halo = up ? 2 * a.nr : 2 * a.nr + 2;
  if (!H->per && L.nx <= 2 * kWave) {
    a.hl = 0;
    a.strips = 1;
  } else {
    a.hl = halo / 2;
    const int64_t ow = 2 * (kWave - 2 * a.hl);
    a.strips = (int)((L.nx + ow - 1) / ow);
  }
  auto blocks = [&](int R) {
    const int64_t rows = (int64_t)R * kMGTileWaves;
    if (!H->per && L.ny <= rows) {
      a.own = (int)L.ny;
      a.y0 = 0;
    } else {
      a.own = (int)(rows - 2 * halo);
      a.y0 = -halo;
    }
    return (int64_t)a.strips * ((L.ny + a.own - 1) / a.own);
  };
  int R = 4;
  int64_t n = blocks(R);
  if (n < 256 && 2 * kMGTileWaves > 3 * halo) n = blocks(R = 2);
  const bool black_first = up && H->relax == 2;
#define CEDA_MG_TILE(RR, PP, UU, CC)                                                                     \
  hipLaunchKernelGGL((k_mg_tile<RR, PP, UU, CC>), dim3((unsigned)n), dim3(kMGTileWaves * kWave), 0, s, a)
#define CEDA_MG_TILE_R(RR)                                                                               \
  if (H->per) {                                                                                          \
    if (!up) CEDA_MG_TILE(RR, true, false, 0);                                                           \
    else if (black_first) CEDA_MG_TILE(RR, true, true, 1);                                               \
    else CEDA_MG_TILE(RR, true, true, 0);                                                                \
  } else {                                                                                               \
    if (!up) CEDA_MG_TILE(RR, false, false, 0);                                                          \
    else if (black_first) CEDA_MG_TILE(RR, false, true, 1);                                              \
    else CEDA_MG_TILE(RR, false, true, 0);                                                               \
  }
  if (R == 4) { CEDA_MG_TILE_R(4) }
  else { CEDA_MG_TILE_R(2) }
#undef CEDA_MG_TILE_R
#undef CEDA_MG_TILE
}

// the hierarchy runs on tiles: every level above the single-workgroup cycle
bool on_tiles(const MGHierarchy* H, int nrelax)
{
  return H->lc < H->nl && nrelax <= kMGTileRelax && H->L[0].nx < (1 << 30) && H->L[0].ny < (1 << 30);
}
// where the correction of level l ends up (levels 1 .. lc)
double* corr(MGHierarchy* H, int l) { return l == H->lc ? H->L[l].x : H->L[l].r; }

// levels 1.. of a cycle on tiles, from L[1].b to corr(1)
void inner_cycle(MGHierarchy* H, hipStream_t s)
{
  for (int l = 1; l < H->lc; l++) tile_level(H, l, H->L[l].b, nullptr, nullptr, H->L[l].x, s);
  coarse_cycle(H, H->L[H->lc].b, H->L[H->lc].x, s);
  for (int l = H->lc - 1; l >= 1; l--) tile_level(H, l, H->L[l].b, H->L[l].x, corr(H, l + 1), H->L[l].r, s);
}

MGHierarchy* build(DiffusionProblem* P)
{
  MGHierarchy* H = new MGHierarchy();
  const bool per = (P->p.kind == DIFFUSION_CEDA_PERIODIC);
  H->per = per ? 1 : 0;
  std::vector<double> fx = P->fx, fy = P->fy, hfx[kMGMaxL], hfy[kMGMaxL];
  int64_t nx = P->p.nx, ny = P->p.ny;
  int l = 0;
  for (;;) {
    MGLevel& L = H->L[l];
    L.nx = nx;
    L.ny = ny;
    CEDA_HIP_CHECK(ceda::dev_malloc(&L.fx, sizeof(double) * (nx + 1)));
    CEDA_HIP_CHECK(ceda::dev_malloc(&L.fy, sizeof(double) * (ny + 1)));
    CEDA_HIP_CHECK(ceda::copy_sync(L.fx, fx.data(), sizeof(double) * (nx + 1), hipMemcpyHostToDevice));
    CEDA_HIP_CHECK(ceda::copy_sync(L.fy, fy.data(), sizeof(double) * (ny + 1), hipMemcpyHostToDevice));
    CEDA_HIP_CHECK(ceda::dev_malloc(&L.x, sizeof(double) * nx * ny));
    CEDA_HIP_CHECK(ceda::dev_malloc(&L.b, sizeof(double) * nx * ny));
    CEDA_HIP_CHECK(ceda::dev_malloc(&L.r, sizeof(double) * nx * ny));
    hfx[l] = fx;
    hfy[l] = fy;
    l++;
    const int64_t cx = nx / 2, cy = ny / 2;
    if (per ? (cx % 2 || cy % 2 || cx < 4 || cy < 4) : (cx < 3 || cy < 3)) break;
    if (l == kMGMaxL) break;
    std::vector<double> cfx(cx + 1), cfy(cy + 1);
    if (per) {
      for (int64_t i = 0; i <= cx; i++) cfx[i] = (fx[i > 0 ? 2 * i - 1 : nx - 1] + fx[2 * i]) / 8.0;
      for (int64_t j = 0; j <= cy; j++) cfy[j] = (fy[j > 0 ? 2 * j - 1 : ny - 1] + fy[2 * j]) / 8.0;
    } else {
      for (int64_t i = 0; i <= cx; i++)
        cfx[i] = (fx[2 * i < nx ? 2 * i : nx] + fx[2 * i + 1 < nx ? 2 * i + 1 : nx]) / 8.0;
      for (int64_t j = 0; j <= cy; j++)
        cfy[j] = (fy[2 * j < ny ? 2 * j : ny] + fy[2 * j + 1 < ny ? 2 * j + 1 : ny]) / 8.0;
    }
    fx.swap(cfx);
    fy.swap(cfy);
    nx = cx;
    ny = cy;
  }
  H->nl = l;
  // the coarse cycle takes the trailing levels whose arrays fit in one
  // workgroup's LDS (none when even the coarsest does not, e.g. a grid that
  // cannot be coarsened)
  int dev = 0;
  CEDA_HIP_CHECK(hipGetDevice(&dev));
  int lds_max = 0;
  CEDA_HIP_CHECK(hipDeviceGetAttribute(&lds_max, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  H->lc = l;
  const size_t lds_dyn_max = (size_t)lds_max;
  while (H->lc > 0 && l - H->lc < kCoarseMaxL && H->L[H->lc - 1].nx * H->L[H->lc - 1].ny <= kMGCoarseCells &&
         mg_coarse_lds(H->L, H->lc - 1, l) <= lds_dyn_max)
    H->lc--;
  H->lc_lds = (H->lc < l) ? mg_coarse_lds(H->L, H->lc, l) : 0;
  if (H->lc_lds > 65536 &&
      hipFuncSetAttribute((const void*)k_mg_coarse, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)H->lc_lds) != hipSuccess) {
    (void)hipGetLastError();
    while (H->lc < l && mg_coarse_lds(H->L, H->lc, l) > 65536) H->lc++;
    H->lc_lds = (H->lc < l) ? mg_coarse_lds(H->L, H->lc, l) : 0;
  }
  if (H->lc < l) {
    std::vector<double> t;
    for (int k = H->lc; k < l; k++) {
      t.insert(t.end(), hfx[k].begin(), hfx[k].end());
      t.insert(t.end(), hfy[k].begin(), hfy[k].end());
    }
    CEDA_HIP_CHECK(ceda::dev_malloc(&H->ctab, sizeof(double) * t.size()));
    CEDA_HIP_CHECK(ceda::copy_sync(H->ctab, t.data(), sizeof(double) * t.size(), hipMemcpyHostToDevice));
  }
  CEDA_HIP_CHECK(ceda::dev_malloc(&H->gamma, sizeof(double)));
  CEDA_HIP_CHECK(ceda::host_malloc(&H->h_gamma, sizeof(double), hipHostMallocDefault));
  return H;
}

}  // namespace

namespace ceda {
void mg_destroy(MGHierarchy* H)
{
  if (!H) return;
  for (int l = 0; l < H->nl; l++) {
    double* ps[] = {H->L[l].fx, H->L[l].fy, H->L[l].x, H->L[l].b, H->L[l].r};
    for (double* p : ps)
      if (p) CEDA_HIP_CHECK(ceda::dev_free(p));
  }
  if (H->gamma) CEDA_HIP_CHECK(ceda::dev_free(H->gamma));
  if (H->ctab) CEDA_HIP_CHECK(ceda::dev_free(H->ctab));
  if (H->h_gamma) CEDA_HIP_CHECK(ceda::host_free(H->h_gamma));
  if (H->graph) CEDA_HIP_CHECK(ceda::graph_exec_destroy(H->graph));
  delete H;
}
}  // namespace ceda

extern "C" {

int MGPSetup(sunrealtype, N_Vector, N_Vector, sunbooleantype, sunbooleantype* jcurPtr, sunrealtype gamma,
             void* user_data)
{
  DiffusionProblem* P = static_cast<DiffusionProblem*>(user_data);
  // periodic grids need even sides (red/black colours consistent across the wrap)
  if (!P || (P->p.kind == DIFFUSION_CEDA_PERIODIC && (P->p.nx % 2 || P->p.ny % 2))) return -1;
  hipStream_t s = P->exec->stream;
  if (!P->mg) P->mg = build(P);
  MGHierarchy* H = P->mg;
  CEDA_HIP_CHECK(hipStreamSynchronize(s));  // the previous gamma may still be read
  *H->h_gamma = gamma;
  CEDA_HIP_CHECK(hipMemcpyAsync(H->gamma, H->h_gamma, sizeof(double), hipMemcpyHostToDevice, s));
  if (H->graph && (H->relax != P->mg_relax || H->nrelax != P->mg_nrelax)) {
    CEDA_HIP_CHECK(ceda::graph_exec_destroy(H->graph));
    H->graph = nullptr;
  }
  if (!H->graph) {
    H->relax = P->mg_relax;
    H->nrelax = P->mg_nrelax;
    hipGraph_t g;
    // no device-wide synchronisation from other threads meanwhile
    std::lock_guard<std::recursive_mutex> lk(ceda::device_sync_mutex());
    CEDA_HIP_CHECK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    if (!on_tiles(H, H->nrelax)) vcycle(H, 0, s);
    else if (H->lc > 0) inner_cycle(H, s);
    else coarse_cycle(H, H->L[0].b, H->L[0].x, s);
    CEDA_HIP_CHECK(hipStreamEndCapture(s, &g));
    CEDA_HIP_CHECK(hipGraphInstantiate(&H->graph, g, nullptr, nullptr, 0));
    CEDA_HIP_CHECK(hipGraphDestroy(g));
  }
  CEDA_HIP_CHECK(hipStreamSynchronize(s));
  if (jcurPtr) *jcurPtr = SUNTRUE;
  return 0;
}

int MGPSolve(sunrealtype, N_Vector, N_Vector, N_Vector r, N_Vector z, sunrealtype, sunrealtype, int,
             void* user_data)
{
  DiffusionProblem* P = static_cast<DiffusionProblem*>(user_data);
  if (!P || !P->mg || !r || !z || N_VGetLength(r) != P->n || N_VGetLength(z) != P->n) return -1;
  MGHierarchy* H = P->mg;
  hipStream_t s = P->exec->stream;
  const size_t bytes = sizeof(double) * (size_t)P->n;
  double *dr = dptr(r), *dz = dptr(z);
  if (on_tiles(H, H->nrelax) && H->lc > 0) {
    const double* b = dr;
    if (dr == dz) {  // the tiles read b while others write x
      CEDA_HIP_CHECK(hipMemcpyAsync(H->L[0].b, dr, bytes, hipMemcpyDeviceToDevice, s));
      b = H->L[0].b;
    }
    tile_level(H, 0, b, nullptr, nullptr, H->L[0].x, s);
    CEDA_HIP_CHECK(hipGraphLaunch(H->graph, s));
    tile_level(H, 0, b, H->L[0].x, corr(H, 1), dz, s);
  } else {
    CEDA_HIP_CHECK(hipMemcpyAsync(H->L[0].b, dr, bytes, hipMemcpyDeviceToDevice, s));
    CEDA_HIP_CHECK(hipGraphLaunch(H->graph, s));
    CEDA_HIP_CHECK(hipMemcpyAsync(dz, H->L[0].x, bytes, hipMemcpyDeviceToDevice, s));
  }
  H->cycles++;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int DiffusionProblem_MGLevels(const DiffusionProblem* P) { return (P && P->mg) ? P->mg->nl : 0; }

int DiffusionProblem_SetMGOptions(DiffusionProblem* P, int relax, int nrelax)
{
  if (!P || (relax != 2 && relax != 3) || nrelax < 0 || nrelax > 16) return -1;
  P->mg_relax = relax;
  P->mg_nrelax = nrelax;
  return 0;
}

long DiffusionProblem_MGNumCycles(const DiffusionProblem* P) { return (P && P->mg) ? P->mg->cycles : 0; }

}  // extern "C"
