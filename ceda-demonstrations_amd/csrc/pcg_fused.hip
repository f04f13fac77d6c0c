// Fused preconditioned CG for the implicit path: (I - gamma J) x = b with J
// the 5-point stencil of the RHS (the analytic Jacobian-vector product,
// exactly laplacian()'s arithmetic, diffusion.cpp:48-53) and the Jacobi or
// multigrid preconditioner.  The algorithm is the integrator's PCG
// (SUNLinSol_PCG, main.cpp:305; Hestenes-Stiefel with z = M r).
//
// An iteration l is two kernels:
//   k_pcg_dir:    the residual test of iteration l-1 and
//                 beta = r.z(l-1) / r.z(l-2); the direction
//                 p_l = z + beta p_{l-1}, formed at the five stencil points
//                 and stored into the other of two direction buffers; and
//                 the partial sums of p_l.Ap with Ap = p_l - gamma * J p_l
//   k_pcg_update: alpha = r.z / p.Ap; x += alpha p, r -= alpha Ap with Ap
//                 formed again from p_l, and the partial sums of |r|^2, r.z
// Ap is never stored: the update kernel reads p_l anyway, and its neighbours
// come from L2.  Nor is z where it is cheap to form: without preconditioner
// z = r, and with the Jacobi diagonal of constant coefficients z = r times
// one number.  So an iteration streams 24 + 40 = 64 bytes per cell (88 with z
// and Ap stored, 176 for the separate vector operations).  With variable
// coefficients z = r / diag is stored by the update (the eight divisions per
// pair of cells of forming it at the stencil's points cost more), and a
// preconditioner given as a callback (multigrid, the learned network) has its
// z = M r enqueued on the same stream after the update, and k_pcg_dot sums
// r.z for the next iteration's test and beta.
//
// The scalars never go to the host: every workgroup first sums the previous
// kernel's per-workgroup partials itself, in one fixed order (every workgroup
// gets bitwise the same alpha or beta), while its first cells' operands are
// already being loaded; the residual test is recorded in the device's solve
// state (running, converged at iteration l, non-finite), which every later
// kernel reads first, returning at once when the solve has ended.  The host
// enqueues
// iterations in batches, of the previous solve's length at first, and reads
// the status once per batch (after a one-workgroup kernel has tested the
// batch's last iteration and written the state to host memory): the iteration
// count, x and the statistics are those of a test after every iteration, and a
// NaN or infinity stops the solve with an error instead of running to the cap.
// The arithmetic of every value is the one of the separate vector operations;
// only the reductions' summation order differs from them (deterministic, not
// bitwise equal), which is why this path is an option of the integrator
// (ARKodeSetDiffusionFastPCG) and the N_Vector PCG stays the reference.
//
// Kernel time per iteration with Jacobi: 2048^2 48.3 us, 5.6 TB/s (63.7 us with
// z and Ap stored); 500 x 480 10.7 us (15.7 us with 938 workgroups, each
// summing as many partials by LDS shuffles before its first load), which is
// two kernels' start, partial sums and tail.
#include <algorithm>
#include <cmath>

#include "arkode_internal.hpp"
#include "diffusion_internal.hpp"
#include "stencil_ops.hpp"

using namespace ceda;

namespace ceda_ark {

namespace {

constexpr int kPcgBlocks = 1024;   // workgroups of the reduction kernels
constexpr int kPcgBatchMax = 32;   // iterations enqueued between host checks
constexpr int kPcgBulkMax = 128;   // the same within the predicted count
constexpr int kPcgTail = 8;        // iterations between host checks past the predicted count
constexpr int kPcgChunk = 4;       // callback preconditioner: iterations between host waits in the bulk
// workspace layout (doubles): partials of p.Ap, of (|r|^2, r.z), of r.z
// (callback preconditioner), then the solve state
constexpr int kOffA = 0, kOffB = kPcgBlocks, kOffC = 3 * kPcgBlocks, kOffState = 4 * kPcgBlocks;
constexpr int kStateDoubles = 8;
constexpr int kWsDoubles = kOffState + kStateDoubles;

// solve state in device memory (doubles): r.z of the current iteration in
// slot l & 1, the status, the iteration it was set at, the last |r|^2 and
// delta.  The status stands in two words, so that no kernel stores one that
// its other wavefronts read: k_pcg_dir returns by kStatus and records its test
// in kTested, k_pcg_update returns by kTested and hands it on to kStatus.
enum { kRz0 = 0, kRz1 = 1, kStatus = 2, kIter = 3, kRr = 4, kDelta = 5, kTested = 6 };
enum { kRunning = 0, kConverged = 1, kNonFinite = 2 };

// x of the lanes `CTRL` (DPP) rows or lanes below; zero where there is none
template <int CTRL, int ROWS>
__device__ inline double dpp_or_zero(double x)
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, ROWS, 0xf, false);
  return __hiloint2double(hi, lo);
}
// the wavefront's sum, in every lane (row scans of 16 lanes, then the rows)
__device__ inline double wave_sum(double v)
{
  v += dpp_or_zero<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
  v += dpp_or_zero<0x112, 0xf>(v);
  v += dpp_or_zero<0x114, 0xf>(v);
  v += dpp_or_zero<0x118, 0xf>(v);
  v += dpp_or_zero<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v += dpp_or_zero<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), kWave - 1),
                          __builtin_amdgcn_readlane(__double2loint(v), kWave - 1));
}

// workgroup sum of NACC accumulators into partials[blockIdx.x * NACC + a]
template <int NACC>
__device__ inline void block_sums(double (&acc)[NACC], double* __restrict__ partials)
{
  __shared__ double s[kBlock / kWave][NACC];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
  for (int a = 0; a < NACC; a++) {
    const double v = wave_sum(acc[a]);
    if (lane == 0) s[wave][a] = v;
  }
  __syncthreads();
  if (threadIdx.x < NACC) {
    double v = s[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < kBlock / kWave; w++) v += s[w][threadIdx.x];
    partials[(int64_t)blockIdx.x * NACC + threadIdx.x] = v;
  }
}

// the sums of NACC accumulators over nblocks per-workgroup partials, returned
// to every thread of the workgroup: thread t adds partials t, t + 256, ... in
// order, then the wavefront sum, then the four wavefront sums in order (every
// workgroup gets bitwise the same values).  TAG: calls of one kernel have
// LDS words of their own.
template <int NACC, int TAG>
__device__ inline void sum_partials(const double* __restrict__ partials, int nblocks, double (&out)[NACC])
{
  __shared__ double s[kBlock / kWave][NACC];
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  double v[NACC] = {};
  for (int b = threadIdx.x; b < nblocks; b += kBlock)
#pragma unroll
    for (int a = 0; a < NACC; a++) v[a] += partials[(int64_t)b * NACC + a];
#pragma unroll
  for (int a = 0; a < NACC; a++) {
    const double t = wave_sum(v[a]);
    if (lane == 0) s[wave][a] = t;
  }
  __syncthreads();
#pragma unroll
  for (int a = 0; a < NACC; a++) {
    out[a] = s[0][a];
#pragma unroll
    for (int w = 1; w < kBlock / kWave; w++) out[a] += s[w][a];
  }
}

__device__ inline bool solve_ended(const double* __restrict__ st, int word = kStatus) { return st[word] != kRunning; }

// Jacobi inverse diagonal from the face coefficients: dinv = 1 / (1 - gp d),
// d = -((ax[i] + ax[i+1]) + (ay[j] + ay[j+1])), exactly k_psetup's value for
// the gamma gp of the last preconditioner setup
struct JacobiDiag {
  const double *ax, *ay;
  double gp;
};
__device__ inline double jac_dinv(const JacobiDiag& J, double sxi, double syj)
{
  const double d = -(sxi + syj);
  return 1.0 / (1.0 - J.gp * d);
}

// the residual test of iteration l-1 from k_pcg_update's partials (|r|^2,
// r.z): converged, non-finite (|r| or beta), else running with
// beta = r.z(l-1) / r.z(l-2).  Workgroup 0 records the outcome, an end in
// `word`; the caller returns when the solve has ended.
// r.z comes from parts_b's second accumulator, or, when parts_z is given
// (a preconditioner callback computed z after the update), from k_pcg_dot's
// partials parts_z.
__device__ inline bool test_iteration(int nparts, const double* __restrict__ parts_b,
                                      const double* __restrict__ parts_z, double* __restrict__ st, int word,
                                      int l, double* beta)
{
  const double rzold = st[(l - 1) & 1], delta = st[kDelta];
  double b2[2], z1[1];
  sum_partials<2, 0>(parts_b, nparts, b2);
  const double rr = b2[0];
  double rznew = b2[1];
  if (parts_z) {
    sum_partials<1, 1>(parts_z, nparts, z1);
    rznew = z1[0];
  }
  const double rnorm = sqrt(rr);
  *beta = rznew / rzold;
  int status = kRunning;
  if (!isfinite(rnorm)) status = kNonFinite;
  else if (rnorm <= delta) status = kConverged;
  else if (!isfinite(*beta)) status = kNonFinite;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st[kRr] = rr;
    st[kIter] = l - 1;
    if (status == kRunning) st[l & 1] = rznew;  // the r.z iteration l uses
    else st[word] = status;
  }
  return status != kRunning;
}

// The cells in units of W of a row: W = 2 pairs (k, k + 1), k even, with
// 16-byte accesses where the rows are even (a pair never straddles a row),
// W = 1 single cells.  XCD-aware grid-stride walk over the units: workgroup b
// runs on XCD b % 8 and, when the grid is a multiple of 8, walks the
// (b % 8)-th of 8 contiguous ranges, so that the rows above and below a unit
// are read by the same XCD at about the same time and come from its L2.  One
// division per thread.
struct PcgGrid {
  int64_t nx, ny;
  const double *fx, *fy;
  int64_t dj;  // rows and units a step advances
  int64_t di;
};
template <int W>
struct UnitWalk {
  int64_t q, end, step, i, j, hn, di, dj;
  __device__ UnitWalk(const PcgGrid& g)
  {
    const int64_t nu = g.nx * g.ny / W;
    const unsigned G = gridDim.x, b = blockIdx.x;
    const int parts = (G % 8 == 0) ? 8 : 1;
    const int64_t per = (nu + parts - 1) / parts;  // (by a constant 1 or 8)
    const int part = (int)(b % parts);
    hn = g.nx / W;
    q = part * per + (int64_t)(b / parts) * kBlock + threadIdx.x;
    end = min(nu, (part + 1) * per);
    step = (int64_t)(G / parts) * kBlock;
    di = g.di;
    dj = g.dj;
    j = nu < ((int64_t)1 << 31) ? (int64_t)((unsigned)q / (unsigned)hn) : q / hn;
    i = q - j * hn;
  }
  __device__ bool valid() const { return q < end; }
  __device__ void next()
  {
    q += step;
    i += di;
    j += dj;
    if (i >= hn) {
      i -= hn;
      j++;
    }
  }
};
// (host) the grid's step in rows and units
template <int W>
PcgGrid pcg_grid(const DiffusionProblem* P, unsigned blocks)
{
  PcgGrid g;
  g.nx = P->p.nx;
  g.ny = P->p.ny;
  g.fx = P->d_fx;
  g.fy = P->d_fy;
  const int64_t step = (int64_t)(blocks / (blocks % 8 == 0 ? 8 : 1)) * kBlock, hn = g.nx / W;
  g.dj = step / hn;
  g.di = step - g.dj * hn;
  return g;
}

template <int W>
__device__ inline void ldw(const double* __restrict__ a, int64_t k, double (&v)[W])
{
  if (W == 2) {
    const double2 t = *reinterpret_cast<const double2*>(a + k);
    v[0] = t.x;
    v[W - 1] = t.y;
  } else v[0] = a[k];
}
template <int W>
__device__ inline void stw(double* __restrict__ a, int64_t k, const double (&v)[W])
{
  if (W == 2) *reinterpret_cast<double2*>(a + k) = make_double2(v[0], v[W - 1]);
  else a[k] = v[0];
}
// a vector at a unit and its neighbours (zero outside a Dirichlet domain)
template <int W>
struct Five {
  double c[W], s[W], n[W], w, e;
};
template <bool PER, int W>
__device__ inline void ld_five(const PcgGrid& g, const UnitWalk<W>& u, const double* __restrict__ a, Five<W>& v)
{
  const int64_t nx = g.nx, ny = g.ny, i = u.i * W, k = u.q * W;
  ldw<W>(a, k, v.c);
  v.w = v.e = 0.0;
#pragma unroll
  for (int t = 0; t < W; t++) v.s[t] = v.n[t] = 0.0;
  if (PER || i > 0) v.w = a[i > 0 ? k - 1 : k + nx - 1];
  if (PER || i + W < nx) v.e = a[i + W < nx ? k + W : k + W - nx];
  if (PER || u.j > 0) ldw<W>(a, u.j > 0 ? k - nx : k + (ny - 1) * nx, v.s);
  if (PER || u.j < ny - 1) ldw<W>(a, u.j < ny - 1 ? k + nx : k - (ny - 1) * nx, v.n);
}
// Ap at the unit: p + (-gamma) J p, N_VLinearSum(1, p, -gamma, Jp) order
template <int W>
__device__ inline void ap_of(const PcgGrid& g, const UnitWalk<W>& u, double gamma, const Five<W>& p, double (&ap)[W])
{
  const int64_t i = u.i * W;
  const double h0 = g.fy[u.j], h1 = g.fy[u.j + 1];
  double f[W + 1];
#pragma unroll
  for (int t = 0; t <= W; t++) f[t] = g.fx[i + t];
#pragma unroll
  for (int t = 0; t < W; t++) {
    const double west = t > 0 ? p.c[t > 0 ? t - 1 : 0] : p.w, east = t < W - 1 ? p.c[t < W - 1 ? t + 1 : 0] : p.e;
    ap[t] = p.c[t] + (-gamma) * cell(f[t], f[t + 1], h0, h1, p.c[t], west, east, p.s[t], p.n[t]);
  }
}

// where z comes from: stored, r times the constant Jacobi inverse diagonal, r
enum { kZStored = 0, kZConst = 1, kZNone = 2 };

template <bool PER, int ZS, int W>
__global__ __launch_bounds__(kBlock) void k_pcg_dir(const PcgGrid g, double gamma, const double* __restrict__ zr,
                                                    JacobiDiag J, const double* __restrict__ pold,
                                                    double* __restrict__ pnew, int nparts,
                                                    const double* __restrict__ parts_b,
                                                    const double* __restrict__ parts_z,
                                                    double* __restrict__ parts_a, double* __restrict__ st, int l)
{
  if (solve_ended(st)) return;
  const bool first = (l == 1);  // the first direction is z itself, already in pold
  UnitWalk<W> u(g);
  Five<W> z = {}, p = {};
  if (u.valid()) {  // in flight during the partial sums
    if (!first) ld_five<PER, W>(g, u, zr, z);
    ld_five<PER, W>(g, u, pold, p);
  }
  const double dz = (ZS == kZConst) ? jac_dinv(J, J.ax[0] + J.ax[1], J.ay[0] + J.ay[1]) : 1.0;
  double beta = 0.0;
  if (!first && test_iteration(nparts, parts_b, parts_z, st, kTested, l, &beta)) return;
  auto dir = [&](double zv, double pv) { return ((ZS == kZConst) ? dz * zv : zv) + beta * pv; };
  double acc[1] = {0.0};
  while (u.valid()) {
    if (!first) {
#pragma unroll
      for (int t = 0; t < W; t++) {
        p.c[t] = dir(z.c[t], p.c[t]);
        p.s[t] = dir(z.s[t], p.s[t]);
        p.n[t] = dir(z.n[t], p.n[t]);
      }
      p.w = dir(z.w, p.w);
      p.e = dir(z.e, p.e);
      stw<W>(pnew, u.q * W, p.c);
    }
    double ap[W];
    ap_of<W>(g, u, gamma, p, ap);
#pragma unroll
    for (int t = 0; t < W; t++) acc[0] += p.c[t] * ap[t];
    u.next();
    if (u.valid()) {
      if (!first) ld_five<PER, W>(g, u, zr, z);
      ld_five<PER, W>(g, u, pold, p);
    }
  }
  block_sums<1>(acc, parts_a);
}

// what the update does about z = M r: nothing (a callback does), r.z with the
// constant Jacobi inverse diagonal or with z = r (not stored), the Jacobi
// inverse diagonal from the face coefficients or from an array (stored)
enum { kUpCallback = 0, kUpConst = 1, kUpNone = 2, kUpJacobi = 3, kUpArray = 4 };

// x += alpha p, r -= alpha Ap.  w: the residual norm is the weighted one, sum
// (r w)^2, else sum r^2.
template <bool PER, int UP, int W>
__global__ __launch_bounds__(kBlock) void k_pcg_update(const PcgGrid g, double gamma, int nparts,
                                                       const double* __restrict__ parts_a,
                                                       double* __restrict__ st, int l,
                                                       const double* __restrict__ p, double* __restrict__ x,
                                                       double* __restrict__ r, double* __restrict__ z,
                                                       const double* __restrict__ dinv, JacobiDiag J,
                                                       const double* __restrict__ w, double* __restrict__ partials)
{
  if (solve_ended(st, kTested)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) st[kStatus] = st[kTested];
    return;
  }
  UnitWalk<W> u(g);
  Five<W> pv = {};
  double xv[W] = {}, rv[W] = {};
  if (u.valid()) {  // in flight during the partial sums
    ld_five<PER, W>(g, u, p, pv);
    ldw<W>(x, u.q * W, xv);
    ldw<W>(r, u.q * W, rv);
  }
  const double dz = (UP == kUpConst) ? jac_dinv(J, J.ax[0] + J.ax[1], J.ay[0] + J.ay[1]) : 1.0;
  const double rz = st[l & 1];
  double pap[1];
  sum_partials<1, 0>(parts_a, nparts, pap);
  const double alpha = rz / pap[0];
  double acc[2] = {0.0, 0.0};
  while (u.valid()) {
    const int64_t k = u.q * W, i = u.i * W;
    double ap[W], zv[W];
    ap_of<W>(g, u, gamma, pv, ap);
#pragma unroll
    for (int t = 0; t < W; t++) {
      xv[t] = xv[t] + alpha * pv.c[t];
      rv[t] = rv[t] + (-alpha) * ap[t];
    }
    stw<W>(x, k, xv);
    stw<W>(r, k, rv);
    double wv[W], dv[W];
    if (w) ldw<W>(w, k, wv);
    if (UP == kUpArray) ldw<W>(dinv, k, dv);
    const double syj = (UP == kUpJacobi) ? J.ay[u.j] + J.ay[u.j + 1] : 0.0;
#pragma unroll
    for (int t = 0; t < W; t++) {
      const double rw = w ? rv[t] * wv[t] : rv[t];
      acc[0] += rw * rw;
      if (UP == kUpCallback) continue;
      zv[t] = rv[t];
      if (UP == kUpConst) zv[t] = dz * rv[t];
      if (UP == kUpJacobi) zv[t] = jac_dinv(J, J.ax[i + t] + J.ax[i + t + 1], syj) * rv[t];
      if (UP == kUpArray) zv[t] = dv[t] * rv[t];
      acc[1] += rv[t] * zv[t];
    }
    if (UP == kUpJacobi || UP == kUpArray) stw<W>(z, k, zv);
    u.next();
    if (u.valid()) {
      ld_five<PER, W>(g, u, p, pv);
      ldw<W>(x, u.q * W, xv);
      ldw<W>(r, u.q * W, rv);
    }
  }
  block_sums<2>(acc, partials);
}

// the state for the host, written to its (pinned) memory
__device__ inline void state_to_host(const double* __restrict__ st, double* __restrict__ host)
{
  __syncthreads();  // the test's own stores
  if (threadIdx.x < kStateDoubles) host[threadIdx.x] = st[threadIdx.x];
}

// the residual test of the last iteration of a batch, so that the host sees it
__global__ __launch_bounds__(kBlock) void k_pcg_check(int nparts, const double* __restrict__ parts_b,
                                                      const double* __restrict__ parts_z, double* st, int l,
                                                      double* host)
{
  if (!solve_ended(st)) {
    double beta;
    test_iteration(nparts, parts_b, parts_z, st, kStatus, l, &beta);
  }
  state_to_host(st, host);
}

// the residual test alone of iteration l (callback preconditioner: before
// z = M r is computed for it): converged or non-finite, recorded as
// test_iteration does; otherwise the state is left for the next iteration's
// full test (beta needs r.z)
__global__ __launch_bounds__(kBlock) void k_pcg_rtest(int nparts, const double* __restrict__ parts_b, double* st, int l,
                                                      double* host)
{
  if (!solve_ended(st)) {
    double b2[2];
    sum_partials<2, 0>(parts_b, nparts, b2);
    const double rnorm = sqrt(b2[0]);
    int status = kRunning;
    if (!isfinite(rnorm)) status = kNonFinite;
    else if (rnorm <= st[kDelta]) status = kConverged;
    if (threadIdx.x == 0 && status != kRunning) {
      st[kRr] = b2[0];
      st[kIter] = l;
      st[kStatus] = status;
    }
  }
  state_to_host(st, host);
}

template <int W>
__global__ __launch_bounds__(kBlock) void k_pcg_dot(int64_t n, const double* __restrict__ a,
                                                    const double* __restrict__ b, double* __restrict__ partials,
                                                    const double* __restrict__ st)
{
  if (st && solve_ended(st)) return;
  double acc[1] = {0.0};
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < n / W; k += (int64_t)gridDim.x * kBlock) {
    double u[W], v[W];
    ldw<W>(a, k * W, u);
    ldw<W>(b, k * W, v);
#pragma unroll
    for (int t = 0; t < W; t++) acc[0] += u[t] * v[t];
  }
  block_sums<1>(acc, partials);
}

__global__ void k_pcg_init(double* __restrict__ st, double rz, double delta)
{
  if (threadIdx.x == 0) {
    st[kRz0] = 0.0;
    st[kRz1] = rz;  // iteration 1 reads slot 1
    st[kStatus] = st[kTested] = kRunning;
    st[kIter] = 0;
    st[kRr] = 0.0;
    st[kDelta] = delta;
  }
}

// two units per thread at least: each workgroup of the next kernel sums all
// partials, and below 1,024 of them a kernel is as long as its start
unsigned blocks_for(int64_t units)
{
  int64_t g = (units + 2 * kBlock - 1) / (2 * kBlock);
  if (g >= 8) g = (g + 7) / 8 * 8;  // (the XCD ranges of UnitWalk)
  if (g > kPcgBlocks) g = kPcgBlocks;
  return (unsigned)(g < 1 ? 1 : g);
}

// the fused solver's workspace (partials and state), allocated on the
// solver's first fused solve and kept with it
void ensure_ws(SUNLinearSolver S)
{
  if (S->d_ws) return;
  CEDA_HIP_CHECK(dev_malloc(&S->d_ws, sizeof(double) * kWsDoubles));
  CEDA_HIP_CHECK(host_malloc(&S->h_ws, sizeof(double) * kStateDoubles, hipHostMallocDefault));
  CEDA_HIP_CHECK(dev_malloc(&S->d_p2, sizeof(double) * vlen(S->r)));
}

}  // namespace

namespace {

struct PcgArgs {
  hipStream_t s;
  unsigned g;
  double gamma;
  const double* zsrc;  // what k_pcg_dir forms z from
  double *z, *x, *r, *pa, *pb, *st;
  const double *pc, *dinv, *w;
  JacobiDiag J;
};

// one iteration's two kernels: p_l into pnew (from pold), x and r
template <bool PER, int W>
void launch_iteration(const DiffusionProblem* P, const PcgArgs& a, int zs, int up, const double* pold, double* pnew, int it)
{
  const PcgGrid g = pcg_grid<W>(P, a.g);
#define CEDA_DIR(Z)                                                                                              \
  hipLaunchKernelGGL((k_pcg_dir<PER, Z, W>), dim3(a.g), dim3(kBlock), 0, a.s, g, a.gamma, a.zsrc, a.J, pold, pnew, \
                     (int)a.g, a.pb, a.pc, a.pa, a.st, it)
#define CEDA_UP(U)                                                                                               \
  hipLaunchKernelGGL((k_pcg_update<PER, U, W>), dim3(a.g), dim3(kBlock), 0, a.s, g, a.gamma, (int)a.g, a.pa, a.st, it, \
                     pnew, a.x, a.r, a.z, a.dinv, a.J, a.w, a.pb)
  if (zs == kZConst) CEDA_DIR(kZConst);
  else if (zs == kZNone) CEDA_DIR(kZNone);
  else CEDA_DIR(kZStored);
  switch (up) {
    case kUpCallback: CEDA_UP(kUpCallback); break;
    case kUpConst: CEDA_UP(kUpConst); break;
    case kUpNone: CEDA_UP(kUpNone); break;
    case kUpJacobi: CEDA_UP(kUpJacobi); break;
    default: CEDA_UP(kUpArray); break;
  }
#undef CEDA_DIR
#undef CEDA_UP
}

}  // namespace

int pcg_fused(ArkMem* A, SUNLinearSolver S, DiffusionProblem* P, int pmode, ARKLsPrecSolveFn ps, void* ud,
              double t, double gamma, N_Vector b, N_Vector x)
{
  // the solver's vectors' stream (the problem is the integrator's user data
  // and lives on the same context)
  hipStream_t s = vstream(S->r);
  const int64_t n = P->n;
  if (vlen(x) != n || vlen(b) != n || vlen(S->r) != n) {
    fprintf(stderr, "[ARKLS ERROR] fused PCG: vector length %lld does not match the problem's %lld cells\n",
            (long long)vlen(x), (long long)n);
    return -1;
  }
  const bool per = P->p.kind == DIFFUSION_CEDA_PERIODIC;
  // pairs of cells: an even row length (every pair in one row, every pair's
  // first cell 16-byte aligned)
  const bool pairs = (P->p.nx % 2 == 0);
  const unsigned g = blocks_for(pairs ? n / 2 : n);
  ensure_ws(S);
  PcgArgs a{};
  a.s = s;
  a.g = g;
  a.gamma = gamma;
  a.pa = S->d_ws + kOffA;
  a.pb = S->d_ws + kOffB;
  double* pc = S->d_ws + kOffC;
  a.pc = pmode == 2 ? pc : nullptr;
  a.st = S->d_ws + kOffState;
  a.x = dptr(x);
  a.r = dptr(S->r);
  a.z = dptr(S->z);
  const bool wl2 = !(A->ls_reltol > 0.0);
  a.w = wl2 ? dptr(A->ewt) : nullptr;
  // the Jacobi inverse diagonal formed in the kernels from the gamma of its
  // last setup (which is what P->diag holds), or P->diag itself
  const bool jac = (pmode == 1 && P->diag_gamma_set);
  a.J = JacobiDiag{per ? P->d_px : P->d_fx, per ? P->d_py : P->d_fy, P->diag_gamma};
  a.dinv = (pmode == 1) ? dptr(P->diag) : nullptr;
  int zs = kZStored, up = kUpCallback;
  if (pmode == 0) zs = kZNone, up = kUpNone;
  else if (jac && P->constant_faces) zs = kZConst, up = kUpConst;
  else if (pmode == 1) up = jac ? kUpJacobi : kUpArray;
  a.zsrc = zs == kZStored ? a.z : a.r;

  N_VConst(0.0, x);
  N_VScale(1.0, b, S->r);
  const double bnorm = wl2 ? N_VWL2Norm(S->r, A->ewt) : sqrt(N_VDotProd(S->r, S->r));
  const double eplifac = (A->epslin > 0.0) ? A->epslin : 0.05;
  const double delta = (A->ls_reltol > 0.0) ? A->ls_reltol * bnorm
                                            : eplifac * A->nlscoef * sqrt((double)A->n);
  if (krylov_nonfinite("fused PCG", "|b|", bnorm)) return -1;
  if (bnorm <= delta) return 0;
  // z = M r
  if (pmode == 2) {
    A->npsolve++;
    if (ps(t, A->zcur, A->fz, S->r, S->z, gamma, delta, 1, ud)) return -1;
  } else if (pmode == 1) {
    A->npsolve++;
    N_VProd(P->diag, S->r, S->z);
  } else N_VScale(1.0, S->r, S->z);
  N_VScale(1.0, S->z, S->p);
  const double rz = N_VDotProd(S->r, S->z);
  if (krylov_nonfinite("fused PCG", "r.z", rz)) return -1;

  // Scalars on the device; the host reads the state once per batch.  The
  // direction of iteration l lives in q[l & 1] (q[1] = S->p holds p_1 = z,
  // which iteration 1 only reads).
  double* q[2] = {S->d_p2, dptr(S->p)};
  hipLaunchKernelGGL(k_pcg_init, dim3(1), dim3(64), 0, s, a.st, rz, delta);
  auto iteration = [&](int it) {
    const double* pold = it == 1 ? q[1] : q[(it - 1) & 1];
    if (pairs) {
      if (per) launch_iteration<true, 2>(P, a, zs, up, pold, q[it & 1], it);
      else launch_iteration<false, 2>(P, a, zs, up, pold, q[it & 1], it);
    } else {
      if (per) launch_iteration<true, 1>(P, a, zs, up, pold, q[it & 1], it);
      else launch_iteration<false, 1>(P, a, zs, up, pold, q[it & 1], it);
    }
  };
  // the solve's end as the state in S->h_ws says it; zlast: z of the
  // converged iterate was counted
  auto ended = [&]() -> int {
    const long iters = (long)S->h_ws[kIter];
    A->nli += iters;
    A->njtimes += iters;
    if (pmode) A->npsolve += iters - 1;  // z of the converged iterate is not computed or used
    S->last_iters = iters;
    if ((int)S->h_ws[kStatus] == kNonFinite) {
      fprintf(stderr, "[ARKLS ERROR] fused PCG: non-finite residual or direction at iteration %ld "
                      "(|r|^2 = %g); linear solve failed\n", iters, S->h_ws[kRr]);
      return -1;
    }
    return 0;
  };
  if (pmode == 2) {
    // Every kernel returns at once after convergence, but the callback's own
    // work would still be spent, so the host enqueues a fraction
    // (A->pcg_bulk, 3/4 by default) of the previous solve's iteration count
    // without waiting and then tests each residual (k_pcg_rtest, one wait)
    // before it calls the preconditioner.
    const long bulk = (S->last_iters > 4) ? (long)(A->pcg_bulk * (double)S->last_iters) : 0;
    for (int it = 1; it <= S->maxl; it++) {
      iteration(it);
      // after the bulk, and every kPcgChunk iterations within it, the host
      // waits for the residual test (chunks keep streams that share a
      // hardware queue interleaved)
      if (it > bulk || it % kPcgChunk == 0) {
        hipLaunchKernelGGL(k_pcg_rtest, dim3(1), dim3(kBlock), 0, s, (int)g, a.pb, a.st, it, S->h_ws);
        CEDA_HIP_CHECK(hipStreamSynchronize(s));
        if ((int)S->h_ws[kStatus] != kRunning) return ended();
      }
      if (ps(t, A->zcur, A->fz, S->r, S->z, gamma, delta, 1, ud)) {
        fprintf(stderr, "[ARKLS ERROR] fused PCG: the preconditioner solve failed at iteration %d\n", it);
        return -1;
      }
      if (pairs) hipLaunchKernelGGL(k_pcg_dot<2>, dim3(g), dim3(kBlock), 0, s, n, a.r, a.z, pc, a.st);
      else hipLaunchKernelGGL(k_pcg_dot<1>, dim3(g), dim3(kBlock), 0, s, n, a.r, a.z, pc, a.st);
    }
  }
  // the batches: most of the previous solve's iterations first, a few at a
  // time after them; doubling ones without a previous solve
  const long predicted = S->last_iters > 16 ? S->last_iters - S->last_iters / 16 : 0;
  int batch = 4;
  for (int l = 1; pmode != 2 && l <= S->maxl;) {
    if (predicted) batch = l <= predicted ? (int)std::min<long>(predicted - l + 1, kPcgBulkMax) : kPcgTail;
    const int last = std::min(S->maxl, l + batch - 1);
    for (int it = l; it <= last; it++) iteration(it);
    hipLaunchKernelGGL(k_pcg_check, dim3(1), dim3(kBlock), 0, s, (int)g, a.pb, nullptr, a.st, last + 1, S->h_ws);
    CEDA_HIP_CHECK(hipStreamSynchronize(s));
    if ((int)S->h_ws[kStatus] != kRunning) return ended();
    l = last + 1;
    batch = std::min(2 * batch, kPcgBatchMax);
  }
  if (pmode == 2) {
    hipLaunchKernelGGL(k_pcg_check, dim3(1), dim3(kBlock), 0, s, (int)g, a.pb, pc, a.st, S->maxl + 1, S->h_ws);
    CEDA_HIP_CHECK(hipStreamSynchronize(s));
  }
  A->nli += S->maxl;
  A->njtimes += S->maxl;
  if (pmode) A->npsolve += S->maxl;
  S->last_iters = S->maxl;
  return (sqrt(S->h_ws[kRr]) < bnorm) ? 1 : 2;
}

}  // namespace ceda_ark
