// Register-tile passes of the super-time-stepping stage loop: up to
// kTileMaxK consecutive stages of
//   Y_j = c0_j*F(t_j, Y_{j-1}) + c1_j*Y_{j-2} + c2_j*Y_n + c3_j*Y_{j-1} + c4_j*F_n
// in one launch, with the whole tile resident in registers.
//
// A workgroup holds a tile of nw*R rows x 128 columns: wavefront w owns R
// consecutive rows, a lane two adjacent columns, and Y_{j-1}, Y_{j-2}, Y_n
// and F_n of those cells stay in registers for the whole pass.  A stage needs
// its neighbours' Y_{j-1}: west and east come from the adjacent lanes (DPP
// wave shifts), south and north from the wavefront's own rows, and only the
// first and last row of each wavefront go through LDS (double-buffered, one
// barrier per stage).  Y_j overwrites Y_{j-2} in place, so the two arrays
// change roles every stage and nothing is moved.  The tile's rim loses one
// cell per stage on every side; wavefronts whose rows are no longer needed
// skip the arithmetic.  The first pass of a step forms Y_1 = c0*Y_n + c1*F_n
// on load, the last one also evaluates F(t_n + h, Y_s).
//
// Against the marching pass (k_pass), which re-forms each row's chain of K
// dependent stages serially, a stage here is one short burst of 2R
// independent cells per lane: it is bound by the FP64 issue rate (about 24
// instructions per cell: 128 x 64 cells of one CU take 1.3 us) or, on small
// grids, by the launch, where k_pass is bound by its dependency chains.
// Per stage, at the best shape of each: 128^2 1.6 us (before: 2.8 us by single
// stages; a 3-stage k_pass 4.9 us), 777 x 1001 periodic 2.2 us (6.6), 2048^2
// 12.0 us (14.8).  The adaptive RKC solve at 128^2 to t = 1 (560 steps of 19
// right-hand sides) went from 49.9 to 29.5 ms, and to 27.9 ms with the products
// of constant coefficients shared between cells (tile_stage_cc), which takes
// 256 uneven problems in a batch from 593 to 536 ms; with more, smaller tiles on
// small grids (the autotuner's choice) and faster reductions it is 19.8 ms.
//
// Every value is formed by cell(), forcing() and lc5() in their order: the
// result is bitwise that of the single-stage kernels.
#include "diffusion_internal.hpp"
#include "stencil_ops.hpp"

namespace ceda {

namespace {

// per-row tables and stage coefficients by wavefront-uniform index: scalar loads
typedef __attribute__((address_space(4))) const double ccdouble;

// neighbour columns: lane i receives lane i-1 (from_west0) or lane i+1
// (from_east0); the end lanes receive zero
__device__ inline double from_west0(double x)
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x138, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x138, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ inline double from_east0(double x)
{
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// 16 wavefronts share a CU's registers: 128 VGPRs each, which R = 4 fills (R = 8
// with 8 wavefronts was measured: 5 to 30 % slower on every grid, its row
// tables spill from the scalar registers)
constexpr int kTileThreads = kTileBatchWaves * kWave;

// what a lane keeps of the tables for its two columns, and a wavefront of
// its R rows (scalar registers)
template <int R>
struct TileTab {
  double fx, fy, mdiag;  // constant coefficients: the faces' values and minus the diagonal
  double Dw0, De0, Dw1, De1, sx0, sx1, cx0, cx1;
  double Ds[R], Dn[R], sy[R], cy[R];
  bool in0, in1;  // the columns lie in the domain
  int64_t j;      // the wavefront's first row
};

// The forcing's factor cx*sy + cy*sx does not change from stage to stage.  Kept
// in registers it costs 4R VGPRs, which the R = 4 tiles do not have: there the
// row's table values pass through an empty asm every stage, so that the
// compiler forms the products again.
constexpr int kHideTab = 4;

// F of the wavefront's rows from Y (S, N: the rows below and above them), then
// lc5 with the stage's coefficients (COMB), the result over prev.  Varying
// coefficients (periodic only)
template <int R, bool COMB>
__device__ __forceinline__ void tile_stage(const TileTab<R>& t, const double (&c)[7], double (&prev)[R][2],
                                           const double (&cur)[R][2], const double (&yn)[R][2],
                                           const double (&fn)[R][2], double2 S, double2 N)
{
#pragma unroll
  for (int q = 0; q < R; q++) {
    // the rows the neighbouring wavefronts wait for first: 0, R-1, 1, 2, ...
    const int r = q == 0 ? 0 : (q == 1 ? R - 1 : q - 1);
    const double s0 = r > 0 ? cur[r > 0 ? r - 1 : 0][0] : S.x, s1 = r > 0 ? cur[r > 0 ? r - 1 : 0][1] : S.y;
    const double n0 = r < R - 1 ? cur[r < R - 1 ? r + 1 : 0][0] : N.x;
    const double n1 = r < R - 1 ? cur[r < R - 1 ? r + 1 : 0][1] : N.y;
    const double w = from_west0(cur[r][1]), e = from_east0(cur[r][0]);
    double f0 = cell(t.Dw0, t.De0, t.Ds[r], t.Dn[r], cur[r][0], w, cur[r][1], s0, n0);
    double f1 = cell(t.Dw1, t.De1, t.Ds[r], t.Dn[r], cur[r][1], cur[r][0], e, s1, n1);
    if (COMB) {
      f0 = lc5(c, f0, prev[r][0], yn[r][0], cur[r][0], fn[r][0]);
      f1 = lc5(c, f1, prev[r][1], yn[r][1], cur[r][1], fn[r][1]);
    }
    prev[r][0] = f0;
    prev[r][1] = f1;
  }
}

// tile_stage where every face coefficient in x is one value and every one in y
// another (the manufactured problem always).  MASK: zero outside the domain
// (the Dirichlet ghosts).  The products of a cell with them
// are formed once and handed to its neighbours, so F takes 3 multiplications
// and 4 additions instead of 5 and 8, the diagonal being one number.  The terms
// and their order are cell()'s; its 0 + t, which only turns a -0 into +0, is
// left out of the stages.
template <int R, bool MMS, bool MASK, bool COMB>
__device__ __forceinline__ void tile_stage_cc(const TileTab<R>& t, int64_t ny, const double (&c)[7],
                                              double (&prev)[R][2], const double (&cur)[R][2],
                                              const double (&yn)[R][2], const double (&fn)[R][2], double2 S, double2 N)
{
  const double T1 = c[5], T2 = c[6];
  double s0 = t.fy * S.x, s1 = t.fy * S.y;  // fy times the rows below, here and above
  double m0 = t.fy * cur[0][0], m1 = t.fy * cur[0][1];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const double n0 = t.fy * (r < R - 1 ? cur[r < R - 1 ? r + 1 : 0][0] : N.x);
    const double n1 = t.fy * (r < R - 1 ? cur[r < R - 1 ? r + 1 : 0][1] : N.y);
    if (!MASK || (t.j + r >= 0 && t.j + r < ny)) {  // else a row of ghosts: prev is and stays zero
      double syj = t.sy[r], cyj = t.cy[r];
      if (MMS && R >= kHideTab) asm volatile("" : "+s"(syj), "+s"(cyj));
      const double p0 = t.fx * cur[r][0], p1 = t.fx * cur[r][1];
      const double w = from_west0(p1), e = from_east0(p0);
      double f0 = t.mdiag * cur[r][0], f1 = t.mdiag * cur[r][1];
      f0 = f0 + w;
      f1 = f1 + p0;
      f0 = f0 + p1;
      f1 = f1 + e;
      f0 = f0 + s0;
      f1 = f1 + s1;
      f0 = f0 + n0;
      f1 = f1 + n1;
      if (!COMB) {
        f0 = 0.0 + f0;
        f1 = 0.0 + f1;
      }
      if (MMS) {
        f0 = f0 + forcing(T1, T2, t.sx0, t.cx0, syj, cyj);
        f1 = f1 + forcing(T1, T2, t.sx1, t.cx1, syj, cyj);
      }
      if (COMB) {
        f0 = lc5(c, f0, prev[r][0], yn[r][0], cur[r][0], fn[r][0]);
        f1 = lc5(c, f1, prev[r][1], yn[r][1], cur[r][1], fn[r][1]);
      }
      if (MASK) {
        f0 = t.in0 ? f0 : 0.0;
        f1 = t.in1 ? f1 : 0.0;
      }
      prev[r][0] = f0;
      prev[r][1] = f1;
    }
    s0 = m0;
    s1 = m1;
    m0 = n0;
    m1 = n1;
  }
}

struct TileGeo {
  const double *fx, *fy, *sx, *sy, *cx, *cy;
  int64_t nx, ny;
  int strips, hl;  // column strips, halo lanes on each side
  int own;         // rows a tile owns
  int y0;          // row offset of a tile's first row from its first owned one
};

// the pass on one tile: K stages with the coefficients sc[8*m .. 8*m+6].  CC:
// constant coefficients, as the manufactured problem (not PER) always has
template <int R, bool PER, bool CC>
__device__ __forceinline__ void tile_pass(const TileGeo& g, const TileIO& o, ccdouble* sc, int strip, int rb,
                                          double2* lds, int nw)
{
  static_assert(PER || CC, "the manufactured problem has constant coefficients");
  constexpr bool MMS = !PER;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
  const int64_t nx = g.nx, ny = g.ny;
  const int64_t c = (int64_t)strip * (kWave - 2 * g.hl) * 2 + 2 * (lane - g.hl);
  const int64_t jown = (int64_t)rb * g.own;
  const int64_t jend = jown + g.own < ny ? jown + g.own : ny;
  TileTab<R> t;
  t.j = jown + g.y0 + (int64_t)wave * R;
  int64_t c0 = c, c1 = c + 1;
  if (PER) {
    while (c0 < 0) c0 += nx;
    while (c0 >= nx) c0 -= nx;
    c1 = c0 + 1 < nx ? c0 + 1 : 0;
  }
  t.in0 = PER || (c0 >= 0 && c0 < nx);
  t.in1 = PER || (c1 >= 0 && c1 < nx);
  t.fx = t.fy = t.mdiag = 0.0;
  if (CC) {
    t.fx = ((ccdouble*)g.fx)[0];
    t.fy = ((ccdouble*)g.fy)[0];
    t.mdiag = -((t.fx + t.fx) + (t.fy + t.fy));
  }
  t.Dw0 = t.De0 = t.Dw1 = t.De1 = t.sx0 = t.sx1 = t.cx0 = t.cx1 = 0.0;
  if (t.in0) {
    if (!CC) t.Dw0 = g.fx[c0];
    if (!CC) t.De0 = g.fx[c0 + 1];
    if (MMS) {
      t.sx0 = g.sx[c0];
      t.cx0 = g.cx[c0];
    }
  }
  if (t.in1) {
    if (!CC) t.Dw1 = g.fx[c1];
    if (!CC) t.De1 = g.fx[c1 + 1];
    if (MMS) {
      t.sx1 = g.sx[c1];
      t.cx1 = g.cx[c1];
    }
  }
  // wavefront-uniform rows: tables through the scalar cache
  ccdouble *fy = (ccdouble*)g.fy, *sy = (ccdouble*)g.sy, *cy = (ccdouble*)g.cy;
  int64_t jr[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    int64_t j = t.j + r;
    if (PER) {
      while (j < 0) j += ny;
      while (j >= ny) j -= ny;
    }
    jr[r] = j;
    const bool ok = PER || (j >= 0 && j < ny);
    t.Ds[r] = (ok && !CC) ? fy[j] : 0.0;
    t.Dn[r] = (ok && !CC) ? fy[j + 1] : 0.0;
    t.sy[r] = (MMS && ok) ? sy[j] : 0.0;
    t.cy[r] = (MMS && ok) ? cy[j] : 0.0;
  }

  double A[R][2], B[R][2], yn[R][2], fn[R][2];  // Y_{j-2}, Y_{j-1}, Y_n, F_n
  // a lane's two columns of a row: one 16-byte access where the rows are even
  // (c0 even, both columns in or both out), else two
  const bool even = (nx & 1) == 0;
  auto ld = [&](const double* __restrict__ p, double (&v)[R][2]) {
#pragma unroll
    for (int r = 0; r < R; r++) {
      v[r][0] = v[r][1] = 0.0;
      if (!PER && (jr[r] < 0 || jr[r] >= ny)) continue;
      const double* q = p + jr[r] * nx;
      if (even) {
        if (t.in0) {
          const double2 x = *reinterpret_cast<const double2*>(q + c0);
          v[r][0] = x.x;
          v[r][1] = x.y;
        }
      } else {
        if (t.in0) v[r][0] = q[c0];
        if (t.in1) v[r][1] = q[c1];
      }
    }
  };
  ld(o.yn, yn);
  ld(o.fn, fn);
  if (o.first) {  // Y_1 = c0 Y_n + c1 F_n (N_VLinearSum order), Y_0 = Y_n
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        B[r][k] = o.a0 * yn[r][k] + o.a1 * fn[r][k];
        A[r][k] = yn[r][k];
      }
  } else {
    ld(o.yjm1, B);
    ld(o.yjm2, A);
  }

  // lds[buffer][wave][first row, last row][lane]
  const int bufsz = nw * 2 * kWave;
  double2* mine = lds + wave * 2 * kWave + lane;
  auto publish = [&](int b, const double (&v)[R][2]) {
    mine[b * bufsz] = make_double2(v[0][0], v[0][1]);
    mine[b * bufsz + kWave] = make_double2(v[R - 1][0], v[R - 1][1]);
  };
  auto south = [&](int b) { return wave > 0 ? mine[b * bufsz - kWave] : make_double2(0.0, 0.0); };
  auto north = [&](int b) { return wave < nw - 1 ? mine[b * bufsz + 2 * kWave] : make_double2(0.0, 0.0); };
  publish(0, B);
  // wavefronts of ghost rows only never compute: their rows are zero for good
  if (!PER && (t.j + R <= 0 || t.j >= ny)) publish(1, B);
  // every cell of the wavefront inside the domain: no masks
  bool mask = false;
  if (!PER) {
    const int64_t cl = (int64_t)strip * (kWave - 2 * g.hl) * 2 - 2 * g.hl;
    mask = t.j < 0 || t.j + R > ny || cl < 0 || cl + 2 * kWave > nx;
    mask = __builtin_amdgcn_readfirstlane((int)mask) != 0;
  }
  const int L = o.K + o.rhs;  // levels of the pass
  // rows still needed after m levels: [jown - (L - m), jend + (L - m))
  auto needed = [&](int m) {
    const int64_t lo = jown - (L - m), hi = jend + (L - m);
    return t.j + R > (PER || lo > 0 ? lo : 0) && t.j < (PER || hi < ny ? hi : ny);
  };
  double cf[7];
  auto coef = [&](int m) {
#pragma unroll
    for (int k = 0; k < 7; k++) cf[k] = sc[8 * m + k];
  };
  auto step = [&](int m, double (&prev)[R][2], const double (&cur)[R][2]) {
    coef(m);
    __syncthreads();
    if (needed(m + 1)) {
      const double2 S = south(m & 1), N = north(m & 1);
      if (CC && !PER && mask) tile_stage_cc<R, MMS, true, true>(t, ny, cf, prev, cur, yn, fn, S, N);
      else if (CC) tile_stage_cc<R, MMS, false, true>(t, ny, cf, prev, cur, yn, fn, S, N);
      else tile_stage<R, true>(t, cf, prev, cur, yn, fn, S, N);
      publish((m + 1) & 1, prev);
    }
  };
  int m = 0;
  for (; m + 1 < o.K; m += 2) {
    step(m, A, B);
    step(m + 1, B, A);
  }
  if (m < o.K) {  // odd: the last stage is in A
    step(m, A, B);
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
      for (int k = 0; k < 2; k++) {
        const double x = A[r][k];
        A[r][k] = B[r][k];
        B[r][k] = x;
      }
  }
  // B = the last stage, A = the one before it
  const bool ownl = lane >= g.hl && lane < kWave - g.hl;
  auto st = [&](double* __restrict__ p, const double (&v)[R][2]) {
    if (!p || !ownl) return;
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int64_t j = t.j + r;
      if (j < jown || j >= jend) continue;
      double* q = p + j * nx + c;
      if (even) {
        if (c < nx) *reinterpret_cast<double2*>(q) = make_double2(v[r][0], v[r][1]);
      } else {
        if (c < nx) q[0] = v[r][0];
        if (c + 1 < nx) q[1] = v[r][1];
      }
    }
  };
  st(o.outA, A);
  st(o.outB, B);
  if (o.rhs) {
    coef(o.K);
    __syncthreads();
    if (needed(L)) {
      const double2 S = south(o.K & 1), N = north(o.K & 1);
      if (CC) tile_stage_cc<R, MMS, false, false>(t, ny, cf, A, B, yn, fn, S, N);
      else tile_stage<R, false>(t, cf, A, B, yn, fn, S, N);
      st(o.outF, A);
    }
  }
}

template <int R, bool PER, bool CC>
__global__ __launch_bounds__(kTileThreads) void k_tile(const TileGeo g, const TileOps o)
{
  extern __shared__ double2 tile_lds[];
  // XCD-aware order (workgroups go round-robin to the 8 XCDs): each XCD takes
  // a contiguous share of the tiles, whose halos then meet in its L2
  const unsigned nb = gridDim.x, b = blockIdx.x;
  const unsigned q = nb >> 3, r = nb & 7u, xcd = b & 7u, loc = b >> 3;
  const unsigned tile = xcd * q + (xcd < r ? xcd : r) + loc;
  const int strip = (int)(tile % (unsigned)g.strips), rb = (int)(tile / (unsigned)g.strips);
  tile_pass<R, PER, CC>(g, o, (ccdouble*)o.c, strip, rb, tile_lds, (int)(blockDim.x / kWave));
}

// column strips and owned rows of tiles of `rows` rows with halo H.  A
// Dirichlet domain no larger than the tile needs no halo: what lies outside is
// the zero ghosts.
void tile_shape(int64_t nx, int64_t ny, bool per, int64_t rows, int H, int& strips, int& hl, int& own, int& y0)
{
  if (!per && nx <= 2 * kWave) {
    hl = 0;
    strips = 1;
  } else {
    hl = (H + 1) / 2;
    const int64_t ow = 2 * (kWave - 2 * hl);
    strips = (int)((nx + ow - 1) / ow);
  }
  if (!per && ny <= rows) {
    own = (int)ny;
    y0 = 0;
  } else {
    own = (int)(rows - 2 * H);
    y0 = -H;
  }
}

// one tile of pass q of its slot (see TileSlot)
template <int R>
__global__ __launch_bounds__(kTileThreads) void k_tile_batch(const TileSlot* __restrict__ slots,
                                                             const TileRef* __restrict__ tiles, int k, int q,
                                                             int adaptive)
{
  extern __shared__ double2 tile_lds[];
  const unsigned nb = gridDim.x, b = blockIdx.x;
  const unsigned bq = nb >> 3, br = nb & 7u, xcd = b & 7u, loc = b >> 3;
  const TileRef ref = tiles[xcd * bq + (xcd < br ? xcd : br) + loc];  // XCD-aware order
  const TileSlot& t = slots[ref.slot];
  TileGeo g;
  g.fx = t.fx;
  g.fy = t.fy;
  g.sx = t.sx;
  g.sy = t.sy;
  g.cx = t.cx;
  g.cy = t.cy;
  g.nx = t.nx;
  g.ny = t.ny;
  g.strips = t.strips;
  g.hl = t.hl;
  g.own = t.own[k];
  g.y0 = t.y0[k];
  // pass q of np of nearly equal lengths (tile_len: the first ones longer)
  const int n = t.s - 1, base = n / t.np, rem = n - base * t.np;
  const int j = 2 + q * base + (q < rem ? q : rem), par = q & 1;
  const bool last = q == t.np - 1;
  TileIO o;
  o.K = base + (q < rem ? 1 : 0);
  o.first = q == 0;
  o.rhs = last && adaptive;
  o.yn = t.yn;
  o.fn = t.fn;
  o.a0 = 1.0;
  o.a1 = t.a1;
  o.yjm2 = t.buf[2 - 2 * par];
  o.yjm1 = t.buf[3 - 2 * par];
  o.outA = last ? nullptr : t.buf[2 * par];
  o.outB = t.buf[2 * par + 1];
  o.outF = t.buf[2 * par];
  ccdouble* sc = (ccdouble*)(t.coef + 8 * (j - 2));
  if (t.per && t.cc) tile_pass<R, true, true>(g, o, sc, ref.strip, ref.rb, tile_lds, kTileBatchWaves);
  else if (t.per) tile_pass<R, true, false>(g, o, sc, ref.strip, ref.rb, tile_lds, kTileBatchWaves);
  else tile_pass<R, false, true>(g, o, sc, ref.strip, ref.rb, tile_lds, kTileBatchWaves);
}

TileGeo tile_geo(const DiffusionProblem* P, const TileCfg& t, int H)
{
  TileGeo g;
  g.fx = P->d_fx;
  g.fy = P->d_fy;
  g.sx = P->d_sx;
  g.sy = P->d_sy;
  g.cx = P->d_cx;
  g.cy = P->d_cy;
  g.nx = P->p.nx;
  g.ny = P->p.ny;
  tile_shape(g.nx, g.ny, P->p.kind == DIFFUSION_CEDA_PERIODIC, (int64_t)t.R * t.nw, H, g.strips, g.hl, g.own, g.y0);
  return g;
}

int64_t tile_blocks(const TileGeo& g) { return g.strips * ((g.ny + g.own - 1) / g.own); }

}  // namespace

// a pass of K stages (and the closing RHS) can run on tiles of this shape (one
// of fewer stages then can too)
bool tile_ok(const DiffusionProblem* P, const TileCfg& t, int K, int rhs)
{
  if (K < 1 || K > kTileMaxK) return false;
  if ((t.R != 1 && t.R != 2 && t.R != 4) || t.nw < 1 || t.nw > 16) return false;
  const int H = K + (rhs ? 1 : 0);
  if (P->p.nx > (int64_t)1 << 30 || P->p.ny > (int64_t)1 << 30) return false;
  const TileGeo g = tile_geo(P, t, H);
  if (g.own < 1 || 2 * g.hl >= kWave) return false;
  // a launch has fewer than 2^32 threads: few rows per tile on a very tall grid
  // (2 x 14,000,000 on tiles that own one row) would have more
  return tile_blocks(g) <= (int64_t)0xffffffff / (t.nw * kWave);
}

void launch_tile(DiffusionProblem* P, const TileCfg& t, const TileOps& o, hipStream_t s)
{
  if (!tile_ok(P, t, o.K, o.rhs)) CEDA_HIP_CHECK(hipErrorInvalidConfiguration);  // (callers check)
  const TileGeo g = tile_geo(P, t, o.K + (o.rhs ? 1 : 0));
  const unsigned grid = (unsigned)tile_blocks(g);
  const unsigned nt = (unsigned)(t.nw * kWave);
  const size_t lds = sizeof(double2) * 2 * 2 * kWave * (size_t)t.nw;  // at most 64 KiB
  const bool per = P->p.kind == DIFFUSION_CEDA_PERIODIC;
#define CEDA_TILE(RR)                                                                                      \
  if (!per) hipLaunchKernelGGL((k_tile<RR, false, true>), dim3(grid), dim3(nt), lds, s, g, o);              \
  else if (P->constant_faces) hipLaunchKernelGGL((k_tile<RR, true, true>), dim3(grid), dim3(nt), lds, s, g, o); \
  else hipLaunchKernelGGL((k_tile<RR, true, false>), dim3(grid), dim3(nt), lds, s, g, o);
  switch (t.R) {
    case 1: CEDA_TILE(1) break;
    case 2: CEDA_TILE(2) break;
    default: CEDA_TILE(4) break;
  }
#undef CEDA_TILE
}

bool tile_slot_geometry(TileSlot& t)
{
  for (int k = 0; k < 2; k++) {
    tile_shape(t.nx, t.ny, t.per, kTileBatchWaves * (k == 0 ? 4 : 2), kTileBatchK + 1, t.strips, t.hl, t.own[k], t.y0[k]);
    if (t.strips > 32767 || (t.ny + t.own[k] - 1) / t.own[k] > 32767) return false;
  }
  return true;
}

int tile_slot_tiles(const TileSlot& t, int k) { return t.strips * ((t.ny + t.own[k] - 1) / t.own[k]); }

void launch_tile_batch(const TileSlot* slots, const TileRef* tiles, int ntiles, int k, int q, int adaptive, hipStream_t s)
{
  if (ntiles <= 0) return;
  const size_t lds = sizeof(double2) * 2 * 2 * kWave * kTileBatchWaves;
  if (k == 0)
    hipLaunchKernelGGL(k_tile_batch<4>, dim3(ntiles), dim3(kTileThreads), lds, s, slots, tiles, k, q, adaptive);
  else
    hipLaunchKernelGGL(k_tile_batch<2>, dim3(ntiles), dim3(kTileThreads), lds, s, slots, tiles, k, q, adaptive);
}

}  // namespace ceda
