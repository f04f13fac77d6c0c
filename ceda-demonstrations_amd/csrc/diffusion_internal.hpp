// Internal interface between the diffusion problem kernels and the
// integrator's fused super-time-stepping path.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "diffusion_hip.h"
#include "nvhip_internal.hpp"

// launch configuration of one stencil kernel kind (the plain RHS or the fused
// STS stage): variant 0 = row-interleaved tiles, rows = rows per wavefront;
// variant 1 = y-marching, rows = consecutive rows per wavefront; nt = 1 uses
// non-temporal loads/stores for the streamed operands
struct StencilCfg {
  int variant = 0;
  int rows = 1;
  int nt = 0;
};

// shape of the register-tile passes (stage_tile.hip): up to K stages per pass
// on tiles of nw wavefronts with R rows each; K = 0: not used
struct TileCfg {
  int K = 0, R = 0, nw = 0;
};

struct LearnedPrec;
struct MGHierarchy;

struct DiffusionProblem {
  DiffusionParams p;
  int64_t n = 0;
  double dx = 0, dy = 0;
  // host copies of the HBM tables (built with the same expressions as the
  // reference so device results are bitwise reproducible)
  std::vector<double> fx, fy, px, py, sx, sy, cx, cy, ax, by;
  double *d_fx = nullptr, *d_fy = nullptr, *d_px = nullptr, *d_py = nullptr;
  double *d_sx = nullptr, *d_sy = nullptr, *d_cx = nullptr, *d_cy = nullptr;
  double *d_ax = nullptr, *d_by = nullptr;
  double* d_tables = nullptr;  // the one allocation the d_ tables above point into
  N_Vector diag = nullptr;  // Jacobi inverse diagonal (udata->diag, main.cpp:223)
  double diag_gamma = 0.0;       // the gamma of the last PSetup, which computed diag
  bool diag_gamma_set = false;   // diag was last written by PSetup
  bool constant_faces = false;   // every face table holds one value (constant coefficients)
  SUNContext ctx = nullptr;
  ceda::Exec* exec = nullptr;
  long nrhs = 0;
  // [0] RHS kernel, [1] fused stage kernel, [2] multi-stage pass (variant =
  // stages per pass K, 0 = single-stage kernels only; rows; nt)
  StencilCfg cfg[3];
  TileCfg tile;  // the autotuner's register-tile shape, where it beats cfg[2]
  LearnedPrec* learned = nullptr;  // network of LearnedPSolve (not owned)
  double learned_out_scale = 1.0;  // its output scale for this problem (LearnedPSetup)
  MGHierarchy* mg = nullptr;       // multigrid hierarchy of MGPSetup/MGPSolve (owned)
  int mg_relax = 2, mg_nrelax = 2;  // V-cycle smoother: PFMG relax type 2|3, sweeps
  bool tuned = false;
};

namespace ceda {

void mg_destroy(MGHierarchy* H);

// One entry of the device-resident stage table of the fused STS path.  Every
// kernel of a step reads its coefficients, time factors and operand pointers
// from its entry, so a captured HIP graph stays valid when h, t and the buffer
// roles change between steps; only the stage count s selects the graph.
struct alignas(16) StageEntry {
  double c[5];          // combination coefficients
  double T1, T2, pad;   // MMS time factors of the RHS evaluated in this kernel
  const double* yjm1;   // stencil input
  const double* yjm2;
  const double* yn;
  const double* fn;
  double* out;
  const void* pad2[3];
};
static_assert(sizeof(StageEntry) == 128, "StageEntry layout");

// out = c0*yn + c1*fn (the first STS stage, N_VLinearSum order)
void launch_stage1_entry(DiffusionProblem* P, const StageEntry* e, hipStream_t s);
// out = c0*F(yjm1) + c1*yjm2 + c2*yn + c3*yjm1 + c4*fn
void launch_fused_entry(DiffusionProblem* P, const StageEntry* e, hipStream_t s);
// out = F(yjm1) with the entry's time factors
void launch_rhs_entry(DiffusionProblem* P, const StageEntry* e, hipStream_t s);

// K consecutive fused stages in one sweep (temporal blocking): stages read
// e[0].yjm1, e[0].yjm2, e[0].yn, e[0].fn; stage K-1 is written to e[K-2].out
// and stage K to e[K-1].out (K = 1..kMaxPassStages).  rows = output rows per
// wavefront tile, nt: bit 0 non-temporal streams, bit 1 Y_n and F_n rows in LDS
// and coefficients re-read.  Bitwise equal to K single-stage launches.
void launch_pass(DiffusionProblem* P, int K, int rows, int nt, const StageEntry* e, hipStream_t s);
// the fewest rows with which the pass's tiles run in `rounds` rounds of the
// wavefronts that the GPU holds (0: unknown)
int pass_fill_rows(const DiffusionProblem* P, int K, int nt, int rounds);
// halo lanes of a K-stage pass (each side of a wavefront strip)
int pass_halo_lanes(int K, int cpl);

// ---- register-tile passes (stage_tile.hip)
constexpr int kTileMaxK = 12;  // stages per pass
// the operands of one pass, by value: K stages with the coefficients
// c[8m .. 8m+4], time factors c[8m+5], c[8m+6]; first: Y_{j-1} = a0 Y_n +
// a1 F_n and Y_{j-2} = Y_n instead of reading them; outA (may be null): the
// next-to-last stage, outB: the last one; rhs: also outF = F(last stage)
// with the time factors c[8K+5], c[8K+6].  Outputs must not alias inputs.
struct TileIO {
  const double *yjm1, *yjm2, *yn, *fn;
  double *outA, *outB, *outF;
  double a0, a1;
  int K, first, rhs, pad;
};
struct TileOps : TileIO {
  double c[8 * (kTileMaxK + 1)];
};
bool tile_ok(const DiffusionProblem* P, const TileCfg& t, int K, int rhs);
void launch_tile(DiffusionProblem* P, const TileCfg& t, const TileOps& o, hipStream_t s);
// passes of a loop of n stages and the length of the next one: equal lengths
__host__ __device__ inline int tile_passes(int n, int K) { return (n + K - 1) / K; }
__host__ __device__ inline int tile_len(int left, int passes) { return (left + passes - 1) / passes; }

// the same passes for many problems in one launch.  A slot is one problem's
// attempt: np passes of up to kTileBatchK stages over its buffers (pass q
// reads buf[2(1-q%2)], buf[2(1-q%2)+1] = Y_{j-2}, Y_{j-1} and writes the other
// two: next-to-last stage, last stage; the last pass leaves F(t_n + h, Y_s)
// in the first of its pair when adaptive)
constexpr int kTileBatchK = 10;
constexpr int kTileBatchWaves = 16;
struct TileSlot {
  const double *fx, *fy, *sx, *sy, *cx, *cy;
  const double *yn, *fn;
  double* buf[4];
  const double* coef;  // stage j's {c0..c4, T1, T2, -} at coef + 8 (j - 2), then the closing RHS's
  double a1;           // Y_1 = Y_n + a1 F_n
  int nx, ny, per, cc, s, np, strips, hl;  // cc: constant coefficients
  int own[2], y0[2];   // rows a tile owns and their offset, R = 4 and R = 2
};
struct TileRef {
  int slot;
  short strip, rb;
};
// a slot's geometry (strips, hl, own, y0) from nx, ny, per; false when the
// problem is too large for TileRef
bool tile_slot_geometry(TileSlot& t);
int tile_slot_tiles(const TileSlot& t, int k);  // tiles with R = 4 (k = 0) or R = 2 (k = 1)
// pass q of the slots whose tiles are listed
void launch_tile_batch(const TileSlot* slots, const TileRef* tiles, int ntiles, int k, int q, int adaptive, hipStream_t s);

// ---- batched super-time-stepping (many independent problems, one launch
// per pass index) ----
constexpr int kMaxPassStages = 6;  // stages per multi-stage pass (one problem)
constexpr int kBatchMaxK = 5;  // stages per pass the batch tile geometry covers
struct BatchDesc {             // per problem, static
  const double *fx, *fy, *sx, *sy, *cx, *cy;
  int64_t nx, ny;
  int per, cpl, rows, strips;
};
struct BatchTile {             // one wavefront tile, problems in slot order
  int slot, prob, strip, rb;
};
int batch_halo_lanes(int cpl);
// column layout and boundary shared by every problem of a batch, so that
// the phase kernel instance holds only that layout's code and registers
enum { kLayoutAny = 0, kLayoutC2Mms = 1, kLayoutC2Per = 2 };
// phase 0: stage 1 of every slot; phase q >= 1: stages j = 2+(q-1)*kmax ..
// j+kmax-1 (clipped at s = stages[slot]) of the slots with j <= s, and the RHS
// at t_n + h (adaptive) of the slots whose last pass was phase q-1; entries of
// slot k start at ent + k*stride; tiles [0, ntiles) must cover exactly those
// slots (a prefix of the slots when they are sorted by s, descending)
void launch_batch_phase(const BatchDesc* desc, const BatchTile* tiles, int ntiles,
                        const StageEntry* ent, int stride, const int* stages, int phase, int kmax,
                        int adaptive, int layout, hipStream_t s);


// one STS stage of the LSRKStep recurrence, fused with the RHS evaluation:
//   out = c0*F(yjm1) + c1*yjm2 + c2*yn + c3*yjm1 + c4*fn
// coef points at 8 device doubles {c0..c4, T1, T2, unused}; F is the diffusion
// RHS with MMS time factors (T1, T2).  Bitwise equal to diffusion() followed
// by N_VLinearCombination(5, ...) in that association order.
void launch_fused_stage(DiffusionProblem* P, const double* coef, const double* yjm1,
                        const double* yjm2, const double* yn, const double* fn,
                        double* out, hipStream_t s);
// f = F(u) with the time factors read from the device (coef[5], coef[6])
void launch_rhs_devtime(DiffusionProblem* P, const double* coef, const double* u,
                        double* f, hipStream_t s);
// host evaluation of the MMS time factors of the forcing (README.md:28)
void mms_time_factors(double t, double* T1, double* T2);

}  // namespace ceda
