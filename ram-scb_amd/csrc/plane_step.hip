// plane_step.hip -- the middle of the split step, DRIFTE, DRIFTMU, the loss
// chain, DRIFTMU, DRIFTE (src/ModRamRun.f90:68-172), on one (K,L) plane per
// block with the plane's cells in registers.
//
// Column c < Q*NE of a block's threads is column K = c mod NE of the R
// consecutive rows of chunk q = c/NE (Q = ceil(NPA/R); R is a template
// constant, so every row lives in a register and the row loops carry no
// bounds tests).  Rows past NPA (the last chunk's, when R does not divide
// NPA) repeat the top row and are never kept; the last chunk holds at least
// two real rows.  LDS carries only what crosses threads: the plane's rows for
// the energy stencil, the three rows beside a chunk for the pitch-angle
// stencil, and the flux terms handed over between chunks.
//
// What bounds it: VALU issue.  A cell takes about 430 vector instructions a
// step (72 a DRIFTE row, 80 a DRIFTMU row, two table-driven exponentials; 522
// by the counters, with the lanes that a 35x72 plane leaves idle; the kernel
// with the plane in LDS that this one replaces took 637), two thirds
// of the issue slots over a launch of 1900 35x72 planes.  Rows in registers
// took the LDS round trips between the pitch-angle sweeps and the loss chain
// out, and with whole chunks per thread six barriers a plane are left of
// eighteen.  The rest is a block's start (one memory round trip, all tables
// in flight with the plane) and its last wave.  Plane launch of 4 species,
// before and after, by events: 35x72 (20x25 grid) 148 -> 96 us, 48x90 (40x48)
// 747 -> 453, 64x90 (20x48) 448 -> 308.
#include <hip/hip_runtime.h>

#include "ctx.h"
#include "sweep_common.h"

namespace ramgpu {

// LDS of the kernel (step_lds_doubles)
struct StepLds {
  double *F;   // NPAP rows of NE+3 energy-stencil positions F(0) .. F(NE+2)
  double *H;   // 4*Q*NE, apart or in F's place: first, second and last row of every chunk, and the flux terms
               // that DRIFTMU hands to the chunk above
  double *cf, *cm, *cl, *lt;  // per-L terms, row by row: 8, 8, 1 (HDNS), 4 (a last row of lt beyond)
  double *kt;  // SKT_N*NE, then EDOT, log(ATLOS) and WAVELO's factor of the plane (NE each)
  double *ex, *red;
  unsigned long long *cmx;
  // SEQ_STEPX: per row {XNE, BASCNE, MU, 1/MU, FNHS*MU, its reciprocal}; 3*NE handed between chunks by the line solves
  double *ct, *cy;
};
// slots of red per wave
constexpr int kStepSums = 7, kStepXSums = kSumSlots;

// Per-row terms of the Coulomb operators and the line solves: XNE(L) =
// NECR(I,J)*BANE(L) with the bounce factor BANE(L) = (1-FNIS/2/FNHS)/(1-MU^2)
// (src/ModRamCoul.f90:167-172; rows L >= NPA-10 take BANE(NPA-11)),
// BASCNE(L) = NECR*BOUNIS/2/BOUNHS (:263), MU, FACMU = FNHS*MU and the
// reciprocals of the last two (those of row 1, MU = 0, are not used).
__device__ inline void step_line_tables(CTab &t, const StepLds &d, int i, int j, int npap) {
  const int NPA = t.npa, I = i + 1, J = j + 1;
  const bool coul = t.coul != 0;
  const double necr = coul ? t.necr[i + (size_t)t.nr * j] : 0.0;
  for (int x = threadIdx.x; x < npap; x += blockDim.x) {
    const int l = min(x, NPA - 1), L = l + 1;
    double *r = d.ct + 6 * x;
    double xne = 0.0, xb = 0.0;
    if (coul) {
      const int lb = min(L, NPA - 11);
      const double mub = t.mu[lb - 1];
      xne = necr * ((1. - GEO3(t.fnis, I, J, lb) / 2. / GEO3(t.fnhs, I, J, lb)) / (1. - mub * mub));
      xb = necr * GEO3(t.bounis, I, J, L) / 2. / GEO3(t.bounhs, I, J, L);
    }
    const double mu = t.mu[l], fac = GEO3(t.fnhs, I, J, L) * mu;
    r[0] = xne;
    r[1] = xb;
    r[2] = mu;
    r[3] = 1.0 / mu;
    r[4] = fac;
    r[5] = 1.0 / fac;
  }
}

// Loads of the descriptor and of a plane's scalars go through the constant
// address space: as plain loads they were vector loads in a chain of two or
// three before the first cell arrived (11000 of a block's 61000 cycles).
//
// SEQ_STEP in place (or from src to dst); SEQ_TAPE out of place: also the
// output of every phase but the last to the tape slots after src, and the
// clamp decisions of the drift phases.  SEQ_STEPX in place with the optional
// processes the problem has on: COULEN and COULMU, WPADIF at the WPI and EMIC
// positions, FLCscatter (src/ModRamRun.f90:81-172).  rec: bit 0 record the
// CFL maxima, bit 1 COULMU's clamp (TimeRamElapsed > 0), bit 2 FLCscatter
// acts (TimeRamElapsed >= Dt_bc).
template <int SEQ, int R>
__global__ void __launch_bounds__(kPlaneMaxThreads, kStepSimdWaves) k_plane_step(Launch L, int rec) {
  constexpr bool TAPE = SEQ == SEQ_TAPE, X = SEQ == SEQ_STEPX;
  constexpr bool kKeepE = R <= 4 && !X, kKeepMu = R <= (TAPE ? 8 : 9) && !X;
  constexpr int kSums = X ? kStepXSums : kStepSums;
  extern __shared__ __align__(16) double sm[];
  for (int vb = blockIdx.x; vb < L.nv; vb += gridDim.x) {
    const CUnit u = const_unit(L, vb);
#define UNIT_DONE continue
#define UNIT_MIXED 0
#define UNIT_THREADS blockDim.x
#include "plane_step_unit.h"
    if (L.nv > (int)gridDim.x) __syncthreads();  // LDS is rewritten for the block's next plane
  }
}

// The same in blocks that may have more threads than the plane needs (not
// SEQ_STEPX, whose barriers depend on its processes).
template <int SEQ, int R>
__device__ __forceinline__ void plane_step_unit(const Launch &L, int rec, const CUnit &u, double *sm) {
  constexpr bool TAPE = SEQ == SEQ_TAPE, X = SEQ == SEQ_STEPX;
  constexpr bool kKeepE = R <= 4 && !X, kKeepMu = R <= (TAPE ? 8 : 9) && !X;
  constexpr int kSums = X ? kStepXSums : kStepSums;
#define UNIT_DONE return
#define UNIT_MIXED 1
#define UNIT_THREADS ((ncol + t.step_cells - 1) / t.step_cells * 64)
#include "plane_step_unit.h"
}

// An ensemble's members in one launch, each with the rows it has alone.
template <int SEQ>
__global__ void __launch_bounds__(kPlaneMaxThreads, kStepSimdWaves) k_plane_mixed(Launch L, int rec) {
  extern __shared__ __align__(16) double sm[];
  for (int vb = blockIdx.x; vb < L.nv; vb += gridDim.x) {
    const CUnit u = const_unit(L, vb);
    switch (u.rows) {
#define ROWS(r) \
  case r: plane_step_unit<SEQ, r>(L, rec, u, sm); break;
      STEP_ROWS(ROWS)
#undef ROWS
    }
    if (L.nv > (int)gridDim.x) __syncthreads();
  }
}

// The row counts are compiled in groups (STEP_PART of the build), each a
// translation unit of its own.
#define STEP_INST(r)                                               \
  template __global__ void k_plane_step<SEQ_STEP, r>(Launch, int); \
  template __global__ void k_plane_step<SEQ_TAPE, r>(Launch, int); \
  template __global__ void k_plane_step<SEQ_STEPX, r>(Launch, int);
#if defined(STEP_ONE)
STEP_INST(STEP_ONE)
#elif STEP_PART == 0
STEP_INST(2) STEP_INST(3) STEP_INST(4) STEP_INST(5)
#elif STEP_PART == 1
STEP_INST(6) STEP_INST(7) STEP_INST(8)
#elif STEP_PART == 2
STEP_INST(9) STEP_INST(10) STEP_INST(11)
#elif STEP_PART == 3
STEP_INST(12) STEP_INST(13)
#elif STEP_PART == 4
STEP_INST(14) STEP_INST(15) STEP_INST(16)
#elif STEP_PART == 5
template __global__ void k_plane_mixed<SEQ_STEP>(Launch, int);
#else
template __global__ void k_plane_mixed<SEQ_TAPE>(Launch, int);
#endif

}  // namespace ramgpu
