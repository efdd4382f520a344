// ramgpu_dev.h -- device-side data of the RAM split step (gfx950).
//
// F2 is kept on the device per species in a [I][J][L][K] layout (K fastest):
// the (K,L) plane of one (I,J) cell is one contiguous run of NE*NPA doubles.
// The radial and local-time sweeps run one thread per line, or per piece of a
// line where the lines are few, with consecutive lanes on consecutive (L,K)
// positions, so every load and store of a wave is one contiguous run; the
// energy and pitch-angle sweeps take a whole (K,L) plane per block, in the
// fused step with its rows in registers (and the loss operators between them),
// as single operators in LDS.
//
// Coefficient tables hold the reference's intermediate quantities (its
// GPA, GPR1.., DRD1.., CMUDOT.. terms) computed in the reference's expression
// order, plus correctly rounded reciprocals of every divisor that is reused
// across cells, so that each Courant number is rebuilt per cell with exactly
// the reference's sequence of roundings.  Tables read together are packed
// together (one base address, consecutive fields).
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>

namespace ramgpu {

constexpr int kMaxSpecies = 8;
constexpr int kLineThreads = 256;      // R/P sweep kernels: one line per thread
constexpr int kPlaneThreads = 512;     // plane adjoint kernels: one (K,L) plane per block
constexpr int kPlaneMaxThreads = 1024; // forward plane kernels: block size chosen per problem
constexpr int kMaxCellsPerThread = 16; // cells of one plane per thread, in every mapping
constexpr int kMaxPlaneCells = kPlaneThreads * kMaxCellsPerThread;  // NE*NPA bound, checked at creation
// SUMRC partial-sum slots of one ram_run: 0..6 the loss chain's (plane
// blocks), 7 the last SUMRC (radial blocks), 8..11 the Coulomb operators'
// (plane blocks: after the first drift half, after COULEN; after the second
// COULMU, after the second COULEN), 12, 13 after the EMIC WPADIFs
constexpr int kSumSlots = 14;
// further slots of partials: ramgpu_sumrc's ELORC, and the blocks' CFL maxima
// of DRIFTR and DRIFTP (cleared by k_finalize)
constexpr int kSlotElorc = kSumSlots, kSlotCflR = kSumSlots + 1, kSlotCflP = kSumSlots + 2, kSlots = kSumSlots + 3;
constexpr int kSumRadial = 7;
constexpr int kSumCoul = 8;
constexpr int kSumEmic = 12;
enum SumAny { ANY_WPI = 1, ANY_EMIC = 2, ANY_CEX = 4 };
// k_finalize's summode: 0 none, 1 one SUMRC (slot 0), 2 the fused step's chain
constexpr int kMuSpread = 4;           // LDS slots per pitch-angle row of DRIFTMU's CFL maximum (by K mod 4)
constexpr int kFinalizeThreads = 1024;  // one block per (problem, species) of k_finalize; also k_ghost's block
constexpr int kGhostPlanes = kFinalizeThreads / 2;  // (K,L) planes per block of k_ghost
constexpr int kCoefCells = 128;         // (I,J) cells per block of k_coef_ij

// packed per-(I,J) terms of the plane sweeps, kij[(i*NT+j)*8 + ..]
enum KijField { KIJ_DRD1, KIJ_DPD1, KIJ_BIJ, KIJ_RBIJ, KIJ_DRM1, KIJ_DPM1, KIJ_DB2, KIJ_MG };
// packed per-(I,J,L) DRIFTE terms, kle[((i*NT+j)*NPA+l)*8 + ..]
enum KleField { KLE_HS, KLE_RHS, KLE_DRD2, KLE_DPD2, KLE_GR, KLE_GP, KLE_DB1, KLE_DI1 };
// packed per-(I,J,L) DRIFTMU terms, klm[((i*NT+j)*NPA+l)*8 + ..]
enum KlmField { KLM_BHS, KLM_RBHS, KLM_DRM2, KLM_DPM2, KLM_CMUDOT, KLM_GMR, KLM_GMP, KLM_DI2 };

// per-species per-K terms of the plane step, kt[(s*SKT_N + field)*NE + k]; the
// charge's sign is folded into EKP and MKP (x/QS == x*QS for QS = +-1)
enum StepKt { SKT_EKPQ, SKT_MKPQ, SKT_SIGV, SKT_DE, SKT_RDE, SKT_WE, SKT_RWE, SKT_EKW, SKT_N };

// All device pointers and scalars of one problem (one ensemble member).
// Lives in device memory; kernels read it through a pointer.
struct Tab {
  int ns, nr, nt, ne, npa;
  double dts, betalim, fraccfl, mdr, dphi, conf1, conf2;
  double omet;  // OME*DTs/DPHI of DRIFTP
  // species
  int charge[kMaxSpecies];
  int cex[kMaxSpecies];
  double rmas[kMaxSpecies];
  // 1-D grid
  const double *rlz, *ekev, *ebnd, *we, *de, *grel, *grbnd, *v, *mu, *wmu, *dmu;
  const int *upa;  // int(UPA(I)), 1-based values
  // geometry in the reference's Fortran layout
  const double *fnhs, *fnis, *bounhs, *bounis, *hdns_f, *didt, *dibndt;
  const double *bnes, *dbdt, *vt, *eir, *eip;
  const int *mgnp;
  const double *fgeos;   // (NS,NT,NE,NPA)
  double *bscale;        // (NS)
  const double *lz, *phi;  // LZ(NR+1), PHI(NT) for the device-side VT of a Kp schedule
  // reciprocals of grid widths: 1/DE(K), 1/WE(K), 1/DMU(L), 1/WMU(L)
  double *rde, *rwe, *rdmu, *rwmu;
  double *rrlz;    // [i] 1/RLZ(I)
  double2 *rsi;    // [i] {RLZ(I)+0.5*MDR, 1/..}                       (DRIFTR)
  double4 *rij;    // [i*NT+j] {CR, BNES(I,J)+BNES(I+1,J), 1/.., outsideMGNP(I,J)}
  double *q1;      // [(l*NR+i)*NT+j] CGR3/(FNHS(I)+FNHS(I+1))         (DRIFTR)
  double4 *pij;    // [i*NT+j] {VT term*P1, EIR term, BNES(I,J)+BNES(I,J1), 1/..}
  double4 *pl;     // [(l*NR+i)*NT+j] {GPA1+GPA2, FNHS(J)+FNHS(J1), 1/.., outsideMGNP(I,J)}
  double *kij;     // [(i*NT+j)*8] KijField
  double *kle;     // [((i*NT+j)*NPA+l)*8] KleField
  double *klm;     // [((i*NT+j)*NPA+l)*8] KlmField
  double2 *kll;    // [(i*NT+j)*NPA+l] {HDNS, 1/FNHS}                   (loss)
  // per species
  double *p4;     // [s][k] DRIFTR P4
  double *ekp;    // [s][k] EBND*1e3*(GRBND+1)/2/GRBND (DRIFTE EDT1 prefix)
  double *mkp;    // [s][k] EKEV*1e3*(GREL+1)/2/GREL   (DRIFTMU EDT prefix)
  double *p2;     // [s][i][k]
  double *edot;   // [s][i][k]
  double *sigv;   // [s][k] 10**Y*V(S,K) of CEPARA
  double *atlos;  // [s][i][k]
  double *rel;    // [s][8]: GREL1, GREL2, sq1, GRZERO, sq0, 1/GREL2, 1/GREL1
  double *kt;     // [s][8][k] the plane step's per-K terms (StepKt)
  double *lt4;    // [l][4] DMU, 1/DMU, WMU, 1/WMU
  int *carry;     // [s][NE*NPA] DRIFTR ghost carry
  double *latl;   // [s][i][k] log(ATLOS): ATLOS**(1/FNHS) = exp(log(ATLOS)/FNHS)
  // WAVELO (electron lifetimes) of the species with wpi[s] set: WALOS1/2/3
  // as wl[(q*NS + s)*NR*NE + i*NE + k], q = 0,1,2; the plasmapause L of each
  // local time; KP of the current step (written by ramgpu_set_kp, the Kp
  // schedules and ramgpu_set_wave_params)
  int wpi[kMaxSpecies];
  double *wl;
  double *wavef;  // [((s*NR + i)*NT + j)*NE + k] exp(-DTs/TAU) of the step (k_coef_ij)
  double *rlpp;   // [j]
  double *kpnow;  // 1 value
  double *lsx;    // [s][3]: LSWAE, LSCOE, LSCSC
  // Coulomb collisions (DoUseCoulomb): the COULPARA tables of every species,
  // (COULE+COULI)(S,K,L) as cc[(s*NPA + l)*NE + k] and {ATA, GTA}(S,K,L) as
  // cag[(s*NPA + l)*NE + k]; COULEN's ghost factors per species, crel[s*5 +
  // ..] = GREL(S,1), GREL(S,2), SQRT((GREL1^2-1)/(GREL2^2-1)), GRZERO(S),
  // SQRT((GRZERO^2-1)/(GREL1^2-1)); NECR (NR,NT) in the reference's layout
  int coul;
  // WPADIF and FLCscatter: per species whether ram_run takes WPADIF at the
  // WPI positions (in place of WAVELO) and at the EMIC positions, and the
  // coefficient tables (F2's device layout; flc null: no FLCscatter)
  int pd_wpi[kMaxSpecies], pd_emic[kMaxSpecies];
  int sum_any;  // SumAny bits: the operators that some species takes
  const double *pdc[kMaxSpecies], *flc[kMaxSpecies];
  double *cc;
  double2 *cag;
  double *crel;
  const double *necr;
  double *ex64;   // [j] 2^(j/64), the table of the loss factors' exponential
  // CFL maxima of max(|C|,floor) over cells inside the magnetopause, as the
  // bit patterns of non-negative doubles (atomicMax order = double order):
  // [s][2+K] E, [s][2+NE+L] Mu (R's and P's: slots kSlotCflR, kSlotCflP)
  unsigned long long *cflmax;
  double *dtdrift;      // [s][4]
  // float reciprocals for exact small-integer division (fast_div)
  float rnt, rne, rp;   // 1/NT, 1/NE, 1/(NE*NPA)
  // row mapping of the forward plane kernels: thread n < plane_chunks*NE
  // owns K = n%NE of the rows of chunk n/NE (plane_chunks_for); the
  // threads above, in a block of any size, are idle
  int plane_chunks;
  int step_cells, step_apart;  // step_wave_cells, step_edges_apart of k_plane_step's shape
  int stepx_apart;             // step_edges_apart of SEQ_STEPX's
  int r_rows, p_rows;          // rows of k_r_rows and k_p_rows; 0: k_r, k_p (line_rows)
  // state
  double *f2;
  double *partials;  // [slot][s][maxblk]
  int maxblk;
  double *energy;    // [s][4]: SETRC, LSDR, LSCHA, LSATM
  // reverse mode of an ensemble (null otherwise): the problem's tape of
  // F2-sized slots, its adjoint lam, the adjoint of each step's FGEOS
  // ([step][NS,NT,NE,NPA]), and its flux-misfit points, weights
  // ([p][NPA]), targets and per-step losses ([step][p])
  double *tape, *lam, *bbar;
  const int *mpts;
  const double *mw, *mtarget;
  double *mloss;
  int mnpts;
};

// One unit of a launch: blocks [b0, b0+nb) of species s of problem tabs[tab];
// rows: the rows per thread of its kernel, where a launch has several.
struct Job {
  int tab, s, b0, nb, rows;
};
constexpr int kMixedRows = -1;  // LineShape, StepShape: each job of the launch by its own rows
// vmap entries: a virtual block's job and its block within the job
constexpr int kVmapShift = 16;
inline __host__ __device__ int vmap_entry(int job, int b) { return (job << kVmapShift) | b; }

// A launch over several units.  With vmap == nullptr the launch covers
// species s0, s0+1, .. of tabs[0], nb blocks each, species after species,
// or with ilv the species of each run of 8 blocks in turn (so the species'
// blocks of one plane land on one XCD, whose L2 then serves the plane's
// species-independent tables to all of them: workgroups go to the 8 XCDs
// in turn); otherwise vmap[vb] is the vmap_entry of virtual block vb.
// Blocks loop over virtual blocks with stride gridDim.x, so the grid may be
// smaller than nv.
// src/dst (sweep kernels): read F2 from src and write to dst (device layout
// of the whole problem) instead of updating tabs[..].f2 in place; null for in
// place.  ssl/dsl name them per problem instead (ensembles): n > 0 is slot
// n-1 of the problem's tape, dsl < 0 its own F2 written out of place, 0 not
// used.
struct Launch {
  const Tab *tabs;
  const Job *jobs;
  const int *vmap;
  int nv, nb, s0, ilv;
  const double *src;
  double *dst;
  int ssl, dsl;
  int bstep;  // reverse mode of an ensemble: the step whose FGEOS adjoint (Tab::bbar) DRIFTR's adjoint feeds
};

template <class T>
inline __host__ __device__ size_t f2_species_stride(const T &t) {
  return (size_t)t.nr * t.nt * t.npa * t.ne;
}

// the input and output F2 of a launch for problem t, and whether they differ
template <class T>
inline __host__ __device__ const double *launch_src(const Launch &L, const T &t) {
  if (L.ssl > 0) return t.tape + (size_t)(L.ssl - 1) * t.ns * f2_species_stride(t);
  return L.src ? L.src : t.f2;
}
template <class T>
inline __host__ __device__ double *launch_dst(const Launch &L, const T &t) {
  if (L.dsl > 0) return t.tape + (size_t)(L.dsl - 1) * t.ns * f2_species_stride(t);
  if (L.dsl < 0) return t.f2;
  return L.dst ? L.dst : t.f2;
}
inline __host__ __device__ bool out_of_place(const Launch &L) { return L.dsl != 0 || (L.dst && L.dst != L.src); }

// block counts of the kernels, per (problem, species)
template <class T>
inline __host__ __device__ int blocks_line_r(const T &t) {  // one thread per line: k_r, k_r_bwd
  return (t.nt * t.ne * t.npa + kLineThreads - 1) / kLineThreads;
}
template <class T>
inline __host__ __device__ int blocks_line_p(const T &t) {  // k_p, k_p_bwd
  return ((t.nr - 1) * t.ne * t.npa + kLineThreads - 1) / kLineThreads;
}
// The sweeps with a line's cells in registers (k_r_rows, k_p_rows): 64 lines
// of one J or I per block, line_chunks waves of `rows` cells.
inline __host__ __device__ int line_chunks(int n, int rows) { return (n + rows - 1) / rows; }
inline __host__ __device__ size_t line_lds_bytes(int chunks, int rows) {
  return (size_t)((4 * chunks + 2) * 64 + 16 + 6 * chunks * rows) * sizeof(double);
}
constexpr int kLineMaxChunks = 16;
// waves per SIMD that the registers leave room for, by rows
constexpr int line_simd_waves(int rows) { return rows <= 2 ? 8 : (rows <= 6 ? 5 : 4); }
template <class T>
inline __host__ __device__ int blocks_r(const T &t) {
  return t.r_rows ? t.nt * ((t.ne * t.npa + 63) / 64) : blocks_line_r(t);
}
template <class T>
inline __host__ __device__ int blocks_p(const T &t) {
  return t.p_rows ? (t.nr - 1) * ((t.ne * t.npa + 63) / 64) : blocks_line_p(t);
}
// out of place DRIFTP also copies the unswept I=1 rows
template <class T>
inline __host__ __device__ int blocks_p_copy(const T &t, bool chunks = true) {
  const int P = t.ne * t.npa;
  if (!t.p_rows || !chunks) return ((t.nr - 1) * P + t.nt * P + kLineThreads - 1) / kLineThreads;
  const int threads = 64 * line_chunks(t.nt, t.p_rows);
  return blocks_p(t) + (t.nt * P + threads - 1) / threads;
}
// blocks of k_ghost, per species
template <class T>
inline __host__ __device__ int ghost_blocks(const T &t) {
  return (t.ne * t.npa + kGhostPlanes - 1) / kGhostPlanes;
}
template <class T>
inline __host__ __device__ int blocks_kl(const T &t) { return (t.nr - 1) * t.nt; }

// LDS bytes of the azimuthal sweep: pl of a block's (I,L) pairs and pij of
// its I values
inline __host__ __device__ size_t azim_lds_bytes(int nt, int ne, int npa) {
  const int npair = (kLineThreads - 1) / ne + 2, ni = (kLineThreads - 1) / (ne * npa) + 2;
  return (size_t)(npair + ni) * nt * 4 * sizeof(double);
}
// LDS bytes of the radial sweep: the face terms of a block's lines, q1 of
// its (J,L) pairs, rij of its J values, rsi and the flags rij(I,NT).w
inline __host__ __device__ size_t radial_lds_bytes(int nr, int ne, int npa) {
  const int npair = (kLineThreads - 1) / ne + 2, nj = (kLineThreads - 1) / (ne * npa) + 2;
  return (size_t)(npair + 4 * nj + 3) * nr * sizeof(double);
}

// LDS bytes of the plane kernel
// LDS of the forward plane kernels; mu_slots: LDS slots per row of DRIFTMU's
// CFL maximum
inline __host__ __device__ size_t plane_lds_bytes(int ne, int npa, int mu_slots = kMuSpread) {
  const size_t P = (size_t)ne * npa;
  return (2 * P + 16 * (size_t)npa + 2 * (size_t)npa + 11 * (size_t)ne + 4 * (size_t)npa + 128 + 64 + 24 +
          2 * (size_t)npa + (size_t)ne + (size_t)mu_slots * npa) * sizeof(double);
}
// Chunks of rows of the forward plane kernels in blocks of T threads: one
// chunk of NE threads per floor(T/NE), at most NPA/2 so that every chunk
// holds two rows or more (the top row L=NPA then never opens a chunk:
// DRIFTMU sets it from the row below, which the same thread holds).  The
// NPA rows are shared out as evenly as they go, the first NPA % chunks
// chunks one row longer.  0 when T < NE.
inline __host__ __device__ int plane_chunks_for(int ne, int npa, int threads) {
  const int q = threads / ne;
  return q < npa / 2 ? q : npa / 2;
}
// the longest chunk's rows
inline __host__ __device__ int plane_max_rows(int npa, int chunks) { return (npa + chunks - 1) / chunks; }
// LDS of the forward plane kernels (PlaneFwd): NPA rows of NE+3 energy
// stencil slots, the K=1 column, T exchange slots, the per-L DRIFTE and
// DRIFTMU terms (16 NPA), HDNS and 1/FNHS (2 NPA), KT_N=11 per-K and LT_N=4
// per-L tables, 128 reduction slots, the 64-entry exp table, PC_N=24 plane
// scalars and the CFL slots (NE + kMuSpread*NPA).
inline __host__ __device__ size_t plane_fwd_lds_bytes(int ne, int npa, int threads) {
  return ((size_t)npa * (ne + 3) + (size_t)npa + (size_t)threads + 16 * (size_t)npa + 2 * (size_t)npa +
          11 * (size_t)ne + 4 * (size_t)npa + 128 + 64 + 24 + (size_t)ne + (size_t)kMuSpread * npa) *
         sizeof(double);
}
// Mapping and LDS of the fused step's plane kernel (k_plane_step).  Q =
// ceil(NPA/R) chunks of R rows of NE threads; a wave takes step_wave_cells
// of the Q*NE columns: 64 where no chunk straddles two waves, else 63, lane 0
// repeating the last column of the wave before.
constexpr size_t kLdsCu = 160 * 1024;  // gfx950
inline __host__ __device__ int step_chunks(int npa, int rows) { return (npa + rows - 1) / rows; }
inline __host__ __device__ int step_wave_cells(int ne) { return 64 % ne == 0 ? 64 : 63; }
inline __host__ __device__ int step_threads(int ne, int npa, int rows) {
  const int w = step_wave_cells(ne);
  return (step_chunks(npa, rows) * ne + w - 1) / w * 64;
}
constexpr int kStepSpread = 2;  // LDS slots per row of DRIFTMU's CFL maximum (by K mod 2)
constexpr int kStepSimdWaves = 4;  // waves per SIMD that the kernel's registers leave room for
// Its LDS in doubles: the plane's rows of NE+3 energy-stencil positions, the
// per-L terms (21 NPAP + 5), 10 per-K terms, the exponential's table, 112
// wave sums, the CFL slots; and 4*Q*NE doubles at the chunks' edges, in the
// rows' place (behind a further barrier) where they would cost a CU a block.
inline __host__ __device__ size_t step_lds_doubles(int ne, int npa, int rows) {
  const size_t q = step_chunks(npa, rows), npap = q * rows, plane = npap * (ne + 3), edges = 4 * q * ne;
  return (plane > edges ? plane : edges) + 1 + 21 * npap + 5 + 10 * (size_t)ne + 64 + 112 + ne +
         (size_t)kStepSpread * npa;
}
// Blocks a CU holds with `lds` bytes each: a block's waves go to the SIMDs in
// turn from the first, so a SIMD takes ceil(waves/4) of each.
inline __host__ __device__ int step_resident(size_t lds, int ne, int npa, int rows) {
  const int simd = (step_threads(ne, npa, rows) / 64 + 3) / 4;
  const int by_waves = kStepSimdWaves / simd, by_lds = (int)(kLdsCu / lds);
  return by_waves < by_lds ? by_waves : by_lds;
}
// The step's plane adjoint (k_plane_adj): a wave takes adj_wave_cells of the
// columns, the two lanes at either end repeating its neighbours'; LDS as the
// forward's with 7*Q*NE doubles at the chunks' edges, in the rows' place, and
// without sums and CFL slots.
inline __host__ __device__ int adj_wave_cells(int ne) { return 64 % ne == 0 ? 64 : 60; }
inline __host__ __device__ int adj_threads(int ne, int npa, int rows) {
  const int w = adj_wave_cells(ne);
  return (step_chunks(npa, rows) * ne + w - 1) / w * 64;
}
inline __host__ __device__ size_t adj_lds_bytes(int ne, int npa, int rows) {
  const size_t q = step_chunks(npa, rows), npap = q * rows, plane = npap * (ne + 3), edges = 7 * q * ne;
  return ((plane > edges ? plane : edges) + 1 + 21 * npap + 5 + 10 * (size_t)ne + 64) * sizeof(double);
}
// SEQ_STEPX's further LDS: wider sums, the per-row terms of the line solves
// and what they hand between chunks
inline __host__ __device__ size_t step_extra_bytes(int ne, int npa, int rows) {
  return (16 * (size_t)(kSumSlots - 7) + 1 + 6 * (size_t)step_chunks(npa, rows) * rows + 3 * (size_t)ne) *
         sizeof(double);
}
// x: SEQ_STEPX
inline __host__ __device__ bool step_edges_apart(int ne, int npa, int rows, bool x = false) {
  const size_t base = step_lds_doubles(ne, npa, rows) * 8 + (x ? step_extra_bytes(ne, npa, rows) : 0);
  const size_t edges = 4 * (size_t)step_chunks(npa, rows) * ne * 8;
  return step_resident(base + edges, ne, npa, rows) >= step_resident(base, ne, npa, rows);
}
inline __host__ __device__ size_t step_lds_bytes(int ne, int npa, int rows, bool x = false) {
  return step_lds_doubles(ne, npa, rows) * 8 + (x ? step_extra_bytes(ne, npa, rows) : 0) +
         (step_edges_apart(ne, npa, rows, x) ? 4 * (size_t)step_chunks(npa, rows) * ne * 8 : 0);
}
// The Coulomb operators' LDS after the forward plane kernels': per L the
// bounce-averaged density XNE, BASCNE, FNHS, BOUNHS, MU, 1/FNHS and 1/MU
// (7 NPA), and COULMU's RL recurrence of every column (NE*NPA).
inline __host__ __device__ size_t plane_coul_lds_bytes(int ne, int npa, int threads) {
  return plane_fwd_lds_bytes(ne, npa, threads) + (7 * (size_t)npa + (size_t)ne * npa) * sizeof(double);
}
// LDS of the pitch-angle line solve (k_pitch_diffusion): RK and RL of each
// of its 64 lines
constexpr int kPitchThreads = 64;
// the species of one k_pitch_diffusion launch and their coefficient tables
struct PitchJob {
  int n;
  int s[kMaxSpecies];
  const double *coef[kMaxSpecies];
};
inline __host__ __device__ size_t pitch_lds_bytes(int npa) { return (size_t)2 * npa * kPitchThreads * sizeof(double); }
// the adjoint kernels record no CFL maxima: their adjoint plane takes the
// place of the CFL slots (NE + mu_slots*NPA doubles)
inline __host__ __device__ size_t plane_bwd_lds_bytes(int ne, int npa) {
  return plane_lds_bytes(ne, npa, 0) - (size_t)ne * sizeof(double) + (size_t)ne * npa * sizeof(double);
}

}  // namespace ramgpu
