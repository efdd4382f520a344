// line_sweep.hip -- DRIFTR and DRIFTP (src/ModRamDrift.f90:139-191, 229-272)
// with a line's cells in registers.
//
// A block takes 64 lines of one J (DRIFTR) or one I (DRIFTP), one per lane, so
// that every load and store of a cell row is one run of 512 bytes; its waves
// take the line's chunks of R cells (R a template constant).  What crosses
// chunks goes through LDS: the old values of the three cells beside a chunk,
// and the flux of its upper face.  The face terms of (I,J) are the same for a
// whole wave; those with an L come with the cells, in one memory round trip.
//
// What bounds it: the chain of memory round trips before the first cell
// (descriptor, cells, ghosts), 6500 of a block's 10000 cycles at 63000 lines;
// the descriptor's fields are fetched in one trip, the ghosts' inputs with the
// cells, the (I,J) terms by the wave's lanes into LDS.  Which launches take it
// rather than one thread per line (k_r, k_p): line_rows.
#include <hip/hip_runtime.h>

#include "ctx.h"
#include "sweep_common.h"

namespace ramgpu {

namespace {

struct LineLds {
  double *H;    // per chunk: first, second and last row (64 lanes each), then the flux of the upper face
  double *red;  // 16: block reductions
  double *T;    // 6 per cell row: its face's terms of (I,J)
};
__device__ __forceinline__ LineLds line_lds(double *sm, int Q) {
  double *const red = sm + (4 * Q + 2) * 64;
  return {sm, red, red + 16};
}

// the block's maximum of m (>= 0) to its place *g, where k_finalize finds it:
// as an atomic maximum on one address per species the 1000 blocks of H+ at
// 20x25x35x72 queued for 5 us (DRIFTR 19.1 -> 14.4 us, DRIFTP 17.5 -> 12.5)
__device__ __forceinline__ void line_max(double m, double *red, int w, int lane, int Q, double *g) {
  for (int off = 32; off > 0; off >>= 1) m = fmax(m, __shfl_down(m, off, 64));
  if (lane == 0) red[w] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int x = 0; x < Q; ++x) m = fmax(m, red[x]);
    *g = m;
  }
}

// the barriers of a unit, for the waves of a mixed launch's block that its
// lines do not need
__device__ __forceinline__ void line_barriers(int n) {
  for (int x = 0; x < n; ++x) __syncthreads();
}

// MODE 0: sweep; 1: sweep and record the CFL maximum; 2: the last sweep of
// ram_run: also the SUMRC partial sum of src/ModRamRun.f90:246-255, then
// F2(:,:,NT)=F2(:,:,1) and the magnetopause mask (:186,197-201).  In mode 2
// the J=NT lines are not swept: the seam overwrites them with the lines J=1,
// whose threads store both.
// MIXED: the block may have more waves than the line has chunks.
template <int MODE, int R, bool MIXED>
__device__ __forceinline__ void r_rows_unit(const Launch &L, const CUnit &u, double *sm) {
  {
    CTab &t = *u.t;
    fetched(t.nr, t.nt, t.ne, t.npa, t.ns, t.rne, t.f2, t.tape, t.q1, t.p4, t.rij, t.rsi, t.betalim,
            t.fgeos, t.fnhs, t.bscale, t.conf1, t.conf2, (int)blockDim.x);
    const int s = u.s, NR = t.nr, NT = t.nt, NE = t.ne, P = NE * t.npa;
    const int G = (P + 63) >> 6, Q = MIXED ? line_chunks(NR, R) : blockDim.x >> 6;
    const int j = u.b / G, q0 = (u.b - j * G) * 64;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const LineLds d = line_lds(sm, Q);
    if (MODE == 2 && j == NT - 1) {
      if (threadIdx.x == 0) t.partials[((size_t)kSumRadial * t.ns + s) * t.maxblk + u.b] = 0.0;
      return;
    }
    if (MIXED && w >= Q) return line_barriers(MODE == 0 ? 2 : 3);
    const int i0 = w * R;
    const bool act = q0 + lane < P;
    const int q = min(q0 + lane, P - 1);
    const int l = fast_div(q, NE, t.rne), k = q - l * NE;
    const int di = NT * P;  // cells between I and I+1; a species has fewer than 2^31 bytes per I
    const size_t off = (size_t)s * f2_species_stride(t) + (size_t)j * P + q0;
    const gptr<const double> fl = as_global(launch_src(L, t) + off);
    const gptr<double> fo = as_global(launch_dst(L, t) + off);
    const unsigned qo = q - q0;
    double f[R], q1[R];
#pragma unroll
    for (int n = 0; n < R; ++n) f[n] = (fl + (size_t)min(i0 + n, NR - 1) * di)[qo];
    const gptr<const double> gq = as_global((const double *)t.q1 + j);
    const unsigned ql = (unsigned)(l * NR) * NT;
#pragma unroll
    for (int n = 0; n < R; ++n) q1[n] = gq[ql + (unsigned)(min(i0 + n, NR - 1) * NT)];
    const bool top = w == Q - 1;
    // FGEOS and FNHS(NR) of the line, for the ghosts F(NR+1), F(NR+2) of
    // inflow lines: loaded with the cells, whether or not the line is one
    double fg = 0.0, fh = 0.0, bs = 0.0;
    if (top) {
      bs = as_global((const double *)t.bscale)[s];
      fg = as_global(t.fgeos)[s + (size_t)t.ns * (j + (size_t)NT * (k + (size_t)NE * l))];
      fh = as_global(t.fnhs)[(NR - 1) + (size_t)(NR + 1) * (j + (size_t)NT * l)];
    }
    const double qn = gq[ql + (unsigned)((NR - 1) * NT)], qm = gq[ql + (unsigned)((NR - 2) * NT)];
    const double p4h = as_global((const double *)t.p4)[(unsigned)(s * NE + k)] * 0.5;
    // the chunk's terms of (I,J): {rij, rsi} of its rows, by the wave's lanes
    double *const T = d.T + 6 * i0;
    for (int e = lane; e < 6 * R; e += 64) {
      const int n = e / 6, x = e - 6 * n, i = min(i0 + n, NR - 1);
      const double *const p = x < 4 ? (const double *)t.rij + (unsigned)(i * NT + j) * 4 + x
                                    : (const double *)t.rsi + (unsigned)(2 * i + x - 4);
      T[e] = *as_global(p);
    }
    const double beta = t.betalim;
    // C(I,J,K,L) as c_radial_of: the factor 1/2 is exact wherever it stands
    auto courant = [&](const double *r, double q1v) __attribute__((always_inline)) {
      return r[0] + div_rn(div_rn(q1v * p4h, r[1], r[2]), r[4], r[5]);
    };
    double *const H = d.H + lane;
    H[(4 * w) * 64] = f[0];
    H[(4 * w + 1) * 64] = f[1];
    H[(4 * w + 2) * 64] = f[R - 1];
    // inflow: C(NR) < 0 (:156-169)
    bool in = false;
    double gh1 = 0.0, gh2 = 0.0, fgh = 0.0;
    if (top) {
      in = courant(d.T + 6 * (NR - 1), qn) < 0;
      // ghost_value's expressions
      const bool outside = d.T[6 * (NR - 1) + 3] == 1.0;
      fg = fg * bs;
      gh1 = (in && !outside) ? fg * t.conf1 * fh : 0.0;
      gh2 = (in && !outside) ? fg * t.conf2 * fh : 0.0;
      // F(NR+1) of face NR-1 when it is upwinded from outside: the line's
      // own ghost on inflow lines, else the one an earlier inflow line left
      fgh = gh1;
      if (!in && courant(d.T + 6 * (NR - 2), qm) < 0) fgh = stale_ghost(*(const Tab *)(unsigned long long)u.t, s, j, k, l);
    }
    __syncthreads();
    if (w == 0) in = courant(d.T + 6 * (NR - 1), qn) < 0;
    double fm = H[(w > 0 ? 4 * w - 2 : 0) * 64];  // F(I-1)
    double up0, up1;
    double cmax = 0.0, hprev = 0.0;
    // the faces above rows 0..R-1 and the cells they bound; twice the face
    // value and the flux, the factor 1/2 (exact) in the update
    auto sweep = [&](auto is_top) __attribute__((always_inline)) {
      constexpr bool TOP = decltype(is_top)::value;
      double f0 = f[0];
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const int i = i0 + n;
        const double f1 = n + 1 < R ? f[n + 1 < R ? n + 1 : 0] : up0;
        double f2 = n + 2 < R ? f[n + 2 < R ? n + 2 : 0] : (n + 2 == R ? up0 : up1);
        if (TOP) f2 = (i == NR - 2) ? fgh : f2;
        const double c = courant(T + 6 * n, q1[n]);
        if (MODE == 1) cmax = (T[6 * n + 3] == 0.0) ? fmax(cmax, fmax(fabs(c), 1E-10)) : cmax;
        const bool neg = c < 0;
        double u2 = face_value2(f0, f1, neg ? f1 : f0, neg ? f2 : fm, neg, c, beta);
        if (TOP) u2 = (i == NR - 1 && !in) ? 2.0 * f0 : u2;  // FBND(NR) = F(NR) on outflow lines
        if (n == 0) u2 = (w == 0) ? (in ? 2.0 * f1 : 0.0) : u2;  // FBND(1) = F(2) on inflow lines, 0 otherwise
        const double h = c * u2;
        fm = f0;
        const double v = fma(0.5, hprev, fma(-0.5, h, f0));
        f0 = f1;
        hprev = h;
        f[n] = row_done((n == 0 && w == 0) ? fm : v);  // cell 1 is not updated
      }
    };
    if (top) {
      // F(NR+1), F(NR+2) follow the line's last cell
#pragma unroll
      for (int n = 2; n < R; ++n) f[n] = (i0 + n == NR) ? gh1 : (i0 + n == NR + 1) ? gh2 : f[n];
      up0 = (i0 + R == NR) ? gh1 : gh2;
      up1 = gh2;
      sweep(Yes());
    } else {
      up0 = H[(4 * w + 4) * 64];
      up1 = H[(4 * w + 5) * 64];
      sweep(No());
    }
    if (!top) H[(4 * w + 3) * 64] = hprev;
    __syncthreads();
    if (w > 0) f[0] = fma(0.5, H[(4 * w - 1) * 64], f[0]);
    double sum = 0.0;
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const int i = i0 + n;
      const bool cell1 = n == 0 && w == 0;
      if (i >= NR) break;
      double v = f[n];
      if (!cell1 && v < 0) v = 1E-15;
      if (MODE == 2) {
        if (!cell1) sum += v;
        if (act) {
          (fo + (size_t)i * di)[qo] = (T[6 * n + 3] == 1.0) ? 1e-31 : v;
          if (j == 0) {
            const double mgs = as_const((const double *)t.rij)[((size_t)i * NT + NT - 1) * 4 + 3];
            (fo + (size_t)i * di + (size_t)(NT - 1) * P)[qo] = (mgs == 1.0) ? 1e-31 : v;
          }
        }
      } else if (act) {
        (fo + (size_t)i * di)[qo] = v;
      }
    }
    if (MODE == 1) line_max(cmax, d.red, w, lane, Q, t.partials + ((size_t)kSlotCflR * t.ns + s) * t.maxblk + u.b);
    if (MODE == 2) {
      // EKEV*WE*WMU is the line's
      double a = 0.0;
      if (act && k >= 1 && l >= 1 && j <= NT - 2) a = sum * (t.ekev[k] * t.we[k] * t.wmu[l]);
      a = wave_sum(a);
      if (lane == 63) d.red[w] = a;
      __syncthreads();
      if (threadIdx.x == 0) {
        double v = 0.0;
        for (int x = 0; x < Q; ++x) v += d.red[x];
        t.partials[((size_t)kSumRadial * t.ns + s) * t.maxblk + u.b] = v;
      }
    }
  }
}

// DRIFTP: rings (I>=2,K,L), periodic in J: F(NT+1) = F(2), F(NT+2) = F(3),
// but for the face J=NT-1 upwinded from above, whose N-1 is 1 (:250-251); the
// flux of face NT is also face 1's (:261-262); F2(I,1) = F2(I,NT) (:272).
// MODE 0: sweep; 1: sweep and record the CFL maximum.
template <int MODE, int R, bool MIXED>
__device__ __forceinline__ void p_rows_unit(const Launch &L, const CUnit &u, double *sm) {
  {
    CTab &t = *u.t;
    fetched(t.nr, t.nt, t.ne, t.npa, t.ns, t.rne, t.f2, t.tape, t.pl, t.p2, t.pij, t.betalim, t.omet,
            (int)blockDim.x);
    const int s = u.s, NR = t.nr, NT = t.nt, NE = t.ne, P = NE * t.npa;
    const int G = (P + 63) >> 6, Q = MIXED ? line_chunks(NT, R) : blockDim.x >> 6;
    const size_t so = (size_t)s * f2_species_stride(t);
    if (u.b >= (NR - 1) * G) {  // out of place: the unswept I=1 rows, a cell per thread
      const int T = 64 * Q, x = (u.b - (NR - 1) * G) * T + threadIdx.x;
      if ((!MIXED || (int)threadIdx.x < T) && x < NT * P) as_global(launch_dst(L, t) + so)[x] = as_global(launch_src(L, t) + so)[x];
      return;
    }
    const int i1 = u.b / G, q0 = (u.b - i1 * G) * 64, i = i1 + 1;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (MIXED && w >= Q) return line_barriers(MODE == 0 ? 2 : 3);
    const LineLds d = line_lds(sm, Q);
    const int j0 = w * R;
    const bool act = q0 + lane < P;
    const int q = min(q0 + lane, P - 1);
    const int l = fast_div(q, NE, t.rne), k = q - l * NE;
    const size_t off = so + (size_t)i * NT * P + q0;
    const gptr<const double> fl = as_global(launch_src(L, t) + off);
    const gptr<double> fo = as_global(launch_dst(L, t) + off);
    const unsigned qo = q - q0;
    double f[R];
#pragma unroll
    for (int n = 0; n < R; ++n) f[n] = (fl + (size_t)min(j0 + n, NT - 1) * P)[qo];
    typedef double d2 __attribute__((ext_vector_type(2)));
    const gptr<const d2> gp = (gptr<const d2>)(const double *)t.pl + (size_t)i * NT * 2;
    const unsigned pl0 = (unsigned)(l * NR) * NT * 2;
    d2 ga[R];
    double gr[R];
#pragma unroll
    for (int n = 0; n < R; ++n) {
      const unsigned e = pl0 + 2 * min(j0 + n, NT - 1);
      ga[n] = gp[e];
      gr[n] = ((gptr<const double>)(gp + e + 1))[0];
    }
    const double p2k = as_global((const double *)t.p2)[(unsigned)((s * NR + i) * NE + k)];
    const double beta = t.betalim, omet = t.omet;
    // the chunk's terms of (I,J): pij of its rows and the flags MGNP(I,J), of
    // pl at L=1, by the wave's lanes
    double *const T = d.T + 6 * j0;
    for (int e = lane; e < 6 * R; e += 64) {
      const int n = e / 6, x = e - 6 * n;
      const unsigned o = (unsigned)(i * NT + min(j0 + n, NT - 1)) * 4;
      T[e] = *as_global(x < 4 ? (const double *)t.pij + o + x : (const double *)t.pl + o + 3);
    }
    double *const H = d.H + lane;
    double *const F3 = H + 4 * Q * 64, *const GN = F3 + 64;
    H[(4 * w) * 64] = f[0];
    H[(4 * w + 1) * 64] = f[1];
    H[(4 * w + 2) * 64] = f[R - 1];
    if (R >= 3 ? w == 0 : w == 1) F3[0] = f[R >= 3 ? 2 : 0];
    __syncthreads();
    const bool top = w == Q - 1;
    double fm = H[(w > 0 ? 4 * w - 2 : 0) * 64];  // F(J-1)
    double up0, up1;
    double cmax = 0.0, hprev = 0.0;
    auto sweep = [&](auto is_top) __attribute__((always_inline)) {
      constexpr bool TOP = decltype(is_top)::value;
      const double F1 = TOP ? H[0] : 0.0;
      double f0 = f[0], hn = 0.0;
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const int j = j0 + n;
        const double f1 = n + 1 < R ? f[n + 1 < R ? n + 1 : 0] : up0;
        const double f2 = n + 2 < R ? f[n + 2 < R ? n + 2 : 0] : (n + 2 == R ? up0 : up1);
        // Courant number of face J (:236-239)
        const double *a = T + 6 * n;
        const double uu = div_rn(p2k * ga[n].x, ga[n].y, gr[n]);
        const double c = div_rn(a[0] - uu - a[1], a[2], a[3]) + omet;
        const bool cell1 = n == 0 && w == 0;  // J=1: no face, no update of its own
        if (MODE == 1 && !cell1) cmax = (a[4] == 0.0) ? fmax(cmax, fmax(fabs(c), 1E-10)) : cmax;
        const bool neg = c < 0;
        const double p = neg ? ((TOP && j == NT - 2) ? F1 : f1) : f0;
        const double h = c * face_value2(f0, f1, p, neg ? f2 : fm, neg, c, beta);
        fm = f0;
        const double v = fma(0.5, hprev, fma(-0.5, h, f0));
        f0 = f1;
        hprev = cell1 ? 0.0 : h;
        if (TOP) hn = (j == NT - 1) ? h : hn;
        f[n] = row_done(v);
      }
      if (TOP) GN[0] = hn;
    };
    if (top) {
      // F(NT+1) = F(2), F(NT+2) = F(3) follow the ring's last cell
      const double f2o = H[64], f3 = F3[0];
#pragma unroll
      for (int n = 2; n < R; ++n) f[n] = (j0 + n == NT) ? f2o : (j0 + n == NT + 1) ? f3 : f[n];
      up0 = (j0 + R == NT) ? f2o : f3;
      up1 = f3;
      sweep(Yes());
    } else {
      up0 = H[(4 * w + 4) * 64];
      up1 = H[(4 * w + 5) * 64];
      sweep(No());
    }
    if (!top) H[(4 * w + 3) * 64] = hprev;
    __syncthreads();
    if (w > 0) f[0] = fma(0.5, H[(4 * w - 1) * 64], f[0]);
    else f[1] = fma(0.5, GN[0], f[1]);
    if (act)
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const int j = j0 + n;
        if (j >= NT) break;
        if (n == 0 && w == 0) continue;
        const double v = (f[n] < 0) ? 1E-15 : f[n];
        (fo + (size_t)j * P)[qo] = v;
        if (j == NT - 1) fo[qo] = v;
      }
    if (MODE == 1) line_max(cmax, d.red, w, lane, Q, t.partials + ((size_t)kSlotCflP * t.ns + s) * t.maxblk + u.b);
  }
}

}  // namespace

template <int MODE, int R>
__global__ void __launch_bounds__(1024, line_simd_waves(R)) k_r_rows(Launch L) {
  extern __shared__ double sm[];
  for (int vb = blockIdx.x; vb < L.nv; vb += gridDim.x) r_rows_unit<MODE, R, false>(L, const_unit(L, vb), sm);
}
template <int MODE, int R>
__global__ void __launch_bounds__(1024, line_simd_waves(R)) k_p_rows(Launch L) {
  extern __shared__ double sm[];
  for (int vb = blockIdx.x; vb < L.nv; vb += gridDim.x) p_rows_unit<MODE, R, false>(L, const_unit(L, vb), sm);
}

// Cells per thread the line kernels are built for: more of them spill.  Of these
// k_r_rows and k_p_rows at 2 cells and k_p_rows at 6 spill up to 7 registers
// (8 to 28 bytes a lane), being held to the waves of line_simd_waves.
#define LINE_ROWS(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8)

// An ensemble's members in one launch, each with the rows it has alone.
template <int MODE>
__global__ void __launch_bounds__(1024, line_simd_waves(8)) k_r_mixed(Launch L) {
  extern __shared__ double sm[];
  for (int vb = blockIdx.x; vb < L.nv; vb += gridDim.x) {
    const CUnit u = const_unit(L, vb);
    switch (u.rows) {
#define ROWS(r) \
  case r: r_rows_unit<MODE, r, true>(L, u, sm); break;
      LINE_ROWS(ROWS)
#undef ROWS
    }
    if (L.nv > (int)gridDim.x) __syncthreads();  // the next unit may lay its LDS out otherwise
  }
}
template <int MODE>
__global__ void __launch_bounds__(1024, line_simd_waves(8)) k_p_mixed(Launch L) {
  extern __shared__ double sm[];
  for (int vb = blockIdx.x; vb < L.nv; vb += gridDim.x) {
    const CUnit u = const_unit(L, vb);
    switch (u.rows) {
#define ROWS(r) \
  case r: p_rows_unit<MODE, r, true>(L, u, sm); break;
      LINE_ROWS(ROWS)
#undef ROWS
    }
    if (L.nv > (int)gridDim.x) __syncthreads();  // the next unit may lay its LDS out otherwise
  }
}

}  // namespace ramgpu

using namespace ramgpu;

namespace ramgpu_host {

// Cells per thread of k_r_rows or k_p_rows for lines of n cells, 0 for one
// thread per line (k_r, k_p), of which a problem has `lines` in all.
// One thread per line walks 20 to 50 dependent steps; with no more than a wave
// of lines per SIMD (line_rows_max) those steps are the sweep's time and cutting
// the line is faster.  Beyond, waves cover for one another and the set-up that
// every chunk repeats costs more (MI355X, by events, us of DRIFTR and DRIFTP by
// one thread per line / by chunks: 2 species of 10x13x11x17 13.7, 10.8 / 8.9,
// 7.4; 20x25x35x72 1 species 18.9, 17.6 / 16.5, 15.6; 4 species 30.4, 24.0 /
// 34.0, 32.1; a step of 1 species 117 / 106, of 2 147 / 155).
// Up to four chunks as long as 8 cells reach; a chunk count from 3 to 5 makes
// no difference there.  The last chunk needs two cells (n mod R = 1 is left out).
int line_rows(int n, long lines, int ncu) {
  if (lines > line_rows_max(ncu)) return 0;
  for (int q : {4, kLineMaxChunks})
    for (int r = 2; r <= 8; ++r)
      if (n % r != 1 && line_chunks(n, r) <= q) return r;
  return 0;
}

// Block and LDS of a context's DRIFTR and DRIFTP.
LineShape r_shape(const ramgpu_ctx *c) {
  if (c->t.r_rows == 0) return {0, kLineThreads, radial_lds_bytes(c->nr, c->ne, c->npa)};
  const int Q = line_chunks(c->nr, c->t.r_rows);
  return {c->t.r_rows, 64 * Q, line_lds_bytes(Q, c->t.r_rows)};
}
LineShape p_shape(const ramgpu_ctx *c, bool chunks) {
  if (c->t.p_rows == 0 || !chunks) return {0, kLineThreads, azim_lds_bytes(c->nt, c->ne, c->npa)};
  const int Q = line_chunks(c->nt, c->t.p_rows);
  return {c->t.p_rows, 64 * Q, line_lds_bytes(Q, c->t.p_rows)};
}

void launch_r(int mode, LineShape sh, dim3 grid, hipStream_t st, const Launch &L) {
  const dim3 blk(sh.threads);
  const size_t lds = sh.lds;
  switch (sh.rows) {
#define ROWS(r)                                                                      \
  case r:                                                                            \
    if (mode == 0) hipLaunchKernelGGL((k_r_rows<0, r>), grid, blk, lds, st, L);      \
    else if (mode == 1) hipLaunchKernelGGL((k_r_rows<1, r>), grid, blk, lds, st, L); \
    else hipLaunchKernelGGL((k_r_rows<2, r>), grid, blk, lds, st, L);                \
    break;
    LINE_ROWS(ROWS)
#undef ROWS
    case kMixedRows:
      if (mode == 0) hipLaunchKernelGGL(k_r_mixed<0>, grid, blk, lds, st, L);
      else if (mode == 1) hipLaunchKernelGGL(k_r_mixed<1>, grid, blk, lds, st, L);
      else hipLaunchKernelGGL(k_r_mixed<2>, grid, blk, lds, st, L);
      break;
    default:
      if (mode == 0) hipLaunchKernelGGL(k_r<0>, grid, blk, lds, st, L);
      else if (mode == 1) hipLaunchKernelGGL(k_r<1>, grid, blk, lds, st, L);
      else hipLaunchKernelGGL(k_r<2>, grid, blk, lds, st, L);
  }
}

void launch_p(int mode, LineShape sh, dim3 grid, hipStream_t st, const Launch &L) {
  const dim3 blk(sh.threads);
  const size_t lds = sh.lds;
  switch (sh.rows) {
#define ROWS(r)                                                                 \
  case r:                                                                       \
    if (mode == 0) hipLaunchKernelGGL((k_p_rows<0, r>), grid, blk, lds, st, L); \
    else hipLaunchKernelGGL((k_p_rows<1, r>), grid, blk, lds, st, L);           \
    break;
    LINE_ROWS(ROWS)
#undef ROWS
    case kMixedRows:
      if (mode == 0) hipLaunchKernelGGL(k_p_mixed<0>, grid, blk, lds, st, L);
      else hipLaunchKernelGGL(k_p_mixed<1>, grid, blk, lds, st, L);
      break;
    default:
      if (mode == 0) hipLaunchKernelGGL(k_p<0>, grid, blk, lds, st, L);
      else hipLaunchKernelGGL(k_p<1>, grid, blk, lds, st, L);
  }
}

}  // namespace ramgpu_host
