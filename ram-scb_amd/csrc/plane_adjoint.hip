// plane_adjoint.hip -- the adjoint of the middle of the split step (DRIFTE,
// DRIFTMU, the loss chain, DRIFTMU, DRIFTE; plane_step.hip), on one (K,L)
// plane per block with the plane's adjoint in registers.
//
// The mapping is the forward kernel's: column c < Q*NE of a block's threads is
// column K = c mod NE of the R consecutive rows of chunk q = c/NE.  A face
// sends partials to the cells K-1 .. K+2 of its row (L-1 .. L+2 of its
// column); along K they reach their cells by wavefront shifts, along L within
// the thread, and across chunks through LDS.  A wave's two lanes at either end
// repeat the neighbouring waves' columns (where no chunk straddles waves, none
// do), so that every owned lane has its face's weights and its four partials
// within the wave.
//
// What bounds it: VALU issue.  The kernel that this one replaces kept x and
// the adjoint in LDS and let the faces add to their cells there, in four
// passes with a barrier each per sweep.  Launch of 475 planes of 35x72 (H+ on
// 20x25): 71 -> 44 us; an ensemble's 3 members up to 18x25x41x60, 2 species:
// 225 -> 129.
#include <hip/hip_runtime.h>

#include "ctx.h"
#include "sweep_common.h"

namespace ramgpu {

namespace {
// the value of v in lane+1 (lane 63: 0)
__device__ __forceinline__ double from_lane_above0(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), 0x130 /* wave_shl:1 */, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x130, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
}  // namespace

// x0: tape slot 0; slots 0..4 hold the inputs of the five phases and slot 7
// the drift phases' clamp decisions (k_plane_step<SEQ_TAPE>).
// MIXED: the block may have more threads than the plane needs (adj_threads).
template <int R, bool MIXED>
__device__ __forceinline__ void plane_adj_unit(const Launch &L, const double *xin, double *adj, const CUnit &u, double *sm) {
  {
    CTab *const tp = u.t;
#define t (*tp)
    fetched(t.ns, t.nr, t.nt, t.ne, t.npa, t.rnt, t.rne, t.f2, t.tape, t.lam, t.kle, t.klm, t.kll, t.lt4, t.kt, t.edot,
            t.latl, t.ex64, t.kij);
    const int NE = t.ne, NPA = t.npa, NT = t.nt, NR = t.nr;
    const int s = u.s, i = 1 + fast_div(u.b, NT, t.rnt), j = u.b - (i - 1) * NT;  // I = i+1 >= 2
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int Q = (NPA + R - 1) / R, NPAP = Q * R, S = NE + 3, ncol = Q * NE;
    const size_t ij = (size_t)i * NT + j;
    const size_t po = (size_t)s * f2_species_stride(t) + ij * ((size_t)NE * NPA);
    const size_t ns = (size_t)t.ns * f2_species_stride(t);
    const double *const x0 = (xin ? xin : launch_src(L, t)) + po;
    double *const ga = (adj ? adj : t.lam) + po;
    const unsigned char *const cb0 = reinterpret_cast<const unsigned char *>((xin ? xin : launch_src(L, t)) + 7 * ns) + po;
    // LDS (adj_lds_bytes)
    double *const F = sm;  // NPAP rows of NE+3 energy-stencil positions; in its place the chunks' edges, 7*ncol
    double *const cf = F + (max(NPAP * S, 7 * ncol) + 1) / 2 * 2;
    double *const cm = cf + 8 * NPAP;
    double *const cl = cm + 8 * NPAP;
    double *const lt = cl + (NPAP + 1) / 2 * 2;
    double *const kt = lt + 4 * (NPAP + 1);
    double *const ex = kt + (SKT_N + 2) * NE;

    const int W = adj_wave_cells(NE), halo = (64 - W) / 2, c_raw = wv * W + lane - halo;
    const int T = MIXED ? (ncol + W - 1) / W * 64 : (int)blockDim.x;
    if (MIXED && tid >= T) {  // whole waves: the unit's barriers
      for (int x = 0; x < (halo ? 10 : 8); ++x) __syncthreads();
      return;
    }
    const bool own = c_raw >= 0 && c_raw < ncol && lane >= halo && lane < halo + W;
    const int c_ = min(max(c_raw, 0), ncol - 1);
    const int q_ = fast_div(c_, NE, t.rne), k_ = c_ - q_ * NE;
#define THREAD_CELLS                                  \
  const int q = fresh(q_), k = fresh(k_), l0 = q * R; \
  (void)k; (void)l0
    // cells of this thread's column, rows past NPA repeating the top row
    auto load = [&](const double *p, double (&v)[R]) __attribute__((always_inline)) {
      THREAD_CELLS;
      const gptr<const double> g = as_global(p);
#pragma unroll
      for (int n = 0; n < R; ++n) v[n] = g[(unsigned)(min(l0 + n, NPA - 1) * NE + k)];
    };
    double y[R], x[R];
    load(ga, y);
    load(x0 + 4 * ns, x);
    {
      typedef double d2 __attribute__((ext_vector_type(2)));
      const gptr<const d2> g0 = (gptr<const d2>)(t.kle + ij * 8 * NPA), g1 = (gptr<const d2>)(t.klm + ij * 8 * NPA),
                           g3 = (gptr<const d2>)t.lt4;
      const gptr<const double> g2 = as_global((const double *)(t.kll + ij * NPA));  // HDNS, 1/FNHS
      const gptr<const double> gk = as_global(t.kt + (size_t)s * SKT_N * NE);
      const gptr<const double> ge = as_global(t.edot + ((size_t)s * NR + i) * NE), gl = as_global(t.latl + ((size_t)s * NR + i) * NE),
                               gx = as_global(t.ex64);
      const int n1 = 4 * NPA, n3 = 2 * NPA, nk = SKT_N * NE;
      d2 *const a0 = (d2 *)cf, *const a1 = (d2 *)cm, *const a3 = (d2 *)lt;
      // rows past NPA: zero terms, so that their faces carry nothing
#pragma unroll 2
      for (int e = tid; e < 4 * NPAP; e += T) {
        const bool in = e < n1;
        const d2 z = {0.0, 0.0}, v0 = in ? g0[(unsigned)e] : z, v1 = in ? g1[(unsigned)e] : z;
        a0[e] = v0;
        a1[e] = v1;
      }
      for (int e = tid; e < 2 * (NPAP + 1); e += T) a3[e] = e < n3 ? g3[(unsigned)e] : d2{0.0, 0.0};
      for (int e = tid; e < NPAP; e += T) cl[e] = e < NPA ? g2[(unsigned)(2 * e)] : 0.0;
      for (int e = tid; e < nk; e += T) kt[e] = gk[(unsigned)e];
      for (int e = tid; e < NE; e += T) {
        kt[nk + e] = ge[(unsigned)e];
        kt[nk + NE + e] = gl[(unsigned)e];
      }
      if (tid < 64) ex[tid] = gx[(unsigned)tid];
    }
#define PLANE_SCALARS                                                                                    \
  CTab &tt = *fresh_uniform(tp);                                                                         \
  const cptr<double> kij = as_const((const double *)tt.kij) + ij * 8;                                    \
  const double rlz = as_const(tt.rlz)[i], rrlz = as_const((const double *)tt.rrlz)[i], beta = tt.betalim; \
  const double bij = kij[KIJ_BIJ], rbij = kij[KIJ_RBIJ]

    // x's rows with DRIFTE's ghosts into LDS, as the forward's rows_out
    auto rows_out = [&]() __attribute__((always_inline)) {
      if (own) {
        THREAD_CELLS;
        double *const Frow = F + l0 * S + k;
        if (k >= 1) {
#pragma unroll
          for (int n = 0; n < R; ++n) Frow[n * S + 1] = x[n];
        }
        if (k == 1) {
          const cptr<double> rel = as_const((const double *)fresh_uniform(tp)->rel) + s * 8;
          const double r0 = rel[0], r1 = rel[1], r2 = rel[2], r3 = rel[3], r4 = rel[4], rr1 = rel[5], rr0 = rel[6];
#pragma unroll
          for (int n = 0; n < R; ++n) {
            const double g1 = div_rn(x[n] * r0, r1, rr1) * r2;
            Frow[n * S] = g1;
            Frow[n * S - 1] = div_rn(g1 * r3, r0, rr0) * r4;
          }
        }
        if (k == NE - 1) {
#pragma unroll
          for (int n = 0; n < R; ++n) Frow[n * S + 2] = Frow[n * S + 3] = 0.0;
        }
      }
      __syncthreads();
    };

    // DRIFTE's adjoint: w, the output adjoint of the updated, unclamped cells
    // (K=1 is not updated), weighs face K by -C/WE(K) and face K-1 by C/WE(K)
    auto adj_e = [&](const unsigned char *cb) __attribute__((always_inline)) {
      THREAD_CELLS;
      PLANE_SCALARS;
      const double *const Frow = F + l0 * S + k;
      const double drd1 = kij[KIJ_DRD1], dpd1 = kij[KIJ_DPD1];
      const cptr<double> rel = as_const((const double *)tt.rel) + s * 8;
      const double dg1 = rel[0] / rel[1] * rel[2], dg0 = dg1 * rel[3] / rel[0] * rel[4];  // dF(1)/dF(2), dF(0)/dF(2)
      const double *const kp = kt + k;
      const double ekp = kp[SKT_EKPQ * NE], edot = kp[SKT_N * NE];
      const double de = kp[SKT_DE * NE], rde = kp[SKT_RDE * NE];
      const double we = kp[SKT_WE * NE], rwe = kp[SKT_RWE * NE];
      const bool top = k + 1 >= NE;
      const double we1 = top ? 1.0 : kp[SKT_WE * NE + 1], rwe1 = top ? 1.0 : kp[SKT_RWE * NE + 1];
      unsigned clamped = 0;
      const gptr<const unsigned char> gc = as_global(cb);
#pragma unroll
      for (int n = 0; n < R; ++n) clamped |= (gc[(unsigned)(min(l0 + n, NPA - 1) * NE + k)] ? 1u : 0u) << n;
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const double *p = Frow + n * S;
        const double ce = c_energy(cf + 8 * (l0 + n), ekp, edot, drd1, dpd1, bij, rbij, rlz, rrlz);
        const bool neg = ce < 0;
        const double f0 = p[1], fp1 = p[2], a = p[neg ? 3 : 0];
        const FaceD D = face_d(f0, fp1, neg ? a : f0, neg ? fp1 : a, ce, div_rn(ce, de, rde), beta);
        const double pass = (k >= 1 && (clamped >> n & 1)) ? 0.0 : y[n];
        const double w = k >= 1 ? pass : 0.0;
        const double wup = from_lane_above0(w);
        const double b = (top ? 0.0 : div_rn(ce, we1, rwe1) * wup) - div_rn(ce, we, rwe) * w;
        // partials to cells K-1, K, K+1, K+2
        double pm = (neg ? 0.0 : D.dm) * b, p0 = (neg ? D.d0 : D.d0 + D.dn) * b;
        double p1 = (neg ? D.d1 + D.dm : D.d1) * b;
        const double p2 = (neg ? D.dn : 0.0) * b;
        if (k <= 1) {  // the ghosts F(0), F(1) are multiples of F(2)
          if (k == 0) {
            p1 = p1 + p0 * dg1 + pm * dg0;
            p0 = 0.0;
          } else {
            p0 = p0 + pm * dg1;
          }
          pm = 0.0;
        }
        double up = from_lane_below0(p2);
        up = p1 + (k >= 1 ? up : 0.0);
        up = from_lane_below0(up);
        const double dn = from_lane_above0(pm);
        y[n] = row_done(((pass + p0) + (k >= 1 ? up : 0.0)) + (top ? 0.0 : dn));
      }
    };

    // DRIFTMU's adjoint: updated cells L=2..NPA-1; the output F2(NPA) is
    // F2(NPA-1)*FNHS(NPA)*MU(NPA)/FNHS(NPA-1)/MU(NPA-1), so its adjoint joins
    // cell NPA-1's; the input F(NPA) only feeds FBND(NPA-1) = F(NPA) and
    // stencils; F(1) = F(2) for the stencil
    auto adj_mu = [&](const unsigned char *cb) __attribute__((always_inline)) {
      THREAD_CELLS;
      PLANE_SCALARS;
      double *const H = F + q * NE + k;
      unsigned clamped = 0;
      const gptr<const unsigned char> gc = as_global(cb);
#pragma unroll
      for (int n = 0; n < R; ++n) clamped |= (gc[(unsigned)(min(l0 + n, NPA - 1) * NE + k)] ? 1u : 0u) << n;
      if (l0 + R >= NPA) {
        const cptr<double> fh = as_const(tt.fnhs) + i + (size_t)(NR + 1) * (j + (size_t)NT * (NPA - 2));
        const cptr<double> mu = as_const(tt.mu) + NPA - 2;
        const double ratio = fh[(size_t)(NR + 1) * NT] * mu[1] / fh[0] / mu[0];
#pragma unroll
        for (int n = 0; n < R; ++n)
          if (l0 + n == NPA - 2) y[n] = y[n] + ratio * y[n + 1 < R ? n + 1 : n];
      }
      // y: now w, the weights of the updated cells; row 1's adjoint passes
      const double pass1 = y[0];
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const bool upd = !(n == 0 && l0 == 0) && l0 + n <= NPA - 2;
        y[n] = row_done((!upd || (clamped >> n & 1)) ? 0.0 : y[n]);
      }
      if (own) {
        H[0] = x[0];
        H[ncol] = x[1];
        H[2 * ncol] = x[R - 1];
        H[3 * ncol] = y[0];
      }
      __syncthreads();
      const double drm1 = kij[KIJ_DRM1], dpm1 = kij[KIJ_DPM1], db2 = kij[KIJ_DB2];
      const double mkp = kt[SKT_MKPQ * NE + k];
      double fm = H[2 * ncol - (q > 0 ? NE : 0)];
      const int cu = (q + 1 < Q) ? NE : 0;
      const double up0 = H[cu], up1 = H[ncol + cu], wup = (q + 1 < Q) ? H[3 * ncol + NE] : 0.0;
      const double *const lr = lt + 4 * l0, *const cmr = cm + 8 * l0;
      double e0 = 0.0, e1 = 0.0, below = 0.0;  // partials to the next two rows, and to the row below the chunk
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const int l = l0 + n;
        const bool row1 = n == 0 && l0 == 0, face = !row1 && l <= NPA - 2;
        const double f0 = x[n], f1 = n + 1 < R ? x[n + 1 < R ? n + 1 : 0] : up0;
        const double f2 = n + 2 < R ? x[n + 2 < R ? n + 2 : 0] : (n + 2 == R ? up0 : up1);
        const double w = y[n], w1 = n + 1 < R ? y[n + 1 < R ? n + 1 : 0] : wup;
        const double c = c_mu(cmr + 8 * n, mkp, drm1, dpm1, db2, bij, rbij, rlz, rrlz);
        const bool neg = c < 0, two = n == 1 && l0 == 0;
        const double fl = two ? f0 : fm;  // F(1) = F(2)
        const FaceD D = face_d(f0, f1, neg ? f2 : f0, neg ? f1 : fl, c, div_rn(c, lr[4 * n], lr[4 * n + 1]), beta);
        // C/WMU(L), C/WMU(L+1); the top rows' weights are 0
        double b = div_rn(c, lr[4 * n + 6], lr[4 * n + 7]) * w1 - div_rn(c, lr[4 * n + 2], lr[4 * n + 3]) * w;
        b = face ? b : 0.0;
        double pm = (neg ? 0.0 : D.dm) * b, p0 = (neg ? D.d0 : D.d0 + D.dn) * b;
        double p1 = (neg ? D.d1 + D.dm : D.d1) * b, p2 = (neg ? D.dn : 0.0) * b;
        if (two) {
          p0 += pm;
          pm = 0.0;
        }
        if (l == NPA - 2) {  // FBND(NPA-1) = F(NPA)
          pm = p0 = p2 = 0.0;
          p1 = b;
        }
        if (n == 0) below = pm;
        else y[n > 0 ? n - 1 : 0] = row_done(y[n > 0 ? n - 1 : 0] + pm);
        y[n] = row_done(((row1 ? pass1 : w) + p0) + e0);
        e0 = e1 + p1;
        e1 = p2;
        fm = f0;
      }
      if (own) {  // for the chunks above and below
        H[4 * ncol] = e0;
        H[5 * ncol] = e1;
        H[6 * ncol] = below;
      }
      __syncthreads();
      if (q > 0) {
        y[0] = y[0] + H[4 * ncol - NE];
        y[1] = y[1] + H[5 * ncol - NE];
      }
      if (q + 1 < Q) y[R - 1] = y[R - 1] + H[6 * ncol + NE];
    };

    rows_out();
    adj_e(cb0 + 3 * ns);  // E2
    load(x0 + 3 * ns, x);
    if (halo) {  // the repeated columns' adjoint, from their owners
      __syncthreads();  // the energy stencil is read
      THREAD_CELLS;
      double *const Y = F + q * NE + k;
      if (own && (lane < 2 * halo || lane >= W)) {
#pragma unroll
        for (int n = 0; n < R; ++n) Y[n * ncol] = y[n];
      }
      __syncthreads();
      if (!own) {
#pragma unroll
        for (int n = 0; n < R; ++n) y[n] = Y[n * ncol];
      }
    }
    __syncthreads();
    adj_mu(cb0 + 2 * ns);  // MU2
    load(x0 + ns, x);
    {  // the chain WAVELO, CEX, ATMOL, ATMOL, CEX, WAVELO (plane_step.hip), reversed
      THREAD_CELLS;
      CTab &tt = *fresh_uniform(tp);
      const bool cex = tt.cex[s] != 0;
      const int upa = as_const(tt.upa)[i];
      const double sigv = kt[SKT_SIGV * NE + k], latl = kt[(SKT_N + 1) * NE + k], dts = tt.dts;
      double wave = 1.0;
      if (tt.wpi[s] != 0 && k >= 1) wave = as_global(tt.wavef + (((size_t)s * NR + i) * NT + j) * NE)[(unsigned)k];
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const int l = l0 + n;
        const bool row1 = n == 0 && l0 == 0;
        const double wf = row1 ? 1.0 : wave;
        const double cxf = cex ? exp_tab(row1 ? 0.0 : -(row_done(sigv) * cl[l] * dts), ex) : 1.0;
        const double af = (l + 1 >= upa) ? exp_tab(latl * cf[8 * l + KLE_RHS], ex) : 1.0;
        y[n] = row_done(((((y[n] * wf) * cxf) * af) * af) * cxf * wf);
      }
    }
    adj_mu(cb0 + ns);  // MU1
    load(x0, x);
    __syncthreads();  // the chunks' edges are read
    rows_out();
    adj_e(cb0);  // E1
    {
      THREAD_CELLS;
      const gptr<double> g = as_global(ga);
      const int nr = own ? min(R, NPA - l0) : 0;
#pragma unroll
      for (int n = 0; n < R; ++n)
        if (n < nr) g[(unsigned)((l0 + n) * NE + k)] = y[n];
    }
#undef t
#undef THREAD_CELLS
#undef PLANE_SCALARS
  }
}

template <int R>
__global__ void __launch_bounds__(kPlaneMaxThreads, kStepSimdWaves) k_plane_adj(Launch L, const double *xin, double *adj) {
  extern __shared__ __align__(16) double sm[];
  for (int vb = blockIdx.x; vb < L.nv; vb += gridDim.x) {
    plane_adj_unit<R, false>(L, xin, adj, const_unit(L, vb), sm);
    if (L.nv > (int)gridDim.x) __syncthreads();  // LDS is rewritten for the block's next plane
  }
}

// An ensemble's members in one launch, each with the rows it has alone.
#if ADJ_PART == 3
__global__ void __launch_bounds__(kPlaneMaxThreads, kStepSimdWaves) k_plane_adj_mixed(Launch L) {
  extern __shared__ __align__(16) double sm[];
  for (int vb = blockIdx.x; vb < L.nv; vb += gridDim.x) {
    const CUnit u = const_unit(L, vb);
    switch (u.rows) {
#define ROWS(r) \
  case r: plane_adj_unit<r, true>(L, nullptr, nullptr, u, sm); break;
      ADJ_ROWS(ROWS)
#undef ROWS
    }
    if (L.nv > (int)gridDim.x) __syncthreads();
  }
}
#endif

// in groups (ADJ_PART of the build), each a translation unit of its own
#define ADJ_INST(r) template __global__ void k_plane_adj<r>(Launch, const double *, double *);
#if defined(ADJ_ONE)
ADJ_INST(ADJ_ONE)
#elif ADJ_PART == 0
ADJ_INST(2) ADJ_INST(3) ADJ_INST(4) ADJ_INST(5)
#elif ADJ_PART == 1
ADJ_INST(6) ADJ_INST(7) ADJ_INST(8)
#elif ADJ_PART == 2
ADJ_INST(9) ADJ_INST(10) ADJ_INST(11) ADJ_INST(12)
#endif

}  // namespace ramgpu
