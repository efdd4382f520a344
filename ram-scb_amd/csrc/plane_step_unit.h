// plane_step_unit.h -- one unit (a plane) of k_plane_step and k_plane_mixed
// (plane_step.hip), included into the bodies of both.  As a function of its own
// the same code takes other registers in k_plane_step: SEQ_STEP at 9 rows (48x90
// planes) then spills two, SEQ_STEPX at 11 rows (35x72) 125 instead of 77, which
// with the last loops' counters signed (131) was 7% of a step with Coulomb
// collisions.
// In scope: SEQ, R, L, rec, u, sm; UNIT_DONE leaves the unit; UNIT_MIXED: the
// block may have more than the plane's UNIT_THREADS.
    CTab *const tp = u.t;
#define t (*tp)
    const int NE = t.ne, NPA = t.npa, NT = t.nt, NR = t.nr;
    const double *const src = launch_src(L, t);
    double *const dst = launch_dst(L, t);
    const size_t sstr = (size_t)u.s * f2_species_stride(t);
    if (u.b >= blocks_kl(t)) {  // out of place: copy plane (I=1, J) of the unswept row
      const size_t off = sstr + (size_t)(u.b - blocks_kl(t)) * NE * NPA;
      block_copy<8>(dst + off, src + off, NE * NPA);
      UNIT_DONE;
    }
    const int s = u.s, i = 1 + fast_div(u.b, NT, t.rnt), j = u.b - (i - 1) * NT;  // I = i+1 >= 2
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int Q = (NPA + R - 1) / R, NPAP = Q * R, S = NE + 3, ncol = Q * NE;
    const size_t ij = (size_t)i * NT + j;
    const size_t po = sstr + ij * ((size_t)NE * NPA);
    StepLds d;
    d.F = sm;
    d.cf = d.F + (max(NPAP * S, 4 * ncol) + 1) / 2 * 2;
    d.cm = d.cf + 8 * NPAP;
    d.cl = d.cm + 8 * NPAP;
    d.lt = d.cl + (NPAP + 1) / 2 * 2;
    d.kt = d.lt + 4 * (NPAP + 1);
    d.ex = d.kt + (SKT_N + 2) * NE;
    d.red = d.ex + 64;
    d.cmx = (unsigned long long *)(d.red + 16 * kSums);
    const bool apart = (X ? t.stepx_apart : t.step_apart) != 0;
#if UNIT_MIXED
    if (tid >= UNIT_THREADS) {  // whole waves: the unit's barriers
      for (int x = 0; x < (apart ? 6 : 8); ++x) __syncthreads();
      UNIT_DONE;
    }
#endif
    d.H = apart ? (double *)(d.cmx + NE + kStepSpread * NPA) : d.F;
    if constexpr (X) {
      const int o = (int)((double *)(d.cmx + NE + kStepSpread * NPA) - sm) + (apart ? 4 * ncol : 0);
      d.ct = sm + (o + 1) / 2 * 2;
      d.cy = d.ct + 6 * NPAP;
    }

    // this thread's column; a wave's lane 0 repeats the last column of the
    // wave before (step_wave_cells), so that every energy face's upper
    // neighbour is the next lane
    const int W = t.step_cells, c_raw = wv * W + lane - (64 - W);
    const bool own = c_raw < ncol && lane >= 64 - W;
    const int c_ = min(max(c_raw, 0), ncol - 1);
    const int q_ = fast_div(c_, NE, t.rne), k_ = c_ - q_ * NE;
    // every phase forms its indices afresh from these (fresh): kept across
    // the phases they would take the registers of the rows
#define THREAD_CELLS                                          \
  const int q = fresh(q_), k = fresh(k_), l0 = q * R;         \
  const int nr = own ? min(R, NPA - l0) : 0; /* real rows */  \
  (void)nr; (void)k

    // loads: the plane's cells, then its tables
    double f[R];
    {
      THREAD_CELLS;
      const gptr<const double> gF = as_global(src + po);
#pragma unroll
      for (int n = 0; n < R; ++n) f[n] = gF[(unsigned)(min(l0 + n, NPA - 1) * NE + k)];
    }
    {
      typedef double d2 __attribute__((ext_vector_type(2)));
      const gptr<const d2> g0 = (gptr<const d2>)(t.kle + ij * 8 * NPA), g1 = (gptr<const d2>)(t.klm + ij * 8 * NPA),
                           g3 = (gptr<const d2>)t.lt4;
      const gptr<const double> g2 = as_global((const double *)(t.kll + ij * NPA));  // HDNS, 1/FNHS
      const int n1 = 4 * NPA, n2 = NPA, n3 = 2 * NPA;
      d2 *const l0_ = (d2 *)d.cf, *const l1_ = (d2 *)d.cm, *const l3_ = (d2 *)d.lt;
      const int T = UNIT_THREADS;
      d2 v0 = {0, 0}, v1 = {0, 0}, v3 = {0, 0};
      double v2 = 0.0;
      if (tid < n1) {
        v0 = g0[(unsigned)tid];
        v1 = g1[(unsigned)tid];
      }
      if (tid < n2) v2 = g2[(unsigned)(2 * tid)];
      if (tid < n3) v3 = g3[(unsigned)tid];
      const gptr<const double> gk = as_global(t.kt + (size_t)s * SKT_N * NE);
      const int nk = SKT_N * NE;
      const double vk = tid < nk ? gk[(unsigned)tid] : 0.0;
      double ve = 0.0, va = 0.0, vx = 0.0;
      if (tid < NE) {
        ve = as_global(t.edot + ((size_t)s * NR + i) * NE)[(unsigned)tid];
        va = as_global(t.latl + ((size_t)s * NR + i) * NE)[(unsigned)tid];
      }
      if (tid < 64) vx = as_global(t.ex64)[(unsigned)tid];
      if (tid < n1) {
        l0_[tid] = v0;
        l1_[tid] = v1;
      }
      if (tid < n2) d.cl[tid] = v2;
      if (tid < n3) l3_[tid] = v3;
      if (tid < nk) d.kt[tid] = vk;
      if (tid < NE) {
        d.kt[SKT_N * NE + tid] = ve;
        d.kt[(SKT_N + 1) * NE + tid] = va;
      }
      if (tid < 64) d.ex[tid] = vx;
      for (int e = tid + T; e < n1; e += T) {  // what one pass did not cover (small blocks)
        l0_[e] = g0[e];
        l1_[e] = g1[e];
      }
      for (int e = tid + T; e < n2; e += T) d.cl[e] = g2[2 * e];
      for (int e = tid + T; e < n3; e += T) l3_[e] = g3[e];
      for (int e = tid + T; e < nk; e += T) d.kt[e] = gk[e];
      for (int e = tid + T; e < NE; e += T) {
        d.kt[SKT_N * NE + e] = t.edot[((size_t)s * NR + i) * NE + e];
        d.kt[(SKT_N + 1) * NE + e] = t.latl[((size_t)s * NR + i) * NE + e];
      }
      // rows past NPA: zero terms, so that their Courant numbers are 0
      for (int e = n1 + tid; e < 4 * NPAP; e += T) l0_[e] = l1_[e] = d2{0.0, 0.0};
      for (int e = n2 + tid; e < NPAP; e += T) d.cl[e] = 0.0;
      for (int e = n3 + tid; e < 2 * (NPAP + 1); e += T) l3_[e] = d2{0.0, 0.0};
      if constexpr (X) step_line_tables(t, d, i, j, NPAP);
      if (rec & 1)
        for (int e = tid; e < NE + kStepSpread * NPA; e += T) d.cmx[e] = 0ull;
    }
    const bool record = (rec & 1) && as_const((const double *)t.kij)[ij * 8 + KIJ_MG] == 0.0;
    // the plane's scalars, read where a phase needs them
#define PLANE_SCALARS                                                                                    \
  CTab &tt = *fresh_uniform(tp);                                                                         \
  const cptr<double> kij = as_const((const double *)tt.kij) + ij * 8;                                    \
  const double rlz = as_const(tt.rlz)[i], rrlz = as_const((const double *)tt.rrlz)[i], beta = tt.betalim; \
  const double bij = kij[KIJ_BIJ], rbij = kij[KIJ_RBIJ]

    // rows into LDS; the thread that holds F(2) forms DRIFTE's relativistic
    // ghosts F(1), F(0) from it (src/ModRamDrift.f90:333-335), or COULEN's,
    // with the square roots of the inverse ratios (src/ModRamCoul.f90:180-181)
    auto rows_out = [&](auto coul) __attribute__((always_inline)) {
      if (own) {
        THREAD_CELLS;
        double *const Frow = d.F + l0 * S + k;
        if (k >= 1) {
#pragma unroll
          for (int n = 0; n < R; ++n) Frow[n * S + 1] = f[n];
        }
        if (k == 1) {
          const cptr<double> rel = as_const((const double *)fresh_uniform(tp)->rel) + s * 8;
          double r2 = rel[2], r4 = rel[4];
          if constexpr (decltype(coul)::value) {
            const cptr<double> crel = as_const((const double *)fresh_uniform(tp)->crel) + s * 5;
            r2 = crel[2];
            r4 = crel[4];
          }
          const double r0 = rel[0], r1 = rel[1], r3 = rel[3], rr1 = rel[5], rr0 = rel[6];
#pragma unroll
          for (int n = 0; n < R; ++n) {
            const double g1 = div_rn(f[n] * r0, r1, rr1) * r2;
            Frow[n * S] = g1;
            Frow[n * S - 1] = div_rn(g1 * r3, r0, rr0) * r4;
          }
        }
        if (k == NE - 1) {  // F(NE+1) = F(NE+2) = 0
#pragma unroll
          for (int n = 0; n < R; ++n) Frow[n * S + 2] = Frow[n * S + 3] = 0.0;
        }
      }
      __syncthreads();
    };
    // the clamp decision of a drift phase, one byte per cell ([L][K])
    auto clamp_byte = [&](unsigned char *cb, int l, int k, double w) { cb[l * NE + k] = (w < 0) ? 1 : 0; };

    // Courant numbers of this thread's cells, kept from the first sweep of a
    // kind for its second where the registers hold them
    double kce[kKeepE ? R : 1], kcm[kKeepMu ? R : 1];

    // DRIFTE (src/ModRamDrift.f90:333-369); K=1 is not updated.  The owner of
    // face K forms F(K) - C(K)/WE(K)*FBND(K) and the term C(K)/WE(K+1)*FBND(K)
    // that the next lane adds.  coul: COULEN instead (src/ModRamCoul.f90:
    // 154-217), the same sweep with CccolE(K) = (COULE+COULI)(S,K,L)*XNE(L) on
    // rows L=2..NPA, no CFL record.
    auto drift_e = [&](auto coul, bool first, unsigned char *cb) __attribute__((always_inline)) {
      constexpr bool COUL = decltype(coul)::value;
      THREAD_CELLS;
      PLANE_SCALARS;
      const double *const Frow = d.F + l0 * S + k;  // row n: Frow[n*S + 0..3] = F(K-1)..F(K+2)
      const double drd1 = kij[KIJ_DRD1], dpd1 = kij[KIJ_DPD1];
      const double *const kt = d.kt + k;
      const double ekp = kt[SKT_EKPQ * NE], edot = kt[SKT_N * NE];
      const double de = kt[SKT_DE * NE], rde = kt[SKT_RDE * NE];
      const double we = kt[SKT_WE * NE], rwe = kt[SKT_RWE * NE];
      const bool top = k + 1 >= NE;  // its upper term goes to a lane that does not use it
      const double we1 = top ? 1.0 : kt[SKT_WE * NE + 1], rwe1 = top ? 1.0 : kt[SKT_RWE * NE + 1];
      const double *const cf = d.cf + 8 * l0;
      double cmax = 0.0, cc[COUL ? R : 1];
      if constexpr (COUL) {
        const gptr<const double> gc = as_global(tt.cc + (size_t)s * NPA * NE);
#pragma unroll
        for (int n = 0; n < R; ++n) cc[n] = gc[(unsigned)(min(l0 + n, NPA - 1) * NE + k)] * d.ct[6 * (l0 + n)];
      }
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const double *p = Frow + n * S;
        double ce;
        if constexpr (COUL) ce = cc[n];
        else ce = (kKeepE && !first) ? kce[kKeepE ? n : 0]
                                     : c_energy(cf + 8 * n, ekp, edot, drd1, dpd1, bij, rbij, rlz, rrlz);
        if (kKeepE && first) kce[n] = ce;
        if (!COUL) cmax = fmax(cmax, fabs(ce));
        const bool neg = ce < 0;
        const double f0 = p[1], fp1 = p[2], a = p[neg ? 3 : 0];
        const double u2 = face_value2(f0, fp1, neg ? fp1 : f0, a, neg, div_rn(ce, de, rde), beta);
        const double h = div_rn(ce, we1, rwe1) * u2;
        const double w = fma(-0.5, div_rn(ce, we, rwe) * u2, f0);
        double v = fma(0.5, from_lane_below0(h), w);
        if (k >= 1) {
          if (TAPE && n < nr) clamp_byte(cb, l0 + n, k, v);
          if (!(COUL && n == 0 && l0 == 0)) f[n] = v < 0 ? 1E-15 : v;
        }
        f[n] = row_done(f[n]);
      }
      if (!COUL && first && record && own) atomic_max_pos(&d.cmx[k], fmax(cmax, 1E-10));
    };

    // DRIFTMU (src/ModRamDrift.f90:413-466).  F(1)=F(2) for the stencil;
    // limiter faces L=2..NPA-2; CDriftMu(1)=0, FBND(1)=0, FBND(NPA-1)=F(NPA);
    // top cell F2(NPA)=F2(NPA-1)*FNHS(NPA)*MU(NPA)/FNHS(NPA-1)/MU(NPA-1).
    // The rows beside the chunk come through LDS, the flux terms at
    // chunk edges likewise.
    auto drift_mu = [&](bool first, unsigned char *cb) __attribute__((always_inline)) {
      THREAD_CELLS;
      PLANE_SCALARS;
      const int c0 = q * NE + k;
      if (own) {
        d.H[c0] = f[0];
        d.H[ncol + c0] = f[1];
        d.H[2 * ncol + c0] = f[R - 1];
      }
      __syncthreads();
      const double drm1 = kij[KIJ_DRM1], dpm1 = kij[KIJ_DPM1], db2 = kij[KIJ_DB2];
      const double mkp = d.kt[SKT_MKPQ * NE + k];
      double fm = d.H[2 * ncol + (q > 0 ? c0 - NE : c0)];
      const int cu = (q + 1 < Q) ? c0 + NE : c0;
      const double up0 = d.H[cu], up1 = d.H[ncol + cu];
      double hprev = 0.0;
      const double *const lt = d.lt + 4 * l0, *const cmr = d.cm + 8 * l0;
      double wn = lt[2], rwn = lt[3];
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const int l = l0 + n;
        const double f0 = f[n], f1 = n + 1 < R ? f[n + 1 < R ? n + 1 : 0] : up0;
        const double f2 = n + 2 < R ? f[n + 2 < R ? n + 2 : 0] : (n + 2 == R ? up0 : up1);
        const double cm = (kKeepMu && !first) ? kcm[kKeepMu ? n : 0]
                                              : c_mu(cmr + 8 * n, mkp, drm1, dpm1, db2, bij, rbij, rlz, rrlz);
        if (kKeepMu && first) kcm[n] = cm;
        if (first && record && own && l >= 1 && l < NPA)
          atomic_max_pos(&d.cmx[NE + kStepSpread * l + (k & (kStepSpread - 1))], fmax(fabs(cm), 1E-32));
        const bool neg = cm < 0;
        const double fl = (n == 1 && l0 == 0) ? f0 : fm;  // F(1) = F(2)
        double u2 = face_value2(f0, f1, neg ? f1 : f0, neg ? f2 : fl, neg, div_rn(cm, lt[4 * n], lt[4 * n + 1]), beta);
        if (l == NPA - 2) u2 = 2.0 * f1;  // FBND(NPA-1) = F(NPA)
        double on = div_rn(cm, wn, rwn) * u2;
        wn = lt[4 * n + 6];
        rwn = lt[4 * n + 7];
        double up = div_rn(cm, wn, rwn) * u2;
        if (n == 0 && l0 == 0) on = up = 0.0;  // face 1: CDriftMu(1) = 0, FBND(1) = 0
        const double v = fma(0.5, hprev, fma(-0.5, on, f0));
        hprev = up;
        fm = f0;
        f[n] = row_done((n == 0 && l0 == 0) ? f0 : v);  // row 1 is not updated
      }
      if (own) d.H[3 * ncol + c0] = hprev;  // for the chunk above
      __syncthreads();
      if (q >= 1) f[0] = fma(0.5, d.H[3 * ncol + c0 - NE], f[0]);
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const bool upd = !(n == 0 && l0 == 0);
        if (TAPE && upd && n < nr && l0 + n <= NPA - 2) clamp_byte(cb, l0 + n, k, f[n]);
        if (f[n] < 0 && upd) f[n] = 1E-15;
      }
      if (l0 + R >= NPA) {  // the top row, from the finished row below it, and its copies above
        const cptr<double> fh = as_const(tt.fnhs) + i + (size_t)(NR + 1) * (j + (size_t)NT * (NPA - 2));
        const cptr<double> mu = as_const(tt.mu) + NPA - 2;
        double b = f[0];
        // row_done: as a plain choice among f[n] the compiler may make it one
        // load at a variable index, which puts the rows into scratch memory
#pragma unroll
        for (int n = 1; n < R - 1; ++n) {
          const double fn = row_done(f[n]);
          b = (l0 + n == NPA - 2) ? fn : b;
        }
        const double topv = b * fh[(size_t)(NR + 1) * NT] * mu[1] / fh[0] / mu[0];
#pragma unroll
        for (int n = 1; n < R; ++n) f[n] = (l0 + n >= NPA - 1) ? topv : f[n];
      }
    };

    // the plane (this thread's cells) to p
    auto store = [&](double *p) __attribute__((always_inline)) {
      THREAD_CELLS;
      const gptr<double> g = as_global(p);
#pragma unroll
      for (int n = 0; n < R; ++n)
        if (n < nr) g[(unsigned)((l0 + n) * NE + k)] = f[n];
    };

    const size_t tn = TAPE ? (size_t)t.ns * f2_species_stride(t) : 0;
    double *const slot = TAPE ? const_cast<double *>(src) + po : nullptr;
    unsigned char *const cb = TAPE ? reinterpret_cast<unsigned char *>(const_cast<double *>(src) + 7 * tn) + po : nullptr;

    // EKEV*WE of this thread's cells in SUMRC (I,K,L>=2, J<=NT-1), else 0
    auto sum_factor = [&](int k) __attribute__((always_inline)) {
      return (own && j <= NT - 2 && k >= 1) ? d.kt[SKT_EKW * NE + k] : 0.0;
    };

    // The loss chain (src/ModRamRun.f90:77-159): SUMRC, [WAVELO, SUMRC],
    // [CEX, SUMRC], ATMOL, SUMRC, ATMOL, SUMRC, [CEX, SUMRC], [WAVELO,
    // SUMRC].  CEX acts on K,L>=2 (its rate is 0 for K=1 and for species
    // without it: a factor of exactly 1), ATMOL on K>=2, L>=UPA(I) (its
    // log(ATLOS) is 0 for K=1), WAVELO on K,L>=2; a weight of 0 leaves a cell
    // out of the sums.
    auto losses = [&]() __attribute__((always_inline)) {
      THREAD_CELLS;
      CTab &tt = *fresh_uniform(tp);
      const bool cex = tt.cex[s] != 0, wpi = tt.wpi[s] != 0;
      const int upa = as_const(tt.upa)[i];
      const double sigv = d.kt[SKT_SIGV * NE + k], latl = d.kt[(SKT_N + 1) * NE + k];
      const double ekw = sum_factor(k);
      double wave = 1.0;
      if (wpi && k >= 1) wave = as_global(tt.wavef + (((size_t)s * NR + i) * NT + j) * NE)[(unsigned)k];
      const double dts = tt.dts;
      const double *const cf = d.cf + 8 * l0, *const cl = d.cl + l0, *const lt = d.lt + 4 * l0;
      double a[5] = {0, 0, 0, 0, 0};
      // two rows at a time, so that their exponentials overlap
#pragma unroll
      for (int n0 = 0; n0 < R; n0 += 2) {
        double cxf[2] = {1.0, 1.0}, af[2] = {1.0, 1.0};
        if (cex)
#pragma unroll
          for (int g = 0; g < 2 && n0 + g < R; ++g)
            cxf[g] = exp_tab((n0 + g == 0 && l0 == 0) ? 0.0 : -(sigv * cl[n0 + g] * dts), d.ex);
        if (l0 + n0 + 2 >= upa)
#pragma unroll
          for (int g = 0; g < 2 && n0 + g < R; ++g)
            af[g] = exp_tab((l0 + n0 + g + 1 >= upa) ? latl * cf[8 * (n0 + g) + KLE_RHS] : 0.0, d.ex);
#pragma unroll
        for (int g = 0; g < 2 && n0 + g < R; ++g) {
          const int n = n0 + g, l = l0 + n;
          const bool row1 = n == 0 && l0 == 0;
          const double qw = (row1 || l >= NPA) ? 0.0 : ekw * lt[4 * n + 2];  // EKEV*WE*WMU
          const double wf = row1 ? 1.0 : wave;
          double x = f[n];
          auto in_sum = [&]() __attribute__((always_inline)) { return (X && row1) ? 0.0 : x; };
          a[0] = fma(in_sum(), qw, a[0]);
          x = x * wf;
          x = x * cxf[g];
          a[1] = fma(in_sum(), qw, a[1]);
          x = x * af[g];
          a[2] = fma(in_sum(), qw, a[2]);
          x = x * af[g];
          a[3] = fma(in_sum(), qw, a[3]);
          x = x * cxf[g];
          a[4] = fma(in_sum(), qw, a[4]);
          f[n] = row_done(x * wf);
#pragma unroll
          for (int m = 0; m < 5; ++m) a[m] = row_done(a[m]);
        }
      }
      // slots: before WAVELO, after it, after CEX, ATMOL, ATMOL, CEX, after
      // WAVELO; each wave's sums in a fixed order, the waves' added up below
      if constexpr (X)
#pragma unroll
        for (int m = 0; m < 5; ++m) a[m] = ekw != 0.0 ? a[m] : 0.0;
      double s7[7] = {a[0], a[0] * wave, a[1], a[2], a[3], a[4], a[4] * wave};
#pragma unroll
      for (int m = 0; m < 7; ++m) s7[m] = wave_sum(s7[m]);
      if (lane == 63)
#pragma unroll
        for (int m = 0; m < 7; ++m) d.red[wv * kSums + m] = s7[m];
    };

    // ---- SEQ_STEPX: the optional processes ---------------------------------
    // SUMRC's partial of the plane as it stands, slot m.  A cell outside the
    // sum is left out of it, not weighed by 0: it may hold anything
    auto sum_slot = [&](int m) __attribute__((always_inline)) {
      THREAD_CELLS;
      const double ekw = sum_factor(k);
      const double *const lt = d.lt + 4 * l0;
      double a = 0.0;
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const bool row1 = n == 0 && l0 == 0;
        a = fma(row1 ? 0.0 : f[n], (row1 || l0 + n >= NPA) ? 0.0 : ekw * lt[4 * n + 2], a);
      }
      a = wave_sum(ekw != 0.0 ? a : 0.0);
      if (lane == 63) d.red[wv * kSums + m] = a;
    };
    // The implicit pitch-angle step of every line (I,J,K>=2): the reference's
    // recurrences in its order, RK(1)=0, RL(1)=-1, RK and RL forward over
    // L=2..NPA-1, back substitution, F2(NPA)=F2(NPA-1).  f holds RP and
    // leaves as the solution; an, gn the couplings.  A line runs through its
    // chunks one after the other, a chunk's rows in one thread's registers:
    // a row costs the latency of the recurrence alone (DENOM, its reciprocal,
    // two quotients), since everything else was formed by all threads.  The
    // other blocks of the CU fill the idle lanes' issue slots.  Plane launch of
    // 4 species, 35x72 (20x25 grid), by events: with Coulomb collisions 422 us
    // (the lines in the plane in LDS, one thread each) -> 213; with WPADIF and
    // FLCscatter too 1430 us a step as one launch per operator -> 416.
    auto solve = [&](double (&an)[R], double (&gn)[R]) __attribute__((always_inline)) {
      THREAD_CELLS;
      const int last = NPA - 2;  // row of L = NPA-1
      const bool line = own && k >= 1;
      double rk = 0.0, rl = -1.0, x = 0.0;
#pragma unroll 1
      for (int qq = 0; qq < Q; ++qq) {
        if (line && q == qq) {
          if (qq > 0) {
            rk = d.cy[k];
            rl = d.cy[NE + k];
          }
#pragma unroll
          for (int n = 0; n < R; ++n) {
            if (n == 0 && qq == 0) {
              f[0] = 0.0;
              an[0] = -1.0;
            } else if (l0 + n <= last) {
              const double den = an[n] + gn[n] + gn[n] * rl + 1;
              double y = __builtin_amdgcn_rcp(den);
              const double e = fma(-den, y, 1.0);
              y = fma(y, fma(e, e, e), y);  // 1/DENOM within an ulp, as div_fast's
              rk = div_rn(f[n] + gn[n] * rk, den, y);
              rl = div_rn(-an[n], den, y);
              f[n] = rk;
              an[n] = rl;
            }
          }
          d.cy[k] = rk;
          d.cy[NE + k] = rl;
        }
        __syncthreads();
      }
      if (q == Q - 1) x = rk / (1 + rl);
#pragma unroll 1
      for (int qq = Q - 1; qq >= 0; --qq) {
        if (line && q == qq) {
          if (qq < Q - 1) x = d.cy[2 * NE + k];
#pragma unroll
          for (int n = R - 1; n >= 0; --n) {
            if (l0 + n < last) x = f[n] - an[n] * x;
            f[n] = x;
          }
          d.cy[2 * NE + k] = x;
        }
        __syncthreads();
      }
    };
    // COULMU (src/ModRamCoul.f90:255-292)
    auto coulmu = [&]() __attribute__((always_inline)) {
      double an[R], gn[R];
      {
        THREAD_CELLS;
        const gptr<const double> cg = as_global((const double *)(fresh_uniform(tp)->cag + (size_t)s * NPA * NE));
#pragma unroll
        for (int n = 0; n < R; ++n) {
          const double2 v = ld_d2(cg, (unsigned)(min(l0 + n, NPA - 1) * NE + k));
          an[n] = v.x;
          gn[n] = v.y;
        }
        const int lm = max(l0 - 1, 0);
        double xbm = d.ct[6 * lm + 1], bhm = d.cm[8 * lm + KLM_BHS];
#pragma unroll
        for (int n = 0; n < R; ++n) {
          const int l = l0 + n;
          const double *r = d.ct + 6 * l;
          const double fh = d.cf[8 * l + KLE_HS], rfh = d.cf[8 * l + KLE_RHS], bh = d.cm[8 * l + KLM_BHS], xb = r[1];
          an[n] = row_done(div_rn(an[n] * xb, fh, rfh) * bh);
          gn[n] = row_done(div_rn(gn[n] * xbm, fh, rfh) * bhm);
          const double rp = div_rn(div_rn(f[n], fh, rfh), r[2], r[3]);
          f[n] = row_done(own && k >= 1 ? rp : f[n]);  // the cell K=1 is not updated
          xbm = xb;
          bhm = bh;
        }
      }
      solve(an, gn);
      {
        THREAD_CELLS;
        const bool clamp = (rec & 2) != 0;
#pragma unroll
        for (int n = 0; n < R; ++n) {
          const int l = l0 + n;
          double v = f[n] * d.cf[8 * l + KLE_HS] * d.ct[6 * l + 2];
          if (clamp && v < 0.) v = 1E-15;
          f[n] = row_done(own && k >= 1 ? v : f[n]);
        }
      }
    };
    // WPADIF (src/ModRamWPI.f90:643-714) and FLCscatter (src/ModRamLoss.f90:
    // 513-575) with the coefficients D of one species (device layout)
    auto diffuse = [&](const double *coef) __attribute__((always_inline)) {
      double an[R], gn[R];
      {
        THREAD_CELLS;
        const gptr<const double> D = as_global(coef + ij * ((size_t)NE * NPA));
#pragma unroll
        for (int n = 0; n < R; ++n) an[n] = D[(unsigned)(min(l0 + n, NPA - 1) * NE + k)];
        const int lm = max(l0 - 1, 0);
        double pm = div_rn(D[(unsigned)(lm * NE + k)], d.lt[4 * lm], d.lt[4 * lm + 1]);
        const double dts = fresh_uniform(tp)->dts;
#pragma unroll
        for (int n = 0; n < R; ++n) {
          const int l = l0 + n;
          const double *r = d.ct + 6 * l, *lt = d.lt + 4 * l;
          const double fac = r[4], rfac = r[5], p = div_rn(an[n], lt[0], lt[1]);
          an[n] = row_done(div_rn(div_rn(p * dts, fac, rfac), lt[2], lt[3]));
          gn[n] = row_done(div_rn(div_rn(pm * dts, fac, rfac), lt[2], lt[3]));
          f[n] = row_done(own && k >= 1 ? div_rn(f[n], fac, rfac) : f[n]);
          pm = p;
        }
      }
      solve(an, gn);
      {
        THREAD_CELLS;
#pragma unroll
        for (int n = 0; n < R; ++n) f[n] = row_done(own && k >= 1 ? f[n] * d.ct[6 * (l0 + n) + 4] : f[n]);
      }
    };
    // CHAREXCHANGE, ATMOL twice (slots 3, 4) and WAVELO on their own
    auto one_loss = [&](int op) __attribute__((always_inline)) {
      THREAD_CELLS;
      CTab &tt = *fresh_uniform(tp);
      const int upa = as_const(tt.upa)[i];
      const double dts = tt.dts, ekw = sum_factor(k);
      const double sigv = d.kt[SKT_SIGV * NE + k], latl = d.kt[(SKT_N + 1) * NE + k];
      double wave = 1.0, a3 = 0.0, a4 = 0.0;
      if (op == 2 && tt.wpi[s] != 0 && k >= 1)
        wave = as_global(tt.wavef + (((size_t)s * NR + i) * NT + j) * NE)[(unsigned)k];
#pragma unroll
      for (int n = 0; n < R; ++n) {
        const int l = l0 + n;
        const bool row1 = n == 0 && l0 == 0;
        if (op == 0) {
          f[n] = row_done(f[n] * exp_tab(row1 ? 0.0 : -(row_done(sigv) * d.cl[l] * dts), d.ex));
        } else if (op == 1) {
          const double af = (l + 1 >= upa) ? exp_tab(row_done(latl) * d.cf[8 * l + KLE_RHS], d.ex) : 1.0;
          const double qw = (row1 || l >= NPA) ? 0.0 : ekw * d.lt[4 * l + 2];
          double x = f[n] * af;
          a3 = fma(row1 ? 0.0 : x, qw, a3);
          x = x * af;
          a4 = row_done(fma(row1 ? 0.0 : x, qw, a4));
          f[n] = row_done(x);
        } else {
          f[n] = row_done(row1 ? f[n] : f[n] * wave);
        }
      }
      if (op == 1) {
        a3 = wave_sum(ekw != 0.0 ? a3 : 0.0);
        a4 = wave_sum(ekw != 0.0 ? a4 : 0.0);
        if (lane == 63) {
          d.red[wv * kSums + 3] = a3;
          d.red[wv * kSums + 4] = a4;
        }
      }
    };
    // [WAVELO or WPADIF], [EMIC WPADIF], [CEX], [FLC], ATMOL, ATMOL and back
    // (src/ModRamRun.f90:91-159), with a SUMRC slot after every operator but
    // FLCscatter, of a species with a line solve in the chain
    auto losses_solves = [&]() {
#pragma unroll 1
      for (int h = 0; h < 2; ++h) {
#pragma unroll 1
        for (int o = 0; o < 4; ++o) {
          const int op = h == 0 ? o : 3 - o;
          CTab &tt = *fresh_uniform(tp);
          if (op == 0) {
            if (h == 0) sum_slot(0);
            if (tt.pd_wpi[s]) diffuse(tt.pdc[s]);
            else if (tt.wpi[s]) one_loss(2);
            sum_slot(h == 0 ? 1 : 6);
          } else if (op == 1) {
            if (tt.pd_emic[s]) diffuse(tt.pdc[s]);
            sum_slot(h == 0 ? kSumEmic : kSumEmic + 1);
          } else if (op == 2) {
            if (tt.cex[s]) one_loss(0);
            sum_slot(h == 0 ? 2 : 5);
          } else if ((rec & 4) && tt.flc[s]) {
            diffuse(tt.flc[s]);
          }
        }
        if (h == 0) one_loss(1);
      }
    };

    rows_out(No());
    drift_e(No(), true, cb);
    if (TAPE) store(slot + tn);
    if (!apart) __syncthreads();  // the energy stencil is read
    drift_mu(true, TAPE ? cb + tn : nullptr);
    if (TAPE) store(slot + 2 * tn);
    if constexpr (X) {
      const bool coul = tp->coul != 0;
      if (coul) {
        sum_slot(kSumCoul);
        if (!apart) __syncthreads();  // the chunks' edge terms are read
        rows_out(Yes());
        drift_e(Yes(), false, nullptr);
        sum_slot(kSumCoul + 1);
        coulmu();
      }
      if (tp->pd_wpi[s] || tp->pd_emic[s] || tp->flc[s]) losses_solves();
      else losses();
      if (coul) {
        coulmu();
        sum_slot(kSumCoul + 2);
        rows_out(Yes());
        drift_e(Yes(), false, nullptr);
        sum_slot(kSumCoul + 3);
        if (!apart) __syncthreads();  // the energy stencil is read
      }
    } else {
      losses();
    }
    if (TAPE) store(slot + 3 * tn);
    drift_mu(false, TAPE ? cb + 2 * tn : nullptr);
    if (TAPE) store(slot + 4 * tn);
    if (!apart) __syncthreads();  // the chunks' edge terms are read
    rows_out(No());
    drift_e(No(), false, TAPE ? cb + 3 * tn : nullptr);
    store(dst + po);
    // SUMRC partials and the CFL maxima, complete since the first DRIFTMU's
    // and the loss chain's next barriers
    if (tid < kSums) {
      double v = 0.0;
      for (int w = 0; w < (int)(UNIT_THREADS >> 6); ++w) v += d.red[w * kSums + tid];
      CTab &tt = *fresh_uniform(tp);
      tt.partials[((size_t)tid * tt.ns + s) * tt.maxblk + u.b] = v;
    }
    if (record) {
      unsigned long long *g = fresh_uniform(tp)->cflmax + (size_t)s * (2 + NE + NPA);
      for (int e = tid; e < NE + NPA; e += UNIT_THREADS) {
        unsigned long long m;
        if (e < NE) {
          m = d.cmx[e];
        } else {
          const unsigned long long *r = d.cmx + NE + kStepSpread * (e - NE);
          m = r[0];
          for (int x = 1; x < kStepSpread; ++x) m = max(m, r[x]);
        }
        // most planes do not raise the maximum: a load decides for less than
        // an atomic on the addresses every plane shares
        if (m > __hip_atomic_load(&g[2 + e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(&g[2 + e], m);
      }
    }
#undef t
#undef THREAD_CELLS
#undef PLANE_SCALARS
#undef UNIT_DONE
#undef UNIT_THREADS
#undef UNIT_MIXED
