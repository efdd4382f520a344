// pitch.hip -- the implicit pitch-angle diffusions, WPADIF
// (src/ModRamWPI.f90:643-714) and FLCscatter (src/ModRamLoss.f90:513-575):
// their coefficient tables, and the operators on their own.  In ram_run they
// run inside the plane kernel (k_plane_step<SEQ_STEPX>).
#include <hip/hip_runtime.h>

#include <vector>

#include "ctx.h"

using namespace ramgpu;

namespace {

using namespace ramgpu_host;

// a species' coefficient table (device layout [I][J][L][K]) from d1 + d2
// (Fortran (NR,NT,NE,NPA), d2 may be null), allocated on first use
int upload_coef(ramgpu_ctx *c, double **slot, const double *d1, const double *d2) {
  const size_t n = (size_t)c->nr * c->nt * c->ne * c->npa;
  if (pitch_lds_bytes(c->npa) > c->lds_limit)
    return fail(RAMGPU_EINVAL, "NPA=%d: the pitch-angle line solve's LDS exceeds the device's", c->npa);
  if (!*slot) {
    void *p = nullptr;
    if (!dev_malloc(c->device, &p, n * sizeof(double)))
      return fail(RAMGPU_ENOMEM, "allocation of a pitch-angle diffusion table failed");
    c->allocs.push_back(p);
    *slot = (double *)p;
  }
  std::vector<double> sum(d1, d1 + n);
  if (d2)
    for (size_t e = 0; e < n; ++e) sum[e] = d1[e] + d2[e];  // ATAW+ATAC, src/ModRamWPI.f90:675
  HIP_TRY(hipMemcpyAsync(c->d_stage, sum.data(), n * sizeof(double), hipMemcpyHostToDevice, c->stream));
  const int rc = launch_f2(c, true, *slot, c->d_stage, 1);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(c->stream));  // the host sum goes out of scope
  return RAMGPU_OK;
}

// the line solves of the species of job in one launch
int run_pitch(ramgpu_ctx *c, const PitchJob &job) {
  if (job.n == 0) return RAMGPU_OK;
  const int lines = (c->nr - 1) * c->nt * (c->ne - 1);
  tbeg(c, RAMGPU_KERNEL_PITCH);
  hipLaunchKernelGGL(k_pitch_diffusion, dim3((lines + kPitchThreads - 1) / kPitchThreads, job.n),
                     dim3(kPitchThreads), pitch_lds_bytes(c->npa), c->stream, c->d_tab, job);
  tend(c);
  return launch_check("k_pitch_diffusion");
}

int run_pitch(ramgpu_ctx *c, int s, const double *coef) {
  PitchJob job{};
  job.n = 1;
  job.s[0] = s;
  job.coef[0] = coef;
  return run_pitch(c, job);
}

}  // namespace

namespace ramgpu_host {

int takes_pitch(const ramgpu_ctx *c) {
  for (int s = 0; s < c->ns; ++s)
    if (c->t.pd_wpi[s] || c->t.pd_emic[s] || c->t.flc[s]) return 1;
  return 0;
}

int forward_only(const ramgpu_ctx *c) {
  if (c->t.coul || takes_pitch(c))
    return fail(RAMGPU_ESTATE,
                "Coulomb collisions, WPADIF or FLC scattering are on: the reverse mode and ensembles do not take "
                "them");
  return RAMGPU_OK;
}

}  // namespace ramgpu_host

extern "C" {

int ramgpu_set_wpadif(ramgpu_ctx *c, int s, const double *d1, const double *d2, int at_wpi, int at_emic) {
  int rc = check_ctx(c);
  if (rc || (rc = check_species(c, s))) return rc;
  if (d1 && (rc = upload_coef(c, &c->d_pdc[s - 1], d1, d2))) return rc;
  c->t.pdc[s - 1] = c->d_pdc[s - 1];
  c->t.pd_wpi[s - 1] = (d1 && at_wpi) ? 1 : 0;
  c->t.pd_emic[s - 1] = (d1 && at_emic) ? 1 : 0;
  c->tab_dirty = true;
  return RAMGPU_OK;
}

int ramgpu_wpadif(ramgpu_ctx *c, int s) {
  int rc = check_ctx(c);
  if (rc || (rc = check_species(c, s))) return rc;
  if (!c->d_pdc[s - 1]) return fail(RAMGPU_ESTATE, "species %d has no WPADIF coefficients (ramgpu_set_wpadif)", s);
  if ((rc = prepare(c))) return rc;
  return run_pitch(c, s - 1, c->d_pdc[s - 1]);
}

int ramgpu_set_flc(ramgpu_ctx *c, int s, const double *coef, double dt_bc) {
  int rc = check_ctx(c);
  if (rc || (rc = check_species(c, s))) return rc;
  c->dt_bc = dt_bc;
  if (!coef) {
    c->t.flc[s - 1] = nullptr;  // the table stays allocated for a later call
    c->tab_dirty = true;
    return RAMGPU_OK;
  }
  double *slot = c->d_flc_mem[s - 1];
  if ((rc = upload_coef(c, &slot, coef, nullptr))) return rc;
  c->d_flc_mem[s - 1] = slot;
  c->t.flc[s - 1] = slot;
  c->tab_dirty = true;
  return RAMGPU_OK;
}

int ramgpu_flcscatter(ramgpu_ctx *c, int s) {
  int rc = check_ctx(c);
  if (rc || (rc = check_species(c, s))) return rc;
  if (!c->t.flc[s - 1]) return fail(RAMGPU_ESTATE, "species %d has no FLC coefficients (ramgpu_set_flc)", s);
  if (c->time_elapsed < c->dt_bc) return RAMGPU_OK;  // src/ModRamLoss.f90:526
  if ((rc = prepare(c))) return rc;
  return run_pitch(c, s - 1, c->t.flc[s - 1]);
}

}  // extern "C"
