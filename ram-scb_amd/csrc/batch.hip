// batch.hip -- ensembles: many independent problems stepped together.
//
// The members are ordinary contexts on one device, each with its own grid
// sizes, species, fields and F2.  A kernel of the split step is one launch
// over all members, or one per shape of its members' kernels where these are
// many blocks each (mixed_launch): a job table lists (member, species, first
// block) units and a per-block map sends each virtual block to its unit, so
// members of different sizes share a grid.  The launches of one step are captured
// once into a HIP graph and replayed per step; the Kp / boundary-scale
// schedule is read on the device through a step counter, so every replay is
// the same graph.  An autotuner picks, per kernel, how many resident blocks
// loop over the virtual blocks (persistent grid) or one block per unit.
//
// A member stepped in an ensemble runs exactly the kernels and arithmetic of
// its own ramgpu_ram_run / ramgpu_ram_run_schedule, so its results are
// bit-identical to stepping it alone.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <numeric>
#include <set>
#include <utility>
#include <vector>

#include "ctx.h"

using namespace ramgpu;
using namespace ramgpu_host;

namespace {

// kernel kinds of an ensemble launch; the last four serve reverse mode: P and
// plane out of place (with the copy lines / planes of the unswept I=1 rows),
// one unit per member (misfit) and a whole-F2 copy per member
enum BatchKind {
  BK_SCHED, BK_COEFIJ, BK_GHOST, BK_R, BK_P, BK_PLANE, BK_FIN, BK_POOP, BK_PLOOP, BK_RB, BK_PB, BK_PLB, BK_MEM,
  BK_COPY, BK_N
};

struct Plan {
  Job *jobs = nullptr;
  int *vmap = nullptr;
  int nv = 0;
  int cap = 0;  // 0: one block per virtual block; else the persistent grid size
  // sweep and plane kinds: the launches, each over the virtual blocks
  // [v0, v0 + nv) of its members: one per shape of the members' kernels (a
  // sweep's is its rows, 0 being one thread per line, and its block), or one
  // with every member's own rows (kMixedRows) where that is faster (mixed_launch)
  struct Group {
    StepShape sh;
    size_t lds;
    int v0, nv;
  };
  std::vector<Group> groups;
};

}  // namespace

struct ramgpu_batch {
  int device = 0;
  std::vector<ramgpu_ctx *> m;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  Tab *d_tabs = nullptr;
  Plan plan[BK_N];
  size_t radial_lds = 0, azim_lds = 0, ghost_lds = 0;
  int mpts_max = 0;  // most satellite points of a member (ensemble adjoint)
  // the largest block and row bound of the members' single-operator plane kernels at creation
  PlaneShape plane{64, 8, 0};
  std::vector<char> wave;  // each member's WAVELO at creation (its coefficient units)
  int sum_ns = 0;
  // DRIFTP and DRIFTR with lines in chunks (line_rows): only if the members'
  // lines together are as few.  DRIFTR's last sweep keeps a member's own
  // choice, which its SUMRC's order of summation goes with.
  bool chunks = false;
  std::vector<int> bs_off;  // first species of member m in a schedule row
  int *d_bsoff = nullptr;
  int *d_step = nullptr;
  double *d_kp = nullptr, *d_bs = nullptr;
  int sched_cap = 0;  // steps the schedule buffers hold
  bool use_graph = true;
  hipGraphExec_t exec[2] = {nullptr, nullptr};  // [0] plain step, [1] scheduled step
  std::vector<void *> allocs;
  int ncu = 256;
  // opt-in per-launch timing (eager steps only): event pairs by kernel kind
  bool timing = false;
  std::vector<hipEvent_t> tev;
  std::vector<int> tkind;
  size_t tused = 0;
};

namespace {

int batch_alloc(ramgpu_batch *b, void **p, size_t bytes) {
  if (!dev_malloc(b->device, p, std::max<size_t>(bytes, 16)))
    return fail(RAMGPU_ENOMEM, "hipMalloc of %zu bytes failed", bytes);
  b->allocs.push_back(*p);
  return RAMGPU_OK;
}

int blocks_of(const ramgpu_batch *b, int kind, const ramgpu_ctx *c) {
  switch (kind) {
    case BK_COEFIJ: return coef_units(c, 256);
    case BK_GHOST: return ghost_blocks(c->t);
    case BK_R: return blocks_r(c->t);
    case BK_P: return b->chunks ? blocks_p(c->t) : blocks_line_p(c->t);
    case BK_PLANE: case BK_PLB: return blocks_kl(c->t);
    case BK_POOP: return blocks_p_copy(c->t, b->chunks);
    case BK_RB: return blocks_line_r(c->t);
    case BK_PB: return blocks_line_p(c->t);
    case BK_PLOOP: return blocks_kl(c->t) + c->nt;
    case BK_COPY: return 256;
    default: return 1;
  }
}

bool per_member(int kind) { return kind == BK_SCHED || kind == BK_COEFIJ || kind == BK_MEM || kind == BK_COPY; }

// Whether members of several kernel shapes go in one launch, each with the
// rows it has alone, in blocks of the widest (the waves a member does not need
// only meet its barriers).  A launch per shape leaves CUs idle and pays its
// latency while it has few blocks; with many, the wide blocks cost more.  A
// step of uneven ensembles on MI355X in us, per shape / mixed (in brackets the
// planes per shape and CU): 4 members up to 14x15x19x41 143 / 86 (0.9), 8 up to
// 24x25x29x61 326 / 238 (1.7), 4 up to 40x41x45x90 380 / 349 (4.8), 32 up to
// 38x39x43x89 1243 / 1232 (4.4), 64 up to 30x31x35x73 1691 / 1728 (6.2), 64 up to
// 41x42x46x90 3653 / 4062 (12.7).
bool mixed_launch(size_t shapes, long units, int ncu) { return shapes > 1 && units <= 4L * ncu * (long)shapes; }

// Job table and block map of one kernel kind, members in order; the sweep
// and plane kinds with the members of one launch together.
int build_plan(ramgpu_batch *b, int kind) {
  std::vector<Job> jobs;
  std::vector<int> vmap;
  const bool plane = kind == BK_PLANE || kind == BK_PLOOP;
  const bool grouped = plane || kind == BK_PLB || kind == BK_R || kind == BK_P || kind == BK_POOP;
  std::vector<size_t> order(b->m.size());
  std::iota(order.begin(), order.end(), size_t(0));
  auto shape_of = [&](const ramgpu_ctx *c, size_t *lds) {
    if (plane) {
      *lds = step_lds_bytes(c->ne, c->npa, c->step.rows);
      return c->step;
    }
    if (kind == BK_PLB) {
      *lds = adj_lds_bytes(c->ne, c->npa, c->adj.rows);
      return c->adj;
    }
    const LineShape h = kind == BK_R ? r_shape(c) : p_shape(c, b->chunks);
    *lds = h.lds;
    return StepShape{h.threads, h.rows};
  };
  auto own_shape = [&](size_t mi) {
    size_t lds;
    const StepShape h = shape_of(b->m[mi], &lds);
    return std::make_pair(h.rows, h.threads);
  };
  std::set<std::pair<int, int>> shapes;
  long units = 0;
  int wide = 0;
  for (size_t mi : order)
    if (grouped && own_shape(mi).first != 0) {
      shapes.insert(own_shape(mi));
      units += (long)b->m[mi]->ns * blocks_of(b, kind, b->m[mi]);
      wide = std::max(wide, own_shape(mi).second);
    }
  const bool mixed = grouped && mixed_launch(shapes.size(), units, b->ncu);
  auto shape = [&](size_t mi) {
    const std::pair<int, int> h = own_shape(mi);
    return (mixed && h.first != 0) ? std::make_pair(kMixedRows, wide) : h;
  };
  if (grouped)
    std::stable_sort(order.begin(), order.end(), [&](size_t x, size_t y) { return shape(x) < shape(y); });
  std::vector<Plan::Group> groups;
  for (size_t o = 0; o < order.size(); ++o) {
    const size_t mi = order[o];
    const ramgpu_ctx *c = b->m[mi];
    int rows = 0;
    if (grouped) {
      size_t lds = 0;
      rows = shape_of(c, &lds).rows;
      const std::pair<int, int> h = shape(mi);
      if (o == 0 || shape(order[o - 1]) != h)
        groups.push_back(Plan::Group{StepShape{h.second, h.first}, 0, (int)vmap.size(), 0});
      groups.back().lds = std::max(groups.back().lds, lds);
    }
    const int nsp = per_member(kind) ? 1 : c->ns;
    const int nb = blocks_of(b, kind, c);
    if (nb >= (1 << kVmapShift) || jobs.size() + nsp >= (1u << (31 - kVmapShift)))
      return fail(RAMGPU_EINVAL, "ensemble too large for the launch tables");
    const int j0 = (int)jobs.size();
    for (int s = 0; s < nsp; ++s) jobs.push_back(Job{(int)mi, s, (int)vmap.size(), nb, rows});
    if (kind == BK_PLANE || kind == BK_PLB) {
      // the species of each run of 8 planes in turn: a plane's species land
      // on one XCD, whose L2 serves them the plane's tables (Launch::ilv)
      for (int g = 0; g < nb; g += 8)
        for (int s = 0; s < nsp; ++s)
          for (int x = g; x < std::min(nb, g + 8); ++x) vmap.push_back(vmap_entry(j0 + s, x));
    } else {
      for (int s = 0; s < nsp; ++s)
        for (int x = 0; x < nb; ++x) vmap.push_back(vmap_entry(j0 + s, x));
    }
    if (grouped) groups.back().nv = (int)vmap.size() - groups.back().v0;
  }
  b->plan[kind].groups = groups;
  Plan &p = b->plan[kind];
  int rc;
  if ((rc = batch_alloc(b, (void **)&p.jobs, jobs.size() * sizeof(Job))) ||
      (rc = batch_alloc(b, (void **)&p.vmap, vmap.size() * sizeof(int))))
    return rc;
  HIP_TRY(hipMemcpy(p.jobs, jobs.data(), jobs.size() * sizeof(Job), hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(p.vmap, vmap.data(), vmap.size() * sizeof(int), hipMemcpyHostToDevice));
  p.nv = (int)vmap.size();
  return RAMGPU_OK;
}

Launch launch_for(const ramgpu_batch *b, int kind) {
  const Plan &p = b->plan[kind];
  Launch L{};
  L.tabs = b->d_tabs;
  L.jobs = p.jobs;
  L.vmap = p.vmap;
  L.nv = p.nv;
  return L;
}

unsigned grid_for(const ramgpu_batch *b, int kind) {
  const Plan &p = b->plan[kind];
  return (unsigned)((p.cap > 0 && p.cap < p.nv) ? p.cap : p.nv);
}

// The fused plane kernel of every member.
void enq_planes(ramgpu_batch *b, int kind, int seq, Launch L, int rec) {
  const Plan &p = b->plan[kind];
  const int *vmap = L.vmap;
  for (const Plan::Group &g : p.groups) {
    L.vmap = vmap + g.v0;
    L.nv = g.nv;
    const int grid = (p.cap > 0 && p.cap < g.nv) ? p.cap : g.nv;
    launch_step(seq, g.sh, dim3((unsigned)grid), g.lds, b->stream, L, rec);
  }
}

// DRIFTR or DRIFTP (kind BK_P or BK_POOP) of every member.  L: the launch's
// slots.
void enq_lines(ramgpu_batch *b, int kind, Launch L, int mode) {
  const Plan &p = b->plan[kind];
  L.jobs = p.jobs;
  for (const Plan::Group &g : p.groups) {
    L.vmap = p.vmap + g.v0;
    L.nv = g.nv;
    const int grid = (p.cap > 0 && p.cap < g.nv) ? p.cap : g.nv;
    const LineShape sh{g.sh.rows, g.sh.threads, g.lds};
    if (kind == BK_R) launch_r(mode, sh, dim3((unsigned)grid), b->stream, L);
    else launch_p(mode, sh, dim3((unsigned)grid), b->stream, L);
  }
}
void enq_r(ramgpu_batch *b, Launch L, int mode) {
  if (mode == 2 || b->chunks) return enq_lines(b, BK_R, L, mode);
  const Plan &p = b->plan[BK_RB];
  L.jobs = p.jobs;
  L.vmap = p.vmap;
  L.nv = p.nv;
  const int cap = b->plan[BK_R].cap, grid = (cap > 0 && cap < p.nv) ? cap : p.nv;
  launch_r(mode, {0, kLineThreads, b->radial_lds}, dim3((unsigned)grid), b->stream, L);
}

void destroy_graphs(ramgpu_batch *b) {
  for (auto &e : b->exec)
    if (e) {
      (void)hipGraphExecDestroy(e);
      e = nullptr;
    }
}

// Bring every member's tables up to date on its own stream and refresh the
// device copies of the member descriptors.
int sync_members(ramgpu_batch *b) {
  int rc;
  std::vector<Tab> tabs;
  for (size_t m = 0; m < b->m.size(); ++m) {
    ramgpu_ctx *c = b->m[m];
    if ((rc = check_ctx(c)) || (rc = forward_only(c)) || (rc = prepare(c))) return rc;
    if (c->plane.threads > b->plane.threads || c->plane.maxc > b->plane.maxc)
      return fail(RAMGPU_ESTATE, "member %zu changed its plane shape after joining the ensemble", m);
    if ((char)takes_wave(c) != b->wave[m])
      return fail(RAMGPU_ESTATE, "member %zu switched WAVELO after joining the ensemble", m);
    HIP_TRY(hipStreamSynchronize(c->stream));
    tabs.push_back(c->t);
  }
  HIP_TRY(hipSetDevice(b->device));
  HIP_TRY(hipMemcpy(b->d_tabs, tabs.data(), tabs.size() * sizeof(Tab), hipMemcpyHostToDevice));
  return RAMGPU_OK;
}

// Event pair around one launch of kind `kind` while timing is on.
void btbeg(ramgpu_batch *b, int kind) {
  if (!b->timing) return;
  if (2 * b->tused + 2 > b->tev.size()) {
    for (int n = 0; n < 2; ++n) {
      hipEvent_t e;
      if (hipEventCreate(&e) != hipSuccess) {
        b->timing = false;
        return;
      }
      b->tev.push_back(e);
    }
  }
  if (b->tkind.size() < b->tused + 1) b->tkind.resize(b->tused + 1);
  b->tkind[b->tused] = kind;
  (void)hipEventRecord(b->tev[2 * b->tused], b->stream);
}

void btend(ramgpu_batch *b) {
  if (!b->timing) return;
  (void)hipEventRecord(b->tev[2 * b->tused + 1], b->stream);
  ++b->tused;
}

// The launches of one ensemble step.  sched: VT / boundary scale of the step
// from the device schedule, then the VT-dependent tables and the ghost carry.
// CFL limits are recorded every step (the same values a member's own
// ram_run reports).
int enqueue_step(ramgpu_batch *b, bool sched) {
  hipStream_t st = b->stream;
  const int M = (int)b->m.size();
  if (sched) {
    btbeg(b, RAMGPU_KERNEL_PREPARE);
    const Launch ls = launch_for(b, BK_SCHED);
    hipLaunchKernelGGL(k_sched, dim3(grid_for(b, BK_SCHED)), dim3(256), 0, st, ls, (const double *)b->d_kp,
                       (const double *)b->d_bs, (const int *)b->d_bsoff, (const int *)b->d_step, M, b->sum_ns);
    const Launch lc = launch_for(b, BK_COEFIJ);
    hipLaunchKernelGGL(k_coef_ij, dim3(grid_for(b, BK_COEFIJ)), dim3(256), 0, st, lc, (const double *)nullptr,
                     (const double *)nullptr);
    const Launch lg = launch_for(b, BK_GHOST);
    hipLaunchKernelGGL(k_ghost, dim3(grid_for(b, BK_GHOST)), dim3(1024), b->ghost_lds, st, lg);
    btend(b);
  }
  const Launch lr = launch_for(b, BK_R), lp = launch_for(b, BK_P), lk = launch_for(b, BK_PLANE),
               lf = launch_for(b, BK_FIN);
  btbeg(b, RAMGPU_KERNEL_R);
  enq_r(b, lr, 1);
  btend(b);
  btbeg(b, RAMGPU_KERNEL_P);
  enq_lines(b, BK_P, lp, 1);
  btend(b);
  btbeg(b, RAMGPU_KERNEL_PLANE);
  enq_planes(b, BK_PLANE, SEQ_STEP, lk, 1);
  btend(b);
  btbeg(b, RAMGPU_KERNEL_P);
  enq_lines(b, BK_P, lp, 0);
  btend(b);
  btbeg(b, RAMGPU_KERNEL_R);
  enq_r(b, lr, 2);
  btend(b);
  btbeg(b, RAMGPU_KERNEL_FINALIZE);
  hipLaunchKernelGGL(k_finalize, dim3(grid_for(b, BK_FIN)), dim3(kFinalizeThreads), 0, st, lf, 15, 2);
  if (sched) hipLaunchKernelGGL(k_tick, dim3(1), dim3(64), 0, st, b->d_step);
  btend(b);
  return launch_check("ensemble step");
}


// ---- reverse mode ----------------------------------------------------------
// The launches of the ensemble adjoint name each member's buffers by tape
// slot (Launch::ssl/dsl, 1-based; 0 = the member's F2 as source, -1 as an
// out-of-place destination), so one launch serves members of any size.

Launch slot_launch(const ramgpu_batch *b, int kind, int ssl, int dsl, int bstep = 0) {
  Launch L = launch_for(b, kind);
  L.ssl = ssl;
  L.dsl = dsl;
  L.bstep = bstep;
  return L;
}

// VT / boundary scale of step `step` from the device schedule, then the
// VT-dependent tables and the ghost carry
void enq_sched(ramgpu_batch *b, int step) {
  hipStream_t st = b->stream;
  hipLaunchKernelGGL(k_setstep, dim3(1), dim3(64), 0, st, b->d_step, step);
  const Launch ls = launch_for(b, BK_SCHED);
  hipLaunchKernelGGL(k_sched, dim3(grid_for(b, BK_SCHED)), dim3(256), 0, st, ls, (const double *)b->d_kp,
                     (const double *)b->d_bs, (const int *)b->d_bsoff, (const int *)b->d_step, (int)b->m.size(),
                     b->sum_ns);
  const Launch lc = launch_for(b, BK_COEFIJ);
  hipLaunchKernelGGL(k_coef_ij, dim3(grid_for(b, BK_COEFIJ)), dim3(256), 0, st, lc, (const double *)nullptr,
                     (const double *)nullptr);
  const Launch lg = launch_for(b, BK_GHOST);
  hipLaunchKernelGGL(k_ghost, dim3(grid_for(b, BK_GHOST)), dim3(1024), b->ghost_lds, st, lg);
}

void enq_copy(ramgpu_batch *b, int ssl, int dsl) {
  const Launch L = slot_launch(b, BK_COPY, ssl, dsl);
  hipLaunchKernelGGL(k_copy_ens, dim3(L.nv), dim3(256), 0, b->stream, L);
}

void enq_misfit(ramgpu_batch *b, int ssl, int step, int adjoint) {
  const Launch L = slot_launch(b, BK_MEM, ssl, 0);
  hipLaunchKernelGGL(k_misfit_ens, dim3(L.nv, std::max(b->mpts_max, 1)), dim3(64), 0, b->stream, L, step, adjoint);
}

// One step with every operator's input on the tape group starting at slot g
// (0-based), the step's output to dsl_out; the arithmetic of enqueue_step.
// With bookkeeping false (a segment recomputed for its tape) the CFL limits
// and the SUMRC chain are not formed: only the states are needed.
void enq_taped_step(ramgpu_batch *b, int g, int dsl_out, bool bookkeeping = true) {
  hipStream_t st = b->stream;
  Launch L = slot_launch(b, BK_R, g + T_R1 + 1, g + T_P1 + 1);
  enq_r(b, L, bookkeeping ? 1 : 0);
  L = slot_launch(b, BK_POOP, g + T_P1 + 1, g + T_E1 + 1);
  enq_lines(b, BK_POOP, L, bookkeeping ? 1 : 0);
  L = slot_launch(b, BK_PLOOP, g + T_E1 + 1, g + T_P2 + 1);
  enq_planes(b, BK_PLOOP, SEQ_TAPE, L, bookkeeping ? 1 : 0);
  L = slot_launch(b, BK_POOP, g + T_P2 + 1, g + T_R2 + 1);
  enq_lines(b, BK_POOP, L, 0);
  L = slot_launch(b, BK_R, g + T_R2 + 1, dsl_out);
  enq_r(b, L, 2);
  if (bookkeeping) {
    const Launch lf = launch_for(b, BK_FIN);
    hipLaunchKernelGGL(k_finalize, dim3(grid_for(b, BK_FIN)), dim3(kFinalizeThreads), 0, st, lf, 15, 2);
  }
}

// adjoint of the step taped at group g: Tab::lam in place, Tab::bbar[step]
void enq_step_bwd(ramgpu_batch *b, int g, int step) {
  hipStream_t st = b->stream;
  Launch L = slot_launch(b, BK_RB, g + T_R2 + 1, 0, step);
  hipLaunchKernelGGL(k_r_bwd<1>, dim3(grid_for(b, BK_RB)), dim3(kLineThreads), b->radial_lds, st, L, nullptr, nullptr,
                     nullptr);
  L = slot_launch(b, BK_PB, g + T_P2 + 1, 0);
  hipLaunchKernelGGL(k_p_bwd, dim3(grid_for(b, BK_PB)), dim3(kLineThreads), b->azim_lds, st, L, nullptr, nullptr);
  L = slot_launch(b, BK_PLB, g + T_E1 + 1, 0);
  const int *vmap = L.vmap;
  for (const Plan::Group &gr : b->plan[BK_PLB].groups) {
    L.vmap = vmap + gr.v0;
    L.nv = gr.nv;
    launch_plane_adj(gr.sh, dim3((unsigned)gr.nv), gr.lds, st, L, nullptr, nullptr);
  }
  L = slot_launch(b, BK_PB, g + T_P1 + 1, 0);
  hipLaunchKernelGGL(k_p_bwd, dim3(grid_for(b, BK_PB)), dim3(kLineThreads), b->azim_lds, st, L, nullptr, nullptr);
  L = slot_launch(b, BK_RB, g + T_R1 + 1, 0, step);
  hipLaunchKernelGGL(k_r_bwd<0>, dim3(grid_for(b, BK_RB)), dim3(kLineThreads), b->radial_lds, st, L, nullptr, nullptr,
                     nullptr);
}

int ensure_graph(ramgpu_batch *b, bool sched) {
  hipGraphExec_t &e = b->exec[sched ? 1 : 0];
  if (e) return RAMGPU_OK;
  hipGraph_t g = nullptr;
  HIP_TRY(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
  const int rc = enqueue_step(b, sched);
  const hipError_t ec = hipStreamEndCapture(b->stream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (ec != hipSuccess) return fail(RAMGPU_EHIP, "graph capture failed: %s", hipGetErrorString(ec));
  const hipError_t ei = hipGraphInstantiate(&e, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (ei != hipSuccess) {
    e = nullptr;
    return fail(RAMGPU_EHIP, "graph instantiation failed: %s", hipGetErrorString(ei));
  }
  return RAMGPU_OK;
}

int run_steps(ramgpu_batch *b, int nsteps, bool sched) {
  int rc;
  const bool graph = b->use_graph && !b->timing;  // per-launch events need eager launches
  if (graph && (rc = ensure_graph(b, sched))) return rc;
  for (int n = 0; n < nsteps; ++n) {
    if (graph) {
      HIP_TRY(hipGraphLaunch(b->exec[sched ? 1 : 0], b->stream));
    } else if ((rc = enqueue_step(b, sched))) {
      return rc;
    }
  }
  return RAMGPU_OK;
}

int finish(ramgpu_batch *b, bool sched, ramgpu_species_out *out) {
  HIP_TRY(hipStreamSynchronize(b->stream));
  size_t o = 0;
  for (ramgpu_ctx *c : b->m) {
    if (sched) c->efield_dirty = true;  // VT and scales now those of the last step
    int rc = fill_out(c, out ? out + o : nullptr);
    if (rc) return rc;
    o += c->ns;
  }
  return RAMGPU_OK;
}

// Upload a per-member Kp / boundary-scale schedule of nsteps steps (bscale
// may be NULL: the members' current scales) and reset the step counter.
int load_schedule(ramgpu_batch *b, int nsteps, const double *kp, const double *bscale) {
  const int M = (int)b->m.size();
  int rc;
  if (nsteps > b->sched_cap) {
    // the graph reads the schedule buffers by address: rebuild it with them
    destroy_graphs(b);
    int cap = std::max(nsteps, 1);
    if ((rc = batch_alloc(b, (void **)&b->d_kp, (size_t)cap * M * sizeof(double))) ||
        (rc = batch_alloc(b, (void **)&b->d_bs, (size_t)cap * b->sum_ns * sizeof(double))))
      return rc;
    b->sched_cap = cap;
  }
  HIP_TRY(hipMemcpyAsync(b->d_kp, kp, (size_t)nsteps * M * sizeof(double), hipMemcpyHostToDevice, b->stream));
  if (bscale) {
    HIP_TRY(hipMemcpyAsync(b->d_bs, bscale, (size_t)nsteps * b->sum_ns * sizeof(double), hipMemcpyHostToDevice,
                           b->stream));
  } else {
    std::vector<double> cur((size_t)nsteps * b->sum_ns);
    for (int mi = 0; mi < M; ++mi) {
      std::vector<double> sc(b->m[mi]->ns);
      HIP_TRY(hipMemcpy(sc.data(), b->m[mi]->d_bscale, sc.size() * sizeof(double), hipMemcpyDeviceToHost));
      for (int n = 0; n < nsteps; ++n)
        for (int s = 0; s < b->m[mi]->ns; ++s) cur[(size_t)n * b->sum_ns + b->bs_off[mi] + s] = sc[s];
    }
    HIP_TRY(hipMemcpy(b->d_bs, cur.data(), cur.size() * sizeof(double), hipMemcpyHostToDevice));
  }
  const int zero = 0;
  HIP_TRY(hipMemcpyAsync(b->d_step, &zero, sizeof(int), hipMemcpyHostToDevice, b->stream));
  HIP_TRY(hipStreamSynchronize(b->stream));
  return RAMGPU_OK;
}

int check_batch(ramgpu_batch *b) {
  if (!b) return fail(RAMGPU_EINVAL, "null ensemble");
  HIP_TRY(hipSetDevice(b->device));
  return RAMGPU_OK;
}

}  // namespace

extern "C" {

int ramgpu_batch_create(ramgpu_batch **out, ramgpu_ctx *const *members, int nmembers) {
  if (!out) return fail(RAMGPU_EINVAL, "null output pointer");
  *out = nullptr;
  if (!members || nmembers < 1) return fail(RAMGPU_EINVAL, "an ensemble needs at least one member");
  const int dev = members[0] ? members[0]->device : -1;
  for (int i = 0; i < nmembers; ++i) {
    if (!members[i]) return fail(RAMGPU_EINVAL, "member %d is null", i);
    if (members[i]->device != dev) return fail(RAMGPU_EINVAL, "member %d is on another device", i);
    for (int j = 0; j < i; ++j)
      if (members[j] == members[i]) return fail(RAMGPU_EINVAL, "member %d appears twice", i);
    const int rc = forward_only(members[i]);
    if (rc) return rc;
  }
  HIP_TRY(hipSetDevice(dev));
  ramgpu_batch *b = new ramgpu_batch();
  b->device = dev;
  b->m.assign(members, members + nmembers);
  auto cleanup = [&](int code) {
    ramgpu_batch_destroy(b);
    return code;
  };
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) == hipSuccess) b->ncu = prop.multiProcessorCount;
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&b->ev0) != hipSuccess || hipEventCreate(&b->ev1) != hipSuccess)
    return cleanup(fail(RAMGPU_EHIP, "stream/event creation failed"));
  int rc;
  if ((rc = batch_alloc(b, (void **)&b->d_tabs, nmembers * sizeof(Tab)))) return cleanup(rc);
  long lines = 0;
  for (ramgpu_ctx *c : b->m) {
    b->bs_off.push_back(b->sum_ns);
    b->sum_ns += c->ns;
    b->radial_lds = std::max(b->radial_lds, radial_lds_bytes(c->nr, c->ne, c->npa));
    b->azim_lds = std::max(b->azim_lds, azim_lds_bytes(c->nt, c->ne, c->npa));
    b->ghost_lds = std::max(b->ghost_lds, (size_t)4 * c->nt * sizeof(double));
    b->plane.threads = std::max(b->plane.threads, c->plane.threads);
    b->plane.maxc = std::max(b->plane.maxc, c->plane.maxc);
    b->wave.push_back((char)takes_wave(c));
    lines += (long)c->ns * std::max(c->nt, c->nr - 1) * c->ne * c->npa;
  }
  b->chunks = lines <= line_rows_max(b->ncu);
  if ((rc = batch_alloc(b, (void **)&b->d_bsoff, nmembers * sizeof(int))) ||
      (rc = batch_alloc(b, (void **)&b->d_step, sizeof(int))))
    return cleanup(rc);
  if (hipMemcpy(b->d_bsoff, b->bs_off.data(), nmembers * sizeof(int), hipMemcpyHostToDevice) != hipSuccess)
    return cleanup(fail(RAMGPU_EHIP, "hipMemcpy failed"));
  for (int k = 0; k < BK_N; ++k)
    if ((rc = build_plan(b, k))) return cleanup(rc);
  *out = b;
  return RAMGPU_OK;
}

int ramgpu_batch_destroy(ramgpu_batch *b) {
  if (!b) return RAMGPU_OK;
  (void)hipSetDevice(b->device);
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  destroy_graphs(b);
  for (void *p : b->allocs) (void)hipFree(p);
  for (hipEvent_t e : b->tev) (void)hipEventDestroy(e);
  if (b->ev0) (void)hipEventDestroy(b->ev0);
  if (b->ev1) (void)hipEventDestroy(b->ev1);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  delete b;
  return RAMGPU_OK;
}

int ramgpu_batch_use_graph(ramgpu_batch *b, int enable) {
  int rc = check_batch(b);
  if (rc) return rc;
  b->use_graph = enable != 0;
  return RAMGPU_OK;
}

int ramgpu_batch_ram_run(ramgpu_batch *b, int nsteps, ramgpu_species_out *out) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (nsteps < 0) return fail(RAMGPU_EINVAL, "nsteps < 0");
  if ((rc = sync_members(b))) return rc;
  HIP_TRY(hipEventRecord(b->ev0, b->stream));
  if ((rc = run_steps(b, nsteps, false))) return rc;
  HIP_TRY(hipEventRecord(b->ev1, b->stream));
  return finish(b, false, out);
}

int ramgpu_batch_ram_run_schedule(ramgpu_batch *b, int nsteps, const double *kp, const double *bscale,
                                  ramgpu_species_out *out) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (nsteps < 0) return fail(RAMGPU_EINVAL, "nsteps < 0");
  if (!kp) return fail(RAMGPU_EINVAL, "kp schedule is null");
  for (size_t mi = 0; mi < b->m.size(); ++mi)
    if (!b->m[mi]->have_lzphi)
      return fail(RAMGPU_ESTATE, "member %zu: ramgpu_set_kp(lz, phi) must precede a Kp schedule", mi);
  if ((rc = load_schedule(b, nsteps, kp, bscale))) return rc;
  if ((rc = sync_members(b))) return rc;
  HIP_TRY(hipEventRecord(b->ev0, b->stream));
  if ((rc = run_steps(b, nsteps, true))) return rc;
  HIP_TRY(hipEventRecord(b->ev1, b->stream));
  return finish(b, true, out);
}

int ramgpu_batch_kernel_timing(ramgpu_batch *b, int enable) {
  int rc = check_batch(b);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(b->stream));
  b->timing = enable != 0;
  b->tused = 0;
  return RAMGPU_OK;
}

int ramgpu_batch_kernel_times(ramgpu_batch *b, double *total_ms, int *launches) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!total_ms || !launches) return fail(RAMGPU_EINVAL, "null output array");
  HIP_TRY(hipStreamSynchronize(b->stream));
  for (int k = 0; k < RAMGPU_KERNEL_KINDS; ++k) {
    total_ms[k] = 0.0;
    launches[k] = 0;
  }
  for (size_t n = 0; n < b->tused; ++n) {
    float f = 0.f;
    HIP_TRY(hipEventElapsedTime(&f, b->tev[2 * n], b->tev[2 * n + 1]));
    total_ms[b->tkind[n]] += f;
    launches[b->tkind[n]] += 1;
  }
  b->tused = 0;
  return RAMGPU_OK;
}

int ramgpu_batch_last_run_ms(ramgpu_batch *b, double *ms) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!ms) return fail(RAMGPU_EINVAL, "ms is null");
  HIP_TRY(hipEventSynchronize(b->ev1));
  float f = 0.f;
  HIP_TRY(hipEventElapsedTime(&f, b->ev0, b->ev1));
  *ms = f;
  return RAMGPU_OK;
}

// Reverse mode of an ensemble: the flux-misfit gradient of every member
// (ramgpu_adjoint_run for each member, all members in the same launches).
// Tape slots of member m, each one F2 of that member: nseg checkpoints,
// then either one tape group per step of a segment (the segment is taped in
// one recomputation) or, when that does not fit the device, seglen states
// plus one group (the segment's states are recomputed, then each step is
// re-taped just before its adjoint).  The arithmetic is the same either way.
int ramgpu_batch_adjoint_run(ramgpu_batch *b, int nsteps, int ckpt_every, const double *kp, const double *bscale,
                             const int *npts, const int *const *pts, const double *const *w,
                             const double *const *target, double *loss, double *const *grad_f2,
                             double *const *grad_fgeos) {
  int rc = check_batch(b);
  if (rc) return rc;
  const int M = (int)b->m.size();
  if (nsteps < 1 || ckpt_every < 1) return fail(RAMGPU_EINVAL, "nsteps and ckpt_every must be >= 1");
  if (!kp) return fail(RAMGPU_EINVAL, "kp schedule is null");
  if (!npts || !pts || !w || !target) return fail(RAMGPU_EINVAL, "misfit points, weights and targets required");
  for (int mi = 0; mi < M; ++mi) {
    const ramgpu_ctx *c = b->m[mi];
    if (!c->have_lzphi) return fail(RAMGPU_ESTATE, "member %d: ramgpu_set_kp(lz, phi) must precede a Kp schedule", mi);
    if (npts[mi] < 1 || !pts[mi] || !w[mi] || !target[mi])
      return fail(RAMGPU_EINVAL, "member %d: misfit points, weights and targets required", mi);
    for (int p = 0; p < npts[mi]; ++p) {
      const int *q = pts[mi] + 4 * p;
      if (q[0] < 1 || q[0] > c->ns || q[1] < 1 || q[1] > c->nr || q[2] < 1 || q[2] > c->nt || q[3] < 1 ||
          q[3] > c->ne)
        return fail(RAMGPU_EINVAL, "member %d: misfit point %d outside the grid", mi, p);
    }
  }
  const int nseg = (nsteps + ckpt_every - 1) / ckpt_every, seglen = std::min(ckpt_every, nsteps);
  set_plane_bwd_lds_limit(b->m[0]->lds_limit);
  // memory plan
  size_t nall = 0, ngall = 0;
  for (ramgpu_ctx *c : b->m) {
    nall += (size_t)c->ns * c->nr * c->nt * c->ne * c->npa;
    ngall += (size_t)c->ns * c->nt * c->ne * c->npa;
  }
  size_t freeb = 0, totb = 0;
  HIP_TRY(hipMemGetInfo(&freeb, &totb));
  freeb += dev_cached(b->device);  // blocks kept from earlier calls serve this one or are given back
  const size_t fixed = 8 * (2 * nall + (grad_fgeos ? (size_t)nsteps * ngall : 0)) + ((size_t)64 << 20);
  const size_t one = (size_t)(nseg + seglen * T_N) * nall * 8, two = (size_t)(nseg + seglen + T_N) * nall * 8;
  // two-level: states, then one re-taped step at a time (forced with
  // RAMGPU_ADJOINT_RETAPE=1, which tests the scheme on small ensembles)
  const char *force = getenv("RAMGPU_ADJOINT_RETAPE");
  bool split;
  if (force && force[0] == '1' && fixed + two <= freeb * 0.92) split = true;
  else if (fixed + one <= freeb * 0.92) split = false;
  else if (fixed + two <= freeb * 0.92) split = true;
  else return fail(RAMGPU_ENOMEM, "ensemble adjoint needs %.1f GB, %.1f GB free", (fixed + two) / 1e9, freeb / 1e9);
  const int nslots = split ? nseg + seglen + T_N : nseg + seglen * T_N;
  const int CK = 0, ST = nseg, TG = split ? nseg + seglen : nseg;
  auto group = [&](int s, int n0) { return split ? TG : TG + (s - n0) * T_N; };
  // buffers
  std::vector<std::pair<void *, size_t>> bufs;
  auto release = [&]() {
    (void)hipStreamSynchronize(b->stream);
    for (const auto &q : bufs) dev_give(b->device, q.first, q.second);
    bufs.clear();
  };
  auto alloc = [&](void **q, size_t bytes) {
    bytes = std::max<size_t>(bytes, 16);
    if (!dev_take(b->device, q, bytes)) return false;
    bufs.emplace_back(*q, bytes);
    return true;
  };
  std::vector<double *> fin(M), fin_e(M);
  for (int mi = 0; mi < M; ++mi) {
    ramgpu_ctx *c = b->m[mi];
    const size_t n = (size_t)c->ns * c->nr * c->nt * c->ne * c->npa, ng = (size_t)c->ns * c->nt * c->ne * c->npa;
    const size_t np = npts[mi];
    void *tape, *lam, *bb = nullptr, *mp, *mw, *mt, *ml, *f, *fe;
    if (!alloc(&tape, (size_t)nslots * n * 8) || !alloc(&lam, n * 8) ||
        (grad_fgeos && grad_fgeos[mi] && !alloc(&bb, (size_t)nsteps * ng * 8)) || !alloc(&mp, np * 4 * sizeof(int)) ||
        !alloc(&mw, np * c->npa * 8) || !alloc(&mt, (size_t)nsteps * np * 8) || !alloc(&ml, (size_t)nsteps * np * 8) ||
        !alloc(&f, n * 8) || !alloc(&fe, (size_t)c->ns * 4 * 8)) {
      release();
      return fail(RAMGPU_ENOMEM, "ensemble adjoint: hipMalloc failed (member %d)", mi);
    }
    HIP_TRY(hipMemcpy(mp, pts[mi], np * 4 * sizeof(int), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(mw, w[mi], np * c->npa * 8, hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(mt, target[mi], (size_t)nsteps * np * 8, hipMemcpyHostToDevice));
    c->t.tape = (double *)tape;
    c->t.lam = (double *)lam;
    c->t.bbar = (double *)bb;
    c->t.mpts = (const int *)mp;
    c->t.mw = (const double *)mw;
    c->t.mtarget = (const double *)mt;
    c->t.mloss = (double *)ml;
    c->t.mnpts = (int)np;
    b->mpts_max = std::max(b->mpts_max, (int)np);
    fin[mi] = (double *)f;
    fin_e[mi] = (double *)fe;
  }
  auto detach = [&]() {  // the members' descriptors no longer name the buffers
    for (ramgpu_ctx *c : b->m) {
      c->t.tape = c->t.lam = c->t.bbar = c->t.mloss = nullptr;
      c->t.mpts = nullptr;
      c->t.mw = c->t.mtarget = nullptr;
      c->t.mnpts = 0;
      c->tab_dirty = true;
      c->efield_dirty = true;  // VT and scales are those of the schedule
    }
    release();
    return sync_members(b);
  };
  if ((rc = load_schedule(b, nsteps, kp, bscale)) || (rc = sync_members(b))) {
    detach();
    return rc;
  }
  hipStream_t st = b->stream;
  const int nlast0 = (nseg - 1) * ckpt_every;
  HIP_TRY(hipEventRecord(b->ev0, st));
  // forward, keeping a checkpoint at the start of every segment; the last
  // segment is taped at once when whole segments are taped
  for (int s = 0; s < nsteps; ++s) {
    enq_sched(b, s);
    if (!split && s >= nlast0) {
      if (s == nlast0) enq_copy(b, 0, group(s, nlast0) + T_R1 + 1);
      const int out = (s == nsteps - 1) ? -1 : group(s + 1, nlast0) + T_R1 + 1;
      enq_taped_step(b, group(s, nlast0), out);
      enq_misfit(b, out < 0 ? 0 : out, s, 0);
    } else {
      if (s % ckpt_every == 0) enq_copy(b, 0, CK + s / ckpt_every + 1);
      enqueue_step(b, false);
      enq_misfit(b, 0, s, 0);
    }
  }
  for (int mi = 0; mi < M; ++mi) {
    ramgpu_ctx *c = b->m[mi];
    const size_t n = (size_t)c->ns * c->nr * c->nt * c->ne * c->npa;
    HIP_TRY(hipMemcpyAsync(fin[mi], c->t.f2, n * 8, hipMemcpyDeviceToDevice, st));
    HIP_TRY(hipMemcpyAsync(fin_e[mi], c->t.energy, (size_t)c->ns * 32, hipMemcpyDeviceToDevice, st));
    const size_t ng = (size_t)c->ns * c->nt * c->ne * c->npa;
    hipLaunchKernelGGL(k_fill, dim3(1024), dim3(256), 0, st, c->t.lam, 0.0, n);
    if (c->t.bbar) hipLaunchKernelGGL(k_fill, dim3(1024), dim3(256), 0, st, c->t.bbar, 0.0, (size_t)nsteps * ng);
  }
  // backward, segment by segment
  for (int g = nseg - 1; g >= 0; --g) {
    const int n0 = g * ckpt_every, n1 = std::min(nsteps, n0 + ckpt_every);
    auto out_of = [&](int s) { return (s == n1 - 1) ? -1 : (split ? ST + (s + 1 - n0) + 1 : group(s + 1, n0) + T_R1 + 1); };
    if (split) {  // the segment's states
      enq_copy(b, CK + g + 1, -1);
      for (int s = n0; s < n1; ++s) {
        enq_copy(b, 0, ST + (s - n0) + 1);
        enq_sched(b, s);
        enqueue_step(b, false);
      }
    } else if (g < nseg - 1) {  // the segment taped
      enq_copy(b, CK + g + 1, group(n0, n0) + T_R1 + 1);
      for (int s = n0; s < n1; ++s) {
        enq_sched(b, s);
        enq_taped_step(b, group(s, n0), out_of(s), false);
      }
    }
    for (int s = n1 - 1; s >= n0; --s) {
      const int out = out_of(s);
      if (split) {
        enq_copy(b, ST + (s - n0) + 1, TG + T_R1 + 1);
        enq_sched(b, s);
        enq_taped_step(b, TG, out, false);  // rewrites the step's output with the same values
      } else {
        enq_sched(b, s);
      }
      enq_misfit(b, out < 0 ? 0 : out, s, 1);
      enq_step_bwd(b, group(s, n0), s);
    }
    if ((rc = launch_check("ensemble adjoint"))) {
      detach();
      return rc;
    }
  }
  HIP_TRY(hipEventRecord(b->ev1, st));
  enq_sched(b, nsteps - 1);  // the members keep the inputs of the last step
  // results; the members are left in the state after the run
  for (int mi = 0; mi < M; ++mi) {
    ramgpu_ctx *c = b->m[mi];
    const size_t n = (size_t)c->ns * c->nr * c->nt * c->ne * c->npa, ng = (size_t)c->ns * c->nt * c->ne * c->npa;
    const size_t np = npts[mi];
    HIP_TRY(hipMemcpyAsync(c->t.f2, fin[mi], n * 8, hipMemcpyDeviceToDevice, st));
    HIP_TRY(hipMemcpyAsync(c->t.energy, fin_e[mi], (size_t)c->ns * 32, hipMemcpyDeviceToDevice, st));
    std::vector<double> lv((size_t)nsteps * np);
    HIP_TRY(hipMemcpyAsync(lv.data(), c->t.mloss, lv.size() * 8, hipMemcpyDeviceToHost, st));
    HIP_TRY(hipStreamSynchronize(st));
    if (loss) {
      double tot = 0.0;
      for (double v : lv) tot += v;
      loss[mi] = tot;
    }
    if (grad_f2 && grad_f2[mi]) {
      HIP_TRY(hipStreamSynchronize(c->stream));
      if ((rc = download_f2(c, grad_f2[mi], c->t.lam))) {
        detach();
        return rc;
      }
    }
    if (c->t.bbar) {
      if ((rc = copy_to_host(b->device, st, grad_fgeos[mi], c->t.bbar, (size_t)nsteps * ng * 8))) {
        detach();
        return rc;
      }
    }
  }
  return detach();
}

// Autotuner: for each sweep kernel (R, P, plane) time the launches of every
// candidate grid -- one block per unit, or 1, 2, 4, 8 resident blocks per CU
// looping over the units -- and keep the fastest.  The members' F2 and
// energy records are saved before and restored after, so tuning leaves the
// ensemble's state unchanged.  ms_best (may be NULL) receives the best
// per-launch times of R, P and plane.
int ramgpu_batch_autotune(ramgpu_batch *b, int reps, double *ms_best) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (reps < 1) reps = 1;
  if ((rc = sync_members(b))) return rc;
  // save state
  std::vector<void *> saved;
  auto release = [&]() {
    for (void *p : saved) (void)hipFree(p);
  };
  for (ramgpu_ctx *c : b->m) {
    const size_t nf = f2_species_stride(c->t) * c->ns * sizeof(double), ne = (size_t)c->ns * 4 * sizeof(double);
    void *p = nullptr, *q = nullptr;
    if (!dev_malloc(b->device, &p, nf) || !dev_malloc(b->device, &q, ne)) {
      if (p) (void)hipFree(p);
      release();
      return fail(RAMGPU_ENOMEM, "autotune: no room to save the state");
    }
    saved.push_back(p);
    saved.push_back(q);
    HIP_TRY(hipMemcpyAsync(p, c->t.f2, nf, hipMemcpyDeviceToDevice, b->stream));
    HIP_TRY(hipMemcpyAsync(q, c->t.energy, ne, hipMemcpyDeviceToDevice, b->stream));
  }
  const int kinds[3] = {BK_R, BK_P, BK_PLANE};
  const int mult[5] = {0, 1, 2, 4, 8};
  hipEvent_t e0 = b->ev0, e1 = b->ev1;
  for (int ki = 0; ki < 3 && rc == RAMGPU_OK; ++ki) {
    const int kind = kinds[ki];
    Plan &p = b->plan[kind];
    float best = 1e30f;
    int best_cap = 0;
    for (int mi = 0; mi < 5; ++mi) {
      p.cap = mult[mi] * b->ncu;
      const Launch L = launch_for(b, kind);
      float tot = 0.f;
      for (int r = 0; r <= reps; ++r) {  // first launch warms up
        (void)hipEventRecord(e0, b->stream);
        if (kind == BK_R) {  // a step's two launches, by their own dispatch
          enq_r(b, L, 0);
          enq_r(b, L, 2);
        } else if (kind == BK_P)
          enq_lines(b, BK_P, L, 0);
        else
          enq_planes(b, kind, SEQ_STEP, L, 0);
        (void)hipEventRecord(e1, b->stream);
        if (hipEventSynchronize(e1) != hipSuccess) {
          rc = fail(RAMGPU_EHIP, "autotune launch failed");
          break;
        }
        float ms = 0.f;
        (void)hipEventElapsedTime(&ms, e0, e1);
        if (r > 0) tot += kind == BK_R ? 0.5f * ms : ms;
      }
      if (rc) break;
      const float avg = tot / reps;
      if (avg < best) {
        best = avg;
        best_cap = p.cap;
      }
    }
    p.cap = best_cap;
    if (ms_best) ms_best[ki] = best;
  }
  // restore state; the tuned shapes change the captured graphs
  size_t o = 0;
  for (ramgpu_ctx *c : b->m) {
    const size_t nf = f2_species_stride(c->t) * c->ns * sizeof(double), ne = (size_t)c->ns * 4 * sizeof(double);
    (void)hipMemcpyAsync(c->t.f2, saved[o], nf, hipMemcpyDeviceToDevice, b->stream);
    (void)hipMemcpyAsync(c->t.energy, saved[o + 1], ne, hipMemcpyDeviceToDevice, b->stream);
    o += 2;
  }
  (void)hipStreamSynchronize(b->stream);
  release();
  destroy_graphs(b);
  return rc;
}

// Grid caps in use: caps[0..2] for R, P, plane (0 = one block per unit).
int ramgpu_batch_get_shapes(ramgpu_batch *b, int *caps) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!caps) return fail(RAMGPU_EINVAL, "caps is null");
  caps[0] = b->plan[BK_R].cap;
  caps[1] = b->plan[BK_P].cap;
  caps[2] = b->plan[BK_PLANE].cap;
  return RAMGPU_OK;
}

int ramgpu_batch_set_shapes(ramgpu_batch *b, const int *caps) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!caps) return fail(RAMGPU_EINVAL, "caps is null");
  for (int i = 0; i < 3; ++i)
    if (caps[i] < 0) return fail(RAMGPU_EINVAL, "negative grid cap");
  b->plan[BK_R].cap = caps[0];
  b->plan[BK_P].cap = caps[1];
  b->plan[BK_PLANE].cap = caps[2];
  destroy_graphs(b);
  return RAMGPU_OK;
}

}  // extern "C"
