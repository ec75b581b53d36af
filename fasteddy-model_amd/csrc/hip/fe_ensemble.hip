/*
 * fe_ensemble.hip -- batched ensemble of unevenly sized LES members on one GPU.
 *
 * The reference advances one model per process: cuda_timeIntDeviceCommence
 * (SRC/TIME_INTEGRATION/CUDA/cuda_timeIntDevice.cu:105-157) launches every tendency
 * kernel of every RK stage over that model's grid, with the launch geometry of
 * SRC/FECUDA/fecuda_Device.cu:110-128.  Small members leave most of an MI355X idle
 * (a 96 x 96 x 64 member is 24 tiles of 64 x 8 columns for 256 compute units), so here
 * all members advance together:
 *   - each member is set up by the plain path (host modules, cuda_gridInit,
 *     cuda_hydroCoreInit, cuda_timeIntInit), then fe_ens_add_member moves its device
 *     state, profiles and surface planes into the ensemble and records its per-stage
 *     kernel arguments (StepArgs) in a device table, one row per member and stage;
 *   - one persistent stage kernel per RK stage (one work-group per compute unit, as
 *     many as the LDS allows) pulls (member, tile, z segment) work items from eight
 *     queues, one per XCD: a work-group serves its own XCD's queue first (the queues
 *     hold contiguous runs of one member's tiles, so neighbours share that XCD's L2)
 *     and then takes what is left in the others;
 *   - the work item runs exactly the tile body of the plain stage kernels
 *     (stage_body / stage_plain_body), with the member's arguments read through the
 *     constant address space, so every member gets the arithmetic of a plain run;
 *   - one RK3 step (counter reset, surface-layer pass, three stage launches, and a
 *     kernel that advances each member's step index, time and microphysics cadence in
 *     the table) is captured once in a hipGraph and replayed per step;
 *   - an autotuner chooses the z-segment length of each member shape (the third
 *     dimension of the TX x TY x L work tile) by timing graph replays.
 * fe_ens_steps_sequential runs the same members one after another through the plain
 * launches (one grid per member and stage, as cuda_timeIntCommence does); the baseline the
 * ensemble is timed against makes the same launches with each grid's plain z segments.
 */


namespace {

struct Member {
  int Nx = 0, Ny = 0, Nz = 0, P = 0, NF = 0, nseg = 1, zseg = 0, ntx = 0, nty = 0, mptf = 0;
  int nseg_plain = 1, zseg_plain = 0;   /* the plain path's own segments for this grid (timed baseline) */
  bool seg_set = false;                 /* segments set by amd_zSegments, fe_ens_set_segments or the autotuner */
  long fs = 0, ps = 0;
  float *S[3] = {nullptr, nullptr, nullptr};
  float *prof = nullptr, *surf = nullptr;
  StepArgs args[3];
};

struct Ens {
  std::vector<Member> mem;
  Variant var;
  bool have_var = false;
  int phys[3] = {0, 0, 0}, surf[3] = {0, 0, 0};
  hipStream_t stream = nullptr;
  StepArgs *dtab = nullptr;
  int *dmptf = nullptr;
  EnsItem *ditems = nullptr;
  size_t nitems_cap = 0;
  unsigned *dctr = nullptr;
  EnsQueues Q;
  int nwg = 0;
  bool seg_old = false;         /* members came since the default segments were chosen */
  bool dirty = true;            /* work items or kernel arguments changed: rebuild and recapture */
  bool host_tab_newer = false;  /* the host rows advanced (sequential steps): upload before a replay */
  hipGraph_t graph = nullptr;
  hipGraphExec_t gexec = nullptr;
  std::string report;
} E;

void ens_host_advance(Member &m) {
  for (int s = 0; s < 3; ++s) {
    StepArgs &a = m.args[s];
    a.step_it = a.step_it + 1;
    a.simTime = a.simTime + a.dt;
    if (m.mptf > 0) a.mpActive = (a.step_it % m.mptf) == 0;
  }
}

void ens_set_segments(Member &m, int n) {
  n = std::max(1, std::min(n, (m.Nz + 1) / 2));
  seg_shape(m.Nz, n, m.zseg, m.nseg);
  for (int s = 0; s < 3; ++s) m.args[s].zseg = m.zseg;
  E.dirty = true;
}

/* Work-groups the chip holds at once: the persistent grid. */
int ens_slots() {
  int dev = 0, ncu = 256;
  hipDeviceProp_t pr;
  if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&pr, dev) == hipSuccess && pr.multiProcessorCount > 0)
    ncu = pr.multiProcessorCount;
  int o1 = 0, o2 = 0, occ = 1;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&o1, E.var.ens_phys, NT, 0) == hipSuccess &&
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&o2, E.var.ens_plain, NT, 0) == hipSuccess)
    occ = std::max(1, std::min(o1, o2));
  return ncu * occ;
}

/* Segments of the members that have none set, chosen for all members together. */
void ens_default_segments() {
  if (!E.seg_old) return;
  E.seg_old = false;
  std::vector<SegMember> mem;
  for (auto &m : E.mem)
    mem.push_back(SegMember{(long)((m.Nx + TX - 1) / TX) * ((m.Ny + TY - 1) / TY), m.Nz, m.seg_set ? m.zseg : 0});
  const int len = ens_segment_length(mem, ens_slots());
  for (auto &m : E.mem)
    if (!m.seg_set) ens_set_segments(m, (m.Nz + len - 1) / len);
}

int ens_drop_graph() {
  if (E.gexec) { HIPCHK(hipGraphExecDestroy(E.gexec)); E.gexec = nullptr; }
  if (E.graph) { HIPCHK(hipGraphDestroy(E.graph)); E.graph = nullptr; }
  return FE_OK;
}

/* One RK3 step of every member on E.stream (captured into the graph). */
int ens_enqueue_step() {
  const int nm = (int)E.mem.size();
  int mx = 0, my = 0;
  for (auto &m : E.mem) { mx = std::max(mx, m.Nx); my = std::max(my, m.Ny); }
  hipLaunchKernelGGL(ens_reset, dim3(1), dim3(64), 0, E.stream, E.dctr, 3 * ENS_NQ);
  for (int s = 0; s < 3; ++s) {
    if (E.surf[s])
      hipLaunchKernelGGL(E.var.ens_surface, dim3((mx + 255) / 256, my, nm), dim3(256), 0, E.stream, (const StepArgs *)E.dtab, s);
    hipLaunchKernelGGL(E.phys[s] ? E.var.ens_phys : E.var.ens_plain, dim3(E.nwg), dim3(NT), 0, E.stream, E.Q, s);
  }
  hipLaunchKernelGGL(ens_advance, dim3((nm + 63) / 64), dim3(64), 0, E.stream, E.dtab, (const int *)E.dmptf, nm);
  HIPCHK(hipGetLastError());
  return FE_OK;
}

/* Work items of every member, longest first, dealt to the eight XCD queues in
 * contiguous runs of about equal work; tables uploaded; the step graph recaptured. */
int ens_build() {
  int rc;
  const int nm = (int)E.mem.size();
  if (nm == 0) return FE_ERR_STATE;
  ens_default_segments();
  /* the tables below are freed and rewritten by null-stream calls, which do not wait for the
   * (non-blocking) ensemble stream */
  HIPCHK(hipStreamSynchronize(E.stream));
  struct T { EnsItem e; int cost; };
  std::vector<T> t;
  for (int i = 0; i < nm; ++i) {
    Member &m = E.mem[i];
    m.ntx = (m.Nx + TX - 1) / TX;
    m.nty = (m.Ny + TY - 1) / TY;
    for (int bz = 0; bz < m.nseg; ++bz) {
      const int z0 = bz * m.zseg, z1 = std::min(m.Nz, z0 + m.zseg);
      const int cost = ens_item_cost(z1 - z0);
      for (int b = 0; b < m.ntx * m.nty; ++b) t.push_back({EnsItem{i, b, m.ntx, bz}, cost});
    }
  }
  std::stable_sort(t.begin(), t.end(), [](const T &x, const T &y) { return x.cost > y.cost; });
  long total = 0;
  for (auto &x : t) total += x.cost;
  std::vector<EnsItem> items(t.size());
  long acc = 0;
  int q = 0;
  for (int k = 0; k < ENS_NQ; ++k) { E.Q.qbeg[k] = 0; E.Q.qlen[k] = 0; }
  for (size_t k = 0; k < t.size(); ++k) {
    while (q < ENS_NQ - 1 && acc >= (long)(q + 1) * total / ENS_NQ) { ++q; E.Q.qbeg[q] = (int)k; }
    items[k] = t[k].e;
    E.Q.qlen[q]++;
    acc += t[k].cost;
  }
  for (int k = q + 1; k < ENS_NQ; ++k) E.Q.qbeg[k] = (int)t.size();
  if (items.size() > E.nitems_cap) {
    if (E.ditems) HIPCHK(hipFree(E.ditems));
    E.ditems = nullptr;
    HIPCHK(hipMalloc(&E.ditems, items.size() * sizeof(EnsItem)));
    E.nitems_cap = items.size();
  }
  HIPCHK(hipMemcpy(E.ditems, items.data(), items.size() * sizeof(EnsItem), hipMemcpyHostToDevice));
  if (E.dtab) HIPCHK(hipFree(E.dtab));
  if (E.dmptf) HIPCHK(hipFree(E.dmptf));
  E.dtab = nullptr; E.dmptf = nullptr;
  HIPCHK(hipMalloc(&E.dtab, (size_t)3 * nm * sizeof(StepArgs)));
  HIPCHK(hipMalloc(&E.dmptf, (size_t)nm * sizeof(int)));
  std::vector<StepArgs> tab((size_t)3 * nm);
  std::vector<int> mptf(nm);
  for (int i = 0; i < nm; ++i) {
    for (int s = 0; s < 3; ++s) tab[(size_t)i * 3 + s] = E.mem[i].args[s];
    mptf[i] = E.mem[i].mptf;
  }
  HIPCHK(hipMemcpy(E.dtab, tab.data(), tab.size() * sizeof(StepArgs), hipMemcpyHostToDevice));
  HIPCHK(hipMemcpy(E.dmptf, mptf.data(), mptf.size() * sizeof(int), hipMemcpyHostToDevice));
  if (!E.dctr) HIPCHK(hipMalloc(&E.dctr, 3 * ENS_NQ * sizeof(unsigned)));
  HIPCHK(hipMemset(E.dctr, 0, 3 * ENS_NQ * sizeof(unsigned)));
  E.Q.tab = E.dtab;
  E.Q.items = E.ditems;
  E.Q.ctr = E.dctr;
  E.nwg = ens_slots();
  if ((rc = ens_drop_graph())) return rc;
  HIPCHK(hipStreamBeginCapture(E.stream, hipStreamCaptureModeThreadLocal));
  rc = ens_enqueue_step();
  hipGraph_t g = nullptr;
  const hipError_t ec = hipStreamEndCapture(E.stream, &g);
  if (rc) { if (g) (void)hipGraphDestroy(g); return rc; }
  HIPCHK(ec);
  E.graph = g;
  HIPCHK(hipGraphInstantiate(&E.gexec, E.graph, nullptr, nullptr, 0));
  E.dirty = false;
  E.host_tab_newer = false;
  return FE_OK;
}

int ens_prepare() {
  if (E.mem.empty()) return FE_ERR_STATE;
  if (E.dirty) return ens_build();
  if (E.host_tab_newer) {
    std::vector<StepArgs> tab(3 * E.mem.size());
    for (size_t i = 0; i < E.mem.size(); ++i)
      for (int s = 0; s < 3; ++s) tab[i * 3 + s] = E.mem[i].args[s];
    HIPCHK(hipMemcpyAsync(E.dtab, tab.data(), tab.size() * sizeof(StepArgs), hipMemcpyHostToDevice, E.stream));
    HIPCHK(hipStreamSynchronize(E.stream));
    E.host_tab_newer = false;
  }
  return FE_OK;
}

/* the device rows (advanced by the replays) back into the host copies */
int ens_pull_tab() {
  std::vector<StepArgs> tab(3 * E.mem.size());
  HIPCHK(hipMemcpyAsync(tab.data(), E.dtab, tab.size() * sizeof(StepArgs), hipMemcpyDeviceToHost, E.stream));
  HIPCHK(hipStreamSynchronize(E.stream));
  for (size_t i = 0; i < E.mem.size(); ++i)
    for (int s = 0; s < 3; ++s) E.mem[i].args[s] = tab[i * 3 + s];
  return FE_OK;
}

/* One step of member m through the plain launches (the plain path's grid and kernels): with
 * the member's current (possibly tuned) z segments, which continues the ensemble bitwise, or
 * (plain_segments) with the segments the plain path chooses for a lone run of this grid, the
 * launches a user running the members one after another would make. */
int ens_plain_step(Member &m, bool plain_segments = false) {
  for (int s = 0; s < 3; ++s) {
    StepArgs a = m.args[s];
    const int nseg = plain_segments ? m.nseg_plain : m.nseg;
    if (plain_segments) a.zseg = m.zseg_plain;
    if (E.surf[s] && a.slSel > 0)
      hipLaunchKernelGGL(E.var.surface, dim3((m.Nx + 255) / 256, m.Ny), dim3(256), 0, E.stream, a);
    hipLaunchKernelGGL(E.phys[s] ? E.var.phys : E.var.plain, dim3(m.ntx, m.nty, nseg), dim3(NT), 0, E.stream, a);
  }
  HIPCHK(hipGetLastError());
  ens_host_advance(m);
  return FE_OK;
}

int ens_free_all() {
  int rc;
  if (E.stream) HIPCHK(hipStreamSynchronize(E.stream));
  if ((rc = ens_drop_graph())) return rc;
  for (auto &m : E.mem) {
    for (int s = 0; s < 3; ++s) if (m.S[s]) HIPCHK(hipFree(m.S[s]));
    if (m.prof) HIPCHK(hipFree(m.prof));
    if (m.surf) HIPCHK(hipFree(m.surf));
  }
  E.mem.clear();
  void *p[] = {E.dtab, E.dmptf, E.ditems, E.dctr};
  for (void *q : p) if (q) HIPCHK(hipFree(q));
  E.dtab = nullptr; E.dmptf = nullptr; E.ditems = nullptr; E.dctr = nullptr; E.nitems_cap = 0;
  E.have_var = false;
  E.dirty = true;
  E.host_tab_newer = false;
  E.report.clear();
  if (!D.fecuda) return xfer_release();        /* no model left to use the pinned slots */
  return FE_OK;
}

/* device time of n graph replays after one untimed replay, in ms */
int ens_time_replays(int n, float &ms) {
  int rc;
  if ((rc = ens_prepare())) return rc;
  HIPCHK(hipGraphLaunch(E.gexec, E.stream));
  hipEvent_t e0, e1;
  HIPCHK(hipEventCreate(&e0));
  HIPCHK(hipEventCreate(&e1));
  HIPCHK(hipEventRecord(e0, E.stream));
  for (int i = 0; i < n; ++i) HIPCHK(hipGraphLaunch(E.gexec, E.stream));
  HIPCHK(hipEventRecord(e1, E.stream));
  HIPCHK(hipEventSynchronize(e1));
  HIPCHK(hipEventElapsedTime(&ms, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return FE_OK;
}

}  // namespace

extern "C" {

/* Move the current plain model (set up through cuda_timeIntInit) into the ensemble as
 * its next member; returns the member index, or a negative FE_ERR_* code.  The plain
 * model keeps its host arrays but no longer has device state (its entry points then
 * return FE_ERR_STATE until it is set up again). */
int fe_ens_add_member(void) {
  if (!D.timeint) return -FE_ERR_STATE;
  if (!g_var_ok || !g_var.ens_plain) {
    fprintf(stderr, "fe_ens_add_member: no ensemble kernels for variant %s\n", g_var_ok ? g_var.name : "none");
    return -FE_ERR_UNSUPPORTED;
  }
  if (lsfSelector == 1) {
    fprintf(stderr, "fe_ens_add_member: large-scale forcing is not supported in the ensemble\n");
    return -FE_ERR_UNSUPPORTED;
  }
  if (D.halo) {
    fprintf(stderr, "fe_ens_add_member: members are periodic grids (no lateral halo storage)\n");
    return -FE_ERR_UNSUPPORTED;
  }
  int ph[3], sf[3];
  for (int s = 0; s < 3; ++s) {
    ph[s] = physics_stage(s) && turbulenceSelector > 0;
    sf[s] = physics_stage(s) && surflayerSelector > 0;
  }
  if (E.have_var) {
    if (strcmp(E.var.name, g_var.name) != 0) {
      fprintf(stderr, "fe_ens_add_member: member variant %s differs from the ensemble's %s\n", g_var.name, E.var.name);
      return -FE_ERR_UNSUPPORTED;
    }
    for (int s = 0; s < 3; ++s)
      if (ph[s] != E.phys[s]) {
        fprintf(stderr, "fe_ens_add_member: members must share the physics-stage schedule (physics_oneRKonly)\n");
        return -FE_ERR_UNSUPPORTED;
      }
  } else {
    E.var = g_var;
    E.have_var = true;
    for (int s = 0; s < 3; ++s) E.phys[s] = ph[s];
    if (!E.stream) HIPCHK(hipStreamCreateWithFlags(&E.stream, hipStreamNonBlocking));
  }
  for (int s = 0; s < 3; ++s) E.surf[s] = E.surf[s] || sf[s];
  HIPCHK(hipStreamSynchronize(D.stream));
  Member m;
  m.Nx = D.Nx; m.Ny = D.Ny; m.Nz = D.Nz; m.P = D.P; m.NF = D.NF; m.fs = D.fs; m.ps = D.ps;
  m.nseg = D.nseg; m.zseg = D.zseg;
  m.nseg_plain = D.nseg; m.zseg_plain = D.zseg;
  m.seg_set = amd_zSegments > 0;
  for (int s = 0; s < 3; ++s) m.S[s] = D.S[s];
  m.prof = D.prof;
  m.surf = D.surf;
  fill_args(m.args[0], 0, m.S[0], m.S[0], m.S[1], 0, nullptr);
  fill_args(m.args[1], 1, m.S[1], m.S[0], m.S[2], 0, nullptr);
  fill_args(m.args[2], 2, m.S[2], m.S[0], m.S[0], 0, nullptr);
  const Variant &var = variant_of(m.args[0]);
  if (E.mem.empty() || E.var.sb) E.var = var;    /* kernels for any weights once a member's weights differ */
  m.mptf = 0;
  if (moistureSelector > 0 && moistureCond > 0 && moistureNvars > 1)
    m.mptf = (int)roundf(fmaxf(moistureMPcallTscale, dt) / dt);
  m.ntx = (m.Nx + TX - 1) / TX;
  m.nty = (m.Ny + TY - 1) / TY;
  /* the device buffers now belong to the ensemble */
  for (int s = 0; s < 3; ++s) D.S[s] = nullptr;
  D.prof = nullptr;
  D.surf = nullptr;
  D.timeint = 0;
  D.hydro = 0;
  D.grid = 0;
  E.mem.push_back(m);
  E.dirty = true;
  E.seg_old = true;
  return (int)E.mem.size() - 1;
}

int fe_ens_count(void) { return (int)E.mem.size(); }

/* info[0..8] = Nx, Ny, Nz, P (row pitch), NF (fields), z segments, segment length,
 * step index, simulation time * 1000 (ms, rounded) */
int fe_ens_member_info(int m, int *info, int n) {
  if (m < 0 || m >= (int)E.mem.size() || !info || n < 9) return FE_ERR_STATE;
  ens_default_segments();
  const Member &q = E.mem[m];
  const int v[9] = {q.Nx, q.Ny, q.Nz, q.P, q.NF, q.nseg, q.zseg, q.args[0].step_it, (int)lroundf(q.args[0].simTime * 1000.f)};
  for (int i = 0; i < 9; ++i) info[i] = v[i];
  return FE_OK;
}

/* Device state of member m ([field][z][y][x], row pitch P), n = NF * Nz * Ny * P floats. */
int fe_ens_member_state(int m, float *out, long n) {
  if (m < 0 || m >= (int)E.mem.size() || !out) return FE_ERR_STATE;
  const Member &q = E.mem[m];
  if (n != (long)q.NF * q.fs) return FE_ERR_UNSUPPORTED;
  int rc;
  if ((rc = xfer_reserve((size_t)n * sizeof(float)))) return rc;
  XferScope scope;
  if ((rc = xfer_down(E.stream, out, q.S[0], (size_t)n * sizeof(float)))) return rc;
  return xfer_finish(E.stream);
}

/* Friction velocity plane of member m ([y][x], pitch P), n = Ny * P floats. */
int fe_ens_member_ustar(int m, float *out, long n) {
  if (m < 0 || m >= (int)E.mem.size() || !out) return FE_ERR_STATE;
  const Member &q = E.mem[m];
  if (n != q.ps) return FE_ERR_UNSUPPORTED;
  HIPCHK(hipStreamSynchronize(E.stream));
  HIPCHK(hipMemcpy(out, q.surf + (long)SF_UST * q.ps, (size_t)n * sizeof(float), hipMemcpyDeviceToHost));
  return FE_OK;
}

/* Set the z-segment count of member m (the autotuner's knob), nseg >= 1. */
int fe_ens_set_segments(int m, int nseg) {
  if (m < 0 || m >= (int)E.mem.size() || nseg < 1) return FE_ERR_STATE;
  ens_set_segments(E.mem[m], nseg);
  E.mem[m].seg_set = true;
  return FE_OK;
}

/* nsteps RK3 steps of every member: one graph replay per step, one synchronisation. */
int fe_ens_steps(int nsteps) {
  int rc;
  if ((rc = ens_prepare())) return rc;
  for (int i = 0; i < nsteps; ++i) HIPCHK(hipGraphLaunch(E.gexec, E.stream));
  HIPCHK(hipStreamSynchronize(E.stream));
  return ens_pull_tab();
}

/* nsteps RK3 steps of each member in turn through the plain launches. */
int fe_ens_steps_sequential(int nsteps) {
  int rc;
  if ((rc = ens_prepare())) return rc;
  if ((rc = ens_pull_tab())) return rc;
  for (auto &m : E.mem)
    for (int i = 0; i < nsteps; ++i)
      if ((rc = ens_plain_step(m))) return rc;
  HIPCHK(hipStreamSynchronize(E.stream));
  E.host_tab_newer = true;
  return FE_OK;
}

/* Device time of each of nsteps steps, in ms, into ms[0..nsteps): with sequential = 0 one
 * ensemble step (all members, one graph replay) per entry; with sequential = 1 the members'
 * plain steps in turn, ms[i] of member i % count, step i / count (nsteps = count * steps),
 * each member launched with the plain path's own z segments for its grid. */
int fe_ens_step_times(int nsteps, int sequential, float *ms) {
  int rc;
  if (!ms || nsteps <= 0) return FE_ERR_STATE;
  if ((rc = ens_prepare())) return rc;
  if (sequential && (rc = ens_pull_tab())) return rc;
  std::vector<hipEvent_t> ev((size_t)nsteps + 1);
  for (auto &e : ev) HIPCHK(hipEventCreate(&e));
  HIPCHK(hipEventRecord(ev[0], E.stream));
  const int nm = (int)E.mem.size();
  for (int i = 0; i < nsteps; ++i) {
    if (sequential) {
      if ((rc = ens_plain_step(E.mem[i % nm], true))) return rc;
    } else {
      HIPCHK(hipGraphLaunch(E.gexec, E.stream));
    }
    HIPCHK(hipEventRecord(ev[i + 1], E.stream));
  }
  HIPCHK(hipEventSynchronize(ev[nsteps]));
  for (int i = 0; i < nsteps; ++i) HIPCHK(hipEventElapsedTime(&ms[i], ev[i], ev[i + 1]));
  for (auto &e : ev) (void)hipEventDestroy(e);
  if (sequential) E.host_tab_newer = true;
  else if ((rc = ens_pull_tab())) return rc;
  return FE_OK;
}

/* Autotuner: for each member shape (Nx, Ny, Nz) in turn, time trial_steps graph replays
 * for every z-segment count whose segments are at least 4 levels long and keep the
 * fastest (coordinate descent from the segments the members have, two passes).  The members'
 * state, surface planes and step rows are saved first and restored after, so tuning
 * leaves the simulation where it was.  A report of the trials and choices is copied
 * into report (len bytes). */
int fe_ens_autotune(int trial_steps, char *report, int len) {
  int rc;
  if (E.mem.empty() || trial_steps < 1) return FE_ERR_STATE;
  if ((rc = ens_prepare())) return rc;
  if ((rc = ens_pull_tab())) return rc;
  /* save */
  std::vector<float *> save(E.mem.size(), nullptr);
  std::vector<Member> rows = E.mem;
  for (size_t i = 0; i < E.mem.size(); ++i) {
    const Member &m = E.mem[i];
    const size_t ns = (size_t)m.NF * m.fs, nsf = (size_t)SF_N * m.ps;
    HIPCHK(hipMalloc(&save[i], (ns + nsf) * sizeof(float)));
    HIPCHK(hipMemcpyAsync(save[i], m.S[0], ns * sizeof(float), hipMemcpyDeviceToDevice, E.stream));
    HIPCHK(hipMemcpyAsync(save[i] + ns, m.surf, nsf * sizeof(float), hipMemcpyDeviceToDevice, E.stream));
  }
  HIPCHK(hipStreamSynchronize(E.stream));
  /* shapes */
  std::vector<std::array<int, 3>> shapes;
  for (auto &m : E.mem) {
    std::array<int, 3> s = {m.Nx, m.Ny, m.Nz};
    if (std::find(shapes.begin(), shapes.end(), s) == shapes.end()) shapes.push_back(s);
  }
  auto set_shape = [&](const std::array<int, 3> &s, int n) {
    for (auto &m : E.mem)
      if (m.Nx == s[0] && m.Ny == s[1] && m.Nz == s[2]) {
        ens_set_segments(m, n);
        m.seg_set = true;
      }
  };
  auto cur = [&](const std::array<int, 3> &s) {
    for (auto &m : E.mem)
      if (m.Nx == s[0] && m.Ny == s[1] && m.Nz == s[2]) return m.nseg;
    return 1;
  };
  char line[256];
  std::string rep;
  float best = 0.f;
  if ((rc = ens_time_replays(trial_steps, best))) return rc;
  snprintf(line, sizeof line, "start: %.4f ms/step\n", best / trial_steps);
  rep += line;
  for (int pass = 0; pass < 2; ++pass) {
    for (auto &s : shapes) {
      const int keep = cur(s);
      int bestn = keep;
      std::vector<int> tried;
      for (int c = 1; c <= s[2]; ++c) {
        int len_, n_;
        seg_shape(s[2], c, len_, n_);
        if (c > 1 && len_ < 4) break;
        if (std::find(tried.begin(), tried.end(), n_) != tried.end() || n_ == keep) continue;
        tried.push_back(n_);
        set_shape(s, n_);
        float t = 0.f;
        if ((rc = ens_time_replays(trial_steps, t))) return rc;
        snprintf(line, sizeof line, "pass %d shape %dx%dx%d: %d segments of %d levels %.4f ms/step\n", pass, s[0], s[1], s[2], n_,
                 len_, t / trial_steps);
        rep += line;
        if (t < best) { best = t; bestn = n_; }
      }
      set_shape(s, bestn);
    }
  }
  for (auto &s : shapes) {
    int len_, n_;
    seg_shape(s[2], cur(s), len_, n_);
    snprintf(line, sizeof line, "choice %dx%dx%d: %d segments of %d levels\n", s[0], s[1], s[2], n_, len_);
    rep += line;
  }
  snprintf(line, sizeof line, "tuned: %.4f ms/step, %d persistent work-groups\n", best / trial_steps, E.nwg);
  rep += line;
  /* restore state, surface planes and step rows (with the tuned segments) */
  for (size_t i = 0; i < E.mem.size(); ++i) {
    Member &m = E.mem[i];
    const size_t ns = (size_t)m.NF * m.fs, nsf = (size_t)SF_N * m.ps;
    HIPCHK(hipMemcpyAsync(m.S[0], save[i], ns * sizeof(float), hipMemcpyDeviceToDevice, E.stream));
    HIPCHK(hipMemcpyAsync(m.surf, save[i] + ns, nsf * sizeof(float), hipMemcpyDeviceToDevice, E.stream));
    for (int s = 0; s < 3; ++s) {
      const int z = m.args[s].zseg;
      m.args[s] = rows[i].args[s];
      m.args[s].zseg = z;
    }
  }
  HIPCHK(hipStreamSynchronize(E.stream));
  for (auto p : save) HIPCHK(hipFree(p));
  E.dirty = true;
  if ((rc = ens_build())) return rc;
  E.report = rep;
  if (report && len > 0) {
    strncpy(report, rep.c_str(), (size_t)len - 1);
    report[len - 1] = 0;
  }
  return FE_OK;
}

int fe_ens_clear(void) { return ens_free_all(); }

}  // extern "C"
