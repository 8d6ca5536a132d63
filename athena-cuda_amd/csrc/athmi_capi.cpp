// athmi_capi.cpp -- host runtime behind include/athmi.h: device memory of the
// instances (SoA planes in HBM, ping-pong state buffers, scratch planes and a
// device-resident clock per instance), the tile work-list of a batch, HIP
// graph capture of one main-loop step, and the AoS<->SoA host transfers.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "athmi.h"
#include "host_problems.hpp"
#include "step_kernels.hpp"
#include "runtime.hpp"

namespace athmi_rt {
thread_local std::string g_err;
}  // namespace athmi_rt

extern "C" {

const char* athmi_last_error(void) { return g_err.c_str(); }

int athmi_create(const athmi_desc* desc, int n, athmi_grid** out) {
  if (!desc || !out || n <= 0) return fail(ATHMI_EINVAL, "athmi_create: bad arguments");
  for (int k = 0; k < n; k++) {
    const athmi_desc& d = desc[k];
    if (d.nx1 < 2 || d.nx2 < 2)
      return fail(ATHMI_EINVAL, "athmi_create: the 2-D integrator needs Nx1 > 1 and Nx2 > 1");
    if (!(d.x1max > d.x1min) || !(d.x2max > d.x2min))
      return fail(ATHMI_EINVAL, "athmi_create: empty domain");
    const int bcs[4] = {d.bc_ix1, d.bc_ox1, d.bc_ix2, d.bc_ox2};
    for (int b : bcs)
      if (b != ATHMI_BC_REFLECT && b != ATHMI_BC_OUTFLOW && b != ATHMI_BC_PERIODIC)
        return fail(ATHMI_EINVAL, "athmi_create: boundary flag must be 1, 2 or 4");
    if (d.flux != ATHMI_FLUX_ROE && d.flux != ATHMI_FLUX_HLLE)
      return fail(ATHMI_EINVAL, "athmi_create: unknown flux");
    if (d.variant != desc[0].variant)
      return fail(ATHMI_EINVAL, "athmi_create: one arithmetic variant per handle");
  }
  if (desc[0].variant != ATHMI_EXACT && desc[0].variant != ATHMI_FAST)
    return fail(ATHMI_EINVAL, "athmi_create: unknown variant");
  int dev = 0, ncu = 0;
  HIP_TRY(hipGetDevice(&dev));
  HIP_TRY(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));

  athmi_grid* g = new athmi_grid();
  g->n = n;
  g->variant = desc[0].variant;
  g->launch = (g->variant == ATHMI_FAST) ? athmi_fast_launch : athmi_exact_launch;
  g->desc.assign(desc, desc + n);
  g->hinst.resize(n);
  g->cpaw_soln.resize(n);
  g->bl.ncu = ncu;
  // faces marched per lane by the x2 predictor (1..16)
  long cols = 0;
  for (int k = 0; k < n; k++) cols += (long)cdiv(desc[k].nx1 + 6, kX2Block) * (desc[k].nx2 + 4);
  g->bl.shape.x2_seg = default_x2_seg(cols);
  g->bl.shape.persist = 0;
  g->bl.shape.xcd_remap = 1;
  g->bl.shape.corr_rows = 1;  // one-row corrector tiles, which follow each other across row ends
  g->bl.shape.x2_kind = 1;  // the two-wave x2 predictor (1.79 against 2.05 ms at 4096^2)
  g->bl.shape.fuse_corner = 1;  // Step 9 corners inside k_final (the autotuner's pick at 4096^2)
  g->bl.shape.strip = 0;        // corrector and final tiles row by row
  g->bl.shape.final_rows = 8;   // 64 x 8 final tiles (1.10 -> 1.07 ms against 64 x 4 at 4096^2)
  // device memory: per instance 2*NSTATE state planes + NSCRATCH scratch planes
  std::vector<size_t> off(n);
  size_t total = 0;
  for (int k = 0; k < n; k++) {
    const athmi_desc& d = desc[k];
    Inst& I = g->hinst[k];
    std::memset(&I, 0, sizeof(I));
    I.nx1 = d.nx1;
    I.nx2 = d.nx2;
    I.is = 4;
    I.ie = d.nx1 + 3;
    I.js = 4;
    I.je = d.nx2 + 3;
    I.sx = d.nx1 + 8;
    I.sy = d.nx2 + 8;
    I.pitch = (int)round_up(I.sx, 16);
    I.flux = d.flux;
    I.bc[0] = d.bc_ix1;
    I.bc[1] = d.bc_ox1;
    I.bc[2] = d.bc_ix2;
    I.bc[3] = d.bc_ox2;
    I.dx1 = (d.x1max - d.x1min) / (double)d.nx1;  // init_grid.c:60
    I.dx2 = (d.x2max - d.x2min) / (double)d.nx2;
    I.gamma = d.gamma;
    I.g1 = d.gamma - 1.0;  // main.c:93-94
    I.g2 = d.gamma - 2.0;
    I.ps = round_up((size_t)I.pitch * I.sy, 64);
    // the kernels address a plane with 32-bit element offsets (bytes < 2^32)
    if (I.ps >= ((size_t)1 << 29)) {
      delete g;
      return fail(ATHMI_EINVAL, "athmi_create: a plane of (Nx1+8) x (Nx2+8) cells exceeds 2^29 "
                                "doubles");
    }
    off[k] = total;
    total += (size_t)(2 * NSTATE + NSCRATCH) * I.ps;
  }
  g->dmem_bytes = total * sizeof(double);
  if (hipMalloc(&g->dmem, g->dmem_bytes) != hipSuccess) {
    delete g;
    return fail(ATHMI_ENOMEM, "athmi_create: hipMalloc of the state failed");
  }
  if (hipMemset(g->dmem, 0, g->dmem_bytes) != hipSuccess) {
    (void)hipFree(g->dmem);
    delete g;
    return fail(ATHMI_EHIP, "athmi_create: clearing the state failed");
  }
  if (hipMalloc(&g->dclk, sizeof(Clock) * n) != hipSuccess ||
      hipMalloc(&g->dinst, inst_lists_bytes(n)) != hipSuccess) {
    athmi_destroy(g);
    return fail(ATHMI_ENOMEM, "athmi_create: hipMalloc of the descriptors failed");
  }
  if (hipHostMalloc(&g->heads, sizeof(ClockHead) * n + sizeof(*g->set_done),
                    hipHostMallocCoherent) != hipSuccess) {
    athmi_destroy(g);
    return fail(ATHMI_ENOMEM, "athmi_create: hipHostMalloc of the clocks failed");
  }
  g->set_done = reinterpret_cast<unsigned long long*>(g->heads + n);
  *g->set_done = 0;
  std::vector<Clock> hc(n);
  for (int k = 0; k < n; k++) {
    std::memset(&hc[k], 0, sizeof(Clock));
    hc[k].cour_no = desc[k].cour_no;
    hc[k].tlim = HUGE_VAL;
    hc[k].tpause = HUGE_VAL;
    hc[k].nlim = -1;
    hc[k].fail_nstep = -1;
    // the reference floors the pressure and steps on (convert_var.c:49): a
    // floor hit is reported, only a non-finite value or d <= 0 stops
    hc[k].fail_stop = ATHMI_FAIL_NONFINITE | ATHMI_FAIL_DENSITY;
    Inst& I = g->hinst[k];
    I.state[0] = g->dmem + off[k];
    I.state[1] = I.state[0] + NSTATE * I.ps;
    I.scratch = I.state[1] + NSTATE * I.ps;
    I.clk = g->dclk + k;
  }
  if (hipMemcpy(g->dclk, hc.data(), sizeof(Clock) * n, hipMemcpyHostToDevice) != hipSuccess) {
    athmi_destroy(g);
    return fail(ATHMI_EHIP, "athmi_create: writing the clocks failed");
  }
  if (hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking) != hipSuccess) {
    athmi_destroy(g);
    return fail(ATHMI_EHIP, "athmi_create: stream creation failed");
  }
  g->own_stream = true;
  int rc = g->refresh_tiles();
  if (rc != ATHMI_OK) {
    athmi_destroy(g);
    return rc;
  }
  *out = g;
  return ATHMI_OK;
}

int athmi_destroy(athmi_grid* g) {
  if (!g) return ATHMI_OK;
  if (g->stream) (void)hipStreamSynchronize(g->stream);
  g->drop_graph();
  if (g->dmem) (void)hipFree(g->dmem);
  if (g->dclk) (void)hipFree(g->dclk);
  if (g->dinst) (void)hipFree(g->dinst);
  if (g->heads) (void)hipHostFree(g->heads);
  if (g->outbuf) (void)hipFree(g->outbuf);
  if (g->own_stream && g->stream) (void)hipStreamDestroy(g->stream);
  delete g;
  return ATHMI_OK;
}

int athmi_count(const athmi_grid* g, int* n) {
  if (!g || !n) return fail(ATHMI_EINVAL, "athmi_count: null argument");
  *n = g->n;
  return ATHMI_OK;
}

static int check_inst(const athmi_grid* g, int inst) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (inst < 0 || inst >= g->n) return fail(ATHMI_EINVAL, "instance index out of range");
  return ATHMI_OK;
}

int athmi_set_spacing(athmi_grid* g, int inst, double dx1, double dx2) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  if (!(dx1 > 0.0) || !(dx2 > 0.0)) return fail(ATHMI_EINVAL, "athmi_set_spacing: dx <= 0");
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->hinst[inst].dx1 = dx1;
  g->hinst[inst].dx2 = dx2;
  return g->refresh_tiles();
}

int athmi_upload(athmi_grid* g, int inst, const double* gas, const double* b1i, const double* b2i,
                 const double* b3i) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  if (!gas || !b1i || !b2i || !b3i) return fail(ATHMI_EINVAL, "athmi_upload: null array");
  Clock c;
  if ((rc = g->read_clock(inst, c))) return rc;
  const Inst& I = g->hinst[inst];
  // the caller's arrays land unchanged in the idle ping-pong buffer (the next
  // step rewrites all of it) and one kernel scatters them into the planes
  const size_t n = (size_t)I.sy * I.sx;
  if ((size_t)I.sy * I.pitch > I.ps) return fail(ATHMI_ESTATE, "athmi_upload: plane layout");
  double* stage = I.state[c.cur ^ 1];
  HIP_TRY(hipMemcpy(stage, gas, sizeof(double) * 8 * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(stage + 8 * n, b1i, sizeof(double) * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(stage + 9 * n, b2i, sizeof(double) * n, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(stage + 10 * n, b3i, sizeof(double) * n, hipMemcpyHostToDevice));
  HIP_TRY(launch_state_unpack(stage, I.state[c.cur], I.ps, I.pitch, I.sx, I.sy, g->stream));
  HIP_TRY(hipStreamSynchronize(g->stream));
  // a new state: the failure word describes states produced from it
  if (c.fail != 0 || c.fail_nstep != -1) {
    c.fail = 0;
    c.fail_nstep = -1;
    if ((rc = g->write_clock_head(inst, c))) return rc;
  }
  return ATHMI_OK;
}

int athmi_download(athmi_grid* g, int inst, double* gas, double* b1i, double* b2i, double* b3i) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  if (!gas || !b1i || !b2i || !b3i) return fail(ATHMI_EINVAL, "athmi_download: null array");
  Clock c;
  if ((rc = g->read_clock(inst, c))) return rc;
  const Inst& I = g->hinst[inst];
  // gathered into the caller's layout in the idle ping-pong buffer, then
  // copied out unchanged
  const size_t n = (size_t)I.sy * I.sx;
  if ((size_t)I.sy * I.pitch > I.ps) return fail(ATHMI_ESTATE, "athmi_download: plane layout");
  double* stage = I.state[c.cur ^ 1];
  HIP_TRY(launch_state_pack(I.state[c.cur], stage, I.ps, I.pitch, I.sx, I.sy, g->stream));
  HIP_TRY(hipStreamSynchronize(g->stream));
  HIP_TRY(hipMemcpy(gas, stage, sizeof(double) * 8 * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(b1i, stage + 8 * n, sizeof(double) * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(b2i, stage + 9 * n, sizeof(double) * n, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(b3i, stage + 10 * n, sizeof(double) * n, hipMemcpyDeviceToHost));
  return ATHMI_OK;
}

int athmi_set_clock(athmi_grid* g, int inst, double dt, double time, int nstep) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  Clock c;
  if ((rc = g->read_clock(inst, c))) return rc;
  c.dt = dt;
  c.time = time;
  c.nstep = nstep;
  return g->write_clock_head(inst, c);
}

int athmi_get_clock(athmi_grid* g, int inst, double* dt, double* time, int* nstep) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  Clock c;
  if ((rc = g->read_clock(inst, c))) return rc;
  if (dt) *dt = c.dt;
  if (time) *time = c.time;
  if (nstep) *nstep = c.nstep;
  return ATHMI_OK;
}

int athmi_get_failure(athmi_grid* g, int inst, int* flags, int* nstep) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  Clock c;
  if ((rc = g->read_clock(inst, c))) return rc;
  if (flags) *flags = c.fail;
  if (nstep) *nstep = c.fail_nstep;
  return ATHMI_OK;
}

int athmi_set_fail_stop(athmi_grid* g, int inst, int mask) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (mask & ~(ATHMI_FAIL_NONFINITE | ATHMI_FAIL_DENSITY | ATHMI_FAIL_PRESSURE))
    return fail(ATHMI_EINVAL, "athmi_set_fail_stop: unknown failure bit");
  const int lo = inst < 0 ? 0 : inst, hi = inst < 0 ? g->n - 1 : inst;
  if (inst >= g->n) return fail(ATHMI_EINVAL, "instance index out of range");
  for (int k = lo; k <= hi; k++) {
    Clock c;
    int rc = g->read_clock(k, c);
    if (rc) return rc;
    c.fail_stop = mask;
    if ((rc = g->write_clock_head(k, c))) return rc;
  }
  return ATHMI_OK;
}

int athmi_set_limits(athmi_grid* g, int inst, double tlim, int nlim) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  const int lo = inst < 0 ? 0 : inst, hi = inst < 0 ? g->n - 1 : inst;
  if (inst >= g->n) return fail(ATHMI_EINVAL, "instance index out of range");
  for (int k = lo; k <= hi; k++) {
    Clock c;
    int rc = g->read_clock(k, c);
    if (rc) return rc;
    c.tlim = tlim;
    c.nlim = nlim;
    if ((rc = g->write_clock_head(k, c))) return rc;
  }
  return ATHMI_OK;
}

int athmi_set_pause(athmi_grid* g, int inst, double t_next) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  const int lo = inst < 0 ? 0 : inst, hi = inst < 0 ? g->n - 1 : inst;
  if (inst >= g->n) return fail(ATHMI_EINVAL, "instance index out of range");
  for (int k = lo; k <= hi; k++) {
    Clock c;
    int rc = g->read_clock(k, c);
    if (rc) return rc;
    c.tpause = t_next;
    if ((rc = g->write_clock_head(k, c))) return rc;
  }
  return ATHMI_OK;
}

int athmi_set_bvals(athmi_grid* g) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  HIP_TRY(g->launch(&g->bl, SK_GHOST_CUR, g->stream));
  return ATHMI_OK;
}

int athmi_new_dt(athmi_grid* g) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  g->clock_written = true;  // by the device
  int rc = issue(g, kSeqNewDt);
  if (rc) return rc;
  HIP_TRY(hipStreamSynchronize(g->stream));
  return ATHMI_OK;
}

// integrate_2d writes only the interior; the ghost zones of the produced
// buffer carry the current values, as an in-place update would leave them
int athmi_integrate(athmi_grid* g) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  g->clock_written = true;  // SK_BEGIN_ONCE
  return issue(g, kSeqIntegrate);
}

static int issue_step(athmi_grid* g) {
  for (int k : kSeqStep) HIP_TRY(g->launch(&g->bl, k, g->stream));
  return ATHMI_OK;
}

int athmi_step(athmi_grid* g) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  const athmi_grid::ClockWork work(g);
  // without the graph every step starts itself: its launches may be captured
  // by the caller and replayed after the host has written the clock. So does
  // every step once the caller has captured any work of the handle: a replay of
  // athmi_integrate leaves its own unconditional start in the clock, and a start
  // launched into a capture has not run
  const bool always = !g->use_graph || g->caller_captured;
  if (g->clock_written || always) {
    HIP_TRY(g->launch(&g->bl, SK_BEGIN_STEP, g->stream));
    g->clock_written = always;
  }
  if (!g->use_graph) return issue_step(g);
  if (!g->graph) {
    std::lock_guard<std::mutex> lk(g->clk_mu);
    hipGraph_t graph;
    HIP_TRY(hipStreamBeginCapture(g->stream, hipStreamCaptureModeThreadLocal));
    int rc = issue_step(g);
    hipError_t e = hipStreamEndCapture(g->stream, &graph);
    if (rc) return rc;
    if (e != hipSuccess) return fail(ATHMI_EHIP, std::string("capture: ") + hipGetErrorString(e));
    e = hipGraphInstantiate(&g->graph, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
      g->graph = nullptr;
      return fail(ATHMI_EHIP, std::string("graph instantiate: ") + hipGetErrorString(e));
    }
  }
  HIP_TRY(hipGraphLaunch(g->graph, g->stream));
  return ATHMI_OK;
}

int athmi_run(athmi_grid* g, int max_steps, int* steps) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  int issued = 0;
  const int chunk = 16;
  while (max_steps < 0 || issued < max_steps) {
    // any instance still running?
    bool running = false;
    {
      std::lock_guard<std::mutex> lk(g->clk_mu);
      const int rc = g->fetch_clocks();
      if (rc) return rc;
      for (int k = 0; k < g->n && !running; k++) {
        Clock c;
        std::memcpy(&c, &g->heads[k], sizeof(ClockHead));
        if (c.time < c.tlim && (c.nlim < 0 || c.nstep < c.nlim) && c.time < c.tpause &&
            (c.fail & c.fail_stop) == 0)
          running = true;
      }
    }
    if (!running) break;
    int m = chunk;
    if (max_steps >= 0) m = std::min(m, max_steps - issued);
    for (int s = 0; s < m; s++) {
      int rc = athmi_step(g);
      if (rc) return rc;
    }
    issued += m;
  }
  {
    std::lock_guard<std::mutex> lk(g->clk_mu);
    const int rc = g->fetch_clocks();
    if (rc) return rc;
  }
  if (steps) *steps = issued;
  return ATHMI_OK;
}

int athmi_divb_max(athmi_grid* g, int inst, double* out) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  if ((rc = issue(g, kSeqDivb))) return rc;
  Clock c;
  if ((rc = g->read_clock(inst, c))) return rc;
  unsigned long long bits = c.divb_bits;
  std::memcpy(out, &bits, sizeof(double));
  return ATHMI_OK;
}

int athmi_profile_steps(athmi_grid* g, int nsteps, double* avg_ms, int nslots) {
  if (!g || !avg_ms || nsteps <= 0 || nslots < NSEPARATE)
    return fail(ATHMI_EINVAL, "athmi_profile_steps: bad arguments");
  // an event after each launch; a step makes at most two per slot (one per solver)
  struct Marks {
    hipStream_t stream;
    std::vector<hipEvent_t> ev;
    std::vector<int> slot;  // of the launch before event k + 1
    hipError_t err = hipSuccess;
    ~Marks() {
      for (hipEvent_t e : ev) (void)hipEventDestroy(e);
    }
    void record() {
      if (err == hipSuccess && slot.size() == ev.size()) {
        hipEvent_t e = nullptr;
        err = hipEventCreate(&e);
        if (err == hipSuccess) ev.push_back(e);
      }
      if (err == hipSuccess) err = hipEventRecord(ev[slot.size()], stream);
    }
    static void launched(void* self, int slot) {
      Marks* m = static_cast<Marks*>(self);
      m->slot.push_back(slot);
      m->record();
    }
  } marks;
  marks.stream = g->stream;
  BatchLaunch bl = g->bl;
  bl.launched = Marks::launched;
  bl.launched_arg = &marks;
  // the step's own launches, or (a caller without their slots) the separate kernels
  const bool own = nslots >= NSLOTS;
  const int shown = own ? NSLOTS : NSEPARATE;
  for (int k = 0; k < shown; k++) avg_ms[k] = 0.0;
  g->clock_written = true;
  const athmi_grid::ClockWork work(g);
  for (int s = 0; s < nsteps; s++) {
    marks.slot.clear();
    marks.record();
    if (own) {
      if (s == 0) HIP_TRY(g->launch(&bl, SK_BEGIN_STEP, g->stream));
      for (int k : kSeqStep) HIP_TRY(g->launch(&bl, k, g->stream));
    } else {
      for (int k : kSeqProfile) HIP_TRY(g->launch(&bl, k, g->stream));
    }
    HIP_TRY(marks.err);
    HIP_TRY(hipEventSynchronize(marks.ev[marks.slot.size()]));
    for (size_t k = 0; k < marks.slot.size(); k++) {
      float ms = 0.f;
      HIP_TRY(hipEventElapsedTime(&ms, marks.ev[k], marks.ev[k + 1]));
      avg_ms[marks.slot[k]] += ms / nsteps;
    }
  }
  return ATHMI_OK;
}

const char* athmi_step_kernel_name(int k) {
  return (k >= 0 && k < NSLOTS) ? kStepNames[k] : "";
}

int athmi_set_stream(athmi_grid* g, void* s) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  HIP_TRY(hipStreamSynchronize(g->stream));
  if (g->own_stream) (void)hipStreamDestroy(g->stream);
  if (s) {
    g->stream = static_cast<hipStream_t>(s);
    g->own_stream = false;
  } else {
    HIP_TRY(hipStreamCreateWithFlags(&g->stream, hipStreamNonBlocking));
    g->own_stream = true;
  }
  g->drop_graph();
  return ATHMI_OK;
}

int athmi_sync(athmi_grid* g) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  HIP_TRY(hipStreamSynchronize(g->stream));
  return ATHMI_OK;
}

int athmi_set_shape(athmi_grid* g, int x2_seg, int persist) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (x2_seg < 1 || x2_seg > 4096 || persist < 0 || persist > 64)
    return fail(ATHMI_EINVAL, "athmi_set_shape: x2_seg in [1,4096], persist in [0,64]");
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->bl.shape.x2_seg = x2_seg;
  g->bl.shape.persist = persist;
  return g->refresh_tiles();
}

// Launch-shape autotuner: every candidate (tile order x x2 marching depth x
// persistent occupancy, then one dimension at a time) runs the same
// `steps` main-loop steps from the same state, timed with HIP events on the
// handle's stream through the step graph; the state and clocks are restored
// after each candidate and the fastest shape is kept.
int athmi_autotune(athmi_grid* g, int steps, int* x2_seg, int* persist, int* xcd_remap,
                   double* ms_per_step) {
  if (!g || steps <= 0) return fail(ATHMI_EINVAL, "athmi_autotune: bad arguments");
  static const int kSeg[] = {2, 4, 8, 16};
  static const int kPersist[] = {0, 1, 2, 4, 8, 16, 32};
  constexpr size_t kFinalists = 6;
  constexpr int kFinalRounds = 3;
  HIP_TRY(hipStreamSynchronize(g->stream));
  std::vector<Clock> hc(g->n);
  HIP_TRY(hipMemcpy(hc.data(), g->dclk, sizeof(Clock) * g->n, hipMemcpyDeviceToHost));
  size_t snap_doubles = 0;
  for (const Inst& I : g->hinst) snap_doubles += NSTATE * I.ps;
  double* snap = nullptr;
  if (hipMalloc(&snap, snap_doubles * sizeof(double)) != hipSuccess)
    return fail(ATHMI_ENOMEM, "athmi_autotune: no room for the state snapshot");
  auto copy_state = [&](bool save) -> int {
    size_t o = 0;
    for (int k = 0; k < g->n; k++) {
      const Inst& I = g->hinst[k];
      double* live = I.state[hc[k].cur];
      const size_t nb = NSTATE * I.ps * sizeof(double);
      HIP_TRY(hipMemcpyAsync(save ? snap + o : live, save ? live : snap + o, nb,
                             hipMemcpyDeviceToDevice, g->stream));
      o += NSTATE * I.ps;
    }
    const athmi_grid::ClockWork work(g);
    HIP_TRY(hipMemcpyAsync(g->dclk, hc.data(), sizeof(Clock) * g->n, hipMemcpyHostToDevice,
                           g->stream));
    g->clock_written = true;
    HIP_TRY(hipStreamSynchronize(g->stream));
    return ATHMI_OK;
  };
  const LaunchShape old = g->bl.shape;
  const bool old_graph = g->use_graph;
  g->use_graph = true;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = copy_state(true);
  double best = HUGE_VAL;
  LaunchShape best_shape = old;
  if (!rc && (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess))
    rc = fail(ATHMI_EHIP, "athmi_autotune: event creation failed");
  // time one shape from the saved state; restores state and clocks
  std::vector<std::pair<double, LaunchShape>> timed;
  auto trial = [&](const LaunchShape& sh, double* out_ms) -> int {
    g->bl.shape = sh;
    int r;
    if ((r = g->refresh_tiles())) return r;
    if ((r = athmi_step(g))) return r;  // capture + first replay, untimed
    // the better of two timed runs from the same state: one short run is
    // sometimes a few percent off (clock ramps, a neighbour's traffic)
    double best_ms = HUGE_VAL;
    for (int rep = 0; rep < 2; rep++) {
      if ((r = copy_state(false))) return r;
      float ms = 0.f;
      if (hipEventRecord(e0, g->stream) != hipSuccess) return fail(ATHMI_EHIP, "event");
      for (int s = 0; s < steps; s++)
        if ((r = athmi_step(g))) return r;
      if (hipEventRecord(e1, g->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
          hipEventElapsedTime(&ms, e0, e1) != hipSuccess)
        return fail(ATHMI_EHIP, "athmi_autotune: event timing failed");
      best_ms = std::min(best_ms, (double)ms / steps);
    }
    *out_ms = best_ms;
    return copy_state(false);
  };
  auto sweep = [&](const LaunchShape& sh) -> int {
    double ms = 0.0;
    const int r = trial(sh, &ms);
    if (!r) timed.emplace_back(ms, sh);
    if (!r && ms < best) {
      best = ms;
      best_shape = sh;
    }
    return r;
  };
  // tile order x x2 marching depth x persistent occupancy
  for (int x2 = 0; !rc && x2 < 2; x2++)
    for (int c = 0; !rc && c < 2; c++)
      for (int a = 0; !rc && a < (int)(sizeof(kSeg) / sizeof(int)); a++)
        for (int b = 0; !rc && b < (int)(sizeof(kPersist) / sizeof(int)); b++) {
          LaunchShape sh = old;
          sh.x2_kind = x2;
          sh.x2_seg = kSeg[a];
          sh.persist = kPersist[b];
          sh.xcd_remap = c;
          rc = sweep(sh);
        }
  // then one dimension at a time at the best shape so far. Each stage times
  // its base again beside the variants: the base's earlier time is the lowest
  // of many short noisy trials, biased low, and a variant measured once would
  // rarely beat it even when faster
  auto stage = [&](const std::vector<LaunchShape>& variants) -> int {
    double stage_best = 0.0;
    LaunchShape stage_shape = best_shape;
    int r = trial(best_shape, &stage_best);
    if (r) return r;
    timed.emplace_back(stage_best, best_shape);
    for (const LaunchShape& sh : variants) {
      double ms = 0.0;
      if ((r = trial(sh, &ms))) return r;
      timed.emplace_back(ms, sh);
      if (ms < stage_best) {
        stage_best = ms;
        stage_shape = sh;
      }
    }
    best = stage_best;
    best_shape = stage_shape;
    return ATHMI_OK;
  };
  auto variants_of = [&](std::initializer_list<int> values, int LaunchShape::*field,
                         int current) {
    std::vector<LaunchShape> v;
    for (int x : values)
      if (x != current) {
        LaunchShape sh = best_shape;
        sh.*field = x;
        v.push_back(sh);
      }
    return v;
  };
  // the x2 marching depth between and around the main sweep's values
  if (!rc)
    rc = stage(variants_of({1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32}, &LaunchShape::x2_seg,
                           best_shape.x2_seg));
  // the corrector's tile height
  if (!rc) rc = stage(variants_of({4, 2, 1}, &LaunchShape::corr_rows, best_shape.corr_rows));
  // tile order of the corrector and final kernels: whole rows or strips
  if (!rc) rc = stage(variants_of({0, 2, 4, 8}, &LaunchShape::strip, best_shape.strip));
  // height of the final-update tiles
  if (!rc)
    rc = stage(variants_of({4, 8, 16}, &LaunchShape::final_rows,
                           final_rows_of(best_shape.final_rows)));
  // fusion depth: the corner emf of Steps 4 and 9 in kernels of their own
  // (0), the Step 9 corners inside the final kernel's tiles (1), and also the
  // Step 4 corners inside the x1 corrector's tiles (2)
  if (!rc) rc = stage(variants_of({0, 1, 2}, &LaunchShape::fuse_corner, best_shape.fuse_corner));
  // single short trials differ by about 1% from run to run: the fastest few
  // shapes, and the stages' winner, run again in turn, and the lowest total
  // time wins
  if (!rc && timed.size() > 1) {
    std::stable_sort(timed.begin(), timed.end(),
                     [](const std::pair<double, LaunchShape>& x,
                        const std::pair<double, LaunchShape>& y) { return x.first < y.first; });
    auto same = [](const LaunchShape& x, const LaunchShape& y) {
      return std::memcmp(&x, &y, sizeof(LaunchShape)) == 0;
    };
    std::vector<LaunchShape> fin{best_shape};
    for (size_t k = 0; k < timed.size() && fin.size() < kFinalists; k++) {
      bool dup = false;
      for (const LaunchShape& f : fin) dup = dup || same(f, timed[k].second);
      if (!dup) fin.push_back(timed[k].second);
    }
    const size_t nf = fin.size();
    std::vector<double> total(nf, 0.0);
    for (int round = 0; !rc && round < kFinalRounds; round++)
      for (size_t f = 0; !rc && f < nf; f++) {
        double ms = 0.0;
        rc = trial(fin[f], &ms);
        total[f] += ms;
      }
    if (!rc) {
      size_t w = 0;
      for (size_t f = 1; f < nf; f++)
        if (total[f] < total[w]) w = f;
      best_shape = fin[w];
      best = total[w] / kFinalRounds;
    }
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (!rc) rc = copy_state(false);
  (void)hipFree(snap);
  g->use_graph = old_graph;
  g->bl.shape = rc ? old : best_shape;
  int rc2 = g->refresh_tiles();
  if (rc) return rc;
  if (rc2) return rc2;
  if (x2_seg) *x2_seg = best_shape.x2_seg;
  if (persist) *persist = best_shape.persist;
  if (xcd_remap) *xcd_remap = best_shape.xcd_remap;
  if (ms_per_step) *ms_per_step = best;
  return ATHMI_OK;
}

int athmi_set_x2_kind(athmi_grid* g, int kind) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (kind != 0 && kind != 1) return fail(ATHMI_EINVAL, "athmi_set_x2_kind: kind must be 0 or 1");
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->bl.shape.x2_kind = kind;
  return g->refresh_tiles();
}

int athmi_set_fusion(athmi_grid* g, int depth) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (depth < 0 || depth > 2)
    return fail(ATHMI_EINVAL, "athmi_set_fusion: depth must be 0, 1 or 2");
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->bl.shape.fuse_corner = depth;
  return g->refresh_tiles();
}

int athmi_set_strip(athmi_grid* g, int tile_cols) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (tile_cols < 0) return fail(ATHMI_EINVAL, "athmi_set_strip: tile_cols must be >= 0");
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->bl.shape.strip = tile_cols;
  return g->refresh_tiles();
}

int athmi_set_final_rows(athmi_grid* g, int rows) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (rows != 4 && rows != 8 && rows != 16)
    return fail(ATHMI_EINVAL, "athmi_set_final_rows: rows must be 4, 8 or 16");
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->bl.shape.final_rows = rows;
  return g->refresh_tiles();
}

int athmi_get_final_rows(const athmi_grid* g, int* rows) {
  if (!g || !rows) return fail(ATHMI_EINVAL, "athmi_get_final_rows: null argument");
  *rows = final_rows_of(g->bl.shape.final_rows);
  return ATHMI_OK;
}

int athmi_get_strip(const athmi_grid* g, int* tile_cols) {
  if (!g || !tile_cols) return fail(ATHMI_EINVAL, "athmi_get_strip: null argument");
  *tile_cols = g->bl.shape.strip;
  return ATHMI_OK;
}

int athmi_get_fusion(const athmi_grid* g, int* depth) {
  if (!g || !depth) return fail(ATHMI_EINVAL, "athmi_get_fusion: null argument");
  *depth = g->bl.shape.fuse_corner;
  return ATHMI_OK;
}

int athmi_get_x2_kind(const athmi_grid* g, int* kind) {
  if (!g || !kind) return fail(ATHMI_EINVAL, "athmi_get_x2_kind: null argument");
  *kind = g->bl.shape.x2_kind;
  return ATHMI_OK;
}

int athmi_set_corr_rows(athmi_grid* g, int rows) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (rows != 1 && rows != 2 && rows != 4)
    return fail(ATHMI_EINVAL, "athmi_set_corr_rows: rows must be 1, 2 or 4");
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->bl.shape.corr_rows = rows;
  return g->refresh_tiles();
}

int athmi_get_shape(const athmi_grid* g, int* x2_seg, int* persist, int* xcd_remap,
                    int* corr_rows) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  if (x2_seg) *x2_seg = g->bl.shape.x2_seg;
  if (persist) *persist = g->bl.shape.persist;
  if (xcd_remap) *xcd_remap = g->bl.shape.xcd_remap;
  if (corr_rows) *corr_rows = g->bl.shape.corr_rows;
  return ATHMI_OK;
}

int athmi_set_tile_order(athmi_grid* g, int xcd_remap) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  HIP_TRY(hipStreamSynchronize(g->stream));
  g->bl.shape.xcd_remap = xcd_remap ? 1 : 0;
  return g->refresh_tiles();
}

int athmi_use_graph(athmi_grid* g, int on) {
  if (!g) return fail(ATHMI_EINVAL, "null handle");
  g->use_graph = on != 0;
  return ATHMI_OK;
}

int athmi_device_state(athmi_grid* g, int inst, double** planes, int* pitch) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  Clock c;
  if ((rc = g->read_clock(inst, c))) return rc;
  const Inst& I = g->hinst[inst];
  for (int q = 0; q < NSTATE; q++) planes[q] = I.state[c.cur] + q * I.ps;
  if (pitch) *pitch = I.pitch;
  return ATHMI_OK;
}

// ---- problem generators ------------------------------------------------------
static int upload_fresh(athmi_grid* g, int inst, const HostState& S) {
  return athmi_upload(g, inst, S.gas.data(), S.b1i.data(), S.b2i.data(), S.b3i.data());
}

int athmi_pgen_blast(athmi_grid* g, int inst, double radius, double pamb, double prat, double b0,
                     double angle_deg, double cx, double cy) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  const HostGeom G = geom_of(g, inst);
  HostState S(G);
  problem_blast(G, S, radius, pamb, prat, b0, angle_deg, cx, cy);
  return upload_fresh(g, inst, S);
}

int athmi_pgen_field_loop(athmi_grid* g, int inst, double rad, double amp, double vflow,
                          int iprob) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  const HostGeom G = geom_of(g, inst);
  HostState S(G);
  problem_field_loop(G, S, rad, amp, vflow, iprob);
  return upload_fresh(g, inst, S);
}

int athmi_pgen_cpaw2d(athmi_grid* g, int inst, double angle, double b_par, double b_perp,
                      double pres, double v_par, double* lambda) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  const HostGeom G = geom_of(g, inst);
  HostState S(G);
  const double lam = problem_cpaw2d(G, S, angle, b_par, b_perp, pres, v_par, &g->cpaw_soln[inst]);
  if (lambda) *lambda = lam;
  return upload_fresh(g, inst, S);
}

int athmi_cpaw2d_l1(athmi_grid* g, int inst, double* out) {
  int rc = check_inst(g, inst);
  if (rc) return rc;
  if (g->cpaw_soln[inst].empty())
    return fail(ATHMI_ESTATE, "athmi_cpaw2d_l1: instance was not set up by athmi_pgen_cpaw2d");
  const HostGeom G = geom_of(g, inst);
  HostState S(G);
  if ((rc = athmi_download(g, inst, S.gas.data(), S.b1i.data(), S.b2i.data(), S.b3i.data())))
    return rc;
  cpaw2d_errors(G, S, g->cpaw_soln[inst], out);
  return ATHMI_OK;
}

}  // extern "C"
