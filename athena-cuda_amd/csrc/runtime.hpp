// runtime.hpp -- internal: the handle behind athmi_grid (device state of the
// instances, tile work-list, stream and step graph) shared by the C-ABI
// translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "athmi.h"
#include "host_problems.hpp"
#include "step_kernels.hpp"

ATHMI_DECLARE_VARIANT(exact)
ATHMI_DECLARE_VARIANT(fast)

using namespace athmi;

namespace athmi_rt {

extern thread_local std::string g_err;

inline int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(expr)                                                                    \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess)                                                                \
      return fail(ATHMI_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_));        \
  } while (0)

typedef hipError_t (*LaunchFn)(const void*, int, hipStream_t);

// transfer.hip: caller layout (gas[sy*sx][8] | b1i | b2i | b3i in `stage`)
// <-> the SoA planes of one state buffer
}  // namespace athmi_rt
namespace athmi {
hipError_t launch_state_unpack(const double* stage, double* st, size_t ps, int pitch, int sx,
                               int sy, hipStream_t s);
hipError_t launch_state_pack(const double* st, double* stage, size_t ps, int pitch, int sx,
                             int sy, hipStream_t s);
// the clocks' heads -> host memory; one head -> the device, then `count` -> host memory
hipError_t launch_clock_publish(const Clock* clk, ClockHead* heads, int n, hipStream_t s);
hipError_t launch_clock_set(Clock* clk, const ClockHead& head, unsigned long long* done,
                            unsigned long long count, hipStream_t s);
// dense [NSTATE][sy][sx] on the device <-> the planes of one state buffer
hipError_t launch_state_dense(double* st, double* dense, size_t ps, int pitch, int sx, int sy,
                              int to_planes, hipStream_t s);
}  // namespace athmi
namespace athmi_rt {

// kernel sequences of the reference's routines
// (a main-loop step is started by the k_end before it, or by SK_BEGIN_STEP
// once the host has written the clock: athmi_grid::clock_written)
const int kSeqStep[] = {SK_PRED, SK_CORNER_P, SK_FINISH, SK_END_STEP};
const int kSeqIntegrate[] = {SK_BEGIN_ONCE, SK_PRED, SK_CORNER_P_CARRY, SK_FINISH_BARE,
                             SK_END_ONCE};
// the step as its separate kernels
const int kSeqProfile[] = {SK_BEGIN_STEP, SK_PRED_X1, SK_PRED_X2, SK_CORNER_P,   SK_CORR,
                           SK_CORR2,      SK_CORNER_C, SK_FINAL,  SK_GHOST_NEXT, SK_END_STEP};
const int kSeqNewDt[] = {SK_CLEAR, SK_DTI, SK_DT_FINAL};
const int kSeqDivb[] = {SK_CLEAR, SK_DIVB};
const char* const kStepNames[] = {"k_begin",   "k_pred_x1",   "k_pred_x2",      "k_corner<pred>",
                                  "k_corr<1>", "k_corr<2>",   "k_corner<corr>", "k_final",
                                  "k_ghost",   "k_end",       "k_pred",         "k_pred_pair",
                                  "k_corr_both", "k_corr_final"};
static_assert(sizeof(kSeqProfile) / sizeof(int) == NSEPARATE, "a slot per separate kernel");
static_assert(sizeof(kStepNames) / sizeof(*kStepNames) == NSLOTS, "a name per slot");

inline size_t round_up(size_t a, size_t b) { return (a + b - 1) / b * b; }

}  // namespace athmi_rt

using namespace athmi_rt;

struct athmi_grid {
  int n = 0;
  int variant = ATHMI_EXACT;
  std::vector<athmi_desc> desc;
  std::vector<Inst> hinst;
  Inst* dinst = nullptr;  // the device lists of bl
  Clock* dclk = nullptr;
  double* dmem = nullptr;
  size_t dmem_bytes = 0;
  BatchLaunch bl{};
  LaunchFn launch = nullptr;
  hipStream_t stream = nullptr;
  bool own_stream = false;
  bool use_graph = true;
  hipGraphExec_t graph = nullptr;
  bool clock_written = true;  // the host wrote a clock since the last main-loop step
  // the clocks as the host last saw them (pinned memory the device writes), and
  // how much work that changes them had been queued by then, of clock_work by now.
  // clk_mu: the heads and the launches that read or write them, and the capture of
  // the step graph (a launch beside it would be captured too); a thread may read
  // the clocks while another steps
  ClockHead* heads = nullptr;
  unsigned long long heads_at = ~0ull;
  std::atomic<unsigned long long> clock_work{0};
  std::mutex clk_mu;
  // writes of clocks queued, and (behind the heads) how many have reached the device
  unsigned long long set_count = 0;
  unsigned long long* set_done = nullptr;
  // the caller has captured work of this handle, which it may replay at any
  // time: the heads are then fetched at every read, and every step starts itself
  std::atomic<bool> caller_captured{false};
  std::vector<std::vector<double>> cpaw_soln;  // initial cpaw2d states (8 planes)
  void* outbuf = nullptr;                      // device staging of the output formats
  size_t outbuf_bytes = 0;

  void drop_graph() {
    if (graph) (void)hipGraphExecDestroy(graph);
    graph = nullptr;
  }
  // the device lists: every instance, and (a batch that mixes the solvers)
  // those of each solver, each with its own tile numbering
  int refresh_tiles() {
    std::vector<unsigned char> img(inst_lists_bytes(n));
    unsigned char* base = reinterpret_cast<unsigned char*>(dinst);
    size_t used = 0;
    auto add = [&](InstList& L, int flux) {
      Inst* I = reinterpret_cast<Inst*>(img.data() + used);
      int m = 0, tot[NKINDS] = {0};
      for (int k = 0; k < n; k++)
        if (flux < 0 || hinst[k].flux == flux) I[m++] = hinst[k];
      int* first = reinterpret_cast<int*>(I + m);
      march_of(I, m, I[0].flux == ATHMI_FLUX_HLLE, bl.ncu, L);
      LaunchShape shape = bl.shape;
      shape.cf_rows = L.cf_rows;
      for (int k = 0; k < m; k++)
        for (int kind = 0; kind < NKINDS; kind++) {
          first[kind * m + k] = I[k].tile0[kind] = tot[kind];
          tot[kind] += tiles_of(kind, I[k].nx1, I[k].nx2, shape);
        }
      L.insts = reinterpret_cast<const Inst*>(base + used);
      L.ninst = m;
      for (int kind = 0; kind < NKINDS; kind++) L.ntiles[kind] = tot[kind];
      used += inst_list_bytes(m);
    };
    bl.outgrows_cache = dmem_bytes > kInfinityCacheBytes;
    int count[2] = {0, 0};
    bl.stale_ghosts = 0;
    bl.thin = 0;
    for (const Inst& I : hinst) {
      count[I.flux]++;
      if (I.nx1 < 4 || I.nx2 < 4) bl.thin = 1;
      if (ghost_fill_reads_stale(I)) bl.stale_ghosts = 1;
    }
    add(bl.all, -1);
    for (int f = 0; f < 2; f++) {
      if (count[f] == n) bl.of_flux[f] = bl.all;
      else if (count[f] == 0) bl.of_flux[f] = InstList{};
      else add(bl.of_flux[f], f);
    }
    HIP_TRY(hipMemcpy(dinst, img.data(), used, hipMemcpyHostToDevice));
    drop_graph();
    return ATHMI_OK;
  }
  // lives around the queueing of work that changes the clocks. The work counts
  // once it is queued: a read that another thread began before then does not pass
  // for one of after
  struct ClockWork {
    athmi_grid* g;
    explicit ClockWork(athmi_grid* g) : g(g) {
      hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
      if (!g->caller_captured && hipStreamIsCapturing(g->stream, &st) == hipSuccess &&
          st != hipStreamCaptureStatusNone) {
        g->wait_clock_set();
        g->caller_captured = true;
      }
    }
    ~ClockWork() { g->clock_work++; }
    ClockWork(const ClockWork&) = delete;
  };
  // waits for the stream, and for the null stream as a blocking copy would: the
  // caller may have replayed captured work there, or written the state's planes.
  // The heads (whose mutex is held) are then the device's
  int fetch_clocks() {
    HIP_TRY(hipStreamSynchronize(nullptr));
    const unsigned long long work = clock_work;
    if (heads_at != work || caller_captured)
      HIP_TRY(launch_clock_publish(dclk, heads, n, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    heads_at = work;
    return ATHMI_OK;
  }
  int read_clock(int k, Clock& c) {
    std::lock_guard<std::mutex> lk(clk_mu);
    const int rc = fetch_clocks();
    if (rc) return rc;
    std::memcpy(&c, &heads[k], sizeof(ClockHead));
    return ATHMI_OK;
  }
  // after read_clock (which has waited for the stream) of the same instance.
  // Work the caller has captured may be replayed on another stream next: it
  // must find the clock written
  int write_clock_head(int k, const Clock& c) {
    std::lock_guard<std::mutex> lk(clk_mu);
    clock_written = true;
    std::memcpy(&heads[k], &c, offsetof(Clock, divb_bits));
    HIP_TRY(launch_clock_set(dclk + k, heads[k], set_done, set_count + 1, stream));
    set_count++;
    if (caller_captured) HIP_TRY(hipStreamSynchronize(stream));
    return ATHMI_OK;
  }
  // until the last write has reached the device. For the first capture, which
  // forbids a wait for its stream; the bound (far above a launch of one wave) keeps
  // a lost device from holding the caller
  void wait_clock_set() const {
    const auto t0 = std::chrono::steady_clock::now();
    while (__atomic_load_n(set_done, __ATOMIC_ACQUIRE) != set_count &&
           std::chrono::steady_clock::now() - t0 < std::chrono::seconds(10))
      std::this_thread::yield();
  }
};

// the reference's Grid geometry of one instance (init_grid.c:25-118)
inline HostGeom geom_of(const athmi_grid* g, int inst) {
  const athmi_desc& d = g->desc[inst];
  const Inst& I = g->hinst[inst];
  HostGeom G;
  G.Nx1 = d.nx1;
  G.Nx2 = d.nx2;
  G.is = I.is;
  G.ie = I.ie;
  G.js = I.js;
  G.je = I.je;
  G.sx = I.sx;
  G.sy = I.sy;
  G.dx1 = I.dx1;
  G.dx2 = I.dx2;
  G.x1_0 = d.x1min;
  G.x2_0 = d.x2min;
  G.idisp = -I.is;
  G.jdisp = -I.js;
  G.gamma_1 = I.g1;
  return G;
}

inline int issue_seq(athmi_grid* g, const int* seq, size_t n) {
  const athmi_grid::ClockWork work(g);
  for (size_t k = 0; k < n; k++) HIP_TRY(g->launch(&g->bl, seq[k], g->stream));
  return ATHMI_OK;
}
#define issue(g, seq) issue_seq((g), (seq), sizeof(seq) / sizeof((seq)[0]))

