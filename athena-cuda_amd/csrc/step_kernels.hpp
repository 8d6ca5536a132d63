// step_kernels.hpp -- data layout shared by the host side and the HIP kernels
// of the CTU+CT step. One "instance" is one 2-D grid (the reference's Grid,
// athena.h:106-120); the plain step is a batch of one instance.
#pragma once
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstddef>
#include <cstdint>

namespace athmi {

// field planes of a state buffer, in Gas order (athena.h:43-52) + interface B
enum Field { F_D = 0, F_M1, F_M2, F_M3, F_E, F_B1C, F_B2C, F_B3C, F_B1I, F_B2I, F_B3I, NSTATE = 11 };

// scratch planes (each Cons1D-shaped group is 7 planes d,Mx,My,Mz,E,By,Bz)
enum Scratch {
  S_UL1 = 0,    // x1-face left states (conserved), predictor
  S_UR1 = 7,    // x1-face right states
  S_F1 = 14,    // x1 predictor fluxes
  S_UL2 = 21,   // x2-face left states (x2 sweep order d,M2,M3,M1,E,B3c,B1c)
  S_UR2 = 28,
  S_F2 = 35,    // x2 predictor fluxes
  S_F1C = 42,   // x1 corrector fluxes
  S_F2C = 49,   // x2 corrector fluxes
  S_ECC = 56,   // cell-centred emf3 at t^n
  S_EMF = 57,   // corner emf3 (predictor, then corrector)
  S_ECH = 58,   // cell-centred emf3 at t^{n+1/2}
  NSCRATCH = 59
};

// optional planes of the predictor's primitive face states, after the 1/2 dt
// MHD source (the Wl, Wr that Steps 1e / 2e hand to the Riemann solver)
enum PrimSave { P_WL1 = 0, P_WR1 = 7, P_WL2 = 14, P_WR2 = 21, NPRIMS = 28 };

enum BcKind { BC_REFLECT = 1, BC_OUTFLOW = 2, BC_PERIODIC = 4 };

constexpr size_t kInfinityCacheBytes = (size_t)256 << 20;

constexpr int kDtSlots = 256;  // partial max slots of the fused dt reduction

// Failure bits of an instance, raised by the step on the state it produces
// (the reference only floors, convert_var.c:49 and new_dt.c:54-55, and steps
// on). Once any is set the main-loop step no longer runs on that instance.
enum FailBits {
  FAIL_NONFINITE = 1,  // a NaN or infinity in d, M1..M3, E or the cell-centred B
  FAIL_DENSITY = 2,    // d <= 0
  FAIL_PRESSURE = 4,   // Gamma_1 (E - KE - ME) below TINY_NUMBER: the pressure floor engages
};

// Device-resident clock of one instance (Grid.dt/time/nstep of athena.h:113-114
// plus the main-loop limits of main.c:217-218).
struct Clock {
  double dt, time, tlim, cour_no;
  double dts;  // dt of the step under way or next: dt, clamped to reach tlim exactly
  double tpause;  // the main-loop step does not run once time >= tpause (an output is due)
  int nstep, nlim, active, cur;  // cur: which ping-pong state buffer holds the state
  int fail;        // FailBits of the states produced so far (0: healthy)
  int fail_nstep;  // nstep of the first state that raised a bit (-1: none)
  int fail_stop;   // FailBits that stop the main-loop step (the others are only reported)
  int steps_run;
  unsigned long long divb_bits;           // max |div B| (bit pattern), diagnostics
  unsigned long long dti_slot[kDtSlots];  // bit patterns of non-negative doubles
};

// a clock without its dt slots, as the host keeps it
struct ClockHead {
  unsigned long long w[offsetof(Clock, dti_slot) / 8];
};
static_assert(offsetof(Clock, dti_slot) % 8 == 0 && offsetof(Clock, divb_bits) % 8 == 0,
              "the head is whole words");

struct Inst {
  int nx1, nx2, is, ie, js, je, sx, sy, pitch, flux;
  int bc[4];          // ix1, ox1, ix2, ox2
  double dx1, dx2, gamma, g1, g2;
  double* state[2];   // two ping-pong buffers of NSTATE planes
  double* scratch;    // NSCRATCH planes
  double* prims;      // NPRIMS planes written by SK_PRED_SAVE
  size_t ps;          // plane stride in doubles
  Clock* clk;
  // first global tile of this instance for each kernel kind
  int tile0[9];
};

// Tile kinds (one per kernel family); tile counts per instance come from
// tiles_of() below so host and device agree on the decomposition.
enum KernelKind {
  K_PRED_X1 = 0,  // cells is-3..ie+3 of rows js-2..je+2 in one sequence, kX1Faces to a tile
  K_PRED_X2,      // columns is-2..ie+2 of segments of faces js-1..je+2, kX2Block to a
                  // tile, in chunks or in one sequence (x2_aligned)
  K_CORR,         // cells [js-1,je+1] x [is-1,ie+1]
  K_CORNER_P,     // corners [js-1,je+2] x [is-1,ie+2]
  K_CORNER_C,     // corners [js,je+1] x [is,ie+1]
  K_FINAL,        // cells [js,je] x [is,ie]
  K_GHOST,        // ghost cells of all planes
  K_INTERIOR,     // cells [js,je] x [is,ie]
  K_CORR_FINAL,   // cells [js,je] x [is,ie] in strips of kCfCols columns, cf_rows rows each
  NKINDS
};

// Work decomposition (tile sizes) shared by host and device
// threads of a predictor-x1 tile (one row segment): two waves, so that the
// workgroups resident on a CU pass their block barriers independently (at one
// wave per SIMD, 4096^2: 2.56 ms with 256 threads, 2.45 with 64, 2.40 with
// 128; at two waves per SIMD the three are within 1%)
constexpr int kX1Block = 128;
constexpr int kX1Faces = kX1Block - 3;      // faces produced per x1 tile
constexpr int kX2Block = 64;                // columns of a predictor-x2 tile
constexpr int kTileX = 64, kTileY = 4;      // 2-D tiles of the cell/corner kernels
constexpr int kCfCols = 62;                 // columns a corrector-and-final wave finishes
constexpr int kGhostBlock = 256;

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

// rows of a final-update tile (64 x 4, 8 or 16 cells; anything else: 4)
inline int final_rows_of(int rows) { return (rows == 8 || rows == 16) ? rows : kTileY; }

// Default faces marched per x2-predictor lane for `cols` lane-columns of x2
// faces (64-column chunks x rows over the batch): shorter segments give more
// workgroups (less tail at the end of the launch) for more halo rows per face.
// The measured best depth grows about as sqrt(cols)/50: 1 at 256^2, 3 at
// 512^2-1024^2, 5 at 2048^2, 8-24 at 4096^2, all within 2-3% of each other.
inline int default_x2_seg(long cols) {
  const long s = std::lround(std::sqrt((double)cols) / 50.0);
  return (int)(s < 1 ? 1 : (s > 16 ? 16 : s));
}

// whether an instance's set_bvals reads ghosts as they were before it (an
// inner reflecting fill across fewer cells than the four ghost layers copies
// outer ghosts the outer fill has not reached yet, set_bvals.c:312-366)
inline bool ghost_fill_reads_stale(const Inst& g) {
  return (g.bc[0] == BC_REFLECT && g.nx1 < 4) || (g.bc[2] == BC_REFLECT && g.nx2 < 4);
}

// Launch shape chosen by the autotuner
struct LaunchShape {
  int x2_seg;        // faces marched per thread in the x2 predictor
  int persist;       // 0: one tile per workgroup; >0: workgroups per CU of a persistent grid
  int xcd_remap;     // 1: contiguous runs of tiles per XCD (L2 locality), 0: launch order
  int corr_rows;     // rows of a corrector tile (kTileX x corr_rows faces): 1, 2 or 4
  int x2_kind;       // x2 predictor: 0 = stencil marched in registers (one wave per
                     // SIMD), 1 = stencil marched in LDS slots (two waves per SIMD)
  int fuse_corner;   // fusion depth. 1: the Step 9 corner emf is computed inside the
                     // final kernel's tiles (no k_corner<corr> launch, no corner plane
                     // round trip); 2: also the Step 4 corner emf inside the x1
                     // corrector's tiles (no k_corner<pred> launch)
  int strip;         // tile order of the corrector and final kernels: 0 = row by row,
                     // s > 0 = strips of s tile columns walked row by row
  int final_rows;    // rows of a final-update tile: 4, 8 or 16 (final_rows_of)
  int cf_rows;       // rows a corrector-and-final wave marches (march_of, per list)
};

// Whether a grid's x2 tiles start on a cache line: whole chunks of 64 columns
// from column 0 (the pitch is a multiple of 16), where they leave less than 3%
// of the lanes idle (HLLE, bound by memory: 3000^2 3303 -> 3255 us a step, 4096^2
// 6165 -> 6097; Roe within 0.3%); otherwise the columns follow each other across
// the segments' ends (at 512^2 whole chunks leave 10% of the lanes idle)
__host__ __device__ inline bool x2_aligned(int nx1) {
  const int lanes = (nx1 + 6 + kX2Block - 1) / kX2Block * kX2Block;
  return 100 * (lanes - (nx1 + 4)) < 3 * lanes;
}

// number of tiles of kind k for a grid of nx1 x nx2 zones
inline int tiles_of(int k, int nx1, int nx2, const LaunchShape& sh) {
  const int sx = nx1 + 8;
  switch (k) {
    case K_PRED_X1: return cdiv((nx2 + 4) * (nx1 + 6) - 3, kX1Faces);
    case K_PRED_X2: {
      const int nseg = cdiv(nx2 + 4, sh.x2_seg);
      return x2_aligned(nx1) ? cdiv(nx1 + 6, kX2Block) * nseg : cdiv((nx1 + 4) * nseg, kX2Block);
    }
    case K_CORR:
      // tiles of one row without strips follow each other across the rows' ends
      if (sh.corr_rows == 1 && sh.strip == 0 && sh.fuse_corner < 2)
        return cdiv((nx1 + 2) * (nx2 + 2), kTileX);
      return cdiv(nx1 + 3, kTileX) * cdiv(nx2 + 3, sh.corr_rows);
    case K_CORNER_P: return cdiv((nx1 + 3) * (nx2 + 3), kTileX * kTileY);
    case K_CORNER_C: return cdiv((nx1 + 1) * (nx2 + 1), kTileX * kTileY);
    case K_FINAL: return cdiv(nx1, kTileX) * cdiv(nx2, final_rows_of(sh.final_rows));
    case K_CORR_FINAL: return cdiv(nx1, kCfCols) * cdiv(nx2, sh.cf_rows);
    case K_GHOST: return cdiv(8 * sx + (nx2 + 1) * 8, kGhostBlock);
    default: return cdiv(nx1, kTileX) * cdiv(nx2, kTileY);
  }
}

// A list of instances on the device and its tile totals per kernel kind. In
// device memory the descriptors are followed by the first tiles again, as a
// dense table [NKINDS][ninst] that find_inst searches (a list of one has none).
struct InstList {
  const Inst* insts;
  int ninst;
  int ntiles[NKINDS];
  int cf_rows;     // rows of a corrector-and-final march
  bool cf_worth;   // whether it beats the separate launches (march_of)
};

// The corrector-and-final march of m instances of one solver on ncu CUs. A march
// of r rows evaluates r + 1 x2 face rows and the x1 fluxes of r + 2 rows; the times
// follow r + 1 (measured with 4 to 24 rows at nine sizes). Twelve (HLLE) or eight
// (Roe) marches run per CU at a time, so the rows are those with the least rounds
// x (r + 1): a nearly empty last round costs as much as a full one (Roe
// 2048 x 1536, two rounds of 13 rows 1248 us a step, of 20 rows 1370, three of 10
// 1313; 1200^2, one round of 12 rows 609, two of 10 697).
// It is worth it where enough of the lanes' rows in these rounds finish cells; the
// fewer the rounds, the more, since all waves then load and compute in step. Roe:
// 1024^2 (0.83 in one round) 462 -> 466 us, 1200^2 (0.87) 629 -> 609, 2048 x 1536 (0.89
// in two) 1309 -> 1248, 4096^2 (0.92 in nine) 6.87 -> 6.27 ms, 100 grids of 200 x 300
// (0.70 at 10 rows) 2.77 -> 2.72, 400 of 128^2 (0.60) 3.08 -> 3.28. HLLE: 768^2
// (0.62 in one) 234 -> 244, 1024^2 (0.79) 396 -> 395, 1200^2 (0.84) 551 -> 513,
// 2048 x 1536 (0.87) 1152 -> 1060, 4096^2 (0.93 in five) 6.09 -> 5.28 ms, 400 grids of
// 128^2 (0.52 at 10 rows) 2.78 -> 2.70. Near the lines the two ways differ by 1%.
inline void march_of(const Inst* insts, int m, bool hlle, int ncu, InstList& list) {
  const long slots = (hlle ? 12L : 8L) * (ncu > 0 ? ncu : 1);
  double cells = 0.0;
  for (int k = 0; k < m; k++) cells += (double)insts[k].nx1 * insts[k].nx2;
  long best = 0, rounds = 0;
  for (int r = 4; r <= 24; r++) {
    long t = 0;
    for (int k = 0; k < m; k++) t += (long)cdiv(insts[k].nx1, kCfCols) * cdiv(insts[k].nx2, r);
    const long n = (t + slots - 1) / slots;
    if (r > 4 && n * (r + 1) >= best) continue;
    best = n * (r + 1);
    rounds = n;
    list.cf_rows = r;
  }
  const double use = cells / ((double)best * slots * kCfCols);
  list.cf_worth = use >= (hlle ? 0.55 + 0.25 / rounds : 0.70 + 0.14 / rounds);
}

// device bytes of a list of n instances, whole descriptors' alignment: the next
// list starts behind it
constexpr size_t inst_list_bytes(size_t n) {
  return (n * (sizeof(Inst) + sizeof(int) * NKINDS) + alignof(Inst) - 1) / alignof(Inst) *
         alignof(Inst);
}
// of the list of all n instances and the two solvers' lists, which share them
// (two odd shares round up once more than their sum does)
constexpr size_t inst_lists_bytes(size_t n) { return 2 * inst_list_bytes(n) + alignof(Inst); }

// Everything a launcher needs for one batch (the instances, the tuned shape
// and the CU count). The kernels that are compiled per Riemann solver take the
// list of the instances that use it; the others take them all.
struct BatchLaunch {
  InstList all;
  InstList of_flux[2];  // by solver (kFluxRoe, kFluxHlle); ninst = 0: not in use
  int stale_ghosts;  // some instance's ghost fill reads stale ghosts (ghost_map.hpp)
  int thin;          // some instance has Nx1 or Nx2 < 4: ghosts may copy ghosts
  // the batch's state and scratch planes outgrow the Infinity Cache: the
  // predictors store past it (measured: 600^2, 247 MB, is slower so, 700^2,
  // 330 MB, faster)
  bool outgrows_cache;
  LaunchShape shape;
  int ncu;
  // called (if set) after every launch of a step's kernel, with its StepSlot
  void (*launched)(void* arg, int slot) = nullptr;
  void* launched_arg = nullptr;
  // a batch of one: its only list, read through descriptor `ins`
  void single(const Inst* ins, int flux) {
    all.insts = ins;
    of_flux[flux] = all;
    of_flux[1 - flux] = InstList{};
  }
};

// Kernels of a main-loop step, as athmi_profile_steps numbers them: the separate
// kernels, then those that hold several stages
enum StepSlot {
  SLOT_BEGIN = 0, SLOT_PRED_X1, SLOT_PRED_X2, SLOT_CORNER_P, SLOT_CORR1, SLOT_CORR2, SLOT_CORNER_C,
  SLOT_FINAL, SLOT_GHOST, SLOT_END,
  NSEPARATE,
  SLOT_PRED = NSEPARATE, SLOT_PRED_PAIR, SLOT_CORR_BOTH, SLOT_CORR_FINAL,
  NSLOTS
};

// Kernels of the pipeline, launched one at a time by athmi_<variant>_launch
enum StepKernel {
  SK_BEGIN_STEP = 0,  // k_begin, main-loop mode
  SK_BEGIN_ONCE,      // k_begin, unconditional (drop-in integrate_2d)
  SK_PRED_X1,
  SK_PRED_X2,
  SK_CORNER_P,
  SK_CORR,            // corrector, x1 faces
  SK_CORR2,           // corrector, x2 faces and emf3 at t^{n+1/2}
  SK_CORNER_C,
  SK_FINAL,
  SK_GHOST_CUR,       // set_bvals on the current buffer
  SK_GHOST_NEXT,      // set_bvals on the buffer this step produces (respects the clock)
  SK_GHOST_CARRY,     // carry current ghost values into the produced buffer
  SK_END_STEP,        // k_end, main-loop mode: the clock of this step, and the next one's start
  SK_END_ONCE,        // k_end, swap only
  SK_CLEAR,           // reset reduction slots
  SK_DTI,             // new_dt partial maxima
  SK_DT_FINAL,        // new_dt.c:93-97
  SK_DIVB,
  SK_PRED,            // both predictors, in one launch or two by the launch shape
  SK_PRED_SAVE,       // in one, storing the primitive face states too (Inst::prims), for the
                      // adjoint's re-run
  SK_CORR_BOTH,       // both corrector parts, in one launch or two by the launch shape
  SK_FINISH,          // SK_CORR_BOTH, SK_CORNER_C and SK_FINAL_GHOST; one launch per solver on
                      // large batches, which then writes no corrector planes
  SK_FINISH_BARE,     // the same without the ghosts (SK_FINAL)
  SK_FINAL_GHOST,     // SK_FINAL and SK_GHOST_NEXT: one launch where every ghost copies a
                      // non-ghost cell
  SK_CORNER_P_CARRY,  // SK_CORNER_P and SK_GHOST_CARRY, in one launch where both are launched
  SK_COUNT
};

}  // namespace athmi

// Launcher exported by each arithmetic variant of step_kernels.hip
// (athmi_exact_launch built with -ffp-contract=off, athmi_fast_launch with FMA).
#define ATHMI_DECLARE_VARIANT(V) \
  extern "C" hipError_t athmi_##V##_launch(const void* bl, int kernel, hipStream_t s);
