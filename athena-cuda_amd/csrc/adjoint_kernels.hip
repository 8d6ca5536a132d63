// adjoint_kernels.hip -- reverse of one CTU+CT step (__integrate_2d__.c:100-537)
// followed by set_bvals (set_bvals.c:114-1031), for one instance.
//
// Given the adjoint of the step's output state (aout) and the forward scratch
// of the step recomputed from its input state S^n (predictor face states,
// conserved and primitive, and fluxes, predictor corner emf, corrector
// fluxes), the kernels below run the step's stages in reverse and accumulate
// the adjoint of S^n into ain:
//   fold        set_bvals: each cell adds the adjoints of the ghosts that copy it
//   update      Steps 9, 11a, 11b, 13 -> corrector fluxes, corner emf, identity
//   correct     Steps 8b / 8c: corrector Riemann fluxes -> corrected face states;
//               Step 7: emf3 at t^{n+1/2} -> half-step face fields, predictor fluxes
//   transverse  Steps 5, 6 and the half-step face fields of Step 4
//   predict     Steps 1c-1e / 2c-2e: sources, prim->cons, predictor fluxes; Step 3
//   plm         Steps 1b / 2b: the PLM reconstruction
//   plm_gather  Steps 1a / 2a: cons->prim
// The corner emf of Steps 9 and 4 is reversed by its inputs: the corrector and
// predictor fluxes' By/Bz and the cell-centred emf3 gather their corners'
// adjoints where their own reverse reads them.
// One launch holds both sweeps (and Step 7, Step 3 beside them), so a reversed
// step is seven launches on one stream. The stages that hold few waves per SIMD
// (correct, predict, plm) run in workgroups of one wave over a row-after-row
// sequence of cells: at 512^2 whole 64-wide tiles left a tenth of the lanes idle.
// Nonlinear stages recompute their forward values with the reference's
// evaluation order (this file is built with -ffp-contract=off, like the exact
// forward kernels), so every branch is the one the forward pass took. The adjoint
// of the input state takes FP64 atomic adds where several threads of one launch
// reach a cell: from the predictor faces' sources and Step 3, and from the two
// sweeps' cons->prim. Their order, and so the last bits, vary from run to run; the
// deterministic reverse stores the faces' terms, gathers them in order and runs
// the two sweeps' gathers one after the other.
#include <hip/hip_runtime.h>

#include "adjoint_device.hpp"
#include "adjoint_kernels.hpp"
#include "ghost_map.hpp"

namespace athmi {
namespace adjk {

using namespace adj;

__device__ __forceinline__ void ADD(double* plane, uint32_t k, double v) {
  unsafeAtomicAdd(plane + k, v);
}
__device__ __forceinline__ Cons7 ld7(const double* base, size_t ps, uint32_t k) {
  return Cons7{base[k], base[ps + k], base[2 * ps + k], base[3 * ps + k], base[4 * ps + k],
               base[5 * ps + k], base[6 * ps + k]};
}
__device__ __forceinline__ void st7(double* base, size_t ps, uint32_t k, const Cons7& u) {
  base[k] = u.d; base[ps + k] = u.mx; base[2 * ps + k] = u.my; base[3 * ps + k] = u.mz;
  base[4 * ps + k] = u.e; base[5 * ps + k] = u.by; base[6 * ps + k] = u.bz;
}
__device__ __forceinline__ void st7(double* base, size_t ps, uint32_t k, const Prim7& w) {
  base[k] = w.d; base[ps + k] = w.vx; base[2 * ps + k] = w.vy; base[3 * ps + k] = w.vz;
  base[4 * ps + k] = w.p; base[5 * ps + k] = w.by; base[6 * ps + k] = w.bz;
}
__device__ __forceinline__ Prim7 ld7p(const double* base, size_t ps, uint32_t k) {
  return Prim7{base[k], base[ps + k], base[2 * ps + k], base[3 * ps + k], base[4 * ps + k],
               base[5 * ps + k], base[6 * ps + k]};
}

constexpr int kWave = 64;     // workgroup of the stages with few waves per SIMD
constexpr int kCells = 256;   // workgroup of the others

// (j, i) of thread `tid` of block b of `n` threads in the range [j0, j1] x
// [i0, i1], taken row after row
__device__ __forceinline__ bool range_ij(int b, int n, int j0, int j1, int i0, int i1, int& j,
                                         int& i) {
  const int e = b * n + (int)threadIdx.x, w = i1 - i0 + 1, r = e / w;
  j = j0 + r;
  i = i0 + (e - r * w);
  return j <= j1;
}

// ---------------------------------------------------------------------------
// The adjoint of set_bvals: the thread of a non-ghost cell sums, field by
// field, the adjoints of the ghosts whose fill copies that cell (in the fixed
// order of for_ghost_images) and adds them. Only the frame of kFrame cells at
// each edge can receive (four cells, and the face past them): e numbers its
// cells, the full rows first.
constexpr int kFrame = 5;
__host__ __device__ inline int frame_cells(int nx1, int nx2) {
  const int w = nx1 + 1, h = nx2 + 1;  // with the faces ie+1, je+1
  const int hr = h < 2 * kFrame ? h : 2 * kFrame, wc = w < 2 * kFrame ? w : 2 * kFrame;
  return hr * w + (h - hr) * wc;
}
__global__ void __launch_bounds__(kCells) ak_fold(AdjArgs a) {
  const Inst& g = a.g;
  const int w = g.nx1 + 1, h = g.nx2 + 1;
  const int hr = min(h, 2 * kFrame), wc = min(w, 2 * kFrame);
  const int e = (int)blockIdx.x * kCells + (int)threadIdx.x;
  if (e >= frame_cells(g.nx1, g.nx2)) return;
  int r, c;
  if (e < hr * w) {
    r = e / w;
    c = e - r * w;
    if (r >= kFrame && h > hr) r += h - hr;
  } else {
    const int f = e - hr * w;
    r = f / wc;
    c = f - r * wc;
    r += kFrame;
    if (c >= kFrame && w > wc) c += w - wc;
  }
  const int j = g.js + r, i = g.is + c;
  double* A = a.aout;
  const size_t ps = g.ps;
  const int pitch = g.pitch;
  const bool cell_i = i <= g.ie, cell_j = j <= g.je;
  const unsigned ix = cell_i ? ghost_images(i, g.is, g.ie, g.bc[0], g.bc[1], false) : 0u;
  const unsigned iy = cell_j ? ghost_images(j, g.js, g.je, g.bc[2], g.bc[3], false) : 0u;
  const unsigned fx = ghost_images(i, g.is, g.ie, g.bc[0], g.bc[1], true);
  const unsigned fy = ghost_images(j, g.js, g.je, g.bc[2], g.bc[3], true);
  // all fields of a class together: their loads are in flight at the same time
  const uint32_t k = (uint32_t)(j * pitch + i);
  double v[NSTATE];
#pragma unroll
  for (int f = 0; f < NSTATE; f++) v[f] = A[f * ps + k];
  auto add = [&](int cls, unsigned mx, unsigned my) {
    for_ghost_images(g, j, i, mx, my, [&](int rr, int cc, bool nx, bool ny) {
      const uint32_t kg = (uint32_t)(rr * pitch + cc);
#pragma unroll
      for (int f = 0; f < NSTATE; f++) {
        if (ghost_class(f) != cls) continue;
        const double x = A[f * ps + kg];
        v[f] += ghost_negates(f, nx, ny) ? -x : x;
      }
    });
#pragma unroll
    for (int f = 0; f < NSTATE; f++)
      if (ghost_class(f) == cls) A[f * ps + k] = v[f];
  };
  if (cell_i && cell_j && (ix | iy)) add(0, ix, iy);
  if (cell_j && (fx | iy)) add(1, fx, iy);
  if (cell_i && (ix | fy)) add(2, ix, fy);
}
__global__ void __launch_bounds__(kCells) ak_clear_ghost(AdjArgs a) {
  const Inst& g = a.g;
  int j, i;
  if (!range_ij(blockIdx.x, kCells, 0, g.sy - 1, 0, g.sx - 1, j, i)) return;
  const uint32_t k = (uint32_t)(j * g.pitch + i);
  const bool gx = i < g.is || i > g.ie, gy = j < g.js || j > g.je;
  if (!gx && !gy) return;
  for (int f = 0; f < NSTATE; f++) {
    // the face at ie+1 of B1i (je+1 of B2i) is not a ghost
    const bool ghost = f == F_B1I   ? (gy || i < g.is || i > g.ie + 1)
                       : f == F_B2I ? (gx || j < g.js || j > g.je + 1)
                                    : true;
    if (ghost) a.aout[f * g.ps + k] = 0.0;
  }
}

// every adjoint plane and ain (start of a reverse pass)
__global__ void __launch_bounds__(256) ak_clear(AdjArgs a) {
  const size_t n_in = (size_t)NSTATE * a.g.ps, n_ab = (size_t)NADJ * a.g.ps;
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n_in + n_ab;
       e += (size_t)gridDim.x * blockDim.x) {
    if (e < n_in) a.ain[e] = 0.0;
    else a.ab[e - n_in] = 0.0;
  }
}

// ---------------------------------------------------------------------------
// Steps 9, 11a, 11b, 13 (:473-534) over [js,je+1] x [is,ie+1]; the corrector
// flux adjoints are stored over [js-1,je+1] x [is-1,ie+1], the faces the
// corrector Riemann reverse reads (zero where no update reads the flux). The
// update's identity part starts ain, over the whole padded grid.
__global__ void __launch_bounds__(kCells) ak_update(AdjArgs a) {
  const Inst& g = a.g;
  int j, i;
  if (!range_ij(blockIdx.x, kCells, 0, g.sy - 1, 0, g.sx - 1, j, i)) return;
  const size_t ps = g.ps;
  const int pitch = g.pitch;
  const double dtodx1 = a.dt / g.dx1, dtodx2 = a.dt / g.dx2;
  const uint32_t k = (uint32_t)(j * pitch + i);
  const double* ao = a.aout;
  // adjoint of the updated value of cell field q at (jj, ii); 0 off the interior.
  // B3i = B3c after the update (Step 13), so B3c carries both adjoints.
  auto cb = [&](int q, int jj, int ii) -> double {
    if (jj < g.js || jj > g.je || ii < g.is || ii > g.ie) return 0.0;
    const uint32_t kk = (uint32_t)(jj * pitch + ii);
    double v = ao[q * ps + kk];
    if (q == F_B3C) v += ao[F_B3I * ps + kk];
    return v;
  };
  const int q_id[6] = {F_D, F_M1, F_M2, F_M3, F_E, F_B3C};
  for (int n = 0; n < 6; n++) a.ain[q_id[n] * ps + k] = cb(q_id[n], j, i);
  a.ain[F_B1C * ps + k] = 0.0;
  a.ain[F_B2C * ps + k] = 0.0;
  a.ain[F_B3I * ps + k] = 0.0;
  if (j < g.js - 1 || j > g.je + 1 || i < g.is - 1 || i > g.ie + 1) {
    a.ain[F_B1I * ps + k] = 0.0;
    a.ain[F_B2I * ps + k] = 0.0;
    return;
  }
  // corrector fluxes; the B2c update of 11a and the B1c update of 11b are
  // overwritten by Step 13, so those components get no adjoint there
  if (i >= g.is) {
    const int q1[7] = {F_D, F_M1, F_M2, F_M3, F_E, -1, F_B3C};
    double* F = a.ab + A_F1C * ps;
    for (int n = 0; n < 7; n++)
      F[n * ps + k] = (q1[n] < 0) ? 0.0 : dtodx1 * (cb(q1[n], j, i) - cb(q1[n], j, i - 1));
  }
  if (j >= g.js) {
    const int q2[7] = {F_D, F_M2, F_M3, F_M1, F_E, F_B3C, -1};
    double* F = a.ab + A_F2C * ps;
    for (int n = 0; n < 7; n++)
      F[n * ps + k] = (q2[n] < 0) ? 0.0 : dtodx2 * (cb(q2[n], j, i) - cb(q2[n], j - 1, i));
  }
  // adjoint of the updated face fields including B1c, B2c = face averages
  auto b1t = [&](int jj, int ii) -> double {
    if (jj < g.js || jj > g.je || ii < g.is || ii > g.ie + 1) return 0.0;
    return ao[F_B1I * ps + (uint32_t)(jj * pitch + ii)] +
           0.5 * (cb(F_B1C, jj, ii) + cb(F_B1C, jj, ii - 1));
  };
  auto b2t = [&](int jj, int ii) -> double {
    if (jj < g.js || jj > g.je + 1 || ii < g.is || ii > g.ie) return 0.0;
    return ao[F_B2I * ps + (uint32_t)(jj * pitch + ii)] +
           0.5 * (cb(F_B2C, jj, ii) + cb(F_B2C, jj - 1, ii));
  };
  a.ain[F_B1I * ps + k] = b1t(j, i);
  a.ain[F_B2I * ps + k] = b2t(j, i);
  if (j < g.js || i < g.is) return;
  a.ab[A_EMFC * ps + k] =
      dtodx2 * (b1t(j, i) - b1t(j - 1, i)) + dtodx1 * (b2t(j, i - 1) - b2t(j, i));
}

// ---------------------------------------------------------------------------
// integrate_emf3_corner (:632-702) reversed, from its inputs' side. Corner K is
// a quarter of four upwinded estimates, picked by the face mass fluxes
//   w1 = F1[K-pitch], w2 = F1[K], w3 = F2[K-1], w4 = F2[K]  (1, 0, or 1/2 at 0);
// each input takes the corners it enters with their weights. The adjoint of a
// corner outside the range of the reversed step is zero, so no input needs a
// range test (a weight is 0, 1/2 or 1 whatever the flux there holds).
__device__ __forceinline__ double upwind_weight(double mass_flux) {
  return (mass_flux > 0.0) ? 1.0 : ((mass_flux < 0.0) ? 0.0 : 0.5);
}
struct CornerGather {
  const double *F1, *F2;  // mass fluxes
  const double* eb;       // adjoint of the corner emf
  uint32_t p;             // pitch
  __device__ double q(uint32_t K) const { return 0.25 * eb[K]; }
  // By of the x1 flux at k: corners k and k + pitch
  __device__ double f1_by(uint32_t k) const {
    const double w3 = upwind_weight(F2[k - 1]), w4 = upwind_weight(F2[k]);
    const double u3 = upwind_weight(F2[k + p - 1]), u4 = upwind_weight(F2[k + p]);
    return q(k) * (-1.0 - (1.0 - w3) - (1.0 - w4)) + q(k + p) * (-1.0 - u3 - u4);
  }
  // Bz of the x2 flux at k: corners k and k + 1
  __device__ double f2_bz(uint32_t k) const {
    const double w1 = upwind_weight(F1[k - p]), w2 = upwind_weight(F1[k]);
    const double u1 = upwind_weight(F1[k + 1 - p]), u2 = upwind_weight(F1[k + 1]);
    return q(k) * ((1.0 - w1) + (1.0 - w2) + 1.0) + q(k + 1) * (u1 + u2 + 1.0);
  }
  // the cell-centred emf at k: its four corners
  __device__ double emf_cc(uint32_t k) const {
    const double q00 = q(k), q01 = q(k + 1), q10 = q(k + p), q11 = q(k + p + 1);
    if (q00 == 0.0 && q01 == 0.0 && q10 == 0.0 && q11 == 0.0) return 0.0;
    const double f1 = upwind_weight(F1[k]), f1i = upwind_weight(F1[k + 1]);
    const double f2 = upwind_weight(F2[k]), f2j = upwind_weight(F2[k + p]);
    return q00 * (-(1.0 - f1) - (1.0 - f2)) + q01 * (-f1i - (1.0 - f2)) +
           q10 * (-(1.0 - f1) - f2j) + q11 * (-f1i - f2j);
  }
};

// ---------------------------------------------------------------------------
// Forward values shared by the corrector stages: half-step face fields
// (:266-275) and the corrected face states (Steps 5, 6), in the exact forward
// order.
struct CorrCtx {
  const Inst& g;
  const double* st;
  const double* sc;
  const double* emf;  // predictor corner emf
  size_t ps;
  int pitch;
  double hdtodx1, hdtodx2;
  __device__ double b1h(uint32_t kk) const {
    return st[F_B1I * ps + kk] - hdtodx2 * (emf[kk + pitch] - emf[kk]);
  }
  __device__ double b2h(uint32_t kk) const {
    return st[F_B2I * ps + kk] + hdtodx1 * (emf[kk + 1] - emf[kk]);
  }
  __device__ double s(int f, uint32_t kk) const { return st[f * ps + kk]; }
  // x1 face k: Step 5a with x2 fluxes at (j+1,i-1),(j,i-1) / (j+1,i),(j,i) and 5b
  __device__ void states_x1(uint32_t k, Cons7& L, Cons7& R) const {
    const double* F2 = sc + S_F2 * ps;
    L = ld7(sc + S_UL1 * ps, ps, k);
    R = ld7(sc + S_UR1 * ps, ps, k);
    const uint32_t a1 = k + pitch - 1, a0 = k - 1, c1 = k + pitch, c0 = k;
    L.d = L.d - hdtodx2 * (F2[a1] - F2[a0]);
    L.mx = L.mx - hdtodx2 * (F2[3 * ps + a1] - F2[3 * ps + a0]);
    L.my = L.my - hdtodx2 * (F2[1 * ps + a1] - F2[1 * ps + a0]);
    L.mz = L.mz - hdtodx2 * (F2[2 * ps + a1] - F2[2 * ps + a0]);
    L.e = L.e - hdtodx2 * (F2[4 * ps + a1] - F2[4 * ps + a0]);
    L.bz = L.bz - hdtodx2 * (F2[5 * ps + a1] - F2[5 * ps + a0]);
    R.d = R.d - hdtodx2 * (F2[c1] - F2[c0]);
    R.mx = R.mx - hdtodx2 * (F2[3 * ps + c1] - F2[3 * ps + c0]);
    R.my = R.my - hdtodx2 * (F2[1 * ps + c1] - F2[1 * ps + c0]);
    R.mz = R.mz - hdtodx2 * (F2[2 * ps + c1] - F2[2 * ps + c0]);
    R.e = R.e - hdtodx2 * (F2[4 * ps + c1] - F2[4 * ps + c0]);
    R.bz = R.bz - hdtodx2 * (F2[5 * ps + c1] - F2[5 * ps + c0]);
    const double hdtodx1_ = hdtodx1;
    double dbx = s(F_B1I, k) - s(F_B1I, k - 1);
    double b1 = s(F_B1C, k - 1), b2 = s(F_B2C, k - 1), b3 = s(F_B3C, k - 1);
    double v3 = s(F_M3, k - 1) / s(F_D, k - 1);
    L.mx = L.mx + hdtodx1_ * b1 * dbx;
    L.my = L.my + hdtodx1_ * b2 * dbx;
    L.mz = L.mz + hdtodx1_ * b3 * dbx;
    L.bz = L.bz + hdtodx1_ * v3 * dbx;
    L.e = L.e + hdtodx1_ * b3 * v3 * dbx;
    dbx = s(F_B1I, k + 1) - s(F_B1I, k);
    b1 = s(F_B1C, k); b2 = s(F_B2C, k); b3 = s(F_B3C, k);
    v3 = s(F_M3, k) / s(F_D, k);
    R.mx = R.mx + hdtodx1_ * b1 * dbx;
    R.my = R.my + hdtodx1_ * b2 * dbx;
    R.mz = R.mz + hdtodx1_ * b3 * dbx;
    R.bz = R.bz + hdtodx1_ * v3 * dbx;
    R.e = R.e + hdtodx1_ * b3 * v3 * dbx;
  }
  // x2 face k: Step 6a with x1 fluxes at (j-1,i+1),(j-1,i) / (j,i+1),(j,i) and 6b
  __device__ void states_x2(uint32_t k, Cons7& L, Cons7& R) const {
    const double* F1 = sc + S_F1 * ps;
    L = ld7(sc + S_UL2 * ps, ps, k);
    R = ld7(sc + S_UR2 * ps, ps, k);
    const uint32_t a1 = k - pitch + 1, a0 = k - pitch, c1 = k + 1, c0 = k;
    L.d = L.d - hdtodx1 * (F1[a1] - F1[a0]);
    L.mx = L.mx - hdtodx1 * (F1[2 * ps + a1] - F1[2 * ps + a0]);
    L.my = L.my - hdtodx1 * (F1[3 * ps + a1] - F1[3 * ps + a0]);
    L.mz = L.mz - hdtodx1 * (F1[1 * ps + a1] - F1[1 * ps + a0]);
    L.e = L.e - hdtodx1 * (F1[4 * ps + a1] - F1[4 * ps + a0]);
    L.by = L.by - hdtodx1 * (F1[6 * ps + a1] - F1[6 * ps + a0]);
    R.d = R.d - hdtodx1 * (F1[c1] - F1[c0]);
    R.mx = R.mx - hdtodx1 * (F1[2 * ps + c1] - F1[2 * ps + c0]);
    R.my = R.my - hdtodx1 * (F1[3 * ps + c1] - F1[3 * ps + c0]);
    R.mz = R.mz - hdtodx1 * (F1[1 * ps + c1] - F1[1 * ps + c0]);
    R.e = R.e - hdtodx1 * (F1[4 * ps + c1] - F1[4 * ps + c0]);
    R.by = R.by - hdtodx1 * (F1[6 * ps + c1] - F1[6 * ps + c0]);
    const uint32_t km = k - pitch;
    double dby = s(F_B2I, k) - s(F_B2I, km);
    double b1 = s(F_B1C, km), b2 = s(F_B2C, km), b3 = s(F_B3C, km);
    double v3 = s(F_M3, km) / s(F_D, km);
    L.mz = L.mz + hdtodx2 * b1 * dby;
    L.mx = L.mx + hdtodx2 * b2 * dby;
    L.my = L.my + hdtodx2 * b3 * dby;
    L.by = L.by + hdtodx2 * v3 * dby;
    L.e = L.e + hdtodx2 * b3 * v3 * dby;
    dby = s(F_B2I, k + pitch) - s(F_B2I, k);
    b1 = s(F_B1C, k); b2 = s(F_B2C, k); b3 = s(F_B3C, k);
    v3 = s(F_M3, k) / s(F_D, k);
    R.mz = R.mz + hdtodx2 * b1 * dby;
    R.mx = R.mx + hdtodx2 * b2 * dby;
    R.my = R.my + hdtodx2 * b3 * dby;
    R.by = R.by + hdtodx2 * v3 * dby;
    R.e = R.e + hdtodx2 * b3 * v3 * dby;
  }
};

__device__ __forceinline__ CorrCtx corr_ctx(const AdjArgs& a) {
  const double dtodx1 = a.dt / a.g.dx1, dtodx2 = a.dt / a.g.dx2;
  return CorrCtx{a.g, a.st, a.sc, a.emfp, a.g.ps, a.g.pitch, 0.5 * dtodx1, 0.5 * dtodx2};
}

// the corners of Step 9 (corrector fluxes) and of Step 4 (predictor fluxes)
__device__ __forceinline__ CornerGather corner_c(const AdjArgs& a) {
  const size_t ps = a.g.ps;
  return CornerGather{a.sc + S_F1C * ps, a.sc + S_F2C * ps, a.ab + A_EMFC * ps,
                      (uint32_t)a.g.pitch};
}
__device__ __forceinline__ CornerGather corner_p(const AdjArgs& a) {
  const size_t ps = a.g.ps;
  return CornerGather{a.sc + S_F1 * ps, a.sc + S_F2 * ps, a.ab + A_EMFP * ps,
                      (uint32_t)a.g.pitch};
}

// Step 8b (X1: x1 faces [js-1,je+1] x [is,ie+1], :438-447) or 8c (x2 faces
// [js,je+1] x [is-1,ie+1], :455-464); the two are independent
template <bool X1, int FLUX>  // FLUX: the grid's Riemann solver
__device__ __forceinline__ void riemann_c(const AdjArgs& a, int block) {
  const Inst& g = a.g;
  int j, i;
  if (X1) {
    if (!range_ij(block, kWave, g.js - 1, g.je + 1, g.is, g.ie + 1, j, i)) return;
  } else {
    if (!range_ij(block, kWave, g.js, g.je + 1, g.is - 1, g.ie + 1, j, i)) return;
  }
  const CorrCtx c = corr_ctx(a);
  const CornerGather corner = corner_c(a);
  const size_t ps = g.ps;
  const uint32_t k = (uint32_t)(j * g.pitch + i);
  const EosC eos{g.gamma, g.g1, g.g2};
  if (X1) {
    Cons7 L, R;
    c.states_x1(k, L, R);
    const double bx = c.b1h(k);
    const Prim7 wl = cons_to_prim(L, bx, eos), wr = cons_to_prim(R, bx, eos);
    Cons7 Lb = zero_cons(), Rb = zero_cons();
    Prim7 Wlb = zero_prim(), Wrb = zero_prim();
    double bxb = 0.0;
    Cons7 Fb = ld7(a.ab + A_F1C * ps, ps, k);
    Fb.by += corner.f1_by(k);
    riemann_b_of<FLUX>(L, R, wl, wr, bx, eos, Fb, Lb, Rb, Wlb, Wrb, bxb);
    cons_to_prim_b(L, bx, eos, Wlb, Lb, bxb);
    cons_to_prim_b(R, bx, eos, Wrb, Rb, bxb);
    st7(a.ab + A_UL1 * ps, ps, k, Lb);
    st7(a.ab + A_UR1 * ps, ps, k, Rb);
    a.ab[A_B1H * ps + k] = bxb;
  } else {
    Cons7 L, R;
    c.states_x2(k, L, R);
    const double bx = c.b2h(k);
    const Prim7 wl = cons_to_prim(L, bx, eos), wr = cons_to_prim(R, bx, eos);
    Cons7 Lb = zero_cons(), Rb = zero_cons();
    Prim7 Wlb = zero_prim(), Wrb = zero_prim();
    double bxb = 0.0;
    Cons7 Fb = ld7(a.ab + A_F2C * ps, ps, k);
    Fb.bz += corner.f2_bz(k);
    riemann_b_of<FLUX>(L, R, wl, wr, bx, eos, Fb, Lb, Rb, Wlb, Wrb, bxb);
    cons_to_prim_b(L, bx, eos, Wlb, Lb, bxb);
    cons_to_prim_b(R, bx, eos, Wrb, Rb, bxb);
    st7(a.ab + A_UL2 * ps, ps, k, Lb);
    st7(a.ab + A_UR2 * ps, ps, k, Rb);
    a.ab[A_B2H * ps + k] = bxb;
  }
}

// Step 7 (:402-431) reversed per cell of [js-1,je+1] x [is-1,ie+1]: stores
// the adjoints of the cell's half-step d, M1, M2 and B1c, B2c; the transverse
// reverse hands them on to the predictor fluxes and the half-step face fields.
__device__ __forceinline__ void half_step(const AdjArgs& a, int block) {
  const Inst& g = a.g;
  int j, i;
  if (!range_ij(block, kWave, g.js - 1, g.je + 1, g.is - 1, g.ie + 1, j, i)) return;
  const size_t ps = g.ps;
  const int pitch = g.pitch;
  const uint32_t k = (uint32_t)(j * pitch + i);
  const double Eb = corner_c(a).emf_cc(k);
  double dhb = 0.0, m1b = 0.0, m2b = 0.0, b1cb = 0.0, b2cb = 0.0;
  if (Eb != 0.0) {
    const CorrCtx c = corr_ctx(a);
    const double h1 = c.hdtodx1, h2 = c.hdtodx2;
    const double* F1 = a.sc + S_F1 * ps;
    const double* F2 = a.sc + S_F2 * ps;
    const double dhalf = c.s(F_D, k) - h1 * (F1[k + 1] - F1[k]) - h2 * (F2[k + pitch] - F2[k]);
    const double m1 = c.s(F_M1, k) - h1 * (F1[ps + k + 1] - F1[ps + k]) -
                      h2 * (F2[3 * ps + k + pitch] - F2[3 * ps + k]);
    const double m2 = c.s(F_M2, k) - h1 * (F1[2 * ps + k + 1] - F1[2 * ps + k]) -
                      h2 * (F2[ps + k + pitch] - F2[ps + k]);
    const double b1c = 0.5 * (c.b1h(k) + c.b1h(k + 1));
    const double b2c = 0.5 * (c.b2h(k) + c.b2h(k + pitch));
    const double emf = (b1c * m2 - b2c * m1) / dhalf;
    b1cb = adiv(Eb * m2, dhalf);
    m2b = adiv(Eb * b1c, dhalf);
    b2cb = -adiv(Eb * m1, dhalf);
    m1b = -adiv(Eb * b2c, dhalf);
    dhb = -adiv(Eb * emf, dhalf);
    a.ain[F_D * ps + k] += dhb;
    a.ain[F_M1 * ps + k] += m1b;
    a.ain[F_M2 * ps + k] += m2b;
  }
  double* ab = a.ab;
  ab[A_HD * ps + k] = dhb;
  ab[A_HM1 * ps + k] = m1b;
  ab[A_HM2 * ps + k] = m2b;
  ab[A_HB1 * ps + k] = b1cb;
  ab[A_HB2 * ps + k] = b2cb;
}

// Steps 8b, 8c and 7 in one launch: blocks [0, n1) the x1 faces, [n1, n1 + n2)
// the x2 faces, the rest Step 7 (they write disjoint planes). The Roe reverse
// holds 512 registers (one wave per SIMD), the HLLE one fits two.
template <int FLUX>
__global__ void __launch_bounds__(kWave, FLUX == kFluxHlle ? 2 : 1) ak_correct(AdjArgs a, int n1,
                                                                              int n2) {
  const int b = blockIdx.x;
  if (b < n1) riemann_c<true, FLUX>(a, b);
  else if (b < n1 + n2) riemann_c<false, FLUX>(a, b - n1);
  else half_step(a, b - n1 - n2);
}

// Steps 5, 6 (:284-393), the half-step face fields of Step 4 (:263-275) and
// the flux part of Step 7, reversed as a gather: each thread owns one cell /
// face / corner position c of [js-2,je+2] x [is-2,ie+2] and stores the
// adjoints of the predictor fluxes and the predictor corner emf there, and
// adds the state adjoints of c. Every adjoint read is zero outside the range
// its writer covers, so no position needs a range test.
//
// The x1-face states at faces c+1 (left) and c (right) both take their 1/2 dt
// source terms from cell c and the face-field difference B1i[c+1] - B1i[c]
// (:296-330), and both are corrected with the x2 fluxes at c and c+pitch
// (left at c+1: at c+1-1): with X1(c) = Lb(c+1) + Rb(c) the sources' adjoint
// is linear in X1(c), and the x2 flux at c receives h2 (X1(c) - X1(c-pitch)).
// Likewise for x2 faces with X2(c) = Lb(c+pitch) + Rb(c).
//
// Tiles of 64 x 4: each position reads its row's and the rows' below values of
// some 40 planes, which a tile's rows share (in the row-after-row order of the
// other stages 47 -> 59 us at 512^2).
__global__ void __launch_bounds__(kTileX* kTileY) ak_transverse(AdjArgs a) {
  const Inst& g = a.g;
  const int i = g.is - 2 + (int)blockIdx.x * kTileX + (int)threadIdx.x;
  const int j = g.js - 2 + (int)blockIdx.y * kTileY + (int)threadIdx.y;
  if (i > g.ie + 2 || j > g.je + 2) return;
  const size_t ps = g.ps;
  const uint32_t pitch = (uint32_t)g.pitch;
  const uint32_t c = (uint32_t)j * pitch + (uint32_t)i;
  const double h1 = 0.5 * a.dt / g.dx1, h2 = 0.5 * a.dt / g.dx2;
  const double* st = a.st;
  const double* ab = a.ab;
  double* ain = a.ain;
  // X1 and X2 components in Cons7 order (d, mx, my, mz, e, by, bz)
  auto X1 = [&](uint32_t kk, int n) {
    return ab[(A_UL1 + n) * ps + kk + 1] + ab[(A_UR1 + n) * ps + kk];
  };
  auto X2 = [&](uint32_t kk, int n) {
    return ab[(A_UL2 + n) * ps + kk + pitch] + ab[(A_UR2 + n) * ps + kk];
  };
  // h_dir * (the source terms' adjoint on the face field), per cell
  //   X.(b1, b2, b3, bt) components: x1 states (mx, my, mz, bz); x2 states
  //   (d, M2, M3, M1, E, B3, B1) -> (mz, mx, my, by)
  auto dbb = [&](uint32_t kk, double h, double xb1, double xb2, double xb3, double xbt,
                 double xe) {
    const double b1 = st[F_B1C * ps + kk], b2 = st[F_B2C * ps + kk], b3 = st[F_B3C * ps + kk];
    const double v3 = st[F_M3 * ps + kk] / st[F_D * ps + kk];
    return h * (xb1 * b1 + xb2 * b2 + xb3 * b3 + xbt * v3 + xe * b3 * v3);
  };
  auto dbb1 = [&](uint32_t kk) {
    return dbb(kk, h1, X1(kk, 1), X1(kk, 2), X1(kk, 3), X1(kk, 6), X1(kk, 4));
  };
  auto dbb2 = [&](uint32_t kk) {
    return dbb(kk, h2, X2(kk, 3), X2(kk, 1), X2(kk, 2), X2(kk, 5), X2(kk, 4));
  };
  // half-step face fields: Riemann part + Step 7's face averages
  auto hb1 = [&](uint32_t kk) {
    return ab[A_B1H * ps + kk] + 0.5 * (ab[A_HB1 * ps + kk] + ab[A_HB1 * ps + kk - 1]);
  };
  auto hb2 = [&](uint32_t kk) {
    return ab[A_B2H * ps + kk] + 0.5 * (ab[A_HB2 * ps + kk] + ab[A_HB2 * ps + kk - pitch]);
  };
  const double* HD = ab + A_HD * ps;
  const double* HM1 = ab + A_HM1 * ps;
  const double* HM2 = ab + A_HM2 * ps;
  // x2 predictor fluxes (d, M2, M3, M1, E, B3, B1): x1 states (d, mx, my, mz, e, bz) were
  // corrected with components (0, 3, 1, 2, 4, 5); Step 7 used d, M1, M2 = (0, 3, 1)
  {
    double* F2b = a.ab + A_F2 * ps;
    const int src[7] = {0, 2, 3, 1, 4, 6, -1};  // x1-state component feeding F2 component
    for (int n = 0; n < 7; n++) {
      double v = (src[n] < 0) ? 0.0 : h2 * (X1(c, src[n]) - X1(c - pitch, src[n]));
      if (n == 0) v += h2 * (HD[c] - HD[c - pitch]);
      if (n == 3) v += h2 * (HM1[c] - HM1[c - pitch]);
      if (n == 1) v += h2 * (HM2[c] - HM2[c - pitch]);
      F2b[n * ps + c] = v;
    }
  }
  // x1 predictor fluxes (d, M1, M2, M3, E, B2, B3): x2 states (d, mx, my, mz, e, by) were
  // corrected with components (0, 2, 3, 1, 4, 6); Step 7 used d, M1, M2 = (0, 1, 2)
  {
    double* F1b = a.ab + A_F1 * ps;
    const int src[7] = {0, 3, 1, 2, 4, -1, 5};  // x2-state component feeding F1 component
    for (int n = 0; n < 7; n++) {
      double v = (src[n] < 0) ? 0.0 : h1 * (X2(c, src[n]) - X2(c - 1, src[n]));
      if (n == 0) v += h1 * (HD[c] - HD[c - 1]);
      if (n == 1) v += h1 * (HM1[c] - HM1[c - 1]);
      if (n == 2) v += h1 * (HM2[c] - HM2[c - 1]);
      F1b[n * ps + c] = v;
    }
  }
  // predictor corner emf from the half-step face fields (:266-275)
  a.ab[A_EMFP * ps + c] = h2 * (hb1(c) - hb1(c - pitch)) + h1 * (hb2(c - 1) - hb2(c));
  // face fields: half-step fields and the source terms' face-field differences
  ain[F_B1I * ps + c] += hb1(c) + dbb1(c - 1) - dbb1(c);
  ain[F_B2I * ps + c] += hb2(c) + dbb2(c - pitch) - dbb2(c);
  // the source terms' cell-centred B and v3 = M3 / d of cell c
  {
    const double b3 = st[F_B3C * ps + c];
    const double d = st[F_D * ps + c], v3 = st[F_M3 * ps + c] / d;
    const double db1 = h1 * (st[F_B1I * ps + c + 1] - st[F_B1I * ps + c]);
    const double db2 = h2 * (st[F_B2I * ps + c + pitch] - st[F_B2I * ps + c]);
    const double x1e = X1(c, 4), x2e = X2(c, 4);
    ain[F_B1C * ps + c] += db1 * X1(c, 1) + db2 * X2(c, 3);
    ain[F_B2C * ps + c] += db1 * X1(c, 2) + db2 * X2(c, 1);
    ain[F_B3C * ps + c] += db1 * (X1(c, 3) + x1e * v3) + db2 * (X2(c, 2) + x2e * v3);
    const double v3b = db1 * (X1(c, 6) + x1e * b3) + db2 * (X2(c, 5) + x2e * b3);
    ain[F_M3 * ps + c] += adiv(v3b, d);
    ain[F_D * ps + c] += -adiv(v3b * v3, d);
  }
}

// Step 3 (:249-255) over [js-2,je+2] x [is-2,ie+2]
__device__ __forceinline__ void emf_cc(const AdjArgs& a, int block) {
  const Inst& g = a.g;
  int j, i;
  if (!range_ij(block, kWave, g.js - 2, g.je + 2, g.is - 2, g.ie + 2, j, i)) return;
  const size_t ps = g.ps;
  const uint32_t k = (uint32_t)(j * g.pitch + i);
  const double Eb = corner_p(a).emf_cc(k);
  if (Eb == 0.0) return;
  const double* st = a.st;
  const double d = st[F_D * ps + k], m1 = st[F_M1 * ps + k], m2 = st[F_M2 * ps + k];
  const double b1 = st[F_B1C * ps + k], b2 = st[F_B2C * ps + k];
  const double e = (b1 * m2 - b2 * m1) / d;
  ADD(a.ain + F_B1C * ps, k, adiv(Eb * m2, d));
  ADD(a.ain + F_M2 * ps, k, adiv(Eb * b1, d));
  ADD(a.ain + F_B2C * ps, k, -adiv(Eb * m1, d));
  ADD(a.ain + F_M1 * ps, k, -adiv(Eb * b2, d));
  ADD(a.ain + F_D * ps, k, -adiv(Eb * e, d));
}

// ---------------------------------------------------------------------------
// Steps 1c-1e / 2c-2e (:156-180, :216-241) reversed per predictor face: the
// Riemann flux, prim->cons and the 1/2 dt MHD source on the transverse field
// (By for x1 faces, Bz for x2 faces), from the face states the forward pass
// stored. X1: faces [js-2,je+2] x [is-1,ie+2]; x2: [js-1,je+2] x [is-2,ie+2].
// Writes the adjoints of the PLM outputs Wl, Wr (the source only adds to them).
template <bool X1, int FLUX>  // FLUX: the grid's Riemann solver
__device__ __forceinline__ void predict(const AdjArgs& a, int block) {
  const Inst& g = a.g;
  int j, i;
  if (X1) {
    if (!range_ij(block, kWave, g.js - 2, g.je + 2, g.is - 1, g.ie + 2, j, i)) return;
  } else {
    if (!range_ij(block, kWave, g.js - 1, g.je + 2, g.is - 2, g.ie + 2, j, i)) return;
  }
  const size_t ps = g.ps;
  const uint32_t stride = X1 ? 1u : (uint32_t)g.pitch;
  const uint32_t k = (uint32_t)(j * g.pitch + i);
  const EosC eos{g.gamma, g.g1, g.g2};
  const double* st = a.st;
  const int bplane = X1 ? F_B1I : F_B2I;  // normal face field
  const int mplane = X1 ? F_M2 : F_M1;    // momentum of the source's velocity
  const double b0 = st[bplane * ps + k];
  Cons7 Ulb = ld7(a.ab + (X1 ? A_UL1 : A_UL2) * ps, ps, k);
  Cons7 Urb = ld7(a.ab + (X1 ? A_UR1 : A_UR2) * ps, ps, k);
  Prim7 wlb = zero_prim(), wrb = zero_prim();
  double b0b = 0.0;
  {
    const Prim7 wl = ld7p(a.pw + (X1 ? P_WL1 : P_WL2) * ps, ps, k);
    const Prim7 wr = ld7p(a.pw + (X1 ? P_WR1 : P_WR2) * ps, ps, k);
    Cons7 Fb = ld7(a.ab + (X1 ? A_F1 : A_F2) * ps, ps, k);
    if (X1) Fb.by += corner_p(a).f1_by(k);
    else Fb.bz += corner_p(a).f2_bz(k);
    riemann_b_of<FLUX>(ld7(a.sc + (X1 ? S_UL1 : S_UL2) * ps, ps, k),
                       ld7(a.sc + (X1 ? S_UR1 : S_UR2) * ps, ps, k), wl, wr, b0, eos, Fb, Ulb,
                       Urb, wlb, wrb, b0b);
    prim_to_cons_b(wl, b0, eos, Ulb, wlb, b0b);
    prim_to_cons_b(wr, b0, eos, Urb, wrb, b0b);
  }
  // source: W.bt += 1/2 dt (M/d)[cell] (B[face+1] - B[face]) / dx, left state
  // from the cell behind the face, right state from the cell ahead
  const double dx = X1 ? g.dx1 : g.dx2;
  const double hdt = 0.5 * a.dt;
  const double bm = st[bplane * ps + k - stride], bp = st[bplane * ps + k + stride];
  const double dl = st[F_D * ps + k - stride], dr = st[F_D * ps + k];
  const double vl = st[mplane * ps + k - stride] / dl, vr = st[mplane * ps + k] / dr;
  const double slb = hdt * (X1 ? wlb.by : wlb.bz), srb = hdt * (X1 ? wrb.by : wrb.bz);
  const double dblb = adiv(slb * vl, dx), vlb = adiv(slb * (b0 - bm), dx);
  const double dbrb = adiv(srb * vr, dx), vrb = adiv(srb * (bp - b0), dx);
  if (a.det) {
    // stored per face; ak_plm_gather adds them to the cells in a fixed order
    double* pc = a.ab + (X1 ? A_PC1 : A_PC2) * ps;
    pc[k] = -dblb;
    pc[ps + k] = b0b + dblb - dbrb;
    pc[2 * ps + k] = dbrb;
    pc[3 * ps + k] = adiv(vlb, dl);
    pc[4 * ps + k] = -adiv(vlb * vl, dl);
    pc[5 * ps + k] = adiv(vrb, dr);
    pc[6 * ps + k] = -adiv(vrb * vr, dr);
  } else {
    ADD(a.ain + bplane * ps, k - stride, -dblb);
    ADD(a.ain + bplane * ps, k, b0b + dblb - dbrb);
    ADD(a.ain + bplane * ps, k + stride, dbrb);
    ADD(a.ain + mplane * ps, k - stride, adiv(vlb, dl));
    ADD(a.ain + F_D * ps, k - stride, -adiv(vlb * vl, dl));
    ADD(a.ain + mplane * ps, k, adiv(vrb, dr));
    ADD(a.ain + F_D * ps, k, -adiv(vrb * vr, dr));
  }
  st7(a.ab + (X1 ? A_WL1 : A_WL2) * ps, ps, k, wlb);
  st7(a.ab + (X1 ? A_WR1 : A_WR2) * ps, ps, k, wrb);
}

// Both sweeps' predictor faces and Step 3 in one launch, as ak_correct (ain
// takes atomic adds from all of them; the deterministic reverse's faces store
// theirs, and Step 3 alone adds).
template <int FLUX>
__global__ void __launch_bounds__(kWave, 1) ak_predict(AdjArgs a, int n1, int n2) {
  const int b = blockIdx.x;
  if (b < n1) predict<true, FLUX>(a, b);
  else if (b < n1 + n2) predict<false, FLUX>(a, b - n1);
  else emf_cc(a, b - n1 - n2);
}

// Steps 1b / 2b reversed for one cell of [js-2,je+2] x [is-2,ie+2]: the PLM
// of cell k produced Wl at the next face and Wr at its own face. Stores the
// adjoints of the primitive states of cells k-1, k, k+1 and of Bxc[k] (22
// planes; zeros where the outputs' adjoints are zero); plm_gather hands them
// through cons->prim.
struct PlmSlot {
  PlmCore c;
  double pad;
};
static_assert((sizeof(PlmSlot) / 8) % 2 == 1, "odd slot stride in doubles");
template <bool X1>
__device__ __forceinline__ void plm(const AdjArgs& a, int block, PlmSlot* slot) {
  const Inst& g = a.g;
  int j, i;
  if (!range_ij(block, kWave, g.js - 2, g.je + 2, g.is - 2, g.ie + 2, j, i)) return;
  const size_t ps = g.ps;
  const uint32_t stride = X1 ? 1u : (uint32_t)g.pitch;
  const uint32_t k = (uint32_t)(j * g.pitch + i);
  double* dst = a.ab + (X1 ? A_PW1 : A_PW2) * ps;
  double olb[7], orb[7];
  bool any = false;
  {
    const Prim7 l = ld7p(a.ab + (X1 ? A_WL1 : A_WL2) * ps, ps, k + stride);
    const Prim7 r = ld7p(a.ab + (X1 ? A_WR1 : A_WR2) * ps, ps, k);
    for (int n = 0; n < 7; n++) {
      olb[n] = arr(l)[n];
      orb[n] = arr(r)[n];
      any = any || olb[n] != 0.0 || orb[n] != 0.0;
    }
  }
  if (!any) {
    for (int n = 0; n < 22; n++) dst[n * ps + k] = 0.0;
    return;
  }
  const EosC eos{g.gamma, g.g1, g.g2};
  const double* st = a.st;
  // cell state in the sweep's order and its normal field
  const int q[7] = {F_D, X1 ? F_M1 : F_M2, X1 ? F_M2 : F_M3, X1 ? F_M3 : F_M1, F_E,
                    X1 ? F_B2C : F_B3C, X1 ? F_B3C : F_B1C};
  const int qx = X1 ? F_B1C : F_B2C;
  auto cons_at = [&](uint32_t kk) {
    return Cons7{st[q[0] * ps + kk], st[q[1] * ps + kk], st[q[2] * ps + kk], st[q[3] * ps + kk],
                 st[q[4] * ps + kk], st[q[5] * ps + kk], st[q[6] * ps + kk]};
  };
  const uint32_t kc[3] = {k - stride, k, k + stride};
  Prim7 W[3];
  for (int c = 0; c < 3; c++) W[c] = cons_to_prim(cons_at(kc[c]), st[qx * ps + kc[c]], eos);
  // the stencil and eigensystem sit in LDS, one per thread, and each reverse
  // stage reads them again: the reverse then fits in registers without spills.
  // A slot is an odd number of doubles long, so that the 8-byte words one
  // field occupies in consecutive lanes' slots fall in distinct LDS banks
  // (68 doubles, an even stride, put lanes 4 or 8 to a bank)
  PlmCore& P = slot[threadIdx.x].c;
  P.prepare(W[0], W[1], W[2], st[qx * ps + k], a.dt / (X1 ? g.dx1 : g.dx2), eos);
  double wb[3][7];
  for (int c = 0; c < 3; c++)
    for (int n = 0; n < 7; n++) wb[c][n] = 0.0;
  double bxcb = 0.0;
  P.back(olb, orb, wb[0], wb[1], wb[2], bxcb);
  for (int c = 0; c < 3; c++)
    for (int n = 0; n < 7; n++) dst[(c * 7 + n) * ps + k] = wb[c][n];
  dst[21 * ps + k] = bxcb;
}

// both sweeps in one launch: blocks [0, n) x1, [n, 2 n) x2. Four one-wave
// workgroups of 40 KB of slots fill a CU's LDS.
__global__ void __launch_bounds__(kWave) ak_plm(AdjArgs a, int n) {
  __shared__ PlmSlot slot[kWave];
  const int b = blockIdx.x;
  if (b < n) plm<true>(a, b, slot);
  else plm<false>(a, b - n, slot);
}

// Steps 1a / 2a reversed per cell: the primitive-state adjoint of cell c sums
// the PLM reverses of cells c+1 (its left neighbour slot), c and c-1, and goes
// through cons->prim once. X1: cells [js-2,je+2] x [is-3,ie+3]; x2:
// [js-3,je+3] x [is-2,ie+2]. Atomic adds: the two sweeps run concurrently.
template <bool X1>
__device__ __forceinline__ void plm_gather(const AdjArgs& a, int block) {
  const Inst& g = a.g;
  int j, i;
  if (X1) {
    if (!range_ij(block, kCells, g.js - 2, g.je + 2, g.is - 3, g.ie + 3, j, i)) return;
  } else {
    if (!range_ij(block, kCells, g.js - 3, g.je + 3, g.is - 2, g.ie + 2, j, i)) return;
  }
  const size_t ps = g.ps;
  const uint32_t stride = X1 ? 1u : (uint32_t)g.pitch;
  const uint32_t k = (uint32_t)(j * g.pitch + i);
  const double* src = a.ab + (X1 ? A_PW1 : A_PW2) * ps;
  double wb[7];
  bool any = false;
  for (int n = 0; n < 7; n++) {
    wb[n] = src[n * ps + k + stride] + src[(7 + n) * ps + k] + src[(14 + n) * ps + k - stride];
    any = any || wb[n] != 0.0;
  }
  double bxb = src[21 * ps + k];
  const int q[7] = {F_D, X1 ? F_M1 : F_M2, X1 ? F_M2 : F_M3, X1 ? F_M3 : F_M1, F_E,
                    X1 ? F_B2C : F_B3C, X1 ? F_B3C : F_B1C};
  const int qx = X1 ? F_B1C : F_B2C;
  if (a.det) {
    // the predictor-face source adjoints of faces k + stride, k and k - stride
    // (the deterministic reverse stores them per face instead of adding them)
    const double* pc = a.ab + (X1 ? A_PC1 : A_PC2) * ps;
    const int bplane = X1 ? F_B1I : F_B2I;
    const int mplane = X1 ? F_M2 : F_M1;
    const double bsum = pc[k + stride] + pc[ps + k] + pc[2 * ps + k - stride];
    const double msum = pc[3 * ps + k + stride] + pc[5 * ps + k];
    const double dsum = pc[4 * ps + k + stride] + pc[6 * ps + k];
    if (bsum != 0.0) ADD(a.ain + bplane * ps, k, bsum);
    if (msum != 0.0) ADD(a.ain + mplane * ps, k, msum);
    if (dsum != 0.0) ADD(a.ain + F_D * ps, k, dsum);
  }
  if (!any && bxb == 0.0) return;
  const EosC eos{g.gamma, g.g1, g.g2};
  const double* st = a.st;
  const Cons7 u{st[q[0] * ps + k], st[q[1] * ps + k], st[q[2] * ps + k], st[q[3] * ps + k],
                st[q[4] * ps + k], st[q[5] * ps + k], st[q[6] * ps + k]};
  Cons7 ub = zero_cons();
  const Prim7 Wb{wb[0], wb[1], wb[2], wb[3], wb[4], wb[5], wb[6]};
  cons_to_prim_b(u, st[qx * ps + k], eos, Wb, ub, bxb);
  for (int n = 0; n < 7; n++) ADD(a.ain + q[n] * ps, k, arr(ub)[n]);
  ADD(a.ain + qx * ps, k, bxb);
}

// blocks [0, n1) x1, the rest x2; `first` skips to the x2 blocks (the
// deterministic reverse launches the sweeps one after the other)
__global__ void __launch_bounds__(kCells) ak_plm_gather(AdjArgs a, int first, int n1) {
  const int b = first + blockIdx.x;
  if (b < n1) plm_gather<true>(a, b);
  else plm_gather<false>(a, b - n1);
}

}  // namespace adjk
}  // namespace athmi

using namespace athmi;
using namespace athmi::adjk;

extern "C" hipError_t athmi_adjoint_launch(const AdjArgs* ap, int kernel, hipStream_t s) {
  const AdjArgs& a = *ap;
  const Inst& g = a.g;
  // blocks of `threads` over a range of (nx2 + dj) x (nx1 + di) positions
  auto blocks = [&](int dj, int di, int threads) {
    return cdiv((g.nx2 + dj) * (g.nx1 + di), threads);
  };
  switch (kernel) {
    case AK_CLEAR:
      hipLaunchKernelGGL(ak_clear, dim3(2048), dim3(256), 0, s, a);
      break;
    case AK_FOLD:
      hipLaunchKernelGGL(ak_fold, dim3(cdiv(frame_cells(g.nx1, g.nx2), kCells)), dim3(kCells), 0, s,
                         a);
      break;
    case AK_CLEAR_GHOST:
      hipLaunchKernelGGL(ak_clear_ghost, dim3(blocks(8, 8, kCells)), dim3(kCells), 0, s, a);
      break;
    case AK_UPDATE:
      hipLaunchKernelGGL(ak_update, dim3(blocks(8, 8, kCells)), dim3(kCells), 0, s, a);
      break;
    case AK_CORRECT: {
      const int n1 = blocks(2, 1, kWave), n2 = blocks(1, 2, kWave), n3 = blocks(2, 2, kWave);
      const auto fn = g.flux == kFluxHlle ? ak_correct<kFluxHlle> : ak_correct<kFluxRoe>;
      hipLaunchKernelGGL(fn, dim3(n1 + n2 + n3), dim3(kWave), 0, s, a, n1, n2);
      break;
    }
    case AK_TRANSVERSE:
      hipLaunchKernelGGL(ak_transverse, dim3(cdiv(g.nx1 + 4, kTileX), cdiv(g.nx2 + 4, kTileY)),
                         dim3(kTileX, kTileY), 0, s, a);
      break;
    case AK_PREDICT: {
      const int n1 = blocks(4, 3, kWave), n2 = blocks(3, 4, kWave), n3 = blocks(4, 4, kWave);
      const auto fn = g.flux == kFluxHlle ? ak_predict<kFluxHlle> : ak_predict<kFluxRoe>;
      hipLaunchKernelGGL(fn, dim3(n1 + n2 + n3), dim3(kWave), 0, s, a, n1, n2);
      break;
    }
    case AK_PLM: {
      const int n = blocks(4, 4, kWave);
      hipLaunchKernelGGL(ak_plm, dim3(2 * n), dim3(kWave), 0, s, a, n);
      break;
    }
    case AK_PLM_GATHER: {
      const int n1 = blocks(4, 6, kCells), n2 = blocks(6, 4, kCells);
      if (a.det) {
        hipLaunchKernelGGL(ak_plm_gather, dim3(n1), dim3(kCells), 0, s, a, 0, n1);
        hipLaunchKernelGGL(ak_plm_gather, dim3(n2), dim3(kCells), 0, s, a, n1, n1);
      } else {
        hipLaunchKernelGGL(ak_plm_gather, dim3(n1 + n2), dim3(kCells), 0, s, a, 0, n1);
      }
      break;
    }
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
