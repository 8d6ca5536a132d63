// adjoint_kernels.hpp -- layout shared by the host side and the adjoint
// (reverse-mode) kernels of one CTU+CT step of a single instance.
#pragma once
#include <hip/hip_runtime.h>

#include "step_kernels.hpp"

namespace athmi {

// adjoint planes (stride Inst::ps, same pitch as the state); each Cons1D-shaped
// group is 7 planes in the sweep's own order. Each plane is stored by one
// kernel over the range its readers cover (entries outside that range stay
// zero from the clear at the start of a reverse pass).
enum AdjPlane {
  A_F1 = 0,     // predictor x1 fluxes
  A_F2 = 7,     // predictor x2 fluxes
  A_B1H = 14,   // half-step face fields, from the corrector Riemann fluxes
  A_B2H = 15,
  A_EMFP = 16,  // corner emf, predictor
  A_F1C = 17,   // corrector x1 fluxes
  A_F2C = 24,   // corrector x2 fluxes
  A_UL1 = 31,   // x1-face states (predictor value = corrected value's identity part)
  A_UR1 = 38,
  A_UL2 = 45,   // x2-face states
  A_UR2 = 52,
  A_WL1 = 59,   // PLM outputs (primitive) at x1 faces before the source terms
  A_WR1 = 66,
  A_WL2 = 73,   // ... at x2 faces
  A_WR2 = 80,
  A_EMFC = 87,  // corner emf, corrector
  A_HD = 88,    // Step 7 per cell: half-step d, M1, M2
  A_HM1 = 89,
  A_HM2 = 90,
  A_HB1 = 91,   // ... and the cell-centred half-step B1c, B2c
  A_HB2 = 92,
  A_PW1 = 93,   // PLM reverse per cell (x1 sweep): adjoints of its 3 stencil cells'
                // primitive states (3 x 7) and of its Bxc (1)
  A_PW2 = 115,  // ... x2 sweep
  A_PC1 = 137,  // deterministic reverse: the predictor-face source adjoints of the x1
                // sweep, per face: B(k-1), B(k), B(k+1), M(k-1), d(k-1), M(k), d(k)
  A_PC2 = 144,  // ... x2 sweep
  NADJ = 151
};

// Everything the adjoint kernels of one step need
struct AdjArgs {
  Inst g;              // the instance (geometry, EOS, pitch, plane stride)
  const double* st;    // S^n: the state the forward pass of this step started from
  const double* sc;    // the forward scratch of this step (predictor + corrector)
  const double* emfp;  // the step's predictor corner emf (Step 4)
  const double* pw;    // NPRIMS planes: the predictor's primitive face states
  double* ab;          // NADJ adjoint planes
  double* ain;         // adjoint of S^n (NSTATE planes), accumulated
  double* aout;        // adjoint of S^{n+1} (NSTATE planes)
  double dt;
  int det;             // 1: deterministic reverse (every sum in a fixed order)
};

enum AdjKernel {
  AK_CLEAR = 0,   // clear all adjoint planes (start of a reverse pass)
  AK_FOLD,        // adjoint of set_bvals on aout: each cell gathers the ghosts that copy it
  AK_CLEAR_GHOST, // clear aout's ghosts (the gradient of ghost values is zero)
  AK_UPDATE,      // Steps 9, 11a, 11b, 13; starts ain
  AK_CORRECT,     // Steps 8b, 8c (corrector fluxes), Step 7 and Step 9's corner emf
  AK_TRANSVERSE,  // Steps 5, 6 and the half-step face fields of Step 4
  AK_PREDICT,     // Steps 1c-1e, 2c-2e (source, prim->cons, predictor flux) per face, Step 4's
                  // corner emf and Step 3
  AK_PLM,         // Steps 1b, 2b (PLM) per cell and sweep
  AK_PLM_GATHER,  // Steps 1a, 2a (cons->prim) per cell, gathering the PLM adjoints
  AK_COUNT
};

}  // namespace athmi

extern "C" hipError_t athmi_adjoint_launch(const athmi::AdjArgs* a, int kernel, hipStream_t s);
