// transfer.hip -- the host-array boundary of one instance: the caller's Gas
// array (8 doubles per cell, athena.h:43-52) and the three interface-field
// arrays, row-major [sy][sx], against the SoA state planes [sy][pitch].
//
// The caller's bytes cross PCIe unchanged into a device staging area and the
// AoS <-> SoA conversion runs here, one thread per padded plane element, so
// the host does no per-cell work. Pure data movement: the values are copied,
// never recomputed.
#include <hip/hip_runtime.h>

#include "step_kernels.hpp"

namespace athmi {
namespace {

constexpr int kXferBlock = 256;
constexpr unsigned kXferMaxBlocks = 16384;

// stage: gas[n][8] | b1i[n] | b2i[n] | b3i[n] with n = sy * sx. Every
// element of the ps-long planes is written: cells from the stage, the pitch
// padding and the tail of each plane with zero.
__global__ void __launch_bounds__(kXferBlock) k_state_unpack(const double* __restrict__ stage,
                                                             double* __restrict__ st, size_t ps,
                                                             int pitch, int sx, int sy) {
  const size_t n = (size_t)sy * sx;
  for (size_t k = (size_t)blockIdx.x * kXferBlock + threadIdx.x; k < ps;
       k += (size_t)gridDim.x * kXferBlock) {
    const size_t j = k / (size_t)pitch, i = k - j * (size_t)pitch;
    const bool cell = j < (size_t)sy && i < (size_t)sx;
    const size_t h = cell ? j * sx + i : 0;
#pragma unroll
    for (int q = 0; q < 8; q++) st[q * ps + k] = cell ? stage[8 * h + q] : 0.0;
    st[F_B1I * ps + k] = cell ? stage[8 * n + h] : 0.0;
    st[F_B2I * ps + k] = cell ? stage[9 * n + h] : 0.0;
    st[F_B3I * ps + k] = cell ? stage[10 * n + h] : 0.0;
  }
}

// the inverse over the sy * sx cells
__global__ void __launch_bounds__(kXferBlock) k_state_pack(const double* __restrict__ st,
                                                           double* __restrict__ stage, size_t ps,
                                                           int pitch, int sx, int sy) {
  const size_t n = (size_t)sy * sx;
  for (size_t h = (size_t)blockIdx.x * kXferBlock + threadIdx.x; h < n;
       h += (size_t)gridDim.x * kXferBlock) {
    const size_t j = h / (size_t)sx, i = h - j * (size_t)sx;
    const size_t k = j * (size_t)pitch + i;
#pragma unroll
    for (int q = 0; q < 8; q++) stage[8 * h + q] = st[q * ps + k];
    stage[8 * n + h] = st[F_B1I * ps + k];
    stage[9 * n + h] = st[F_B2I * ps + k];
    stage[10 * n + h] = st[F_B3I * ps + k];
  }
}

// dense [NSTATE][sy][sx] on the device <-> the planes' cells (the pitch padding
// is neither read nor written). One launch for the eleven planes: as eleven
// 2-D copies the four conversions of a gradient took 0.5 ms at any size.
__global__ void __launch_bounds__(kXferBlock) k_state_dense(double* st, double* dense, size_t ps,
                                                            int pitch, int sx, int sy,
                                                            int to_planes) {
  const size_t n = (size_t)sy * sx;
  for (size_t h = (size_t)blockIdx.x * kXferBlock + threadIdx.x; h < n;
       h += (size_t)gridDim.x * kXferBlock) {
    const size_t j = h / (size_t)sx, i = h - j * (size_t)sx;
    const size_t k = j * (size_t)pitch + i;
    double v[NSTATE];
#pragma unroll
    for (int q = 0; q < NSTATE; q++) v[q] = to_planes ? dense[q * n + h] : st[q * ps + k];
#pragma unroll
    for (int q = 0; q < NSTATE; q++)
      if (to_planes) st[q * ps + k] = v[q];
      else dense[q * n + h] = v[q];
  }
}

// The clocks' heads (everything but the dt slots) to host memory, and one head
// from the launch's arguments to the device: the host reads and writes clocks
// without a copy command, which costs some 15 us a time where a launch costs 4.
constexpr int kHeadWords = (int)(sizeof(ClockHead) / 8);
__global__ void __launch_bounds__(kXferBlock) k_clock_publish(const Clock* __restrict__ clk,
                                                              ClockHead* __restrict__ heads,
                                                              int n) {
  const int e = (int)(blockIdx.x * kXferBlock + threadIdx.x), k = e / kHeadWords;
  if (k >= n) return;
  const int w = e - k * kHeadWords;
  heads[k].w[w] = reinterpret_cast<const unsigned long long*>(clk + k)[w];
}
// (the count of writes that have reached the device follows, for a host that
// cannot wait for the stream)
__global__ void __launch_bounds__(64) k_clock_set(Clock* clk, ClockHead head,
                                                  unsigned long long* done,
                                                  unsigned long long count) {
  // up to divb_bits, which only the device writes
  for (int w = threadIdx.x; w < (int)(offsetof(Clock, divb_bits) / 8); w += 64)
    reinterpret_cast<unsigned long long*>(clk)[w] = head.w[w];
  __threadfence_system();
  if (threadIdx.x == 0)
    __hip_atomic_store(done, count, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

unsigned blocks_for(size_t n) {
  const size_t b = (n + kXferBlock - 1) / kXferBlock;
  return (unsigned)(b < kXferMaxBlocks ? (b ? b : 1) : kXferMaxBlocks);
}

}  // namespace

hipError_t launch_state_unpack(const double* stage, double* st, size_t ps, int pitch, int sx,
                               int sy, hipStream_t s) {
  hipLaunchKernelGGL(k_state_unpack, dim3(blocks_for(ps)), dim3(kXferBlock), 0, s, stage, st, ps,
                     pitch, sx, sy);
  return hipGetLastError();
}

hipError_t launch_state_pack(const double* st, double* stage, size_t ps, int pitch, int sx,
                             int sy, hipStream_t s) {
  hipLaunchKernelGGL(k_state_pack, dim3(blocks_for((size_t)sy * sx)), dim3(kXferBlock), 0, s,
                     st, stage, ps, pitch, sx, sy);
  return hipGetLastError();
}

hipError_t launch_clock_publish(const Clock* clk, ClockHead* heads, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_clock_publish, dim3(cdiv(n * kHeadWords, kXferBlock)), dim3(kXferBlock), 0,
                     s, clk, heads, n);
  return hipGetLastError();
}

hipError_t launch_clock_set(Clock* clk, const ClockHead& head, unsigned long long* done,
                            unsigned long long count, hipStream_t s) {
  hipLaunchKernelGGL(k_clock_set, dim3(1), dim3(64), 0, s, clk, head, done, count);
  return hipGetLastError();
}

hipError_t launch_state_dense(double* st, double* dense, size_t ps, int pitch, int sx, int sy,
                              int to_planes, hipStream_t s) {
  hipLaunchKernelGGL(k_state_dense, dim3(blocks_for((size_t)sy * sx)), dim3(kXferBlock), 0, s, st,
                     dense, ps, pitch, sx, sy, to_planes);
  return hipGetLastError();
}

}  // namespace athmi
