// Three-sweep local Hpsi (T + V) on nx x ny x nz grids: the z sweeps are the
// tiles of fft3_tiles.hpp with run-time x and y extents, one set of kernels per
// z length; the x-y sweep is one kernel per workgroup size that picks the plans
// of its two axes at run time.  Kernels for every pair of x and y lengths would
// be several hundred; a plan is a few kilobytes of code, and one uniform switch
// per axis and direction costs nothing beside a plane's loads.
//
// Five pencil passes move 176 B per point and band and add V_nl psi and the
// Taylor terms in passes of their own; the three sweeps move 112 with both
// fused.  Against the pencil passes: Hpsi at 48 x 60 x 72 x 101 bands 817 -> 738
// us (674 since its z tiles are dealt per XCD), at 25 x 45 x 27 x 45 86 -> 67 us,
// at 80 x 90 x 96 x 20 508 -> 499 us; the ETRS step at 32 x 25 x 90 x 60 1519 ->
// 1295 us, the interacting step at 60 x 36 x 27 x 43 2.53 -> 2.07 ms, the adjoint
// of 8 steps at 20 x 60 x 36 x 12 (whose fused half steps need the sweeps) 20.1 ->
// 11.3 ms.
#pragma once

#include "fft3_tiles.hpp"

namespace inqamd {

// Kernels of one z length (explicitly instantiated over the fft3_rect_z*.hip)
enum rect_z_kernel : int {
  RECT_Z_FWD,          // z forward
  RECT_Z_BWD,          // z backward with V psi + V_nl psi
  RECT_Z_BWD_ACC,      // ... and the Taylor sums
  RECT_Z_BWD_FWD,      // ... transforming its output forward
  RECT_Z_BWD_ACC_FWD,  // ... both
  RECT_Z_INV,          // z inverse (G-space Hpsi)
  RECT_Z_KIN,          // z forward with the kinetic term (G-space Hpsi)
  RECT_Z_PREPARE       // LDS attributes of them all
};

// Launches `k` for z length nz; false when nz is not in this file's list
bool rect_z_launch_a(const fft3_args &a, int nz, rect_z_kernel k, hipStream_t stream);
bool rect_z_launch_b(const fft3_args &a, int nz, rect_z_kernel k, hipStream_t stream);
bool rect_z_launch_c(const fft3_args &a, int nz, rect_z_kernel k, hipStream_t stream);

// Kernels of the x-y planes, by threads of their workgroups (explicitly instantiated
// over the fft3_rect_x*.hip)
enum rect_planes : int {
  RECT_KINETIC,    // forward, 1/2 |G+k+A|^2, back
  RECT_GATHER,     // psi at the owned points (G-space Hpsi)
  RECT_POTENTIAL,  // to real space, V psi + V_nl psi, back (G-space Hpsi)
  RECT_MOMENTS,    // sums of |psi^|^2 into rows (fft3_moments)
  RECT_XY_PREPARE  // LDS attributes of them all
};

// Most elements of a plane for a workgroup of NT threads
constexpr int rect_elements(int NT) {
  return NT == 128 ? 1280 : (NT == 256 ? 3072 : (NT == 512 ? 5120 : 10240));
}

inline size_t rect_xy_lds(const int n[3]) { return (size_t)n[0] * (n[1] | 1) * sizeof(cplx); }

// Launches `what` for planes of n[0] x n[1] <= rect_elements(NT)
template <int NT>
void rect_xy_launch(const fft3_args &a, const int n[3], rect_planes what, double *rows,
                    hipStream_t stream);

// (length, radices of the z tiles): the lengths up to 96 that two or three
// butterflies reach, from 20 on (shorter axes leave the sweeps' tiles mostly
// empty), the cubic grids' with their plans
#define INQAMD_RECT_Z_A(X) \
  X(20, 5, 4, 1)           \
  X(24, 8, 3, 1)           \
  X(25, 5, 5, 1)           \
  X(27, 9, 3, 1)           \
  X(28, 7, 4, 1)           \
  X(30, 6, 5, 1)           \
  X(32, 8, 4, 1)           \
  X(36, 6, 6, 1)
#define INQAMD_RECT_Z_B(X) \
  X(40, 8, 5, 1)           \
  X(42, 7, 6, 1)           \
  X(45, 9, 5, 1)           \
  X(48, 8, 6, 1)           \
  X(50, 10, 5, 1)          \
  X(54, 9, 6, 1)           \
  X(56, 8, 7, 1)           \
  X(60, 12, 5, 1)
#define INQAMD_RECT_Z_C(X) \
  X(64, 8, 8, 1)           \
  X(70, 10, 7, 1)          \
  X(72, 8, 9, 1)           \
  X(75, 5, 5, 3)           \
  X(80, 8, 2, 5)           \
  X(84, 12, 7, 1)          \
  X(90, 10, 9, 1)          \
  X(96, 8, 4, 3)

// The same lengths with the radices of the x-y planes: two stages wherever the
// butterflies allow (each stage is an LDS pass and a barrier)
#define INQAMD_RECT_XY(X) \
  X(20, 5, 4, 1)          \
  X(24, 6, 4, 1)          \
  X(25, 5, 5, 1)          \
  X(27, 9, 3, 1)          \
  X(28, 7, 4, 1)          \
  X(30, 6, 5, 1)          \
  X(32, 8, 4, 1)          \
  X(36, 6, 6, 1)          \
  X(40, 8, 5, 1)          \
  X(42, 7, 6, 1)          \
  X(45, 9, 5, 1)          \
  X(48, 8, 6, 1)          \
  X(50, 10, 5, 1)         \
  X(54, 9, 6, 1)          \
  X(56, 8, 7, 1)          \
  X(60, 10, 6, 1)         \
  X(64, 8, 8, 1)          \
  X(70, 10, 7, 1)         \
  X(72, 9, 8, 1)          \
  X(75, 5, 5, 3)          \
  X(80, 10, 8, 1)         \
  X(84, 12, 7, 1)         \
  X(90, 10, 9, 1)         \
  X(96, 12, 8, 1)

constexpr int RECT_MAX_LEN = 96;

}  // namespace inqamd
