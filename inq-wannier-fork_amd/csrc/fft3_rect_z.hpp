// z-sweep kernels of fft3_rect.hpp, included by the files that instantiate them.
#pragma once

#include "fft3_rect.hpp"
#include "projector_dev.hpp"

namespace inqamd {

constexpr int RECT_TY = 8;  // y values of a 64-column tile (4 of a 32-column one)

template <int R0, int R1, int R2, int SIGN, bool PRE>
__global__ __launch_bounds__(z_threads(R0 * R1 * R2)) void rect_z_fwd_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  constexpr int TB = Z_COLS / RECT_TY;
  const int nbt = (a.nb + TB - 1) / TB;
  const long tiles = (long)a.nx * ((a.ny + RECT_TY - 1) / RECT_TY) * nbt;
  if (blockIdx.x >= tiles) {
    phase_block(a, (int)(blockIdx.x - tiles));
    return;
  }
  const long t = a.xcd ? xcd_tile(blockIdx.x, tiles, nbt) : (long)blockIdx.x;
  z_fwd_tile<R0, R1, R2, RECT_TY, z_threads(R0 * R1 * R2), SIGN, true, PRE>(a, t, lds);
}

template <int R0, int R1, int R2, bool ACC, bool FWD>
__global__ __launch_bounds__(z_bwd_threads(R0 * R1 * R2, ACC || FWD))
__attribute__((amdgpu_waves_per_eu(z_bwd_waves(R0 * R1 * R2))))
void rect_z_bwd_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  constexpr int L = R0 * R1 * R2;
  constexpr bool T = ACC || FWD;
  constexpr int ZC = z_bwd_cols(L, T), TY = ZC == Z_COLS ? RECT_TY : RECT_TY / 2, TB = ZC / TY;
  const long t =
      T && !a.xcd ? (long)blockIdx.x : xcd_tile(blockIdx.x, gridDim.x, (a.nb + TB - 1) / TB);
  z_bwd_epi_tile<R0, R1, R2, TY, z_bwd_threads(L, T), ACC, false, FWD, ZC, true>(a, t, lds);
}

template <int R0, int R1, int R2, bool MM>
__global__ __launch_bounds__(z_threads(R0 * R1 * R2))
__attribute__((amdgpu_waves_per_eu(z_bwd_waves(R0 * R1 * R2))))
void rect_z_kin_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  constexpr int TB = Z_COLS / RECT_TY;
  const long t = a.xcd ? xcd_tile(blockIdx.x, gridDim.x, (a.nb + TB - 1) / TB) : (long)blockIdx.x;
  z_bwd_epi_tile<R0, R1, R2, RECT_TY, z_threads(R0 * R1 * R2), false, true, false, Z_COLS, true, MM>(
      a, t, lds);
}

template <typename K>
static void rect_lds(K kernel, size_t bytes) {
  if (bytes > 65536)
    INQAMD_HIP_CHECK(hipFuncSetAttribute((const void *)kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

template <int R0, int R1, int R2, bool ACC, bool FWD>
static void rect_z_bwd(const fft3_args &a, hipStream_t stream, bool prepare) {
  constexpr int L = R0 * R1 * R2, ZC = z_bwd_cols(L, ACC || FWD);
  constexpr int TY = ZC == Z_COLS ? RECT_TY : RECT_TY / 2, TB = ZC / TY;
  if (prepare) {
    rect_lds(rect_z_bwd_kernel<R0, R1, R2, ACC, FWD>, z_bwd_lds(L, ZC));
    return;
  }
  const long tiles = (long)a.nx * ((a.ny + TY - 1) / TY) * ((a.nb + TB - 1) / TB);
  hipLaunchKernelGGL((rect_z_bwd_kernel<R0, R1, R2, ACC, FWD>), dim3((unsigned)tiles),
                     dim3(z_bwd_threads(L, ACC || FWD)), z_bwd_lds(L, ZC), stream, a);
  INQAMD_HIP_CHECK(hipGetLastError());
}

template <int R0, int R1, int R2>
static void rect_z_run(const fft3_args &a, rect_z_kernel k, hipStream_t stream) {
  constexpr int L = R0 * R1 * R2, TB = Z_COLS / RECT_TY;
  constexpr size_t zl = (size_t)L * Z_COLS * sizeof(cplx);
  const long tiles = (long)a.nx * ((a.ny + RECT_TY - 1) / RECT_TY) * ((a.nb + TB - 1) / TB);
  const bool prep = k == RECT_Z_PREPARE;
  if (prep) {
    rect_lds(rect_z_fwd_kernel<R0, R1, R2, -1, false>, zl);
    rect_lds(rect_z_fwd_kernel<R0, R1, R2, +1, false>, zl);
    rect_lds(rect_z_fwd_kernel<R0, R1, R2, +1, true>, zl);
    rect_lds(rect_z_kin_kernel<R0, R1, R2, false>, z_bwd_lds(L));
    rect_lds(rect_z_kin_kernel<R0, R1, R2, true>, z_bwd_lds(L));
  }
  if (prep || k == RECT_Z_BWD) rect_z_bwd<R0, R1, R2, false, false>(a, stream, prep);
  if (prep || k == RECT_Z_BWD_ACC) rect_z_bwd<R0, R1, R2, true, false>(a, stream, prep);
  if (prep || k == RECT_Z_BWD_FWD) rect_z_bwd<R0, R1, R2, false, true>(a, stream, prep);
  if (prep || k == RECT_Z_BWD_ACC_FWD) rect_z_bwd<R0, R1, R2, true, true>(a, stream, prep);
  if (k == RECT_Z_FWD)
    hipLaunchKernelGGL((rect_z_fwd_kernel<R0, R1, R2, -1, false>),
                       dim3((unsigned)(tiles + phase_blocks(a, z_threads(L)))),
                       dim3(z_threads(L)), zl, stream, a);
  if (k == RECT_Z_INV && a.pre_kin)
    hipLaunchKernelGGL((rect_z_fwd_kernel<R0, R1, R2, +1, true>), dim3((unsigned)tiles),
                       dim3(z_threads(L)), zl, stream, a);
  if (k == RECT_Z_INV && !a.pre_kin)
    hipLaunchKernelGGL((rect_z_fwd_kernel<R0, R1, R2, +1, false>), dim3((unsigned)tiles),
                       dim3(z_threads(L)), zl, stream, a);
  if (k == RECT_Z_KIN && a.mm_phi)
    hipLaunchKernelGGL((rect_z_kin_kernel<R0, R1, R2, true>), dim3((unsigned)tiles),
                       dim3(z_threads(L)), z_bwd_lds(L), stream, a);
  if (k == RECT_Z_KIN && !a.mm_phi)
    hipLaunchKernelGGL((rect_z_kin_kernel<R0, R1, R2, false>), dim3((unsigned)tiles),
                       dim3(z_threads(L)), z_bwd_lds(L), stream, a);
  INQAMD_HIP_CHECK(hipGetLastError());
}

#define INQAMD_RECT_Z_CASE(L, R0, R1, R2) \
  case L: rect_z_run<R0, R1, R2>(a, k, stream); return true;

}  // namespace inqamd
