// Launches of the nx x ny x nz three-sweep Hpsi (see fft3_rect.hpp).
#include "fft3_rect_xy.hpp"

namespace inqamd {

extern template void rect_xy_launch<128>(const fft3_args &, const int[3], rect_planes, double *,
                                         hipStream_t);
extern template void rect_xy_launch<256>(const fft3_args &, const int[3], rect_planes, double *,
                                         hipStream_t);
extern template void rect_xy_launch<512>(const fft3_args &, const int[3], rect_planes, double *,
                                         hipStream_t);
extern template void rect_xy_launch<1024>(const fft3_args &, const int[3], rect_planes, double *,
                                          hipStream_t);

// The kinetic planes after the workgroups of the projector
// (projector_beside_planes)
__global__ __launch_bounds__(P4_NT) __attribute__((amdgpu_waves_per_eu(4)))
void rect_xy_proj_kernel(const fft3_args a, int nz, const project_expand_args pa, int ntile,
                         int nproj) {
  extern __shared__ cplx lds[];
  if ((int)blockIdx.x < nproj)
    p4_block(pa, blockIdx.x, ntile, lds);
  else
    rect_xy_plane<P4_NT>(a, nz, blockIdx.x - nproj, lds);
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
static void rect_xy(const fft3_args &a, const int n[3], rect_planes what, hipStream_t stream,
                    double *rows = nullptr) {
  const int el = n[0] * n[1];
  if (el <= rect_elements(128))
    rect_xy_launch<128>(a, n, what, rows, stream);
  else if (el <= rect_elements(256))
    rect_xy_launch<256>(a, n, what, rows, stream);
  else if (el <= rect_elements(512))
    rect_xy_launch<512>(a, n, what, rows, stream);
  else
    rect_xy_launch<1024>(a, n, what, rows, stream);
}

static bool rect_length(int L) {
  switch (L) {
#define INQAMD_RECT_CASE(LL, R0, R1, R2) case LL:
    INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
      return true;
    default: return false;
  }
}

bool fft3_rect_supported(const int n[3], size_t max_lds) {
  return rect_length(n[0]) && rect_length(n[1]) && rect_length(n[2]) &&
         n[0] * n[1] <= rect_elements(1024) && rect_xy_lds(n) <= max_lds &&
         z_bwd_lds(n[2]) <= max_lds;
}

static void rect_z(const fft3_args &a, int nz, rect_z_kernel k, hipStream_t stream) {
  if (rect_z_launch_a(a, nz, k, stream) || rect_z_launch_b(a, nz, k, stream) ||
      rect_z_launch_c(a, nz, k, stream))
    return;
  throw error{ERR_UNSUPPORTED, "three-sweep Hpsi: unsupported z length"};
}

void fft3_rect_prepare(const int n[3]) {
  const size_t lds = rect_xy_lds(n);
  if (lds > 65536)
    INQAMD_HIP_CHECK(hipFuncSetAttribute((const void *)rect_xy_proj_kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
  fft3_moments_prepare(n);
  rect_z(fft3_args{}, n[2], RECT_Z_PREPARE, nullptr);
}

// As fft3_projector: planes of a 512-thread workgroup's size, or few of them
bool fft3_rect_projector(const int n[3], int nb) {
  const int el = n[0] * n[1];
  return el <= rect_elements(P4_NT) &&
         (el > rect_elements(P4_NT / 2) || (long)nb * n[2] <= PROJ_FEW_PLANES);
}

void fft3_rect_local_hamiltonian(const fft3_args &a, const int n[3], hipStream_t stream, int sweep,
                                 bool fwd_next, const project_expand_args *proj) {
  if (sweep < 0 || sweep == 0) rect_z(a, n[2], RECT_Z_FWD, stream);
  if ((sweep < 0 || sweep == 1) && proj) {
    const int ntile = (proj->nbc + P4_BANDS - 1) / P4_BANDS, np = ntile * a.nproj;
    const size_t lds = rect_xy_lds(n) > P4_BLOCK_LDS ? rect_xy_lds(n) : P4_BLOCK_LDS;
    hipLaunchKernelGGL(rect_xy_proj_kernel, dim3((unsigned)((long)a.nb * n[2] + np)), dim3(P4_NT),
                       lds, stream, a, n[2], *proj, ntile, np);
    INQAMD_HIP_CHECK(hipGetLastError());
  } else if (sweep < 0 || sweep == 1) {
    rect_xy(a, n, RECT_KINETIC, stream);
  }
  if (sweep < 0 || sweep == 2)
    rect_z(a, n[2],
           a.acc1 ? (fwd_next ? RECT_Z_BWD_ACC_FWD : RECT_Z_BWD_ACC)
                  : (fwd_next ? RECT_Z_BWD_FWD : RECT_Z_BWD),
           stream);
}

bool fft3_moments_supported(const int n[3], size_t max_lds) {
  return rect_length(n[0]) && rect_length(n[1]) && n[0] * n[1] <= rect_elements(1024) &&
         rect_xy_lds(n) <= max_lds;
}

void fft3_moments_prepare(const int n[3]) { rect_xy(fft3_args{}, n, RECT_XY_PREPARE, nullptr); }

void fft3_moments(const fft3_args &a, const int n[3], double *rows, hipStream_t stream) {
  rect_xy(a, n, RECT_MOMENTS, stream, rows);
}

void fft3_rect_fourier_hamiltonian(const fft3_args &a, const int n[3], hipStream_t stream,
                                   fourier_half half) {
  if (half == G_INVERSE) {
    rect_z(a, n[2], RECT_Z_INV, stream);
    if (a.zoff) rect_xy(a, n, RECT_GATHER, stream);
    return;
  }
  rect_xy(a, n, RECT_POTENTIAL, stream);
  fft3_args k = a;
  k.scale = 1.0;  // (the planes took 1/N)
  rect_z(k, n[2], RECT_Z_KIN, stream);
}

}  // namespace inqamd
