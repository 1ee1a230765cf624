// Three-sweep local part of Hpsi (T + V) for one system on a cubic grid
// L x L x L: one launch per sweep over a band chunk (tile bodies in
// fft3_tiles.hpp).  The projector's V_nl psi (precomputed per owned point)
// and the Taylor accumulations acc += c * hpsi are added in the last sweep's
// write.
//
// Traffic per band: 2 x 16N (z_fwd) + 2 x 16N (xy_kin) + 3 x 16N (z_bwd_epi)
// = 112 N bytes, against 176 N for five pencil passes; run per band chunk
// so W stays resident in the Infinity Cache between sweeps.

#include "fft3_tiles.hpp"
#include "projector_dev.hpp"

#include <cstdlib>

namespace inqamd {

// Shapes of the one-system kernels: z tiles of TY y x 64/TY bands, x-y
// planes with plane_threads(L) or twice as many threads.  The defaults (8,
// 2x: measured fastest at 64^3 x 256) can be overridden through INQAMD_Z_TY
// (8 or 16) and INQAMD_XY_WIDE (0 or 1).

template <int R0, int R1, int R2, int TY>
__global__ __launch_bounds__(z_threads(R0 * R1 * R2)) void z_fwd_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  constexpr int TB = Z_COLS / TY;
  const long tiles = z_tiles<TY>(R0 * R1 * R2, a.nb);
  if (blockIdx.x >= tiles) {
    phase_block(a, (int)(blockIdx.x - tiles));
    return;
  }
  const long t = a.xcd ? xcd_tile(blockIdx.x, tiles, (a.nb + TB - 1) / TB) : (long)blockIdx.x;
  z_fwd_tile<R0, R1, R2, TY, z_threads(R0 * R1 * R2)>(a, t, lds);
}

constexpr int wide_threads(int L) {
  return 2 * plane_threads(L) > 1024 ? 1024 : 2 * plane_threads(L);
}

template <int R0, int R1, int R2, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(xy_kin_waves<R0, R1, R2, NT>())))
void xy_kin_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  xy_kin_plane<R0, R1, R2, NT>(a, blockIdx.x, lds);
}

// The same planes after the workgroups of the projector (projector_beside_planes)
constexpr int proj_plane_threads(int L) { return wide_threads(L) < P4_NT ? wide_threads(L) : P4_NT; }

template <int R0, int R1, int R2>
constexpr size_t xy_proj_lds() {
  return xy_kin_lds<R0, R1, R2>() > P4_BLOCK_LDS ? xy_kin_lds<R0, R1, R2>() : P4_BLOCK_LDS;
}

template <int R0, int R1, int R2>
__global__ __launch_bounds__(P4_NT) __attribute__((amdgpu_waves_per_eu(4)))
void xy_proj_kernel(const fft3_args a, const project_expand_args pa, int ntile, int nproj) {
  extern __shared__ cplx lds[];
  if ((int)blockIdx.x < nproj)
    p4_block(pa, blockIdx.x, ntile, lds);
  else
    xy_kin_plane<R0, R1, R2, proj_plane_threads(R0 * R1 * R2)>(a, blockIdx.x - nproj, lds);
}

// TY: y values of a 64-column tile (8 or 16); a 32-column tile takes TY / 2
// (the same bands per tile)
constexpr int z_bwd_ty(int L, bool taylor, int ty) {
  return z_bwd_cols(L, taylor) == Z_COLS ? ty : ty / 2;
}

template <int R0, int R1, int R2, int TY, bool ACC, bool FWD>
__global__ __launch_bounds__(z_bwd_threads(R0 * R1 * R2, ACC || FWD))
__attribute__((amdgpu_waves_per_eu(z_bwd_waves(R0 * R1 * R2))))
void z_bwd_epi_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  constexpr int L = R0 * R1 * R2;
  // the plain Hpsi's tiles dealt per XCD (64^3 x 256 Hpsi 1.495 -> 1.480
  // ms); the Taylor forms keep the natural order (their steps ran 1 % slower
  // dealt per XCD)
  constexpr bool T = ACC || FWD;
  constexpr int TB = z_bwd_cols(L, T) / z_bwd_ty(L, T, TY);
  const long t =
      T && !a.xcd ? (long)blockIdx.x : xcd_tile(blockIdx.x, gridDim.x, (a.nb + TB - 1) / TB);
  z_bwd_epi_tile<R0, R1, R2, z_bwd_ty(L, T, TY), z_bwd_threads(L, T), ACC, false, FWD,
                 z_bwd_cols(L, T)>(a, t, lds);
}

template <int R0, int R1, int R2, int TY, bool ACC, bool FWD>
static void z_bwd_launch(const fft3_args &a, hipStream_t stream) {
  constexpr int L = R0 * R1 * R2, ZC = z_bwd_cols(L, ACC || FWD);
  const long tiles = z_tiles<z_bwd_ty(L, ACC || FWD, TY), ZC>(L, a.nb);
  hipLaunchKernelGGL((z_bwd_epi_kernel<R0, R1, R2, TY, ACC, FWD>), dim3((unsigned)tiles),
                     dim3(z_bwd_threads(L, ACC || FWD)), z_bwd_lds(L, ZC), stream, a);
}

// G-space Hpsi sweeps
template <int R0, int R1, int R2, int TY, bool PRE>
__global__ __launch_bounds__(z_threads(R0 * R1 * R2)) void z_inv_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  constexpr int TB = Z_COLS / TY;
  const long t = a.xcd ? xcd_tile(blockIdx.x, gridDim.x, (a.nb + TB - 1) / TB) : (long)blockIdx.x;
  z_fwd_tile<R0, R1, R2, TY, z_threads(R0 * R1 * R2), +1, false, PRE>(a, t, lds);
}

template <int R0, int R1, int R2, int NT, bool GATHER>
__global__ __launch_bounds__(NT) void xy_real_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  xy_real_plane<R0, R1, R2, NT, GATHER>(a, xcd_tile(blockIdx.x, gridDim.x, a.nb), lds);
}

template <int R0, int R1, int R2, int TY, bool MM>
__global__ __launch_bounds__(z_threads(R0 * R1 * R2))
__attribute__((amdgpu_waves_per_eu(z_bwd_waves(R0 * R1 * R2))))
void z_kin_kernel(const fft3_args a) {
  extern __shared__ cplx lds[];
  constexpr int TB = Z_COLS / TY;
  const long t = a.xcd ? xcd_tile(blockIdx.x, gridDim.x, (a.nb + TB - 1) / TB) : (long)blockIdx.x;
  z_bwd_epi_tile<R0, R1, R2, TY, z_threads(R0 * R1 * R2), false, true, false, Z_COLS, false, MM>(
      a, t, lds);
}

static int z_ty_choice() {
  static const int ty = [] {
    const char *e = getenv("INQAMD_Z_TY");
    return e && atoi(e) == 16 ? 16 : 8;
  }();
  return ty;
}

static bool xy_wide_choice() {
  static const bool w = [] {
    const char *e = getenv("INQAMD_XY_WIDE");
    return !(e && atoi(e) == 0);
  }();
  return w;
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
template <typename K>
static void ensure_lds(K kernel, size_t bytes) {
  if (bytes > 65536)
    INQAMD_HIP_CHECK(hipFuncSetAttribute((const void *)kernel,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
}

template <int R0, int R1, int R2>
static void prepare3() {
  constexpr int L = R0 * R1 * R2;
  const size_t zl = (size_t)L * Z_COLS * sizeof(cplx), pl = (size_t)L * (L + 1) * sizeof(cplx);
  ensure_lds(z_fwd_kernel<R0, R1, R2, 8>, zl);
  ensure_lds(z_fwd_kernel<R0, R1, R2, 16>, zl);
  ensure_lds(xy_kin_kernel<R0, R1, R2, plane_threads(L)>, xy_kin_lds<R0, R1, R2>());
  ensure_lds(xy_kin_kernel<R0, R1, R2, wide_threads(L)>, xy_kin_lds<R0, R1, R2>());
  if constexpr (L <= PROJ_MAX_LEN) ensure_lds(xy_proj_kernel<R0, R1, R2>, xy_proj_lds<R0, R1, R2>());
  ensure_lds(z_inv_kernel<R0, R1, R2, 8, false>, zl);
  ensure_lds(z_inv_kernel<R0, R1, R2, 8, true>, zl);
  ensure_lds(z_kin_kernel<R0, R1, R2, 8, false>, z_bwd_lds(L));
  ensure_lds(z_kin_kernel<R0, R1, R2, 8, true>, z_bwd_lds(L));
  ensure_lds(xy_real_kernel<R0, R1, R2, wide_threads(L), true>, pl);
  ensure_lds(xy_real_kernel<R0, R1, R2, wide_threads(L), false>, pl);
  const size_t zbp = z_bwd_lds(L, z_bwd_cols(L, false)), zba = z_bwd_lds(L, z_bwd_cols(L, true));
  ensure_lds(z_bwd_epi_kernel<R0, R1, R2, 8, false, false>, zbp);
  ensure_lds(z_bwd_epi_kernel<R0, R1, R2, 16, false, false>, zbp);
  ensure_lds(z_bwd_epi_kernel<R0, R1, R2, 8, true, false>, zba);
  ensure_lds(z_bwd_epi_kernel<R0, R1, R2, 16, true, false>, zba);
  ensure_lds(z_bwd_epi_kernel<R0, R1, R2, 8, false, true>, zba);
  ensure_lds(z_bwd_epi_kernel<R0, R1, R2, 16, false, true>, zba);
  ensure_lds(z_bwd_epi_kernel<R0, R1, R2, 8, true, true>, zba);
  ensure_lds(z_bwd_epi_kernel<R0, R1, R2, 16, true, true>, zba);
}

// proj: the launch of the x-y planes with the projector's workgroups
// sweep: -1 all three, 0/1/2 one of them; fwd_next: the last sweep also
// transforms its output forward in z into W (Taylor chains)
template <int R0, int R1, int R2, int TY, int NT>
static void launch3v(const fft3_args &a, hipStream_t stream, int sweep, bool fwd_next,
                     const project_expand_args *proj) {
  constexpr int L = R0 * R1 * R2;
  const long ztiles = z_tiles<TY>(L, a.nb);
  const size_t zlds = (size_t)L * Z_COLS * sizeof(cplx);
  const size_t plds = xy_kin_lds<R0, R1, R2>();
  if (sweep < 0 || sweep == 0) {
    hipLaunchKernelGGL((z_fwd_kernel<R0, R1, R2, TY>),
                       dim3((unsigned)(ztiles + phase_blocks(a, z_threads(L)))),
                       dim3(z_threads(L)), zlds, stream, a);
    INQAMD_HIP_CHECK(hipGetLastError());
  }
  if (sweep < 0 || sweep == 1) {
    if (proj) {
      if constexpr (L <= PROJ_MAX_LEN) {
        const int ntile = (proj->nbc + P4_BANDS - 1) / P4_BANDS, np = ntile * a.nproj;
        hipLaunchKernelGGL((xy_proj_kernel<R0, R1, R2>), dim3((unsigned)((long)a.nb * L + np)),
                           dim3(P4_NT), (xy_proj_lds<R0, R1, R2>()), stream, a, *proj, ntile, np);
      } else {
        throw error{ERR_UNSUPPORTED, "no plane kernel with the projector for this length"};
      }
    } else {
      hipLaunchKernelGGL((xy_kin_kernel<R0, R1, R2, NT>), dim3((unsigned)((long)a.nb * L)),
                         dim3(NT), plds, stream, a);
    }
    INQAMD_HIP_CHECK(hipGetLastError());
  }
  if (sweep < 0 || sweep == 2) {
    const bool acc = a.acc1 != nullptr;
    if (fwd_next && acc)
      z_bwd_launch<R0, R1, R2, TY, true, true>(a, stream);
    else if (fwd_next)
      z_bwd_launch<R0, R1, R2, TY, false, true>(a, stream);
    else if (acc)
      z_bwd_launch<R0, R1, R2, TY, true, false>(a, stream);
    else
      z_bwd_launch<R0, R1, R2, TY, false, false>(a, stream);
    INQAMD_HIP_CHECK(hipGetLastError());
  }
}

template <int R0, int R1, int R2>
static void launch3(const fft3_args &a, hipStream_t stream, int sweep, bool fwd_next,
                    const project_expand_args *proj) {
  constexpr int L = R0 * R1 * R2;
  const bool wide = a.xy_wide ? a.xy_wide == 2 : xy_wide_choice();
  const int ty = a.z_ty ? a.z_ty : z_ty_choice();
  if (ty == 16) {
    if (wide)
      launch3v<R0, R1, R2, 16, wide_threads(L)>(a, stream, sweep, fwd_next, proj);
    else
      launch3v<R0, R1, R2, 16, plane_threads(L)>(a, stream, sweep, fwd_next, proj);
  } else {
    if (wide)
      launch3v<R0, R1, R2, 8, wide_threads(L)>(a, stream, sweep, fwd_next, proj);
    else
      launch3v<R0, R1, R2, 8, plane_threads(L)>(a, stream, sweep, fwd_next, proj);
  }
}

template <int R0, int R1, int R2>
static void launch_fourier(const fft3_args &a, hipStream_t stream, fourier_half half) {
  constexpr int L = R0 * R1 * R2, NT = wide_threads(L);
  const dim3 tiles((unsigned)z_tiles<8>(L, a.nb)), planes((unsigned)((long)a.nb * L));
  const size_t plds = (size_t)L * (L + 1) * sizeof(cplx);
  if (half == G_INVERSE) {
    const size_t zlds = (size_t)L * Z_COLS * sizeof(cplx);
    if (a.pre_kin)
      hipLaunchKernelGGL((z_inv_kernel<R0, R1, R2, 8, true>), tiles, dim3(z_threads(L)), zlds,
                         stream, a);
    else
      hipLaunchKernelGGL((z_inv_kernel<R0, R1, R2, 8, false>), tiles, dim3(z_threads(L)), zlds,
                         stream, a);
    INQAMD_HIP_CHECK(hipGetLastError());
    if (a.zoff)
      hipLaunchKernelGGL((xy_real_kernel<R0, R1, R2, NT, true>), planes, dim3(NT), plds, stream, a);
    INQAMD_HIP_CHECK(hipGetLastError());
    return;
  }
  hipLaunchKernelGGL((xy_real_kernel<R0, R1, R2, NT, false>), planes, dim3(NT), plds, stream, a);
  INQAMD_HIP_CHECK(hipGetLastError());
  fft3_args k = a;
  k.scale = 1.0;  // (the planes took 1/N)
  if (a.mm_phi)
    hipLaunchKernelGGL((z_kin_kernel<R0, R1, R2, 8, true>), tiles, dim3(z_threads(L)),
                       z_bwd_lds(L), stream, k);
  else
    hipLaunchKernelGGL((z_kin_kernel<R0, R1, R2, 8, false>), tiles, dim3(z_threads(L)),
                       z_bwd_lds(L), stream, k);
  INQAMD_HIP_CHECK(hipGetLastError());
}

void fft3_fourier_hamiltonian(const fft3_args &a, int L, hipStream_t stream, fourier_half half) {
  switch (L) {
#define INQAMD_FFT3_CASE(LL, R0, R1, R2) \
  case LL: launch_fourier<R0, R1, R2>(a, stream, half); return;
    INQAMD_FFT3_TABLE(INQAMD_FFT3_CASE)
#undef INQAMD_FFT3_CASE
    default: throw error{ERR_UNSUPPORTED, "G-space three-sweep Hpsi: unsupported grid length"};
  }
}

bool fft3_supported(int L, size_t max_lds) {
  switch (L) {
#define INQAMD_FFT3_CASE(LL, R0, R1, R2) case LL:
    INQAMD_FFT3_TABLE(INQAMD_FFT3_CASE)
#undef INQAMD_FFT3_CASE
      return (size_t)L * (L + 1) * sizeof(cplx) <= max_lds && z_bwd_lds(L) <= max_lds;
    default: return false;
  }
}

void fft3_prepare(int L) {
  switch (L) {
#define INQAMD_FFT3_CASE(LL, R0, R1, R2) \
  case LL: prepare3<R0, R1, R2>(); return;
    INQAMD_FFT3_TABLE(INQAMD_FFT3_CASE)
#undef INQAMD_FFT3_CASE
    default: return;
  }
}

void fft3_local_hamiltonian(const fft3_args &a, int L, hipStream_t stream, int sweep,
                            bool fwd_next, const project_expand_args *proj) {
  switch (L) {
#define INQAMD_FFT3_CASE(LL, R0, R1, R2) \
  case LL: launch3<R0, R1, R2>(a, stream, sweep, fwd_next, proj); return;
    INQAMD_FFT3_TABLE(INQAMD_FFT3_CASE)
#undef INQAMD_FFT3_CASE
    default: throw error{ERR_UNSUPPORTED, "three-sweep Hpsi: unsupported grid length"};
  }
}

// The planes then run in workgroups of P4_NT threads: at 48 to 64 they do so
// anyway (384 to 512), below that only where the launch is too small for the
// idle threads to matter.
bool fft3_projector(int L, int nb, int xy_wide) {
  if (xy_wide ? xy_wide != 2 : !xy_wide_choice()) return false;
  return L <= PROJ_MAX_LEN && (L >= 48 || (long)nb * L <= PROJ_FEW_PLANES);
}

}  // namespace inqamd
