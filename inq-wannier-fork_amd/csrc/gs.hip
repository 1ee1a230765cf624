// Ground-state pieces: operations::laplacian_add, operations::preconditioner
// (Teter-Payne-Allan), operations::orthogonalize,
// eigensolvers::steepest_descent on G-space orbitals and
// ground_state::subspace_diagonalization, the eigensolver steps of
// ground_state/calculator.hpp:150-180.
//
// Steepest descent keeps hphi, the residual and H residual in a workspace of
// three [N][max_bands] arrays allocated on first use.  Its per-band sums run
// as fused streaming passes (partial sums per point chunk, then a fixed-order
// sum over chunks, so results do not depend on scheduling):
//   pass 1  eig = <hphi|phi>, norm = <phi|phi>
//   pass 2  residual = hphi - (eig/norm) phi, written, with the kinetic sums
//           of the preconditioner sum 1/2|G|^2 |r|^2 and sum |r|^2
//   pass 3  residual *= K(1/2|G|^2 / kinetic)
//   H residual (G-space Hpsi)
//   pass 4  <r|r>, <phi|r>, <r|Hr>, <phi|Hr> and the step lambda per band (on
//           three-sweep grids in the sweep that writes H residual)
//   pass 5  phi += lambda r, hphi += lambda Hr, with pass 2 of the next step, whose
//           eig and norm follow from this step's sums
// orthogonalize forms S = dV Phi^H Phi (gram.hip),
// factors it (S = R R^H, R lower: cholesky.hip) and applies Phi <- Phi R^-H in
// place (rotate.hip); the subspace diagonalisation diagonalises dV Phi^H H Phi with
// rocSOLVER ZHEEVD.

#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdlib>
#include <vector>

#include "internal.hpp"
#include "inq_amd.h"

namespace inqamd {
namespace {

// The per-band reductions run in blocks of 256 threads over a chunk of points and
// BT = 64 or 16 bands, 256 / BT lanes of points per band: 16 where 64 would leave
// a quarter of the lanes or more without a band (the descent at 40^3 x 48 bands
// 2.54 -> 1.90 ms together with the shorter chunks).  Chunks of up to
// GS_CHUNK points, shorter where that would leave fewer than GS_BLOCKS blocks
// (125 for 40^3 x 48, on 256 CUs).
constexpr long GS_CHUNK = 512;
constexpr long GS_CHUNK_MIN = 64;
constexpr long GS_BLOCKS = 2048;

struct gs_state {
  cplx *hphi = nullptr, *res = nullptr, *hres = nullptr;  // [N][max_bands] each
  double *part = nullptr;   // [nchunk][max_bands][8] partial sums
  double *band = nullptr;   // [max_bands][16] per-band results
  rocblas_handle blas = nullptr;
  cplx *S = nullptr;        // [max_bands]^2 device overlap / rotation
  cplx *T = nullptr;        // [max_bands]^2 rotation of orthogonalize
  cplx *chol = nullptr;     // scratch of the Cholesky factorisation
  double *eig = nullptr;    // [2 max_bands] eigenvalues + tridiagonal work
  cplx *ip_part = nullptr;  // [max_bands]^2 scratch of inner products in one slice
  rocblas_int *info = nullptr;
};

#define GS_BLAS_CHECK(expr)                                                              \
  do {                                                                                   \
    rocblas_status _s = (expr);                                                          \
    if (_s != rocblas_status_success)                                                    \
      throw ::inqamd::error{::inqamd::ERR_HIP, std::string(#expr) + ": " +              \
                                                   rocblas_status_to_string(_s)};        \
  } while (0)

// Launch shape of the per-band reductions over nst bands
struct gs_shape {
  int bt;       // bands per block
  long groups;  // blocks of bands
  long chunk;   // points per partial sum
  long nchunk;
};

gs_shape shape(const handle &h, int nst) {
  gs_shape g;
  g.bt = nst % 64 == 0 || nst % 64 > 48 ? 64 : 16;
  g.groups = (nst + g.bt - 1) / g.bt;
  g.chunk = (h.npoint * g.groups + GS_BLOCKS - 1) / GS_BLOCKS;
  g.chunk = g.chunk < GS_CHUNK_MIN ? GS_CHUNK_MIN : (g.chunk > GS_CHUNK ? GS_CHUNK : g.chunk);
  g.nchunk = (h.npoint + g.chunk - 1) / g.chunk;
  return g;
}

// Most partial sums (chunks x bands) of any nst <= max_bands: chunks of
// GS_CHUNK, or GS_BLOCKS blocks of at most 64 bands (and a chunk cut short in
// each band group), or the rows of the line sums
long most_partials(const handle &h) {
  const long full = (h.npoint + GS_CHUNK - 1) / GS_CHUNK * h.max_bands;
  const long split = (GS_BLOCKS + h.max_bands / 16 + 1) * 64;
  const long line = h.three_sweep ? line_sum_rows(h.n[0], h.n[1]) * h.max_bands : 0;
  return std::max(full, std::max(split, line));
}

gs_state &state(handle &h) {
  if (!h.gs) h.gs = new gs_state();
  return *static_cast<gs_state *>(h.gs);
}

void *dalloc(size_t bytes) {
  void *p = nullptr;
  if (hipMalloc(&p, bytes) != hipSuccess)
    throw error{ERR_MEMORY, "device allocation of " + std::to_string(bytes) + " bytes failed"};
  return p;
}

void ensure_reductions(handle &h) {
  gs_state &g = state(h);
  if (!g.part) {
    g.part = (double *)dalloc((size_t)most_partials(h) * 8 * sizeof(double));
    g.band = (double *)dalloc((size_t)h.max_bands * 16 * sizeof(double));
  }
}

void ensure_workspace(handle &h) {
  gs_state &g = state(h);
  ensure_reductions(h);
  if (!g.hphi) {
    const size_t orb = (size_t)h.npoint * h.max_bands * sizeof(cplx);
    g.hphi = (cplx *)dalloc(orb);
    g.res = (cplx *)dalloc(orb);
    g.hres = (cplx *)dalloc(orb);
  }
}

void ensure_blas(handle &h) {
  gs_state &g = state(h);
  if (!g.blas) {
    rotate_prepare();
    GS_BLAS_CHECK(rocblas_create_handle(&g.blas));
  }
  if (!g.S) g.S = (cplx *)dalloc((size_t)h.max_bands * h.max_bands * sizeof(cplx));
  if (!g.T) g.T = (cplx *)dalloc((size_t)h.max_bands * h.max_bands * sizeof(cplx));
  if (!g.chol) g.chol = (cplx *)dalloc((size_t)cholesky_scratch(h.max_bands) * sizeof(cplx));
  if (!g.eig) g.eig = (double *)dalloc((size_t)2 * h.max_bands * sizeof(double));
  if (!g.info) g.info = (rocblas_int *)dalloc(sizeof(rocblas_int));
  if (!g.ip_part)
    g.ip_part = (cplx *)dalloc((size_t)h.max_bands * h.max_bands * sizeof(cplx));
  GS_BLAS_CHECK(rocblas_set_stream(g.blas, h.stream));
}

// Grid geometry for the G-space kernels: G covariant = 2 pi m with m the
// symmetric index (fourier_space.hpp:66-81), |G|^2 through the reciprocal
// lattice rows b_i (which carry the 2 pi).
struct gspace {
  int n0, n1, n2;
  double b[9];
  __device__ void m_of(long point, int &m0, int &m1, int &m2) const {
    const unsigned p = (unsigned)point;  // (grids have fewer than 2^31 points)
    const unsigned t = p / (unsigned)n2;
    const int iz = (int)(p - t * (unsigned)n2);
    const int iy = (int)(t % (unsigned)n1), ix = (int)(t / (unsigned)n1);
    m0 = ix >= (n0 + 1) / 2 ? ix - n0 : ix;
    m1 = iy >= (n1 + 1) / 2 ? iy - n1 : iy;
    m2 = iz >= (n2 + 1) / 2 ? iz - n2 : iz;
  }
  __device__ double g2(int m0, int m1, int m2) const {
    const double gx = m0 * b[0] + m1 * b[3] + m2 * b[6];
    const double gy = m0 * b[1] + m1 * b[4] + m2 * b[7];
    const double gz = m0 * b[2] + m1 * b[5] + m2 * b[8];
    return gx * gx + gy * gy + gz * gz;
  }
};

gspace geometry(const handle &h) {
  gspace g;
  g.n0 = h.n[0];
  g.n1 = h.n[1];
  g.n2 = h.n[2];
  for (int i = 0; i < 9; i++) g.b[i] = h.rlat[i];
  return g;
}

unsigned grid1(long total) {
  long b = (total + 255) / 256;
  return (unsigned)(b > 65536 ? 65536 : b);
}

// ---------------------------------------------------------------------------
// laplacian_add (laplacian.hpp:24-38)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void laplacian_add_kernel(gspace geo, const cplx *__restrict__ ff,
                                                            cplx *__restrict__ out, long ld,
                                                            int nst, long npoint, double factor,
                                                            double c0, double c1, double c2) {
  const long total = npoint * nst;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < total; i += (long)gridDim.x * 256) {
    const long p = i / nst;
    const int b = (int)(i % nst);
    int m0, m1, m2;
    geo.m_of(p, m0, m1, m2);
    const double two_pi = 6.283185307179586476925286766559;
    const double gdot = two_pi * (c0 * m0 + c1 * m1 + c2 * m2);
    const double lapl = factor * (-geo.g2(m0, m1, m2) + gdot);
    const cplx f = ff[p * ld + b];
    cplx o = out[p * ld + b];
    o.x += lapl * f.x;
    o.y += lapl * f.y;
    out[p * ld + b] = o;
  }
}

// ---------------------------------------------------------------------------
// per-band reductions: block (chunk, band group); thread = band x lane
// ---------------------------------------------------------------------------
template <int NV, int BT, class F>
__device__ __forceinline__ void band_partials(long npoint, long chunk, int nst, double *part,
                                              F term) {
  constexpr int LANES = 256 / BT;
  __shared__ double red[4][BT][NV];
  const int bb = threadIdx.x % BT;
  const int lane = threadIdx.x / BT;
  const int b = blockIdx.y * BT + bb;
  const long p0 = (long)blockIdx.x * chunk;
  const long p1 = p0 + chunk < npoint ? p0 + chunk : npoint;
  double acc[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) acc[v] = 0.0;
  if (b < nst)
    for (long p = p0 + lane; p < p1; p += LANES) term(p, b, acc);
  // the lanes of a band within each wave by a butterfly, the waves in order
#pragma unroll
  for (int w = BT; w < 64; w <<= 1)
#pragma unroll
    for (int v = 0; v < NV; v++) acc[v] += __shfl_xor(acc[v], w, 64);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) < BT)
#pragma unroll
    for (int v = 0; v < NV; v++) red[wave][bb][v] = acc[v];
  __syncthreads();
  if (threadIdx.x < BT && b < nst) {
#pragma unroll
    for (int v = 0; v < NV; v++) {
      double s = red[0][bb][v];
      for (int l = 1; l < 4; l++) s += red[l][bb][v];
      part[((long)blockIdx.x * nst + b) * 8 + v] = s;
    }
  }
}

// pass 1: eig = sum conj(hphi) phi, norm = sum |phi|^2
template <int BT>
__global__ __launch_bounds__(256) void eig_norm_partial(const cplx *__restrict__ hphi, long hld,
                                                        const cplx *__restrict__ phi, long ld,
                                                        int nst, long npoint, long chunk, double *part) {
  band_partials<3, BT>(npoint, chunk, nst, part, [&](long p, int b, double *a) {
    const cplx h = hphi[p * hld + b], f = phi[p * ld + b];
    a[0] += h.x * f.x + h.y * f.y;
    a[1] += h.x * f.y - h.y * f.x;
    a[2] += f.x * f.x + f.y * f.y;
  });
}

// pass 2: residual = hphi - evn phi (shift.hpp:19-31 with factor -1), and
// the preconditioner's sums 1/2|G|^2 |r|^2, |r|^2 (preconditioner.hpp:42)
template <int BT>
__global__ __launch_bounds__(256) void residual_partial(gspace geo, const cplx *__restrict__ hphi,
                                                        long hld, const cplx *__restrict__ phi,
                                                        long ld, cplx *__restrict__ res, long rld,
                                                        const double *__restrict__ band, int nst,
                                                        long npoint, long chunk, double *part) {
  band_partials<2, BT>(npoint, chunk, nst, part, [&](long p, int b, double *a) {
    const double er = band[b * 16 + 3], ei = band[b * 16 + 4];  // evn
    const cplx h = hphi[p * hld + b], f = phi[p * ld + b];
    cplx r;
    r.x = h.x + (-1.0) * (er * f.x - ei * f.y);
    r.y = h.y + (-1.0) * (er * f.y + ei * f.x);
    res[p * rld + b] = r;
    int m0, m1, m2;
    geo.m_of(p, m0, m1, m2);
    const double lap = -0.5 * (-geo.g2(m0, m1, m2));
    const double r2 = r.x * r.x + r.y * r.y;
    a[0] += lap * r2;
    a[1] += r2;
  });
}

// pass 4: m0 = <r|r>, m1 = <phi|r>, m2 = <r|Hr>, m3 = <phi|Hr>
template <int BT>
__global__ __launch_bounds__(256) void mm_partial(const cplx *__restrict__ phi, long ld,
                                                  const cplx *__restrict__ res,
                                                  const cplx *__restrict__ hres, long rld, int nst,
                                                  long npoint, long chunk, double *part) {
  band_partials<8, BT>(npoint, chunk, nst, part, [&](long p, int b, double *a) {
    line_sums(a, phi[p * ld + b], res[p * rld + b], hres[p * rld + b]);
  });
}

// Sums of the NV partials of band b over all point chunks, by one 256-thread
// workgroup (strided over chunks, then a tree in LDS: a fixed order).
// Thread 0 gets the totals in `out`.
template <int NV>
__device__ __forceinline__ void band_sums(const double *part, long nchunk, int nst, int b,
                                          double *out) {
  __shared__ double red[256][NV];
  double acc[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) acc[v] = 0.0;
  for (long c = threadIdx.x; c < nchunk; c += 256)
#pragma unroll
    for (int v = 0; v < NV; v++) acc[v] += part[(c * nst + b) * 8 + v];
#pragma unroll
  for (int v = 0; v < NV; v++) red[threadIdx.x][v] = acc[v];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
#pragma unroll
      for (int v = 0; v < NV; v++) red[threadIdx.x][v] += red[threadIdx.x + w][v];
    __syncthreads();
  }
  if (threadIdx.x == 0)
#pragma unroll
    for (int v = 0; v < NV; v++) out[v] = red[0][v];
}

// band record: [0..1] eig, [2] norm, [3..4] eig/norm, [5] kinetic, [6] lambda
// (one workgroup of 256 threads per band)
__global__ __launch_bounds__(256) void eig_norm_final(const double *part, long nchunk, int nst,
                                                      double dV, double *band) {
  const int b = blockIdx.x;
  double t[3];
  band_sums<3>(part, nchunk, nst, b, t);
  if (threadIdx.x != 0) return;
  const double er = dV * t[0], ei = dV * t[1], nn = dV * t[2];
  band[b * 16 + 0] = er;
  band[b * 16 + 1] = ei;
  band[b * 16 + 2] = nn;
  band[b * 16 + 3] = er / nn;
  band[b * 16 + 4] = ei / nn;
}

__global__ __launch_bounds__(256) void kinetic_final(const double *part, long nchunk, int nst,
                                                     double *band) {
  const int b = blockIdx.x;
  double t[2];
  band_sums<2>(part, nchunk, nst, b, t);
  // overlap_diagonal_normalized: the volume element cancels
  if (threadIdx.x == 0) band[b * 16 + 5] = t[0] / t[1];
}

// lambda (steepest_descent.hpp:56-68), and the eig and norm of phi + lambda r from
// those of phi and the same sums: <r|H phi> = conj(<phi|H r>), lambda is real
__global__ __launch_bounds__(256) void lambda_final(const double *part, long nchunk, int nst,
                                                    double dV, double *band) {
  const int b = blockIdx.x;
  double t[8];
  band_sums<8>(part, nchunk, nst, b, t);
  if (threadIdx.x != 0) return;
  // m0 = <r|r>, m1 = <phi|r>, m2 = <r|Hr>, m3 = <phi|Hr>, m4 = eig, m5 = norm
  double m[8];
  for (int v = 0; v < 8; v++) m[v] = dV * t[v];
  const double m4r = band[b * 16 + 0], m4i = band[b * 16 + 1], m5r = band[b * 16 + 2];
  // real parts of the complex products
  auto re = [](double ar, double ai, double br, double bi) { return ar * br - ai * bi; };
  const double ca = re(m[0], m[1], m[6], m[7]) - re(m[4], m[5], m[2], m[3]);
  const double cb = re(m5r, 0.0, m[4], m[5]) - re(m4r, m4i, m[0], m[1]);
  const double cc = re(m4r, m4i, m[2], m[3]) - re(m[6], m[7], m5r, 0.0);
  const double den = cb + sqrt(cb * cb - 4.0 * ca * cc);
  const double lam = fabs(den) < 1e-15 ? 0.0 : 2.0 * cc / den;
  band[b * 16 + 6] = lam;
  const double er = m4r + lam * (2.0 * m[6] + lam * m[4]), ei = m4i - lam * lam * m[5];
  const double nn = m5r + lam * (2.0 * m[2] + lam * m[0]);
  band[b * 16 + 0] = er;
  band[b * 16 + 1] = ei;
  band[b * 16 + 2] = nn;
  band[b * 16 + 3] = er / nn;
  band[b * 16 + 4] = ei / nn;
}

// pass 3: phi(G) *= K(1/2 |G|^2 / kinetic_b) (preconditioner.hpp:45-52).
// A wave takes one grid point at a time, its lanes the bands: the point's
// G vector is worked out once per point (the index divisions of a flat
// per-element loop cost more than the memory traffic).
constexpr int PRECOND_POINT_WAVES = 65536;  // waves of the grid-stride loop at most

__global__ __launch_bounds__(256) void precondition_kernel(gspace geo, cplx *__restrict__ phi,
                                                           long ld, int nst, long npoint,
                                                           const double *__restrict__ band) {
  const int lane = threadIdx.x & 63;
  const long nwaves = (long)gridDim.x * 4;
  for (long p = ((long)blockIdx.x * 256 + threadIdx.x) >> 6; p < npoint; p += nwaves) {
    int m0, m1, m2;
    geo.m_of(p, m0, m1, m2);
    const double g2 = geo.g2(m0, m1, m2);
    // four bands per lane in flight (a band past nst reads the lane's first
    // band and is not stored)
    for (int b0 = lane; b0 < nst; b0 += 256) {
      cplx f[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int b = b0 + 64 * j;
        f[j] = phi[p * ld + (b < nst ? b : b0)];
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int b = b0 + 64 * j;
        if (b < nst) {
          const double k = tpa_k(-0.5 * (-g2) / band[b * 16 + 5]);
          phi[p * ld + b] = mk(f[j].x * k, f[j].y * k);
        }
      }
    }
  }
}

// pass 5 (steepest_descent.hpp:70-77) of the last step, which leaves hphi:
// phi += lambda r over the grid of the partial-sum passes (point chunk x
// band group; the lanes of a point chunk stride its points)
template <int BT>
__global__ __launch_bounds__(256) void sd_update_phi(cplx *__restrict__ phi, long ld,
                                                     const cplx *__restrict__ res, long rld,
                                                     int nst, long npoint, long chunk,
                                                     const double *__restrict__ band) {
  const int bb = threadIdx.x % BT;
  const int lane = threadIdx.x / BT;
  const int b = blockIdx.y * BT + bb;
  if (b >= nst) return;
  const long p0 = (long)blockIdx.x * chunk;
  const long p1 = p0 + chunk < npoint ? p0 + chunk : npoint;
  const double lam = band[b * 16 + 6];
  for (long p = p0 + lane; p < p1; p += 256 / BT) {
    cplx f = phi[p * ld + b];
    const cplx r = res[p * rld + b];
    f.x += lam * r.x;
    f.y += lam * r.y;
    phi[p * ld + b] = f;
  }
}

// pass 5 of a step fused with pass 2 of the next: the residual of the updated phi
// and hphi over the old one.  Seven arrays move instead of the nine of an update
// with the sums of eig and norm and a residual pass after it: steepest descent at
// 40^3 x 48 bands 1535 -> 1479 us, at 64^3 x 256 with the diagonalisation 49.5 ->
// 48.0 ms.
template <int BT>
__global__ __launch_bounds__(256) void sd_update_residual(gspace geo, cplx *__restrict__ phi,
                                                          long ld, cplx *__restrict__ res,
                                                          cplx *__restrict__ hphi,
                                                          const cplx *__restrict__ hres, long rld,
                                                          int nst, long npoint,
                                                          const double *__restrict__ band,
                                                          long chunk, double *part) {
  band_partials<2, BT>(npoint, chunk, nst, part, [&](long p, int b, double *a) {
    const double er = band[b * 16 + 3], ei = band[b * 16 + 4], lam = band[b * 16 + 6];
    cplx f = phi[p * ld + b];
    cplx r = res[p * rld + b];
    cplx h = hphi[p * rld + b];
    const cplx hr = hres[p * rld + b];
    f.x += lam * r.x;
    f.y += lam * r.y;
    h.x += lam * hr.x;
    h.y += lam * hr.y;
    phi[p * ld + b] = f;
    hphi[p * rld + b] = h;
    r.x = h.x + (-1.0) * (er * f.x - ei * f.y);
    r.y = h.y + (-1.0) * (er * f.y + ei * f.x);
    res[p * rld + b] = r;
    int m0, m1, m2;
    geo.m_of(p, m0, m1, m2);
    const double lap = -0.5 * (-geo.g2(m0, m1, m2));
    const double r2 = r.x * r.x + r.y * r.y;
    a[0] += lap * r2;
    a[1] += r2;
  });
}

// Launches a reduction kernel in the shape of nst bands
#define GS_REDUCE(kernel, g, stream, ...)                                                  \
  do {                                                                                     \
    const dim3 grid_((unsigned)(g).nchunk, (unsigned)(g).groups);                          \
    if ((g).bt == 64)                                                                      \
      hipLaunchKernelGGL(kernel<64>, grid_, dim3(256), 0, stream, __VA_ARGS__);            \
    else                                                                                   \
      hipLaunchKernelGGL(kernel<16>, grid_, dim3(256), 0, stream, __VA_ARGS__);            \
    check_launch();                                                                        \
  } while (0)

void check_launch() { INQAMD_HIP_CHECK(hipGetLastError()); }

// Row-major Hermitian M[r][c] = alpha sum_p conj(A[p][r]) B[p][c] over all grid
// points (operations::overlap, overlap.hpp:26-60).  Uses hn2.
void inner_products(handle &h, const cplx *A, long lda, const cplx *B, long ldb, int nst,
                    double alpha, cplx *out) {
  ensure_blas(h);
  // (several slices take at most a quarter of hn2)
  cplx *part = gram_slices(h.npoint, nst) > 1 ? h.hn2 : state(h).ip_part;
  gram(A, lda, B, ldb, nst, h.npoint, alpha, part, out, h.stream);
}

// The K(1/2|G|^2/kinetic) scaling of operations::preconditioner for
// fourier_space orbitals (preconditioner.hpp:39-55), given the residual-type
// kinetic sums already in the band records.
void preconditioner_kinetic(handle &h, int nst) {
  gs_state &g = state(h);
  hipLaunchKernelGGL(kinetic_final, dim3(nst), dim3(256), 0, h.stream,
                     (const double *)g.part, shape(h, nst).nchunk, nst, g.band);
  check_launch();
}

void precondition_apply(handle &h, cplx *phi, long ld, int nst) {
  gs_state &g = state(h);
  preconditioner_kinetic(h, nst);
  const long waves = h.npoint < PRECOND_POINT_WAVES ? h.npoint : PRECOND_POINT_WAVES;
  hipLaunchKernelGGL(precondition_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0,
                     h.stream, geometry(h), phi, ld, nst, h.npoint, (const double *)g.band);
  check_launch();
}

// kinetic sums of phi alone (preconditioner.hpp:42) into the partial buffer
template <int BT>
__global__ __launch_bounds__(256) void kinetic_partial(gspace geo, const cplx *__restrict__ phi,
                                                       long ld, int nst, long npoint,
                                                       long chunk, double *part) {
  band_partials<2, BT>(npoint, chunk, nst, part, [&](long p, int b, double *a) {
    const cplx f = phi[p * ld + b];
    int m0, m1, m2;
    geo.m_of(p, m0, m1, m2);
    const double lap = -0.5 * (-geo.g2(m0, m1, m2));
    const double r2 = f.x * f.x + f.y * f.y;
    a[0] += lap * r2;
    a[1] += r2;
  });
}

}  // namespace

static bool gspace_sweeps(const handle &h) {
  static const bool sweeps = [] {
    const char *e = getenv("INQAMD_GSPACE_SWEEPS");
    return !(e && atoi(e) == 0);
  }();
  return h.three_sweep && sweeps;
}

// ks_hamiltonian::operator() on fourier_space orbitals (ks_hamiltonian.hpp:
// 156-176): to_real, the real-space operator, to_fourier.  Uses hn and hn2.
void hamiltonian_fourier(handle &h, const cplx *phi, long ld, cplx *hphi, long hld, int nst) {
  if (gspace_sweeps(h)) {
    hamiltonian_fourier_sweeps(h, phi, ld, hphi, hld, nst);
    return;
  }
  fft3d(h, phi, ld, h.hn, nst, nst, +1, 1.0 / (double)h.npoint);
  hamiltonian_apply(h, h.hn, nst, h.hn2, nst, nst, KA_CURRENT);
  fft3d(h, h.hn2, nst, hphi, hld, nst, -1, 1.0);
}

void preconditioner(handle &h, cplx *phi, long ld, int nst) {
  ensure_reductions(h);
  gs_state &g = state(h);
  const gs_shape rs = shape(h, nst);
  GS_REDUCE(kinetic_partial, rs, h.stream, geometry(h), (const cplx *)phi, ld, nst, h.npoint,
            rs.chunk, g.part);
  precondition_apply(h, phi, ld, nst);
}

// Phi <- Phi T (row-major T, `upper` triangular with zeros below): out[p][j] =
// sum_i phi[p][i] T[i][j].  Bands beyond LDS go through a ZGEMM into hn, as the
// column-major out^T = T_cm * Phi^T.
static void rotate_bands(handle &h, cplx *phi, long ld, int nst, bool upper) {
  gs_state &g = state(h);
  if (rotate_supported(nst, h.max_lds)) {
    rotate(phi, ld, nst, h.npoint, g.T, upper, h.max_lds, h.stream);
    return;
  }
  const rocblas_double_complex one = {1.0, 0.0}, zero = {0.0, 0.0};
  GS_BLAS_CHECK(rocblas_zgemm(g.blas, rocblas_operation_none, rocblas_operation_none, nst,
                              (rocblas_int)h.npoint, nst, &one,
                              reinterpret_cast<const rocblas_double_complex *>(g.T), nst,
                              reinterpret_cast<const rocblas_double_complex *>(phi), (int)ld,
                              &zero, reinterpret_cast<rocblas_double_complex *>(h.hn), nst));
  copy(h, h.hn, nst, phi, ld, nst);
}

// operations::orthogonalize (orthogonalize.hpp:25-32): S = dV Phi^H Phi,
// S = R R^H (R lower: zpotrf on the row-major S, cholesky.hpp:29-80),
// Phi <- Phi R^-H (invert_triangular + rotate, rotate.hpp:147-156).
void orthogonalize(handle &h, cplx *phi, long ld, int nst, double dV) {
  ensure_blas(h);
  gs_state &g = state(h);
  // S[i][j] = dV sum_p conj(phi_pi) phi_pj, row-major
  inner_products(h, phi, ld, phi, ld, nst, dV, g.S);
  cholesky_rotation(g.S, nst, g.chol, g.T, g.info, h.stream);
  // phi stays as it is where S has no factor
  rocblas_int band = -1;
  INQAMD_HIP_CHECK(
      hipMemcpyAsync(&band, g.info, sizeof(band), hipMemcpyDeviceToHost, h.stream));
  INQAMD_HIP_CHECK(hipStreamSynchronize(h.stream));
  if (band >= 0)
    throw error{ERR_ARGUMENT, "orthogonalize: overlap matrix is not positive definite (band " +
                                  std::to_string(band) + ")"};
  rotate_bands(h, phi, ld, nst, true);
}

// eigensolvers::steepest_descent (steepest_descent.hpp:23-88) on
// fourier_space orbitals with the G-space Hamiltonian.
void steepest_descent(handle &h, cplx *phi, long ld, int nst, bool precond) {
  ensure_workspace(h);
  gs_state &g = state(h);
  const long rl = nst;
  const gs_shape rs = shape(h, nst);
  const long nchunk = rs.nchunk;
  // fourier_space::volume_element (fourier_space.hpp:41-44)
  const double dV = h.volume / ((double)h.npoint * (double)h.npoint);
  const dim3 fg(nst);
  hamiltonian_fourier(h, phi, ld, g.hphi, rl, nst);
  const int num_steps = 5;
  for (int istep = 0; istep < num_steps; istep++) {
    // passes 1 and 2 (after the first step, pass 4's sums and the last update)
    if (istep == 0) {
      GS_REDUCE(eig_norm_partial, rs, h.stream, (const cplx *)g.hphi, rl, (const cplx *)phi, ld,
                nst, h.npoint, rs.chunk, g.part);
      hipLaunchKernelGGL(eig_norm_final, fg, dim3(256), 0, h.stream, (const double *)g.part,
                         nchunk, nst, dV, g.band);
      check_launch();
      GS_REDUCE(residual_partial, rs, h.stream, geometry(h), (const cplx *)g.hphi, rl,
                (const cplx *)phi, ld, g.res, rl, (const double *)g.band, nst, h.npoint, rs.chunk,
                g.part);
    }
    // pass 3, H residual and pass 4: in the first and last of the sweeps where they
    // make H residual
    long mm_rows = nchunk;
    if (gspace_sweeps(h)) {
      fourier_extra e{g.res, nullptr, phi, ld, g.part};
      if (precond) {
        preconditioner_kinetic(h, nst);
        e.kinetic = g.band + 5;
      }
      hamiltonian_fourier_sweeps(h, g.res, rl, g.hres, rl, nst, &e);
      mm_rows = line_sum_rows(h.n[0], h.n[1]);
    } else {
      if (precond) precondition_apply(h, g.res, rl, nst);
      hamiltonian_fourier(h, g.res, rl, g.hres, rl, nst);
      GS_REDUCE(mm_partial, rs, h.stream, (const cplx *)phi, ld, (const cplx *)g.res,
                (const cplx *)g.hres, rl, nst, h.npoint, rs.chunk, g.part);
    }
    hipLaunchKernelGGL(lambda_final, fg, dim3(256), 0, h.stream, (const double *)g.part, mm_rows,
                       nst, dV, g.band);
    check_launch();
    if (istep != num_steps - 1)
      GS_REDUCE(sd_update_residual, rs, h.stream, geometry(h), phi, ld, g.res, g.hphi,
                (const cplx *)g.hres, rl, nst, h.npoint, (const double *)g.band, rs.chunk, g.part);
    else
      GS_REDUCE(sd_update_phi, rs, h.stream, phi, ld, (const cplx *)g.res, rl, nst, h.npoint,
                rs.chunk, (const double *)g.band);
  }
  orthogonalize(h, phi, ld, nst, dV);
}

// ground_state::subspace_diagonalization (subspace_diagonalization.hpp:16-25)
// on real-space orbitals: H_sub = dV Phi^H (H Phi) (overlap.hpp:26-60), its
// eigenpairs (matrix::diagonalize, here rocSOLVER ZHEEVD), Phi <- Phi V
// (rotate, rotate.hpp:63).  Eigenvalues ascending into eig_host.
void subspace_diagonalization(handle &h, cplx *phi, long ld, int nst, double *eig_host) {
  ensure_workspace(h);
  ensure_blas(h);
  gs_state &g = state(h);
  hamiltonian_apply(h, phi, ld, g.hphi, nst, nst, KA_CURRENT);
  // H_sub[r][c] = dV sum_p conj(phi[p][r]) hphi[p][c], row-major (dV = V/N);
  // read as a column-major matrix that is conj(H_sub)
  inner_products(h, phi, ld, g.hphi, nst, nst, h.volume / (double)h.npoint, g.S);
  // eigenvectors w_k of conj(H_sub) are conj(v_k), v_k those of H_sub
  GS_BLAS_CHECK(rocsolver_zheevd(g.blas, rocblas_evect_original, rocblas_fill_upper, nst,
                                 reinterpret_cast<rocblas_double_complex *>(g.S), nst, g.eig,
                                 g.eig + h.max_bands, g.info));
  // out[p][k] = sum_i phi[p][i] v_k[i] = sum_i phi[p][i] conj(W(i, k))
  adjoint_matrix(g.S, nst, g.T, h.stream);
  rotate_bands(h, phi, ld, nst, false);
  rocblas_int info = 0;
  INQAMD_HIP_CHECK(hipMemcpyAsync(eig_host, g.eig, (size_t)nst * sizeof(double),
                                  hipMemcpyDeviceToHost, h.stream));
  INQAMD_HIP_CHECK(hipMemcpyAsync(&info, g.info, sizeof(info), hipMemcpyDeviceToHost, h.stream));
  INQAMD_HIP_CHECK(hipStreamSynchronize(h.stream));
  if (info != 0)
    throw error{ERR_ARGUMENT, "subspace_diagonalization: eigensolver did not converge (info " +
                                  std::to_string(info) + ")"};
}

void gs_release(handle &h) {
  if (!h.gs) return;
  gs_state *g = static_cast<gs_state *>(h.gs);
  for (void *p : {(void *)g->hphi, (void *)g->res, (void *)g->hres, (void *)g->part,
                  (void *)g->band, (void *)g->S, (void *)g->T, (void *)g->chol, (void *)g->eig, (void *)g->info,
                  (void *)g->ip_part})
    if (p) (void)hipFree(p);
  if (g->blas) (void)rocblas_destroy_handle(g->blas);
  delete g;
  h.gs = nullptr;
}

}  // namespace inqamd

using namespace inqamd;

extern "C" {

int inqamd_laplacian_add(inqamd_hamiltonian_t h, const void *ff, void *laplff, int nst, int ld,
                         double factor, const double gradcoeff_contra[3]) {
  if (!h) return INQAMD_ERR_ARGUMENT;
  return guarded(h, [&] {
    check_orbital(*h, ff, "ff");
    check_orbital(*h, laplff, "laplff");
    check_bands(*h, nst, ld, false);
    INQAMD_REQUIRE(gradcoeff_contra, "gradcoeff is null");
    hipLaunchKernelGGL(laplacian_add_kernel, dim3(grid1(h->npoint * nst)), dim3(256), 0,
                       h->stream, geometry(*h), (const cplx *)ff, (cplx *)laplff, (long)ld, nst,
                       h->npoint, factor, gradcoeff_contra[0], gradcoeff_contra[1],
                       gradcoeff_contra[2]);
    check_launch();
  });
}

int inqamd_preconditioner(inqamd_hamiltonian_t h, void *phi, int nst, int ld) {
  if (!h) return INQAMD_ERR_ARGUMENT;
  return guarded(h, [&] {
    check_orbital(*h, phi, "phi");
    check_bands(*h, nst, ld, true);
    preconditioner(*h, (cplx *)phi, ld, nst);
  });
}

int inqamd_orthogonalize(inqamd_hamiltonian_t h, void *phi, int nst, int ld, int fourier) {
  if (!h) return INQAMD_ERR_ARGUMENT;
  return guarded(h, [&] {
    check_orbital(*h, phi, "phi");
    check_bands(*h, nst, ld, true);
    // real_space::volume_element V/N, fourier_space::volume_element V/N^2
    // (real_space.hpp:150-152, fourier_space.hpp:41-44)
    const double dV = fourier ? h->volume / ((double)h->npoint * (double)h->npoint)
                              : h->volume / (double)h->npoint;
    orthogonalize(*h, (cplx *)phi, ld, nst, dV);
  });
}

int inqamd_subspace_diagonalization(inqamd_hamiltonian_t h, void *phi, int nst, int ld,
                                    double *eigenvalues) {
  if (!h) return INQAMD_ERR_ARGUMENT;
  return guarded(h, [&] {
    check_orbital(*h, phi, "phi");
    check_bands(*h, nst, ld, true);
    INQAMD_REQUIRE(eigenvalues, "eigenvalues is null");
    subspace_diagonalization(*h, (cplx *)phi, ld, nst, eigenvalues);
  });
}

int inqamd_steepest_descent(inqamd_hamiltonian_t h, void *phi, int nst, int ld, int precondition) {
  if (!h) return INQAMD_ERR_ARGUMENT;
  return guarded(h, [&] {
    check_orbital(*h, phi, "phi");
    check_bands(*h, nst, ld, true);
    steepest_descent(*h, (cplx *)phi, ld, nst, precondition != 0);
  });
}

}  // extern "C"
