// phi <- phi M on nst bands, in place (operations::rotate, rotate.hpp:63, 147-156), M
// an nst x nst matrix, upper triangular or full, on v_mfma_f64_16x16x4f64 (rows 16
// points, depth four bands of phi, columns 16 bands of the result; four
// instructions per complex tile).
//
// A workgroup holds its points' rows in LDS and writes the results over them, so
// phi is read and written once: the library's product went to another array and
// was copied back (steepest descent at 40^3 x 48 bands 1475 -> 1432 us, at 30 x 36 x
// 40 x 130 3089 -> 2991 us, at 64^3 x 256 with the diagonalisation 47.99 -> 47.71 ms).  LDS rows are an odd number of 16-byte slots apart, which
// spreads the 16 points of an operand over the banks; M's operand is 16 contiguous
// bands of four rows, from L2.  A wave takes RT row tiles and one column tile at
// a time, up to the last row that the triangle has in that column.
//   up to 64 bands: 64 points, four waves of one row tile each through all the
//     column tiles (66 KB at most: two workgroups per CU; bound by memory)
//   above, while 32 rows fit in LDS: 32 points, two row tiles per wave, so that
//     M comes from L2 at 8 B per cycle and CU; eight waves take the column tiles
//     from both ends in turn (equal work in a triangle)
//   above: 16 points
#include "internal.hpp"
#include "projector_dev.hpp"

namespace inqamd {
namespace {

constexpr int rotate_stride(int nst) { return (nst + 3) / 4 * 4 + 1; }

template <int RT, int RG, int NW, bool TRI>
__global__ __launch_bounds__(64 * NW) void rotate_kernel(cplx *phi, long ld, int nst, long npoint,
                                                         const cplx *__restrict__ M) {
  constexpr int P = 16 * RT * RG;  // points
  constexpr int RW = P / NW;       // rows a wave loads
  static_assert(NW % RG == 0 && P % NW == 0, "whole rows and row groups per wave");
  extern __shared__ cplx lds[];
  const int stride = rotate_stride(nst);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long p0 = (long)blockIdx.x * P;
  // rows past the grid and bands up to a multiple of four are zero
  for (int b = lane; b < stride - 1; b += 64) {
    cplx v[RW];
#pragma unroll
    for (int r = 0; r < RW; r++) {
      const long p = p0 + wave + r * NW;
      v[r] = p < npoint && b < nst ? phi[p * ld + b] : mk(0.0, 0.0);
    }
#pragma unroll
    for (int r = 0; r < RW; r++) lds[(wave + r * NW) * stride + b] = v[r];
  }
  __syncthreads();

  const int nct = (nst + 15) / 16;
  const int col = mfma_col_b(lane), k = mfma_k(lane);
  constexpr int WG = NW / RG;  // waves of a row group
  const int rg = wave % RG, w = wave / RG;
  const cplx *row = lds + (long)(rg * RT * 16 + mfma_row_a(lane)) * stride + k;
  for (int t = 0; t * WG < nct; t++) {
    const int ct = t * WG + (t & 1 ? WG - 1 - w : w);
    if (ct >= nct) continue;
    const int c = 16 * ct + col;
    const int kend = TRI && 16 * ct + 16 < nst ? 16 * ct + 16 : nst;
    const cplx *m = M + (c < nst ? c : nst - 1);
    auto load = [&](int i) {
      const cplx v = m[(long)(i + k < nst ? i + k : nst - 1) * nst];
      return i + k < nst ? v : mk(0.0, 0.0);
    };
    v4d re[RT], im[RT];
#pragma unroll
    for (int q = 0; q < RT; q++) re[q] = im[q] = v4d{0.0, 0.0, 0.0, 0.0};
    constexpr int U = 4;  // steps whose operands of M are loaded ahead
    cplx ring[U];
#pragma unroll
    for (int u = 0; u < U; u++) ring[u] = load(4 * u);
    // (every lane runs every instruction; the loop's bounds are the wave's)
    for (int i0 = 0; i0 < kend; i0 += 4 * U) {
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int i = i0 + 4 * u;
        if (i < kend) {
          const cplx b = ring[u];
          ring[u] = load(i + 4 * U);
          cplx a[RT];
#pragma unroll
          for (int q = 0; q < RT; q++) a[q] = row[(long)q * 16 * stride + i];
#pragma unroll
          for (int q = 0; q < RT; q++) {
            re[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q].x, b.x, re[q], 0, 0, 0);
            im[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q].x, b.y, im[q], 0, 0, 0);
          }
#pragma unroll
          for (int q = 0; q < RT; q++) {
            re[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[q].y, b.y, re[q], 0, 0, 0);
            im[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q].y, b.x, im[q], 0, 0, 0);
          }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < RT; q++) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const long p = p0 + (rg * RT + q) * 16 + mfma_row_d(lane, v);
        if (p < npoint && c < nst) phi[p * ld + c] = mk(re[q][v], im[q][v]);
      }
    }
  }
}

// out[i][k] = conj(W[k][i]) (row-major)
__global__ __launch_bounds__(256) void adjoint_kernel(const cplx *__restrict__ W, int n,
                                                      cplx *__restrict__ out) {
  const long e = blockIdx.x * 256L + threadIdx.x;
  if (e >= (long)n * n) return;
  const int i = (int)(e / n), k = (int)(e % n);
  const cplx v = W[(long)k * n + i];
  out[e] = mk(v.x, -v.y);
}

template <int RT, int RG, int NW>
void rotate_launch(cplx *phi, long ld, int nst, long npoint, const cplx *M, bool tri,
                   hipStream_t stream) {
  constexpr int P = 16 * RT * RG;
  const size_t lds = (size_t)P * rotate_stride(nst) * sizeof(cplx);
  const dim3 grid((unsigned)((npoint + P - 1) / P));
  if (tri)
    hipLaunchKernelGGL((rotate_kernel<RT, RG, NW, true>), grid, dim3(64 * NW), lds, stream, phi,
                       ld, nst, npoint, M);
  else
    hipLaunchKernelGGL((rotate_kernel<RT, RG, NW, false>), grid, dim3(64 * NW), lds, stream, phi,
                       ld, nst, npoint, M);
  INQAMD_HIP_CHECK(hipGetLastError());
}

}  // namespace

void rotate_prepare() {
  for (const void *k : {(const void *)rotate_kernel<1, 4, 4, true>,
                        (const void *)rotate_kernel<1, 4, 4, false>,
                        (const void *)rotate_kernel<2, 1, 8, true>,
                        (const void *)rotate_kernel<2, 1, 8, false>,
                        (const void *)rotate_kernel<1, 1, 8, true>,
                        (const void *)rotate_kernel<1, 1, 8, false>})
    INQAMD_HIP_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
}

bool rotate_supported(int nst, size_t max_lds) {
  return (size_t)16 * rotate_stride(nst) * sizeof(cplx) <= max_lds;
}

void rotate(cplx *phi, long ld, int nst, long npoint, const cplx *M, bool upper, size_t max_lds,
            hipStream_t stream) {
  if (nst <= 64)
    rotate_launch<1, 4, 4>(phi, ld, nst, npoint, M, upper, stream);
  else if ((size_t)32 * rotate_stride(nst) * sizeof(cplx) <= max_lds)
    rotate_launch<2, 1, 8>(phi, ld, nst, npoint, M, upper, stream);
  else
    rotate_launch<1, 1, 8>(phi, ld, nst, npoint, M, upper, stream);
}

void adjoint_matrix(const cplx *W, int n, cplx *out, hipStream_t stream) {
  hipLaunchKernelGGL(adjoint_kernel, dim3((unsigned)(((long)n * n + 255) / 256)), dim3(256), 0,
                     stream, W, n, out);
  INQAMD_HIP_CHECK(hipGetLastError());
}

}  // namespace inqamd
