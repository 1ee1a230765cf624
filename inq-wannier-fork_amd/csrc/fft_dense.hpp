// The DFT-matrix product of fft_dense.hip on a 16-column tile, shared with the
// field passes (fields.hip).
#pragma once

#include "fft.hpp"
#include "fft_dft.hpp"

namespace inqamd {

constexpr int DENSE_B = 16;
typedef double v4d __attribute__((ext_vector_type(4)));

// Lane layout of v_mfma_f64_16x16x4f64 (see projector_dev.hpp): lane l holds
// A[l % 16][l / 16], B[l / 16][l % 16] and D[4 v + l / 16][l % 16], v = 0..3.
struct dense_acc {
  v4d pr, pi, qr, qi;
};

// P and Q of the wave's rows k = 16 wave + ... over the hp rows (hp a multiple
// of 4, zero beyond h) of U and D
__device__ __forceinline__ dense_acc dense_product(const cplx *U, const cplx *D, const cplx *tw,
                                                   int L, int hp) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int k = 16 * wave + (lane & 15), n0 = lane >> 4, c = lane & 15;
  // table index (k n) mod L, advanced by 4 k mod L per step
  int idx = (int)((unsigned)(k * n0) % (unsigned)L);
  const int inc = (int)((unsigned)(4 * k) % (unsigned)L);
  dense_acc a;
  a.pr = a.pi = a.qr = a.qi = v4d{0.0, 0.0, 0.0, 0.0};
  for (int n = n0; n < hp; n += 4) {
    const cplx w = tw[idx];  // cos - i sin
    const cplx u = U[n * DENSE_B + c], d = D[n * DENSE_B + c];
    a.pr = __builtin_amdgcn_mfma_f64_16x16x4f64(w.x, u.x, a.pr, 0, 0, 0);
    a.pi = __builtin_amdgcn_mfma_f64_16x16x4f64(w.x, u.y, a.pi, 0, 0, 0);
    a.qr = __builtin_amdgcn_mfma_f64_16x16x4f64(-w.y, d.x, a.qr, 0, 0, 0);
    a.qi = __builtin_amdgcn_mfma_f64_16x16x4f64(-w.y, d.y, a.qi, 0, 0, 0);
    idx += inc;
    idx -= idx >= L ? L : 0;
  }
  return a;
}

// y_k and y_{L-k} of accumulator row v: P +- i sign Q
__device__ __forceinline__ void dense_pair(const dense_acc &a, int v, int sign, cplx &lo, cplx &hi) {
  const double s = sign;
  const cplx iq = mk(-s * a.qi[v], s * a.qr[v]);
  lo = mk(a.pr[v] + iq.x, a.pi[v] + iq.y);
  hi = mk(a.pr[v] - iq.x, a.pi[v] - iq.y);
}

__host__ __device__ constexpr int dense_rows(int L) { return (L / 2 + 1 + 3) / 4 * 4; }
constexpr int dense_waves(int L) { return (L / 2 + 1 + 15) / 16; }

// Most lengths whose tiles fit the default LDS limit and 384 threads
constexpr int DENSE_MAX_LEN = 191;

}  // namespace inqamd
