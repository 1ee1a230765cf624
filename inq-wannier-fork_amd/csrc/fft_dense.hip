// Pencil passes of the lengths without a butterfly plan (fft_plan.hip): the
// transform as a product with the DFT matrix on the FP64 matrix cores.
//
// With h = floor(L/2), u_n = x_n + x_{L-n} and d_n = x_n - x_{L-n} (u_0 = x_0,
// and u_h = x_h where L is even; their d are 0),
//   P_k = sum_{n <= h} cos(2 pi k n / L) u_n,  Q_k = sum_{n <= h} sin(2 pi k n / L) d_n
//   y_k = P_k + i sign Q_k,  y_{L-k} = P_k - i sign Q_k,   k <= h,
// so two real (h+1) x (h+1) matrices on complex columns replace the complex
// L x L one: a quarter of its multiply-adds.  A workgroup takes 16 columns (one
// per (pencil, band), as in fft_plan.hip) and one wave each block of 16 rows k;
// v_mfma_f64_16x16x4f64 has rows k, depth four n, columns the 16 columns, and
// four of them per step (P and Q, real and imaginary parts).  The wave that
// holds y_k holds y_{L-k} too, so the kinetic pass forms the inverse's u and d
// in registers.
//
// At L = 67 a tile's 108 matrix instructions take about 1700 cycles of its CU
// against about 4200 for its 34 KB of memory traffic; the work grows with L^2
// and meets the traffic near 192.  Before, such lengths ran O(p^2) butterflies
// for every prime p > 5 from LDS, with a table lookup and an integer modulo per
// product.  Both transforms of 67 x 61 x 53 x 9 bands 23.4 ms -> 112 us (3.3
// TB/s over six passes), of 44 x 46 x 52 x 30 1329 -> 161 us, of 33 x 65 x 71 x
// 40 12.5 ms -> 277 us; errors against 64-bit references as before (1.2e-15,
// 7.8e-16, 7.9e-16).
#include "fft_dense.hpp"

namespace inqamd {

// LDS: U and D [hp][16], the table [L]
template <int MODE>
__global__ __launch_bounds__(384) void fft_dense_kernel(const fft_pass_args a) {
  extern __shared__ cplx lds[];
  const int L = a.len, h = L / 2, hp = dense_rows(L);
  cplx *U = lds, *D = lds + hp * DENSE_B, *tw = lds + 2 * hp * DENSE_B;

  const unsigned ncol = (unsigned)a.nst * (unsigned)a.c1 * (unsigned)a.c2;
  const unsigned g = blockIdx.x * DENSE_B + threadIdx.x % DENSE_B;
  const bool ok = g < ncol;
  const unsigned q = (ok ? g : 0) / (unsigned)a.nst;
  const int b = (int)((ok ? g : 0) - q * (unsigned)a.nst);
  const int o2 = (int)(q / (unsigned)a.c1);
  const int o1 = (int)(q - (unsigned)o2 * (unsigned)a.c1);
  const long base = o1 * a.s1 + o2 * a.s2;
  const cplx *in = a.in + base * a.in_ld + b;
  cplx *out = a.out + base * a.out_ld + b;
  const long istep = a.stride * a.in_ld, ostep = a.stride * a.out_ld;

  for (int i = threadIdx.x; i < L; i += blockDim.x) tw[i] = a.tw[i];
  const int nstep = blockDim.x / DENSE_B, c = threadIdx.x % DENSE_B;
  for (int n = threadIdx.x / DENSE_B; n < hp; n += nstep) {
    cplx u = mk(0.0, 0.0), d = u;
    if (n <= h) {
      const int m = n == 0 ? 0 : L - n;
      const cplx x = in[n * istep], y = in[m * istep];
      const bool pair = m != n;
      u = pair ? cadd(x, y) : x;
      d = pair ? csub(x, y) : d;
    }
    U[n * DENSE_B + c] = u;
    D[n * DENSE_B + c] = d;
  }
  __syncthreads();

  // this lane's outputs: rows k(v) and L - k(v), column lane % 16 = c
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int k0 = 16 * wave + (lane >> 4);

  cplx pre[4][2];
  if constexpr (MODE == FFT_EPILOGUE) {
    // V psi of the outputs, loaded before the product (rows past h load row 0)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int k = k0 + 4 * v;
      const int lo = k <= h ? k : 0, hi = lo ? L - lo : 0;
      const long p0 = base + (long)lo * a.stride, p1 = base + (long)hi * a.stride;
      pre[v][0] = cscale(a.V[p0], a.psi[p0 * a.psi_ld + b]);
      pre[v][1] = cscale(a.V[p1], a.psi[p1 * a.psi_ld + b]);
    }
  }

  dense_acc acc = dense_product(U, D, tw, L, hp);
  int sign = a.sign;
  if constexpr (MODE == FFT_KINETIC) {
    const double inv2pi = 0.15915494309189533576888376337251;
    const int m1 = symmetric_index(o1, a.n[a.ax1]);
    const int m2 = symmetric_index(o2, a.n[a.ax2]);
    double gfix[3], bax[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const double kc = (a.rlat[0 * 3 + d] * a.kA[0] + a.rlat[1 * 3 + d] * a.kA[1] +
                         a.rlat[2 * 3 + d] * a.kA[2]) * inv2pi;
      gfix[d] = m1 * a.rlat[a.ax1 * 3 + d] + m2 * a.rlat[a.ax2 * 3 + d] + kc;
      bax[d] = a.rlat[a.ax * 3 + d];
    }
    auto kin = [&](int i, cplx v) {
      const int m = symmetric_index(i, L);
      const double q0 = m * bax[0] + gfix[0], q1 = m * bax[1] + gfix[1], q2 = m * bax[2] + gfix[2];
      return cscale(0.5 * (q0 * q0 + q1 * q1 + q2 * q2), v);
    };
    __syncthreads();  // every wave has read U and D
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int k = k0 + 4 * v;
      if (k <= h) {  // (rows past h stay zero)
        cplx lo, hi;
        dense_pair(acc, v, -1, lo, hi);
        const bool pair = k != 0 && L - k != k;
        lo = kin(k, lo);
        hi = pair ? kin(L - k, hi) : mk(0.0, 0.0);
        U[k * DENSE_B + c] = cadd(lo, hi);
        D[k * DENSE_B + c] = pair ? csub(lo, hi) : mk(0.0, 0.0);
      }
    }
    __syncthreads();
    acc = dense_product(U, D, tw, L, hp);
    sign = 1;
  }

  if (!ok) return;
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int k = k0 + 4 * v;
    if (k <= h) {
      cplx lo, hi;
      dense_pair(acc, v, sign, lo, hi);
      lo = cscale(a.scale, lo);
      hi = cscale(a.scale, hi);
      if constexpr (MODE == FFT_EPILOGUE) {
        lo = cadd(lo, pre[v][0]);
        hi = cadd(hi, pre[v][1]);
      }
      out[k * ostep] = lo;
      if (k != 0 && L - k != k) out[(L - k) * ostep] = hi;
    }
  }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
template <int MODE>
static void dense_launch(const fft_pass_args &a, unsigned nblocks, hipStream_t stream) {
  const size_t lds = (size_t)(2 * dense_rows(a.len) * DENSE_B + a.len) * sizeof(cplx);
  hipLaunchKernelGGL(fft_dense_kernel<MODE>, dim3(nblocks), dim3(64 * dense_waves(a.len)), lds,
                     stream, a);
  INQAMD_HIP_CHECK(hipGetLastError());
}

// Up to 128 every length without a plan; up to 191 those that need a butterfly
// of a prime above 5 (the others run the stages of fft.hip, whose work grows
// more slowly than the product's; both transforms of 169 x 182 x 191 take 408 us,
// 311 ms by such butterflies, of 98^3 x 4 bands 211 us and 1248).  191 is the longest whose six waves and
// 52 KB of LDS fit the launch bound and the default LDS limit.
bool fft_dense_launch(const fft_pass_args &a, int mode, hipStream_t stream) {
  if (a.len > DENSE_MAX_LEN) return false;
  if (a.len > 128) {
    bool rough = false;
    for (int s = 0; s < a.nstages; s++) rough = rough || a.radix[s] == 7 || a.radix[s] > 8;
    if (!rough) return false;
  }
  const long ncol = (long)a.nst * a.c1 * a.c2;
  if (ncol > (1L << 31) - DENSE_B) return false;  // columns are numbered in 32 bits
  const unsigned nblocks = (unsigned)((ncol + DENSE_B - 1) / DENSE_B);
  switch (mode) {
    case FFT_PLAIN: dense_launch<FFT_PLAIN>(a, nblocks, stream); return true;
    case FFT_KINETIC: dense_launch<FFT_KINETIC>(a, nblocks, stream); return true;
    case FFT_EPILOGUE: dense_launch<FFT_EPILOGUE>(a, nblocks, stream); return true;
    default: return false;
  }
}

}  // namespace inqamd
