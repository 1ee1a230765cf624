// Plan-specialised register-resident pencil passes.
//
// The first Stockham stage reads HBM into registers, the last stage writes
// registers to HBM, and LDS only exchanges data between stages, in place.  The
// radix sequence is a template parameter, so every stage's span,
// butterfly count and twiddle stride are compile-time constants and a kernel
// holds only the registers its own radices need.  The Hpsi epilogue loads
// the psi and V values of the elements a thread will write before the FFT
// stages start, so their latency overlaps the transform.
//
// A workgroup takes PLAN_B consecutive columns of the pass, a column being one
// (pencil, band) pair numbered pencil * nst + band: band counts that are no
// multiple of the tile leave no idle lanes, and where the rows are compact
// (ld = nst) a tile's accesses along x and y are whole aligned 256-byte runs
// whatever the band count.  Bound by HBM: six passes of 230 MB at 45 x 54 x 80
// x 37 bands take 253 us (5.4 TB/s, where a copy reaches 5.7), against 454 with
// run-time plans for 45 and 54 and tiles of 16 bands (37 of 48 lanes) along
// every axis; 64^3 x 128 1239 -> 1222 us, and one field of 64^3 (nst = 1, 15 of
// 16 lanes idle before) 381 -> 237 us for its Hartree and PBE potentials.
//
// Instantiated for the lengths tabulated below; the others (98 and 105 among them)
// go to fft_dense.hip and fft.hip.

#include "fft.hpp"
#include "fft_dft.hpp"
#include "fft_stage.hpp"

namespace inqamd {

constexpr int PLAN_B = 16;

template <int MODE, int R0, int R1, int R2>
__global__ __launch_bounds__(plan_threads(R0 * R1 * R2, PLAN_B)) void fft_plan_kernel(
    const fft_pass_args a) {
  using P = plan3<R0, R1, R2>;
  constexpr int B = PLAN_B;
  constexpr int LEN = P::LEN;
  constexpr int NT = plan_threads(LEN, B);
  constexpr int RL = P::NSTAGE == 1 ? R0 : (P::NSTAGE == 2 ? R1 : R2);  // last radix
  constexpr int NBL = LEN / RL;
  constexpr int NBFL = (NBL * B + NT - 1) / NT;
  static_assert(NT % B == 0, "a thread works on one column");
  __shared__ cplx lds[LEN * B];

  // this thread's column; one past the last loads column 0 and stores nothing
  const unsigned ncol = (unsigned)a.nst * (unsigned)a.c1 * (unsigned)a.c2;
  const unsigned g = blockIdx.x * B + threadIdx.x % B;
  const bool ok = g < ncol;
  const unsigned q = (ok ? g : 0) / (unsigned)a.nst;
  const int b = (int)((ok ? g : 0) - q * (unsigned)a.nst);
  const int o2 = (int)(q / (unsigned)a.c1);
  const int o1 = (int)(q - (unsigned)o2 * (unsigned)a.c1);
  const long base = o1 * a.s1 + o2 * a.s2;
  const cplx *in = a.in + base * a.in_ld + b;
  cplx *out = a.out + base * a.out_ld + b;
  const long istep = a.stride * a.in_ld, ostep = a.stride * a.out_ld;

  auto gl = [&](int i, int) -> cplx { return in[i * istep]; };
  auto ll = [&](int i, int bb) -> cplx { return lds[i * B + bb]; };
  auto ls = [&](int i, int bb, cplx v, int, int) { lds[i * B + bb] = v; };

  if constexpr (MODE == FFT_EPILOGUE) {
    // prefetch V psi for the outputs of the last stage: thread element
    // (q, r) is pencil point j + r*NBL with j = w / B (span NBL = LEN/RL)
    cplx pre[NBFL][RL];
    const cplx *psi = a.psi + base * a.psi_ld + b;
    const double *V = a.V + base;
#pragma unroll
    for (int q = 0; q < NBFL; q++) {
      const int w = threadIdx.x + q * NT;
      const int j = w / B;
#pragma unroll
      for (int r = 0; r < RL; r++) {
        pre[q][r] = mk(0.0, 0.0);
        if (NBFL * NT == NBL * B || w < NBL * B) {
          const long p = (long)(j + r * NBL) * a.stride;
          pre[q][r] = cscale(V[p], psi[p * a.psi_ld]);
        }
      }
    }
    // the last stage stores butterfly slot (q, r) at pencil point j + r*NBL,
    // the point whose V psi was prefetched into pre[q][r]
    auto gs = [&](int i, int, cplx v, int q, int r) {
      if (ok) out[i * ostep] = cadd(cscale(a.scale, v), pre[q][r]);
    };
    run_plan<P, R0, R1, R2, B, NT>(a.tw, a.sign, false, gl, ll, ls, gs, false);
  } else {
    auto gs = [&](int i, int, cplx v, int, int) {
      if (ok) out[i * ostep] = cscale(a.scale, v);
    };
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
      auto ks = [&](int i, int bb, cplx v, int, int) {
        const int m = symmetric_index(i, LEN);
        const double q0 = m * bax[0] + gfix[0], q1 = m * bax[1] + gfix[1], q2 = m * bax[2] + gfix[2];
        lds[i * B + bb] = cscale(0.5 * (q0 * q0 + q1 * q1 + q2 * q2), v);
      };
      run_plan<P, R0, R1, R2, B, NT>(a.tw, -1, false, gl, ll, ls, ks, true);
      run_plan<P, R0, R1, R2, B, NT>(a.tw, +1, true, ll, ll, ls, gs, false);
    } else {
      run_plan<P, R0, R1, R2, B, NT>(a.tw, a.sign, false, gl, ll, ls, gs, false);
    }
  }
}

// ---------------------------------------------------------------------------
// host: (length -> radix sequence) table
// ---------------------------------------------------------------------------
template <int MODE, int R0, int R1, int R2>
static void plan_launch(const fft_pass_args &a, unsigned nblocks, hipStream_t stream) {
  constexpr int NT = plan_threads(R0 * R1 * R2, PLAN_B);
  hipLaunchKernelGGL((fft_plan_kernel<MODE, R0, R1, R2>), dim3(nblocks), dim3(NT), 0, stream, a);
  INQAMD_HIP_CHECK(hipGetLastError());
}

// Two stages wherever two butterflies of at most 12 reach the length: every
// further stage is an LDS round trip and two barriers
#define INQAMD_PLAN_TABLE(X) \
  X(8, 8, 1, 1)              \
  X(9, 3, 3, 1)              \
  X(10, 5, 2, 1)             \
  X(12, 4, 3, 1)             \
  X(14, 7, 2, 1)             \
  X(15, 5, 3, 1)             \
  X(16, 4, 4, 1)             \
  X(18, 6, 3, 1)             \
  X(20, 5, 4, 1)             \
  X(21, 7, 3, 1)             \
  X(24, 6, 4, 1)             \
  X(25, 5, 5, 1)             \
  X(27, 9, 3, 1)             \
  X(28, 7, 4, 1)             \
  X(30, 6, 5, 1)             \
  X(32, 8, 4, 1)             \
  X(35, 7, 5, 1)             \
  X(36, 6, 6, 1)             \
  X(40, 8, 5, 1)             \
  X(42, 7, 6, 1)             \
  X(45, 9, 5, 1)             \
  X(48, 8, 6, 1)             \
  X(49, 7, 7, 1)             \
  X(50, 10, 5, 1)            \
  X(54, 9, 6, 1)             \
  X(56, 8, 7, 1)             \
  X(60, 10, 6, 1)            \
  X(63, 9, 7, 1)             \
  X(64, 8, 8, 1)             \
  X(70, 10, 7, 1)            \
  X(72, 9, 8, 1)             \
  X(75, 5, 5, 3)             \
  X(80, 10, 8, 1)            \
  X(81, 9, 9, 1)             \
  X(84, 12, 7, 1)            \
  X(90, 10, 9, 1)            \
  X(96, 12, 8, 1)            \
  X(100, 10, 10, 1)          \
  X(108, 12, 9, 1)           \
  X(112, 8, 7, 2)            \
  X(120, 12, 10, 1)          \
  X(125, 5, 5, 5)            \
  X(126, 9, 7, 2)            \
  X(128, 8, 4, 4)

template <int MODE>
static bool plan_dispatch(const fft_pass_args &a, unsigned nblocks, hipStream_t stream) {
  switch (a.len) {
#define INQAMD_PLAN_CASE(L, R0, R1, R2) \
  case L: plan_launch<MODE, R0, R1, R2>(a, nblocks, stream); return true;
    INQAMD_PLAN_TABLE(INQAMD_PLAN_CASE)
#undef INQAMD_PLAN_CASE
    default: return false;
  }
}

bool fft_plan_launch(const fft_pass_args &a, int mode, hipStream_t stream) {
  const long ncol = (long)a.nst * a.c1 * a.c2;
  if (ncol > (1L << 31) - PLAN_B) return false;  // columns are numbered in 32 bits
  const unsigned nblocks = (unsigned)((ncol + PLAN_B - 1) / PLAN_B);
  switch (mode) {
    case FFT_PLAIN: return plan_dispatch<FFT_PLAIN>(a, nblocks, stream);
    case FFT_KINETIC: return plan_dispatch<FFT_KINETIC>(a, nblocks, stream);
    case FFT_EPILOGUE: return plan_dispatch<FFT_EPILOGUE>(a, nblocks, stream);
    default: return false;
  }
}

}  // namespace inqamd
