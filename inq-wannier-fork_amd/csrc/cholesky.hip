// Cholesky factor of the overlap matrix and the rotation T = R^-H it gives
// (S = R R^H, R lower; operations::orthogonalize, orthogonalize.hpp:25-32), on
// the device.
//
// Blocks of 32: one launch per block column k updates every trailing block
//   S_ij -= L_ik L_jk^H,  L_ik = S_ik R_kk^-H,   i >= j > k,
// each workgroup forming its own two L blocks (the products are small, a launch
// between them is not), and the workgroup of block (k+1, k+1) factors it and
// inverts the factor before the next launch.  A last launch forms R^-1 by block
// forward substitution, eight columns per workgroup.  Bound by the chain of
// diagonal blocks: 32 steps of one barrier each, n / 32 of them.
//
// On the host (two triple loops with the matrix copied out and back) this left
// the GPU idle for 7.2 ms at 256 bands: a ground-state iteration at 64^3 x 256
// takes 59.8 ms against 67.0.
#include "internal.hpp"

namespace inqamd {

namespace {

constexpr int CH_B = 32;        // block
constexpr int CH_P = CH_B + 1;  // padded row of an LDS block
constexpr int CH_NT = 256;
constexpr int CH_C = 8;         // columns per workgroup of the inverse

// Element (i, j) of the n x n row-major A; the identity beyond its edge
__device__ __forceinline__ cplx padded(const cplx *A, int n, int i, int j) {
  return i < n && j < n ? A[(long)i * n + j] : mk(i == j ? 1.0 : 0.0, 0.0);
}

// out[q][p] = sum_m X[r + 16 q][m] conj(Y[c + 16 p][m]) with r = thread / 16, c =
// thread % 16
__device__ __forceinline__ void block_product(const cplx *X, const cplx *Y, cplx (&out)[2][2]) {
  const int r = threadIdx.x / 16, c = threadIdx.x % 16;
#pragma unroll
  for (int q = 0; q < 2; q++)
#pragma unroll
    for (int p = 0; p < 2; p++) out[q][p] = mk(0.0, 0.0);
#pragma unroll 4
  for (int m = 0; m < CH_B; m++) {
    const cplx x[2] = {X[r * CH_P + m], X[(r + 16) * CH_P + m]};
    const cplx y[2] = {Y[c * CH_P + m], Y[(c + 16) * CH_P + m]};
#pragma unroll
    for (int q = 0; q < 2; q++)
#pragma unroll
      for (int p = 0; p < 2; p++) out[q][p] = cadd(out[q][p], cmulconj(x[q], y[p]));
  }
}

// Calls f(q, p, row, column) for the four elements of block_product's layout
template <class F>
__device__ __forceinline__ void block_each(F f) {
  const int r = threadIdx.x / 16, c = threadIdx.x % 16;
#pragma unroll
  for (int q = 0; q < 2; q++)
#pragma unroll
    for (int p = 0; p < 2; p++) f(q, p, r + 16 * q, c + 16 * p);
}

// Factors the Hermitian block in D (LDS, lower triangle) and inverts the factor
// in W (LDS).  Columns and rows stay unscaled until the end: with d_k the pivot,
// D[i][j] -= D[i][k] conj(D[j][k]) / d_k and W[i] -= D[i][k] W[k] / d_k, so a step
// is one pass and one barrier.  *info gets the first band whose pivot is not
// positive.
__device__ void factor_block(cplx *D, cplx *W, int kb, int n, cplx *L, cplx *inv, int *info) {
  block_each([&](int, int, int i, int j) { W[i * CH_P + j] = mk(i == j ? 1.0 : 0.0, 0.0); });
  __syncthreads();
  for (int k = 0; k < CH_B - 1; k++) {
    const double rd = 1.0 / D[k * CH_P + k].x;
    block_each([&](int, int, int i, int j) {
      if (i > k) {
        const cplx l = cscale(rd, D[i * CH_P + k]);
        if (j > k && j <= i)
          D[i * CH_P + j] = csub(D[i * CH_P + j], cmulconj(l, D[j * CH_P + k]));
        if (j <= k) W[i * CH_P + j] = csub(W[i * CH_P + j], cmul(l, W[k * CH_P + j]));
      }
    });
    __syncthreads();
  }
  if (threadIdx.x == 0 && *info < 0)
    for (int k = 0; k < CH_B; k++)
      if (!(D[k * CH_P + k].x > 0.0)) {
        *info = kb * CH_B + k;
        break;
      }
  block_each([&](int, int, int i, int j) {
    const cplx zero = mk(0.0, 0.0);
    const double ri = 1.0 / sqrt(D[i * CH_P + i].x), dj = D[j * CH_P + j].x;
    inv[i * CH_B + j] = j <= i ? cscale(ri, W[i * CH_P + j]) : zero;
    const int gi = kb * CH_B + i, gj = kb * CH_B + j;
    if (gi < n && gj < n)
      L[(long)gi * n + gj] = j < i ? cscale(1.0 / sqrt(dj), D[i * CH_P + j])
                                   : (j == i ? mk(sqrt(dj), 0.0) : zero);
  });
}

// The first diagonal block
__global__ __launch_bounds__(CH_NT) void cholesky_first_kernel(const cplx *A, int n, cplx *L,
                                                               cplx *inv, int *info) {
  __shared__ cplx D[CH_B * CH_P], W[CH_B * CH_P];
  if (threadIdx.x == 0) *info = -1;
  block_each([&](int, int, int i, int j) { D[i * CH_P + j] = padded(A, n, i, j); });
  __syncthreads();
  factor_block(D, W, 0, n, L, inv, info);
}

// Block column kb done: workgroup t updates trailing block (i, j), i >= j > kb,
// numbered row by row; t = 0 is (kb + 1, kb + 1).  L_ik goes to L (the
// workgroups of a row and a column read S_ik, so it stays in A).
__global__ __launch_bounds__(CH_NT) void cholesky_step_kernel(cplx *A, int n, int kb, cplx *L,
                                                              cplx *inv, int *info) {
  __shared__ cplx X[CH_B * CH_P], Y[CH_B * CH_P], V[CH_B * CH_P];
  int i = 0, t = blockIdx.x;
  while (t > i) t -= ++i;
  const int bi = kb + 1 + i, bj = kb + 1 + t;
  const cplx *ivk = inv + (long)kb * CH_B * CH_B;
  block_each([&](int, int, int r, int c) {
    X[r * CH_P + c] = padded(A, n, bi * CH_B + r, kb * CH_B + c);
    Y[r * CH_P + c] = padded(A, n, bj * CH_B + r, kb * CH_B + c);
    V[r * CH_P + c] = ivk[r * CH_B + c];
  });
  __syncthreads();
  cplx li[2][2], lj[2][2], u[2][2];
  block_product(X, V, li);
  block_product(Y, V, lj);
  __syncthreads();
  block_each([&](int q, int p, int r, int c) {
    X[r * CH_P + c] = li[q][p];
    Y[r * CH_P + c] = lj[q][p];
    if (t == 0 && bi * CH_B + r < n)  // (kb is a whole block: its columns are in range)
      L[(long)(bi * CH_B + r) * n + kb * CH_B + c] = li[q][p];
  });
  __syncthreads();
  block_product(X, Y, u);
  const bool diagonal = blockIdx.x == 0;
  if (diagonal) __syncthreads();  // X becomes the block to factor
  block_each([&](int q, int p, int r, int c) {
    const int gi = bi * CH_B + r, gj = bj * CH_B + c;
    const cplx v = csub(padded(A, n, gi, gj), u[q][p]);
    if (diagonal)
      X[r * CH_P + c] = v;
    else if (gi < n && gj < n)
      A[(long)gi * n + gj] = v;
  });
  if (!diagonal) return;
  __syncthreads();
  factor_block(X, Y, kb + 1, n, L, inv + (long)(kb + 1) * CH_B * CH_B, info);
}

// T = (R^-1)^H for columns [CH_C strip, ...) of block column j of R^-1: block rows
// i = j, j + 1, ...: X_j = R_jj^-1, X_i = -R_ii^-1 sum_{j <= k < i} L_ik X_k.
// R^-1[r][c] is kept as T[c][r] = conj; T is zero below its diagonal.
__global__ __launch_bounds__(CH_NT) void cholesky_inverse_kernel(const cplx *L, const cplx *inv,
                                                                 int n, cplx *T) {
  __shared__ cplx M[CH_B * CH_P], X[CH_B][CH_C + 1];
  const int nblk = (n + CH_B - 1) / CH_B;
  const int j = blockIdx.x / (CH_B / CH_C), c0 = j * CH_B + blockIdx.x % (CH_B / CH_C) * CH_C;
  const int r = threadIdx.x / CH_C, c = threadIdx.x % CH_C, gc = c0 + c;
  // rows above the block column (its own block is written below)
  for (int i = threadIdx.x / CH_C; i < j * CH_B; i += CH_NT / CH_C)
    if (gc < n) T[(long)gc * n + i] = mk(0.0, 0.0);
  for (int i = j; i < nblk; i++) {
    cplx s = mk(0.0, 0.0);
    if (i > j) {
      for (int k = j; k < i; k++) {
        block_each([&](int, int, int a, int b) {
          M[a * CH_P + b] = padded(L, n, i * CH_B + a, k * CH_B + b);
        });
        const cplx x = gc < n && k * CH_B + r < n ? T[(long)gc * n + k * CH_B + r] : mk(0.0, 0.0);
        X[r][c] = mk(x.x, -x.y);
        __syncthreads();
#pragma unroll 4
        for (int m = 0; m < CH_B; m++) s = cadd(s, cmul(M[r * CH_P + m], X[m][c]));
        __syncthreads();
      }
      X[r][c] = mk(-s.x, -s.y);
    } else {
      X[r][c] = mk(j * CH_B + r == gc ? 1.0 : 0.0, 0.0);
    }
    block_each([&](int, int, int a, int b) {
      M[a * CH_P + b] = inv[((long)i * CH_B + a) * CH_B + b];
    });
    __syncthreads();
    s = mk(0.0, 0.0);
#pragma unroll 4
    for (int m = 0; m < CH_B; m++) s = cadd(s, cmul(M[r * CH_P + m], X[m][c]));
    const int gr = i * CH_B + r;
    if (gr < n && gc < n) T[(long)gc * n + gr] = mk(s.x, -s.y);
    __syncthreads();
  }
}

}  // namespace

long cholesky_scratch(int n) {
  return (long)n * n + (long)((n + CH_B - 1) / CH_B) * CH_B * CH_B;
}

// T (row-major, upper triangular) = R^-H of the Hermitian S = R R^H (its lower
// triangle is read, S is overwritten); scratch of cholesky_scratch(n) elements;
// *info (device) = the first band whose pivot is not positive, or -1.
void cholesky_rotation(cplx *S, int n, cplx *scratch, cplx *T, int *info, hipStream_t stream) {
  cplx *L = scratch, *inv = scratch + (long)n * n;
  const int nblk = (n + CH_B - 1) / CH_B;
  hipLaunchKernelGGL(cholesky_first_kernel, dim3(1), dim3(CH_NT), 0, stream, (const cplx *)S, n, L,
                     inv, info);
  INQAMD_HIP_CHECK(hipGetLastError());
  for (int kb = 0; kb + 1 < nblk; kb++) {
    const int m = nblk - kb - 1;
    hipLaunchKernelGGL(cholesky_step_kernel, dim3(m * (m + 1) / 2), dim3(CH_NT), 0, stream, S, n,
                       kb, L, inv, info);
    INQAMD_HIP_CHECK(hipGetLastError());
  }
  hipLaunchKernelGGL(cholesky_inverse_kernel, dim3(nblk * (CH_B / CH_C)), dim3(CH_NT), 0, stream,
                     (const cplx *)L, (const cplx *)inv, n, T);
  INQAMD_HIP_CHECK(hipGetLastError());
}

}  // namespace inqamd
