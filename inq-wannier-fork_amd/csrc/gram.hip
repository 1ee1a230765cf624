// Inner products of two sets of bands, M[r][c] = alpha sum_p conj(A[p][r]) B[p][c]
// (operations::overlap, overlap.hpp:26-60), where M is Hermitian: the overlap
// matrix (A = B) and the subspace Hamiltonian (B = H A).
//
// Only the upper triangle is formed, in 16 x 16 tiles of v_mfma_f64_16x16x4f64
// (rows r, depth four points, columns c; four instructions per complex tile).  A
// lane's operand of either side is one band of one point, so a wave's load is
// four runs of 256 contiguous bytes and goes from memory to the instruction
// without LDS.  A wave keeps a block of T x T tiles (the T (T + 1) / 2 of the upper
// triangle where the block is on the diagonal) in registers over its share of the
// points: with T = 4 a step of four points is 64 instructions of 64 cycles on eight
// loads, so one wave per SIMD keeps the matrix core busy; with few bands the
// tiles' registers leave room for more waves and the loads are the bound.  The
// point sum is split over workgroups (gram_slices) and their results are added in
// order.
//
// A strided-batched library product formed the whole square and idled most of its
// 64 x 64 tiles at few bands: 40^3 x 48 bands 118 -> 35 us, 96^3 x 8 1506 -> about
// 65 us; steepest descent there 1623 -> 1534 and 5246 -> 3805 us, at 64^3 x 20
// 3134 -> 2726 us, at 30 x 36 x 40 x 130 3396 -> 3246 us, the ground-state step
// at 64^3 x 256 50.7 -> 49.4 ms.
#include "internal.hpp"
#include "projector_dev.hpp"

namespace inqamd {
namespace {

struct gram_args {
  const cplx *A, *B;
  long lda, ldb;
  int nst;
  long npoint, chunk;  // points per slice
  cplx *part;          // [slice][nst][nst]
  int nblk, npair_off; // blocks of bands; pairs off the diagonal
};

// Rows rb..., columns cb..., points [p0, p1); SAME: A is B
template <int T, bool DIAG, bool SAME>
__device__ __forceinline__ void gram_block(const gram_args &a, int rb, int cb, long p0, long p1,
                                           cplx *part, double (*red)[64][8]) {
  constexpr int NT = DIAG ? T * (T + 1) / 2 : T * T;
  constexpr bool ONE = DIAG && SAME;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = mfma_col_b(lane), k = mfma_k(lane);
  v4d re[NT], im[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) re[t] = im[t] = v4d{0.0, 0.0, 0.0, 0.0};
  // bands past the last read it again; their products are not stored
  const cplx *pa[T], *pb[T];
#pragma unroll
  for (int i = 0; i < T; i++) {
    const int r = rb + 16 * i + col, c = cb + 16 * i + col;
    pa[i] = a.A + (r < a.nst ? r : a.nst - 1);
    pb[i] = a.B + (c < a.nst ? c : a.nst - 1);
  }
  cplx fa[T], fb[T];
  auto load = [&](long p) {  // points past the last are zero
    const long q = p + k;
    const bool in = q < p1;
    const long oa = (in ? q : p1 - 1) * a.lda, ob = (in ? q : p1 - 1) * a.ldb;
#pragma unroll
    for (int i = 0; i < T; i++) {
      fa[i] = pa[i][oa];
      if constexpr (!ONE) fb[i] = pb[i][ob];
    }
    if (!in) {
#pragma unroll
      for (int i = 0; i < T; i++) fa[i] = fb[i] = mk(0.0, 0.0);
    }
  };
  // (uniform over the wave: every lane runs every instruction)
  long p = p0 + 4 * wave;
  if (p < p1) load(p);
  while (p < p1) {
    cplx xa[T], xb[T];
#pragma unroll
    for (int i = 0; i < T; i++) {
      xa[i] = fa[i];
      xb[i] = ONE ? fa[i] : fb[i];
    }
    p += 16;
    if (p < p1) load(p);
#pragma unroll
    for (int h = 0; h < 2; h++) {
      int t = 0;
#pragma unroll
      for (int i = 0; i < T; i++) {
#pragma unroll
        for (int j = DIAG ? i : 0; j < T; j++, t++) {
          re[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(h ? xa[i].y : xa[i].x,
                                                       h ? xb[j].y : xb[j].x, re[t], 0, 0, 0);
          im[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(h ? -xa[i].y : xa[i].x,
                                                       h ? xb[j].x : xb[j].y, im[t], 0, 0, 0);
        }
      }
    }
  }
  // the waves' tiles in wave order
  int t = 0;
#pragma unroll
  for (int i = 0; i < T; i++) {
#pragma unroll
    for (int j = DIAG ? i : 0; j < T; j++, t++) {
      __syncthreads();
#pragma unroll
      for (int v = 0; v < 4; v++) {
        red[wave][lane][v] = re[t][v];
        red[wave][lane][4 + v] = im[t][v];
      }
      __syncthreads();
      // thread: lane layout of element v = wave
      const int r = rb + 16 * i + mfma_row_d(lane, wave), c = cb + 16 * j + mfma_col_d(lane);
      cplx s = mk(0.0, 0.0);
      for (int w = 0; w < 4; w++) s = cadd(s, mk(red[w][lane][wave], red[w][lane][4 + wave]));
      if (r < a.nst && c < a.nst) part[(long)r * a.nst + c] = s;
    }
  }
}

// Workgroup: slice blockIdx.x, pair of band blocks blockIdx.y (those off the
// diagonal, which have more tiles, first).  The pairs of a slice run at about the
// same time on one XCD where gridDim.x is a multiple of 8, and share its loads in
// L2.  OFF: there are pairs off the diagonal (their tiles'
// registers would cost a lone block its other waves).
template <int T, bool SAME, bool OFF>
__global__ __launch_bounds__(256) void gram_kernel(const gram_args a) {
  __shared__ double red[4][64][8];
  const long p0 = (long)blockIdx.x * a.chunk;
  const long p1 = p0 + a.chunk < a.npoint ? p0 + a.chunk : a.npoint;
  cplx *part = a.part + (long)blockIdx.x * a.nst * a.nst;
  const int y = blockIdx.y;
  if (y >= a.npair_off) {
    const int b = (y - a.npair_off) * 16 * T;
    gram_block<T, true, SAME>(a, b, b, p0, p1, part, red);
    return;
  }
  if constexpr (OFF) {
    int i = 0, o = y;
    while (o >= a.nblk - 1 - i) o -= a.nblk - 1 - i++;
    gram_block<T, false, SAME>(a, i * 16 * T, (i + 1 + o) * 16 * T, p0, p1, part, red);
  }
}

// The slices in order, 16 lanes of them per element, and the other triangle
__global__ __launch_bounds__(256) void gram_sum_kernel(const cplx *__restrict__ part, int nslice,
                                                       int nst, double alpha,
                                                       cplx *__restrict__ out) {
  __shared__ cplx red[16][16];
  const int e = threadIdx.x & 15, l = threadIdx.x >> 4;
  const long n = (long)nst * nst, g = (long)blockIdx.x * 16 + e;
  const int r = (int)(g / nst), c = (int)(g % nst);
  const bool ok = g < n && r <= c;
  cplx s = mk(0.0, 0.0);
  if (ok)
    for (int k = l; k < nslice; k += 16) s = cadd(s, part[(long)k * n + g]);
  red[l][e] = s;
  __syncthreads();
  if (l != 0 || !ok) return;
  for (int k = 1; k < 16; k++) s = cadd(s, red[k][e]);
  s = cscale(alpha, s);
  if (r == c) s.y = 0.0;
  out[(long)r * nst + c] = s;
  out[(long)c * nst + r] = mk(s.x, -s.y);
}

template <int T, bool OFF>
void gram_launch(const gram_args &a, unsigned slices, hipStream_t stream) {
  const dim3 grid(slices, (unsigned)(a.npair_off + a.nblk));
  if (a.A == a.B && a.lda == a.ldb)
    hipLaunchKernelGGL((gram_kernel<T, true, OFF>), grid, dim3(256), 0, stream, a);
  else
    hipLaunchKernelGGL((gram_kernel<T, false, OFF>), grid, dim3(256), 0, stream, a);
  INQAMD_HIP_CHECK(hipGetLastError());
}

constexpr int GRAM_BLOCKS = 1024;  // workgroups of a launch, about

}  // namespace

// Slices of the point sum: about GRAM_BLOCKS workgroups over the pairs of band
// blocks, results of at most a quarter of the bands' own size; whole multiples of 8
// where there are that many, any number below (one slice for all of them there took
// 28.7 ms where an orthogonalisation at 48^3 x 961 bands takes 22.4, and 2990 us for
// 1490 at 24^3 x 433)
int gram_slices(long npoint, int nst) {
  const int nblk = (nst + 63) / 64, pairs = nblk * (nblk + 1) / 2;
  long c = GRAM_BLOCKS / pairs;
  if (c > npoint / (4L * nst)) c = npoint / (4L * nst);
  if (c > 512) c = 512;
  if (c >= 8) c = c / 8 * 8;
  return c < 1 ? 1 : (int)c;
}

// part: gram_slices nst^2 values of scratch
void gram(const cplx *A, long lda, const cplx *B, long ldb, int nst, long npoint, double alpha,
          cplx *part, cplx *out, hipStream_t stream) {
  const int slices = gram_slices(npoint, nst);
  gram_args a;
  a.A = A;
  a.B = B;
  a.lda = lda;
  a.ldb = ldb;
  a.nst = nst;
  a.npoint = npoint;
  a.chunk = (npoint + slices - 1) / slices;
  a.part = part;
  a.nblk = (nst + 63) / 64;
  a.npair_off = a.nblk * (a.nblk - 1) / 2;
  const int tiles = (nst + 15) / 16;
  const int T = (tiles + a.nblk - 1) / a.nblk;  // (3 or 4 where there are several blocks)
  if (T == 1)
    gram_launch<1, false>(a, slices, stream);
  else if (T == 2)
    gram_launch<2, false>(a, slices, stream);
  else if (T == 3)
    a.nblk > 1 ? gram_launch<3, true>(a, slices, stream) : gram_launch<3, false>(a, slices, stream);
  else
    a.nblk > 1 ? gram_launch<4, true>(a, slices, stream) : gram_launch<4, false>(a, slices, stream);
  const long n = (long)nst * nst;
  hipLaunchKernelGGL(gram_sum_kernel, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, stream,
                     (const cplx *)part, slices, nst, alpha, out);
  INQAMD_HIP_CHECK(hipGetLastError());
}

}  // namespace inqamd
