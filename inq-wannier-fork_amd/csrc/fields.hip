// Spectral passes over single real fields: the Hartree potential and the
// gradient corrections of the exchange-correlation potential.
//
// A field of a few megabytes lives in the caches, so these passes are bound by
// the latency of their launches, not by memory: the transforms of an axis, the
// multiplications in G space, the point functions and the sums are fused until
// every launch is one direction change:
//   rho   x forward from the real field; y forward
//   V_H   z forward, x 4 pi / |G|^2, z back; y back; x back to the real field
//   PBE   z forward, x i G_d, z back (three components); y back; x back, sigma and
//         the point function, x forward of the flux; y forward; z forward,
//         sum_d i G_d, z back; y back; x back, added to v, with the sum of rho v
// Twelve launches for both against 27 with a pass of its own for each of these
// steps, and one copy of the sums to the host against three: poisson and xc("pbe")
// of a 64^3 density 254 -> 187 us, of 24^3 207 -> 134, of 96^3 395 -> 313, of 53 x
// 61 x 67 290 -> 208; the interacting step of 60 x 36 x 27 x 43 bands 1.76 -> 1.60
// ms.  The x and z passes use the DFT-matrix product (fft_dense.hpp): any length, one
// instantiation, and at these sizes a transform is a microsecond of matrix
// instructions.
#include "fields.hpp"

#include "fft_dense.hpp"
#include "xc_point.hpp"

namespace inqamd {

namespace {

struct field_geo {
  int n[3];
  double b[9];  // reciprocal lattice rows
  const cplx *tw;
  int L;        // the transformed axis
};

// A tile's LDS and columns
struct field_tile {
  cplx *U, *D, *tw;
  int L, h, hp, c, k0;
  unsigned g;  // this thread's column
  bool ok;
  __device__ field_tile(const field_geo &f, unsigned ncol, cplx *lds) {
    L = f.L;
    h = L / 2;
    hp = dense_rows(L);
    U = lds;
    D = lds + hp * DENSE_B;
    tw = lds + 2 * hp * DENSE_B;
    c = threadIdx.x % DENSE_B;
    const unsigned col = blockIdx.x * DENSE_B + c;
    ok = col < ncol;
    g = ok ? col : 0;
    k0 = 16 * (threadIdx.x >> 6) + ((threadIdx.x & 63) >> 4);
    for (int i = threadIdx.x; i < L; i += blockDim.x) tw[i] = f.tw[i];
  }
  __device__ bool pair(int k) const { return k != 0 && L - k != k; }
  // U and D of the column's elements ld(i), i < L; ends with a barrier
  template <class LD>
  __device__ void load(LD ld) {
    __syncthreads();  // earlier products have read U and D
    for (int n = threadIdx.x / DENSE_B; n < hp; n += blockDim.x / DENSE_B) {
      cplx u = mk(0.0, 0.0), d = u;
      if (n <= h) {
        const cplx x = ld(n);
        u = x;
        if (pair(n)) {
          const cplx y = ld(L - n);
          u = cadd(x, y);
          d = csub(x, y);
        }
      }
      U[n * DENSE_B + c] = u;
      D[n * DENSE_B + c] = d;
    }
    __syncthreads();
  }
  // U and D from values in the layout of a product's output, val(v, k, hi):
  // element k (hi = false) or L - k of the lane's row v
  template <class VAL>
  __device__ void refill(VAL val) {
    __syncthreads();
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int k = k0 + 4 * v;
      if (k <= h) {
        const cplx lo = val(v, k, false);
        cplx u = lo, d = mk(0.0, 0.0);
        if (pair(k)) {
          const cplx hi = val(v, L - k, true);
          u = cadd(lo, hi);
          d = csub(lo, hi);
        }
        U[k * DENSE_B + c] = u;
        D[k * DENSE_B + c] = d;
      }
    }
    __syncthreads();
  }
  __device__ dense_acc product() const { return dense_product(U, D, tw, L, hp); }
  // f(v, element, hi) for the lane's outputs
  template <class F>
  __device__ void each(F f) const {
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int k = k0 + 4 * v;
      if (k <= h) {
        f(v, k, false);
        if (pair(k)) f(v, L - k, true);
      }
    }
  }
};

// The lane's outputs of a product as values
struct field_values {
  cplx v[4][2];
  __device__ void from(const dense_acc &a, int sign) {
#pragma unroll
    for (int r = 0; r < 4; r++) dense_pair(a, r, sign, v[r][0], v[r][1]);
  }
};

// i G_d x scale
__device__ __forceinline__ cplx i_g(double g, cplx x) { return mk(-g * x.y, g * x.x); }

// Sums of NV values per thread over the workgroup into red[block][NV]
template <int NV>
__device__ __forceinline__ void tile_sums(double (&a)[NV], double *red) {
  __shared__ double sh[6][NV];
#pragma unroll
  for (int v = 0; v < NV; v++)
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) a[v] += __shfl_xor(a[v], w, 64);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int v = 0; v < NV; v++) sh[threadIdx.x >> 6][v] = a[v];
  __syncthreads();
  if (threadIdx.x == 0)
#pragma unroll
    for (int v = 0; v < NV; v++) {
      double s = sh[0][v];
      for (int w = 1; w < (int)blockDim.x / 64; w++) s += sh[w][v];
      red[(long)blockIdx.x * NV + v] = s;
    }
}

// x forward of a real field: columns (y, z), stride ny nz
__global__ __launch_bounds__(384) void field_x_forward(const field_geo f,
                                                       const double *__restrict__ rho,
                                                       cplx *__restrict__ out) {
  extern __shared__ cplx lds[];
  const long s = (long)f.n[1] * f.n[2];
  field_tile t(f, (unsigned)s, lds);
  t.load([&](int i) { return mk(rho[i * s + t.g], 0.0); });
  field_values y;
  y.from(t.product(), -1);
  t.each([&](int v, int i, bool hi) {
    if (t.ok) out[i * s + t.g] = y.v[v][hi];
  });
}

// x back to the real part of the field
__global__ __launch_bounds__(384) void field_x_back(const field_geo f, const cplx *__restrict__ in,
                                                    double *__restrict__ out) {
  extern __shared__ cplx lds[];
  const long s = (long)f.n[1] * f.n[2];
  field_tile t(f, (unsigned)s, lds);
  t.load([&](int i) { return in[i * s + t.g]; });
  field_values y;
  y.from(t.product(), +1);
  t.each([&](int v, int i, bool hi) {
    if (t.ok) out[i * s + t.g] = y.v[v][hi].x;
  });
}

// ... added to v, with the sums of rho v (gga_finish of the general path)
__global__ __launch_bounds__(384) void field_x_back_add(const field_geo f,
                                                        const cplx *__restrict__ in,
                                                        const double *__restrict__ rho,
                                                        double *__restrict__ vxc,
                                                        double *__restrict__ red) {
  extern __shared__ cplx lds[];
  const long s = (long)f.n[1] * f.n[2];
  field_tile t(f, (unsigned)s, lds);
  t.load([&](int i) { return in[i * s + t.g]; });
  field_values y;
  y.from(t.product(), +1);
  double a[1] = {0.0};
  t.each([&](int v, int i, bool hi) {
    if (t.ok) {
      const long p = i * s + t.g;
      const double x = vxc[p] + y.v[v][hi].x;
      vxc[p] = x;
      a[0] += rho[p] * x;
    }
  });
  tile_sums<1>(a, red);
}

// G of column (x, y) and z index i
struct field_g {
  double g0[3], bz[3];
  int nz;
  __device__ field_g(const field_geo &f, unsigned col) {
    const int ix = (int)(col / (unsigned)f.n[1]), iy = (int)(col - (unsigned)ix * f.n[1]);
    const int m0 = symmetric_index(ix, f.n[0]), m1 = symmetric_index(iy, f.n[1]);
    nz = f.n[2];
#pragma unroll
    for (int d = 0; d < 3; d++) {
      g0[d] = m0 * f.b[d] + m1 * f.b[3 + d];
      bz[d] = f.b[6 + d];
    }
  }
  __device__ double operator()(int d, int i) const {
    return g0[d] + symmetric_index(i, nz) * bz[d];
  }
};

// z forward, the periodic Poisson kernel (-4 pi / N)(-1 / |G|^2), 0 where
// |G|^2 < 1e-6 (poisson.hpp:29-35, 69-84), z back: columns are pencils
__global__ __launch_bounds__(384) void field_z_poisson(const field_geo f,
                                                       const cplx *__restrict__ in,
                                                       cplx *__restrict__ out, double scal) {
  extern __shared__ cplx lds[];
  field_tile t(f, (unsigned)f.n[0] * (unsigned)f.n[1], lds);
  const field_g G(f, t.g);
  const long base = (long)t.g * f.n[2];
  t.load([&](int i) { return in[base + i]; });
  field_values y;
  y.from(t.product(), -1);
  t.refill([&](int v, int i, bool hi) {
    const double gx = G(0, i), gy = G(1, i), gz = G(2, i);
    const double g2 = gx * gx + gy * gy + gz * gz;
    return cscale(scal * (g2 < 1e-6 ? 0.0 : -1.0 / g2), y.v[v][hi]);
  });
  y.from(t.product(), +1);
  t.each([&](int v, int i, bool hi) {
    if (t.ok) out[base + i] = y.v[v][hi];
  });
}

// z forward of one field, x i G_d / N and z back for its three components
// (out[d], fields of `field` elements)
__global__ __launch_bounds__(384) void field_z_gradient(const field_geo f,
                                                        const cplx *__restrict__ in,
                                                        cplx *__restrict__ out, long field,
                                                        double inv_n) {
  extern __shared__ cplx lds[];
  field_tile t(f, (unsigned)f.n[0] * (unsigned)f.n[1], lds);
  const field_g G(f, t.g);
  const long base = (long)t.g * f.n[2];
  t.load([&](int i) { return in[base + i]; });
  field_values y, w;
  y.from(t.product(), -1);
  for (int d = 0; d < 3; d++) {
    t.refill([&](int v, int i, bool hi) { return i_g(G(d, i) * inv_n, y.v[v][hi]); });
    w.from(t.product(), +1);
    t.each([&](int v, int i, bool hi) {
      if (t.ok) out[d * field + base + i] = w.v[v][hi];
    });
  }
}

// z forward of three components, sum_d i G_d / N, z back
__global__ __launch_bounds__(384) void field_z_divergence(const field_geo f,
                                                          const cplx *__restrict__ in, long field,
                                                          cplx *__restrict__ out, double inv_n) {
  extern __shared__ cplx lds[];
  field_tile t(f, (unsigned)f.n[0] * (unsigned)f.n[1], lds);
  const field_g G(f, t.g);
  const long base = (long)t.g * f.n[2];
  field_values y, w;
#pragma unroll
  for (int v = 0; v < 4; v++) w.v[v][0] = w.v[v][1] = mk(0.0, 0.0);
  for (int d = 0; d < 3; d++) {
    t.load([&](int i) { return in[d * field + base + i]; });
    y.from(t.product(), -1);
    t.each([&](int v, int i, bool hi) {
      w.v[v][hi] = cadd(w.v[v][hi], i_g(G(d, i), y.v[v][hi]));
    });
  }
  t.refill([&](int v, int, bool hi) { return cscale(inv_n, w.v[v][hi]); });
  y.from(t.product(), +1);
  t.each([&](int v, int i, bool hi) {
    if (t.ok) out[base + i] = y.v[v][hi];
  });
}

// x back of the three gradient components, the GGA's point function of n and
// sigma (the real parts, xc_term.hpp:267-292), x forward of the flux -2 vs grad n
// in their place; vxc = vn, sums of e n
__global__ __launch_bounds__(384) void field_x_gga(const field_geo f, cplx *g, long field,
                                                   const double *__restrict__ rho, int which,
                                                   double *__restrict__ vxc,
                                                   double *__restrict__ red) {
  extern __shared__ cplx lds[];
  const long s = (long)f.n[1] * f.n[2];
  field_tile t(f, (unsigned)s, lds);
  double gr[3][4][2];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    t.load([&](int i) { return g[d * field + i * s + t.g]; });
    field_values y;
    y.from(t.product(), +1);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      gr[d][v][0] = y.v[v][0].x;
      gr[d][v][1] = y.v[v][1].x;
    }
  }
  double a[1] = {0.0};
  t.each([&](int v, int i, bool hi) {
    const long p = i * s + t.g;
    const double r = rho[p], n = r < 0.0 ? 0.0 : r;
    const double gx = gr[0][v][hi], gy = gr[1][v][hi], gz = gr[2][v][hi];
    double e, vn, vs;
    gga_point(n, gx * gx + gy * gy + gz * gz, which, e, vn, vs);
    if (t.ok) {
      vxc[p] = vn;
      a[0] += e * n;
    }
#pragma unroll
    for (int d = 0; d < 3; d++) gr[d][v][hi] *= -2.0 * vs;
  });
#pragma unroll
  for (int d = 0; d < 3; d++) {
    t.refill([&](int v, int, bool hi) { return mk(gr[d][v][hi], 0.0); });
    field_values y;
    y.from(t.product(), -1);
    t.each([&](int v, int i, bool hi) {
      if (t.ok) g[d * field + i * s + t.g] = y.v[v][hi];
    });
  }
  tile_sums<1>(a, red);
}

// Totals of up to FIELD_SUMS rows of partial sums: one workgroup per row, threads
// strided over the partials, a butterfly per wave, the waves in order
__global__ __launch_bounds__(256) void field_totals(const field_sum_rows r, double *out) {
  __shared__ double sh[4];
  const double *x = r.part[blockIdx.x];
  const int n = r.n[blockIdx.x], st = r.stride[blockIdx.x];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += x[(long)i * st];
#pragma unroll
  for (int w = 32; w > 0; w >>= 1) s += __shfl_xor(s, w, 64);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = ((sh[0] + sh[1]) + sh[2]) + sh[3];
}

field_geo geo(const handle &h, int axis) {
  field_geo f;
  for (int d = 0; d < 3; d++) f.n[d] = h.n[d];
  for (int d = 0; d < 9; d++) f.b[d] = h.rlat[d];
  f.tw = h.axis[axis].tw;
  f.L = h.n[axis];
  return f;
}

// Launch shape of a pass along `axis`
struct field_launch {
  dim3 grid, block;
  size_t lds;
  field_launch(const handle &h, int axis) {
    const int L = h.n[axis];
    const long ncol = h.npoint / L;
    grid = dim3((unsigned)((ncol + DENSE_B - 1) / DENSE_B));
    block = dim3(64 * dense_waves(L));
    lds = (size_t)(2 * dense_rows(L) * DENSE_B + L) * sizeof(cplx);
  }
};

#define FIELD_LAUNCH(kernel, h, axis, ...)                                              \
  do {                                                                                  \
    const field_launch l_(h, axis);                                                     \
    hipLaunchKernelGGL(kernel, l_.grid, l_.block, l_.lds, (h).stream, geo(h, axis),     \
                       __VA_ARGS__);                                                    \
    INQAMD_HIP_CHECK(hipGetLastError());                                                \
  } while (0)

}  // namespace

// All lengths that the product takes.  Its work grows with the length, but the
// passes still win where they end: PBE of 120^3 353 us against 426 with a pass for
// each step, of 144^3 1475 against 1675, of 180^3 2916 against 3140, of 191 x 190 x
// 187 1918 against 2214 (only 128^3, whose strides are powers of two, 555 against
// 486); Poisson of 144^3 340 against 669, of 180^3 596 against 1160.
bool fields_supported(const handle &h) {
  return h.n[0] <= DENSE_MAX_LEN && h.n[1] <= DENSE_MAX_LEN && h.n[2] <= DENSE_MAX_LEN;
}

long field_partials(const handle &h) {
  return (h.npoint / h.n[0] + DENSE_B - 1) / DENSE_B;
}

void field_forward_xy(handle &h, const double *rho, cplx *c) {
  FIELD_LAUNCH(field_x_forward, h, 0, rho, c);
  fft_y_pass(h, c, 1, -1);
}

void field_hartree(handle &h, const cplx *c, cplx *work, double *vh) {
  const double scal = (-4.0 * 3.14159265358979323846) / (double)h.npoint;
  FIELD_LAUNCH(field_z_poisson, h, 2, c, work, scal);
  fft_y_pass(h, work, 1, +1);
  FIELD_LAUNCH(field_x_back, h, 0, (const cplx *)work, vh);
}

void field_gga(handle &h, const cplx *c, cplx *g3, cplx *work, const double *rho, int which,
               double *vxc, double *red_e, double *red_v) {
  const double inv_n = 1.0 / (double)h.npoint;
  FIELD_LAUNCH(field_z_gradient, h, 2, c, g3, h.npoint, inv_n);
  fft_y_pass(h, g3, 3, +1);
  FIELD_LAUNCH(field_x_gga, h, 0, g3, h.npoint, rho, which, vxc, red_e);
  fft_y_pass(h, g3, 3, -1);
  FIELD_LAUNCH(field_z_divergence, h, 2, (const cplx *)g3, h.npoint, work, inv_n);
  fft_y_pass(h, work, 1, +1);
  FIELD_LAUNCH(field_x_back_add, h, 0, (const cplx *)work, rho, vxc, red_v);
}

void field_sums(handle &h, const field_sum_rows &r, int nrows, double *out) {
  hipLaunchKernelGGL(field_totals, dim3(nrows), dim3(256), 0, h.stream, r, out);
  INQAMD_HIP_CHECK(hipGetLastError());
}

}  // namespace inqamd
