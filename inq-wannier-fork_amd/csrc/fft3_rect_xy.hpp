// x-y planes of the nx x ny x nz three-sweep Hpsi (see fft3_rect.hpp), included by the
// files that instantiate them.
//
// A workgroup transforms one (band, z) plane W[b][z][.][.] of nx x ny in LDS
// (rows padded to an odd count of 16-byte elements), like the cubic planes, but
// the number of columns of each axis's transform is a run-time value: butterfly w
// is butterfly w / C of column w % C, by a float reciprocal (exact: w < 2^14).
// Workgroups of 128 to 1024 threads by the size of the plane: a thread holds at
// most two butterflies between a stage's loads and its stores (18 elements at 128
// and 512 threads, 20 at 256, 16 at 1024).  The sweep is bound by the barriers
// between the stages, which the other planes of a CU fill.

#pragma once

#include "fft3_rect.hpp"
#include "projector_dev.hpp"

namespace inqamd {

// Most columns beside an axis of length L
constexpr int rect_columns(int L, int NT) {
  return rect_elements(NT) / L < RECT_MAX_LEN ? rect_elements(NT) / L : RECT_MAX_LEN;
}

template <int R, int L, int NT>
struct rect_regs {
  static constexpr int NBF = (L / R * rect_columns(L, NT) + NT - 1) / NT;
  cplx v[NBF][R];
};

// Columns of one axis's transform
struct rect_cols {
  int C;
  float inv;
  __device__ void split(int w, int &j, int &c) const {
    j = (int)(((float)w + 0.5f) * inv);
    c = w - j * C;
  }
};

// Calls f(q, j, c) for each butterfly of this thread
template <int R, int L, int NT, class F>
__device__ __forceinline__ void rect_each(const rect_cols &k, F f) {
#pragma unroll
  for (int q = 0; q < rect_regs<R, L, NT>::NBF; q++) {
    const int w = threadIdx.x + q * NT;
    int j, c;
    k.split(w, j, c);
    if (j < L / R) f(q, j, c);
  }
}

template <int R, int L, int NT, class LD>
__device__ __forceinline__ void rect_load(rect_regs<R, L, NT> &in, const rect_cols &k, LD ld) {
  rect_each<R, L, NT>(k, [&](int q, int j, int c) {
#pragma unroll
    for (int r = 0; r < R; r++) in.v[q][r] = ld(j + r * (L / R), c);
  });
}

template <int R, int NS, int L, int NT>
__device__ __forceinline__ void rect_compute(rect_regs<R, L, NT> &in, const rect_cols &k,
                                             const cplx *__restrict__ tw, int sign) {
  rect_each<R, L, NT>(k, [&](int q, int j, int) {
    if constexpr (NS > 1) {
      const int kk = j % NS;
#pragma unroll
      for (int r = 1; r < R; r++)
        in.v[q][r] = cmul(in.v[q][r], twiddle(tw, r * kk * (L / (NS * R)), sign));
    }
    dft<R>(in.v[q], sign);
  });
}

template <int R, int NS, int L, int NT, class ST>
__device__ __forceinline__ void rect_store(rect_regs<R, L, NT> &in, const rect_cols &k, ST st) {
  rect_each<R, L, NT>(k, [&](int q, int j, int c) {
    const int base = (j / NS) * NS * R + j % NS;
#pragma unroll
    for (int r = 0; r < R; r++) st(base + r * NS, c, in.v[q][r]);
  });
}

// One in-place LDS stage (between barriers)
template <int R, int NS, int L, int NT, class LD, class ST>
__device__ __forceinline__ void rect_stage(const rect_cols &k, const cplx *tw, int sign, LD ld,
                                           ST st) {
  rect_regs<R, L, NT> in;
  rect_load<R, L, NT>(in, k, ld);
  rect_compute<R, NS, L, NT>(in, k, tw, sign);
  __syncthreads();
  rect_store<R, NS, L, NT>(in, k, st);
  __syncthreads();
}

// The stages of an axis from `first` (global or LDS) to `last` (LDS or global)
// through ld / st in LDS; FROM_LDS, TO_LDS: whether the ends share the array
template <int R0, int R1, int R2, int NT, bool FROM_LDS, bool TO_LDS, class FL, class LD, class ST,
          class LS>
__device__ __forceinline__ void rect_axis(const rect_cols &k, const cplx *tw, int sign, FL first,
                                          LD ld, ST st, LS last) {
  constexpr int L = R0 * R1 * R2;
  static_assert(R1 > 1, "at least two stages");
  {
    rect_regs<R0, L, NT> in;
    rect_load<R0, L, NT>(in, k, first);
    rect_compute<R0, 1, L, NT>(in, k, tw, sign);
    if (FROM_LDS) __syncthreads();
    rect_store<R0, 1, L, NT>(in, k, st);
    __syncthreads();
  }
  if constexpr (R2 > 1) rect_stage<R1, R0, L, NT>(k, tw, sign, ld, st);
  constexpr int RL = R2 > 1 ? R2 : R1, NSL = L / RL;
  rect_regs<RL, L, NT> in;
  rect_load<RL, L, NT>(in, k, ld);
  rect_compute<RL, NSL, L, NT>(in, k, tw, sign);
  if (TO_LDS) __syncthreads();
  rect_store<RL, NSL, L, NT>(in, k, last);
  if (TO_LDS) __syncthreads();
}

// The y axis of the kinetic plane: forward, x 1/2 |G+k+A|^2 (and the copy of the
// transform before it), inverse.  The forward's last stage holds in butterfly j
// the outputs j + r L/RL, the inputs of the first stage of the inverse run with
// the radices in reverse order, so that stage starts from the registers.
template <int R0, int R1, int R2, int NT, class LD, class ST, class KIN>
__device__ __forceinline__ void rect_y_kinetic(const rect_cols &k, const cplx *tw, LD ld, ST st,
                                               KIN kin) {
  constexpr int L = R0 * R1 * R2;
  constexpr int RL = R2 > 1 ? R2 : R1, NSL = L / RL;
  rect_stage<R0, 1, L, NT>(k, tw, -1, ld, st);
  if constexpr (R2 > 1) rect_stage<R1, R0, L, NT>(k, tw, -1, ld, st);
  {
    rect_regs<RL, L, NT> in;
    rect_load<RL, L, NT>(in, k, ld);
    rect_compute<RL, NSL, L, NT>(in, k, tw, -1);
    rect_each<RL, L, NT>(k, [&](int q, int j, int c) {
#pragma unroll
      for (int r = 0; r < RL; r++) in.v[q][r] = kin(j + r * NSL, c, in.v[q][r]);
    });
    rect_compute<RL, 1, L, NT>(in, k, tw, +1);
    __syncthreads();
    rect_store<RL, 1, L, NT>(in, k, st);
    __syncthreads();
  }
  if constexpr (R2 > 1) rect_stage<R1, RL, L, NT>(k, tw, +1, ld, st);
  rect_stage<R0, L / R0, L, NT>(k, tw, +1, ld, st);
}

// Plane `plane` = band * nz + z
template <int NT>
__device__ __forceinline__ void rect_xy_plane(const fft3_args &a, int nz, long plane, cplx *lds) {
  const int nx = a.nx, ny = a.ny, pad = ny | 1;
  const int z = (int)(plane % nz);
  cplx *W = a.W + plane * nx * ny;
  const rect_cols kx = {ny, 1.0f / (float)ny}, ky = {nx, 1.0f / (float)nx};

  // x axis: element (i = x, c = y); y axis: (i = y, c = x)
  auto gx = [&](int i, int c) -> cplx { return W[i * ny + c]; };
  auto wx = [&](int i, int c, cplx v) { W[i * ny + c] = v; };
  auto lx = [&](int i, int c) -> cplx { return lds[i * pad + c]; };
  auto sx = [&](int i, int c, cplx v) { lds[i * pad + c] = v; };
  auto ly = [&](int i, int c) -> cplx { return lds[c * pad + i]; };
  auto sy = [&](int i, int c, cplx v) { lds[c * pad + i] = v; };

  switch (nx) {
#define INQAMD_RECT_CASE(L, R0, R1, R2)                                                   \
  case L:                                                                                \
    rect_axis<R0, R1, R2, NT, false, true>(kx, a.twx, -1, gx, lx, sx, sx);               \
    break;
    INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
  }
  // 1/2 |G + k + A|^2 with G = m_x b0 + m_y b1 + m_z b2 (cartesian)
  double kc[3], gz[3], b0[3], b1[3];
  xy_kc(a, kc);
  const int mz = symmetric_index(z, nz);
#pragma unroll
  for (int d = 0; d < 3; d++) {
    gz[d] = mz * a.rlat[2 * 3 + d] + kc[d];
    b0[d] = a.rlat[0 * 3 + d];
    b1[d] = a.rlat[1 * 3 + d];
  }
  cplx *G = a.gdump ? a.gdump + plane * nx * ny : nullptr;
  auto kin = [&](int i, int c, cplx v) -> cplx {
    if (G) G[c * ny + i] = v;
    const int my = symmetric_index(i, ny), mx = symmetric_index(c, nx);
    const double q0 = mx * b0[0] + my * b1[0] + gz[0];
    const double q1 = mx * b0[1] + my * b1[1] + gz[1];
    const double q2 = mx * b0[2] + my * b1[2] + gz[2];
    return cscale(0.5 * (q0 * q0 + q1 * q1 + q2 * q2), v);
  };
  switch (ny) {
#define INQAMD_RECT_CASE(L, R0, R1, R2)                                                   \
case L: rect_y_kinetic<R0, R1, R2, NT>(ky, a.twy, ly, sy, kin); break;
    INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
  }
  switch (nx) {
#define INQAMD_RECT_CASE(L, R0, R1, R2)                                                   \
case L:                                                                                \
  rect_axis<R0, R1, R2, NT, true, false>(kx, a.twx, +1, lx, lx, sx, wx);               \
  break;
    INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
  }
}

// The planes of the G-space Hpsi (xy_real_plane of the cubic grids)
template <int NT, bool GATHER>
__device__ __forceinline__ void rect_real_plane(const fft3_args &a, int nz, long t, cplx *lds) {
  const int nx = a.nx, ny = a.ny, pad = ny | 1;
  const int z = (int)(t / a.nb), b = (int)(t - (long)z * a.nb);
  const int zo = a.zoff ? a.zoff[z] : 0, zn = a.zoff ? a.zoff[z + 1] - zo : 0;
  if constexpr (GATHER) {
    if (zn == 0) return;
  }
  cplx *W = a.W + ((long)b * nz + z) * nx * ny;
  const rect_cols kx = {ny, 1.0f / (float)ny}, ky = {nx, 1.0f / (float)nx};
  auto gx = [&](int i, int c) -> cplx { return W[i * ny + c]; };  // (i = x, c = y)
  auto wx = [&](int i, int c, cplx v) { W[i * ny + c] = v; };
  auto lx = [&](int i, int c) -> cplx { return lds[i * pad + c]; };
  auto sx = [&](int i, int c, cplx v) { lds[i * pad + c] = v; };
  auto ly = [&](int i, int c) -> cplx { return lds[c * pad + i]; };  // (i = y, c = x)
  auto sy = [&](int i, int c, cplx v) { lds[c * pad + i] = v; };
  const double *V = a.V + z;
  auto sv = [&](int i, int c, cplx v) {
    if constexpr (!GATHER) v = cscale(a.scale * V[((long)c * ny + i) * nz], v);
    lds[c * pad + i] = v;
  };
  auto slot = [&](int k) {
    const int xy = a.zxy[zo + k];
    return (xy >> 16) * pad + (xy & 0xffff);
  };
  const int own0 = !GATHER && (int)threadIdx.x < zn ? a.zown[zo + threadIdx.x] : 0;
  switch (nx) {
#define INQAMD_RECT_CASE(L, R0, R1, R2) \
  case L: rect_axis<R0, R1, R2, NT, false, true>(kx, a.twx, +1, gx, lx, sx, sx); break;
    INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
  }
  cplx first = mk(0.0, 0.0);
  if (own0) first = a.Qe[(long)(own0 >> OWN_COUNT_BITS) * a.ldQ + b];
  switch (ny) {
#define INQAMD_RECT_CASE(L, R0, R1, R2) \
  case L: rect_axis<R0, R1, R2, NT, true, true>(ky, a.twy, +1, ly, ly, sy, sv); break;
    INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
  }
  if constexpr (GATHER) {
    for (int k = threadIdx.x; k < zn; k += NT)
      a.S[(long)(zo + k) * a.ldS + b] = cscale(a.scale, lds[slot(k)]);
  } else {
    if (zn > 0) {
      for (int k = threadIdx.x; k < zn; k += NT) {
        const int own = k < NT ? own0 : a.zown[zo + k];
        const int e0 = own >> OWN_COUNT_BITS, cnt = own & OWN_MAX_COUNT;
        cplx v = k < NT ? first : a.Qe[(long)e0 * a.ldQ + b];
        for (int j = 1; j < cnt; j++) v = cadd(v, a.Qe[(long)(e0 + j) * a.ldQ + b]);
        const int e = slot(k);
        lds[e] = cadd(lds[e], v);
      }
      __syncthreads();
    }
    switch (ny) {
#define INQAMD_RECT_CASE(L, R0, R1, R2) \
  case L: rect_axis<R0, R1, R2, NT, true, true>(ky, a.twy, -1, ly, ly, sy, sy); break;
      INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
    }
    switch (nx) {
#define INQAMD_RECT_CASE(L, R0, R1, R2) \
  case L: rect_axis<R0, R1, R2, NT, true, false>(kx, a.twx, -1, lx, lx, sx, wx); break;
      INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
    }
  }
}

// Plane `plane` = band * nz + z of W (psi transformed in z): the sums of |psi^|^2 m_c
// over the plane, m_0 = 1 and m_1..3 the symmetric indices (x, y, z), into
// rows[offset of the band in psi x nz + z][8] (complex, like the other G-space
// moments), so that the order of their sum is the same for any chunks.  Nothing is
// written back: two sweeps, 48 N bytes per band, where three pencil passes and a pass over
// their result moved 112 (density, dipole, energies and current of 36 x 36 x 90 x 48
// bands 540 -> 496 us, of 64^3 x 64 1130 -> 1033 us, of 96^3 x 8 878 -> 827 us).
template <int NT>
__device__ __forceinline__ void rect_moments_plane(const fft3_args &a, int nz, long plane,
                                                   cplx *lds, double *rows) {
  const int nx = a.nx, ny = a.ny, pad = ny | 1;
  const cplx *W = a.W + plane * nx * ny;
  const rect_cols kx = {ny, 1.0f / (float)ny}, ky = {nx, 1.0f / (float)nx};
  auto gx = [&](int i, int c) -> cplx { return W[i * ny + c]; };  // (i = x, c = y)
  auto lx = [&](int i, int c) -> cplx { return lds[i * pad + c]; };
  auto sx = [&](int i, int c, cplx v) { lds[i * pad + c] = v; };
  auto ly = [&](int i, int c) -> cplx { return lds[c * pad + i]; };  // (i = y, c = x)
  auto sy = [&](int i, int c, cplx v) { lds[c * pad + i] = v; };
  switch (nx) {
#define INQAMD_RECT_CASE(L, R0, R1, R2) \
  case L: rect_axis<R0, R1, R2, NT, false, true>(kx, a.twx, -1, gx, lx, sx, sx); break;
    INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
  }
  double s[3] = {0.0, 0.0, 0.0};
  auto sum = [&](int i, int c, cplx v) {
    const double t = v.x * v.x + v.y * v.y;
    s[0] += t;
    s[1] += symmetric_index(c, nx) * t;
    s[2] += symmetric_index(i, ny) * t;
  };
  switch (ny) {
#define INQAMD_RECT_CASE(L, R0, R1, R2) \
  case L: rect_axis<R0, R1, R2, NT, true, false>(ky, a.twy, -1, ly, ly, sy, sum); break;
    INQAMD_RECT_XY(INQAMD_RECT_CASE)
#undef INQAMD_RECT_CASE
  }
  // the lanes of a wave by a butterfly, the waves in order
  double *red = reinterpret_cast<double *>(lds);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; k++) {
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) s[k] += __shfl_xor(s[k], w, 64);
    if ((threadIdx.x & 63) == 0) red[(threadIdx.x >> 6) * 3 + k] = s[k];
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int w = 1; w < NT / 64; w++)
    for (int k = 0; k < 3; k++) s[k] += red[w * 3 + k];
  const int cb = (int)(plane / nz), z = (int)(plane - (long)cb * nz);
  double *r = rows + ((long)(cb + (cb >> (3 + a.glog)) * a.gskip) * nz + z) * 8;
  r[0] = s[0];
  r[2] = s[1];
  r[4] = s[2];
  r[6] = symmetric_index(z, nz) * s[0];
  r[1] = r[3] = r[5] = r[7] = 0.0;
}

template <int NT, int MODE>
__global__ __launch_bounds__(NT) void rect_xy_kernel(const fft3_args a, int nz) {
  extern __shared__ cplx lds[];
  if constexpr (MODE == RECT_KINETIC)
    rect_xy_plane<NT>(a, nz, blockIdx.x, lds);
  else
    rect_real_plane<NT, MODE == RECT_GATHER>(a, nz, xcd_tile(blockIdx.x, gridDim.x, a.nb), lds);
}

template <int NT>
__global__ __launch_bounds__(NT) void rect_moments_kernel(const fft3_args a, int nz, double *rows) {
  extern __shared__ cplx lds[];
  rect_moments_plane<NT>(a, nz, blockIdx.x, lds, rows);
}

template <int NT>
void rect_xy_launch(const fft3_args &a, const int n[3], rect_planes what, double *rows,
                    hipStream_t stream) {
  const dim3 planes((unsigned)((long)a.nb * n[2])), nt(NT);
  const size_t lds = rect_xy_lds(n);
  auto attribute = [&](const void *k) {
    if (lds > 65536)
      INQAMD_HIP_CHECK(
          hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 163840));
  };
  switch (what) {
    case RECT_KINETIC:
      hipLaunchKernelGGL((rect_xy_kernel<NT, RECT_KINETIC>), planes, nt, lds, stream, a, n[2]);
      break;
    case RECT_GATHER:
      hipLaunchKernelGGL((rect_xy_kernel<NT, RECT_GATHER>), planes, nt, lds, stream, a, n[2]);
      break;
    case RECT_POTENTIAL:
      hipLaunchKernelGGL((rect_xy_kernel<NT, RECT_POTENTIAL>), planes, nt, lds, stream, a, n[2]);
      break;
    case RECT_MOMENTS:
      hipLaunchKernelGGL(rect_moments_kernel<NT>, planes, nt, lds, stream, a, n[2], rows);
      break;
    case RECT_XY_PREPARE:
      attribute((const void *)rect_xy_kernel<NT, RECT_KINETIC>);
      attribute((const void *)rect_xy_kernel<NT, RECT_GATHER>);
      attribute((const void *)rect_xy_kernel<NT, RECT_POTENTIAL>);
      attribute((const void *)rect_moments_kernel<NT>);
      return;
  }
  INQAMD_HIP_CHECK(hipGetLastError());
}

}  // namespace inqamd
