// Batched complex128 3-D FFT over INQ's [x][y][z][band] layout, built from
// one-axis "pencil" passes.  Each pass stages a tile of `len` points x B
// contiguous bands in LDS, runs a mixed-radix Stockham FFT there and writes
// the tile back, optionally fused with the kinetic multiply (fwd, x T(G), bwd
// in one pass) or with the Hpsi epilogue (x 1/N + V psi).
#pragma once

#include "common.hpp"

#include <vector>

namespace inqamd {

constexpr int FFT_MAX_STAGES = 12;
constexpr int FFT_MAX_GENERIC_RADIX = 31;  // largest radix with a register-resident butterfly
constexpr int FFT_BLOCK = 256;

enum fft_mode : int { FFT_PLAIN = 0, FFT_KINETIC = 1, FFT_EPILOGUE = 2 };

// Ownership-map word of a grid point: first entry << OWN_COUNT_BITS | entry count.
constexpr int OWN_COUNT_BITS = 8;
constexpr int OWN_MAX_COUNT = (1 << OWN_COUNT_BITS) - 1;

struct fft_axis_plan {
  int len = 0;
  int nstages = 0;
  int radix[FFT_MAX_STAGES] = {};
  cplx *tw = nullptr;  // device: W_len^k = exp(-2 pi i k / len), k < len
};

// Arguments of one pencil pass (passed by value to the kernel).
struct fft_pass_args {
  const cplx *in;
  long in_ld;
  cplx *out;
  long out_ld;
  int nst;
  int len;
  long stride;  // point stride along the transformed axis
  int c1;       // other axis 1 (fastest varying over workgroups)
  long s1;
  int c2;
  long s2;
  int nstages;
  int radix[FFT_MAX_STAGES];
  const cplx *tw;
  double scale;
  int sign;
  // FFT_KINETIC: element (i, o1, o2) sits at grid coords c[ax]=i, c[ax1]=o1, c[ax2]=o2
  int n[3];
  int ax, ax1, ax2;
  double rlat[9];      // reciprocal lattice rows (include 2 pi)
  const double *kA;    // device, covariant k + A
  // FFT_EPILOGUE: out = scale * fft + V[p] * psi[p][b]
  const double *V;
  const cplx *psi;
  long psi_ld;
};

// Factor len into radices (8, 4, 2, 3, 5, then the remaining primes; those
// above FFT_MAX_GENERIC_RADIX run a direct O(R^2) stage from LDS).
// Returns false if that takes more than FFT_MAX_STAGES stages.
bool fft_factor(int len, std::vector<int> &radices);

// Host twiddle table exp(-2 pi i k/len), evaluated in long double.
std::vector<cplx> fft_twiddles(int len);

// Band tile chosen for a given nst and axis length.
int fft_band_tile(int nst, int len);

// Launch one pencil pass of the given mode on `stream`.
void fft_launch_pass(const fft_pass_args &a, int mode, hipStream_t stream);

// Plan-specialised pass (fft_plan.hip) for the tabulated lengths; returns
// false when the length has no instantiation.
bool fft_plan_launch(const fft_pass_args &a, int mode, hipStream_t stream);

// DFT-matrix pass on the matrix cores (fft_dense.hip) for the lengths that it
// takes; false for the others.
bool fft_dense_launch(const fft_pass_args &a, int mode, hipStream_t stream);

// Powers H^n psi that a Taylor chain keeps before one sweep adds them to its sums
constexpr int TAYLOR_PENDING = 3;

struct project_expand_args;  // internal.hpp

// The projector phases e^{+-i(k+A).r} of a call, computed by extra workgroups of
// its first sweep (pos == nullptr: none)
struct phase_args {
  const float *pos;
  const int *uent;
  int nsph, nent;
  cplx *sph, *ent;
};

// Arguments of the three-sweep local Hamiltonian (fft3.hip) on a band chunk
// of a cubic L^3 grid (or an nx x ny x nz one: fft3_rect.hpp).
struct fft3_args {
  const cplx *psi;   // chunk's first band, INQ layout, leading dimension ld
  long ld;
  cplx *hpsi;        // output, leading dimension hld
  long hld;
  cplx *W;           // band-major intermediate [nb][L][L][L]
  int nb;
  // psi, hpsi, Qe and the accumulators hold chunk band cb at offset
  // cb + (cb >> (3 + glog)) * gskip: groups of 8 << glog bands
  // (gskip 0: the chunk's bands are contiguous)
  int gskip, glog;
  const double *V;   // [N]
  const double *kA;  // device covariant k + A
  double rlat[9];
  const cplx *tw;    // W_L^k table (of the z axis)
  double scale;      // 1/N
  // nx x ny x nz grids (fft3_rect.hpp): extents and tables of the other axes
  int nx, ny;
  const cplx *twx, *twy;
  // projector apply fused into the last sweep (own == nullptr: not fused):
  // hpsi(p, b) += sum_{j < cnt} Qe[e0 + j][b] with own[p] = (e0 << OWN_COUNT_BITS) | cnt
  // (own[p] = -1 where no sphere reaches)
  const int *own;
  const cplx *Qe;        // [nent][ldQ], offset to the chunk's first band
  long ldQ;
  // or (Pc != nullptr, Qe unused) V_nl psi expanded at the owned points
  // from the projector coefficients: hpsi(p, b) += sum_{j < cnt}
  // phase_ent[e] sum_{lm < nlmP} ent_mat[e][lm] Pc[(ent_sph[e] nlmP + lm) ldPc + b],
  // e = e0 + j (Pc offset to the chunk's first band; ent_sph[e0] = own_sph[p])
  const cplx *Pc;
  long ldPc;
  int nlmP;
  const int *ent_sph;     // [nent] sphere of each ownership entry
  const int *own_sph;     // [N] sphere of a point's first entry (0 where unowned)
  const double *ent_mat;  // [nent][4] projector values at the entry's point
  const cplx *phase_ent;  // [nent] e^{-i(k+A).r} of the call
  // Taylor sums (acc1 == nullptr / acc2 == nullptr: unused), chunk-offset:
  //   acc1 = src1 + sum_{j < npend} pc1[j] pend[j] + c1 hpsi, terms in this order
  //   acc2 = acc2 + sum_{j < npend} pc2[j] pend[j] + c2 hpsi
  // with src1 the old acc1 or the state that the sum starts from, and pend the
  // earlier powers that no sum holds yet (each at its own points only, so hpsi
  // may be written over pend[0])
  cplx *acc1;
  long acc1_ld;
  const cplx *src1;
  long src1_ld;
  double c1re, c1im;
  cplx *acc2;
  long acc2_ld;
  double c2re, c2im;
  int npend;
  const cplx *pend[TAYLOR_PENDING];
  long pend_ld;
  double pc1re[TAYLOR_PENDING], pc1im[TAYLOR_PENDING];
  double pc2re[TAYLOR_PENDING], pc2im[TAYLOR_PENDING];
  // optional copy of psi's forward transform (before the kinetic factor),
  // band-major [nb][kz][kx][ky] like W, chunk-offset (nullptr: none)
  cplx *gdump;
  // hpsi not written at all (the last term of a Taylor chain: only the
  // accumulators need it)
  int skip_store;
  // the phases of the projector, in workgroups after the z forward tiles
  phase_args phase;
  int nproj;  // spheres of the projector that an x-y launch carries
  // deal z tiles per XCD also in the sweeps that run them in natural order
  // (rows that start off a 128-byte line: neighbouring band tiles share lines)
  int xcd;
  // launch shapes (0: the process default): z tiles of z_ty y values, x-y
  // planes with plane_threads(L) (xy_wide 1) or twice as many (2)
  int z_ty, xy_wide;
  // G-space Hpsi sweeps: G-space orbitals whose 1/2 |G+k+A|^2 multiple the
  // last sweep adds (fft3_fourier_hamiltonian)
  const cplx *kin_in;
  long kin_ld;
  // its planes: the owned points of plane z are rows [zoff[z], zoff[z + 1]) of
  // zxy (x << 16 | y), zown (ownership words) and S (zoff == nullptr: none);
  // psi at the owned points goes to S [row][ldS], V_nl psi comes from Qe, both
  // with the chunk's band cb at column cb
  const int *zoff, *zxy, *zown;
  cplx *S;
  long ldS;
  // and the preconditioner its first sweep applies to psi, in place (pre_kin ==
  // nullptr: none): K(1/2 |G|^2 / pre_kin[16 b]) for the chunk's band at offset b
  cplx *pre_psi;
  const double *pre_kin;
  // and the partial sums of the line search over them (mm_phi == nullptr: none):
  // for each (x, y rows) of the grid and band mm_band0 + b, the eight of
  // line_sums over phi, kin_in and hpsi into mm_part[row][mm_nst][8]
  const cplx *mm_phi;
  long mm_ld;
  double *mm_part;
  int mm_nst, mm_band0;
};

// K of Teter, Payne and Allan (preconditioner.hpp:30-37)
__device__ __forceinline__ double tpa_k(double x) {
  const double num = ((8.0 * x + 12.0) * x + 18.0) * x + 27.0;
  const double den = (((16.0 * x + 8.0) * x + 12.0) * x + 18.0) * x + 27.0;
  return num / den;
}

// <r|r>, <f|r>, <r|h>, <f|h> (real, imaginary) of one element
// (steepest_descent.hpp:47-51)
__device__ __forceinline__ void line_sums(double *a, cplx f, cplx r, cplx h) {
  a[0] += r.x * r.x + r.y * r.y;
  a[1] += r.x * r.y - r.y * r.x;
  a[2] += f.x * r.x + f.y * r.y;
  a[3] += f.x * r.y - f.y * r.x;
  a[4] += r.x * h.x + r.y * h.y;
  a[5] += r.x * h.y - r.y * h.x;
  a[6] += f.x * h.x + f.y * h.y;
  a[7] += f.x * h.y - f.y * h.x;
}

// Rows of those partial sums
inline long line_sum_rows(int nx, int ny) { return (long)nx * ((ny + 7) / 8); }

// G-space Hpsi on the chunk's bands from phi (`psi` and `kin_in`): hpsi =
// FFT(V psi + V_nl psi) + 1/2 |G+k+A|^2 phi with psi = IFFT(phi).
// G_INVERSE: z inverse into W and, with owned points, psi there into S (for
// the projector, which leaves V_nl psi in Qe).  G_FORWARD: the planes (x and y
// inverse, potential terms, x and y forward) and the z forward write with the
// kinetic term.
enum fourier_half : int { G_INVERSE, G_FORWARD };
void fft3_fourier_hamiltonian(const fft3_args &a, int L, hipStream_t stream, fourier_half half);

// True when the three-sweep kernels exist for length L and fit in max_lds.
bool fft3_supported(int L, size_t max_lds);
// Sets the kernels' LDS attributes for length L (once, before any launch).
void fft3_prepare(int L);
// hpsi = IFFT(1/2|G+k+A|^2 FFT(psi)) / N + V psi for the chunk's bands: all
// three sweeps (sweep < 0) or only sweep 0 (z forward), 1 (x-y) or 2 (z back).
// proj: the chunk's projector coefficients, by workgroups of the x-y launch
// (lengths and workgroup shapes of fft3_projector only).
void fft3_local_hamiltonian(const fft3_args &a, int L, hipStream_t stream, int sweep = -1,
                            bool fwd_next = false, const project_expand_args *proj = nullptr);
// Whether the x-y launch of nb bands on an L^3 grid may carry the projector;
// xy_wide as in fft3_args.
bool fft3_projector(int L, int nb, int xy_wide);

// The same sweeps on an n[0] x n[1] x n[2] grid (fft3_rect.hip): true when every
// length has a plan there and the plane and the z tile fit in max_lds.
bool fft3_rect_supported(const int n[3], size_t max_lds);
void fft3_rect_prepare(const int n[3]);
void fft3_rect_local_hamiltonian(const fft3_args &a, const int n[3], hipStream_t stream, int sweep,
                                 bool fwd_next, const project_expand_args *proj = nullptr);
bool fft3_rect_projector(const int n[3], int nb);
void fft3_rect_fourier_hamiltonian(const fft3_args &a, const int n[3], hipStream_t stream,
                                   fourier_half half);

// G-space moments of the chunk's bands from W after the z forward sweep, rows
// [nst n[2]][8] offset to the chunk's first band, bands at the offsets that they
// have in psi (fft3_rect.hip; cubic grids too); where both plane axes have plans
bool fft3_moments_supported(const int n[3], size_t max_lds);
// Sets their LDS attributes (once, before any launch; fft3_rect_prepare does too)
void fft3_moments_prepare(const int n[3]);
void fft3_moments(const fft3_args &a, const int n[3], double *rows, hipStream_t stream);

}  // namespace inqamd
