// Fused spectral passes over single fields (fields.hip).
#pragma once

#include "internal.hpp"

namespace inqamd {

// Rows of partial sums for one totals launch: n[r] values at stride[r]
constexpr int FIELD_SUMS = 4;
struct field_sum_rows {
  const double *part[FIELD_SUMS];
  int n[FIELD_SUMS], stride[FIELD_SUMS];
};

// Whether every axis is short enough for these passes
bool fields_supported(const handle &h);
// Partial sums (one per workgroup) of a pass along x
long field_partials(const handle &h);

// c = the x and y transforms of the real field rho
void field_forward_xy(handle &h, const double *rho, cplx *c);
// vh = the periodic Hartree potential of c = field_forward_xy(rho)
void field_hartree(handle &h, const cplx *c, cplx *work, double *vh);
// A GGA (which: 1 exchange, 2 correlation, 3 both) of rho, c its field_forward_xy:
// vxc, and the partial sums of e n (red_e) and rho vxc (red_v); g3 three fields
void field_gga(handle &h, const cplx *c, cplx *g3, cplx *work, const double *rho, int which,
               double *vxc, double *red_e, double *red_v);
// out[r] = the total of row r (device)
void field_sums(handle &h, const field_sum_rows &r, int nrows, double *out);

// hamiltonian.hip: the y transforms of nf consecutive fields, in place
void fft_y_pass(handle &h, cplx *c, int nf, int sign);

}  // namespace inqamd
