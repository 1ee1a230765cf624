// z-sweep kernels of fft3_rect.hpp, lengths of INQAMD_RECT_Z_B.
#include "fft3_rect_z.hpp"

namespace inqamd {

bool rect_z_launch_b(const fft3_args &a, int nz, rect_z_kernel k, hipStream_t stream) {
  switch (nz) {
    INQAMD_RECT_Z_B(INQAMD_RECT_Z_CASE)
    default: return false;
  }
}

}  // namespace inqamd
