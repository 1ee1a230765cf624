// x-y planes of fft3_rect.hpp in workgroups of 1024 threads.
#include "fft3_rect_xy.hpp"

namespace inqamd {

template void rect_xy_launch<1024>(const fft3_args &, const int[3], rect_planes, double *,
                                 hipStream_t);

}  // namespace inqamd
