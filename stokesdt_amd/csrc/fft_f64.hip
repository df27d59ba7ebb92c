// Two-stage transforms of the SPME meshes, double instances.
#include <algorithm>
#include "fft_kernels.hpp"

namespace sdt {

template struct Fft2Launch<double>;

}  // namespace sdt
