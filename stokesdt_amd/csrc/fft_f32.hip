// Two-stage transforms of the SPME meshes, float instances.
#include <algorithm>
#include "fft_kernels.hpp"

namespace sdt {

template struct Fft2Launch<float>;

}  // namespace sdt
