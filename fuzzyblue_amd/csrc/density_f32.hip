// density_f32.hip — the scattering density kernels of FP32 mode.
#include "density.hpp"

namespace fbk {
template struct DensityLaunch<float>;
}  // namespace fbk
