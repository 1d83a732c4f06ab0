// density_f64.hip — the scattering density kernels of precision mode.
#include "density.hpp"

namespace fbk {
template struct DensityLaunch<double>;
}  // namespace fbk
