// Transform passes of the lengths below (compile-time engines; see wfft_passes.h)
#include "wfft_passes.h"

namespace mc {

template struct Passes<double, 162>;
template struct Passes<float, 162>;
template struct Passes<double, 180>;
template struct Passes<float, 180>;
template struct Passes<double, 200>;
template struct Passes<float, 200>;
template struct Passes<double, 216>;
template struct Passes<float, 216>;
template struct Passes<double, 256>;
template struct Passes<float, 256>;

}  // namespace mc
