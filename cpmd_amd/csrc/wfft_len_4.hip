// Transform passes of the lengths below (compile-time engines; see wfft_passes.h)
#include "wfft_passes.h"

namespace mc {

template struct Passes<double, 60>;
template struct Passes<float, 60>;
template struct Passes<double, 64>;
template struct Passes<float, 64>;
template struct Passes<double, 72>;
template struct Passes<float, 72>;
template struct Passes<double, 80>;
template struct Passes<float, 80>;
template struct Passes<double, 90>;
template struct Passes<float, 90>;
template struct Passes<double, 96>;
template struct Passes<float, 96>;

}  // namespace mc
