// Transform passes of the lengths below (compile-time engines; see wfft_passes.h)
#include "wfft_passes.h"

namespace mc {

template struct Passes<double, 100>;
template struct Passes<float, 100>;
template struct Passes<double, 108>;
template struct Passes<float, 108>;
template struct Passes<double, 120>;
template struct Passes<float, 120>;
template struct Passes<double, 144>;
template struct Passes<float, 144>;
template struct Passes<double, 150>;
template struct Passes<float, 150>;
template struct Passes<double, 160>;
template struct Passes<float, 160>;

}  // namespace mc
