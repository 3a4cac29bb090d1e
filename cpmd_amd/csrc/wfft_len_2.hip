// Transform passes of the lengths below (compile-time engines; see wfft_passes.h)
#include "wfft_passes.h"

namespace mc {

template struct Passes<double, 128>;
template struct Passes<float, 128>;
template struct Passes<double, 192>;
template struct Passes<float, 192>;

}  // namespace mc
