// Transform passes of the lengths below (compile-time engines; see wfft_passes.h)
#include "wfft_passes.h"

namespace mc {

template struct Passes<double, 224>;
template struct Passes<float, 224>;
template struct Passes<double, 240>;
template struct Passes<float, 240>;

}  // namespace mc
