// Transform passes of the lengths below (compile-time engines; see wfft_passes.h)
#include "wfft_passes.h"

namespace mc {

template struct Passes<double, 270>;
template struct Passes<float, 270>;
template struct Passes<double, 288>;
template struct Passes<float, 288>;
template struct Passes<double, 300>;
template struct Passes<float, 300>;
template struct Passes<double, 320>;
template struct Passes<float, 320>;

}  // namespace mc
