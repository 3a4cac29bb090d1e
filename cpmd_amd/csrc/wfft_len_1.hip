// Transform passes of the lengths below (compile-time engines; see wfft_passes.h)
#include "wfft_passes.h"

namespace mc {

template struct Passes<double, 16>;
template struct Passes<float, 16>;
template struct Passes<double, 18>;
template struct Passes<float, 18>;
template struct Passes<double, 24>;
template struct Passes<float, 24>;
template struct Passes<double, 30>;
template struct Passes<float, 30>;
template struct Passes<double, 32>;
template struct Passes<float, 32>;
template struct Passes<double, 36>;
template struct Passes<float, 36>;
template struct Passes<double, 40>;
template struct Passes<float, 40>;
template struct Passes<double, 48>;
template struct Passes<float, 48>;
template struct Passes<double, 54>;
template struct Passes<float, 54>;

}  // namespace mc
