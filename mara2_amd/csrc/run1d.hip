// run1d.hip -- runs of 1-D blocks on chip (run1d.hpp) with binary64 fluxes,
// compiled without contraction.
#include "run1d.hpp"

namespace mara {
namespace run1d {
void launch_f64(const Args& a) { launch<double>(a); }
void courant_f64(const Args& a) { launch_courant<double>(a); }
} // namespace run1d
} // namespace mara
