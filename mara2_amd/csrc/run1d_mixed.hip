// run1d_mixed.hip -- runs of 1-D blocks on chip (run1d.hpp) with the mixed
// form's binary32 fluxes, compiled with contraction like mixed.hip.
#include "run1d.hpp"

namespace mara {
namespace run1d {
void launch_f32(const Args& a) { launch<float>(a); }
void courant_f32(const Args& a) { launch_courant<float>(a); }
} // namespace run1d
} // namespace mara
