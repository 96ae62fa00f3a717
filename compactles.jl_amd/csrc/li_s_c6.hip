// Explicit instantiation: float line operators, q=1 M=2 sym=0.
#include "cles_line.hpp"

namespace cles {
template void launch_epi<float, 1, 2, 0>(const HostPlan &, int, const View3 &, const float *, const EpiArgs &,
                                            hipStream_t, const LineFields &, const HostPlan *);
}  // namespace cles
