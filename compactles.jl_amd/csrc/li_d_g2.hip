// Explicit instantiation: double line operators, q=2 M=4 sym=0.
#include "cles_line.hpp"

namespace cles {
template void launch_epi<double, 2, 4, 0>(const HostPlan &, int, const View3 &, const double *, const EpiArgs &,
                                            hipStream_t, const LineFields &, const HostPlan *);
}  // namespace cles
