// Explicit instantiation: double line operators, q=1 M=4 sym=1.
#include "cles_line.hpp"

namespace cles {
template void launch_epi<double, 1, 4, 1>(const HostPlan &, int, const View3 &, const double *, const EpiArgs &,
                                            hipStream_t, const LineFields &, const HostPlan *);
}  // namespace cles
