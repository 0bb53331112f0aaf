// F64 instantiation of the coupling kernels (coupling_kernel.hpp).
#include "coupling_kernel.hpp"

namespace phx {
template void launch_separable_zy<double>(const SepParams&, int, hipStream_t, bool);
template bool launch_separable_x<double>(const SepParams&, const CoupParams&, bool, hipStream_t, hipEvent_t,
                                                  const EpFork&);
}  // namespace phx
