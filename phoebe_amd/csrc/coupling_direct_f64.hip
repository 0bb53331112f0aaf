// F64 instantiation of the direct coupling transform (coupling_direct.hpp).
#include "coupling_direct.hpp"

namespace phx {
template void launch_coupling<double>(const CoupParams&, bool, hipStream_t);
}  // namespace phx
