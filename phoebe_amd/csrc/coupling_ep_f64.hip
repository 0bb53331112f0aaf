// F64 instantiation of the split last stage's epilogue (sep_epilogue.hpp).
#include "sep_epilogue.hpp"

namespace phx {
template void launch_ep2<double>(EpParams, int, int, bool, hipStream_t);
}  // namespace phx
