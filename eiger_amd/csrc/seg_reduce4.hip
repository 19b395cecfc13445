// Segmented reduction, 4-byte keys.
#include "eg_seg_launch_impl.hpp"

namespace eg {
template void launch_seg<4, kMaxOps>(const SegArgs&, int, const AggSpec&, const OutSpec&, hipStream_t);
}  // namespace eg
