// Segmented reduction, 8-byte keys, few states.
#include "eg_seg_launch_impl.hpp"

namespace eg {
template void launch_seg<8, kSegFewOps>(const SegArgs&, int, const AggSpec&, const OutSpec&, hipStream_t);
}  // namespace eg
