// Partition unit kernels: 4-byte keys, partitioned columns.
#include "eg_part_launch_impl.hpp"

namespace eg {
template void launch_part_agg<4, false>(const KeyDesc&, const AggSpec&, const int64_t*, const agg::Unit*, int, const GTable&,
                                       const OutSpec&, const agg::OutClaims&, int64_t, int, size_t, int, int64_t,
                                       hipStream_t);
}  // namespace eg
