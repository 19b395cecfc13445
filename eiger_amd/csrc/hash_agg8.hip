// Hash aggregation kernels that flush with atomics, 8-byte keys.
#include "eg_hash_launch_impl.hpp"

namespace eg {
template HashLaunch prepare_hash_agg<8, false>(bool, const HashTuning&, int64_t, const AggSpec&, const HashLayout&, bool);
template void launch_hash_agg<8>(const HashLaunch&, const KeyDesc&, int64_t, const AggSpec&, const GTable&,
                                  const HashLayout&, unsigned long long*, hipStream_t);
}  // namespace eg
