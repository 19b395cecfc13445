// Hash aggregation kernels that store their tables, 4-byte keys.
#include "eg_hash_launch_impl.hpp"

namespace eg {
template HashLaunch prepare_hash_agg<4, true>(bool, const HashTuning&, int64_t, const AggSpec&, const HashLayout&,
                                              bool);
}  // namespace eg
