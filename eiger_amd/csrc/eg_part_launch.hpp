// eg_part_launch.hpp -- launch of the partition unit kernel: one translation
// unit instantiates it per key width and row layout (part_agg_*.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "eg_agg_kernels.hpp"
#include "eg_internal.hpp"

namespace eg {

// The unit kernel (specialised for the request once that is compiled) over
// `nunits` units of the partitioned columns; GATHER: values through the row
// ids `perm`.
template <int KB, bool GATHER>
void launch_part_agg(const KeyDesc& key, const AggSpec& spec, const int64_t* perm, const agg::Unit* units, int nunits,
                     const GTable& gt, const OutSpec& os, const agg::OutClaims& claims, int64_t capacity, int cr,
                     size_t lds, int block, int64_t rows, hipStream_t s);

}  // namespace eg
