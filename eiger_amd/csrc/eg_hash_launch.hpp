// eg_hash_launch.hpp -- launch of the hash aggregation kernel: one translation
// unit instantiates it per key width and ending (hash_agg*.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "eg_agg_kernels.hpp"
#include "eg_hash_table.hpp"
#include "eg_internal.hpp"

namespace eg {

// A chosen kernel and its persistent grid.
struct HashLaunch {
    using Kern = void (*)(KeyDesc, int64_t, AggSpec, GTable, int, int, int, int, unsigned long long*);
    Kern kern = nullptr;          // the generic kernel of the value layout
    hipFunction_t fn = nullptr;   // the specialised one, if it is available
    int block = 0;
    int64_t grid = 0;
};

// Picks the compiled value layout (vector loads for up to two 4/8-byte
// columns on 16-byte aligned data, else typed loads), the specialised kernel
// when use_jit and it is loaded, and the grid.  STORE: the kernel whose blocks
// store their tables instead of flushing them (see agg::flush_lds).
template <int KB, bool STORE>
HashLaunch prepare_hash_agg(bool vec, const HashTuning& t, int64_t n, const AggSpec& spec, const HashLayout& L,
                            bool use_jit);

// priv: room for one stored table per block of h.grid (STORE kernels).
template <int KB>
void launch_hash_agg(const HashLaunch& h, const KeyDesc& key, int64_t n, const AggSpec& spec, const GTable& gt,
                     const HashLayout& L, unsigned long long* priv, hipStream_t s);

}  // namespace eg
