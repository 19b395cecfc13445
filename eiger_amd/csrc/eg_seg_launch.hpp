// eg_seg_launch.hpp -- launch of the segmented reduction: one translation unit
// instantiates it per key width and number of states (seg_reduce*.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "eg_internal.hpp"
#include "eg_spec.hpp"

namespace eg {

constexpr int kSegB = 256;
// 2048-row tiles: the turned column and five states leave five workgroups a CU.
constexpr int kSegItems = 8;
// Tiles that add to one address when a group covers them all.
constexpr uint32_t kSegSpan = 128;

// Requests of at most this many states take kernels unrolled for that many,
// half the code and 67 instead of 88 registers (40M rows of int64 keys and
// doubles, three states: 1.64 against 1.75 ms a call); others kMaxOps.
constexpr int kSegFewOps = 6;

struct SegArgs {
    const void* keys;
    const int64_t* perm;
    int64_t n;
    const uint32_t* head_off;
    uint32_t ntiles;
    unsigned long long* bstate;
    unsigned long long* bkey;
    uint32_t* btrail;
};

template <int KB, int MO>
void launch_seg(const SegArgs& a, int is_signed, const AggSpec& spec, const OutSpec& os, hipStream_t s);

}  // namespace eg
