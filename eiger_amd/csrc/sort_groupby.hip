// sort_groupby.hip -- sort-based group-by (gamax::groupby::sort::groupby and
// groupby_gfur, operators/groupby/groupby_sort.cu:346-479).
//
// The reference sorts (key, value) pairs once per aggregation request and runs
// cub::DeviceReduce::ReduceByKey per request (groupby_sort.cu:32-78,
// 363-419).  Here:
//   1. key_range: min/max of the radix-ordered keys; only the bits of
//      (key - min) are sorted, so dense keys take few passes (the reference
//      only narrows the bit range under hint.zero_based_ids,
//      groupby_sort.cu:222-246; the range here is exact and always applies).
//   2. one LSD radix sort carrying every value column (SORT) or the row ids
//      (SORT_GFUR: values are gathered through the permutation, like the
//      reference's permutation_iterator, groupby_sort.cu:429-479);
//   3. a segmented reduction that computes every aggregation in one pass:
//      seg_heads_kernel counts group heads per tile, a scan gives each
//      tile its first group index, and seg_reduce_kernel folds each lane's
//      consecutive rows in registers, merges runs that cross lanes through LDS
//      states, writes the tile's complete groups and hands the group that
//      crosses into the next tile to seg_tail_kernel through a per-tile
//      boundary state.
// Output rows are in ascending key order, as in the reference.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "eg_device.hpp"
#include "eg_internal.hpp"
#include "eg_lds_table.hpp"
#include "eg_radix.hpp"
#include "eg_seg_launch.hpp"

namespace eg {
namespace {

using namespace lds;

// Group heads of one tile of T = kSegB * ITEMS sorted rows: thread t takes
// rows t, t + kSegB, ... of the tile, so a wave's loads are consecutive (a
// lane walking its own ITEMS rows made every load 64 cache lines: 40M int64
// keys took 768 us).
template <int ITEMS, int KB>
__global__ __launch_bounds__(kSegB) void seg_heads_kernel(const void* __restrict__ keys, int64_t n, uint32_t* heads)
{
    const int64_t base = (int64_t)blockIdx.x * (kSegB * ITEMS) + threadIdx.x;
    auto key_at = [&](int64_t r) -> uint64_t {
        return KB == 4 ? (uint64_t)((const uint32_t*)keys)[r] : ((const uint64_t*)keys)[r];
    };
    uint64_t k[ITEMS], p[ITEMS];
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int64_t r = base + (int64_t)i * kSegB;
        k[i] = r < n ? key_at(r) : 0ull;
        p[i] = r < n && r > 0 ? key_at(r - 1) : 0ull;
    }
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int64_t r = base + (int64_t)i * kSegB;
        c += r < n && (r == 0 || k[i] != p[i]) ? 1u : 0u;
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) c += __shfl_xor(c, off);
    __shared__ uint32_t ws[4];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) heads[blockIdx.x] = ws[0] + ws[1] + ws[2] + ws[3];
}

// Writes the groups that continue past the tile of their head (one lane per
// tile).  A group that covers the first tile of later spans has a partial
// state at each of those: the wave collects them.  Such a group covers all
// tiles from its head's to the next span's first, so a wave's 64 tiles hold
// the head of at most one.
__global__ void seg_tail_kernel(uint32_t ntiles, const uint32_t* head_off, unsigned long long* bstate,
                                const unsigned long long* bkey, const uint32_t* btrail, AggSpec spec, int kb,
                                int is_signed, OutSpec os)
{
    const int nops = spec.nops;
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const bool trail = t < ntiles && btrail[t] != 0u;
    const uint32_t groups = trail ? head_off[t + 1] : 0u;  // this one is the last of them
    const uint32_t next = (t & ~(kSegSpan - 1u)) + kSegSpan;
    const bool spans = trail && next < ntiles && head_off[next + 1] == groups;
    if (const uint64_t m = __ballot(spans)) {
        const int src = __ffsll((unsigned long long)m) - 1;
        const uint32_t g = __shfl(groups, src), first = __shfl(next, src);
        for (int a = 0; a < nops; ++a) {
            const int32_t cls = dev::class_of(spec, a);
            uint64_t v = 0ull;
            int have = 0;
            for (uint64_t s = first + (uint64_t)lane * kSegSpan; s < ntiles && head_off[s + 1] == g; s += 64 * kSegSpan) {
                const uint64_t x = bstate[(size_t)s * nops + a];
                v = have ? dev::combine(cls, v, x) : x;
                have = 1;
            }
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) {
                const uint64_t x = __shfl_down((unsigned long long)v, off);
                const int other = __shfl_down(have, off);
                if (lane + off < 64 && other) {
                    v = have ? dev::combine(cls, v, x) : x;
                    have = 1;
                }
            }
            v = __shfl((unsigned long long)v, 0);
            if (lane == src) {
                unsigned long long* dst = bstate + (size_t)t * nops + a;
                *dst = dev::combine(cls, *dst, v);
            }
        }
    }
    if (trail)
        dev::emit_group(os, (int64_t)groups - 1, dev::enc64(dev::widen_key(bkey[t], kb, is_signed)),
                        bstate + (size_t)t * nops, (int64_t)1);
}

}  // namespace

// Segmented reduction of rows already ordered by key (equal keys adjacent):
// writes every group into freshly allocated outputs.  perm: optional row
// gather for the value columns (GFUR).
Result reduce_sorted(const Plan& plan, const void* sorted_keys, const AggSpec& spec, const int64_t* perm,
                     hipStream_t s)
{
    const int64_t n = plan.rows;
    const int kb = plan.key.bytes;
    constexpr int items = kSegItems;
    const int T = kSegB * items;
    const int64_t ntiles64 = (n + T - 1) / T;
    if (ntiles64 >= ((int64_t)1 << 31)) raise(EG_ERR_UNSUPPORTED, "too many rows for the segmented reduction");
    const uint32_t ntiles = (uint32_t)ntiles64;

    DevBuf heads((size_t)(ntiles + 1) * 4, s), head_off((size_t)(ntiles + 1) * 4, s);
    fill_zero(heads.get(), (size_t)(ntiles + 1) * 4, s);
    {
        KernelTimer timer("seg_heads", s);
        auto kern = kb == 4 ? seg_heads_kernel<items, 4> : seg_heads_kernel<items, 8>;
        hipLaunchKernelGGL(kern, dim3(ntiles), dim3(kSegB), 0, s, sorted_keys, n, heads.get<uint32_t>());
        EG_LAUNCH_CHECK();
    }
    // head_off[t] = groups whose head lies before tile t; head_off[ntiles] = G
    const uint64_t groups = scan_exclusive_u32(heads.get<uint32_t>(), head_off.get<uint32_t>(), (int64_t)ntiles + 1, s, true);

    Result res;
    OutSpec os;
    alloc_outputs(plan, (int64_t)groups, s, res, os);
    DevBuf bstate((size_t)ntiles * spec.nops * 8 + 8, s), bkey((size_t)ntiles * 8, s), btrail((size_t)ntiles * 4, s);
    fill_zero(bstate.get(), (size_t)ntiles * spec.nops * 8 + 8, s);
    fill_zero(btrail.get(), (size_t)ntiles * 4, s);
    const int sg = plan.key.is_signed;
    const SegArgs sa{sorted_keys, perm, n, head_off.get<uint32_t>(), ntiles, bstate.get<unsigned long long>(),
                     bkey.get<unsigned long long>(), btrail.get<uint32_t>()};
    const bool few = spec.nops <= kSegFewOps;
    if (kb == 4) (few ? launch_seg<4, kSegFewOps> : launch_seg<4, kMaxOps>)(sa, sg, spec, os, s);
    else (few ? launch_seg<8, kSegFewOps> : launch_seg<8, kMaxOps>)(sa, sg, spec, os, s);
    hipLaunchKernelGGL(seg_tail_kernel, dim3((ntiles + 255) / 256), dim3(256), 0, s, ntiles,
                       (const uint32_t*)head_off.get<uint32_t>(), bstate.get<unsigned long long>(),
                       (const unsigned long long*)bkey.get<unsigned long long>(), (const uint32_t*)btrail.get<uint32_t>(),
                       spec, kb, sg, os);
    EG_LAUNCH_CHECK();
    EG_HIP(hipStreamSynchronize(s));
    return res;
}

Result run_sort(const Plan& plan, const eg_groupby_hint& hint, bool gfur, hipStream_t s)
{
    (void)hint;
    const int64_t n = plan.rows;
    const int kb = plan.key.bytes;
    KeyRange range;
    const RangeCol rc{plan.key.data, plan.key_type, kb};
    key_ranges(&rc, 1, n, s, &range);
    const uint64_t mn = range.min, span = range.max - range.min;
    const int bits = span == 0 ? 0 : 64 - __builtin_clzll(span);
    // low bits that every key shares are zero in key - min: no digit covers them
    const int low = span == 0 ? 0 : __builtin_ctzll(range.varying);

    RadixKeys rk{};
    rk.data = plan.key.data;
    rk.bytes = kb;
    rk.type = plan.key_type;
    rk.mode = DIG_KEY;
    rk.kmin = mn;
    SortBuffers b;
    b.keys_in = plan.key.data;
    DevBuf ka((size_t)n * kb, s), kbuf((size_t)n * kb, s);
    b.keys_a = ka.get();
    b.keys_b = kbuf.get();
    std::vector<DevBuf> bufs;
    AggSpec spec = plan.spec;
    if (gfur) {
        b.pay_in.push_back(Payload{nullptr, nullptr, 8, 1});
        bufs.emplace_back((size_t)n * 8, s);
        bufs.emplace_back((size_t)n * 8, s);
        b.pay_a.push_back(bufs[0].get());
        b.pay_b.push_back(bufs[1].get());
    } else {
        for (int c = 0; c < spec.nvcols; ++c) {
            const int by = spec.cols[c].bytes;
            b.pay_in.push_back(Payload{spec.cols[c].data, nullptr, by, 0});
            bufs.emplace_back((size_t)n * by, s);
            bufs.emplace_back((size_t)n * by, s);
            b.pay_a.push_back(bufs[bufs.size() - 2].get());
            b.pay_b.push_back(bufs[bufs.size() - 1].get());
        }
    }
    const void* sorted_keys = nullptr;
    std::vector<const void*> sorted_pay;
    radix_sort(rk, b, n, low, bits, s, &sorted_keys, sorted_pay);
    const int64_t* perm = nullptr;
    if (gfur) perm = (const int64_t*)sorted_pay[0];
    else
        for (int c = 0; c < spec.nvcols; ++c) spec.cols[c].data = sorted_pay[(size_t)c];
    return reduce_sorted(plan, sorted_keys, spec, perm, s);
}

}  // namespace eg
