// hash_groupby.hip -- hash-based group-by for MI355X (gfx950).
//
// Replaces gamax::groupby::hash::groupby (operators/groupby/groupby_hash.cu:302-426).
// The reference builds dense group ids with a cuco static_set of row indices,
// then runs a second pass of per-row global atomics (compute_groupid_kernel
// :48-75, compute_aggregation :77-99).  Here one streaming pass does both:
//
//   1. hash_agg_kernel: a persistent grid, one workgroup per CU slot.  Each
//      workgroup keeps private open-addressing tables in LDS holding the
//      encoded key and every aggregation state inline.  For small group counts
//      the table is replicated R times (R up to 64) and lane l uses replica
//      l mod R, so lanes of a wave never collide on one LDS address; the
//      replicas are merged in LDS before the flush.  Rows are read with
//      16-byte vector loads, four consecutive rows per lane, and the next
//      tile is loaded while the current one is aggregated.  A row that
//      cannot find a slot within `probe_limit` probes spills to the HBM
//      table.  Hot keys (many lanes of a wave on one group) are combined by
//      the wave first (eg_atomics.hpp) so one atomic per state is issued.
//      The finished table goes into the HBM table with atomics, or, where
//      that would cost more (store_pays), is stored as it stands.
//   2. hash_merge_kernel, after stored tables: combines the same slots of
//      every workgroup's table and adds the result to the HBM table.
//   3. hash_compact_kernel: scans the HBM table and writes the final key and
//      output columns at wave-aggregated positions.
//
// Up to 4096 rows one workgroup does all of it in one launch, straight to the
// outputs (hash_tiny_kernel).
//
// The HBM table stores slots of W = 2^k 64-bit words [enc key | states...]
// (AoS, so a random update touches one cache line).  The all-zero word is
// "empty" for keys and the identity of every state, so the table is cleared
// with a plain zero fill.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <type_traits>
#include <vector>

#include "eg_agg_kernels.hpp"
#include "eg_atomics.hpp"
#include "eg_device.hpp"
#include "eg_hash_launch.hpp"
#include "eg_hash_table.hpp"
#include "eg_internal.hpp"
#include "eg_lds_table.hpp"

namespace eg {
namespace {

using namespace lds;

__global__ __launch_bounds__(agg::kMergeBlock) void hash_merge_kernel(const unsigned long long* priv, int nb, int cr,
                                                                     AggSpec spec, GTable gt, int key8)
{
    agg::table_merge(priv, nb, cr, spec, gt, key8 != 0);
}

// Groups at indices from `capacity` on are not written (the caller sees the
// count and re-runs the compaction with room for them).
template <int R>
__global__ __launch_bounds__(256) void hash_compact_kernel(GTable gt, OutSpec os, unsigned long long* counter,
                                                           int64_t capacity)
{
    __shared__ unsigned long long sh[17];
    compact_groups<R>(gt, counter, sh, [&](int64_t idx, uint64_t enc, const unsigned long long* st) {
        if (idx < capacity) dev::emit_group(os, idx, enc, st, 1);
    });
}

// Compaction of gt into os from *counter on (grid and slots per thread by size).
void launch_compact(const GTable& gt, const OutSpec& os, unsigned long long* counter, hipStream_t s,
                    int64_t capacity = INT64_MAX)
{
    const DeviceInfo& di = device_info();
    const uint64_t total = gt.mask + 2;
    const bool wide = total >= kCompactWideSlots;
    const int64_t per = 256 * (wide ? kCompactSlots : 1);
    const int64_t grid = std::max<int64_t>(1, std::min<int64_t>((int64_t)((total + per - 1) / per), (int64_t)di.num_cus * 8));
    KernelTimer timer("hash_compact", s);
    if (wide)
        hipLaunchKernelGGL(hash_compact_kernel<kCompactSlots>, dim3((unsigned)grid), dim3(256), 0, s, gt, os, counter,
                           capacity);
    else hipLaunchKernelGGL(hash_compact_kernel<1>, dim3((unsigned)grid), dim3(256), 0, s, gt, os, counter, capacity);
    EG_LAUNCH_CHECK();
}

// Whether the workgroups' tables are better stored and merged than flushed
// with atomics.  A flush costs one atomic per state for each group a block
// holds, serialised across the blocks on the groups' lines; storing costs the
// merge's launch (5 us) and 2-8% of the row loop, whose kernel is the slower
// one.  Measured on both sides, two and five states, us flushed / stored:
// 2^16 rows, 200 groups 45/48, 400 54/50; 2^18, 64 47/48, 128 51/49;
// 2^20, 16 52/49, 1000 306/60; 2^26, 64 248/244, 128 274/246; 2^28 (five
// states), 16 766/832, 200 789/796, 400 891/808.  Above two value columns a
// block has half the threads: 2^26 rows, 12 states, 100 groups 1025/1100.
// Below 16 blocks a flush meets little: 16,000 rows of unknown groups, ten of
// them 42/47, 1000 of them 57/63.
bool store_pays(int64_t rows, int64_t groups, int nvcols)
{
    const int64_t tile = nvcols <= 2 ? 4096 : 2048;
    const int64_t tiles = (rows + tile - 1) / tile;
    const int64_t blocks = std::min<int64_t>(tiles, device_info().num_cus);
    return blocks >= 16 && blocks * groups >= 5000 + tiles;
}

// The aggregation of n rows into gt.  `scratch` (optional): where the blocks'
// tables are stored, allocated here; without it (callers that must not
// allocate), or without room for it, every block flushes into gt with atomics.
// use_jit: take the specialised kernel once it is loaded (loading a module
// allocates device memory for its code, so callers that must not allocate pass
// false and always run the generic kernel).
template <int KB>
void aggregate(bool vec, const HashTuning& t, const KeyDesc& key, int64_t n, const AggSpec& spec, const GTable& gt,
               const HashLayout& L, hipStream_t s, bool use_jit, DevBuf* scratch)
{
    if (scratch && L.cr > 0) {
        const HashLaunch h = prepare_hash_agg<KB, true>(vec, t, n, spec, L, use_jit);
        try {
            *scratch = DevBuf((size_t)h.grid * (size_t)(1 + spec.nops) * (L.cr + 1) * 8, s);
        } catch (const std::bad_alloc&) {
            // no room (a small memory pool): flush with atomics
        }
        if (unsigned long long* priv = scratch->get<unsigned long long>()) {
            launch_hash_agg<KB>(h, key, n, spec, gt, L, priv, s);
            const int grid = (L.cr + 1 + agg::kMergeSlots - 1) / agg::kMergeSlots;
            const size_t lds = (size_t)lds_table_words(spec.nops, agg::kMergeCr, 0, 8) * 8;
            if (enable_dynamic_lds((const void*)hash_merge_kernel) < lds) raise(EG_ERR_DEVICE, "hash merge: LDS");
            KernelTimer timer("hash_merge", s);
            hipLaunchKernelGGL(hash_merge_kernel, dim3((unsigned)grid), dim3(agg::kMergeBlock), lds, s,
                               (const unsigned long long*)priv, (int)h.grid, L.cr, spec, gt, KB == 8 ? 1 : 0);
            EG_LAUNCH_CHECK();
            return;
        }
    }
    const HashLaunch h = prepare_hash_agg<KB, false>(vec, t, n, spec, L, use_jit);
    launch_hash_agg<KB>(h, key, n, spec, gt, L, nullptr, s);
}

bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

}  // namespace

HashLayout plan_hash_layout(int nops, int key_bytes, int64_t group_bound, int64_t expected, const HashTuning& t)
{
    const DeviceInfo& di = device_info();
    HashLayout L;
    auto bytes_of = [&](int cr_log2, int rep_log2) {
        return (size_t)lds::lds_table_words(nops, 1 << cr_log2, rep_log2, key_bytes) * 8;
    };
    const size_t budget = (size_t)di.max_lds;
    // replicas: the most (<= 64) that still give every replica >= 2x the group bound
    int best_c = -1, best_r = 0;
    for (int rl = 6; rl >= 0; --rl) {
        if (t.replicas > 0 && (1 << rl) > t.replicas) continue;
        int cl = -1;
        for (int c = 14; c >= 4; --c)
            if (bytes_of(c, rl) <= budget && (t.lds_slots == 0 || ((1 << c) << rl) <= t.lds_slots)) {
                cl = c;
                break;
            }
        if (cl < 0) continue;
        if (rl == 0 || (int64_t)(1 << cl) >= 2 * group_bound) {
            best_c = cl;
            best_r = rl;
            break;
        }
    }
    if (best_c >= 0 && group_bound <= (int64_t)t.lds_max_ratio * ((int64_t)1 << best_c)) {
        L.cr = 1 << best_c;
        L.rep_log2 = best_r;
        if (best_r == 0) {
            // one table: every multiple of four slots the LDS holds (a larger
            // table keeps more of the keys that arrive, and fewer rows spill)
            auto bytes_cr = [&](int cr) { return (size_t)lds::lds_table_words(nops, cr, 0, key_bytes) * 8; };
            const int cap = t.lds_slots > 0 ? t.lds_slots : (1 << 14);
            while (L.cr + 4 <= cap && bytes_cr(L.cr + 4) + 1024 <= budget) L.cr += 4;  // 1 KB for static LDS
        }
        L.lds_bytes = (size_t)lds::lds_table_words(nops, L.cr, L.rep_log2, key_bytes) * 8;
    }
    // A table much smaller than the group count still catches the hot keys
    // (they arrive early); keep the probing short so cold rows spill cheaply.
    const int64_t slots = std::max(L.cr, 1);
    L.probe_limit = expected > 4 * slots ? 2 : expected > slots ? 4 : 16;
    L.peel_min = t.peel_min;
    return L;
}

int hash_lds_slots(int nops, int key_bytes)
{
    static std::atomic<int> known[2][kMaxOps + 1];  // the same on every device of one architecture
    nops = std::min(std::max(nops, 1), kMaxOps);
    std::atomic<int>& slots = known[key_bytes == 8 ? 1 : 0][nops];
    if (slots == 0) slots = plan_hash_layout(nops, key_bytes, (int64_t)1 << 30, 0, HashTuning{}).cr;
    return slots;
}

// ---- tiny inputs ---------------------------------------------------------------
// A whole group-by in one workgroup and one launch: up to kTinyRows rows, four
// a thread, into an LDS table that has room for every row being its own group;
// the groups go straight to the outputs and their count to pinned host memory.
// The general path's launches (fill, one-block aggregation of an LDS-wide
// table, compaction, copy) take 29 us for 3000 rows, this kernel 9.
namespace {
constexpr int kTinyRows = 4096;
constexpr int kTinyBlock = 1024;

template <int KB, int NV>
__global__ __launch_bounds__(kTinyBlock) void hash_tiny_kernel(KeyDesc key, int n, AggSpec spec, OutSpec os, int cr,
                                                               int peel_min, int64_t* count)
{
    constexpr int J = kTinyRows / kTinyBlock;
    using KT = typename LdsKey<KB>::T;
    extern __shared__ __align__(16) unsigned long long smem[];
    __shared__ uint32_t wsum[kTinyBlock / 64];
    const int t = threadIdx.x, lane = dev::lane_id();
    LdsTable<KB, true> tab(smem, spec.nops, cr, 0);
    uint64_t k[J], raw[J][NV];
    bool valid[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int r = j * kTinyBlock + t;
        valid[j] = r < n;
        k[j] = valid[j] ? (KB == 4 ? (uint64_t)((const uint32_t*)key.data)[r] : ((const uint64_t*)key.data)[r]) : 0ull;
    }
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        if (c >= spec.nvcols) break;
        const void* p = spec.cols[c].data;
        auto column = [&](auto w) {  // the width switched on once per column
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const int r = j * kTinyBlock + t;
                raw[j][c] = valid[j] ? dev::load_raw(p, decltype(w)::value, r) : 0ull;
            }
        };
        switch (spec.cols[c].bytes) {
        case 1: column(std::integral_constant<int, 1>{}); break;
        case 2: column(std::integral_constant<int, 2>{}); break;
        case 4: column(std::integral_constant<int, 4>{}); break;
        default: column(std::integral_constant<int, 8>{}); break;
        }
    }
    const int words = LdsTable<KB>::words(spec.nops, cr, 0);
    for (int i = t; i < words; i += kTinyBlock) smem[i] = 0ull;
    __syncthreads();
    dev::HotTags hot;
#pragma unroll
    for (int j = 0; j < J; ++j) {
        if (j * kTinyBlock >= n) break;  // uniform
        uint64_t cv[NV];
#pragma unroll
        for (int c = 0; c < NV; ++c) cv[c] = c < spec.nvcols ? dev::canon(raw[j][c], spec.cols[c].conv) : 0ull;
        // never spills: the table has more slots than rows and every one is probed
        lds_row<dev::RtOps, KB, NV>(tab, true, 0, lane, key, spec, k[j], cv, valid[j], cr, peel_min, hot);
    }
    __syncthreads();
    uint32_t mine = 0;  // this thread's groups, in slots t, t + kTinyBlock, ...
    auto slot_key = [&](int sl, KT& kw) {
        kw = 0;
        if (sl < cr) {
            kw = tab.keys[sl];
            return kw != 0;
        }
        return sl == cr && tab.side[0] != 0ull;
    };
    for (int sl = t; sl <= cr; sl += kTinyBlock) {
        KT kw;
        mine += slot_key(sl, kw) ? 1u : 0u;
    }
    uint32_t at = dev::block_excl_scan<kTinyBlock>(mine, wsum);
    if (t == kTinyBlock - 1) *count = (int64_t)(at + mine);
    for (int sl = t; sl <= cr; sl += kTinyBlock) {
        KT kw;
        if (!slot_key(sl, kw)) continue;
        dev::emit_group(os, (int64_t)at, lds_to_enc64<KB>(kw, key.is_signed), tab.st + sl, (int64_t)tab.T);
        ++at;
    }
}

// LDS slots of a tiny table: a quarter more than the rows, whole buckets.
int tiny_slots(int64_t n) { return (int)(((n + n / 4 + 8) + kBucket - 1) / kBucket * kBucket); }

template <int KB>
bool run_tiny(const Plan& plan, const HashTuning& t, hipStream_t s, Result& res)
{
    const int nv = plan.spec.nvcols;
    auto kern = nv <= 1 ? hash_tiny_kernel<KB, 1> : nv <= 2 ? hash_tiny_kernel<KB, 2> : hash_tiny_kernel<KB, kMaxVCols>;
    const int cr = tiny_slots(plan.rows);
    const size_t lds = (size_t)lds_table_words(plan.spec.nops, cr, 0, KB) * 8;
    if (enable_dynamic_lds((const void*)kern) < lds) return false;
    OutSpec os;
    alloc_outputs(plan, plan.rows, s, res, os);
    int64_t* count = pinned_i64(1);
    KernelTimer timer("hash_agg", s);
    hipLaunchKernelGGL(kern, dim3(1), dim3(kTinyBlock), lds, s, plan.key, (int)plan.rows, plan.spec, os, cr, t.peel_min,
                       count);
    EG_LAUNCH_CHECK();
    EG_HIP(hipStreamSynchronize(s));
    res.num_groups = *(volatile int64_t*)count;
    return true;
}
}  // namespace

// Group bounds up to which run_hash allocates the outputs before it reads
// the group count (at most 40 bytes a group for the benchmark's requests).
constexpr int64_t kEarlyOutputRows = (int64_t)1 << 22;

Result run_hash(const Plan& plan, int64_t group_bound, int64_t expected, bool callers, hipStream_t s, const HashTuning& t)
{
    const int64_t n = plan.rows;
    const int nops = plan.spec.nops;
    const int W = table_words_per_slot(nops);
    const int KB = plan.key.bytes;
    if (n <= kTinyRows) {
        Result res;
        if (KB == 4 ? run_tiny<4>(plan, t, s, res) : run_tiny<8>(plan, t, s, res)) return res;
    }
    // A caller's bound is the better guess of whether the keys outnumber the LDS
    // slots: the estimate is short of skewed ones (2^28 rows, five states, 4096
    // groups and bound at Zipf 1.2 2.57 -> 2.08 ms; uniform 7.43 -> 7.8).  A
    // bound made of the estimate has its headroom on top (2^26 rows, 16 states,
    // 1000 groups 1.06 ms by the estimate, 2.34 by the bound).
    const HashLayout L = plan_hash_layout(nops, KB, group_bound, callers ? group_bound : std::min(group_bound, expected), t);

    bool vec = aligned16(plan.key.data);
    for (int c = 0; c < plan.spec.nvcols; ++c) vec = vec && aligned16(plan.spec.cols[c].data);

    int64_t bound = std::max<int64_t>(1, std::min<int64_t>(group_bound, n));
    expected = std::max<int64_t>(1, std::min(expected, bound));
    int64_t slots = t.table_slots > 0 ? t.table_slots : 1024;
    while (slots < 2 * bound) slots <<= 1;

    // With a modest bound the outputs are allocated for it before the table is
    // read, and the compaction runs right after the aggregation: one
    // synchronisation per call instead of two (a bound the groups exceed
    // costs one more compaction into exact outputs).
    const bool early = bound <= kEarlyOutputRows;
    for (;;) {
        HbmTable ht(slots, W, s);
        // before the stored tables, which take only room that is left
        Result eres;
        OutSpec eos;
        if (early) alloc_outputs(plan, bound, s, eres, eos);
        DevBuf scratch;
        // above twice the LDS slots the tables hold different keys and flush (3M
        // rows in 400k groups 329 us, 622 stored and merged)
        DevBuf* stored = expected <= 2 * (int64_t)L.cr && store_pays(n, expected, plan.spec.nvcols) ? &scratch : nullptr;
        if (KB == 4) aggregate<4>(vec, t, plan.key, n, plan.spec, ht.gt, L, s, true, stored);
        else aggregate<8>(vec, t, plan.key, n, plan.spec, ht.gt, L, s, true, stored);
        if (early) launch_compact(ht.gt, eos, ht.gt.meta + 3, s, bound);  // meta[3]: zeroed with the table
        int64_t meta[3];
        ht.read_meta(meta, s);
        scratch = DevBuf();  // for the outputs allocated below, or the retry's table
        if (meta[2] != 0) {
            // The table filled up: the group bound was too small.  Retry with a
            // table sized for every row being its own group.
            if (slots >= 2 * n) raise(EG_ERR_CAPACITY, "hash table overflow");
            timing_count("hash_retry");
            int64_t ns = slots;
            while (ns < 2 * n) ns <<= 1;
            slots = ns;
            continue;
        }
        const int64_t groups = meta[0] + (meta[1] != 0 ? 1 : 0);
        if (early && groups <= bound) {
            eres.num_groups = groups;
            return eres;  // read_meta synchronised after the compaction
        }
        Result res;
        OutSpec os;
        alloc_outputs(plan, groups, s, res, os);
        if (groups > 0) {
            DevBuf counter(8, s);
            fill_zero(counter.get(), 8, s);
            ht.compact(os, counter.get<unsigned long long>(), s);
        }
        EG_HIP(hipStreamSynchronize(s));
        return res;
    }
}

// ---- no-allocation variant ---------------------------------------------------------
// The HBM table of run_hash_noalloc lives in this array: one copy per device,
// loaded with the module and held until the process ends.  Host code never
// passes the array's name to a kernel (on the host it only stands for the
// symbol); it uses the device address that hipGetSymbolAddress returns for
// the current device, looked up once per device.
namespace {
__device__ __align__(256) unsigned long long scratch[kNoAllocScratchBytes / 8];

unsigned long long* scratch_ptr()
{
    static std::mutex mu;
    static std::vector<void*> ptrs;
    int dev = 0;
    EG_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(mu);
    if ((size_t)dev >= ptrs.size()) ptrs.resize((size_t)dev + 1, nullptr);
    if (!ptrs[(size_t)dev]) {
        void* p = nullptr;
        EG_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) raise(EG_ERR_DEVICE, "no device address for the group-by scratch");
        ptrs[(size_t)dev] = p;
    }
    return static_cast<unsigned long long*>(ptrs[(size_t)dev]);
}
}  // namespace

int64_t run_hash_noalloc(const Plan& plan, int64_t group_bound, const OutSpec& os, int64_t capacity, hipStream_t s)
{
    const int64_t n = plan.rows;
    const int nops = plan.spec.nops;
    const int W = table_words_per_slot(nops);
    const int KB = plan.key.bytes;
    const HashTuning t;
    const HashLayout L = plan_hash_layout(nops, KB, group_bound, group_bound, t);
    bool vec = aligned16(plan.key.data);
    for (int c = 0; c < plan.spec.nvcols; ++c) vec = vec && aligned16(plan.spec.cols[c].data);

    // table: slots * W words, then the side slot (W words) and 4 meta words;
    // meta[3] is the compaction's output counter
    const size_t max_words = kNoAllocScratchBytes / 8;
    auto words_of = [&](int64_t slots) { return (size_t)slots * (size_t)W + (size_t)W + 4; };
    const int64_t bound = std::max<int64_t>(1, std::min<int64_t>(group_bound, n));
    int64_t slots = 1024;
    while (slots < 2 * bound) slots <<= 1;
    if (words_of(slots) > max_words)
        raise(EG_ERR_CAPACITY, "groups_upper_bound " + std::to_string(group_bound) + " needs a table of " +
                                   std::to_string(words_of(slots) * 8) + " bytes, above the " +
                                   std::to_string(kNoAllocScratchBytes) + "-byte no-allocation scratch");
    int64_t max_slots = slots;
    while (words_of(max_slots * 2) <= max_words) max_slots <<= 1;

    unsigned long long* base = scratch_ptr();
    for (;;) {
        GTable gt;
        gt.base = base;
        gt.side = base + (size_t)slots * W;
        gt.meta = gt.side + W;
        gt.mask = (uint64_t)slots - 1;
        gt.W = W;
        fill_zero(base, words_of(slots) * 8, s);  // a kernel: every call starts from an empty table
        if (KB == 4) aggregate<4>(vec, t, plan.key, n, plan.spec, gt, L, s, false, nullptr);
        else aggregate<8>(vec, t, plan.key, n, plan.spec, gt, L, s, false, nullptr);
        int64_t meta[3] = {0, 0, 0};
        EG_HIP(hipMemcpyAsync(meta, gt.meta, sizeof meta, hipMemcpyDeviceToHost, s));
        EG_HIP(hipStreamSynchronize(s));
        if (meta[2] != 0) {
            // more groups than the bound said: once more with the largest
            // table the scratch holds
            if (slots < max_slots) {
                slots = max_slots;
                continue;
            }
            raise(EG_ERR_CAPACITY, "more groups than the no-allocation scratch's table holds (" +
                                       std::to_string(slots / 2) + " at load 1/2)");
        }
        const int64_t groups = meta[0] + (meta[1] != 0 ? 1 : 0);
        if (groups > capacity)
            raise(EG_ERR_CAPACITY, std::to_string(groups) + " groups exceed the output capacity of " +
                                       std::to_string(capacity) + " rows");
        if (groups > 0) {
            launch_compact(gt, os, gt.meta + 3, s);
        }
        EG_HIP(hipStreamSynchronize(s));
        return groups;
    }
}

// ---- HbmTable ---------------------------------------------------------------------
int table_words_per_slot(int nops)
{
    int p = 1;
    while (p < 1 + nops) p <<= 1;
    return p;
}

HbmTable::HbmTable(int64_t slots, int W, hipStream_t s, int64_t extra_words)
    : buf((size_t)(slots * W + W + 4 + extra_words) * 8, s)
{
    const size_t words = (size_t)(slots * W + W + 4 + extra_words);
    fill_zero(buf.get(), words * 8, s);
    gt.base = buf.get<unsigned long long>();
    gt.side = gt.base + (size_t)slots * W;
    gt.meta = gt.side + W;
    gt.mask = (uint64_t)slots - 1;
    gt.W = W;
    extra = extra_words > 0 ? gt.meta + 4 : nullptr;
}

void HbmTable::read_meta(int64_t* out3, hipStream_t s)
{
    int64_t* h = pinned_i64(4);
    EG_HIP(hipMemcpyAsync(h, gt.meta, 3 * sizeof(int64_t), hipMemcpyDeviceToHost, s));
    EG_HIP(hipStreamSynchronize(s));
    out3[0] = h[0];
    out3[1] = h[1];
    out3[2] = h[2];
}

void HbmTable::compact(const OutSpec& os, unsigned long long* counter, hipStream_t s)
{
    launch_compact(gt, os, counter, s);
}

}  // namespace eg
