// eg_seg_launch_impl.hpp -- the segmented reduction and its launch, included
// by the translation units that instantiate them.
#pragma once

#include <type_traits>

#include "eg_device.hpp"
#include "eg_lds_table.hpp"
#include "eg_seg_launch.hpp"

namespace eg {
namespace {

using namespace lds;

__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* wsum, uint32_t* total)
{
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t y = __shfl_up(x, off);
        if (lane >= off) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    uint32_t add = 0, tot = 0;
    for (int i = 0; i < kSegB / 64; ++i) {
        if (i < w) add += wsum[i];
        tot += wsum[i];
    }
    *total = tot;
    __syncthreads();
    return x - v + add;
}

// Largest tile u with head_off[u] <= g (the tile holding group g's head).
__device__ __forceinline__ uint32_t owner_tile(const uint32_t* head_off, uint32_t ntiles, uint32_t g)
{
    uint32_t lo = 0, hi = ntiles;  // head_off has ntiles + 1 entries
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (head_off[mid] <= g) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Writes group g from states held in registers.
template <int MO>
__device__ __forceinline__ void emit_regs(const OutSpec& os, int64_t g, uint64_t key_enc, const uint64_t (&acc)[MO])
{
    dev::store_bytes(os.key_data, os.key_bytes, g, dev::dec64(key_enc));
    for (int j = 0; j < os.nouts; ++j) {
        const OutDesc& o = os.outs[j];
        uint64_t st[2] = {0ull, 0ull};
#pragma unroll
        for (int a = 0; a < MO; ++a) {
            if (a == o.op) st[0] = acc[a];
            if (a == o.op2) st[1] = acc[a];
        }
        const uint64_t s = st[0];
        switch (o.code) {
        case OUT_U64: dev::store_bytes(o.data, 8, g, s); break;
        case OUT_F32: ((float*)o.data)[g] = (float)__longlong_as_double((long long)s); break;
        case OUT_F64: ((double*)o.data)[g] = __longlong_as_double((long long)s); break;
        case OUT_MAX_I: dev::store_bytes(o.data, o.bytes, g, s ^ dev::kSign64); break;
        case OUT_MIN_I: dev::store_bytes(o.data, o.bytes, g, (~s) ^ dev::kSign64); break;
        case OUT_MAX_U: dev::store_bytes(o.data, o.bytes, g, s); break;
        case OUT_MIN_U: dev::store_bytes(o.data, o.bytes, g, ~s); break;
        case OUT_MAX_F: dev::store_double_as(o.data, o.bytes, g, dev::unord_f64(s)); break;
        case OUT_MIN_F: dev::store_double_as(o.data, o.bytes, g, dev::unord_f64(~s)); break;
        case OUT_ANY:
            if (o.is_float && o.bytes == 4) ((float*)o.data)[g] = (float)__longlong_as_double((long long)s);
            else dev::store_bytes(o.data, o.bytes, g, s);
            break;
        default: {
            const double cnt = (double)st[1];
            const double sum = (o.code == OUT_AVG_I) ? (double)(int64_t)s
                             : (o.code == OUT_AVG_U) ? (double)s
                             : __longlong_as_double((long long)s);
            ((double*)o.data)[g] = sum / cnt;
            break;
        }
        }
    }
}

// One tile of sorted rows (ITEMS consecutive rows per lane).  Each column is
// read lane by lane and turned through LDS (a lane reading its own
// consecutive rows makes every load 64 cache lines: 40M rows of int64 keys and
// double values took 583 us).  A run
// (rows of one key) that starts and ends inside a lane is folded in registers
// and written straight out.  Runs that cross lane boundaries meet in LDS:
// slot L (nops states) collects the group whose head is in lane L, slot
// kSegB the group whose head lies before the tile.  A continuation run finds
// its slot through a max-scan of "last lane with a head".  The tile's last
// group, if it continues into the next tile, goes to the tile's boundary
// state instead; the continuation group of an earlier tile's head is added
// to that tile's boundary state, or, if the group began before this tile's
// kSegSpan tiles, to the state of the first of those (which has no heads, so
// no use for it): at most kSegSpan tiles meet at one address.  Every tile of
// one group of 64M rows at one address, five states, took 2.60 ms a call,
// this way 1.23.
template <int KB, int MO, class VL>
__global__ __launch_bounds__(kSegB) void seg_reduce_kernel(SegArgs sa, int is_signed, AggSpec spec, OutSpec os)
{
    constexpr int ITEMS = kSegItems;
    const void* keys = sa.keys;
    const int64_t* perm = sa.perm;
    const int64_t n = sa.n;
    const uint32_t* __restrict__ head_off = sa.head_off;
    const uint32_t ntiles = sa.ntiles;
    unsigned long long* bstate = sa.bstate;
    unsigned long long* bkey = sa.bkey;
    uint32_t* btrail = sa.btrail;
    constexpr int T = kSegB * ITEMS;
    constexpr int kSlots = kSegB + 1;
    constexpr int NV = VL::NV > 0 ? VL::NV : 1;
    constexpr int kb = KB;
    extern __shared__ unsigned long long slot[];  // nops * kSlots
    __shared__ unsigned long long turn[kSegB * (ITEMS + 1)];  // a column of the tile, one word of padding per lane
    __shared__ uint32_t wsum[kSegB / 64];
    __shared__ int wmax[kSegB / 64];
    __shared__ uint32_t s_tile_cont;

    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const uint32_t tile = blockIdx.x;
    const int64_t tstart = (int64_t)tile * T;
    const int64_t r0 = tstart + (int64_t)t * ITEMS;
    const int nops = spec.nops;
    for (int i = t; i < nops * kSlots; i += kSegB) slot[i] = 0ull;
    if (t == 0) s_tile_cont = 0u;

    uint64_t k[ITEMS];
    bool head[ITEMS];
    uint32_t nheads = 0;
    auto key_at = [&](int64_t r) -> uint64_t {
        return KB == 4 ? (uint64_t)((const uint32_t*)keys)[r] : ((const uint64_t*)keys)[r];
    };
    // load(r) for every row of the tile, into this lane's consecutive rows
    auto turned = [&](auto load, uint64_t (&o)[ITEMS]) {
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            const int e = i * kSegB + t;
            const int64_t r = tstart + e;
            turn[e + e / ITEMS] = r < n ? load(r) : 0ull;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) o[i] = turn[t * (ITEMS + 1) + i];
    };
    turned(key_at, k);
    uint64_t prev = 0ull;
    if (r0 > 0 && r0 < n) prev = t > 0 ? turn[(t - 1) * (ITEMS + 1) + ITEMS - 1] : key_at(r0 - 1);
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int64_t r = r0 + i;
        head[i] = r < n && (r == 0 || k[i] != prev);
        nheads += head[i] ? 1u : 0u;
        prev = k[i];
    }
    const int64_t r_end = r0 + ITEMS;  // first row after this lane
    bool next_head = r_end >= n;
    if (!next_head) next_head = (t + 1 < kSegB ? turn[(t + 1) * (ITEMS + 1)] : key_at(r_end)) != k[ITEMS - 1];
    __syncthreads();  // turn is free again
    // groups whose head precedes this lane within the tile, and the tile total
    uint32_t tile_heads = 0;
    const uint32_t hbefore = block_excl_scan(nheads, wsum, &tile_heads);
    // owner of a continuation: the last lane before this one with a head (-1: before the tile)
    int mine = nheads > 0 ? t : -1;
    int incl = mine;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(incl, off);
        if (lane >= off) incl = y > incl ? y : incl;
    }
    if (lane == 63) wmax[w] = incl;
    __syncthreads();  // also orders the slot clearing above
    int prev_max = -1;
    for (int i = 0; i < w; ++i) prev_max = wmax[i] > prev_max ? wmax[i] : prev_max;
    int excl = __shfl_up(incl, 1);
    if (lane == 0) excl = -1;
    excl = excl > prev_max ? excl : prev_max;
    const int owner = excl < 0 ? kSegB : excl;  // slot of a continuation run

    const uint32_t hbase = head_off[tile];
    const bool last_cont_tile = [&] {
        const int64_t nx = tstart + T;
        return nx < n && key_at(nx) == key_at(nx - 1);
    }();

    uint64_t acc[MO];
#pragma unroll
    for (int a = 0; a < MO; ++a) acc[a] = 0ull;
    bool have = false, cont = r0 < n && r0 > 0 && !head[0];
    uint32_t hseen = 0;          // heads of this lane seen so far
    uint64_t run_key = 0;
    auto to_slot = [&](int sidx) {
#pragma unroll
        for (int a = 0; a < MO; ++a)
            if (a < nops) dev::apply_atomic(dev::class_of(spec, a), &slot[(size_t)a * kSlots + sidx], acc[a]);
    };
    // closes the current run; `closed`: the run ends inside this lane
    auto finish = [&](bool closed) {
        if (!have) return;
        if (cont) {
            to_slot(owner);
            if (owner == kSegB) s_tile_cont = 1u;
        } else if (closed) {
            emit_regs(os, (int64_t)hbase + hbefore + hseen - 1, dev::enc64(dev::widen_key(run_key, kb, is_signed)), acc);
        } else {
            to_slot(t);
        }
    };
    // values of the lane's rows (wide layouts: typed loads row by row)
    uint64_t rawv[VL::GEN ? 1 : NV][ITEMS];
    if constexpr (!VL::GEN && VL::NV >= 1) {
        auto column = [&](auto c) {
            constexpr int C = decltype(c)::value;
            constexpr int W = VL::template width<C>();
            const void* data = spec.cols[C].data;
            turned([&](int64_t r) -> uint64_t {
                const int64_t x = perm ? perm[r] : r;
                return W == 4 ? (uint64_t)((const uint32_t*)data)[x] : ((const uint64_t*)data)[x];
            }, rawv[C]);
        };
        column(std::integral_constant<int, 0>{});
        if constexpr (VL::NV >= 2) {
            __syncthreads();
            column(std::integral_constant<int, 1>{});
        }
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int64_t r = r0 + i;
        if (r >= n) break;
        if (head[i]) {
            finish(true);
            have = false;
            cont = false;
            ++hseen;
            run_key = k[i];
        }
        uint64_t cv[NV], raw[NV];
        if constexpr (VL::GEN) {
            load_row<VL>(spec, perm ? perm[r] : r, true, raw);
        } else {
#pragma unroll
            for (int c = 0; c < NV; ++c) raw[c] = VL::NV > 0 ? rawv[c][i] : 0ull;
        }
        canon_row<VL, NV>(spec, raw, cv);
#pragma unroll
        for (int a = 0; a < MO; ++a) {
            if (a < nops) {
                const OpDesc od = spec.ops[a];
                uint64_t v = 1ull;
#pragma unroll
                for (int c = 0; c < NV; ++c)
                    if (c == od.col) v = cv[c];
                const uint64_t o = dev::operand(od, v);
                acc[a] = have ? dev::combine(dev::class_of(spec, a), acc[a], o) : o;
            }
        }
        have = true;
    }
    // the lane's last run: complete when the next row starts a new group
    finish(next_head);
    __syncthreads();

    // groups collected in slots: the one with its head in this lane
    const bool owns_open = have && !cont && !next_head;
    if (owns_open) {
        const uint32_t gidx = hbase + hbefore + hseen - 1;
        if (last_cont_tile && hbefore + hseen == tile_heads) {
            // the tile's last group continues into the next tile
            unsigned long long* dst = bstate + (size_t)tile * nops;
            for (int a = 0; a < nops; ++a)
                dev::apply_atomic(dev::class_of(spec, a), dst + a, slot[(size_t)a * kSlots + t]);
            bkey[tile] = run_key;
            btrail[tile] = 1u;
        } else {
            dev::emit_group(os, (int64_t)gidx, dev::enc64(dev::widen_key(run_key, kb, is_signed)), slot + t,
                            (int64_t)kSlots);
        }
    }
    if (t == 0 && s_tile_cont) {
        // continuation of a group whose head is in an earlier tile
        const uint32_t first = tile & ~(kSegSpan - 1u);
        const bool from_before = head_off[first] == hbase && (first != tile || tile_heads == 0u);
        const uint32_t own = from_before ? first : owner_tile(head_off, ntiles, hbase - 1u);
        unsigned long long* dst = bstate + (size_t)own * nops;
        for (int a = 0; a < nops; ++a)
            dev::apply_atomic(dev::class_of(spec, a), dst + a, slot[(size_t)a * kSlots + kSegB]);
    }
}

}  // namespace

template <int KB, int MO>
void launch_seg(const SegArgs& a, int is_signed, const AggSpec& spec, const OutSpec& os, hipStream_t s)
{
    const size_t lds = (size_t)spec.nops * (kSegB + 1) * 8;
    lds::with_vlayout(spec, true, [&](auto vl) {
        auto kern = seg_reduce_kernel<KB, MO, decltype(vl)>;
        if (enable_dynamic_lds((const void*)kern) < lds) raise(EG_ERR_UNSUPPORTED, "segmented reduction slots too large");
        KernelTimer timer("segreduce", s);
        hipLaunchKernelGGL(kern, dim3(a.ntiles), dim3(kSegB), lds, s, a, is_signed, spec, os);
        EG_LAUNCH_CHECK();
    });
}

}  // namespace eg
