// eg_hash_launch_impl.hpp -- the hash aggregation kernel and its launch,
// included by the translation units that instantiate them.
#pragma once

#include <algorithm>

#include "eg_hash_launch.hpp"
#include "eg_jit.hpp"
#include "eg_lds_table.hpp"

namespace eg {
namespace {
using agg::max_block;

template <int KB, class VL, bool STORE>
__global__ __launch_bounds__(max_block<VL::NV>()) void hash_agg_kernel(KeyDesc key, int64_t n, AggSpec spec,
                                                                        GTable gt, int cr, int rep_log2,
                                                                        int probe_limit, int peel_min,
                                                                        unsigned long long* priv)
{
    agg::hash_agg<KB, VL, dev::RtOps, STORE>(key, n, spec, gt, cr, rep_log2, probe_limit, peel_min, priv);
}

}  // namespace

template <int KB, bool STORE>
HashLaunch prepare_hash_agg(bool vec, const HashTuning& t, int64_t n, const AggSpec& spec, const HashLayout& L,
                            bool use_jit)
{
    const DeviceInfo& di = device_info();
    HashLaunch h;
    lds::with_vlayout(spec, vec, [&](auto vl) {
        using VL = decltype(vl);
        h.kern = hash_agg_kernel<KB, VL, STORE>;
        enable_dynamic_lds((const void*)h.kern);
        h.block = std::min(t.block, max_block<VL::NV>());
        // the kernel with this request's ops compiled in, once it is available
        const jit::Kind kind = STORE ? jit::Kind::HASH_AGG_STORE : jit::Kind::HASH_AGG;
        if (use_jit) h.fn = jit::lookup(kind, KB, jit::vlayout_name<VL>(), spec, n);
    });
    const int64_t tile = (int64_t)h.block * lds::kRows;
    const int64_t want = (n + tile - 1) / tile;
    int per_cu = t.blocks_per_cu;
    if (per_cu <= 0) {
        if (h.fn) per_cu = jit::occupancy(h.fn, h.block, L.lds_bytes);
        else EG_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, h.kern, h.block, L.lds_bytes));
    }
    h.grid = std::max<int64_t>(1, std::min<int64_t>(want, (int64_t)di.num_cus * std::max(per_cu, 1)));
    return h;
}

template <int KB>
void launch_hash_agg(const HashLaunch& h, const KeyDesc& key, int64_t n, const AggSpec& spec, const GTable& gt,
                     const HashLayout& L, unsigned long long* priv, hipStream_t s)
{
    KernelTimer timer("hash_agg", s);
    if (h.fn) {
        KeyDesc a_key = key;
        int64_t a_n = n;
        AggSpec a_spec = spec;
        GTable a_gt = gt;
        int a_cr = L.cr, a_rep = L.rep_log2, a_probe = L.probe_limit, a_peel = L.peel_min;
        unsigned long long* a_priv = priv;
        void* args[] = {&a_key, &a_n, &a_spec, &a_gt, &a_cr, &a_rep, &a_probe, &a_peel, &a_priv};
        if (jit::launch(h.fn, (unsigned)h.grid, (unsigned)h.block, L.lds_bytes, s, args)) return;
    }
    hipLaunchKernelGGL(h.kern, dim3((unsigned)h.grid), dim3(h.block), L.lds_bytes, s, key, n, spec, gt, L.cr,
                       L.rep_log2, L.probe_limit, L.peel_min, priv);
    EG_LAUNCH_CHECK();
}

}  // namespace eg
