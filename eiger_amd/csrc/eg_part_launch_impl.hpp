// eg_part_launch_impl.hpp -- the unit kernel and its launch, included by the
// translation units that instantiate them.
#pragma once

#include "eg_jit.hpp"
#include "eg_lds_table.hpp"
#include "eg_part_launch.hpp"

namespace eg {
namespace {

using namespace lds;
using agg::kPBMax;
using agg::OutClaims;
using agg::Unit;

// Eight waves per SIMD: two 1024-thread workgroups per CU, which the LDS
// table is sized for (without the bound the compiler's scalar registers
// alone leave room for only one).
template <int KB, class VL, bool GATHER>
__global__ __launch_bounds__(kPBMax, 8) void part_agg_kernel(KeyDesc key, AggSpec spec, const int64_t* perm,
                                                       const Unit* units, GTable gt, OutSpec os,
                                                       OutClaims claims, int64_t capacity,
                                                       int cr, int probe, int peel_min)
{
    agg::part_agg<KB, VL, dev::RtOps, GATHER>(key, spec, perm, units, gt, os, claims, capacity, cr, probe,
                                              peel_min);
}

}  // namespace

template <int KB, bool GATHER>
void launch_part_agg(const KeyDesc& key, const AggSpec& spec, const int64_t* perm, const Unit* units, int nunits,
                     const GTable& gt, const OutSpec& os, const OutClaims& claims, int64_t capacity, int cr,
                     size_t lds, int block, int64_t rows, hipStream_t s)
{
    lds::with_vlayout(spec, true, [&](auto vl) {
        using VL = decltype(vl);
        auto kern = part_agg_kernel<KB, VL, GATHER>;
        if (enable_dynamic_lds((const void*)kern) < lds) raise(EG_ERR_UNSUPPORTED, "partition LDS table too large");
        KernelTimer timer("partition_agg", s);
        int probe = 16, peel_min = default_peel_min();  // probe: buckets of four slots
        // the kernel with this request's ops compiled in, once it is available
        const jit::Kind kind = GATHER ? jit::Kind::PART_AGG_GATHER : jit::Kind::PART_AGG;
        if (hipFunction_t f = jit::lookup(kind, KB, jit::vlayout_name<VL>(), spec, rows, &os)) {
            KeyDesc a_key = key;
            AggSpec a_spec = spec;
            const int64_t* a_perm = perm;
            const Unit* a_units = units;
            GTable a_gt = gt;
            OutSpec a_os = os;
            OutClaims a_claims = claims;
            int64_t a_cap = capacity;
            int a_cr = cr;
            void* args[] = {&a_key, &a_spec, &a_perm, &a_units, &a_gt, &a_os, &a_claims, &a_cap, &a_cr,
                            &probe, &peel_min};
            if (jit::launch(f, (unsigned)nunits, (unsigned)block, lds, s, args)) return;
        }
        hipLaunchKernelGGL(kern, dim3(nunits), dim3(block), lds, s, key, spec, perm, units, gt, os, claims, capacity,
                           cr, probe, peel_min);
        EG_LAUNCH_CHECK();
    });
}

}  // namespace eg
