// Launch side of egs_scatter_fused.h for one element type; included by egs_fused_<type>.hip.
#pragma once
#include "egs_jobs.h"

namespace egs {
namespace host {

template <class TT, bool W_NMAJOR, int KS>
int launch_scatter_fused_one(const ScatterFusedParams &p, size_t lds, int blocks, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s)
{
    static LdsGrant told_plain, told_dw, told_dwt, told_multi;      // one set per template instantiation
    if constexpr (TT::ES != 2) { dw = nullptr; dwt = nullptr; }     // the small weight gradients exist for 16-bit types only
    const char *name = "scatter_fused_kernel";
    if (p.experts_per_pass < p.E && p.tab_seg != nullptr) {
        name = "scatter_fused_multi_table_kernel";
        static LdsGrant told_multi_tab;
        const int rc_lds = allow_large_lds((const void *)scatter_fused_multi_table_kernel<TT, W_NMAJOR, KS>, told_multi_tab, lds,
                                           "hipFuncSetAttribute(scatter_fused_multi_table_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        hipLaunchKernelGGL((scatter_fused_multi_table_kernel<TT, W_NMAJOR, KS>), dim3(blocks), dim3(kFusedThreads), lds, s, p);
    } else if (p.experts_per_pass < p.E) {
        // several passes over groups of experts: a launch of its own (a weight gradient of the same call follows alone)
        name = "scatter_fused_multi_kernel";
        const int rc_lds = allow_large_lds((const void *)scatter_fused_multi_kernel<TT, W_NMAJOR, KS>, told_multi, lds,
                                           "hipFuncSetAttribute(scatter_fused_multi_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        hipLaunchKernelGGL((scatter_fused_multi_kernel<TT, W_NMAJOR, KS>), dim3(blocks), dim3(kFusedThreads), lds, s, p);
    } else if (p.run > 1) {             // (a weight gradient of the same call follows alone)
        name = "scatter_fused_runs_kernel";
        static LdsGrant told_runs[2];
        constexpr bool kHolds = KS <= 2;
        // Rows stay in registers where that saves a workgroup ten units' loads or more; bringing them into operand order ahead of the first slice
        // and a pass over the table are its price.  Of 507 sizes, us, held / not: B18 T76 E2 K3 I896 J64 two units in runs of two 13.9 / 11.7, B85
        // T286 E4 K48 I160 J64 eight in runs of two 15.8 / 13.6; from this line on 4 of 361 are more than 3 % slower, on average 0.90 of it.
        const int units = p.E * ((p.K + 31) / 32);
        const bool hold = kHolds && units <= kFusedHeldUnits && units * (p.run - 1) >= 10;
        const auto kernel = hold ? scatter_fused_runs_kernel<TT, W_NMAJOR, KS, kHolds> : scatter_fused_runs_kernel<TT, W_NMAJOR, KS, false>;
        const int rc_lds = allow_large_lds((const void *)kernel, told_runs[hold], lds, "hipFuncSetAttribute(scatter_fused_runs_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kFusedThreads), lds, s, p);
    } else if (p.tab_seg != nullptr && dwt != nullptr && !dwt->wide && TT::ES == 2) {
      if constexpr (TT::ES == 2) {
        name = "scatter_fused_dwtile_table_kernel";
        static LdsGrant told_dwt_tab;
        const size_t tile_lds = dw_tile_lds(kFusedThreads / 64);
        const size_t need = lds > tile_lds ? lds : tile_lds;
        const int rc_lds = allow_large_lds((const void *)scatter_fused_dwtile_table_kernel<TT, W_NMAJOR, KS>, told_dwt_tab, need,
                                           "hipFuncSetAttribute(scatter_fused_dwtile_table_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        hipLaunchKernelGGL((scatter_fused_dwtile_table_kernel<TT, W_NMAJOR, KS>), dim3(blocks + dwt->blocks), dim3(kFusedThreads), need,
                           s, p, dwt->q, blocks);
        dwt->done = true;
      }
    } else if (p.tab_seg != nullptr && dw == nullptr && (dwt == nullptr || dwt->wide || TT::ES != 2)) {
        name = "scatter_fused_table_kernel";
        static LdsGrant told_tab;
        const int rc_lds = allow_large_lds((const void *)scatter_fused_table_kernel<TT, W_NMAJOR, KS>, told_tab, lds,
                                           "hipFuncSetAttribute(scatter_fused_table_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        hipLaunchKernelGGL((scatter_fused_table_kernel<TT, W_NMAJOR, KS>), dim3(blocks), dim3(kFusedThreads), lds, s, p);
    } else if (dwt != nullptr && !dwt->wide) {
      if constexpr (TT::ES == 2) {
        name = "scatter_fused_dwtile_kernel";
        const size_t tile_lds = dw_tile_lds(kFusedThreads / 64);
        const size_t need = lds > tile_lds ? lds : tile_lds;
        const int rc_lds = allow_large_lds((const void *)scatter_fused_dwtile_kernel<TT, W_NMAJOR, KS>, told_dwt, need,
                                           "hipFuncSetAttribute(scatter_fused_dwtile_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        hipLaunchKernelGGL((scatter_fused_dwtile_kernel<TT, W_NMAJOR, KS>), dim3(blocks + dwt->blocks), dim3(kFusedThreads), need,
                           s, p, dwt->q, blocks);
        dwt->done = true;
      }
    } else if (dw != nullptr) {
      if constexpr (TT::ES == 2) {
        name = "scatter_fused_dw_kernel";
        const size_t dw_lds = (size_t)kDwSmallLdsBytes * (kFusedThreads / kThreads);       // one 16 KB tile per wavefront
        const size_t need = lds > dw_lds ? lds : dw_lds;
        const int rc_lds = allow_large_lds((const void *)scatter_fused_dw_kernel<TT, W_NMAJOR, KS>, told_dw, need,
                                           "hipFuncSetAttribute(scatter_fused_dw_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        hipLaunchKernelGGL((scatter_fused_dw_kernel<TT, W_NMAJOR, KS>), dim3(blocks + dw->blocks), dim3(kFusedThreads), need, s, p,
                           dw->q, blocks);
        dw->done = true;
      }
    } else {
        const int rc_lds = allow_large_lds((const void *)scatter_fused_kernel<TT, W_NMAJOR, KS>, told_plain, lds,
                                           "hipFuncSetAttribute(scatter_fused_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        hipLaunchKernelGGL((scatter_fused_kernel<TT, W_NMAJOR, KS>), dim3(blocks), dim3(kFusedThreads), lds, s, p);
    }
    EGS_CHECK_LAUNCH(name);
    return EGS_OK;
}

template <class TT, bool W_NMAJOR>
int launch_scatter_fused_ks(const ScatterFusedParams &p, int R, size_t lds, int blocks, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s)
{
    switch (R / (4 * TT::VEC)) {        // MFMA steps of four 16-byte chunks
    case 1: return launch_scatter_fused_one<TT, W_NMAJOR, 1>(p, lds, blocks, dw, dwt, s);
    case 2: return launch_scatter_fused_one<TT, W_NMAJOR, 2>(p, lds, blocks, dw, dwt, s);
    default: return launch_scatter_fused_one<TT, W_NMAJOR, 4>(p, lds, blocks, dw, dwt, s);
    }
}

}  // namespace host
}  // namespace egs
