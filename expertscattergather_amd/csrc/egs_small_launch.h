// Launch side of rows_small_kernel (egs_small.h) for one element type; included by egs_small_<type>.hip.
#pragma once
#include "egs_jobs.h"

namespace egs {
namespace host {

// ---- launch of a rows job, alone or sharing the launch with a weight gradient of the same call (its one-pass form,
// or the first pass of its split form)
template <class TT, bool W_NMAJOR, int KS, int TN, bool GATHER, bool OUT_F32>
int launch_rows_small_one(SmallRowsJob &j, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s)
{
    if constexpr (GATHER) {
        if (j.p.act != ACT_NONE) {
            if (dw != nullptr || dwt != nullptr) return EGS_ERR_UNSUPPORTED;        // (backward products have no activation)
            hipLaunchKernelGGL((rows_small_kernel<TT, W_NMAJOR, KS, TN, GATHER, OUT_F32, true>), dim3(j.blocks), dim3(kThreads), j.lds, s, j.p);
            EGS_CHECK_LAUNCH("rows_small_kernel");
            return EGS_OK;
        }
        if (dwt != nullptr) {       // dwt->wide, and j regridded for 8 wavefronts per workgroup (see pair_gather_with_dw_tile)
            static LdsGrant told;
            const size_t tile_lds = dw_tile_lds(kDwWideThreads / 64, 64);
            const int rc = allow_large_lds((const void *)rows_dw_tile_kernel<TT, W_NMAJOR, KS, TN>, told, tile_lds,
                                           "hipFuncSetAttribute(rows_dw_tile_kernel)");
            if (rc != EGS_OK) return rc;
            hipLaunchKernelGGL((rows_dw_tile_kernel<TT, W_NMAJOR, KS, TN>), dim3(j.blocks + dwt->blocks), dim3(kDwWideThreads),
                               tile_lds, s, j.p, dwt->q, j.blocks);
            EGS_CHECK_LAUNCH("rows_dw_tile_kernel");
            dwt->done = true;
            return EGS_OK;
        }
    }
    if (dw != nullptr) {
        hipLaunchKernelGGL((rows_dw_small_kernel<TT, W_NMAJOR, KS, TN, GATHER, OUT_F32>), dim3(j.blocks + dw->blocks),
                           dim3(kThreads), j.lds, s, j.p, dw->q, j.blocks);
        dw->done = true;
    } else {
        hipLaunchKernelGGL((rows_small_kernel<TT, W_NMAJOR, KS, TN, GATHER, OUT_F32>), dim3(j.blocks), dim3(kThreads),
                           j.lds, s, j.p);
    }
    EGS_CHECK_LAUNCH(dw != nullptr ? "rows_dw_small_kernel" : "rows_small_kernel");
    return EGS_OK;
}

template <class TT, bool W_NMAJOR, int TN, bool GATHER, bool OUT_F32>
int launch_rows_small_ks(SmallRowsJob &j, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s)
{
    switch (j.R) {
    case 32: return launch_rows_small_one<TT, W_NMAJOR, 1, TN, GATHER, OUT_F32>(j, dw, dwt, s);
    case 64: return launch_rows_small_one<TT, W_NMAJOR, 2, TN, GATHER, OUT_F32>(j, dw, dwt, s);
    default: return launch_rows_small_one<TT, W_NMAJOR, 4, TN, GATHER, OUT_F32>(j, dw, dwt, s);
    }
}

template <class TT, bool GATHER, bool OUT_F32>
int launch_rows_small_tn(SmallRowsJob &j, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s)
{
    if (j.p.N <= 64)
        return j.nmajor ? launch_rows_small_ks<TT, true, 4, GATHER, OUT_F32>(j, dw, dwt, s)
                        : launch_rows_small_ks<TT, false, 4, GATHER, OUT_F32>(j, dw, dwt, s);
    return j.nmajor ? launch_rows_small_ks<TT, true, 8, GATHER, OUT_F32>(j, dw, dwt, s)
                    : launch_rows_small_ks<TT, false, 8, GATHER, OUT_F32>(j, dw, dwt, s);
}

template <class TT>
int launch_rows_small_tt(SmallRowsJob &j, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s)
{
    if (j.gather) return launch_rows_small_tn<TT, true, false>(j, dw, dwt, s);
    return j.out_f32 ? launch_rows_small_tn<TT, false, true>(j, dw, dwt, s) : launch_rows_small_tn<TT, false, false>(j, dw, dwt, s);
}

}  // namespace host
}  // namespace egs
