// Launch side of egs_tiled.h for one element type; included by egs_tiled_<type>.hip, which each instantiate their share.
#pragma once
#include "egs_host.h"
#include "egs_split_f32.h"

namespace egs {
namespace host {

template <class TT, int WES, bool W_TRANS, int TN>
int launch_tiled_one(TiledRowsParams &p, hipStream_t s)
{
    p.m_tiles = ceil_div(p.B * p.K, 64);
    p.n_tiles = ceil_div(p.N, 16 * TN);
    const int64_t total = (int64_t)p.E * p.m_tiles * p.n_tiles;
    if (total > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    static LdsGrant told;
    constexpr size_t lds = TiledLds<TT, W_TRANS, TN>::BYTES;
    const int rc = allow_large_lds((const void *)tiled_rows_kernel<TT, WES, W_TRANS, TN>, told, lds, "hipFuncSetAttribute(tiled_rows_kernel)");
    if (rc != EGS_OK) return rc;
    hipLaunchKernelGGL((tiled_rows_kernel<TT, WES, W_TRANS, TN>), dim3((unsigned)(8 * ((total + 7) / 8))), dim3(kThreads), lds, s, p);
    EGS_CHECK_LAUNCH("tiled_rows_kernel");
    return EGS_OK;
}

template <class TT, int WES, bool W_TRANS>
int launch_tiled(TiledRowsParams &p, hipStream_t s)
{
    // (offsets inside an expert's matrix are 32-bit, the slab past its end included)
    const bool huge = (uint64_t)p.R * p.N * WES + 128ull * p.N * WES + 4096 > 0xff000000ull;
    // Every 16-byte read of A stays inside A, and every one of W between the start of an expert's matrix and the end of W: the last
    // expert's own matrix has to hold one (all others' then do)
    if (p.a_bytes < 16 || (uint64_t)p.R * p.N * WES < 16 || huge) {
        hipLaunchKernelGGL((tiny_rows_kernel<TT, WES, W_TRANS>), dim3(grid_1d((size_t)p.B * p.E * p.K * p.N)), dim3(kThreads), 0, s, p);
        EGS_CHECK_LAUNCH("tiny_rows_kernel");
        return EGS_OK;
    }
    const int tn = tiled_columns(p.E, (int64_t)p.B * p.K, p.N, TT::ES == 4);
    if constexpr (TT::ES == 4) {
        if (tn == 5) return launch_tiled_one<TT, WES, W_TRANS, 5>(p, s);
    }
    return tn == 6 ? launch_tiled_one<TT, WES, W_TRANS, 6>(p, s)
                   : tn == 4 ? launch_tiled_one<TT, WES, W_TRANS, 4>(p, s) : launch_tiled_one<TT, WES, W_TRANS, 2>(p, s);
}

template <class TT>
int launch_tiled_dw(TiledDwParams &p, hipStream_t s)
{
    const size_t w_elems = (size_t)p.E * p.I * p.J;
    if (p.x_bytes < 16 || p.y_bytes < 16) {
        hipLaunchKernelGGL(tiny_dw_kernel<TT>, dim3(grid_1d(w_elems)), dim3(kThreads), 0, s, p);
        EGS_CHECK_LAUNCH("tiny_dw_kernel");
        return EGS_OK;
    }
    if constexpr (TT::ES == 4) {
        if (p.split32) {
            p.i_tiles = ceil_div(p.I, SplitDwLds::T); p.j_tiles = ceil_div(p.J, SplitDwLds::T);
            const int64_t tiles = (int64_t)p.E * p.i_tiles * p.j_tiles * p.S;
            if (tiles > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
            static_assert(SplitDwLds::BYTES <= 64 * 1024, "no grant needed");
            hipLaunchKernelGGL(tiled_dw_split_kernel, dim3((unsigned)(8 * ((tiles + 7) / 8))), dim3(kThreads), SplitDwLds::BYTES, s, p);
            EGS_CHECK_LAUNCH("tiled_dw_split_kernel");
            return EGS_OK;
        }
    }
    if (p.wide) {
        typedef TiledDwWide<TT> L;
        p.i_tiles = ceil_div(p.I, L::TI); p.j_tiles = ceil_div(p.J, L::TJ);
        const int64_t wide = (int64_t)p.E * p.i_tiles * p.j_tiles;
        if (wide > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
        static LdsGrant told;
        const int rc = allow_large_lds((const void *)tiled_dw_wide_kernel<TT>, told, L::BYTES, "hipFuncSetAttribute(tiled_dw_wide_kernel)");
        if (rc != EGS_OK) return rc;
        hipLaunchKernelGGL(tiled_dw_wide_kernel<TT>, dim3((unsigned)(8 * ((wide + 7) / 8))), dim3(kThreads), L::BYTES, s, p);
        EGS_CHECK_LAUNCH("tiled_dw_wide_kernel");
        return EGS_OK;
    }
    const int64_t total = (int64_t)p.E * p.i_tiles * p.j_tiles * p.S;
    if (total > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    static_assert(TiledDw<TT>::BYTES <= 64 * 1024, "no grant needed");
    hipLaunchKernelGGL(tiled_dw_kernel<TT>, dim3((unsigned)(8 * ((total + 7) / 8))), dim3(kThreads), TiledDw<TT>::BYTES, s, p);
    EGS_CHECK_LAUNCH("tiled_dw_kernel");
    return EGS_OK;
}

}  // namespace host
}  // namespace egs
