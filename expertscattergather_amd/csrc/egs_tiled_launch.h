// Launch side of egs_tiled.h for one element type; included by egs_tiled_<type>.hip, which each instantiate their share.
#pragma once
#include "egs_host.h"

namespace egs {
namespace host {

template <class TT, int WES, bool W_TRANS, int TM, int TN, bool DEEP = false>
int launch_tiled_one(TiledRowsParams &p, hipStream_t s)
{
    p.m_tiles = ceil_div(p.B * p.K, 64 * TM);
    p.n_tiles = ceil_div(p.N, 16 * TN);
    const int64_t total = (int64_t)p.E * p.m_tiles * p.n_tiles;
    if (total > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    static LdsGrant told;
    constexpr size_t lds = TiledLds<TT, W_TRANS, TM, TN>::BYTES;
    const int rc = allow_large_lds((const void *)tiled_rows_kernel<TT, WES, W_TRANS, TM, TN, DEEP>, told, lds, "hipFuncSetAttribute(tiled_rows_kernel)");
    if (rc != EGS_OK) return rc;
    hipLaunchKernelGGL((tiled_rows_kernel<TT, WES, W_TRANS, TM, TN, DEEP>), dim3((unsigned)(8 * ((total + 7) / 8))), dim3(kThreads), lds, s, p);
    EGS_CHECK_LAUNCH("tiled_rows_kernel");
    return EGS_OK;
}

template <class TT, int WES, bool W_TRANS>
int launch_tiled(TiledRowsParams &p, hipStream_t s)
{
    // (offsets inside an expert's matrix are 32-bit, the slab past its end included)
    const bool huge = (uint64_t)p.R * p.N * WES + 128ull * p.N * WES + 4096 > 0xff000000ull;
    if (p.a_bytes < 16 || p.w_bytes < 16 || huge) {
        hipLaunchKernelGGL((tiny_rows_kernel<TT, WES, W_TRANS>), dim3(grid_1d((size_t)p.B * p.E * p.K * p.N)), dim3(kThreads), 0, s, p);
        EGS_CHECK_LAUNCH("tiny_rows_kernel");
        return EGS_OK;
    }
    // Tile shape.  Columns: what covers N with the least left over, at most 128.  Rows: 128 where that still gives every CU two
    // workgroups, else 64.  Then narrower columns while the device (256 CUs) is not covered: these products are bound by the
    // latency of their slabs, and rows fetched again by the next column tile come out of the L2.
    const int64_t Me = (int64_t)p.B * p.K;
    const int at_most_8 = ceil_div(ceil_div(p.N, ceil_div(p.N, 128)), 16);
    int tn = at_most_8 <= 2 ? 2 : at_most_8 <= 4 ? 4 : at_most_8 <= 6 ? at_most_8 : 8;
    auto tiles = [&](int bm) { return (int64_t)p.E * ((Me + bm - 1) / bm) * ceil_div(p.N, 16 * tn); };
    const int tm = Me > 64 && tiles(128) >= 512 ? 2 : 1;
    while (tm == 1 && tn > 2 && tiles(64) < 256) tn = tn > 4 ? 4 : 2;
    if (tm == 1 && tn <= 4 && tiles(64) <= 512)
        return tn == 2 ? launch_tiled_one<TT, WES, W_TRANS, 1, 2, true>(p, s) : launch_tiled_one<TT, WES, W_TRANS, 1, 4, true>(p, s);
    switch (tm * 16 + tn) {
    case 16 + 2: return launch_tiled_one<TT, WES, W_TRANS, 1, 2>(p, s);
    case 16 + 4: return launch_tiled_one<TT, WES, W_TRANS, 1, 4>(p, s);
    case 16 + 5: return launch_tiled_one<TT, WES, W_TRANS, 1, 5>(p, s);
    case 16 + 6: return launch_tiled_one<TT, WES, W_TRANS, 1, 6>(p, s);
    case 16 + 8: return launch_tiled_one<TT, WES, W_TRANS, 1, 8>(p, s);
    case 32 + 2: return launch_tiled_one<TT, WES, W_TRANS, 2, 2>(p, s);
    case 32 + 4: return launch_tiled_one<TT, WES, W_TRANS, 2, 4>(p, s);
    case 32 + 5: return launch_tiled_one<TT, WES, W_TRANS, 2, 5>(p, s);
    case 32 + 6: return launch_tiled_one<TT, WES, W_TRANS, 2, 6>(p, s);
    default: return launch_tiled_one<TT, WES, W_TRANS, 2, 8>(p, s);
    }
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
    const int64_t total = (int64_t)p.E * p.i_tiles * p.j_tiles * p.S;
    if (total > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    static_assert(TiledDw<TT>::BYTES <= 64 * 1024, "no grant needed");
    hipLaunchKernelGGL(tiled_dw_kernel<TT>, dim3((unsigned)(8 * ((total + 7) / 8))), dim3(kThreads), TiledDw<TT>::BYTES, s, p);
    EGS_CHECK_LAUNCH("tiled_dw_kernel");
    return EGS_OK;
}

}  // namespace host
}  // namespace egs
