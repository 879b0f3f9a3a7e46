// Launch side of egs_tiled.h for one element type; included by egs_tiled_<type>.hip, which each instantiate their share.
#pragma once
#include "egs_host.h"
#include "egs_split_f32.h"

namespace egs {
namespace host {

// a weight gradient as a launch, or as the first workgroups of one
struct TiledDwGrid { int blocks; size_t lds; TiledDwKind kind; };

// false: operands that tiny_dw_kernel takes, or more tiles than a grid holds
template <class TT>
bool tiled_dw_grid(TiledDwParams &p, TiledDwGrid &g)
{
    if (p.x_bytes < 16 || p.y_bytes < 16) return false;
    g.kind = TT::ES == 4 && p.split32 ? TILED_DW_SPLIT : p.wide ? TILED_DW_WIDE : TILED_DW;
    if (g.kind == TILED_DW_SPLIT) {
        p.i_tiles = ceil_div(p.I, SplitDwLds::T); p.j_tiles = ceil_div(p.J, SplitDwLds::T);
        g.lds = SplitDwLds::BYTES;
    } else if (g.kind == TILED_DW_WIDE) {
        typedef TiledDwWide<TT> L;
        p.i_tiles = ceil_div(p.I, L::TI); p.j_tiles = ceil_div(p.J, L::TJ);
        g.lds = L::BYTES;
    } else {
        g.lds = TiledDw<TT>::BYTES;
    }
    const int64_t tiles = (int64_t)p.E * p.i_tiles * p.j_tiles * p.S;       // (the wide tiles are not split)
    if (tiles > INT32_MAX / 2) return false;
    g.blocks = (int)(8 * ((tiles + 7) / 8));
    return true;
}

// Two launches where the product's written-out kernel (one or two slabs), which more workgroups of a CU run side by side than the shared launch's loop,
// gains more than the sharing saves: many tiles of product, enough of the weight gradient's to fill the device on their own, in chains that are
// not long against the product.  us, one launch / two: bf16 dY and dW B41 T1715 E119 K224 I32 J25 90 / 74, B90 T1835 E94 K138 I32 J25 100 / 84, f32 B113
// T319 E117 K63 I32 J55 158 / 135, f32 dX and dW B98 T555 E63 K217 I32 J64 323 / 276; not bf16 B43 T1534 E102 K139 I39 J160 191 / 189.  Of 1542 backward
// calls (most of them of short reductions and large) 56 go this way, 6 of them more than 3 % slower for it (1.05); of 1045 others of that kind 7 are left that
// two launches would run more than 3 % faster (at worst 1.14), where one in 37 was (1.21).
template <class TT>
bool tiled_apart(const TiledRowsParams &p, int blocks, const TiledDwParams &q, const TiledDwGrid &g)
{
    const int slabs = ceil_div(p.R, 8 * TT::VEC);
    if (g.kind != TILED_DW || slabs > 2 || g.blocks < 400) return false;
    const double tiles = blocks * (TT::ES == 4 ? 2.0 : 1.0), steps = (double)q.B * q.K / q.S / 128;        // fp32 tiles take twice as long
    return tiles >= 4096 * (2 * slabs - 1) && tiles >= 0.6 * g.blocks * steps;
}

template <class TT, int TN, int KIND>
int launch_tiled_pair(const TiledRowsParams &p, int blocks, size_t lds, const TiledDwParams &q, const TiledDwGrid &g, hipStream_t s)
{
    static LdsGrant told;
    if (g.lds > lds) lds = g.lds;
    const int rc = allow_large_lds((const void *)tiled_pair_kernel<TT, TN, KIND>, told, lds, "hipFuncSetAttribute(tiled_pair_kernel)");
    if (rc != EGS_OK) return rc;
    // The longer chains first: the slabs of 128 bytes that a product's workgroup goes through, against 32 picks at a time of an expert.  Of 4255
    // calls with either first 121 are more than 3 % slower than the other way by this line (with the weight gradient always first 245): us, it /
    // the product first, f32 dY and dW B6 T47 E52 K10 I686 J160 45 / 29, B2 T124 E115 K16 I960 J32 32 / 21, B15 T98 E79 K46 I64 J31 15 / 23.5.
    const int dw_first = ceil_div(p.R, 8 * TT::VEC) <= q.B * q.K / 32 + 6;
    hipLaunchKernelGGL((tiled_pair_kernel<TT, TN, KIND>), dim3((unsigned)(g.blocks + blocks)), dim3(kThreads), lds, s, p, q, dw_first ? g.blocks : blocks, dw_first);
    EGS_CHECK_LAUNCH("tiled_pair_kernel");
    note_launch("tiled_rows_kernel");           // (the weight gradient's name follows from dw_general)
    return EGS_OK;
}

template <class TT, int WES, bool W_TRANS, int TN>
int launch_tiled_one(TiledRowsParams &p, TiledDwJob *dw, hipStream_t s)
{
    p.m_tiles = ceil_div(p.B * p.K, 64);
    p.n_tiles = ceil_div(p.N, 16 * TN);
    const int64_t total = (int64_t)p.E * p.m_tiles * p.n_tiles;
    if (total > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    constexpr size_t lds = TiledLds<TT, W_TRANS, TN>::BYTES;
    const int blocks = (int)(8 * ((total + 7) / 8));
    if constexpr (!W_TRANS && WES == TT::ES) {
        TiledDwGrid g;
        if (dw != nullptr && !dw->done && tiled_dw_grid<TT>(dw->q, g) && (int64_t)g.blocks + blocks <= INT32_MAX / 2 &&
            !tiled_apart<TT>(p, blocks, dw->q, g)) {
            int rc;
            if (TT::ES == 4 && g.kind == TILED_DW_SPLIT) rc = launch_tiled_pair<TT, TN, TT::ES == 4 ? TILED_DW_SPLIT : TILED_DW>(p, blocks, lds, dw->q, g, s);
            else if (g.kind == TILED_DW_WIDE) rc = launch_tiled_pair<TT, TN, TILED_DW_WIDE>(p, blocks, lds, dw->q, g, s);
            else rc = launch_tiled_pair<TT, TN, TILED_DW>(p, blocks, lds, dw->q, g, s);
            dw->name = g.kind == TILED_DW_SPLIT ? "tiled_dw_split_kernel" : g.kind == TILED_DW_WIDE ? "tiled_dw_wide_kernel" : "tiled_dw_kernel";
            dw->done = rc == EGS_OK;
            return rc;
        }
    }
    static LdsGrant told;
    const int slabs = ceil_div(p.R, 8 * TT::VEC);
    const auto kernel = slabs <= 1   ? tiled_rows_kernel<TT, WES, W_TRANS, TN, 1>
                        : slabs == 2 ? tiled_rows_kernel<TT, WES, W_TRANS, TN, 2>
                        : slabs == 3 ? tiled_rows_kernel<TT, WES, W_TRANS, TN, 3>
                        : slabs == 4 ? tiled_rows_kernel<TT, WES, W_TRANS, TN, 4> : tiled_rows_kernel<TT, WES, W_TRANS, TN, 0>;
    const int rc = allow_large_lds((const void *)tiled_rows_kernel<TT, WES, W_TRANS, TN, 0>, told, lds, "hipFuncSetAttribute(tiled_rows_kernel)");
    if (rc != EGS_OK) return rc;
    const size_t held = slabs <= 4 ? TiledLds<TT, W_TRANS, TN>::ONE_STAGE : lds;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kThreads), held, s, p);
    EGS_CHECK_LAUNCH("tiled_rows_kernel");
    return EGS_OK;
}

template <class TT, int WES, bool W_TRANS>
int launch_tiled(TiledRowsParams &p, TiledDwJob *dw, hipStream_t s)
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
        if (tn == 5) return launch_tiled_one<TT, WES, W_TRANS, 5>(p, dw, s);
    }
    return tn == 6 ? launch_tiled_one<TT, WES, W_TRANS, 6>(p, dw, s)
                   : tn == 4 ? launch_tiled_one<TT, WES, W_TRANS, 4>(p, dw, s) : launch_tiled_one<TT, WES, W_TRANS, 2>(p, dw, s);
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
    TiledDwGrid g;
    if (!tiled_dw_grid<TT>(p, g)) return EGS_ERR_BAD_SHAPE;
    if constexpr (TT::ES == 4) {
        if (g.kind == TILED_DW_SPLIT) {
            static_assert(SplitDwLds::BYTES <= 64 * 1024, "no grant needed");
            hipLaunchKernelGGL(tiled_dw_split_kernel, dim3((unsigned)g.blocks), dim3(kThreads), g.lds, s, p);
            EGS_CHECK_LAUNCH("tiled_dw_split_kernel");
            return EGS_OK;
        }
    }
    if (g.kind == TILED_DW_WIDE) {
        static LdsGrant told;
        const int rc = allow_large_lds((const void *)tiled_dw_wide_kernel<TT>, told, g.lds, "hipFuncSetAttribute(tiled_dw_wide_kernel)");
        if (rc != EGS_OK) return rc;
        hipLaunchKernelGGL(tiled_dw_wide_kernel<TT>, dim3((unsigned)g.blocks), dim3(kThreads), g.lds, s, p);
        EGS_CHECK_LAUNCH("tiled_dw_wide_kernel");
        return EGS_OK;
    }
    static_assert(TiledDw<TT>::BYTES <= 64 * 1024, "no grant needed");
    hipLaunchKernelGGL(tiled_dw_kernel<TT>, dim3((unsigned)g.blocks), dim3(kThreads), g.lds, s, p);
    EGS_CHECK_LAUNCH("tiled_dw_kernel");
    return EGS_OK;
}

}  // namespace host
}  // namespace egs
