// Launches that several translation units have a part in: the small-expert products, weight gradients that may share another kernel's
// launch, and the one-kernel scatter; their launch entry points (one file per element type, so that the many variants compile in parallel).
#pragma once
#include "egs_host.h"
#include "egs_scatter_aux.h"
#include "egs_small.h"
#include "egs_dw_tile.h"
#include "egs_scatter_fused.h"

namespace egs {
namespace host {

// one launch of rows_small_kernel, or its share of a heterogeneous launch
struct SmallRowsJob {
    SmallRowsParams p;
    int R, act_dtype, blocks;
    bool nmajor, gather, out_f32;
    size_t lds;
};

// one launch of dw_small_kernel (or its share of a heterogeneous launch) plus the second pass
struct SmallDwJob {
    SmallDwParams q;
    int blocks, act_dtype;
    size_t w_elems;
    bool done;          // set once the first pass has been enqueued
};

// one launch of dw_tile_kernel (or its share of a heterogeneous launch): the whole weight gradient, no second pass
struct DwTileJob {
    DwTileParams q;
    int blocks, act_dtype;
    bool wide;          // 32 x 64 tiles and 8 wavefronts (dw_tile_wide_kernel) instead of 32 x 32 and 4
    bool done;          // set once it has been enqueued
};

// ---- egs_small_<type>.hip
int launch_rows_small_f16(SmallRowsJob &j, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s);
int launch_rows_small_bf16(SmallRowsJob &j, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s);

// ---- egs_fused_<type>.hip
int launch_fused_f32(const ScatterFusedParams &p, bool w_nmajor, int R, size_t lds, int blocks, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s);
int launch_fused_f16(const ScatterFusedParams &p, bool w_nmajor, int R, size_t lds, int blocks, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s);
int launch_fused_bf16(const ScatterFusedParams &p, bool w_nmajor, int R, size_t lds, int blocks, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s);

}  // namespace host
}  // namespace egs
