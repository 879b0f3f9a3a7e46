// Launch side of the tiled weight gradient: tiled_dw_kernel, tiled_dw_wide_kernel for few picks, or dw_dl_kernel for large well-formed 16-bit
// shapes, followed by the fixed-order sum over splits.
#include "egs_host.h"
#include "egs_dw_dl.h"
#include "egs_dw_strip.h"

namespace egs {
namespace host {

namespace {

template <class TT, int TP, int BQ>
int launch_dw_strip_one(const DwDlParams &q, int grid, hipStream_t s)
{
    static LdsGrant told;
    const int rc = allow_large_lds((const void *)dw_strip_kernel<TT, TP, BQ>, told, DwStrip<TP, BQ>::BYTES, "hipFuncSetAttribute(dw_strip_kernel)");
    if (rc != EGS_OK) return rc;
    hipLaunchKernelGGL((dw_strip_kernel<TT, TP, BQ>), dim3((unsigned)grid), dim3(kDlThreads), (DwStrip<TP, BQ>::BYTES), s, q);
    EGS_CHECK_LAUNCH("dw_strip_kernel");
    return EGS_OK;
}
template <class TT>
int launch_dw_strip(const DwDlParams &q, int tp, int bq, int grid, hipStream_t s)
{
    return bq == 128 ? launch_dw_strip_one<TT, 4, 128>(q, grid, s) : tp == 2 ? launch_dw_strip_one<TT, 2, 64>(q, grid, s)
         : tp == 3 ? launch_dw_strip_one<TT, 3, 64>(q, grid, s) : launch_dw_strip_one<TT, 4, 64>(q, grid, s);
}

}  // namespace

int dw_general(const void *Xs, const void *Ys, const void *Ind, void *dW, void *workspace, const egs_dims *d,
               int64_t ldx_b, int64_t ldx_t, int act_dtype, int out_dtype, int ind_dtype, int dw_layout,
               const DwPlan &pl, hipStream_t s)
{
    const size_t w_elems = (size_t)d->E * d->I * d->J;
    const int ES = elem_size(act_dtype);
    DwParams p;
    memset(&p, 0, sizeof(p));
    p.Xs = (const char *)Xs; p.Ys = (const char *)Ys; p.Ind = Ind;
    p.part = (float *)workspace; p.dW = (char *)dW;
    p.B = d->B; p.T = d->T; p.E = d->E; p.K = d->K; p.I = d->I; p.J = d->J;
    p.ldx_b = ldx_b; p.ldx_t = ldx_t;
    p.ind_dtype = ind_dtype;
    p.out_dtype = out_dtype; p.dw_layout = dw_layout;
    const uint64_t x_span = d->B > 0 && d->T > 0
        ? ((uint64_t)(d->B - 1) * (uint64_t)ldx_b + (uint64_t)(d->T - 1) * (uint64_t)ldx_t + (uint64_t)d->I) * ES : 0;
    const uint64_t y_span = (uint64_t)d->B * d->E * d->K * d->J * ES;
    if (dw_big_takes(pl, Xs, Ys, dW, d, ldx_b, ldx_t, act_dtype)) {
        DwDlParams q;
        q.d = p;
        q.d.i_tiles = pl.b_i_tiles; q.d.j_tiles = pl.b_j_tiles; q.d.S = pl.b_S; q.d.rows_per_split = pl.b_rows_per_split;
        q.x_bytes = (uint32_t)x_span; q.y_bytes = (uint32_t)y_span;
        const int64_t per_e = (int64_t)pl.b_i_tiles * pl.b_j_tiles * pl.b_S;
        const int64_t grid = pl.b_tp != 0 ? (d->E * per_e + 7) / 8 * 8 : 8 * ceil_div(d->E, 8) * per_e;
        if (grid > INT32_MAX) return EGS_ERR_BAD_SHAPE;
        // 128-column tiles: three 48 KB stages of 64 rows (C4: 42.2 -> 37.9 us per weight gradient with its sum over
        // splits); 256-column tiles: four 32 KB stages of 32 rows (C3: 178 -> 174 us)
        if (pl.b_tp != 0) {
            const int rc = act_dtype == EGS_F16 ? launch_dw_strip<ElemF16>(q, pl.b_tp, pl.b_bq, (int)grid, s)
                                                : launch_dw_strip<ElemBF16>(q, pl.b_tp, pl.b_bq, (int)grid, s);
            if (rc != EGS_OK) return rc;
        } else if (act_dtype == EGS_F16) {
            if (pl.b_bq == 256) hipLaunchKernelGGL((dw_dl_kernel<ElemF16, 256, 4, 32>), dim3((unsigned)grid), dim3(kDlThreads), 0, s, q);
            else hipLaunchKernelGGL((dw_dl_kernel<ElemF16, 128, 3>), dim3((unsigned)grid), dim3(kDlThreads), 0, s, q);
        } else {
            if (pl.b_bq == 256) hipLaunchKernelGGL((dw_dl_kernel<ElemBF16, 256, 4, 32>), dim3((unsigned)grid), dim3(kDlThreads), 0, s, q);
            else hipLaunchKernelGGL((dw_dl_kernel<ElemBF16, 128, 3>), dim3((unsigned)grid), dim3(kDlThreads), 0, s, q);
        }
        if (pl.b_tp == 0) EGS_CHECK_LAUNCH("dw_dl_kernel");
        if (pl.b_S > 1) {       // partials are in the output's layout, I % 8 == 0 and J % 8 == 0: vectorised plain sum
            hipLaunchKernelGGL(dw_reduce4_kernel, dim3(grid_1d(w_elems / 4, 4096)), dim3(kThreads), 0, s,
                               (const float *)workspace, (char *)dW, pl.b_S, w_elems / 4, out_dtype);
            EGS_CHECK_LAUNCH("dw_reduce4_kernel");
        }
        return EGS_OK;
    }
    // operands of less than 16 bytes, which tiny_dw_kernel takes: whole sums, however many picks
    const bool split32 = pl.split32 && x_span < (1ull << 31) && y_span < (1ull << 31);
    const int S = x_span < 16 || y_span < 16 ? 1 : split32 ? pl.f_S : pl.S;
    TiledDwParams q;
    memset(&q, 0, sizeof(q));
    q.Xs = p.Xs; q.Ys = p.Ys; q.Ind = Ind; q.dW = S > 1 ? (char *)workspace : (char *)dW;
    q.x_bytes = (int64_t)x_span; q.y_bytes = (int64_t)y_span;
    q.ldx_b = ldx_b; q.ldx_t = ldx_t;
    q.B = d->B; q.T = d->T; q.E = d->E; q.K = d->K; q.I = d->I; q.J = d->J;
    q.ind_dtype = ind_dtype; q.out_dtype = out_dtype; q.eji = dw_layout != 0;
    q.i_tiles = pl.i_tiles; q.j_tiles = pl.j_tiles; q.S = S; q.picks_per_split = split32 ? pl.f_picks_per_split : pl.picks_per_split;
    q.wide = pl.wide; q.split32 = split32;
    q.edges = (d->I * ES) % 16 != 0 || (d->J * ES) % 16 != 0;
    const int rc = act_dtype == EGS_F32 ? tiled_dw_f32(q, s) : act_dtype == EGS_F16 ? tiled_dw_f16(q, s) : tiled_dw_bf16(q, s);
    if (rc != EGS_OK || S <= 1) return rc;
    hipLaunchKernelGGL(tiled_dw_sum_kernel, dim3(grid_1d((w_elems + 3) / 4, 4096)), dim3(kThreads), 0, s, (const float *)workspace,
                       (char *)dW, S, (int64_t)w_elems, out_dtype);
    EGS_CHECK_LAUNCH("tiled_dw_sum_kernel");
    return EGS_OK;
}


}  // namespace host
}  // namespace egs
