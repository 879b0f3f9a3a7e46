// Host side of the library: argument validation, workspace plans, kernel selection and the C ABI
// declared in include/egs_hip.h.  The launches of kernels that are templates live in units of their own, so that
// they build side by side: egs_rows_launch.hip (products), egs_stream_launch.hip (few rows), egs_f8_launch.hip, egs_dw_launch.hip
// (weight gradients), egs_tiled_*.hip (any size), egs_small_*.hip and egs_fused_*.hip (small experts), egs_sum_launch.hip (tables and
// sums), egs_pass_launch.hip, egs_mlp_launch.hip, egs_bias.hip, egs_router.hip.
#include "egs_host.h"
#include "../../include/egs_hip_testing.h"
#include "egs_device.h"
#include "egs_jobs.h"
#include "egs_small_f32.h"

#include <atomic>
#include <mutex>

using namespace egs;
using namespace egs::host;

namespace egs {
namespace host {

std::atomic<bool> g_force_generic{false};
static thread_local char g_hip_error_buf[256] = "";

int hip_fail(hipError_t err, const char *what)
{
    snprintf(g_hip_error_buf, sizeof(g_hip_error_buf), "%s: %s", what, hipGetErrorString(err));
    return EGS_ERR_HIP;
}
const char *last_hip_error() { return g_hip_error_buf; }

struct LaunchLog { bool on; size_t len; char text[1024]; };
static thread_local LaunchLog g_launch_log = {false, 0, ""};
void note_launch(const char *what)
{
    LaunchLog &l = g_launch_log;
    if (!l.on) return;
    const size_t n = strlen(what);
    if (l.len + n + 2 > sizeof(l.text)) return;
    if (l.len > 0) l.text[l.len++] = ',';
    memcpy(l.text + l.len, what, n + 1);
    l.len += n;
}

static std::mutex g_lds_mutex;
int allow_large_lds(const void *fn, LdsGrant &grant, size_t lds, const char *what)
{
    if (lds <= 64 * 1024) return EGS_OK;
    int dev = -1;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return hip_fail(err, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return EGS_ERR_UNSUPPORTED;
    if (grant.bytes[dev].load(std::memory_order_acquire) >= lds) return EGS_OK;
    std::lock_guard<std::mutex> lock(g_lds_mutex);
    if (grant.bytes[dev].load(std::memory_order_relaxed) >= lds) return EGS_OK;
    err = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return hip_fail(err, what);
    grant.bytes[dev].store((uint32_t)lds, std::memory_order_release);
    return EGS_OK;
}

}  // namespace host
}  // namespace egs

namespace {

// ------------------------------------------------------------------------------ built-in scratch
// Device memory that exists from the moment the library's code object is loaded, for the one entry
// point that serves callers which cannot allocate (egs_dw_builtin_scratch).  Every GPU the library
// runs on holds its own copy of the array, at its own address, until the process ends.
// The array's name is only a host-side handle: host code never passes it to a kernel or a copy.  The
// device address is looked up once per device (with that device current) and kept.
static __device__ __align__(256) unsigned char scratch[EGS_BUILTIN_SCRATCH_BYTES];

std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices];              // per device: address of that device's copy of `scratch`

int builtin_scratch_ptr(void **out)
{
    int dev = -1;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess) return hip_fail(err, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return EGS_ERR_UNSUPPORTED;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void *ptr = nullptr;
        err = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess) return hip_fail(err, "hipGetSymbolAddress(scratch)");
        if (ptr == nullptr) return EGS_ERR_HIP;
        g_scratch_ptr[dev] = ptr;
    }
    *out = g_scratch_ptr[dev];
    return EGS_OK;
}

bool act_dtype_ok(int d) { return d == EGS_F32 || d == EGS_F16 || d == EGS_BF16; }
bool ind_dtype_ok(int d) { return d >= EGS_IND_I16 && d <= EGS_IND_U8; }
bool layout_ok(int l) { return l == EGS_W_EIJ || l == EGS_W_EJI; }
bool mode_ok(int m) { return m == EGS_SCATTER_DETERMINISTIC || m == EGS_SCATTER_ATOMIC || m == EGS_SCATTER_COMPACT; }

int check_dims(const egs_dims *d)
{
    if (d == nullptr) return EGS_ERR_NULL_POINTER;
    if (d->B < 0 || d->T < 0 || d->E < 0 || d->K < 0 || d->I < 0 || d->J < 0) return EGS_ERR_BAD_SHAPE;
    // row counts and per-batch pick counts are held in 32-bit ints inside the kernels
    if ((int64_t)d->B * d->K > INT32_MAX || (int64_t)d->E * d->K > INT32_MAX) return EGS_ERR_BAD_SHAPE;
    if ((int64_t)d->B * d->T > INT32_MAX) return EGS_ERR_BAD_SHAPE;
    return EGS_OK;
}

// ------------------------------------------------------------------------------ plans
struct ScatterPlan {
    size_t seg_off_at, perm_at, rank_at, cnt_at, long_tab_at, long_part_at, rows_at;   // byte offsets inside the workspace
    size_t bytes;
};

// Workspace of the GEMM-scatter, for the kernels that will run:
//   fp32 atomic mode and the one-kernel scatter of small experts (`fused`) need none;
//   otherwise: routing table (segment offsets, picks in token order, scratch ranks, optional global counters),
//   long-segment records and partial rows, and the product rows in pick order - fp32 in deterministic mode
//   (fp32 accumulation with one final rounding), the element type in atomic ("fast") mode with 16-bit types
//   (half the traffic, one extra rounding per pick; the summation order is still fixed).
//   the one-kernel scatter in passes (SCATTER_PASS) needs nothing either (it sorts each pass's picks in LDS);
enum ScatterPath { SCATTER_FUSED, SCATTER_PASS, SCATTER_ROWS };

ScatterPlan plan_scatter(const egs_dims *d, int mode, int act_dtype, ScatterPath path)
{
    ScatterPlan pl;
    memset(&pl, 0, sizeof(pl));
    const size_t N = (size_t)d->E * d->K;
    if (mode == EGS_SCATTER_ATOMIC && act_dtype == EGS_F32) return pl;
    if (path == SCATTER_FUSED || path == SCATTER_PASS) return pl;
    const size_t row_es = (mode != EGS_SCATTER_ATOMIC || act_dtype == EGS_F32) ? 4 : (size_t)elem_size(act_dtype);
    size_t at = 0;
    pl.seg_off_at = at; at += align_up((size_t)d->B * ((size_t)d->T + 1) * 4, 256);
    pl.perm_at = at;    at += align_up((size_t)d->B * N * 4, 256);
    pl.rank_at = at;    at += align_up((size_t)d->B * N * 4, 256);
    pl.cnt_at = at;     at += d->T > kCsrLdsTokens ? align_up((size_t)d->B * d->T * 4, 256) : 0;
    // long segments (tokens picked more than kLongSegment times): records and fp32 partial rows
    pl.long_tab_at = at;  at += align_up((size_t)d->B * long_tab_stride((int)N) * 4, 256);
    pl.long_part_at = at; at += align_up((size_t)d->B * long_max_slots((int)N) * d->I * 4, 256);
    pl.rows_at = at;    at += align_up((size_t)d->B * N * product_ld(d->I) * row_es, 256);
    pl.bytes = at;
    return pl;
}

// Experts of few picks: dW itself is what takes the time, and tiled_dw_wide_kernel writes it as whole rows.  Each of its workgroups
// goes through all picks, so there have to be enough of them for the number of picks.  us, this kernel and the next best: bf16 B1
// T256 E128 K4 I1024 J128 16 and 82, B3 T169 E86 K58 I384 J64 11 and 17; with fewer tiles bf16 B4 E6 K21 I64 J64 6.7 and 4.5.
// Sizes that only tiled_dw_kernel takes otherwise: fp32 B16 E50 K32 I300 J150 41 and 58 (750 tiles), bf16 B20 E60 K100 I500 J250 76
// and 138 (960), fp32 B32 E128 K64 I100 J75 110 and 102 (512), bf16 B6 E20 K80 I100 J60 15 and 7 (40).
int64_t dw_wide_tiles(const egs_dims *d, int act_dtype)
{
    return (int64_t)d->E * ceil_div(d->I, 64) * ceil_div(d->J, act_dtype == EGS_F32 ? 64 : 128);
}
bool dw_few_picks(const egs_dims *d, int act_dtype) { return (int64_t)d->B * d->K <= 256 && dw_wide_tiles(d, act_dtype) >= 256; }

// fp32: 32-pick slabs that the 64 x 64 tiles of tiled_dw_split_kernel go through in all
int64_t dw_split32_slabs(const egs_dims *d)
{
    return (int64_t)d->E * ceil_div(d->I, 64) * ceil_div(d->J, 64) * (((int64_t)d->B * d->K + 31) / 32);
}

// Is tiled_dw_split_kernel, in the parts of `pl`, the faster one?  Some hundred slabs are needed in any case.
// Against tiled_dw_wide_kernel, which has the same tiles: from 64 picks on (us, it / that: 12 picks 19.6 / 16.8, 20 picks 9.4 / 8.5, 34 picks
// 12.7 / 12.0, 48 level, 99 picks at B3 E150 I70 J130 0.91 of it, 155 picks at B1 T712 E125 I369 J128 28.4 / 34.5).
// Against the 32 x 32 tiles of tiled_dw_kernel by the time that the fullest CU takes, fitted to 1101 sizes alone on the device: up to three
// workgroups of it on a CU, two of those, each some us, and some for every 32 picks (128) that a CU's workgroups go through, plus the
// second pass.  Within 10 and 12 % of the time at 95 % of the sizes; by it 13 sizes are 3 % slower than on the fp32 instruction and none more
// than 10 %.  us, it / that: B53 T97 E29 K41 I111 J75 30 / 43, B12 T121 E52 K61 I272 J31 (59 % of the tiles empty) 30 / 18.6, B26 T665 E30 K30 I523
// J32 33 / 23.5, B20 T289 E33 K163 I693 J29 111 / 90.
bool dw_split32_pays(const egs_dims *d, const DwPlan &pl)
{
    const int64_t Me = (int64_t)d->B * d->K;
    if (Me < 512 && dw_split32_slabs(d) < 600) return false;
    if (pl.wide) return Me >= 64;
    const int64_t split = ((int64_t)d->E * ceil_div(d->I, 64) * ceil_div(d->J, 64) * pl.f_S + 255) / 256;
    const int64_t plain = ((int64_t)d->E * pl.i_tiles * pl.j_tiles * pl.S + 255) / 256;
    const double elems = (double)d->E * d->I * d->J;
    const double split_us = 6.2 * (double)((split + 2) / 3) + 0.56 * (double)split * (pl.f_picks_per_split / 32) + (pl.f_S > 1 ? 1.9 + 2.5e-6 * pl.f_S * elems : 0.0);
    const double plain_us = 2.7 + 3.4 * (double)((plain + 1) / 2) + 1.08 * (double)plain * (((int64_t)pl.picks_per_split + 127) / 128) +
                            (pl.S > 1 ? 3.0 + 2.8e-6 * pl.S * elems : 0.0);
    return split_us < plain_us;
}

// 16-bit weight gradients in strips: the tile (32 tp x bq) and the number of splits of the picks that dw_strip_kernel is expected to be
// the fastest with, and the us that takes: rounds of workgroups over the CUs, each some us and some more for every 1000 picks, fitted to
// times alone on the device.
struct DwStripPlan { int tp, bq, S, rows_per_split; double us; };

DwStripPlan dw_strip_plan(const egs_dims *d)
{
    struct Width { int tp, bq; double start, per_pick; };
    static constexpr Width widths[] = {{2, 64, 2.4, 5.8e-3}, {3, 64, 3.0, 7.3e-3}, {4, 64, 2.6, 10.0e-3}, {4, 128, 4.5, 11.7e-3}};
    constexpr double second_pass = 4.0, per_sum = 2e-6;
    const int64_t Me = (int64_t)d->B * d->K;
    DwStripPlan best = {0, 0, 0, 0, 0.0};
    for (const Width &w : widths) {
        if (w.bq == 128 && d->J <= 64) continue;
        const int64_t tiles = (int64_t)d->E * ceil_div(d->I, 32 * w.tp) * ceil_div(d->J, w.bq), most = tiles < 256 ? 256 / tiles : 1;
        for (int64_t n = 1; n <= most; n += most > 1 ? most - 1 : 1) {
            const int64_t rows = ((Me + n - 1) / n + 127) / 128 * 128, S = (Me + rows - 1) / rows;
            const double us = (double)((tiles * S + 255) / 256) * (w.start + (double)rows * w.per_pick) +
                              (S > 1 ? second_pass + (double)S * d->E * d->I * d->J * per_sum : 0.0);
            if (best.tp == 0 || us < best.us) best = {w.tp, w.bq, (int)S, (int)(rows < INT32_MAX ? rows : INT32_MAX), us};
        }
    }
    return best;
}

// Up to 64 output columns, against the 32 x 64 and 32 x 32 tiles of make_dw_tile, modelled the same way.  us, strips / those: B64 T256 E32 K32
// I768 J64 18.8 / 28.4, B2 T1000 E60 K200 I640 J48 12 / 20, B8 T4096 E128 K256 I1024 J64 95 / 147, B100 T500 E6 K100 I448 J64 18 / 33, B20
// T900 E14 K64 I1024 J32 10.4 / 11.6, B7 T500 E80 K64 I192 J64 5.6 / 9.2; not taken: I256 J64 at E32 and 2048 picks 13.2 / 10.0, B40 T400
// E16 K40 I640 J24 11.8 / 11.3, B1 T2000 E8 K250 I256 J64 4.7 / 3.7.  Where those are not taken the general tiles always lose: B3 T120 E5
// K90 I200 J56 4.3 / 8.6, B17 T2218 E4 K63 I224 J32 9.3 / 13.2, B2 T300 E100 K100 I160 J32 5.4 / 10.4, B30 T200 E4 K20 I136 J24 5.6 / 9.3.
bool dw_strip_narrow(const egs_dims *d, int act_dtype, DwStripPlan *plan = nullptr)
{
    const int64_t Me = (int64_t)d->B * d->K;
    if (act_dtype == EGS_F32 || d->I % 8 || d->J % 8 || d->I <= 128 || d->J > 64 || d->J < 8 || Me < 128 || d->E == 0) return false;
    const int64_t narrow = (int64_t)d->E * ceil_div(d->I, 32) * ceil_div(d->J, 32), wide = (int64_t)d->E * ceil_div(d->I, 32);
    const bool alone = narrow < 128 || d->I > 2048 || dw_few_picks(d, act_dtype);       // make_dw_tile refuses these
    if (alone && plan == nullptr) return true;
    const DwStripPlan strip = dw_strip_plan(d);
    if (plan != nullptr) *plan = strip;
    if (alone) return true;
    const double tile = d->J > 32 && (narrow > 256 || Me >= 4096) ? (double)((wide + 255) / 256) * (2.9 + (double)Me * 3.0e-3)
                                                                  : (double)((narrow + 511) / 512) * (2.9 + (double)Me * 5.0e-3);
    return strip.us < 0.95 * tile;
}

// More columns, against the 256-row tiles of dw_dl_kernel and their sum over splits (an XCD takes whole experts there).  us, strips / those:
// B6 T1100 E20 K150 I328 J136 10.1 / 24.2, B16 T1024 E64 K128 I512 J128 30 / 37, B12 T1000 E5 K100 I1000 J256 12 / 26, B8 T1024 E16 K128
// I512 J256 13 / 30, B40 T300 E40 K40 I256 J192 17 / 40, B3 T1000 E90 K250 I736 J200 64 / 83; not taken: B8 T4096 E128 K256 I1024 J256
// 219 / 180.  (With fewer than 256 picks the general tiles are as fast: B1 T4000 E64 K250 I1024 J256 30.3 / 31.6, B1 T700 E120 K150 I384
// J256 20.5 / 20.0.)  With up to 128 rows and more than 128 columns the general tiles are the alternative: B4 T500 E30 K100 I96 J192
// 5.8 / 9.7, B20 T400 E12 K50 I64 J256 7.9 / 11.1, B30 T300 E40 K40 I32 J160 9.6 / 15.0, B6 T2000 E3 K200 I128 J224 10.0 / 11.6.
bool dw_strip_broad(const egs_dims *d, int act_dtype, const DwPlan &pl, DwStripPlan &strip)
{
    if (act_dtype == EGS_F32 || d->I % 8 || d->J % 8 || d->J <= 64 || d->I < 32 || d->E == 0) return false;
    if (!pl.big_ok && (d->I > 128 || d->J <= 128 || (int64_t)d->B * d->K < 128)) return false;
    // (half the rows of a strip empty, and CUs enough to fill with less: I32 J192 E46 7568 picks 42 / 32, J144 E117 1204 picks 18.4 / 16.8)
    if (d->I <= 32 && (int64_t)d->E * ceil_div(d->J, 64) >= 128 && (int64_t)d->B * d->K >= 384) return false;
    strip = dw_strip_plan(d);
    if (!pl.big_ok) return true;
    const int64_t on_xcd = (int64_t)ceil_div(d->E, 8) * pl.b_i_tiles * pl.b_j_tiles * pl.b_S;
    const double per_round = pl.b_bq == 256 ? 9.5 + pl.b_rows_per_split * 39e-3 : 7.0 + pl.b_rows_per_split * 20e-3;
    const double us = (double)((on_xcd + 31) / 32) * per_round + (pl.b_S > 1 ? 3.5 + (double)pl.b_S * d->E * d->I * d->J * 0.45e-6 : 0.0);
    return strip.us < 0.95 * us;
}

DwPlan plan_dw(const egs_dims *d, int act_dtype)
{
    DwPlan pl;
    memset(&pl, 0, sizeof(pl));
    // any shape: 32 x 64 tiles (fp32: 32 x 32), the picks split only where there are more than a workgroup's four wavefronts
    // reduce in about the time the second pass would cost (1024) and too few tiles to fill the device
    const int64_t Me = (int64_t)d->B * d->K;
    pl.i_tiles = ceil_div(d->I, 32);
    pl.j_tiles = ceil_div(d->J, act_dtype == EGS_F32 ? 32 : 64);
    const int64_t base = (int64_t)d->E * pl.i_tiles * pl.j_tiles;
    int64_t S = base > 0 ? 512 / base : 1;
    if (S > (Me + 1023) / 1024) S = (Me + 1023) / 1024;
    if (S < 1) S = 1;
    int64_t rows = Me > 0 ? ((Me + S - 1) / S + 127) / 128 * 128 : 128;
    S = Me > 0 ? (Me + rows - 1) / rows : 1;
    pl.S = (int)S;
    pl.picks_per_split = (int)(rows < INT32_MAX ? rows : INT32_MAX);
    pl.wide = Me <= 128 || (Me <= 512 && dw_wide_tiles(d, act_dtype) >= 256) || dw_wide_tiles(d, act_dtype) >= 768;
    if (act_dtype == EGS_F32 && Me > 0) {
        // two workgroups per CU where that leaves four slabs or more to each
        const int64_t tiles = (int64_t)d->E * ceil_div(d->I, 64) * ceil_div(d->J, 64);
        int64_t parts = tiles > 0 ? 512 / tiles : 1;
        if (parts > Me / 128) parts = Me / 128;
        if (parts < 1) parts = 1;
        rows = ((Me + parts - 1) / parts + 31) / 32 * 32;
        pl.f_S = (int)((Me + rows - 1) / rows);
        pl.f_picks_per_split = (int)(rows < INT32_MAX ? rows : INT32_MAX);
        pl.split32 = dw_split32_pays(d, pl);
        if (pl.split32 && S < pl.f_S) S = pl.f_S;       // workspace for either
    }
    pl.bytes_general = S > 1 ? align_up((size_t)S * d->E * d->I * d->J * 4, 256) : 256;     // never none: this path always has a workspace

    // large 16-bit shapes: 256 x 256 (or 256 x 128) tiles, 64-row slabs, splits only to give every CU a workgroup
    // (C4: 2 splits 42 us, 4 splits 49 us, none 50 us)
    pl.big_ok = act_dtype != EGS_F32 && d->I % 8 == 0 && d->J % 8 == 0 && d->I > 128 && d->J > 64 && Me >= 256 && d->E > 0;
    if (pl.big_ok) {
        pl.b_bq = d->J > 128 ? 256 : 128;
        pl.b_i_tiles = ceil_div(d->I, 256);
        pl.b_j_tiles = ceil_div(d->J, pl.b_bq);
        const int64_t tiles = (int64_t)d->E * pl.b_i_tiles * pl.b_j_tiles;
        int64_t s3 = (256 + tiles - 1) / tiles;
        const int64_t most = (Me + 255) / 256;              // at least four slabs per split
        if (s3 > most) s3 = most;
        if (s3 > 32) s3 = 32;
        if (s3 < 1) s3 = 1;
        int64_t r3 = ((Me + s3 - 1) / s3 + 63) / 64 * 64;
        s3 = (Me + r3 - 1) / r3;
        pl.b_S = (int)s3;
        pl.b_rows_per_split = (int)r3;
        pl.bytes_big = s3 > 1 ? align_up((size_t)s3 * d->E * d->I * d->J * 4, 256) : 0;
    }

    DwStripPlan strip;
    if (dw_strip_narrow(d, act_dtype, &strip) || dw_strip_broad(d, act_dtype, pl, strip)) {
        pl.big_ok = true;
        pl.b_bq = strip.bq;
        pl.b_tp = strip.tp;
        pl.b_i_tiles = ceil_div(d->I, 32 * strip.tp);
        pl.b_j_tiles = ceil_div(d->J, strip.bq);
        pl.b_S = strip.S;
        pl.b_rows_per_split = strip.rows_per_split;
        // never less than the 256-row tiles ask for: which sizes fit a scratch of a given size does not depend on the choice between the two
        const size_t bytes = strip.S > 1 ? align_up((size_t)strip.S * d->E * d->I * d->J * 4, 256) : 0;
        if (bytes > pl.bytes_big) pl.bytes_big = bytes;
    }

    // small experts: 64 x 64 tiles, up to 1024 picks per workgroup, enough workgroups to cover the device
    pl.small_ok = act_dtype != EGS_F32 && d->I % 8 == 0 && d->J % 8 == 0 && d->I >= 8 && d->J >= 8 && d->I <= 128 &&
                  d->J <= 128 && Me > 0 && d->E > 0 && !dw_few_picks(d, act_dtype);
    if (pl.small_ok) {
        pl.s_i_tiles = ceil_div(d->I, 64);
        pl.s_j_tiles = ceil_div(d->J, 64);
        const int64_t tiles = (int64_t)d->E * pl.s_i_tiles * pl.s_j_tiles;
        int64_t s2 = (256 + tiles - 1) / tiles;
        const int64_t need = (Me + kDwSmallMaxRows - 1) / kDwSmallMaxRows, most = (Me + 127) / 128;
        if (s2 < need) s2 = need;
        if (s2 > most) s2 = most;
        int64_t r2 = ((Me + s2 - 1) / s2 + 127) / 128 * 128;
        s2 = (Me + r2 - 1) / r2;
        pl.s_S = (int)s2;
        pl.s_rows_per_split = (int)r2;
        pl.bytes_small = s2 > 1 ? align_up((size_t)s2 * d->E * d->I * d->J * 4, 256) : 0;
    }
    return pl;
}

// ------------------------------------------------------------------------------ small-expert fast paths
constexpr uint64_t kSpan32 = 0xFFFFFFFFull;      // the small kernels address with 32-bit byte offsets

bool small_shape_ok(int act_dtype, int R, int N)
{
    return act_dtype != EGS_F32 && (R == 32 || R == 64 || R == 128) && N % 8 == 0 && N >= 8 && N <= 128;
}

// A routing table in caller-owned memory (egs_routing_table_bytes): seg [B][T+1], perm [B][E*K], the picks of each batch
// element in a stable order by token.  Built once per Ind by a gather forward, read by the one-kernel scatters that follow.
struct RoutingTable { int32_t *seg, *perm; };


// Workgroup -> (expert, row tile) map of the small-expert row kernels (decode_rows_block): which operand is worth keeping
// XCD-local - the source rows, each read by ~E*K/T experts and fetched from beyond the L2 once per XCD that uses them,
// or W(e), fetched once per XCD that runs one of the expert's row tiles.  Row tiles take the XCDs only where that leaves none
// idle: in groups of eight, or 2 / 4 of them on 4 / 2 XCDs each.
// whether the routing table that rides in a gather launch is built by two workgroups per batch element
// (csr_count_half_body) instead of one: its shares must fit the registers and its counters a modest piece of LDS, there must
// be picks enough to split, and the launch must not grow beyond what the device holds at once (two of these kernels'
// workgroups fit a CU)
bool table_split_pays(const egs_dims *d, int nwaves, int gather_blocks, int round_blocks)
{
    const int64_t N = (int64_t)d->E * d->K;
    return N >= 256 && N <= (int64_t)nwaves * 1024 && csr_half_lds(d->T, nwaves) <= 64 * 1024 &&
           (int64_t)gather_blocks + 2 * (int64_t)d->B <= round_blocks;
}
int rows_xcd_map(const egs_dims *d, int R, int N, int es, int tiles_per_e)
{
    const double picks_per_token = (double)d->E * d->K / (d->T > 0 ? d->T : 1);
    const double x_bytes = (double)d->B * d->T * R * es, w_bytes = (double)d->E * R * N * es;
    const double by_expert = x_bytes * (picks_per_token < 8 ? (picks_per_token < 1 ? 1 : picks_per_token) : 8) + w_bytes;
    const double by_rows = x_bytes + w_bytes * (tiles_per_e < 8 ? tiles_per_e : 8);
    if (by_rows >= by_expert) return 0;
    if (tiles_per_e == 2 || tiles_per_e == 4) return 8 / tiles_per_e;
    return (tiles_per_e % 8 == 0 || tiles_per_e > 16) ? 1 : 0;
}
int rows_xcd_blocks(int map, int tiles_per_e, int E)
{
    return map == 0 ? 8 * ceil_div(E, 8) * tiles_per_e : map == 1 ? 8 * ceil_div(tiles_per_e, 8) * E : 8 * ceil_div(E, map);
}

bool make_gather_small(const void *X, const void *W, const void *Ind, void *Y, const egs_dims *d, int64_t ldx_b,
                       int64_t ldx_t, int act_dtype, int w_dtype, int ind_dtype, int w_layout, SmallRowsJob &j,
                       const RoutingTable *build = nullptr, int act = ACT_NONE)
{
    const int R = d->I, N = d->J;
    if (g_force_generic || w_dtype != act_dtype || !small_shape_ok(act_dtype, R, N)) return false;
    if (!aligned_to(X, 16) || !aligned_to(W, 16) || !aligned_to(Y, 16)) return false;
    if ((ldx_b * 2) % 16 || (ldx_t * 2) % 16 || d->T == 0) return false;
    const int64_t Me = (int64_t)d->B * d->K;
    if (Me == 0 || d->E == 0) return false;
    const uint64_t x_span = ((uint64_t)(d->B - 1) * (uint64_t)ldx_b + (uint64_t)(d->T - 1) * (uint64_t)ldx_t + R) * 2;
    if (x_span > kSpan32 || (uint64_t)d->E * R * N * 2 > kSpan32 || (uint64_t)Me * d->E * N * 2 > kSpan32) return false;
    memset(&j, 0, sizeof(j));
    SmallRowsParams &p = j.p;
    p.A = (const char *)X; p.W = (const char *)W; p.Ind = Ind; p.C = (char *)Y;
    p.B = d->B; p.T = d->T; p.E = d->E; p.K = d->K; p.N = N;
    p.lda_b = ldx_b; p.lda_t = ldx_t; p.ind_dtype = ind_dtype;
    p.tiles_per_e = (int)((Me + 255) / 256);
    if ((int64_t)8 * (ceil_div(d->E, 8) + 1) * (p.tiles_per_e + 8) > INT32_MAX / 2) return false;
    p.rows_share_xcd = rows_xcd_map(d, R, N, 2, p.tiles_per_e);
    p.act = act;
    j.R = R; j.act_dtype = act_dtype; j.gather = true; j.out_f32 = false; j.lds = 0;
    j.nmajor = (w_layout == EGS_W_EIJ);                 // [E,I,J] = [E,R,N]
    if (build != nullptr) {             // the routing table of a later scatter rides along: B more workgroups, first in line
        p.csr_blocks = d->B;
        p.seg_off = build->seg; p.perm = build->perm;
        j.lds = csr_count_lds(d->T, 4);
        // ... or 2 B, each ranking half of the picks (the ranking is what the build consists of, and the gather's workgroups
        // alone take less time than one workgroup's whole table: B64 T256 E32 K32, 6.8 -> 6.3 us for the launch)
        const int gather_blocks = rows_xcd_blocks(p.rows_share_xcd, p.tiles_per_e, p.E);
        if (table_split_pays(d, 4, gather_blocks, 512)) { p.csr_blocks = 2 * d->B; p.csr_split = 1; j.lds = csr_half_lds(d->T, 4); }
    }
    j.blocks = rows_xcd_blocks(p.rows_share_xcd, p.tiles_per_e, p.E) + p.csr_blocks;
    return true;
}

// product rows of the scatter in pick order; with `ride` the routing table is built by extra
// workgroups of the same launch
bool make_scatter_rows_small(const void *Y, const void *W, void *rows, bool rows_f32, const egs_dims *d, int act_dtype,
                             int w_layout, bool ride, const void *Ind, int ind_dtype, int32_t *seg_off, int32_t *perm,
                             int32_t *rank_tmp, int32_t *long_tab, SmallRowsJob &j)
{
    const int R = d->J, N = d->I;
    if (g_force_generic || !small_shape_ok(act_dtype, R, N)) return false;
    if (!aligned_to(Y, 16) || !aligned_to(W, 16)) return false;
    const int64_t Me = (int64_t)d->B * d->K;
    if (Me == 0 || d->E == 0) return false;
    if ((uint64_t)Me * d->E * R * 2 > kSpan32 || (uint64_t)d->E * R * N * 2 > kSpan32 ||
        (uint64_t)Me * d->E * N * 4 > kSpan32) return false;
    memset(&j, 0, sizeof(j));
    SmallRowsParams &p = j.p;
    p.A = (const char *)Y; p.W = (const char *)W; p.C = (char *)rows;
    p.B = d->B; p.T = d->T; p.E = d->E; p.K = d->K; p.N = N;
    p.tiles_per_e = (int)((Me + 255) / 256);
    if (ride) {
        p.csr_blocks = d->B; p.Ind = Ind; p.ind_dtype = ind_dtype;
        p.seg_off = seg_off; p.perm = perm; p.rank_tmp = rank_tmp; p.long_tab = long_tab;
        j.lds = csr_count_lds(d->T, 4);
    }
    if ((int64_t)8 * ceil_div(d->E, 8) * p.tiles_per_e + p.csr_blocks > INT32_MAX / 2) return false;
    j.R = R; j.act_dtype = act_dtype; j.gather = false; j.out_f32 = rows_f32;
    j.nmajor = (w_layout == EGS_W_EJI);                 // [E,J,I] = [E,R,N]
    j.blocks = 8 * ceil_div(p.E, 8) * p.tiles_per_e + p.csr_blocks;
    return true;
}

bool make_dw_small(const void *Xs, const void *Ys, const void *Ind, void *dW, void *workspace, const egs_dims *d,
                   int64_t ldx_b, int64_t ldx_t, int act_dtype, int out_dtype, int ind_dtype, int dw_layout,
                   const DwPlan &pl, SmallDwJob &j)
{
    if (!pl.small_ok || g_force_generic || d->T == 0) return false;
    const uint64_t x_span = ((uint64_t)(d->B - 1) * (uint64_t)ldx_b + (uint64_t)(d->T - 1) * (uint64_t)ldx_t + d->I) * 2;
    if (!aligned_to(Xs, 16) || !aligned_to(Ys, 16) || !aligned_to(dW, 16) || (ldx_b * 2) % 16 || (ldx_t * 2) % 16) return false;
    if (x_span > kSpan32 || (uint64_t)d->B * d->E * d->K * d->J * 2 > kSpan32) return false;
    if ((int64_t)8 * ceil_div(d->E, 8) * pl.s_i_tiles * pl.s_j_tiles * pl.s_S > INT32_MAX / 2) return false;
    memset(&j, 0, sizeof(j));
    SmallDwParams &q = j.q;
    q.Xs = (const char *)Xs; q.Ys = (const char *)Ys; q.Ind = Ind; q.part = (float *)workspace; q.dW = (char *)dW;
    q.B = d->B; q.T = d->T; q.E = d->E; q.K = d->K; q.I = d->I; q.J = d->J;
    q.ldx_b = ldx_b; q.ldx_t = ldx_t; q.ind_dtype = ind_dtype;
    q.i_tiles = pl.s_i_tiles; q.j_tiles = pl.s_j_tiles; q.S = pl.s_S; q.rows_per_split = pl.s_rows_per_split;
    q.out_dtype = out_dtype; q.dw_layout = dw_layout;
    j.blocks = 8 * ceil_div(d->E, 8) * pl.s_i_tiles * pl.s_j_tiles * pl.s_S;
    j.act_dtype = act_dtype;
    j.w_elems = (size_t)d->E * d->I * d->J;
    return true;
}

// The one-pass weight gradient (32 x 32 tiles of dW(e), every workgroup reduces all picks of its expert) is taken
// when its tiles alone fill the device; with fewer tiles the picks are split instead (dw_small_kernel + second pass).
// `shared`: in the launch of a scatter, where strips would be one or two launches of their own (gather's backward, us, with strips / shared:
// B50 T45 E16 K45 I160 J64 28.5 / 19.8, B12 T1243 E15 K21 I192 J64 17.6 / 13.6, B20 T396 E10 K85 I256 J64 20.9 / 18.5, B26 T165 E5 K121 I608 J64
// 36.2 / 37.4).
bool make_dw_tile(const void *Xs, const void *Ys, const void *Ind, void *dW, const egs_dims *d, int64_t ldx_b, int64_t ldx_t,
                  int act_dtype, int out_dtype, int ind_dtype, int dw_layout, DwTileJob &j, bool wide = false, bool shared = false)
{
    if (g_force_generic) return false;
    const int ES = elem_size(act_dtype);
    // (fp32, the bf16 instruction's 64 x 64 tiles / these, us, by slabs: 4096 (B64 T256 E32 K32 I128 J64) 21 / 20, 9450 (B16 T61 E14 K45 I960 J96)
    // 30 / 50, 16384 43 / 66 and 46 / 60; with 32 columns of a tile empty (I32 J96, 7676) 41 / 30)
    if (ES == 4 && d->I > 32 && d->J > 32 && dw_split32_slabs(d) >= 8192) return false;
    if (!shared && dw_strip_narrow(d, act_dtype)) return false;
    if (d->I % 8 || d->J % 8 || d->I < 8 || d->J < 8 || d->I > 2048 || d->J > 128) return false;
    const int64_t Me = (int64_t)d->B * d->K;
    if (Me == 0 || d->E == 0 || d->T == 0) return false;
    if (dw_few_picks(d, act_dtype)) return false;
    if (ES == 2 && d->I > 128 && d->J > 64 && Me >= 256) return false;      // the 256-row tiles of the direct-to-LDS kernel do better there
    const int it = ceil_div(d->I, 32), jt = ceil_div(d->J, wide ? 64 : 32);
    if ((int64_t)d->E * it * jt < (wide ? 64 : 128)) return false;
    if (!aligned_to(Xs, 16) || !aligned_to(Ys, 16) || !aligned_to(dW, 16) || (ldx_b * ES) % 16 || (ldx_t * ES) % 16) return false;
    const uint64_t x_span = ((uint64_t)(d->B - 1) * (uint64_t)ldx_b + (uint64_t)(d->T - 1) * (uint64_t)ldx_t + d->I) * ES;
    const uint64_t y_span = (uint64_t)Me * d->E * d->J * ES;
    if (x_span >= (1ull << 31) || y_span >= (1ull << 31)) return false;
    if ((int64_t)8 * ceil_div(d->E, 8) * it * jt > INT32_MAX / 2) return false;
    memset(&j, 0, sizeof(j));
    DwTileParams &q = j.q;
    q.Xs = (const char *)Xs; q.Ys = (const char *)Ys; q.Ind = Ind; q.dW = (char *)dW;
    q.B = d->B; q.T = d->T; q.E = d->E; q.K = d->K; q.I = d->I; q.J = d->J;
    q.ldx_b = ldx_b; q.ldx_t = ldx_t; q.ind_dtype = ind_dtype;
    q.i_tiles = it; q.j_tiles = jt;
    q.out_dtype = out_dtype; q.dw_layout = dw_layout;
    q.x_bytes = (uint32_t)x_span; q.y_bytes = (uint32_t)y_span;
    j.blocks = 8 * ceil_div(d->E, 8) * it * jt;
    j.act_dtype = act_dtype;
    j.wide = wide;
    return true;
}

// Which tile a one-pass weight gradient launched on its own should use.  32 x 64 tiles fetch whole 128-byte lines on
// the Ys side and send half the requests per pick; 32 x 32 tiles only win when they fill the device exactly once and the
// reduction is short (16-bit, the reference's default shape: 10.1 against 10.6 us; E48: 15.0 / 11.5, B160: 24.5 / 21.2,
// I256: 16.3 / 12.5 us).
// In fp32 a wide tile is twice the matrix instructions for the same four wavefronts, so only the tile count decides
// (default shape 19.5 / 30.1 us, B160: 41.7 / 67.3, E48: 36.2 / 30.5, I256: 36.6 / 31.0 us).
bool dw_tile_wide_alone(const egs_dims *d, int act_dtype)
{
    constexpr int64_t kCUs = 256;
    const int64_t narrow_tiles = (int64_t)d->E * ceil_div(d->I, 32) * ceil_div(d->J, 32);
    if (d->J <= 32) return false;
    return narrow_tiles > kCUs || (act_dtype != EGS_F32 && (int64_t)d->B * d->K >= 4096);
}

int launch_dw_tile_alone(DwTileJob &j, hipStream_t s)
{
    if (j.act_dtype == EGS_F32) {
        // four wavefronts either way; both sizes of staging tiles need more than the default LDS limit
        static LdsGrant told_narrow, told_wide;
        const size_t lds = dw_tile_lds(kThreads / 64, j.wide ? 64 : 32, 4);
        const int rc = j.wide
            ? allow_large_lds((const void *)dw_tile_wide_f32_kernel, told_wide, lds, "hipFuncSetAttribute(dw_tile_wide_f32_kernel)")
            : allow_large_lds((const void *)dw_tile_kernel<ElemF32>, told_narrow, lds, "hipFuncSetAttribute(dw_tile_kernel)");
        if (rc != EGS_OK) return rc;
        if (j.wide) hipLaunchKernelGGL(dw_tile_wide_f32_kernel, dim3(j.blocks), dim3(kThreads), lds, s, j.q);
        else hipLaunchKernelGGL(dw_tile_kernel<ElemF32>, dim3(j.blocks), dim3(kThreads), lds, s, j.q);
    } else if (j.wide) {
        static LdsGrant told_bf16, told_f16;
        const size_t lds = dw_tile_lds(kDwWideThreads / 64, 64);
        const int rc = j.act_dtype == EGS_BF16
            ? allow_large_lds((const void *)dw_tile_wide_kernel<ElemBF16>, told_bf16, lds, "hipFuncSetAttribute(dw_tile_wide_kernel)")
            : allow_large_lds((const void *)dw_tile_wide_kernel<ElemF16>, told_f16, lds, "hipFuncSetAttribute(dw_tile_wide_kernel)");
        if (rc != EGS_OK) return rc;
        if (j.act_dtype == EGS_BF16) hipLaunchKernelGGL(dw_tile_wide_kernel<ElemBF16>, dim3(j.blocks), dim3(kDwWideThreads), lds, s, j.q);
        else hipLaunchKernelGGL(dw_tile_wide_kernel<ElemF16>, dim3(j.blocks), dim3(kDwWideThreads), lds, s, j.q);
    } else {
        const size_t lds = dw_tile_lds(kThreads / 64);
        if (j.act_dtype == EGS_BF16) hipLaunchKernelGGL(dw_tile_kernel<ElemBF16>, dim3(j.blocks), dim3(kThreads), lds, s, j.q);
        else hipLaunchKernelGGL(dw_tile_kernel<ElemF16>, dim3(j.blocks), dim3(kThreads), lds, s, j.q);
    }
    EGS_CHECK_LAUNCH(j.act_dtype == EGS_F32 ? (j.wide ? "dw_tile_wide_f32_kernel" : "dw_tile_kernel") : (j.wide ? "dw_tile_wide_kernel" : "dw_tile_kernel"));
    j.done = true;
    return EGS_OK;
}

// ---- fp32 gather of small experts (W(e) in LDS, fp32 matrix instruction)
// Two 16-pick row tiles per wavefront and eight wavefronts per workgroup: two wavefronts per SIMD, so that one's waits
// (row transposition, LDS fragment reads) sit under the other's matrix instructions (default shape 18.4 -> 16.8 us against
// four row tiles and four wavefronts)
constexpr int kSmallF32Waves = 8;       // 16 / TQ with TQ = 2 below

template <bool W_NMAJOR, int KS>
int launch_gather_small_f32_ks(const SmallRowsParams &p, int blocks, hipStream_t s)
{
    constexpr int TQ = 2, threads = 64 * (16 / TQ);
    static_assert(threads == 64 * kSmallF32Waves, "wavefronts per workgroup");
    size_t lds = rows_small_f32_lds(16 * KS, p.N);
    const size_t csr_lds = p.csr_split ? csr_half_lds(p.T, kSmallF32Waves) : csr_count_lds(p.T, kSmallF32Waves);
    if (p.csr_blocks > 0 && csr_lds > lds) lds = csr_lds;
    switch (p.N / 16) {
    case 1: hipLaunchKernelGGL((rows_small_f32_kernel<W_NMAJOR, KS, 1, TQ>), dim3(blocks), dim3(threads), lds, s, p); break;
    case 2: hipLaunchKernelGGL((rows_small_f32_kernel<W_NMAJOR, KS, 2, TQ>), dim3(blocks), dim3(threads), lds, s, p); break;
    case 3: hipLaunchKernelGGL((rows_small_f32_kernel<W_NMAJOR, KS, 3, TQ>), dim3(blocks), dim3(threads), lds, s, p); break;
    default: hipLaunchKernelGGL((rows_small_f32_kernel<W_NMAJOR, KS, 4, TQ>), dim3(blocks), dim3(threads), lds, s, p); break;
    }
    EGS_CHECK_LAUNCH("rows_small_f32_kernel");
    return EGS_OK;
}

// `used` reports whether the shape and operands qualified
// whether the fp32 small-expert gather takes these sizes and operands
bool gather_small_f32_takes(const void *X, const void *W, const void *Y, const egs_dims *d, int64_t ldx_b, int64_t ldx_t)
{
    const int R = d->I, N = d->J;
    if (g_force_generic || !(R == 32 || R == 64 || R == 128) || N % 16 != 0 || N < 16 || N > 64 || d->T == 0) return false;
    if (!aligned_to(X, 16) || !aligned_to(W, 16) || !aligned_to(Y, 16) || (ldx_b * 4) % 16 || (ldx_t * 4) % 16) return false;
    const int64_t Me = (int64_t)d->B * d->K;
    if (Me == 0 || d->E == 0) return false;
    const uint64_t x_span = ((uint64_t)(d->B - 1) * (uint64_t)ldx_b + (uint64_t)(d->T - 1) * (uint64_t)ldx_t + R) * 4;
    if (x_span > kSpan32 || (uint64_t)d->E * R * N * 4 > kSpan32 || (uint64_t)Me * d->E * N * 4 > kSpan32) return false;
    const int tiles_per_e = (int)((Me + 255) / 256);
    return (int64_t)8 * (ceil_div(d->E, 8) + 1) * (tiles_per_e + 8) <= INT32_MAX / 2;
}

// `build` (optional): the routing table of a later scatter over the same Ind is built by B more workgroups of the launch
int gather_small_f32(const void *X, const void *W, const void *Ind, void *Y, const egs_dims *d, int64_t ldx_b, int64_t ldx_t,
                     int ind_dtype, int w_layout, hipStream_t s, bool &used, const RoutingTable *build = nullptr)
{
    used = false;
    if (!gather_small_f32_takes(X, W, Y, d, ldx_b, ldx_t)) return EGS_OK;
    const int R = d->I, N = d->J;
    const int64_t Me = (int64_t)d->B * d->K;
    SmallRowsParams p;
    memset(&p, 0, sizeof(p));
    p.A = (const char *)X; p.W = (const char *)W; p.Ind = Ind; p.C = (char *)Y;
    p.B = d->B; p.T = d->T; p.E = d->E; p.K = d->K; p.N = N;
    p.lda_b = ldx_b; p.lda_t = ldx_t; p.ind_dtype = ind_dtype;
    p.tiles_per_e = (int)((Me + 255) / 256);
    if ((int64_t)8 * (ceil_div(d->E, 8) + 1) * (p.tiles_per_e + 8) > INT32_MAX / 2) return EGS_OK;
    p.rows_share_xcd = rows_xcd_map(d, R, N, 4, p.tiles_per_e);
    if (build != nullptr) {
        p.csr_blocks = d->B; p.seg_off = build->seg; p.perm = build->perm;
        if (table_split_pays(d, kSmallF32Waves, rows_xcd_blocks(p.rows_share_xcd, p.tiles_per_e, p.E), 512)) { p.csr_blocks = 2 * d->B; p.csr_split = 1; }
    }
    const int blocks = rows_xcd_blocks(p.rows_share_xcd, p.tiles_per_e, p.E) + p.csr_blocks;
    used = true;
    const bool nmajor = (w_layout == EGS_W_EIJ);        // [E,I,J] = [E,R,N]
    switch (R) {
    case 32: return nmajor ? launch_gather_small_f32_ks<true, 2>(p, blocks, s) : launch_gather_small_f32_ks<false, 2>(p, blocks, s);
    case 64: return nmajor ? launch_gather_small_f32_ks<true, 4>(p, blocks, s) : launch_gather_small_f32_ks<false, 4>(p, blocks, s);
    default: return nmajor ? launch_gather_small_f32_ks<true, 8>(p, blocks, s) : launch_gather_small_f32_ks<false, 8>(p, blocks, s);
    }
}

// `dwt` (one-pass weight gradient) shares the launch of a gather only; `dw` (first pass of the split form) any rows job
int launch_rows_small_job(SmallRowsJob &j, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s)
{
    return j.act_dtype == EGS_BF16 ? launch_rows_small_bf16(j, dw, dwt, s) : launch_rows_small_f16(j, dw, dwt, s);
}

int launch_dw_small_alone(SmallDwJob &j, hipStream_t s)
{
    if (j.act_dtype == EGS_BF16) hipLaunchKernelGGL(dw_small_kernel<ElemBF16>, dim3(j.blocks), dim3(kThreads), 0, s, j.q);
    else hipLaunchKernelGGL(dw_small_kernel<ElemF16>, dim3(j.blocks), dim3(kThreads), 0, s, j.q);
    EGS_CHECK_LAUNCH("dw_small_kernel");
    j.done = true;
    return EGS_OK;
}

int launch_dw_reduce4(const SmallDwJob &j, hipStream_t s)
{
    if (j.q.S <= 1) return EGS_OK;
    hipLaunchKernelGGL(dw_reduce4_kernel, dim3(grid_1d(j.w_elems / 4, 2048)), dim3(kThreads), 0, s,
                       (const float *)j.q.part, j.q.dW, j.q.S, j.w_elems / 4, j.q.out_dtype);
    EGS_CHECK_LAUNCH("dw_reduce4_kernel");
    return EGS_OK;
}

// sums over product rows; the second pass of the weight gradient `dw`, where it waits for one, shares the launch if it can
int segment_sum_with(const void *rows, bool rows_f32, const int32_t *seg_off, const int32_t *perm, int32_t *long_tab, float *long_part,
                     void *Out, const egs_dims *d, int act_dtype, SmallDwJob *dw, hipStream_t s)
{
    const bool waits = dw != nullptr && dw->done && dw->q.S > 1;
    DwSecondPass second = {};
    if (waits) second = {(const float *)dw->q.part, dw->q.dW, dw->q.S, dw->q.out_dtype, dw->w_elems, false};
    const int rc = launch_segment_sum(rows, rows_f32, seg_off, perm, long_tab, long_part, Out, d, act_dtype, waits ? &second : nullptr, s);
    if (second.done) dw->q.S = 1;
    return rc;
}

// ------------------------------------------------------------------------------ fused small-expert scatter
// Does the one-kernel scatter of small experts (product rows stay in LDS, no workspace) take this problem, and in how
// many passes over groups of experts?  experts_per_pass == E: one pass.
struct FusedPlan { bool ok; int experts_per_pass; size_t lds; };

FusedPlan scatter_fused_plan(const void *Y, const void *W, const void *Out, const egs_dims *d, int act_dtype)
{
    const FusedPlan no = {false, 0, 0};
    const int R = d->J, N = d->I;
    const int64_t NP = (int64_t)d->E * d->K;
    if (g_force_generic || !(R == 32 || R == 64 || (R == 128 && act_dtype != EGS_F32))) return no;
    const int ES = elem_size(act_dtype);
    if (N < kFusedCols || N % kFusedCols != 0 || NP < 1 || NP > 4096 || d->T < 1 || d->B < 1) return no;
    if (!aligned_to(Y, 16) || !aligned_to(W, 16) || !aligned_to(Out, 16)) return no;
    if ((uint64_t)d->B * NP * R * ES > kSpan32 || (uint64_t)d->E * R * N * ES > kSpan32) return no;
    const int slices = N / kFusedCols;
    const int64_t blocks = (int64_t)8 * ceil_div(d->B, 8) * slices;
    if (blocks > INT32_MAX / 2 || (int64_t)d->B * slices < 8) return no;        // fewer workgroups are not worth it
    const size_t budget = 156 * 1024;
    if (NP <= 1024 && scatter_fused_lds(d->T, (int)NP) <= budget) return {true, d->E, scatter_fused_lds(d->T, (int)NP)};
    // groups of experts: as few passes as the rows' share of LDS allows, of equal size
    if (d->T > (kFusedThreads >> 3) * kFusedMultiTokens) return no;
    const size_t fixed = scatter_fused_lds(d->T, (int)NP, 0);
    if (fixed >= budget) return no;
    const int64_t fit = (int64_t)((budget - fixed) / ((size_t)d->K * kFusedCols * 4));     // experts whose rows fit
    if (fit < 1) return no;
    const int passes = ceil_div(d->E, (int)(fit < d->E ? fit : d->E));
    if (passes < 2 || passes > kFusedMaxPasses) return no;
    const int per_pass = ceil_div(d->E, passes);
    return {true, per_pass, scatter_fused_lds(d->T, (int)NP, per_pass * d->K)};
}

// whether the one-kernel scatter planned as `fp` can take its routing table from memory: what the kernel's registers stage
// (one pass: 1024 picks, T + 1 <= 2048 offsets; in passes: 2048 picks, T <= 512, 16-bit types - in fp32 the pass kernel
// measured slower with the table than sorting for itself: 131 against 128 us for gather + scatter + gather backward at
// B64 T256 E60 K32 I128 J64)
bool fused_reads_table(const FusedPlan &fp, const egs_dims *d, int act_dtype)
{
    if (!fp.ok) return false;
    const int64_t NP = (int64_t)d->E * d->K;
    if (fp.experts_per_pass == d->E) return NP <= 1024 && d->T + 1 <= 2048;
    return act_dtype != EGS_F32 && NP <= 2048 && d->T <= 512;
}

// More slices than CUs: runs of slices with one sort.  A CU does its workgroups' slices one after the other, however many fit
// its LDS, and a sort takes 0.6 of a slice's time; the run with the shortest rounds was the fastest at 12 of 12 sizes (B64
// T256 E32 K32 I768 J64: runs of 6, 61 -> 47 us; B128 T64 E8 K16 I1024 J64: 16, 73 -> 37).
int fused_run(const FusedPlan &fp, const egs_dims *d)
{
    const int slices = d->I / kFusedCols;
    int run = 1;
    if (fp.experts_per_pass == d->E) {
        double least = 0;
        for (int r = 1; r <= slices; ++r) {
            const double cost = (double)(((int64_t)d->B * ceil_div(slices, r) + 255) / 256) * (r + 0.6);
            if (r == 1 || cost < least) { least = cost; run = r; }
        }
    }
    return run;
}

// GEMM-scatter of small experts in one kernel; the caller has checked scatter_fused_plan().  Both scatter modes
// take it: it is bitwise reproducible and needs no workspace.
int scatter_fused(const void *Y, const void *W, const void *Ind, void *Out, const egs_dims *d, int act_dtype, int ind_dtype,
                  int w_layout, SmallDwJob *dw, DwTileJob *dwt, hipStream_t s, const RoutingTable *use = nullptr)
{
    const int R = d->J, N = d->I;
    const int64_t NP = (int64_t)d->E * d->K;
    const FusedPlan fp = scatter_fused_plan(Y, W, Out, d, act_dtype);
    if (!fp.ok) return EGS_ERR_UNSUPPORTED;
    const size_t lds = fp.lds;
    const int slices = N / kFusedCols;
    const int run = fused_run(fp, d);
    const int64_t blocks = (int64_t)8 * ceil_div(d->B, 8) * ceil_div(slices, run);
    ScatterFusedParams p;
    memset(&p, 0, sizeof(p));
    p.A = (const char *)Y; p.W = (const char *)W; p.Ind = Ind; p.out = (char *)Out;
    p.B = d->B; p.T = d->T; p.E = d->E; p.K = d->K; p.N = N;
    p.ind_dtype = ind_dtype;
    p.slices = slices;
    p.run = run;
    p.experts_per_pass = fp.experts_per_pass;
    if (use != nullptr && fused_reads_table(fp, d, act_dtype)) { p.tab_seg = use->seg; p.tab_perm = use->perm; }
    p.perm_at = (int32_t)((int64_t)fp.experts_per_pass * d->K * kFusedCols * 4);
    p.cnt_at = p.perm_at + (int32_t)(NP * 4);
    p.zero_at = (int32_t)scatter_fused_zero_at(d->T, (int)NP, fp.experts_per_pass * d->K);
    // where the rows come from a small-expert gather (256 picks of one expert per workgroup, row tiles mapped to XCDs), the
    // batch elements of one of its row tiles - 256 / K of them - were written on one XCD
    p.xcd_batch = (d->K == 32 || d->K == 64 || d->K == 128 || d->K == 256) ? 256 / d->K : 2;
    const bool nmajor = (w_layout == EGS_W_EJI);        // [E,J,I] = [E,R,N]
    return act_dtype == EGS_F32 ? launch_fused_f32(p, nmajor, R, lds, (int)blocks, nullptr, nullptr, s)
         : act_dtype == EGS_F16 ? launch_fused_f16(p, nmajor, R, lds, (int)blocks, dw, dwt, s) : launch_fused_bf16(p, nmajor, R, lds, (int)blocks, dw, dwt, s);
}

// whether the weight gradient's 32 x 32 tiles share the launch of a gather backward's one-kernel scatter: it runs in one pass and they come
// after it in one round of workgroups (I = 256: 42.9 us sharing, 37 us as two launches with 32 x 64 tiles)
bool gather_backward_shares(const FusedPlan &fp, const egs_dims *d, int act_dtype)
{
    return act_dtype != EGS_F32 && fp.ok && fp.experts_per_pass == d->E && fused_run(fp, d) == 1 &&
           (int64_t)d->E * ceil_div(d->I, 32) * ceil_div(d->J, 32) <= 256;
}

// Which weight-gradient kernel takes these operands, and the workspace it needs.  egs_workspace_bytes asks with
// stand-in operands (dense, 16-byte aligned); the entry points ask with the real ones, so what is planned and what
// runs agree by construction.
enum DwPath { DW_TILE, DW_SMALL, DW_BIG, DW_GENERAL };
struct DwChoice { DwPath path; size_t bytes; };

DwChoice dw_choose(const void *Xs, const void *Ys, void *dW, const egs_dims *d, int64_t ldx_b, int64_t ldx_t, int act_dtype,
                   const DwPlan &pl)
{
    DwTileJob tj;
    if (make_dw_tile(Xs, Ys, nullptr, dW, d, ldx_b, ldx_t, act_dtype, act_dtype, 0, 0, tj)) return {DW_TILE, 0};
    SmallDwJob sj;
    if (make_dw_small(Xs, Ys, nullptr, dW, nullptr, d, ldx_b, ldx_t, act_dtype, act_dtype, 0, 0, pl, sj)) return {DW_SMALL, pl.bytes_small};
    if (dw_big_takes(pl, Xs, Ys, dW, d, ldx_b, ldx_t, act_dtype)) return {DW_BIG, pl.bytes_big};
    return {DW_GENERAL, pl.bytes_general};
}

void *const kStandInPtr = (void *)(uintptr_t)4096;      // aligned, never dereferenced

size_t dw_bytes_planned(const egs_dims *d, int act_dtype)
{
    return dw_choose(kStandInPtr, kStandInPtr, kStandInPtr, d, (int64_t)d->T * d->I, d->I, act_dtype, plan_dw(d, act_dtype)).bytes;
}

// Is the one-kernel scatter the faster one?  A model of its time and of product rows with their sums, fitted to 2000 sizes alone on the device
// (within 14 and 9 % of most): the turns that its workgroups take at the CUs, each a sort of the picks and then, for every slice, units of 32
// picks of one expert, empty places included, and sums of all tokens; against the rows written and read, the tiles they are made in,
// the weights, the output, and the indices that every group of 32 tokens looks through.  What it loses are many experts of few picks (units
// mostly empty: bf16 B1 T2127 E83 K5 I640 J128 34 us, 13 as rows; f32 B91 T338 E64 K5 I192 J64 82 / 30), few batch elements with many tokens
// (f32 B9 T454 E28 K5 I96 J64 16.3 / 10.3) and slices by the hundred of few picks (f16 B21 T416 E125 K5 I896 J128 94 / 32; not of full units: f16 B80
// T269 E43 K23 I928 J64 85 / 126).  Of 2481 other calls that either takes 507 go by rows, 4 of them more than 3 % slower for it (1.11), and all
// take 0.93 of the one kernel's time in 16 bits and 0.83 in fp32 (0.89 and 0.77 are the least: the margin is on its side, for it needs no workspace).
// A weight gradient that shares a launch with either counts 3 or 4 us for it.  Zipf-distributed picks, whose hot tokens one group of threads adds up
// here and many there, make it lose more (its time 1.0 to 1.5 of the rows' on average in one pass); a call can't know.
// In passes (more than 1024 picks) it loses to the rows by 1.3 on average (1.85 in fp32) and by 3 with Zipf-distributed picks; the
// model keeps 184 of 379 scatters there (1.18 of the rows' time; bf16 B78 T43 E49 K25 I96 J32 17.8 / 28.7) and one whose table comes with the
// gather's launch, and the others take 0.55 of the time they took.
// Up to kRowsInsteadBytes of workspace, a little more than 380000 random sizes of up to 128 batch elements ask for: a call of thousands of them would
// want a hundred times its operands and more than a card has (bf16 B1852 T22 E252 K7 I1536 J32: 20 GB of rows for 0.36, B93597 T82 E250 K2 I1952 J32 378 GB).
constexpr size_t kRowsInsteadBytes = 1ull << 30;
bool fused_model_pays(const FusedPlan &fp, const egs_dims *d, int act_dtype, double extra_us, double margin = 1.15)
{
    if (plan_scatter(d, EGS_SCATTER_DETERMINISTIC, act_dtype, SCATTER_ROWS).bytes > kRowsInsteadBytes) return true;
    const bool f32 = act_dtype == EGS_F32, passes = fp.experts_per_pass != d->E;
    const int run_slices = passes ? 1 : fused_run(fp, d);
    if (!passes && scatter_fused_holds(d->E, d->K, d->J * elem_size(act_dtype), run_slices)) return true;     // 0.70 (fp32: 0.83) of the rows' time
    const double T = d->T / 256.0, N = (double)d->E * d->K / 1024.0, run = run_slices, steps = d->J / 32.0;
    const double units = (double)d->E * ceil_div(d->K, 32) / 8.0;       // of a wavefront
    const int64_t groups = (int64_t)d->B * ceil_div(d->I / kFusedCols, run_slices), at_once = fp.lds <= 80 * 1024 ? 512 : 256;
    const double turns = groups > at_once ? (double)((groups + at_once - 1) / at_once) * (at_once / 256) : groups > 256 ? groups / 256.0 : 1.0;
    const double pass_turns = std::max(1.0, groups / 256.0), resort = groups > 256 ? N : 0.0;       // in passes the picks are sorted again
    const double fused_us =
        passes ? f32 ? 3.5 + 12.4 * resort + pass_turns * (4.7 * N + units * (0.45 + 1.26 * steps) + 2.6 * T + 1.2)
                     : 1.6 + 7.7 * resort + pass_turns * (5.2 * N + units * (0.21 + 0.32 * steps) + 2.8 * T + 3.6)
        : f32  ? 3.4 + turns * (2.23 * N + run * (1.84 + units * (0.15 + 1.3 * steps) + 1.26 * T))
               : 4.0 + turns * (0.16 * T + 2.25 * N + run * (1.1 + units * (0.195 + 0.31 * steps) + 0.88 * T));
    const double es = elem_size(act_dtype), picks = (double)d->B * d->E * d->K, out = (double)d->B * d->T;
    const double rows_mb = picks * d->I * 4e-6, out_mb = out * d->I * es * 1e-6, w_mb = (double)d->E * d->I * d->J * es * 1e-6;
    const double tiles = (double)(((int64_t)d->B * d->K + 63) / 64) * d->E * ceil_div(d->I, 96) / 768.0, scans = out * d->E * d->K * 1e-6 / 32.0;
    const double rows_us = f32 ? 9.6 + 0.236 * rows_mb + 13.3 * picks * d->I * d->J * 2e-9 + 0.096 * out_mb + 0.14 * w_mb + 2.63 * tiles + 0.006 * d->E +
                                     1.43e-4 * out + 0.95 * scans
                               : 9.4 + 0.364 * rows_mb + 0.30 * out_mb + 0.183 * w_mb + 1.23 * tiles + 0.005 * d->E + 3.0e-5 * out + 0.64 * scans;
    return fused_us + extra_us < margin * rows_us;
}

// Layout of a caller-owned routing table, for the sizes whose one-kernel scatter can read one (fused_reads_table: one pass of any type, or 16-bit types in
// passes); `ok` false: a table would not be used; `worth` false: none is asked for, and one that is given is
// built, and read where the one-kernel scatter runs.
struct TableLayout { bool ok, worth; size_t perm_at, bytes; };
TableLayout routing_table_layout(const egs_dims *d, int act_dtype)
{
    TableLayout l = {false, false, 0, 0};
    if (!(act_dtype == EGS_F16 || act_dtype == EGS_BF16 || act_dtype == EGS_F32)) return l;
    const FusedPlan fp = scatter_fused_plan(kStandInPtr, kStandInPtr, kStandInPtr, d, act_dtype);
    if (!fused_reads_table(fp, d, act_dtype)) return l;
    // the table pays only when its build rides in the gather forward's launch (as a launch of its own it costs more than
    // the two scatters save): the small-expert gather of the type must take these sizes too
    if (act_dtype == EGS_F32) {
        if (!gather_small_f32_takes(kStandInPtr, kStandInPtr, kStandInPtr, d, (int64_t)d->T * d->I, d->I) ||
            csr_count_lds(d->T, kSmallF32Waves) > 64 * 1024)
            return l;
    } else {
        SmallRowsJob gj;
        if (!make_gather_small(kStandInPtr, kStandInPtr, kStandInPtr, kStandInPtr, d, (int64_t)d->T * d->I, d->I, act_dtype,
                               act_dtype, EGS_IND_I32, EGS_W_EIJ, gj))
            return l;
    }
    l.ok = true;
    // The table spares a scatter its sort, not the units of a few picks each: as product rows fp32 B69 T57 E111 K6 I32 J64 takes 17 us (42.9 in one
    // kernel), B4 T39 E65 K9 I64 J64 10 (27.6).  (16 bits: 0.83 of the rows' step.)
    l.worth = act_dtype != EGS_F32 || fused_model_pays(fp, d, act_dtype, -2.0 * d->E * d->K / 1024.0, 1.7);
    l.perm_at = align_up((size_t)d->B * (d->T + 1) * 4, 256);
    l.bytes = l.perm_at + align_up((size_t)d->B * d->E * d->K * 4, 256);
    return l;
}

// ------------------------------------------------------------------------------ which scatter
// What a scatter is launched with: nothing, a weight gradient whose launch the product rows would share (tiled_pair_kernel), or one that
// shares the one-kernel scatter's.
enum ScatterWith { SCATTER_ALONE, SCATTER_WITH_TILED_DW, SCATTER_WITH_DW_TILES };

// a gather's backward, by its sizes alone (what is planned and what runs then agree whatever the operands)
ScatterWith gather_backward_with(const egs_dims *d, int act_dtype)
{
    const FusedPlan fp = scatter_fused_plan(kStandInPtr, kStandInPtr, kStandInPtr, d, act_dtype);
    DwTileJob j;
    if (gather_backward_shares(fp, d, act_dtype) && make_dw_tile(kStandInPtr, kStandInPtr, nullptr, kStandInPtr, d, (int64_t)d->T * d->I, d->I, act_dtype,
                                                                 act_dtype, 0, 0, j, false, true))
        return SCATTER_WITH_DW_TILES;
    const DwChoice dw = dw_choose(kStandInPtr, kStandInPtr, kStandInPtr, d, (int64_t)d->T * d->I, d->I, act_dtype, plan_dw(d, act_dtype));
    return dw.path == DW_GENERAL ? SCATTER_WITH_TILED_DW : SCATTER_ALONE;
}

bool scatter_fused_pays(const FusedPlan &fp, const egs_dims *d, int act_dtype, bool gather_backward)
{
    if (routing_table_layout(d, act_dtype).worth) return true;
    if (fp.experts_per_pass == d->E && small_shape_ok(act_dtype, d->J, d->I)) return true;      // the rows of small experts and their sums: 1.34 times its time
    const ScatterWith with = gather_backward ? gather_backward_with(d, act_dtype) : SCATTER_ALONE;
    return fused_model_pays(fp, d, act_dtype, with == SCATTER_WITH_TILED_DW ? 3.0 : with == SCATTER_WITH_DW_TILES ? -4.0 : 0.0);
}

// The one-kernel scatters come first where they apply and pay (they need no workspace).  Beyond them
// the product rows go through the workspace, unless the caller asks for the compact mode: the one-kernel scatter in
// passes keeps them in LDS and sorts each pass's picks there too, for any number of picks per batch element and with no
// workspace at all - at B16 T1024 E64 K128 I512 J128 in 136 us under Zipf routing and 133 us under even routing, where
// the product rows through 270 MB of workspace take 120 and 105 us.
// `given`: bytes of the caller's workspace; one that does not hold the rows is enough for the one-kernel scatter.  (In the atomic mode its
// fp32 sums are more precise than rows in the element type, so there it is not a matter of time.)
ScatterPath scatter_choose(const void *Y, const void *W, const void *Out, const egs_dims *d, int act_dtype, int mode, bool gather_backward = false,
                           size_t given = SIZE_MAX)
{
    const FusedPlan fp = scatter_fused_plan(Y, W, Out, d, act_dtype);
    if (fp.ok && (mode != EGS_SCATTER_DETERMINISTIC || scatter_fused_pays(fp, d, act_dtype, gather_backward) ||
                  plan_scatter(d, mode, act_dtype, SCATTER_ROWS).bytes > given))
        return SCATTER_FUSED;
    if (mode == EGS_SCATTER_COMPACT && scatter_pass_plan(Y, W, Out, d, act_dtype).ok) return SCATTER_PASS;
    return SCATTER_ROWS;
}
size_t scatter_bytes_planned(const egs_dims *d, int mode, int act_dtype, bool gather_backward)
{
    return plan_scatter(d, mode, act_dtype, scatter_choose(kStandInPtr, kStandInPtr, kStandInPtr, d, act_dtype, mode, gather_backward)).bytes;
}

// checks a table argument of an entry point; fills `t` when the table is to be used
int check_table_arg(void *table, size_t table_bytes, const egs_dims *d, int act_dtype, RoutingTable &t, bool &have)
{
    have = false;
    if (table == nullptr) return EGS_OK;
    const TableLayout l = routing_table_layout(d, act_dtype);
    if (!l.ok) return EGS_ERR_UNSUPPORTED;
    if (!aligned_to(table, 256)) return EGS_ERR_ALIGNMENT;
    if (table_bytes < l.bytes) return EGS_ERR_WORKSPACE;
    t.seg = (int32_t *)table;
    t.perm = (int32_t *)((char *)table + l.perm_at);
    have = true;
    return EGS_OK;
}

// ------------------------------------------------------------------------------ implementations
int gather_gemm_impl(const void *X, const void *W, const void *Ind, void *Y, const float *w_scale,
                     const egs_dims *d, int64_t ldx_b, int64_t ldx_t, int act_dtype, int w_dtype, int ind_dtype,
                     int w_layout, hipStream_t s, const RoutingTable *build = nullptr, int act = ACT_NONE, const void *bias = nullptr, TiledDwJob *tdw = nullptr)
{
    const int ES = elem_size(act_dtype), WES = elem_size(w_dtype);
    if (w_scale == nullptr) {
        SmallRowsJob j;
        if (make_gather_small(X, W, Ind, Y, d, ldx_b, ldx_t, act_dtype, w_dtype, ind_dtype, w_layout, j, build, act)) {
            const int rc = launch_rows_small_job(j, nullptr, nullptr, s);
            return rc == EGS_OK && bias != nullptr ? bias_rows(Y, bias, d, act_dtype, s) : rc;
        }
    }
    if (w_scale == nullptr && act_dtype == EGS_F32 && w_dtype == EGS_F32) {
        bool used = false;
        const int rc = gather_small_f32(X, W, Ind, Y, d, ldx_b, ldx_t, ind_dtype, w_layout, s, used, build);
        if (used) return rc == EGS_OK && bias != nullptr ? bias_rows(Y, bias, d, act_dtype, s) : rc;
    }
    if (build != nullptr) {             // no launch for the table to ride in: a launch of its own
        const int rc = launch_routing_table(Ind, ind_dtype, d, build->seg, build->perm, nullptr, nullptr, nullptr, s);
        if (rc != EGS_OK) return rc;
    }
    RowsGemmParams p;
    memset(&p, 0, sizeof(p));
    p.A = (const char *)X; p.W = (const char *)W; p.Ind = Ind; p.C = (char *)Y; p.w_scale = w_scale;
    p.B = d->B; p.T = d->T; p.E = d->E; p.K = d->K;
    p.act = act; p.bias = bias;
    p.R = d->I; p.N = d->J;
    p.lda_b = ldx_b; p.lda_t = ldx_t;
    p.ind_dtype = ind_dtype;
    const bool w_trans = (w_layout == EGS_W_EIJ);       // [E,I,J]: the reduction index selects the row
    p.a_vec = aligned_to(X, 16) && (ldx_b * ES) % 16 == 0 && (ldx_t * ES) % 16 == 0;
    const int64_t w_row = w_trans ? d->J : d->I;
    p.w_vec = WES == 1 ? (aligned_to(W, 8) && w_row % 8 == 0) : (aligned_to(W, 16) && (w_row * WES) % 16 == 0);
    {
        const uint64_t span = d->B > 0 && d->T > 0
            ? ((uint64_t)(d->B - 1) * (uint64_t)ldx_b + (uint64_t)(d->T - 1) * (uint64_t)ldx_t + (uint64_t)d->I) * ES : 0;
        p.a_bytes = span < (1ull << 31) ? (uint32_t)span : 0;
    }
    const int rc = rows_gemm_gather(p, act_dtype, w_dtype == EGS_FP8_E4M3, w_trans, s, tdw);
    return rc == EGS_OK && bias != nullptr && !p.bias_done ? bias_rows(Y, bias, d, act_dtype, s) : rc;
}

int gemm_scatter_rows(const void *Y, const void *W, const void *Ind, void *Out, void *workspace,
                      const egs_dims *d, int act_dtype, int ind_dtype, int w_layout, int mode, SmallDwJob *dw,
                      DwTileJob *dwt, hipStream_t s, const RoutingTable *use, const void *bias, bool &bias_done, TiledDwJob *tdw, ScatterPath path);

// The picks that sums without a routing table look through: 4096 a batch element, or twice that for few tokens of short rows, where the launch for the
// table takes as long as the sums.  us: bf16 B1 T2941 E47 K157 I32 J160 25.8 -> 13.9, B2 T1832 E59 K79 I32 J20 21.7 -> 12.8, f32 B2 T440 E27 K162 I32 J40
// 20 -> 13; 68 random scatters take 0.76 of their time, 16 under Zipf routing 0.92 (one of them is 4 % slower); 160 of 4097 to 4224 picks 0.70, under Zipf
// routing 0.87 (11 slower, f16 B34 T252 E57 K72 I68 J37 44 -> 61).  Longer rows take 0.78 to 0.83, under Zipf
// routing 1.2 to 1.4: a hot token's rows are many workgroups' with a table, and one's here.
bool token_sums_take(const egs_dims *d)
{
    const int64_t N = (int64_t)d->E * d->K;
    const bool few = N > kTokenSumPicks && N <= kTokenSumPicksFew && d->I <= 128 && (int64_t)d->B * d->T <= 16384;
    return N >= 1 && (N <= kTokenSumPicks || few);
}

// Sums that find their picks themselves, or a launch for the routing table and sums that use it?  What the launch takes (us), more for long
// sequences, and what its sums lose on tokens of many picks and on the output, against what the others do once more for every group of tokens:
// look through all indices.  Of 361 sizes on the device alone two are more than 3 % slower by this, and the scatters take 0.68 of what they
// took with a table in all of them (0.678 is the least): us, table / without, bf16 B2 T2696 E5 K6 I64 J32 45.9 / 9.4, B3 T3776 E78 K8 I32 J64 23.5 / 11.2,
// B85 T2791 E85 K36 I128 J128 93 / 111, f16 B103 T2302 E40 K28 I32 J21 37.5 / 50.8.
bool token_sums_pay(const egs_dims *d)
{
    const double tokens = (double)d->B * d->T, N = (double)d->E * d->K;
    return 1.33e-4 * tokens + 1.25e-9 * tokens * N < 3.0 + 2.3e-3 * d->T + 0.6 * N / d->T + 4e-7 * tokens * d->I;
}
// The product rows of small experts: their launch can take the table along (`rides`), one workgroup per batch element, which ranks the
// picks longer than the products take where there are many; the sums with it are the faster ones for few picks, and with hot tokens.
// us, riding / without: bf16 B1 T476 E47 K81 I56 J32 20.9 / 12.4, B9 T130 E56 K52 I32 J32 22 / 16.5; B5 T39 E102 K30 I96 J64 (78 picks a token) 23 /
// 32.5, B6 T70 E4 K9 I32 J64 7.8 / 10.6.  Of 489 sizes 78 go this way and 3 are more than 3 % slower.
bool small_token_sums_pay(const egs_dims *d, bool rides)
{
    const int64_t N = (int64_t)d->E * d->K;
    if (!token_sums_take(d) || d->T < 1) return false;
    if (N > kTokenSumPicks) return true;
    return rides ? d->B <= 32 && N >= 1500 && N <= 32 * (int64_t)d->T : token_sums_pay(d);
}

// `dw` (optional): a weight gradient of the same call whose first pass may share the product
// launch and whose second pass may share the reduction launch; `tdw` (optional): one in the tiled kernels, which a tiled product takes along
int gemm_scatter_impl(const void *Y, const void *W, const void *Ind, void *Out, void *workspace,
                      const egs_dims *d, int act_dtype, int ind_dtype, int w_layout, int mode, ScatterPath path, SmallDwJob *dw,
                      DwTileJob *dwt, hipStream_t s, const RoutingTable *use = nullptr, const void *bias = nullptr, TiledDwJob *tdw = nullptr)
{
    bool bias_done = false;
    const int rc = gemm_scatter_rows(Y, W, Ind, Out, workspace, d, act_dtype, ind_dtype, w_layout, mode, dw, dwt, s, use, bias, bias_done, tdw, path);
    return rc == EGS_OK && bias != nullptr && !bias_done ? bias_scatter(Out, bias, Ind, d, act_dtype, ind_dtype, s) : rc;
}

int gemm_scatter_rows(const void *Y, const void *W, const void *Ind, void *Out, void *workspace,
                      const egs_dims *d, int act_dtype, int ind_dtype, int w_layout, int mode, SmallDwJob *dw,
                      DwTileJob *dwt, hipStream_t s, const RoutingTable *use, const void *bias, bool &bias_done, TiledDwJob *tdw, ScatterPath path)
{
    bias_done = false;
    const int ES = elem_size(act_dtype);
    const size_t out_elems = (size_t)d->B * d->T * d->I;
    if (out_elems == 0) return EGS_OK;
    const bool fused = path == SCATTER_FUSED;
    const ScatterPlan pl = plan_scatter(d, mode, act_dtype, path);
    char *ws = (char *)workspace;
    const int N = d->E * d->K;

    RowsGemmParams p;
    memset(&p, 0, sizeof(p));
    p.A = (const char *)Y; p.W = (const char *)W; p.Ind = Ind;
    p.B = d->B; p.T = d->T; p.E = d->E; p.K = d->K;
    p.R = d->J; p.N = d->I;
    p.ind_dtype = ind_dtype;
    const bool w_trans = (w_layout == EGS_W_EJI);       // [E,J,I]: the reduction index j selects the row
    p.a_vec = aligned_to(Y, 16) && ((int64_t)d->J * ES) % 16 == 0;
    const int64_t w_row = w_trans ? d->I : d->J;
    p.w_vec = aligned_to(W, 16) && (w_row * ES) % 16 == 0;
    {
        const uint64_t span = (uint64_t)d->B * d->E * d->K * d->J * ES;
        p.a_bytes = span < (1ull << 31) ? (uint32_t)span : 0;
    }

    if (mode == EGS_SCATTER_ATOMIC && act_dtype == EGS_F32) {
        float *acc32 = (float *)Out;
        hipLaunchKernelGGL(fill_zero_f32_kernel, dim3(grid_1d(out_elems / 4 + 1)), dim3(kThreads), 0, s, acc32, out_elems,
                           (int)aligned_to(acc32, 16));
        EGS_CHECK_LAUNCH("fill_zero_f32_kernel");
        p.C = (char *)acc32;
        return rows_gemm_scatter(p, act_dtype, w_trans, EPI_ATOMIC_F32, s);
    }

    if (fused) return scatter_fused(Y, W, Ind, Out, d, act_dtype, ind_dtype, w_layout, dw, dwt, s, use);   // small experts: one kernel
    // compact mode, thousands of picks per batch element: one kernel in passes, nothing in the workspace
    if (path == SCATTER_PASS) return scatter_pass(Y, W, Ind, Out, d, act_dtype, ind_dtype, w_layout, s);

    // routing table (picks in token order) + product rows in pick order, then one fixed-order
    // gather-and-sum per token that writes every output row exactly once
    int32_t *seg_off = (int32_t *)(ws + pl.seg_off_at);
    int32_t *perm = (int32_t *)(ws + pl.perm_at);
    int32_t *rank_tmp = (int32_t *)(ws + pl.rank_at);
    int32_t *cnt = d->T > kCsrLdsTokens ? (int32_t *)(ws + pl.cnt_at) : nullptr;
    int32_t *long_tab = (int32_t *)(ws + pl.long_tab_at);
    float *long_part = (float *)(ws + pl.long_part_at);
    void *rows = ws + pl.rows_at;
    bool rows_f32 = (mode != EGS_SCATTER_ATOMIC);
    // small experts: the sort rides along with the product when its histograms are small
    const bool can_ride = csr_count_lds(d->T, 4) <= 16 * 1024 && N <= 4096 && N > 0;
    const bool token_sums = !(dw != nullptr && dw->q.S > 1) && small_token_sums_pay(d, can_ride), ride = can_ride && !token_sums;
    SmallRowsJob j;
    int rc;
    if (N > 0 && make_scatter_rows_small(Y, W, rows, rows_f32, d, act_dtype, w_layout, ride, Ind, ind_dtype, seg_off, perm,
                                         rank_tmp, long_tab, j)) {
        if (!ride && !token_sums) {
            rc = launch_routing_table(Ind, ind_dtype, d, seg_off, perm, rank_tmp, cnt, long_tab, s);
            if (rc != EGS_OK) return rc;
        }
        rc = launch_rows_small_job(j, dw, nullptr, s);
        if (rc == EGS_OK && token_sums) return launch_token_sum(rows, rows_f32, Ind, ind_dtype, Out, d, act_dtype, s);
    } else {
        rows_f32 = mode != EGS_SCATTER_ATOMIC || act_dtype == EGS_F32;   // fast mode: rows in the element type
        // Product rows that one launch writes and the next reads back are still in the 256 MB memory-side
        // cache when there are few enough of them.  A call with more is processed as groups of batch
        // elements (independent of each other; the routing tables of all of them are built with the first
        // group): the largest groups whose rows take at most 144 MB, provided the weights, which every
        // group reads again, fit beside them and the groups still fill the 256-row tiles of the product
        // kernel.  C4: 2 groups of 8, 142 -> 123 us; C3: 8 groups of 1, 600 -> 565 us.  Smaller groups than
        // necessary lose more in the product kernel than the cache returns (C4, groups of 4: 168 us).
        int G = d->B;
        {
            const uint64_t per_b = (uint64_t)N * d->I * (rows_f32 ? 4 : ES);
            const uint64_t keep = 144ull << 20;
            if (per_b > 0 && per_b * d->B > (192ull << 20) && per_b <= keep) {
                const int fit = (int)(keep / per_b);
                const int groups = ceil_div(d->B, fit);
                const int g = ceil_div(d->B, groups);
                const uint64_t w_bytes = (uint64_t)d->E * d->I * d->J * ES;
                const int64_t rows_e = (int64_t)g * d->K;                     // rows per expert and group
                const int64_t padded = (rows_e + 255) / 256 * 256;
                if (groups > 1 && rows_e >= 256 && padded * 100 <= rows_e * 115 && w_bytes <= keep / 2) G = g;
            }
        }
        p.C = (char *)rows;
        p.seg_off = seg_off; p.perm = perm; p.rank_tmp = rank_tmp; p.long_tab = long_tab;
        // Whether the rows come with the bias is each group's own answer: a last group with fewer rows per expert than the large
        // product kernel takes runs the tiled one, which adds it.  Consecutive groups without it get it in one launch.
        int bare = 0;                   // batch elements from here up to the current group have no bias yet
        auto add_bias_up_to = [&](int b_end) -> int {
            if (bias == nullptr || bare >= b_end) return EGS_OK;
            egs_dims part = *d;
            part.B = b_end - bare;
            return bias_scatter((char *)Out + (size_t)bare * d->T * d->I * ES, bias, (const char *)Ind + (size_t)bare * N * ind_size(ind_dtype),
                                &part, act_dtype, ind_dtype, s);
        };
        bool token_sums = false;
        for (int b0 = 0; b0 < d->B; b0 += G) {
            egs_dims sub = *d;
            sub.B = d->B - b0 < G ? d->B - b0 : G;
            p.A = (const char *)Y + (size_t)b0 * N * d->J * ES;
            p.B = sub.B;
            const uint64_t span = (uint64_t)sub.B * N * d->J * ES;
            p.a_bytes = span < (1ull << 31) ? (uint32_t)span : 0;
            // the routing table may ride along with the (first) product launch (large shapes); otherwise it is a launch of its own
            p.csr_blocks = b0 == 0 && N > 0 ? d->B : 0; p.csr_done = 0;
            p.bias = bias; p.bias_done = 0;
            p.own_sums = b0 == 0 && (G == d->B || d->I % 4 != 0) && token_sums_take(d) && !(dw != nullptr && dw->done && dw->q.S > 1);
            rc = rows_gemm_scatter(p, act_dtype, w_trans, rows_f32 ? EPI_STORE_F32 : EPI_STORE, s, tdw);
            if (rc == EGS_OK && p.bias_done) {
                rc = add_bias_up_to(b0);
                bare = b0 + sub.B;
            }
            // Few picks, and the table would be a launch of its own for one launch of sums: sums that do without it.  us, product and
            // sums with the table riding along / without a table: bf16 B54 T1123 E15 K23 I192 J320 33 / 40, B14 T2048 E64 K60 I512 J128
            // 50 / 57, B16 T512 E16 K64 I256 J256 24.5 / 26.9, B8 T2048 E32 K100 I512 J256 38.0 / 36.3; three groups of f16 B61 T1657
            // E78 K45 I384 J384 234 / 272.  With a launch for the table: B53 T97 E29 K41 I111 J75 fp32 54 / 35.  Groups share one table: it is the
            // faster way for them but where rows are not whole pieces of four columns, which its sums add and store with half as many in flight: 120
            // scatters of two to nine groups of such rows take 0.90 of the time without it (0.94 under Zipf routing; up to one pick a token 0.70, f16
            // B101 T3838 E10 K116 I791 J47 680 / 376; from four on they are level, from sixteen on 1.04).
            if (b0 == 0)
                token_sums = p.own_sums && !p.csr_done;
            if (rc == EGS_OK && token_sums) {
                rc = launch_token_sum(rows, rows_f32, (const char *)Ind + (size_t)b0 * N * ind_size(ind_dtype), ind_dtype,
                                      (char *)Out + (size_t)b0 * d->T * d->I * ES, &sub, act_dtype, s);
            } else {
                if (rc == EGS_OK && b0 == 0 && !p.csr_done)
                    rc = launch_routing_table(Ind, ind_dtype, d, seg_off, perm, rank_tmp, cnt, long_tab, s);
                if (rc == EGS_OK)
                    rc = segment_sum_with(rows, rows_f32, seg_off + (size_t)b0 * (d->T + 1), perm + (size_t)b0 * N,
                                          long_tab + (size_t)b0 * long_tab_stride(N), long_part + (size_t)b0 * long_max_slots(N) * d->I,
                                          (char *)Out + (size_t)b0 * d->T * d->I * ES, &sub, act_dtype, b0 + G >= d->B ? dw : nullptr, s);
            }
            if (rc != EGS_OK) return rc;
        }
        bias_done = true;
        return add_bias_up_to(d->B);
    }
    if (rc != EGS_OK) return rc;
    return segment_sum_with(rows, rows_f32, seg_off, perm, long_tab, long_part, Out, d, act_dtype, dw, s);
}

int dw_impl(const void *Xs, const void *Ys, const void *Ind, void *dW, void *workspace, const egs_dims *d,
            int64_t ldx_b, int64_t ldx_t, int act_dtype, int out_dtype, int ind_dtype, int dw_layout, hipStream_t s)
{
    if ((size_t)d->E * d->I * d->J == 0) return EGS_OK;
    DwPlan pl = plan_dw(d, act_dtype);
    switch (dw_choose(Xs, Ys, dW, d, ldx_b, ldx_t, act_dtype, pl).path) {
    case DW_TILE: {
        DwTileJob jt;
        make_dw_tile(Xs, Ys, Ind, dW, d, ldx_b, ldx_t, act_dtype, out_dtype, ind_dtype, dw_layout, jt, dw_tile_wide_alone(d, act_dtype));
        return launch_dw_tile_alone(jt, s);
    }
    case DW_SMALL: {
        SmallDwJob j;
        make_dw_small(Xs, Ys, Ind, dW, workspace, d, ldx_b, ldx_t, act_dtype, out_dtype, ind_dtype, dw_layout, pl, j);
        const int rc = launch_dw_small_alone(j, s);
        return rc != EGS_OK ? rc : launch_dw_reduce4(j, s);
    }
    default:
        return dw_general(Xs, Ys, Ind, dW, workspace, d, ldx_b, ldx_t, act_dtype, out_dtype, ind_dtype, dw_layout, pl, s);
    }
}

// ------------------------------------------------------------------------------ validation
int validate_gather(const void *X, const void *W, const void *Ind, const void *Y, const float *w_scale,
                    const egs_dims *d, int64_t ldx_b, int64_t ldx_t, int act_dtype, int w_dtype, int ind_dtype,
                    int w_layout)
{
    int rc = check_dims(d);
    if (rc != EGS_OK) return rc;
    if (!act_dtype_ok(act_dtype) || !ind_dtype_ok(ind_dtype)) return EGS_ERR_BAD_DTYPE;
    if (w_dtype == EGS_FP8_E4M3) {
        if (act_dtype != EGS_BF16) return EGS_ERR_UNSUPPORTED;    // fp8 weights pair with bf16 activations
        if (w_scale == nullptr) return EGS_ERR_NULL_POINTER;
    } else if (w_dtype != act_dtype) {
        return act_dtype_ok(w_dtype) ? EGS_ERR_UNSUPPORTED : EGS_ERR_BAD_DTYPE;
    }
    if (!layout_ok(w_layout)) return EGS_ERR_BAD_LAYOUT;
    const size_t y_elems = (size_t)d->B * d->E * d->K * d->J;
    if (y_elems == 0) return EGS_OK;
    if (Y == nullptr || Ind == nullptr) return EGS_ERR_NULL_POINTER;
    if (d->I > 0 && (X == nullptr || W == nullptr)) return EGS_ERR_NULL_POINTER;
    if (d->I > 0 && d->T == 0) return EGS_OK;                      // every pick is out of range
    if (ldx_t < d->I || (d->B > 1 && ldx_b < 0)) return EGS_ERR_BAD_STRIDE;
    const int ES = elem_size(act_dtype);
    if (!aligned_to(X, ES) || !aligned_to(Y, ES) || !aligned_to(W, elem_size(w_dtype))) return EGS_ERR_ALIGNMENT;
    return EGS_OK;
}

int validate_scatter(const void *Y, const void *W, const void *Ind, const void *Out, const void *workspace,
                     size_t workspace_bytes, const egs_dims *d, int act_dtype, int ind_dtype, int w_layout, int mode, ScatterPath &path,
                     bool gather_backward = false)
{
    path = SCATTER_ROWS;
    int rc = check_dims(d);
    if (rc != EGS_OK) return rc;
    if (!act_dtype_ok(act_dtype) || !ind_dtype_ok(ind_dtype)) return EGS_ERR_BAD_DTYPE;
    if (!layout_ok(w_layout)) return EGS_ERR_BAD_LAYOUT;
    if (!mode_ok(mode)) return EGS_ERR_BAD_MODE;
    const size_t out_elems = (size_t)d->B * d->T * d->I;
    if (out_elems == 0) return EGS_OK;
    if (Out == nullptr) return EGS_ERR_NULL_POINTER;
    const size_t picks = (size_t)d->B * d->E * d->K;
    if (picks > 0 && Ind == nullptr) return EGS_ERR_NULL_POINTER;
    if (picks > 0 && d->J > 0 && (Y == nullptr || W == nullptr)) return EGS_ERR_NULL_POINTER;
    path = scatter_choose(Y, W, Out, d, act_dtype, mode, gather_backward, aligned_to(workspace, 256) && workspace != nullptr ? workspace_bytes : 0);
    const size_t need = plan_scatter(d, mode, act_dtype, path).bytes;
    if (need > 0 && (workspace == nullptr || workspace_bytes < need)) return EGS_ERR_WORKSPACE;
    if (need > 0 && !aligned_to(workspace, 256)) return EGS_ERR_ALIGNMENT;
    const int ES = elem_size(act_dtype);
    if (!aligned_to(Y, ES) || !aligned_to(Out, ES) || !aligned_to(W, ES)) return EGS_ERR_ALIGNMENT;
    return EGS_OK;
}

int validate_dw(const void *Xs, const void *Ys, const void *Ind, const void *dW, const void *workspace,
                size_t workspace_bytes, const egs_dims *d, int64_t ldx_b, int64_t ldx_t, int act_dtype,
                int out_dtype, int ind_dtype, int dw_layout)
{
    int rc = check_dims(d);
    if (rc != EGS_OK) return rc;
    if (!act_dtype_ok(act_dtype) || !act_dtype_ok(out_dtype) || !ind_dtype_ok(ind_dtype)) return EGS_ERR_BAD_DTYPE;
    if (!layout_ok(dw_layout)) return EGS_ERR_BAD_LAYOUT;
    const size_t w_elems = (size_t)d->E * d->I * d->J;
    if (w_elems == 0) return EGS_OK;
    if (dW == nullptr) return EGS_ERR_NULL_POINTER;
    const size_t picks = (size_t)d->B * d->K;
    if (picks > 0 && (Xs == nullptr || Ys == nullptr || Ind == nullptr)) return EGS_ERR_NULL_POINTER;
    if (picks > 0 && d->T > 0 && (ldx_t < d->I || (d->B > 1 && ldx_b < 0))) return EGS_ERR_BAD_STRIDE;
    const size_t need = picks > 0 ? dw_choose(Xs, Ys, const_cast<void *>(dW), d, ldx_b, ldx_t, act_dtype, plan_dw(d, act_dtype)).bytes : 0;
    if (need > 0 && (workspace == nullptr || workspace_bytes < need)) return EGS_ERR_WORKSPACE;
    if (need > 0 && !aligned_to(workspace, 256)) return EGS_ERR_ALIGNMENT;
    const int ES = elem_size(act_dtype);
    if (!aligned_to(Xs, ES) || !aligned_to(Ys, ES) || !aligned_to(dW, elem_size(out_dtype))) return EGS_ERR_ALIGNMENT;
    return EGS_OK;
}

}  // namespace

// ================================================================================ C ABI
extern "C" {

int egs_abi_version(void) { return EGS_ABI_VERSION; }

const char *egs_status_string(int status)
{
    switch (status) {
    case EGS_OK: return "ok";
    case EGS_ERR_NULL_POINTER: return "null pointer argument";
    case EGS_ERR_BAD_SHAPE: return "negative or too large dimension";
    case EGS_ERR_BAD_DTYPE: return "Unknown dtype";
    case EGS_ERR_BAD_LAYOUT: return "unknown weight layout";
    case EGS_ERR_BAD_MODE: return "unknown scatter mode";
    case EGS_ERR_WORKSPACE: return "workspace missing or too small";
    case EGS_ERR_ALIGNMENT: return "pointer not aligned to its element size (workspace: 256 bytes)";
    case EGS_ERR_HIP: return "HIP runtime error";
    case EGS_ERR_UNSUPPORTED: return "unsupported dtype combination";
    case EGS_ERR_BAD_STRIDE: return "source stride smaller than its row";
    case EGS_ERR_SCRATCH_LIMIT: return "sizes need more scratch than the built-in buffer holds (EGS_BUILTIN_SCRATCH_BYTES)";
    default: return "unknown status";
    }
}

const char *egs_last_hip_error(void) { return last_hip_error(); }

void egs_testing_force_generic(int on) { g_force_generic.store(on != 0); }

void egs_testing_launch_log_begin(void)
{
    g_launch_log.on = true; g_launch_log.len = 0; g_launch_log.text[0] = 0;
}

size_t egs_testing_launch_log_end(char *buf, size_t n)
{
    const size_t len = g_launch_log.len;
    if (buf != nullptr && n > 0) {
        const size_t c = len < n - 1 ? len : n - 1;
        memcpy(buf, g_launch_log.text, c);
        buf[c] = 0;
    }
    g_launch_log.on = false; g_launch_log.len = 0; g_launch_log.text[0] = 0;
    return len;
}

size_t egs_workspace_bytes(int op, int mode, const egs_dims *d, int act_dtype)
{
    if (check_dims(d) != EGS_OK || !act_dtype_ok(act_dtype)) return 0;
    if (!mode_ok(mode)) mode = EGS_SCATTER_DETERMINISTIC;
    switch (op) {
    case EGS_OP_GATHER_GEMM: return 0;
    case EGS_OP_GEMM_SCATTER: return scatter_bytes_planned(d, mode, act_dtype, false);
    case EGS_OP_DW: return dw_bytes_planned(d, act_dtype);
    case EGS_OP_GATHER_BACKWARD: return scatter_bytes_planned(d, mode, act_dtype, true) + dw_bytes_planned(d, act_dtype);
    case EGS_OP_SCATTER_BACKWARD: return dw_bytes_planned(d, act_dtype);
    default: return 0;
    }
}

int egs_gather_gemm(const void *X, const void *W, const void *Ind, void *Y, const float *w_scale,
                    const egs_dims *d, int64_t ldx_b, int64_t ldx_t,
                    int act_dtype, int w_dtype, int ind_dtype, int w_layout, void *stream)
{
    int rc = validate_gather(X, W, Ind, Y, w_scale, d, ldx_b, ldx_t, act_dtype, w_dtype, ind_dtype, w_layout);
    if (rc != EGS_OK) return rc;
    if ((size_t)d->B * d->E * d->K * d->J == 0) return EGS_OK;
    return gather_gemm_impl(X, W, Ind, Y, w_scale, d, ldx_b, ldx_t, act_dtype, w_dtype, ind_dtype, w_layout,
                            (hipStream_t)stream);
}

int egs_gemm_scatter(const void *Y, const void *W, const void *Ind, void *Out,
                     void *workspace, size_t workspace_bytes, const egs_dims *d,
                     int act_dtype, int ind_dtype, int w_layout, int mode, void *stream)
{
    ScatterPath path;
    int rc = validate_scatter(Y, W, Ind, Out, workspace, workspace_bytes, d, act_dtype, ind_dtype, w_layout, mode, path);
    if (rc != EGS_OK) return rc;
    return gemm_scatter_impl(Y, W, Ind, Out, workspace, d, act_dtype, ind_dtype, w_layout, mode, path, nullptr, nullptr,
                             (hipStream_t)stream);
}

int egs_dw(const void *Xsrc, const void *Ysrc, const void *Ind, void *dW,
           void *workspace, size_t workspace_bytes, const egs_dims *d,
           int64_t ldx_b, int64_t ldx_t,
           int act_dtype, int out_dtype, int ind_dtype, int dw_layout, void *stream)
{
    int rc = validate_dw(Xsrc, Ysrc, Ind, dW, workspace, workspace_bytes, d, ldx_b, ldx_t, act_dtype, out_dtype,
                         ind_dtype, dw_layout);
    if (rc != EGS_OK) return rc;
    return dw_impl(Xsrc, Ysrc, Ind, dW, workspace, d, ldx_b, ldx_t, act_dtype, out_dtype, ind_dtype, dw_layout,
                   (hipStream_t)stream);
}

int egs_dw_builtin_scratch(const void *Xsrc, const void *Ysrc, const void *Ind, void *dW, const egs_dims *d,
                           int64_t ldx_b, int64_t ldx_t,
                           int act_dtype, int out_dtype, int ind_dtype, int dw_layout, void *stream)
{
    int rc = check_dims(d);
    if (rc != EGS_OK) return rc;
    if (!act_dtype_ok(act_dtype)) return EGS_ERR_BAD_DTYPE;
    if (!layout_ok(dw_layout)) return EGS_ERR_BAD_LAYOUT;
    const size_t need = dw_choose(Xsrc, Ysrc, dW, d, ldx_b, ldx_t, act_dtype, plan_dw(d, act_dtype)).bytes;
    if (need > (size_t)EGS_BUILTIN_SCRATCH_BYTES) return EGS_ERR_SCRATCH_LIMIT;
    // the remaining checks are those of egs_dw; the stand-in address only has to look like a valid workspace
    rc = validate_dw(Xsrc, Ysrc, Ind, dW, need > 0 ? (const void *)(uintptr_t)256 : nullptr, need, d, ldx_b, ldx_t, act_dtype,
                     out_dtype, ind_dtype, dw_layout);
    if (rc != EGS_OK) return rc;
    if ((size_t)d->E * d->I * d->J == 0) return EGS_OK;
    void *ws = nullptr;
    if (need > 0) {
        rc = builtin_scratch_ptr(&ws);
        if (rc != EGS_OK) return rc;
    }
    // the partial sums of every split are written before the second pass reads them: nothing in the
    // buffer has to start at zero
    return dw_impl(Xsrc, Ysrc, Ind, dW, ws, d, ldx_b, ldx_t, act_dtype, out_dtype, ind_dtype, dw_layout,
                   (hipStream_t)stream);
}

int egs_expert_gather_forward(const void *X, const void *W, const void *Ind, void *Y,
                              const egs_dims *d, int64_t ldx_b, int64_t ldx_t,
                              int dtype, int ind_dtype, void *stream)
{
    return egs_gather_gemm(X, W, Ind, Y, nullptr, d, ldx_b, ldx_t, dtype, dtype, ind_dtype, EGS_W_EIJ, stream);
}

static int gather_backward_impl(const void *X, const void *W, const void *Ind, const void *grad_Y,
                                void *grad_X, void *grad_W,
                                void *workspace, size_t workspace_bytes, const egs_dims *d,
                                int64_t ldx_b, int64_t ldx_t,
                                int dtype, int ind_dtype, int mode, void *stream, void *table, size_t table_bytes)
{
    int rc = check_dims(d);
    if (rc != EGS_OK) return rc;
    if (!act_dtype_ok(dtype)) return EGS_ERR_BAD_DTYPE;
    if (!mode_ok(mode)) return EGS_ERR_BAD_MODE;
    if (grad_X == nullptr && (size_t)d->B * d->T * d->I > 0) return EGS_ERR_NULL_POINTER;
    RoutingTable tab;
    bool have_tab = false;
    rc = check_table_arg(table, table_bytes, d, dtype, tab, have_tab);
    if (rc != EGS_OK) return rc;
    const size_t ws_dw = (size_t)d->B * d->K > 0 && (size_t)d->E * d->I * d->J > 0 && grad_W != nullptr
        ? dw_choose(X, grad_Y, grad_W, d, ldx_b, ldx_t, dtype, plan_dw(d, dtype)).bytes : 0;
    // the weight gradient's part is at the end of what the scatter needs
    const size_t given = workspace != nullptr && aligned_to(workspace, 256) && workspace_bytes > ws_dw ? workspace_bytes - ws_dw : 0;
    const size_t ws_scatter = plan_scatter(d, mode, dtype, scatter_choose(grad_Y, W, grad_X, d, dtype, mode, true, given)).bytes;
    if (ws_scatter + ws_dw > 0 && (workspace == nullptr || workspace_bytes < ws_scatter + ws_dw)) return EGS_ERR_WORKSPACE;
    // validate both halves before enqueuing anything
    ScatterPath path;
    rc = validate_scatter(grad_Y, W, Ind, grad_X, workspace, ws_scatter, d, dtype, ind_dtype, EGS_W_EIJ, mode, path, true);
    if (rc != EGS_OK) return rc;
    void *ws2 = workspace ? (char *)workspace + ws_scatter : nullptr;
    rc = validate_dw(X, grad_Y, Ind, grad_W, ws2, ws_dw, d, ldx_b, ldx_t, dtype, dtype, ind_dtype, EGS_W_EIJ);
    if (rc != EGS_OK) return rc;
    // grad_X[b,t,i] = sum_picks sum_j grad_Y[b,e,k,j] * W[e,i,j];  grad_W[e,i,j] = sum X[b,Ind,i] * grad_Y[b,e,k,j].
    // The two are independent: for small experts the weight gradient shares the scatter's launches.
    hipStream_t s = (hipStream_t)stream;
    const size_t w_elems = (size_t)d->E * d->I * d->J;
    const DwPlan dpl = plan_dw(d, dtype);
    SmallDwJob dwj;
    DwTileJob dwt;
    // 32 x 32 tiles when they can share the launch of the one-kernel scatter, else what suits a launch of its own
    const bool shares_launch = path == SCATTER_FUSED && gather_backward_shares(scatter_fused_plan(grad_Y, W, grad_X, d, dtype), d, dtype);
    const bool dw_tile = w_elems > 0 && make_dw_tile(X, grad_Y, Ind, grad_W, d, ldx_b, ldx_t, dtype, dtype, ind_dtype, EGS_W_EIJ, dwt,
                                                     !shares_launch && dw_tile_wide_alone(d, dtype), shares_launch);
    const bool dw_small = !dw_tile && w_elems > 0 && make_dw_small(X, grad_Y, Ind, grad_W, ws2, d, ldx_b, ldx_t, dtype, dtype,
                                                                   ind_dtype, EGS_W_EIJ, dpl, dwj);
    TiledDwJob tdw;
    const bool dw_tiled = !dw_tile && !dw_small && w_elems > 0 && make_tiled_dw(X, grad_Y, Ind, grad_W, ws2, d, ldx_b, ldx_t, dtype, dtype, ind_dtype,
                                                                                EGS_W_EIJ, dpl, tdw);
    rc = gemm_scatter_impl(grad_Y, W, Ind, grad_X, workspace, d, dtype, ind_dtype, EGS_W_EIJ, mode, path, dw_small ? &dwj : nullptr,
                           dw_tile ? &dwt : nullptr, s, have_tab ? &tab : nullptr, nullptr, dw_tiled ? &tdw : nullptr);
    if (rc != EGS_OK) return rc;
    if (w_elems == 0) return EGS_OK;
    if (dw_tile) return dwt.done ? EGS_OK : launch_dw_tile_alone(dwt, s);
    if (dw_small) {
        if (!dwj.done) { rc = launch_dw_small_alone(dwj, s); if (rc != EGS_OK) return rc; }
        return launch_dw_reduce4(dwj, s);       // no-op when the reduction launch already did it
    }
    return dw_general(X, grad_Y, Ind, grad_W, ws2, d, ldx_b, ldx_t, dtype, dtype, ind_dtype, EGS_W_EIJ, dpl, s, dw_tiled ? &tdw : nullptr);
}

int egs_expert_gather_backward(const void *X, const void *W, const void *Ind, const void *grad_Y,
                               void *grad_X, void *grad_W,
                               void *workspace, size_t workspace_bytes, const egs_dims *d,
                               int64_t ldx_b, int64_t ldx_t,
                               int dtype, int ind_dtype, int mode, void *stream)
{
    return gather_backward_impl(X, W, Ind, grad_Y, grad_X, grad_W, workspace, workspace_bytes, d, ldx_b, ldx_t, dtype, ind_dtype,
                                mode, stream, nullptr, 0);
}

int egs_expert_gather_backward_table(const void *X, const void *W, const void *Ind, const void *table, size_t table_bytes,
                                     const void *grad_Y, void *grad_X, void *grad_W,
                                     void *workspace, size_t workspace_bytes, const egs_dims *d,
                                     int64_t ldx_b, int64_t ldx_t,
                                     int dtype, int ind_dtype, int mode, void *stream)
{
    return gather_backward_impl(X, W, Ind, grad_Y, grad_X, grad_W, workspace, workspace_bytes, d, ldx_b, ldx_t, dtype, ind_dtype,
                                mode, stream, const_cast<void *>(table), table_bytes);
}

int egs_expert_scatter_forward(const void *Y, const void *W, const void *Ind, void *Out,
                               void *workspace, size_t workspace_bytes, const egs_dims *d,
                               int dtype, int ind_dtype, int mode, void *stream)
{
    return egs_gemm_scatter(Y, W, Ind, Out, workspace, workspace_bytes, d, dtype, ind_dtype, EGS_W_EJI, mode, stream);
}

int egs_expert_scatter_bias_forward(const void *Y, const void *W, const void *bias, const void *Ind, const void *table, size_t table_bytes,
                                    void *Out, void *workspace, size_t workspace_bytes, const egs_dims *d,
                                    int dtype, int ind_dtype, int mode, void *stream)
{
    ScatterPath path;
    int rc = validate_scatter(Y, W, Ind, Out, workspace, workspace_bytes, d, dtype, ind_dtype, EGS_W_EJI, mode, path);
    if (rc != EGS_OK) return rc;
    if (bias != nullptr && !aligned_to(bias, elem_size(dtype))) return EGS_ERR_ALIGNMENT;
    RoutingTable tab;
    bool have_tab = false;
    rc = check_table_arg(const_cast<void *>(table), table_bytes, d, dtype, tab, have_tab);
    if (rc != EGS_OK) return rc;
    return gemm_scatter_impl(Y, W, Ind, Out, workspace, d, dtype, ind_dtype, EGS_W_EJI, mode, path, nullptr, nullptr,
                             (hipStream_t)stream, have_tab ? &tab : nullptr, bias);
}

int egs_expert_scatter_forward_table(const void *Y, const void *W, const void *Ind, const void *table, size_t table_bytes,
                                     void *Out, void *workspace, size_t workspace_bytes, const egs_dims *d,
                                     int dtype, int ind_dtype, int mode, void *stream)
{
    return egs_expert_scatter_bias_forward(Y, W, nullptr, Ind, table, table_bytes, Out, workspace, workspace_bytes, d, dtype, ind_dtype, mode, stream);
}

size_t egs_routing_table_bytes(const egs_dims *d, int dtype)
{
    if (check_dims(d) != EGS_OK) return 0;
    const TableLayout l = routing_table_layout(d, dtype);
    return l.ok && l.worth ? l.bytes : 0;
}

int egs_expert_gather_act_forward(const void *X, const void *W, const void *bias, const void *Ind, void *Y, void *table, size_t table_bytes,
                                  const egs_dims *d, int64_t ldx_b, int64_t ldx_t,
                                  int dtype, int ind_dtype, int activation, void *stream)
{
    int rc = validate_gather(X, W, Ind, Y, nullptr, d, ldx_b, ldx_t, dtype, dtype, ind_dtype, EGS_W_EIJ);
    if (rc != EGS_OK) return rc;
    const int act = activation & ~EGS_ACT_ROUND_FIRST;
    if (act < EGS_ACT_NONE || act > EGS_ACT_GELU_TANH) return EGS_ERR_BAD_MODE;
    if (act <= EGS_ACT_RELU) activation = act;      // the same values either way
    if (dtype == EGS_F32 && act != EGS_ACT_NONE) return EGS_ERR_UNSUPPORTED;      // the approximations are for 16-bit results
    if (bias != nullptr && (act != EGS_ACT_NONE || !aligned_to(bias, elem_size(dtype)))) return act != EGS_ACT_NONE ? EGS_ERR_UNSUPPORTED : EGS_ERR_ALIGNMENT;
    RoutingTable tab;
    bool have_tab = false;
    rc = check_table_arg(table, table_bytes, d, dtype, tab, have_tab);
    if (rc != EGS_OK) return rc;
    if ((size_t)d->B * d->E * d->K * d->J == 0) return EGS_OK;
    return gather_gemm_impl(X, W, Ind, Y, nullptr, d, ldx_b, ldx_t, dtype, dtype, ind_dtype, EGS_W_EIJ, (hipStream_t)stream,
                            have_tab ? &tab : nullptr, activation, bias);
}

int egs_expert_gather_forward_table(const void *X, const void *W, const void *Ind, void *Y, void *table, size_t table_bytes,
                                    const egs_dims *d, int64_t ldx_b, int64_t ldx_t,
                                    int dtype, int ind_dtype, void *stream)
{
    return egs_expert_gather_act_forward(X, W, nullptr, Ind, Y, table, table_bytes, d, ldx_b, ldx_t, dtype, ind_dtype, EGS_ACT_NONE, stream);
}

int egs_expert_scatter_backward(const void *Y, const void *W, const void *Ind, const void *grad_Out,
                                void *grad_Y, void *grad_W,
                                void *workspace, size_t workspace_bytes, const egs_dims *d,
                                int64_t ldg_b, int64_t ldg_t,
                                int dtype, int ind_dtype, void *stream)
{
    int rc = validate_gather(grad_Out, W, Ind, grad_Y, nullptr, d, ldg_b, ldg_t, dtype, dtype, ind_dtype, EGS_W_EJI);
    if (rc != EGS_OK) return rc;
    rc = validate_dw(grad_Out, Y, Ind, grad_W, workspace, workspace_bytes, d, ldg_b, ldg_t, dtype, dtype, ind_dtype,
                     EGS_W_EJI);
    if (rc != EGS_OK) return rc;
    // grad_Y[b,e,k,j] = sum_i grad_Out[b,Ind,i] * W[e,j,i];  grad_W[e,j,i] = sum grad_Out[b,Ind,i] * Y[b,e,k,j].
    // Independent of each other: for small experts they share one launch.
    hipStream_t s = (hipStream_t)stream;
    const size_t y_elems = (size_t)d->B * d->E * d->K * d->J, w_elems = (size_t)d->E * d->I * d->J;
    const DwPlan dpl = plan_dw(d, dtype);
    SmallRowsJob gj;
    SmallDwJob dwj;
    const bool g_small = y_elems > 0 && make_gather_small(grad_Out, W, Ind, grad_Y, d, ldg_b, ldg_t, dtype, dtype, ind_dtype,
                                                          EGS_W_EJI, gj);
    DwTileJob dwt;
    if (g_small && w_elems > 0 &&
        make_dw_tile(grad_Out, Y, Ind, grad_W, d, ldg_b, ldg_t, dtype, dtype, ind_dtype, EGS_W_EJI, dwt, /*wide=*/true)) {
        // One launch: the gather regridded to 8 wavefronts per workgroup, the weight-gradient workgroups first in launch
        // order (they run longest).  The launch's LDS size admits one workgroup per CU, so the two bodies never share a
        // CU (sharing one costs the sum of their times); with more workgroups than CUs the gather's fill the CUs the
        // weight gradient leaves and then follow on each CU as it frees (B64 T256 E48 K32 I128 J64: 26.5 -> 21.1 us
        // against two launches, B128 E32: 30.9 -> 21.3 us).
        SmallRowsJob g8 = gj;
        const int64_t Me = (int64_t)d->B * d->K;
        g8.p.tiles_per_e = (int)((Me + 511) / 512);
        // (row tiles on the XCDs in groups of eight only: with four row tiles on two XCDs each this launch measured
        // 11.4 against 11.05 us at B64 T256 E32 K32 I128 J64 - its other half reads the same rows expert by expert)
        g8.p.rows_share_xcd = g8.p.tiles_per_e % 8 == 0 ? rows_xcd_map(d, d->I, d->J, 2, g8.p.tiles_per_e) : 0;
        g8.blocks = rows_xcd_blocks(g8.p.rows_share_xcd, g8.p.tiles_per_e, g8.p.E);
        if ((int64_t)g8.blocks + dwt.blocks <= INT32_MAX / 2) return launch_rows_small_job(g8, nullptr, &dwt, s);
    }
    const bool dw_tile = w_elems > 0 && make_dw_tile(grad_Out, Y, Ind, grad_W, d, ldg_b, ldg_t, dtype, dtype, ind_dtype, EGS_W_EJI, dwt,
                                                     dw_tile_wide_alone(d, dtype));
    if (dw_tile) {
        if (y_elems > 0) {
            rc = gather_gemm_impl(grad_Out, W, Ind, grad_Y, nullptr, d, ldg_b, ldg_t, dtype, dtype, ind_dtype, EGS_W_EJI, s);
            if (rc != EGS_OK) return rc;
        }
        return launch_dw_tile_alone(dwt, s);
    }
    const bool dw_small = !dw_tile && w_elems > 0 && make_dw_small(grad_Out, Y, Ind, grad_W, workspace, d, ldg_b, ldg_t, dtype,
                                                                   dtype, ind_dtype, EGS_W_EJI, dpl, dwj);
    if (g_small && dw_small) {
        rc = launch_rows_small_job(gj, &dwj, nullptr, s);
        if (rc != EGS_OK) return rc;
        return launch_dw_reduce4(dwj, s);
    }
    TiledDwJob tdw;
    const bool dw_tiled = !dw_small && w_elems > 0 && make_tiled_dw(grad_Out, Y, Ind, grad_W, workspace, d, ldg_b, ldg_t, dtype, dtype, ind_dtype,
                                                                    EGS_W_EJI, dpl, tdw);
    if (y_elems > 0) {
        rc = gather_gemm_impl(grad_Out, W, Ind, grad_Y, nullptr, d, ldg_b, ldg_t, dtype, dtype, ind_dtype, EGS_W_EJI, s, nullptr, ACT_NONE, nullptr,
                              dw_tiled ? &tdw : nullptr);
        if (rc != EGS_OK) return rc;
    }
    if (dw_tiled) return dw_general(grad_Out, Y, Ind, grad_W, workspace, d, ldg_b, ldg_t, dtype, dtype, ind_dtype, EGS_W_EJI, dpl, s, &tdw);
    return dw_impl(grad_Out, Y, Ind, grad_W, workspace, d, ldg_b, ldg_t, dtype, dtype, ind_dtype, EGS_W_EJI, s);
}

int egs_stream_capture_id(void *stream, unsigned long long *id)
{
    if (id == nullptr) return EGS_ERR_NULL_POINTER;
    *id = 0;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long cid = 0;
    const hipError_t err = hipStreamGetCaptureInfo((hipStream_t)stream, &status, &cid);
    if (err != hipSuccess) return hip_fail(err, "hipStreamGetCaptureInfo");
    if (status == hipStreamCaptureStatusActive) *id = cid;
    return EGS_OK;
}

int egs_validate_indices(const void *Ind, int ind_dtype, int64_t n, int32_t T, int32_t *d_bad_count, void *stream)
{
    if (n < 0) return EGS_ERR_BAD_SHAPE;
    if (!ind_dtype_ok(ind_dtype)) return EGS_ERR_BAD_DTYPE;
    if (n == 0) return EGS_OK;
    if (Ind == nullptr || d_bad_count == nullptr) return EGS_ERR_NULL_POINTER;
    hipLaunchKernelGGL(validate_indices_kernel, dim3(grid_1d((size_t)n, 1024)), dim3(kThreads), 0, (hipStream_t)stream,
                       Ind, ind_dtype, n, T, d_bad_count);
    EGS_CHECK_LAUNCH("validate_indices_kernel");
    return EGS_OK;
}

}  // extern "C"
