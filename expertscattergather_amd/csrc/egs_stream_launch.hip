// Launch side of rows_stream_kernel (egs_rows_stream.h)
#include "egs_host.h"
#include "egs_rows_stream.h"

namespace egs {
namespace host {
namespace {

template <class TT, int WES, bool W_TRANS, int MT>
int launch_stream(RowsStreamParams &p, hipStream_t s)
{
    typedef RowsStreamLds<WES, MT> L;
    p.m_tiles = ceil_div(p.B * p.K, L::BM);
    p.n_tiles = ceil_div(p.N, L::BN);
    const int64_t total = (int64_t)p.E * p.m_tiles * p.n_tiles;
    if (total > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    static_assert(L::BYTES <= 64 * 1024, "no grant needed");
    const dim3 grid((unsigned)(8 * ((total + 7) / 8)));
    // Weights of which two - a layer has a gather's and a scatter's - do not stay in the memory-side cache (256 MB) go past the caches.  Over 157 sizes,
    // past them against not, two weights in turn: 90 to 130 MB 1.07 to 1.13 of the time, to 150 MB 1.00 to 1.02, from there on 0.91 to 0.96
    // (B4 T512 E256 K8 I2048 J512, fp8, a gather and a scatter: 181 us and 188).  A call repeated by itself with the same weights finds them there
    // up to 256 MB, and loses 12 %: no layer does that.  (16-bit weights by 64 rows are always more.)
    constexpr bool kAlways = WES == 2 && MT == 4;
    const bool once = kAlways || (p.m_tiles == 1 && (uint64_t)p.E * p.R * p.N * WES > (128ull << 20));
    if (once) hipLaunchKernelGGL((rows_stream_kernel<TT, WES, W_TRANS, MT, true>), grid, dim3(kThreads), L::BYTES, s, p);
    else hipLaunchKernelGGL((rows_stream_kernel<TT, WES, W_TRANS, MT, kAlways>), grid, dim3(kThreads), L::BYTES, s, p);
    EGS_CHECK_LAUNCH("rows_stream_kernel");
    return EGS_OK;
}
template <class TT, int WES, bool W_TRANS>
int launch_stream(RowsStreamParams &p, int mt, hipStream_t s)
{
    return mt == 2 ? launch_stream<TT, WES, W_TRANS, 2>(p, s) : launch_stream<TT, WES, W_TRANS, 4>(p, s);
}

// fp8 weights: is this kernel faster than tiled_rows_kernel?  Both by the time of the fullest CU, fitted to 1565
// sizes of up to 128 rows: a fixed part, and for every 64 reduction elements what a CU's workgroups take side by side, three of this kernel's
// or two of the other's.  By it 23 sizes are 3 % slower than they could be, none 15 %.  us, it / that: R1792 N352 Me84 E236 64 / 90, R640
// N480 Me70 E165 27 / 37; not taken: R384 N304 Me102 E69 12.4 / 11.1, R1408 N144 Me50 E70 14.9 / 13.5, R1920 N144 Me28 E30 16.2 / 14.0.
bool stream_fp8_pays(int64_t E, int64_t Me, int R, int N)
{
    const auto rounds = [](int64_t n, int per, double alone, double each) {
        const int64_t rest = n % per;
        const auto round = [&](int64_t k) { return (double)k * each > alone ? (double)k * each : alone; };
        return (double)(n / per) * round(per) + (rest ? round(rest) : 0.0);
    };
    const int tn = tiled_columns(E, Me, N, false);
    const int64_t stream = (E * ((Me + 31) / 32) * ceil_div(N, 128) + 255) / 256, tiled = (E * ((Me + 63) / 64) * ceil_div(N, 16 * tn) + 255) / 256;
    const double slabs = R / 64;
    return 2.5 + 1.3 * (double)((stream + 2) / 3) + slabs * rounds(stream, 3, 0.37, 0.25) < 4.8 + slabs * rounds(tiled, 2, 0.14 + 0.064 * tn, 0.06 + 0.062 * tn);
}

}  // namespace

int rows_stream(RowsGemmParams &p, int act_dtype, bool fp8_w, bool w_trans, bool gather, int epi, bool &used, hipStream_t s)
{
    used = false;
    const int64_t Me = (int64_t)p.B * p.K;
    if (g_force_generic || act_dtype == EGS_F32 || (fp8_w && !w_trans) || !p.a_vec || !p.w_vec || p.a_bytes == 0 || !aligned_to(p.W, 16) || !aligned_to(p.C, 16) ||
        p.R % 64 != 0 || p.N % (fp8_w ? 16 : 8) != 0 || (uint64_t)p.R * p.N * (fp8_w ? 1 : 2) >= (1ull << 31))
        return EGS_OK;
    // us, this kernel and tiled_rows_kernel, bf16 weights unless said otherwise.  Long reductions of few rows: R2048 N512 Me32 E256 fp8 53 / 80, bf16 106 / 120;
    // R2048 N384 Me28 E22 13.2 / 17.4, R1472 N64 Me24 E210 10.5 / 14.1, R704 N256 Me30 E206 17.4 / 19.2 (fp8 11.9 / 18.0).  Short ones are over before
    // three slabs are on their way: R128 N1408 Me116 E88 62 / 53, R192 N384 Me120 E103 13.1 / 11.1, R256 N704 Me30 E206 33 / 31.
    const int cols = fp8_w ? 128 : 64;
    if (Me > 128 || p.R < 384 || p.N < cols) return EGS_OK;
    // Where it is the faster one, measured at 2300 sizes.  One round of workgroups, three to a CU, or a single row tile.  More rows than that
    // have every weight fetched by several row tiles in turn, and rows_strip_kernel's or tiled_rows_kernel's 64 columns fetch it once: us, it and
    // those, R1984 N256 Me128 E114 42 / 24, R640 N128 Me99 E196 18.6 / 12.3, R1216 N184 Me120 E159 34 / 20, R960 N408 Me64 E254 66 / 41; kept:
    // R1408 N128 Me116 E88 14.1 / 17.2, R576 N320 Me76 E40 7.8 / 10.0.  Weight rows that are no whole 128-byte lines cost a second line per piece,
    // which shows in more than a round (R1280 N312 Me26 E251 51 / 37, R1344 N400 Me17 E203 53 / 39).  Up to 64 rows also 64 at a time where the
    // weights come from memory in any case (R2048 N512 Me64 E256 121 / 139; 102 such sizes 0.85 to 1.04 of the other's time).
    const int64_t tiles = (int64_t)p.E * ceil_div(p.N, cols), row_tiles = (Me + 31) / 32;
    if (fp8_w) {
        if (!(tiles >= 1024 && Me <= 64) && !stream_fp8_pays(p.E, Me, p.R, p.N)) return EGS_OK;
    } else {
        const bool lines = !w_trans || p.N % 64 == 0;
        const bool from_memory = Me <= 64 && tiles >= 1024 && (uint64_t)p.E * p.R * p.N * 2 > (320ull << 20);
        if (row_tiles * tiles > 768 && !(lines && (Me <= 32 || from_memory))) return EGS_OK;
    }
    RowsStreamParams q;
    memset(&q, 0, sizeof(q));
    q.A = p.A; q.W = p.W; q.Ind = p.Ind; q.C = p.C; q.w_scale = p.w_scale; q.bias = (const char *)p.bias;
    q.lda_b = p.lda_b; q.lda_t = p.lda_t; q.a_bytes = p.a_bytes;
    q.B = p.B; q.T = p.T; q.E = p.E; q.K = p.K; q.R = p.R; q.N = p.N; q.ldc = p.N;
    q.ind_dtype = p.ind_dtype; q.gather = gather; q.out_f32 = epi == EPI_STORE_F32; q.act = p.act;
    // 64 rows at a time where there are workgroups enough to keep the weights coming (fp8 R2048 N512 Me64 E256 66 / 76), else 32 (R640 N320 Me81 E117
    // 18.3 / 21.8)
    const int mt = Me > 32 && (int64_t)p.E * ceil_div(p.N, cols) >= 1024 ? 4 : 2;
    const int rc = fp8_w ? launch_stream<ElemBF16, 1, true>(q, mt, s)
                 : act_dtype == EGS_BF16 ? (w_trans ? launch_stream<ElemBF16, 2, true>(q, mt, s) : launch_stream<ElemBF16, 2, false>(q, mt, s))
                                         : (w_trans ? launch_stream<ElemF16, 2, true>(q, mt, s) : launch_stream<ElemF16, 2, false>(q, mt, s));
    if (rc != EGS_OK) return rc;
    p.bias_done = p.bias != nullptr;
    used = true;
    return EGS_OK;
}

}  // namespace host
}  // namespace egs
