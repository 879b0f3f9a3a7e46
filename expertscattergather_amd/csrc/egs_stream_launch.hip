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
    if (p.m_tiles == 1 && (uint64_t)p.E * p.R * p.N * WES > (128ull << 20)) hipLaunchKernelGGL((rows_stream_kernel<TT, WES, W_TRANS, MT, true>), grid, dim3(kThreads), L::BYTES, s, p);
    else hipLaunchKernelGGL((rows_stream_kernel<TT, WES, W_TRANS, MT, false>), grid, dim3(kThreads), L::BYTES, s, p);
    EGS_CHECK_LAUNCH("rows_stream_kernel");
    return EGS_OK;
}
template <class TT, int WES, bool W_TRANS>
int launch_stream(RowsStreamParams &p, int mt, hipStream_t s)
{
    return mt == 2 ? launch_stream<TT, WES, W_TRANS, 2>(p, s) : launch_stream<TT, WES, W_TRANS, 4>(p, s);
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
    // R2048 N384 Me28 E22 13.2 / 17.4, R1472 N64 Me24 E210 10.5 / 14.1, R576 N320 Me76 E40 7.8 / 10.0, R704 N256 Me30 E206 17.4 / 19.2 (fp8
    // 11.9 / 18.0), R1408 N128 Me116 E88 14.1 / 17.2, R640 N320 Me81 E117 18.3 / 18.7; level from 128 rows.  Short ones are over before three slabs are on
    // their way: R128 N1408 Me116 E88 62 / 53, R192 N384 Me120 E103 13.1 / 11.1, R256 N704 Me30 E206 33 / 31.
    const int cols = fp8_w ? 128 : 64;
    if (Me > 128 || p.R < 384 || p.N < cols) return EGS_OK;
    RowsStreamParams q;
    memset(&q, 0, sizeof(q));
    q.A = p.A; q.W = p.W; q.Ind = p.Ind; q.C = p.C; q.w_scale = p.w_scale; q.bias = (const char *)p.bias;
    q.lda_b = p.lda_b; q.lda_t = p.lda_t; q.a_bytes = p.a_bytes;
    q.B = p.B; q.T = p.T; q.E = p.E; q.K = p.K; q.R = p.R; q.N = p.N; q.ldc = p.N;
    q.ind_dtype = p.ind_dtype; q.gather = gather; q.out_f32 = epi == EPI_STORE_F32; q.act = p.act;
    // 64 rows at a time where there are workgroups enough to keep the weights coming (R2048 N512 Me64 E256 fp8 66 / 76, bf16 121 / 139), else 32
    // (R640 N320 Me81 E117 18.3 / 21.8)
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
