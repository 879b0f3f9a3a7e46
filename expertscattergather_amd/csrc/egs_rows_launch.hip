// Launch side of the rows x weight products: rows_gemm_dl_kernel for large well-formed 16-bit shapes, rows_gemm_kernel for other
// 16-bit shapes that fill its tiles, rows_strip_kernel for mid-sized ones, rows_atomic_f32_kernel for fp32 atomics on the output, else the tiled kernels of egs_tiled.h.
#include "egs_host.h"
#include "egs_rows_gemm_dl.h"
#include "egs_rows_strip.h"

namespace egs {
namespace host {
namespace {

// ------------------------------------------------------------------------------ rows-GEMM dispatch
// fp32 atomics on the output: the one epilogue that the tiled kernels of egs_tiled.h do not have.  128 x 128 tiles only for long reductions
// that fill the chip with them, where their half as many operand bytes count; else 64 x 64, of which a CU takes several.  us, 128 then
// 64: R2048 N1024 Me512 E32 617, 695; R1024 N1024 Me512 E32 374, 387; R2048 N200 Me400 E32 187, 171; R2048 N512 Me256 E16 187, 101; R512
// N128 Me4000 E16 109, 102; R128 N512 Me2048 E64 390, 304 (Zipf-routed 490, 362); R196 N220 Me51 E15 34, 14.4; R64 N96 Me4800 E60 181, 125
template <bool W_TRANS>
int launch_rows_atomic(RowsGemmParams &p, hipStream_t s)
{
    const int Me = p.B * p.K;
    const bool large = (p.R >= 1024 && (int64_t)p.E * ceil_div(Me, 128) * ceil_div(p.N, 128) >= 512) ||
                       (int64_t)8 * ceil_div(p.E, 8) * ceil_div(Me, 64) * ceil_div(p.N, 64) > INT32_MAX;       // (more than a grid holds)
    const int tile = large ? 128 : 64;
    p.m_tiles = ceil_div(Me, tile); p.n_tiles = ceil_div(p.N, tile);
    const int64_t grid = (int64_t)8 * ceil_div(p.E, 8) * p.m_tiles * p.n_tiles;
    if (grid > INT32_MAX) return EGS_ERR_BAD_SHAPE;
    if (large)
        hipLaunchKernelGGL((rows_atomic_f32_kernel<128, 128, 32, 2, 2, W_TRANS>), dim3((unsigned)grid), dim3(256), 0, s, p);
    else
        hipLaunchKernelGGL((rows_atomic_f32_kernel<64, 64, 32, 4, 1, W_TRANS>), dim3((unsigned)grid), dim3(256), 0, s, p);
    EGS_CHECK_LAUNCH("rows_atomic_f32_kernel");
    return EGS_OK;
}

// Which operand to keep in one XCD's L2 (4 MB each), by the bytes that then come from beyond it.  Row tiles outermost: the source
// once and the weights again for every row tile (for every XCD, if they fit).  Experts outermost: the weights once and a source
// row for every pick.  us, row tiles / experts outermost: bf16 R672 N96 Me2262 E99 106 / 69, f16 R1744 N104 Me2380 E70 235 / 204,
// f16 R896 N64 Me2405 E215 183 / 151; the other way bf16 R768 N64 Me2048 E32 18.5 / 19.7.  A source that fits is kept by either:
// f16 R64 N256 Me13157 E29 132 / 121; and where the weights are the larger operand the count promises more than row tiles
// outermost keep: f16 R1408 N32 Me140 E165 15.7 / 13.4.
bool rows_outermost(const RowsGemmParams &p, int ES, int WES)
{
    const double fits = 3.5e6, x = (double)p.B * p.T * p.R * ES, w = (double)p.E * p.R * p.N * WES;
    const double picked = (double)p.E * p.B * p.K * p.R * ES, row_tiles = ((double)p.B * p.K + 63) / 64;
    return x > fits && x > w && (x < picked ? x : picked) + w * (w <= fits ? 8 : row_tiles) < 1.05 * (picked + w);
}

// anything the direct-to-LDS kernels do not take
int launch_rows_tiled(RowsGemmParams &p, int act_dtype, bool fp8_w, bool w_trans, bool gather, int epi, hipStream_t s, TiledDwJob *dw)
{
    TiledRowsParams q;
    memset(&q, 0, sizeof(q));
    const int ES = elem_size(act_dtype), WES = fp8_w ? 1 : ES;
    q.A = p.A; q.W = p.W; q.Ind = p.Ind; q.C = p.C; q.w_scale = p.w_scale;
    q.a_bytes = gather && p.T < 1 ? 0 : (gather ? (int64_t)(p.B - 1) * p.lda_b + (int64_t)(p.T - 1) * p.lda_t + p.R : (int64_t)p.B * p.E * p.K * p.R) * ES;
    q.w_bytes = (int64_t)p.E * p.R * p.N * WES;
    q.lda_b = p.lda_b; q.lda_t = p.lda_t;
    q.B = p.B; q.T = p.T; q.E = p.E; q.K = p.K; q.R = p.R; q.N = p.N;
    q.ldc = gather ? p.N : product_ld(p.N);
    q.ind_dtype = p.ind_dtype; q.gather = gather; q.out_f32 = epi == EPI_STORE_F32; q.act = p.act; q.bias = (const char *)p.bias;
    p.bias_done = p.bias != nullptr;
    q.rows_major = gather && rows_outermost(p, ES, WES);
    if (fp8_w) return tiled_rows_fp8w(q, w_trans, s);
    return act_dtype == EGS_F32 ? tiled_rows_f32(q, w_trans, dw, s) : act_dtype == EGS_F16 ? tiled_rows_f16(q, w_trans, dw, s) : tiled_rows_bf16(q, w_trans, dw, s);
}

// Large 16-bit products that are not for the direct-to-LDS loads (reduction not a multiple of 64, or shorter than 128); `used`: they
// are taken here.  Worth it where 128 x 128 or 256 x 256 tiles are filled: by rows and columns, by the experts on each XCD and in the
// last round of workgroups.  At 212 shapes the product of the three separated what these tiles win (the 102 above the lines: 0.94 to
// 1.67 times, 1.26 on average) from what the small ones do (the others: 0.55 to 1.39, 0.95 on average); fp32 rows are bound by their
// stores more, so that their line lies lower.
template <class TT, bool GATHER, bool W_TRANS, int EPI>
int launch_rows_large(RowsGemmParams &p, bool &used, hipStream_t s)
{
    used = false;
    const int64_t Me = (int64_t)p.B * p.K;
    if (g_force_generic || Me < 192 || p.N < 96 || p.R % 8 != 0 || p.N % 8 != 0 || !p.a_vec || !p.w_vec || !aligned_to(p.C, 16) ||
        p.act != ACT_NONE || p.bias != nullptr || p.w_scale != nullptr)
        return EGS_OK;
    const bool big = p.N >= 192 && p.R >= 128;
    const int tile = big ? 256 : 128;
    const int64_t m_tiles = (Me + tile - 1) / tile, n_tiles = ceil_div(p.N, tile), grid = 8 * ceil_div(p.E, 8) * m_tiles * n_tiles;
    if (grid > INT32_MAX / 2) return EGS_OK;
    const int64_t tiles = p.E * m_tiles * n_tiles, round = big ? 256 : 512;         // workgroups that run at once
    const double filled = (double)Me * p.N / ((double)m_tiles * n_tiles * tile * tile) * p.E / (8 * ceil_div(p.E, 8)) *
                          tiles / ((tiles + round - 1) / round * round);
    if (filled < (EPI == EPI_STORE_F32 ? 0.6 : 0.7)) return EGS_OK;
    p.m_tiles = (int)m_tiles; p.n_tiles = (int)n_tiles;
    if (big) hipLaunchKernelGGL((rows_gemm_kernel<TT, 256, 256, 2, 4, GATHER, W_TRANS, EPI>), dim3((unsigned)grid), dim3(512), 0, s, p);
    else hipLaunchKernelGGL((rows_gemm_kernel<TT, 128, 128, 2, 2, GATHER, W_TRANS, EPI>), dim3((unsigned)grid), dim3(256), 0, s, p);
    EGS_CHECK_LAUNCH("rows_gemm_kernel");
    used = true;
    return EGS_OK;
}

// The direct-to-LDS pipeline for large, well-formed 16-bit products; `used`: it takes this one
template <class TT, int WES, bool GATHER, bool W_TRANS, int EPI>
int launch_rows_dl(RowsGemmParams &p, bool &used, hipStream_t s)
{
    used = false;
    const int Me = p.B * p.K;
    const int e_groups = ceil_div(p.E, 8);
    const bool well_formed = !g_force_generic && Me >= 256 && p.R >= 128 && p.R % 64 == 0 && p.N % (WES == 1 ? 16 : 8) == 0 && p.a_vec && p.w_vec &&
                             p.a_bytes != 0 && (uint64_t)p.R * p.N * 2 < (1ull << 31) && (WES == 1 || p.w_scale == nullptr) &&
                             (WES == 2 || aligned_to(p.W, 16)) && aligned_to(p.C, 16);
    if (!well_formed) return EGS_OK;
    if (p.N >= 192) {
        // 256 x 256 x 64 slabs, two stages.  256 x 128 tiles of
        // four wavefronts on 32-deep slabs, two workgroups to a CU, measured for these shapes: gather at C3 156 -> 170 us
        // (gathered rows fetched once per column tile), fp32 product rows at C3 38.7 -> 40.2 us per group and at C5
        // 1.80 -> 2.09 ms; at C4 31.9 -> 28.7 us, which the table workgroups riding along take back
        p.m_tiles = ceil_div(Me, 256); p.n_tiles = ceil_div(p.N, 256);
        int64_t grid = (int64_t)8 * e_groups * p.m_tiles * p.n_tiles;
        if (grid > INT32_MAX) return EGS_ERR_BAD_SHAPE;
        const size_t smem = GATHER ? 0 : (size_t)dl_smem_bytes_scatter(256, 256, 64, 2);
        p.csr_threads = 512;            // as many wavefronts as the histograms leave room for
        while (p.csr_threads > kWave && csr_count_lds(p.T, p.csr_threads / kWave) > smem) p.csr_threads >>= 1;
        if (GATHER || csr_count_lds(p.T, p.csr_threads / kWave) > smem) p.csr_blocks = 0;
        // many picks per batch element: several workgroups per table, each ranking a share whose wavefront
        // slices (512 picks) stay in registers; one workgroup ranking 32768 picks outlasts the product tiles
        // of its launch (C3: 100 against 38 us; with eight parts the launch takes 54 us, one more round of workgroups)
        p.csr_parts = 1;
        if (p.csr_blocks > 0) {
            const int64_t per = (int64_t)(p.csr_threads / kWave) * 512;
            const int64_t parts = ((int64_t)p.E * p.K + per - 1) / per;
            p.csr_parts = (int)(parts < 1 ? 1 : parts > 8 ? 8 : parts);
            p.csr_blocks *= p.csr_parts;
        }
        p.tile_blocks = (int)grid;
        p.stream_rows = !GATHER && EPI == EPI_STORE_F32 && (uint64_t)Me * p.E * p.N * 4 > (256ull << 20);
        // A workgroup per CU goes through its share of the tiles without refilling its pipeline between them (bf16 B1 T4096 E128 K256
        // I1024 J256, a group of the long-sequence configuration: 37.8 -> 36.5 us in a kernel trace); where table workgroups come first
        // the shares would end at different times (B8 T1024 E64 K128 I512 J128: 36 -> 40 us), and rows that are streamed need the LDS
        // for that.
        if (!GATHER && EPI == EPI_STORE_F32 && p.csr_blocks == 0 && !p.stream_rows && grid > 256) grid = 256;
        grid += p.csr_blocks;
        if (grid > INT32_MAX) return EGS_ERR_BAD_SHAPE;
        p.csr_done = p.csr_blocks > 0;
        // fp8 weights: a stage is 32 KB of rows + 16 KB of weight bytes, so three fit (C5 gather 1058 -> 1024 us)
        constexpr int STAGES = WES == 1 && GATHER ? 3 : 2;
        hipLaunchKernelGGL((rows_gemm_dl_kernel<TT, WES, 256, 256, 64, STAGES, GATHER, W_TRANS, EPI>), dim3((unsigned)grid), dim3(512), 0, s, p);
        EGS_CHECK_LAUNCH("rows_gemm_dl_kernel");
        used = true;
        return EGS_OK;
    }
    // 65..191 output columns.  The gathers of large, well-formed 16-bit shapes: 256 x 128 tiles of four wavefronts in three
    // stages of 32-deep slabs (75 KB), compiled for two
    // wavefronts per SIMD so that TWO workgroups share a CU and one's loads and stores run under the other's
    // matrix instructions: C4 gather 29.5 -> 21.5 us against 64-deep slabs in two stages with one workgroup per
    // CU.  (Left to itself the compiler gives a four-wavefront workgroup 144 + 128 accumulator registers, which
    // keeps a second workgroup off the CU whatever the LDS size.)
    if constexpr (WES == 2 && GATHER) {
        if (p.N > 64) {
            p.m_tiles = ceil_div(Me, 256); p.n_tiles = ceil_div(p.N, 128);
            const int64_t grid = (int64_t)8 * e_groups * p.m_tiles * p.n_tiles;
            if (grid > INT32_MAX) return EGS_ERR_BAD_SHAPE;
            p.csr_blocks = 0;
            hipLaunchKernelGGL((rows_gemm_dl_kernel<TT, 2, 256, 128, 32, 3, true, W_TRANS, EPI_STORE>), dim3((unsigned)grid),
                               dim3(dl_threads(256, 128)), 0, s, p);
            EGS_CHECK_LAUNCH("rows_gemm_dl_kernel");
            used = true;
        }
    }
    return EGS_OK;
}

// the two for 16-bit operands, in this order
template <class TT, bool GATHER, bool W_TRANS, int EPI>
int launch_rows_16(RowsGemmParams &p, bool &used, hipStream_t s)
{
    const int rc = launch_rows_dl<TT, 2, GATHER, W_TRANS, EPI>(p, used, s);
    if (used || rc != EGS_OK) return rc;
    p.csr_blocks = 0; p.csr_done = 0;
    return launch_rows_large<TT, GATHER, W_TRANS, EPI>(p, used, s);
}
template <class TT, bool GATHER, int EPI>
int launch_rows_16_w(RowsGemmParams &p, bool w_trans, bool &used, hipStream_t s)
{
    return w_trans ? launch_rows_16<TT, GATHER, true, EPI>(p, used, s) : launch_rows_16<TT, GATHER, false, EPI>(p, used, s);
}

template <class TT, bool W_TRANS, int WES = 2>
int launch_rows_strip(RowsStripParams &p, hipStream_t s)
{
    typedef RowsStripLds L;
    p.m_tiles = ceil_div(p.B * p.K, L::BM);
    p.n_tiles = ceil_div(p.N, L::BN);
    const int64_t total = (int64_t)p.E * p.m_tiles * p.n_tiles;
    if (total > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    static_assert(L::BYTES <= 64 * 1024, "no grant needed");
    hipLaunchKernelGGL((rows_strip_kernel<TT, W_TRANS, WES>), dim3((unsigned)(8 * ((total + 7) / 8))), dim3(kStripThreads), L::BYTES, s, p);
    EGS_CHECK_LAUNCH("rows_strip_kernel");
    return EGS_OK;
}

// the parameters of either kind of weights; false: operands that the kernel can't take
bool make_rows_strip(const RowsGemmParams &p, int act_dtype, int wes, bool gather, int epi, RowsStripParams &q)
{
    if (g_force_generic || act_dtype == EGS_F32 || !p.a_vec || !p.w_vec || p.a_bytes == 0 || !aligned_to(p.W, 16) || !aligned_to(p.C, 16) ||
        p.R % 8 != 0 || p.N % (wes == 1 ? 16 : 8) != 0 || (uint64_t)p.R * p.N * 2 >= (1ull << 31))
        return false;
    memset(&q, 0, sizeof(q));
    q.A = p.A; q.W = p.W; q.w_scale = p.w_scale; q.Ind = p.Ind; q.C = p.C; q.bias = (const char *)p.bias;
    q.lda_b = p.lda_b; q.lda_t = p.lda_t; q.a_bytes = p.a_bytes;
    q.B = p.B; q.T = p.T; q.E = p.E; q.K = p.K; q.R = p.R; q.N = p.N; q.ldc = gather ? p.N : product_ld(p.N);
    q.ind_dtype = p.ind_dtype; q.gather = gather; q.out_f32 = epi == EPI_STORE_F32; q.act = p.act;
    q.rows_major = gather && rows_outermost(p, 2, wes);
    return true;
}

// Mid-sized 16-bit products; `used`: rows_strip_kernel takes this one.  Against tiled_rows_kernel, us, strips / that: R768 N64 Me2048 E32 16.4 /
// 20.7, R328 N136 Me900 E20 10.3 / 13.9, R136 N328 12.5 / 13.8, R800 N64 Me1628 E34 18 / 22, R896 N128 Me232 E83 14.3 / 17.5, R704 N224
// Me85 E114 12.9 / 18.4; not with little work, counted in full tiles of 128 x 64
// (R352 N64 Me252 E18: 35, 6.2 / 5.3, R96 N48 Me576 E13: 44, 5.1 / 4.6, R160 N128 Me468 E8: 58, 5.5 / 4.8), nor up to 64 rows, which are one
// tile of that too (773 sizes 0.89 to 1.24 of its time, level on average: R80 N1920 Me40 E248 57 / 52 with the sums, R464 N1792 Me24 E194 99 / 86;
// 65 to 128 rows, two of them, 0.86), nor with columns mostly empty (R896 N32 Me119 E53 9.6 / 7.9, R288 N32 Me2080 E35 10.2 / 9.8) unless there are
// many and long ones (1972 strips, R800 N32 Me2146 E116 42 / 47; but R160 N32 Me1920 E103 35.7 / 32.3).  Of 4992 such products, 1686 of them
// taken, 21 were more than 3 % slower; since that kernel has reductions of up to four slabs written out, 105 of 895 taken ones of those are, on average
// still 0.98 of its time (R64 N576 Me2814 E14 20.8 / 20.5; with half a strip of columns empty R72 N96 Me9699 E61 60 / 47, R48 N96 Me1560 E116 21.6 / 17.6).
int rows_strip(RowsGemmParams &p, int act_dtype, bool w_trans, bool gather, int epi, bool &used, hipStream_t s)
{
    used = false;
    const int64_t Me = (int64_t)p.B * p.K, strips = p.E * ((Me + 127) / 128) * ceil_div(p.N, 64);
    const double full = (double)Me * p.N * p.E / (128 * 64);
    const bool half_empty = 10 * (int64_t)p.N < 6 * 64 * ceil_div(p.N, 64);
    if (full < 70 || Me <= 64 || (half_empty && (strips < 1500 || p.R < 400)) || p.w_scale != nullptr) return EGS_OK;
    RowsStripParams q;
    if (!make_rows_strip(p, act_dtype, 2, gather, epi, q)) return EGS_OK;
    const int rc = act_dtype == EGS_BF16 ? (w_trans ? launch_rows_strip<ElemBF16, true>(q, s) : launch_rows_strip<ElemBF16, false>(q, s))
                                         : (w_trans ? launch_rows_strip<ElemF16, true>(q, s) : launch_rows_strip<ElemF16, false>(q, s));
    if (rc != EGS_OK) return rc;
    p.csr_blocks = 0; p.csr_done = 0;
    p.bias_done = p.bias != nullptr;
    used = true;
    return EGS_OK;
}

// How much of the matrix work of 256 x 256 tiles, a round of one per CU at a time, is asked for: rows, columns, experts on each XCD and the last
// round are rarely full.
double dl_filled(const RowsGemmParams &p)
{
    const int64_t Me = (int64_t)p.B * p.K, tiles = 8 * (int64_t)ceil_div(p.E, 8) * ((Me + 255) / 256) * ceil_div(p.N, 256);
    return (double)p.E * Me * p.N / 65536 / (double)(256 * ((tiles + 255) / 256));
}

// fp8 weights in strips; `used`: they are taken.  By a model (us) of each of the three kernels that such a product can go to, fitted to 900 sizes of 65
// rows or more (within 4 % of most, tiled_rows_kernel 7): the turns at the fullest CU, three strips, two small tiles or one of 256 x 256 side by side,
// the weights' bytes and the results.
// Against 256 x 256 tiles on the direct-to-LDS loads 160 of 205 sizes are taken, none of them slower, and all take 0.76 of their time (0.757 is the
// least): B6 T220 E34 K61 I1664 J256 49 -> 26.5, B13 T189 E23 K36 I1408 J384 44 -> 30, B9 T575 E215 K35 I1536 J320 172 -> 118; not B31 T324 E65 K26
// I1536 J480 142 / 158.  Against tiled_rows_kernel 440 of 699, 3 of them more than 3 % slower (1.04), and all take 0.917 of their time (0.913):
// B15 T1637 E229 K7 I896 J192 30 -> 22, B16 T591 E166 K21 I1536 J144 82 -> 60, B15 T785 E27 K14 I768 J208 12.5 -> 10.4; not B9 T126 E41 K20 I1408
// J256 19.2 / 22.3, B3 T104 E32 K34 I1024 J64 9.8 / 11.5.
int rows_strip_fp8(RowsGemmParams &p, bool w_trans, bool &used, hipStream_t s)
{
    used = false;
    RowsStripParams q;
    const int64_t Me = (int64_t)p.B * p.K;
    if (!w_trans || Me <= 64 || !make_rows_strip(p, EGS_BF16, 1, true, EPI_STORE, q)) return EGS_OK;
    const auto per_cu = [](int64_t n) { return (n + 255) / 256; };
    const double slabs = p.R / 64.0, weights = (double)p.E * p.R * p.N * 1e-6, results = (double)p.E * Me * p.N * 1e-6;
    const double strips_us = 4.8 + slabs * cu_turns(per_cu(p.E * ((Me + 127) / 128) * ceil_div(p.N, 64)), 3, 0.41, 0.35) + 0.026 * weights + 0.63 * results;
    double other_us;
    if (Me >= 256 && p.N >= 192 && p.R >= 128 && p.R % 64 == 0) {
        const int64_t tiles = ((Me + 255) / 256) * ceil_div(p.N, 256);
        other_us = 2.9 + (double)per_cu(8 * ceil_div(p.E, 8) * tiles) * (9.9 + 1.2 * slabs) + 0.365 * slabs * (double)(p.E * tiles) / 256 + 0.054 * weights;
    } else {
        const int tn = tiled_columns(p.E, Me, p.N, false);
        const int64_t tiles = per_cu(p.E * ((Me + 63) / 64) * ceil_div(p.N, 16 * tn));
        other_us = 5.1 + slabs * cu_turns(tiles, 2, 0.112 + 0.062 * tn, 0.048 + 0.06 * tn) + 0.52 * (double)((tiles + 1) / 2) + 0.0057 * weights;
    }
    if (strips_us >= 0.97 * other_us) return EGS_OK;
    const int rc = launch_rows_strip<ElemBF16, true, 1>(q, s);
    if (rc != EGS_OK) return rc;
    p.csr_blocks = 0; p.csr_done = 0;
    p.bias_done = p.bias != nullptr;
    used = true;
    return EGS_OK;
}

}  // namespace

// `used`: rows_stream_kernel takes this product
int rows_stream(RowsGemmParams &p, int act_dtype, bool fp8_w, bool w_trans, bool gather, int epi, bool &used, hipStream_t s);

int rows_gemm_gather(RowsGemmParams &p, int act_dtype, bool fp8_w, bool w_trans, hipStream_t s, TiledDwJob *dw)
{
    if (p.B * p.K == 0 || p.E == 0 || p.N == 0) return EGS_OK;
    bool used = false;
    int rc = rows_stream(p, act_dtype, fp8_w, w_trans, true, EPI_STORE, used, s);      // (fewer rows than any other but the general kernel)
    if (used || rc != EGS_OK) return rc;
    // Too few 256-row tiles for the CUs: us, strips / the direct-to-LDS tiles, R1024 N256 Me1200 E5 (25 of 256 columns) 12 / 26, R512 N256 Me1024
    // E16 (64) 11.7 / 18, R448 N128 Me600 E50 (150 of 128 columns) 10.8 / 15, R256 N256 Me1600 E20 (140) 15.0 / 15.0, R448 N128 Me936 E71 (284)
    // 22 / 21
    const int64_t dl_tiles = p.E * (((int64_t)p.B * p.K + 255) / 256) * ceil_div(p.N, p.N >= 192 ? 256 : 128);
    if (!fp8_w && p.N > 64 && dl_tiles <= (p.N >= 192 ? 100 : 200)) {
        rc = rows_strip(p, act_dtype, w_trans, true, EPI_STORE, used, s);
        if (used || rc != EGS_OK) return rc;
    }
    if (fp8_w) {
        rc = rows_strip_fp8(p, w_trans, used, s);
        if (used || rc != EGS_OK) return rc;
    }
    if (fp8_w) { if (w_trans) rc = launch_rows_dl<ElemBF16, 1, true, true, EPI_STORE>(p, used, s); }
    else if (act_dtype == EGS_F16) rc = launch_rows_16_w<ElemF16, true, EPI_STORE>(p, w_trans, used, s);
    else if (act_dtype == EGS_BF16) rc = launch_rows_16_w<ElemBF16, true, EPI_STORE>(p, w_trans, used, s);
    if (used || rc != EGS_OK) return rc;
    if (!fp8_w) rc = rows_strip(p, act_dtype, w_trans, true, EPI_STORE, used, s);
    if (used || rc != EGS_OK) return rc;
    return launch_rows_tiled(p, act_dtype, fp8_w, w_trans, true, EPI_STORE, s, dw);
}

int rows_gemm_scatter(RowsGemmParams &p, int act_dtype, bool w_trans, int epi, hipStream_t s, TiledDwJob *dw)
{
    if (p.B * p.K == 0 || p.E == 0 || p.N == 0) return EGS_OK;
    if (epi == EPI_ATOMIC_F32) return w_trans ? launch_rows_atomic<true>(p, s) : launch_rows_atomic<false>(p, s);
    bool used = false;
    int rc = EGS_OK;
    // 256 x 256 tiles that are half empty, and few picks for each token (at most four, and with sums that find their picks themselves): strips without
    // a table, whose ranking outlasts the products that it rides with.  More picks a token are less of a gain, and a hot token's rows are many
    // workgroups' with a table; more rows than 256 MB are kept out of the caches by those tiles (B21 T138 E234 K13 I1152 J320, 294 MB, 203 / 220 us).
    // us, tiles and table / strips: bf16 B8 T3637 E42 K41 I544 J192 46 / 30.5, B11 T3988 E5 K29 I512 J192 31.5 / 20.8, B48 T1641 E28 K29 I320 J192 56 /
    // 42.  Of 326 sizes 158 are taken, in 0.84 of their time; 4 of them are more than 3 % slower (the worst 1.10).
    if (p.own_sums && epi == EPI_STORE_F32 && p.N >= 192 && (int64_t)p.E * p.K <= 4 * (int64_t)p.T && dl_filled(p) < 0.5 &&
        (uint64_t)p.B * p.K * p.E * p.N * 4 <= (256ull << 20)) {
        rc = rows_strip(p, act_dtype, w_trans, false, epi, used, s);
        if (used || rc != EGS_OK) return rc;
    }
    if (act_dtype == EGS_F16)
        rc = epi == EPI_STORE ? launch_rows_16_w<ElemF16, false, EPI_STORE>(p, w_trans, used, s) : launch_rows_16_w<ElemF16, false, EPI_STORE_F32>(p, w_trans, used, s);
    else if (act_dtype == EGS_BF16)
        rc = epi == EPI_STORE ? launch_rows_16_w<ElemBF16, false, EPI_STORE>(p, w_trans, used, s) : launch_rows_16_w<ElemBF16, false, EPI_STORE_F32>(p, w_trans, used, s);
    if (used || rc != EGS_OK) return rc;
    p.csr_blocks = 0; p.csr_done = 0;
    rc = rows_stream(p, act_dtype, false, w_trans, false, epi, used, s);
    if (used || rc != EGS_OK) return rc;
    rc = rows_strip(p, act_dtype, w_trans, false, epi, used, s);
    if (used || rc != EGS_OK) return rc;
    return launch_rows_tiled(p, act_dtype, false, w_trans, false, epi, s, dw);
}

}  // namespace host
}  // namespace egs
