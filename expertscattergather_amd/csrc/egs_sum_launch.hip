// Launch side of the sums over product rows (segment_sum_kernel with a routing table, token_sum_kernel without) and of the routing
// table as a launch of its own.
#include "egs_host.h"
#include "egs_scatter_aux.h"
#include "egs_small.h"

namespace egs {
namespace host {

// routing table of the deterministic scatter as a launch of its own: counting sort with
// per-wavefront histograms when they fit in LDS, bitonic sort in LDS for long sequences, else
// the one-wavefront counting sort
int launch_routing_table(const void *Ind, int ind_dtype, const egs_dims *d, int32_t *seg_off, int32_t *perm,
                         int32_t *rank_tmp, int32_t *cnt, int32_t *long_tab, hipStream_t s)
{
    const int64_t N = (int64_t)d->E * d->K;
    if (N >= 1) {
        // as many wavefronts as the per-wavefront histograms leave room for (up to 148 KB of LDS)
        const size_t budget = 148 * 1024;
        int nw = (int)((N + 63) / 64);
        if (nw > 16) nw = 16;
        while (nw > 1 && csr_count_lds(d->T, nw) > budget) nw >>= 1;
        const size_t lds = csr_count_lds(d->T, nw);
        if (lds <= budget) {
            // Several workgroups per table where a wavefront has more than four chunks of 64 picks, which it ranks one after the other: 16 us
            // for the 18 chunks of 17670 picks.  Every part also counts all picks, so not below that (us more with two parts at one to three
            // chunks: 0.5 to 1.3), and as many as there are CUs for, one workgroup each: scatters at B46 T1359 E128 K84 with one part 94.7, two
            // 84.5, four 81.8, six 94.0; B99 T1086 E128 K181 314, 306, 314, 328; B1 T1133 E64 K211 41.7, 31.9, 28.3 and with eight 25.8.
            const int64_t per = (int64_t)nw * 128, want = N <= 2 * per ? 1 : (N + per - 1) / per;
            const int64_t most = d->B >= 256 ? 1 : 256 / d->B < 8 ? 256 / d->B : 8;
            const int parts = (int)(want > most ? most : want);
            const auto kernel = parts > 1 ? csr_count_kernel<true> : csr_count_kernel<false>;
            static LdsGrant told[2];
            const int rc_lds = allow_large_lds((const void *)kernel, told[parts > 1], lds, "hipFuncSetAttribute(csr_count_kernel)");
            if (rc_lds != EGS_OK) return rc_lds;
            hipLaunchKernelGGL(kernel, dim3(d->B * parts), dim3(64 * nw), lds, s, Ind, ind_dtype, d->T, (int32_t)N, seg_off, perm, rank_tmp, long_tab, parts);
            EGS_CHECK_LAUNCH("csr_count_kernel");
            return EGS_OK;
        }
    }
    int NP = 1, QB = 0;
    while (NP < N) { NP <<= 1; ++QB; }
    const bool sortable = N >= 1 && NP <= 32768 && (((uint64_t)d->T << QB) <= 0xFFFFFFFFull);
    if (sortable) {
        const size_t lds = (size_t)NP * 4;
        static LdsGrant told;
        const int rc_lds = allow_large_lds((const void *)csr_sort_kernel, told, lds, "hipFuncSetAttribute(csr_sort_kernel)");
        if (rc_lds != EGS_OK) return rc_lds;
        int threads = NP / 2;
        if (threads < 64) threads = 64;
        if (threads > 1024) threads = 1024;
        hipLaunchKernelGGL(csr_sort_kernel, dim3(d->B), dim3(threads), lds, s, Ind, ind_dtype, d->T, (int32_t)N, NP, QB, seg_off, perm, long_tab);
        EGS_CHECK_LAUNCH("csr_sort_kernel");
        return EGS_OK;
    }
    const size_t lds = d->T > kCsrLdsTokens ? 0 : (size_t)d->T * 4;
    hipLaunchKernelGGL(csr_build_kernel, dim3(d->B), dim3(kWave), lds, s, Ind, ind_dtype, d->T, (int32_t)N, seg_off, perm, cnt, long_tab);
    EGS_CHECK_LAUNCH("csr_build_kernel");
    return EGS_OK;
}

// more product rows than the memory-side cache (256 MB) holds until they are read
static bool rows_stream_by(const egs_dims *d, size_t row_bytes) { return (uint64_t)d->B * d->E * d->K * row_bytes > (256ull << 20); }

template <class TT, class PT>
void launch_segment_sum8(const SegSumParams &sp, int seg_blocks, bool stream, hipStream_t s)
{
    if (stream) hipLaunchKernelGGL((segment_sum_kernel<TT, PT, 8, true>), dim3(seg_blocks), dim3(kThreads), 0, s, sp);
    else hipLaunchKernelGGL((segment_sum_kernel<TT, PT, 8>), dim3(seg_blocks), dim3(kThreads), 0, s, sp);
}

// fixed-order reduction of the product rows per token; when `reduce` is given (and qualifies) the
// second pass of that weight gradient shares the launch
int launch_segment_sum(const void *rows, bool rows_f32, const int32_t *seg_off, const int32_t *perm, int32_t *long_tab,
                       float *long_part, void *Out, const egs_dims *d, int act_dtype, DwSecondPass *reduce, hipStream_t s)
{
    const int N = d->E * d->K;
    const bool vw4 = d->I % 4 == 0 && aligned_to(Out, 16);
    // eight elements of a row per thread (16 bytes of a 16-bit row, two 16-byte loads of an fp32 row): half the threads,
    // table look-ups and address arithmetic per row
    const bool vw8 = vw4 && d->I % 8 == 0 && aligned_to(rows, 16) && reduce == nullptr;
    const int iv = vw8 ? d->I / 8 : vw4 ? d->I / 4 : d->I;
    SegSumParams sp;
    memset(&sp, 0, sizeof(sp));
    sp.P = rows; sp.seg_off = seg_off; sp.perm = perm; sp.out = (char *)Out;
    sp.B = d->B; sp.T = d->T; sp.N = N; sp.I = d->I; sp.ldp = product_ld(d->I);
    while ((1 << sp.tpr_log2) < iv && sp.tpr_log2 < 8) ++sp.tpr_log2;      // threads sharing an output row (<= 256)
    sp.gx = ceil_div(d->T, kThreads >> sp.tpr_log2);
    sp.gy = d->B;
    while ((int64_t)sp.gx * sp.gy > (1 << 22)) sp.gy = (sp.gy + 1) / 2;     // stride loop over batch elements beyond that
    sp.long_tab = long_tab; sp.long_part = long_part;
    const int64_t all_seg_blocks = (int64_t)sp.gx * sp.gy + (int64_t)d->B * long_max_slots(N);
    if (all_seg_blocks > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    const int seg_blocks = (int)all_seg_blocks;
    const bool fuse = reduce != nullptr && vw4;
    const int red_blocks = fuse ? grid_1d(reduce->w_elems / 4, 1024) : 0;
#define EGS_SEGSUM(TT, PT)                                                                                                  \
    do {                                                                                                                    \
        if (fuse) hipLaunchKernelGGL((segsum_dwreduce_kernel<TT, PT, 4>), dim3(seg_blocks + red_blocks), dim3(kThreads), 0, \
                                     s, sp, seg_blocks, reduce->part, reduce->dW, reduce->S, reduce->w_elems / 4,           \
                                     reduce->out_dtype);                                                                    \
        else if (vw8) launch_segment_sum8<TT, PT>(sp, seg_blocks, rows_stream_by(d, (size_t)sp.ldp * sizeof(PT)), s);       \
        else if (vw4) hipLaunchKernelGGL((segment_sum_kernel<TT, PT, 4>), dim3(seg_blocks), dim3(kThreads), 0, s, sp);      \
        else hipLaunchKernelGGL((segment_sum_kernel<TT, PT, 1>), dim3(seg_blocks), dim3(kThreads), 0, s, sp);               \
    } while (0)
    if (act_dtype == EGS_F32) EGS_SEGSUM(ElemF32, float);
    else if (act_dtype == EGS_F16) { if (rows_f32) EGS_SEGSUM(ElemF16, float); else EGS_SEGSUM(ElemF16, uint16_t); }
    else { if (rows_f32) EGS_SEGSUM(ElemBF16, float); else EGS_SEGSUM(ElemBF16, uint16_t); }
#undef EGS_SEGSUM
    EGS_CHECK_LAUNCH(fuse ? "segsum_dwreduce_kernel" : "segment_sum_kernel");
    if (fuse) reduce->done = true;
    return EGS_OK;
}

// the same without a routing table, for up to kTokenSumPicks picks per batch element
int launch_token_sum(const void *rows, bool rows_f32, const void *Ind, int ind_dtype, void *Out, const egs_dims *d, int act_dtype, hipStream_t s)
{
    TokenSumParams p;
    memset(&p, 0, sizeof(p));
    p.P = rows; p.Ind = Ind; p.out = (char *)Out;
    p.B = d->B; p.T = d->T; p.N = d->E * d->K; p.I = d->I; p.ldp = product_ld(d->I);
    p.ind_dtype = ind_dtype;
    // at most 64 threads (256 columns) per row, so that a hot token's segment has at least four groups of threads to share it
    p.tpr_log2 = 3;
    while ((4 << p.tpr_log2) < d->I && p.tpr_log2 < 6) ++p.tpr_log2;
    p.c_blocks = ceil_div(d->I, 4 << p.tpr_log2);
    // tokens per workgroup: one per group of threads, more (each workgroup reads all indices of its batch element) once that
    // alone makes a thousand workgroups
    const int groups = kThreads >> p.tpr_log2;
    p.tb = groups;
    while (p.tb < kTokenSumTokens && (int64_t)d->B * ceil_div(d->T, p.tb) * p.c_blocks > 1024) p.tb *= 2;
    p.t_blocks = ceil_div(d->T, p.tb);
    const int64_t grid = (int64_t)d->B * p.t_blocks * p.c_blocks;
    if (grid > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    const size_t lds = token_sum_lds(p.N);
    const bool stream = rows_stream_by(d, (size_t)p.ldp * (rows_f32 ? 4 : 2));
    const bool wave = p.tpr_log2 == 6;
#define EGS_TOKSUM(TT, PT)                                                                                              \
    do {                                                                                                                \
        const auto kernel = wave ? (stream ? token_sum_kernel<TT, PT, true, true> : token_sum_kernel<TT, PT, true, false>)       \
                                 : (stream ? token_sum_kernel<TT, PT, false, true> : token_sum_kernel<TT, PT, false, false>);    \
        hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kThreads), lds, s, p);                                    \
    } while (0)
    if (act_dtype == EGS_F32) EGS_TOKSUM(ElemF32, float);
    else if (act_dtype == EGS_F16) { if (rows_f32) EGS_TOKSUM(ElemF16, float); else EGS_TOKSUM(ElemF16, uint16_t); }
    else { if (rows_f32) EGS_TOKSUM(ElemBF16, float); else EGS_TOKSUM(ElemBF16, uint16_t); }
#undef EGS_TOKSUM
    EGS_CHECK_LAUNCH("token_sum_kernel");
    return EGS_OK;
}

}  // namespace host
}  // namespace egs
