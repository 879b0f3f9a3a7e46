// Weight gradient for 16-bit shapes with many picks, on the direct-to-LDS pipeline, in tiles small enough to give every CU one:
//
//   dW(e, i, j) = sum_{m in split s} Xs[b, Ind[m], i] * Ys[m, j]
//
// A workgroup owns 32 TP (64, 96 or 128) rows of dW(e), columns of Xs, by BQ = 64 columns, or 128 by 128, and goes through the picks
// in slabs of 128 or 64, whose rows stay [pick][column] in LDS: direct 16-byte loads by row offsets from a table decoded from Ind
// beforehand, fragments by LDS transpose reads, NST - 1 slabs in flight, one barrier per slab.  The eight wavefronts are two halves of a
// slab's picks by a 2 x 2 grid of the tile; the halves' sums meet in LDS at the end, in that order.  Rows that do not exist get an
// offset outside the buffer descriptor and arrive as zeros.  Consecutive tiles of an expert share an XCD, and every XCD gets as many.
//
// What bounds it is the rows' way from the memory-side cache into the eight L2s, which the gather makes 88 MB long at B64 T256 E32 K32
// I768 J64: 18.9 us there, of which 4 before the first slab, with 256 workgroups of 96 columns; tiles of 32 columns, a wavefront-private
// stage each and the wavefronts' sums met in LDS took 28.4 us.  Wider tiles read less and fill fewer CUs, so the host picks the width by
// the rounds it makes (dw_strip_plan); 256 x 256 tiles with the picks split to fill the CUs took 24 us at B6 T1100 E20 K150 I328 J136,
// strips of 96 take 10.
//
// Preconditions (checked by the host): I % 8 == 0, J % 8 == 0, 16-byte aligned rows, operands below 2 GiB.
#pragma once
#include "egs_dw_dl.h"

namespace egs {

template <int TP, int BQ_> struct DwStrip {
    static constexpr int BP = 32 * TP, BQ = BQ_, SLAB = BQ == 64 ? 128 : 64;
    static constexpr int P_BYTES = SLAB * BP * 2, Q_BYTES = SLAB * BQ * 2, STAGE = P_BYTES + Q_BYTES;
    static constexpr int NST = STAGE <= 32 * 1024 ? 4 : 3;
    static constexpr int ROWS = STAGE > 40 * 1024 ? 1024 : 2048;    // picks whose offsets are in LDS at a time
    static constexpr int BYTES = NST * STAGE + 8 * ROWS;
    static_assert(BYTES <= 160 * 1024, "LDS of a CU");
};

template <class TT, int TP, int BQ>
__global__ __launch_bounds__(kDlThreads) void dw_strip_kernel(DwDlParams pp)
{
    static_assert(TT::ES == 2, "16-bit element types");
    typedef DwStrip<TP, BQ> L;
    constexpr int PL = L::P_BYTES / 8192, QL = L::Q_BYTES / 8192;       // loads per wavefront and slab (1 KB each)
    constexpr int NQ = BQ / 32, KH = L::SLAB / 64;          // 16-column tiles and 32-pick steps per wavefront
    constexpr int PCR = L::BP / 8, QCR = L::BQ / 8;         // 16-byte chunks per row
    extern __shared__ __attribute__((aligned(1024))) char smem_strip[];
    uint32_t *const x_voff = reinterpret_cast<uint32_t *>(smem_strip + L::NST * L::STAGE), *const y_voff = x_voff + L::ROWS;

    const DwParams &p = pp.d;
    const int per_e = p.i_tiles * p.j_tiles * p.S, lin = balanced_tile((int)blockIdx.x, p.E * per_e);
    if (lin < 0) return;
    const int e = lin / per_e, tile = lin - e * per_e, s = tile / (p.i_tiles * p.j_tiles), ij = tile - s * (p.i_tiles * p.j_tiles);
    const int i0 = ij / p.j_tiles * L::BP, j0 = ij % p.j_tiles * BQ;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = lane & 15, g = lane >> 4;
    const int Me = p.B * p.K;
    const int row_begin = s * p.rows_per_split, row_end = min(Me, row_begin + p.rows_per_split);
    const u32x4 rs_x = make_rsrc(p.Xs, pp.x_bytes), rs_y = make_rsrc(p.Ys, pp.y_bytes);

    // what a load's lanes fetch: row of the slab and byte offset of its column chunk, kVoffInvalid outside
    int p_row[PL], q_row[QL];
    uint32_t p_col[PL], q_col[QL];
#pragma unroll
    for (int jj = 0; jj < PL; ++jj) {
        const int at = (wave * PL + jj) * 64 + lane, row = at / PCR, pc = at - row * PCR;
        const int col = i0 + ((((pc >> 1) ^ tr_key<L::BP>(row)) << 1) | (pc & 1)) * 8;
        p_row[jj] = row;
        p_col[jj] = col < p.I ? (uint32_t)col * 2u : kVoffInvalid;
    }
#pragma unroll
    for (int jj = 0; jj < QL; ++jj) {
        const int at = (wave * QL + jj) * 64 + lane, row = at / QCR, pc = at - row * QCR;
        const int col = j0 + ((((pc >> 1) ^ tr_key<BQ>(row)) << 1) | (pc & 1)) * 8;
        q_row[jj] = row;
        q_col[jj] = col < p.J ? (uint32_t)col * 2u : kVoffInvalid;
    }
    auto issue = [&](int slab, int stage) {
        char *base = smem_strip + stage * L::STAGE;
#pragma unroll
        for (int jj = 0; jj < PL; ++jj) {
            const uint32_t ro = x_voff[slab * L::SLAB + p_row[jj]];
            direct_load16(rs_x, (ro == kVoffInvalid || p_col[jj] == kVoffInvalid) ? kVoffInvalid : ro + p_col[jj], 0, base + (wave * PL + jj) * 1024);
        }
#pragma unroll
        for (int jj = 0; jj < QL; ++jj) {
            const uint32_t ro = y_voff[slab * L::SLAB + q_row[jj]];
            direct_load16(rs_y, (ro == kVoffInvalid || q_col[jj] == kVoffInvalid) ? kVoffInvalid : ro + q_col[jj], 0, base + L::P_BYTES + (wave * QL + jj) * 1024);
        }
    };

    // fragment addresses: a lane supplies row 32 ks + 8 g + 4 h + a/4 and four columns 4 (a%4) of a 16-column tile, and receives column a
    // of rows 8 g + 4 h .. + 3.  Keys repeat every 32 rows, so a step adds a constant.
    const int half = wave >> 2, wi = (wave >> 1) & 1, wj = wave & 1;
    int p_at[2][TP], q_at[2][NQ];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = half * (L::SLAB / 2) + g * 8 + h * 4 + (a >> 2);
#pragma unroll
        for (int x = 0; x < TP; ++x) p_at[h][x] = row * (L::BP * 2) + (((wi * TP + x) ^ tr_key<L::BP>(row)) << 5) + (a & 3) * 8;
#pragma unroll
        for (int y = 0; y < NQ; ++y) q_at[h][y] = L::P_BYTES + row * (L::BQ * 2) + (((wj * NQ + y) ^ tr_key<BQ>(row)) << 5) + (a & 3) * 8;
    }
    f32x4 acc[TP][NQ];
#pragma unroll
    for (int x = 0; x < TP; ++x)
#pragma unroll
        for (int y = 0; y < NQ; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int stage) {
        const char *st = smem_strip + stage * L::STAGE;
#pragma unroll
        for (int k = 0; k < KH; ++k) {
            u32x4 pf[TP], qf[NQ];
#pragma unroll
            for (int x = 0; x < TP; ++x) {
                const u32x2 lo = lds_read_tr16(st + p_at[0][x] + k * 32 * L::BP * 2), hi = lds_read_tr16(st + p_at[1][x] + k * 32 * L::BP * 2);
                pf[x] = u32x4{lo[0], lo[1], hi[0], hi[1]};
            }
#pragma unroll
            for (int y = 0; y < NQ; ++y) {
                const u32x2 lo = lds_read_tr16(st + q_at[0][y] + k * 32 * L::BQ * 2), hi = lds_read_tr16(st + q_at[1][y] + k * 32 * L::BQ * 2);
                qf[y] = u32x4{lo[0], lo[1], hi[0], hi[1]};
            }
#pragma unroll
            for (int x = 0; x < TP; ++x)
#pragma unroll
                for (int y = 0; y < NQ; ++y) mma_chunk<TT>(acc[x][y], qf[y], pf[x]);
        }
    };

    int stage = 0;
    for (int chunk0 = row_begin; chunk0 < row_end; chunk0 += L::ROWS) {
        const int rows = min(L::ROWS, row_end - chunk0), nsl = (rows + L::SLAB - 1) / L::SLAB;
        __syncthreads();            // the previous chunk's offsets and stages are no longer being read
        for (int r = tid; r < nsl * L::SLAB; r += kDlThreads) {
            uint32_t xo = kVoffInvalid, yo = kVoffInvalid;
            if (r < rows) {
                const int m = chunk0 + r, b = m / p.K;
                const int64_t pick = ((int64_t)b * p.E + e) * p.K + (m - b * p.K);
                const int32_t t = load_token(p.Ind, p.ind_dtype, pick, p.T);
                if (t >= 0) {
                    xo = (uint32_t)(((int64_t)b * p.ldx_b + (int64_t)t * p.ldx_t) * 2);
                    yo = (uint32_t)(pick * p.J * 2);
                }
            }
            x_voff[r] = xo;
            y_voff[r] = yo;
        }
        __syncthreads();
#pragma unroll
        for (int st = 0; st < L::NST - 1; ++st)
            if (st < nsl) issue(st, stage + st < L::NST ? stage + st : stage + st - L::NST);
        for (int sl = 0; sl < nsl; ++sl) {
            const int later = min(nsl - 1 - sl, L::NST - 2);        // slabs requested after this one
            if (L::NST >= 4 && later >= 2) wait_vmem<(L::NST >= 4 ? 2 : 0) * (PL + QL)>();
            else if (later >= 1) wait_vmem<PL + QL>();
            else wait_vmem<0>();
            __syncthreads();        // slab sl landed everywhere; the stage of slab sl - 1 is free
            if (sl + L::NST - 1 < nsl) issue(sl + L::NST - 1, stage + L::NST - 1 < L::NST ? stage + L::NST - 1 : stage - 1);
            multiply(stage);
            if (++stage == L::NST) stage = 0;
        }
    }

    // the second half's sums join the first's; each half then stores one half of the columns
    __syncthreads();
    f32x4 *const meet = reinterpret_cast<f32x4 *>(smem_strip) + (wave & 3) * (TP * NQ * 64) + lane;
#pragma unroll
    for (int x = 0; x < TP; ++x)
#pragma unroll
        for (int y = 0; y < NQ / 2; ++y) meet[(x * NQ + (half ^ 1) * (NQ / 2) + y) * 64] = half ? acc[x][y] : acc[x][NQ / 2 + y];
    __syncthreads();
#pragma unroll
    for (int y = 0; y < NQ / 2; ++y) {
        const int j = j0 + wj * (BQ / 2) + (half * (NQ / 2) + y) * 16 + g * 4;
        if (j >= p.J) break;            // J % 8 == 0: the four columns are all in or all out
#pragma unroll
        for (int x = 0; x < TP; ++x) {
            const f32x4 other = meet[(x * NQ + half * (NQ / 2) + y) * 64];
            f32x4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = half ? other[r] + acc[x][NQ / 2 + y][r] : acc[x][y][r] + other[r];
            const int i = i0 + wi * 16 * TP + x * 16 + a;
            if (i >= p.I) continue;
            const size_t at = p.dw_layout == 0 ? ((size_t)e * p.I + i) * p.J + j : ((size_t)e * p.J + j) * p.I + i;
            const size_t step = p.dw_layout == 0 ? 1 : (size_t)p.I;
            if (p.S > 1 || p.out_dtype == 0) {      // partial sums in the output's layout, or an fp32 output
                float *dst = (p.S > 1 ? p.part + (size_t)s * p.E * p.I * p.J : reinterpret_cast<float *>(p.dW)) + at;
                if (step == 1) *reinterpret_cast<f32x4 *>(dst) = v;
                else
#pragma unroll
                    for (int r = 0; r < 4; ++r) dst[r * step] = v[r];
            } else {
                const u32x2 w = p.out_dtype == 1 ? u32x2{pack2<ElemF16>(v[0], v[1]), pack2<ElemF16>(v[2], v[3])}
                                                 : u32x2{pack2<ElemBF16>(v[0], v[1]), pack2<ElemBF16>(v[2], v[3])};
                uint16_t *dst = reinterpret_cast<uint16_t *>(p.dW) + at;
                if (step == 1) *reinterpret_cast<u32x2 *>(dst) = w;
                else
#pragma unroll
                    for (int r = 0; r < 4; ++r) dst[r * step] = (uint16_t)(w[r >> 1] >> ((r & 1) * 16));
            }
        }
    }
}

}  // namespace egs
