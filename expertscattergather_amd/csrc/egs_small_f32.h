// Gather-GEMM for small experts in fp32: Y[b,e,k,:] = X[b, Ind[b,e,k], :] . W(e), reduction length 32/64/128, 16..64
// output columns (the reference's default shape in its own precision: B64 T256 E32 K32 I128 J64 fp32).
//
// The products go through the bf16 matrix instruction, three pieces per value (egs_split.h).  W(e) is split once per workgroup, into
// three LDS planes in operand order: a lane's eight weights of 32 reduction steps are 16 bytes, steps 4 g .. + 3 of the first
// sixteen and then of the second, as the rows' 16-byte chunks give them.  The gathered rows go global -> registers -> operand order
// (coalesced 64-byte runs per row, then the 4 x 16 lane transposition) and are split there.  One wavefront = 32 picks of one
// expert, a workgroup 256; one barrier (W(e) in place).  A wavefront multiplies and stores its 16-pick row tiles one after the
// other, the first tile's rows requested before the barrier and the others after it.
// us in a graph, three pieces / the fp32 instruction, which was the roof with 138 TFLOP/s: B64 T256 E32 K32 I128 J64 13.4 / 15.5 (the matrix
// instructions take 3, indices, rows and W(e) the rest), E60 21.7 / 26.7, I64 9.2 / 10.3, B160 J48 22.4 / 28.4, B8 T100 E16 9.4 / 11.5; level for
// 16 columns.  (The one-kernel scatter does not gain: it would split every weight once per batch element, 20.0 / 18.8.)
//
// Replaces the reference's expert_gather_kernel (egs/triton_kernels.py:49-143) on these shapes.
#pragma once
#include "egs_small.h"
#include "egs_split.h"

namespace egs {

// bytes of a column in a plane: 16 more than the weights take, so that the 16 lanes of a read spread over the banks
__host__ __device__ constexpr int rows_small_f32_column(int R) { return R * 2 + 16; }
__host__ __device__ constexpr size_t rows_small_f32_lds(int R, int N) { return (size_t)3 * N * rows_small_f32_column(R); }

// Requirements (checked by the launcher): fp32, R == 16 * KS in {32, 64, 128}, N == 16 * TN <= 64, rows of A, W and C
// 16-byte aligned, every tensor below 4 GiB.  W is [E,R,N] (W_NMAJOR) or [E,N,R].
// TQ = 16-pick row tiles per wavefront (4, or 2 with twice the wavefronts: a workgroup covers 256 picks either way)
template <bool W_NMAJOR, int KS, int TN, int TQ = 4>
__global__ __launch_bounds__(64 * (16 / TQ), 4) void rows_small_f32_kernel(SmallRowsParams p)
{
    constexpr int R = 16 * KS, N = 16 * TN, COL = rows_small_f32_column(R), PLANE = N * COL;
    constexpr int PW = 16 * TQ, NTHREADS = 64 * (256 / PW);     // picks per wavefront, threads per workgroup
    extern __shared__ __attribute__((aligned(16))) char w_lds[];       // [3][N][COL]
    int e, tile;
    int bid = (int)blockIdx.x;
    // routing-table build of a later scatter riding along (csr_blocks = B, or 0): one workgroup per batch element, first in line
    if (bid < p.csr_blocks) {
        if (p.csr_split)
            csr_count_half_body(reinterpret_cast<int32_t *>(w_lds), bid >> 1, bid & 1, (int)threadIdx.x, NTHREADS, p.Ind,
                                p.ind_dtype, p.T, p.E * p.K, p.seg_off, p.perm);
        else
            csr_count_body(reinterpret_cast<int32_t *>(w_lds), bid, bid, (int)threadIdx.x, NTHREADS, p.Ind, p.ind_dtype, p.T,
                           p.E * p.K, p.seg_off, p.perm, nullptr, nullptr);
        return;
    }
    bid -= p.csr_blocks;
    if (!decode_rows_block(bid, p.rows_share_xcd, p.tiles_per_e, p.E, e, tile)) return;       // uniform per workgroup
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = lane & 15, g = lane >> 4;
    const int Me = p.B * p.K;
    const int m0 = (tile * (256 / PW) + wave) * PW;
    const bool live_wave = m0 < Me;

    // the index load goes first: the chain index -> row is the long one (lanes beyond the wavefront's picks repeat them
    // and own nothing)
    const int m_lane = m0 + lane % PW;
    const int mm_lane = min(m_lane, Me - 1);
    const int b_lane = mm_lane / p.K;
    const int64_t pick = ((int64_t)b_lane * p.E + e) * p.K + (mm_lane - b_lane * p.K);
    // (no branch around any load of the prologue, also where a wavefront has no picks left - its clamped addresses are valid:
    // behind a branch the compiler loses track of the order of the outstanding loads and makes the first matrix instruction
    // wait for all of them, the rows of the last slab included)
    const uint64_t t_word = load_index_word(p.Ind, p.ind_dtype, pick);

    // W(e) -> registers (all loads in flight behind the index load), LDS as [column][reduction] further down
    const char *We = p.W + (size_t)e * R * N * 4;
    constexpr int W_CHUNKS = R * N / 4, W_UNITS = KS / 2 * TN, NWAVES = NTHREADS / 64;
    constexpr int W_IT = W_NMAJOR ? 2 * ((W_UNITS + NWAVES - 1) / NWAVES) : (W_CHUNKS + NTHREADS - 1) / NTHREADS;
    // Which 16-byte chunk a thread takes.  [N][R]: consecutive threads, consecutive chunks.  [R][N]: a wavefront takes 32 reduction
    // rows x 16 columns per two loads, lanes 4 q .. 4 q + 3 the four chunks of rows 2 q and 2 q + 1, whose pieces go to LDS in pairs;
    // the 64 pairs of one write (columns 16 apart in steps of 4 lanes) fall on 64 different banks.
    auto w_chunk = [&](int i) -> int {
        if constexpr (!W_NMAJOR) {
            const int c = tid + i * NTHREADS;
            return c < W_CHUNKS ? c : -1;
        } else {
            const int u = wave + (i >> 1) * NWAVES;                         // (32-row block, 16-column group) of these two loads
            if (W_UNITS % NWAVES != 0 && u >= W_UNITS) return -1;
            return ((u / TN) * 32 + (lane >> 2) * 2 + (i & 1)) * (N / 4) + (u % TN) * 4 + (lane & 3);
        }
    };
    u32x4 wv[W_IT];
#pragma unroll
    for (int i = 0; i < W_IT; ++i) {
        const int c = w_chunk(i);
        wv[i] = *reinterpret_cast<const u32x4 *>(We + (size_t)max(c, 0) * 16);
    }

    const int64_t t_raw = decode_index_word(t_word, p.Ind, p.ind_dtype, pick);
    const int32_t t = (t_raw < 0 || t_raw >= (int64_t)p.T) ? -1 : (int32_t)t_raw;
    const uint32_t aoff = t >= 0 ? (uint32_t)(((int64_t)b_lane * p.lda_b + (int64_t)t * p.lda_t) * 4) : 0u;
    const uint32_t coff = (uint32_t)(pick * N * 4);
    const int state = (m_lane < Me && lane < PW) ? (t >= 0 ? 1 : 2) : 0;  // 0: nothing to store, 1: store the product, 2: store zeros (bad index)
    // gathered rows: lanes 4r .. 4r+3 fetch the four 16-byte chunks of a 16-deep slab of row 16 tq + r
    uint32_t xo[TQ];
#pragma unroll
    for (int tq = 0; tq < TQ; ++tq) xo[tq] = (uint32_t)__shfl((int)aoff, tq * 16 + (lane >> 2), kWave) + (uint32_t)((lane & 3) * 16);
    // every 16-deep slab of every row tile goes in flight now, the first row tile's first
    // The first row tile's slabs are requested now, the others after the barrier: a CU's eight wavefronts push 160 KB
    // through its one address path in this prologue (2560 cycles at 64 bytes a cycle), a wavefront cannot go on to
    // its LDS writes before its requests are accepted, and the barrier waits for the last of them - with every slab
    // requested here the first matrix instruction started 4700 cycles after the indices had arrived.
    u32x4 xr[TQ][KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) xr[0][s] = *reinterpret_cast<const u32x4 *>(p.A + xo[0] + s * 64);
    __builtin_amdgcn_sched_barrier(0);
    // reduction step k of a column: 32-step block, its lane group, which of its two sixteens
    auto w_at = [](int n, int k) -> int { return n * COL + (k >> 5) * 64 + ((k >> 2) & 3) * 16 + ((k >> 4) & 1) * 8 + (k & 3) * 2; };
#pragma unroll
    for (int i = 0; i < W_IT; i += W_NMAJOR ? 2 : 1) {
        const int c = w_chunk(i);
        if (c < 0) continue;
        if constexpr (!W_NMAJOR) {
            const int n = c / (R / 4), k4 = c - n * (R / 4);
            u32x2 piece[3];
            split_chunk(wv[i], piece);
#pragma unroll
            for (int x = 0; x < 3; ++x) *reinterpret_cast<u32x2 *>(w_lds + x * PLANE + w_at(n, 4 * k4)) = piece[x];
        } else {
            const int r = c / (N / 4), n4 = c - r * (N / 4);                // an even row and the next, four columns
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                uint32_t piece[3];
                split_pair(bits_f32(wv[i][y]), bits_f32(wv[i + 1][y]), piece);
#pragma unroll
                for (int x = 0; x < 3; ++x) *reinterpret_cast<uint32_t *>(w_lds + x * PLANE + w_at(4 * n4 + y, r)) = piece[x];
            }
        }
    }
    __syncthreads();                    // W(e) is in place
    if (!live_wave) return;
#pragma unroll
    for (int tq = 1; tq < TQ; ++tq)
#pragma unroll
        for (int s = 0; s < KS; ++s) xr[tq][s] = *reinterpret_cast<const u32x4 *>(p.A + xo[tq] + s * 64);
    __builtin_amdgcn_sched_barrier(0);

    // Row tiles are multiplied and stored one after the other (TG = 1), so that the stores of one run under the matrix
    // instructions of the next instead of all at the kernel's end - as long as a tile alone keeps four accumulators
    // busy (consecutive matrix instructions on one accumulator would wait for each other); narrower outputs take the
    // row tiles of the wavefront together (TG = TQ).
    constexpr int TG = TN >= 3 ? 1 : TQ;
#pragma unroll
    for (int t0 = 0; t0 < TQ; t0 += TG) {
        f32x4 acc[TG][TN];
#pragma unroll
        for (int t = 0; t < TG; ++t)
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) acc[t][tn] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; s += 2) {
            u32x4 xf[TG][3];
#pragma unroll
            for (int t = 0; t < TG; ++t) {
                u32x2 lo[3], hi[3];
                split_chunk(lanes_4a_g_to_16g_a(xr[t0 + t][s], lane), lo);
                split_chunk(lanes_4a_g_to_16g_a(xr[t0 + t][s + 1], lane), hi);
#pragma unroll
                for (int x = 0; x < 3; ++x) xf[t][x] = u32x4{lo[x][0], lo[x][1], hi[x][0], hi[x][1]};
            }
            u32x4 wf[TN][3];
#pragma unroll
            for (int x = 0; x < 3; ++x)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
                    wf[tn][x] = *reinterpret_cast<const u32x4 *>(w_lds + x * PLANE + (tn * 16 + a) * COL + s * 32 + g * 16);
            // piece by piece over all accumulators: consecutive matrix instructions then go to different ones
#pragma unroll
            for (int c = 0; c < 6; ++c)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                    for (int t = 0; t < TG; ++t) mma_chunk<ElemBF16>(acc[t][tn], wf[tn][kSplitP[c]], xf[t][kSplitQ[c]]);
        }
        // not all finite: these row tiles again, by the fp32 instruction, weights straight from memory.  (Only what is stored counts:
        // a pick that does not exist multiplied some row or other.)
        float odd = 0.f;
#pragma unroll
        for (int t = 0; t < TG; ++t) {
            float one = 0.f;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) one = not_finite(acc[t][tn], 4, one);
            if (__shfl(state, (t0 + t) * 16 + a, kWave) == 1) odd += one;
        }
        if (__any(odd != odd)) {
            f32x4 again[TG][TN];
#pragma unroll
            for (int t = 0; t < TG; ++t)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) again[t][tn] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KS; ++s)
#pragma unroll
                for (int t = 0; t < TG; ++t) {
                    const u32x4 x = lanes_4a_g_to_16g_a(xr[t0 + t][s], lane);
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int k = s * 16 + g * 4 + c;
#pragma unroll
                        for (int tn = 0; tn < TN; ++tn) {
                            const int n = tn * 16 + a;
                            const float w = *reinterpret_cast<const float *>(We + (uint32_t)((W_NMAJOR ? k * N + n : n * R + k) * 4));
                            again[t][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, bits_f32(x[c]), again[t][tn], 0, 0, 0);
                        }
                    }
                }
#pragma unroll
            for (int t = 0; t < TG; ++t)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn) split_result(acc[t][tn], again[t][tn]);
        } else {
#pragma unroll
            for (int t = 0; t < TG; ++t)
#pragma unroll
                for (int tn = 0; tn < TN; ++tn)
#pragma unroll
                    for (int x = 0; x < 4; ++x) acc[t][tn][x] *= kSplitUnscale;
        }
        // lane (a, g) holds, for pick 16 tq + a, columns 16 tn + 4 g .. + 3: the four lanes g of a pick write 64 contiguous bytes
#pragma unroll
        for (int t = 0; t < TG; ++t) {
            const int tq = t0 + t;
            const int st = __shfl(state, tq * 16 + a, kWave);
            const uint32_t co = (uint32_t)__shfl((int)coff, tq * 16 + a, kWave);
            if (st == 0) continue;
#pragma unroll
            for (int tn = 0; tn < TN; ++tn) {
                const f32x4 v = st == 2 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[t][tn];
                *reinterpret_cast<f32x4 *>(p.C + co + (tn * 16 + g * 4) * 4) = v;
            }
        }
    }
}

}  // namespace egs
