// The fp32 weight gradient on the bf16 matrix instruction (egs_split.h says how).
#pragma once
#include "egs_split.h"
#include "egs_tiled.h"

namespace egs {

// ------------------------------------------------------------------------------ weight gradient
// LDS: three planes of 32 picks x 64 columns of both operands, 32-byte units XOR-swizzled by bits 1 and 3 of
// the pick so that the 16 row pieces of a transpose read fall two deep on every bank; byte offsets of the rows of TAB picks
struct SplitDwLds {
    static constexpr int T = 64, PL = 32 * T * 2, STAGE = 6 * PL;
    static constexpr int RS = T + 4;                                    // floats per row of the results
    static_assert(T * RS * 4 <= STAGE, "the results fit");
    static constexpr int TAB = 512, BYTES = STAGE + TAB * 8;
};

// tiled_dw_wide_kernel (egs_tiled.h) for fp32 with the picks split over workgroups where there are few tiles: a 64 x 64 tile of dW(e)
// per workgroup, wavefronts 2 x 2; slabs of 32 picks, fetched two ahead.  A slab's fragments go into registers as soon as it is in LDS;
// one barrier later the next slab is split and written under the matrix instructions of this one.
// What bounds it is instruction issue: per slab and wavefront 24 matrix instructions (384 cycles) and 126 vector instructions of two to
// four, 104 of which split (16 of them the factor: B53 T97 E29 K41 I111 J75 26.3 us without, 27.5 with, in a trace); hence buffer loads (a pick
// that does not exist needs no masks) and 32-bit offsets (with 64-bit ones and masks 70 vector instructions more, 151 us for 135 at the first of
// these).  us in a graph, the fp32 instruction / this: B30 T46 E73 K44 I384 J169 182 / 130, B53 T97 E29 K41 I111 J75 40.7 / 29.6, B16 T512
// E64 K64 I256 J128 61 / 42, B33 T1697 E37 K79 I64 J256 71 / 40.
// (The products rows x weights gain less, 1.05 to 1.18 times above 12000 slabs and lose below: not taken there.)
static __device__ __forceinline__ void tiled_dw_split_body(const TiledDwParams &p, const int block)
{
    typedef SplitDwLds L;
    constexpr int ES = 4, TI = L::T, TJ = L::T, XL = 16, NX = 32 * XL / kThreads;         // 16 chunks of four columns per pick
    extern __shared__ __attribute__((aligned(16))) char smem_split_dw[];
    u32x2 *tab = reinterpret_cast<u32x2 *>(smem_split_dw + L::STAGE);                     // [TAB] byte offsets of a pick's X and Y rows
    const int per_e = p.i_tiles * p.j_tiles * p.S;
    const int lin = balanced_tile(block, p.E * per_e);
    if (lin < 0) return;
    const int e = lin / per_e;
    int rest = lin - e * per_e;
    const int split = rest / (p.i_tiles * p.j_tiles);
    rest -= split * (p.i_tiles * p.j_tiles);
    const int i0 = (rest / p.j_tiles) * TI, j0 = (rest % p.j_tiles) * TJ;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = lane & 15, g = lane >> 4;
    const int wi0 = (wave >> 1) * 32, wj0 = (wave & 1) * 32;
    const int Me = p.B * p.K;
    const int lo = split * p.picks_per_split, hi = min(Me, lo + p.picks_per_split), nslabs = max(0, (hi - lo + 31) >> 5);
    const int xp = tid / XL, xc = tid % XL;
    const int x_last = (int)(p.x_bytes - 16), y_last = (int)(p.y_bytes - 16);
    const __amdgpu_buffer_rsrc_t rs_x = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(p.Xs), 0, (int)p.x_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rs_y = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(p.Ys), 0, (int)p.y_bytes, 0x00020000);

    auto pick_of = [&](int m, int &b) -> int64_t {
        b = m / p.K;
        return ((int64_t)b * p.E + e) * p.K + (m - b * p.K);
    };
    auto make_tab = [&](int s) {                                        // from slab s on (two slabs beyond the last are looked up)
        for (int at = tid; at < L::TAB && lo + s * 32 + at < hi + 96; at += kThreads) {
            const int m = lo + s * 32 + at;
            int b;
            const int64_t pick = pick_of(min(m, Me - 1), b);
            const int64_t t = decode_index_word(load_index_word(p.Ind, p.ind_dtype, pick), p.Ind, p.ind_dtype, pick);
            const bool ok = m < hi && t >= 0 && t < (int64_t)p.T;
            tab[at] = ok ? u32x2{(uint32_t)(((int64_t)b * p.ldx_b + t * p.ldx_t) * ES), (uint32_t)(pick * p.J * ES)} : u32x2{kVoffInvalid, kVoffInvalid};
        }
    };
    // Picks that do not exist have an offset outside the descriptors and arrive as zeros on both sides.  Columns past a row are the next
    // row's: they reach only results that are not stored.  A chunk that would pass the end of its operand is read early and shifted.
    u32x4 rx[2][NX], ry[2][NX];
    int shift_x[2][NX], shift_y[2][NX];
    const int xcol = (i0 + xc * 4) * ES, ycol = (j0 + xc * 4) * ES;
    auto issue = [&](int s, int q) {
        auto fetch = [&](__amdgpu_buffer_rsrc_t rsrc, int at, int last, int &shift) -> u32x4 {
            const int from = min(at, last);                             // (signed: what does not exist stays outside)
            shift = at - from;
            return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, from, 0, 0));
        };
        const u32x2 *row = tab + s % (L::TAB / 32) * 32;
#pragma unroll
        for (int h = 0; h < NX; ++h) {
            const u32x2 at = row[h * (kThreads / XL) + xp];
            rx[q][h] = fetch(rs_x, (int)(at[0] + (uint32_t)xcol), x_last, shift_x[q][h]);
            ry[q][h] = fetch(rs_y, (int)(at[1] + (uint32_t)ycol), y_last, shift_y[q][h]);
        }
    };
    auto at = [](int pick, int unit) -> int { return pick * 128 + ((unit ^ (((pick >> 1) & 1) | ((pick >> 2) & 2))) << 5); };
    auto put_chunk = [&](int q, int c) {                                // chunk c < 2 NX of this thread's
        auto one = [&](char *plane0, int r, const u32x4 &v) {
            u32x2 piece[3];
            split_chunk(v, piece);
#pragma unroll
            for (int x = 0; x < 3; ++x) *reinterpret_cast<u32x2 *>(plane0 + x * L::PL + at(r, xc >> 2) + (xc & 3) * 8) = piece[x];
        };
        if (c < NX) one(smem_split_dw, c * (kThreads / XL) + xp, rx[q][c]);
        else one(smem_split_dw + 3 * L::PL, (c - NX) * (kThreads / XL) + xp, ry[q][c - NX]);
    };
    auto settle = [&](int q) {
        if (!p.edges) return;
        int any = 0;
#pragma unroll
        for (int h = 0; h < NX; ++h) any |= shift_x[q][h] | shift_y[q][h];
        if (__any(any)) {
#pragma unroll
            for (int h = 0; h < NX; ++h) { rx[q][h] = shift_right_bytes(rx[q][h], min(shift_x[q][h], 15)); ry[q][h] = shift_right_bytes(ry[q][h], min(shift_y[q][h], 15)); }
        }
    };
    f32x4 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 xf[2][3], yf[2][3];
    auto read = [&]() {
        // transpose reads: lane (a, g) points at pick 8 g + 4 h + a / 4, columns 4 (a % 4) .. + 3
        auto frag = [&](const char *plane, int unit) -> u32x4 {
            const char *from = plane + at(g * 8 + (a >> 2), unit) + (a & 3) * 8;
            const u32x2 l = lds_read_tr16(from), h = lds_read_tr16(from + 4 * 128);
            return u32x4{l[0], l[1], h[0], h[1]};
        };
#pragma unroll
        for (int x = 0; x < 3; ++x)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                xf[i][x] = frag(smem_split_dw + x * L::PL, (wi0 >> 4) + i);
                yf[i][x] = frag(smem_split_dw + (3 + x) * L::PL, (wj0 >> 4) + i);
            }
    };
    // Piece by piece over all accumulators, the smallest first; `between(t)` is issued behind the matrix instructions of product t < 6.
    auto multiply = [&](auto between) {
#pragma unroll
        for (int t = 0; t < 6; ++t) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) mma_chunk<ElemBF16>(acc[x][y], yf[y][kSplitP[t]], xf[x][kSplitQ[t]]);
            between(t);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    if (nslabs > 0) {
        make_tab(0);
        __syncthreads();
        issue(0, 0);
        issue(1, 1);
        settle(0);
#pragma unroll
        for (int c = 0; c < 2 * NX; ++c) put_chunk(0, c);
        issue(2, 0);
    }
    for (int s0 = 0; s0 < nslabs; s0 += 2) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {                                   // (a last odd round's second slab is zeros)
            const int s = s0 + q;
            __syncthreads();
            read();
            __syncthreads();
            if ((s + 3) % (L::TAB / 32) == 0) { make_tab(s + 3); __syncthreads(); }
            settle(q ^ 1);
            multiply([&](int t) {
                if (t < 2 * NX) put_chunk(q ^ 1, t);                    // (past the last slab: zeros, which nobody reads)
                if (t == 5) issue(s + 3, q ^ 1);
            });
            if (s + 1 >= nslabs) break;
        }
    }

    // ---------------- not all finite: the wavefront's part again, by the fp32 instruction, straight from memory.  (Only what is stored
    // counts: columns past a row hold whatever follows it in memory.)
    float odd = 0.f;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) odd = not_finite(acc[x][y], i0 + wi0 + x * 16 + a < p.I ? p.J - (j0 + wj0 + y * 16 + g * 4) : 0, odd);
    f32x4 again[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) again[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (__any(odd != odd)) {
        // 32 picks at a time, their offsets looked up by a lane each, the next ones' while these multiply.  (B53 T97 E29 K41 I111 J75 with a
        // row of NaN: 55 us; four picks at a time, each with loads that wait for its own, 117; the fp32 instruction throughout 42.)
        auto look_up = [&](int m0, uint32_t &xo, uint32_t &yo) {
            int b;
            const int m = m0 + (lane & 31);
            const int64_t pick = pick_of(min(m, Me - 1), b);
            const int32_t t = load_token(p.Ind, p.ind_dtype, pick, p.T);
            const bool ok = m < hi && t >= 0;
            xo = ok ? (uint32_t)(((int64_t)b * p.ldx_b + (int64_t)t * p.ldx_t) * ES) : kVoffInvalid;
            yo = ok ? (uint32_t)(pick * p.J * ES) : kVoffInvalid;
        };
        uint32_t xo, yo;
        look_up(lo, xo, yo);
#pragma unroll 1
        for (int m0 = lo; m0 < hi; m0 += 32) {
            float xv[8][2], yv[8][2];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t xk = (uint32_t)__shfl((int)xo, k * 4 + g, kWave), yk = (uint32_t)__shfl((int)yo, k * 4 + g, kWave);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    xv[k][h] = bits_f32(__builtin_amdgcn_raw_buffer_load_b32(rs_x, (int)(xk + (uint32_t)(i0 + wi0 + h * 16 + a) * ES), 0, 0));
                    yv[k][h] = bits_f32(__builtin_amdgcn_raw_buffer_load_b32(rs_y, (int)(yk + (uint32_t)(j0 + wj0 + h * 16 + a) * ES), 0, 0));
                }
            }
            look_up(m0 + 32, xo, yo);
#pragma unroll
            for (int k = 0; k < 8; ++k)
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < 2; ++y) again[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(yv[k][y], xv[k][x], again[x][y], 0, 0, 0);
        }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) split_result(acc[x][y], again[x][y]);

    // ---------------- lane (a, g) holds rows i0 + wi0 + 16 x + a, columns j0 + wj0 + 16 y + 4 g .. + 3; through LDS, so that whole
    // row (or, [E,J,I], column) segments leave
    __syncthreads();
    float *red = reinterpret_cast<float *>(smem_split_dw);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) *reinterpret_cast<f32x4 *>(red + (wi0 + x * 16 + a) * L::RS + wj0 + y * 16 + g * 4) = acc[x][y];
    __syncthreads();
    const bool eji = p.eji != 0;
    const int out_dtype = p.S > 1 ? 0 : p.out_dtype;
    const int oes = out_dtype == 0 ? 4 : 2;
    const int64_t part = p.S > 1 ? (int64_t)split * p.E * p.I * p.J : 0;
    auto pack = [&](float x, float y) -> uint32_t { return out_dtype == 1 ? pack2<ElemF16>(x, y) : pack2<ElemBF16>(x, y); };
#pragma unroll 1
    for (int v = tid; v < TI * TJ / 4; v += kThreads) {
        int gi, gj;
        f32x4 r;
        if (eji) {
            const int il = (v & 15) * 4, jl = v >> 4;
            const float *from = red + il * L::RS + jl;
            gi = i0 + il; gj = j0 + jl;
            r = f32x4{from[0], from[L::RS], from[2 * L::RS], from[3 * L::RS]};
        } else {
            const int il = v >> 4, jl = (v & 15) * 4;
            gi = i0 + il; gj = j0 + jl;
            r = *reinterpret_cast<const f32x4 *>(red + il * L::RS + jl);
        }
        if (gi >= p.I || gj >= p.J) continue;
        const int live = min(4, eji ? p.I - gi : p.J - gj);
        char *dst = p.dW + (part + (eji ? ((int64_t)e * p.J + gj) * p.I + gi : ((int64_t)e * p.I + gi) * p.J + gj)) * oes;
        if (live == 4) {
            if (oes == 4) *reinterpret_cast<f32x4_any *>(dst) = r;
            else *reinterpret_cast<u32x2_any *>(dst) = u32x2{pack(r[0], r[1]), pack(r[2], r[3])};
        } else {
            for (int x = 0; x < live; ++x) {
                if (oes == 4) reinterpret_cast<float *>(dst)[x] = r[x];
                else reinterpret_cast<uint16_t *>(dst)[x] = (uint16_t)(pack(r[x], 0.f) & 0xffffu);
            }
        }
    }
}

static __global__ __launch_bounds__(kThreads, 3) void tiled_dw_split_kernel(TiledDwParams p) { tiled_dw_split_body(p, (int)blockIdx.x); }

// ------------------------------------------------------------------------------ product and weight gradient of a backward call in one launch
// dY or dX's product rows and the weight gradient do not depend on each other, and at most sizes that come here neither fills the device: each
// is a chain of round trips of 5 to 15 us with a launch of its own.  The workgroups with the longer chains come
// first (launch_tiled_pair); the bodies are those of the kernels alone (the same bits; the product's the loop, also for the short reductions that are
// written out where it is alone, and then sometimes faster apart: tiled_apart).  Against two launches with the kernels as they are, 393 scatter backward
// calls of random sizes take 0.73 of the time and 389 gather backward calls, sums and all, 0.84; none is more than 1.6 % slower.
// us in a graph, two launches / one: bf16 B3 T607 E7 K90 I768 J19 dY and dW 15.3 / 8.3, B4 T201 E17 K6 I352 J31 11.3 / 6.3, f32 B66 T52 E5 K5 I431 J27
// 19.3 / 10.8, f32 B30 T706 E66 K21 I866 J192 253 / 248.
enum TiledDwKind { TILED_DW, TILED_DW_WIDE, TILED_DW_SPLIT };
template <class TT, int TN, int KIND>
__global__ __launch_bounds__(kThreads, 3) void tiled_pair_kernel(TiledRowsParams r, TiledDwParams d, int first_blocks, int dw_first)
{
    const bool first = (int)blockIdx.x < first_blocks;
    const int block = (int)blockIdx.x - (first ? 0 : first_blocks);
    if (first != (dw_first != 0)) tiled_rows_body<TT, TT::ES, false, TN>(r, block);
    else if constexpr (KIND == TILED_DW_SPLIT) tiled_dw_split_body(d, block);
    else if constexpr (KIND == TILED_DW_WIDE) tiled_dw_wide_body<TT>(d, block);
    else tiled_dw_body<TT>(d, block);
}

}  // namespace egs
