// Tiled rows x weight products and weight gradients for operands of ANY size and alignment: odd row lengths, views that
// start anywhere, few picks, few experts.  The specialised kernels (egs_small*.h, egs_rows_gemm_dl.h, egs_rows_gemm.h,
// egs_dw_tile.h, egs_dw_dl.h) take the shapes they are made for; everything else runs here.
//
// What such calls are bound by is not arithmetic but the chain  index -> row -> LDS -> matrix instruction  and the number of
// workgroups: a 95 x 65 expert with 74 picks is one 128 x 128 tile, and the kernel this replaces walked its three 32-deep
// slabs one memory round trip after the other, reading rows that do not start on 16 bytes element by element.  Hence:
//   * every operand is read 16 bytes at a time wherever a row starts (global memory takes any alignment); the one chunk per
//     tensor that would reach past its end is read a little earlier and shifted, row tails are masked in the last slab;
//   * two slabs are in flight in registers and the LDS tile is double-buffered: one barrier per slab;
//   * tiles are 64 rows x 32 .. 96 columns, so that a ragged width wastes little and a small problem still has
//     many workgroups; workgroups are dealt to the XCDs evenly for any number of experts.
#pragma once
#include <type_traits>

#include "egs_device.h"

namespace egs {

typedef u32x4 u32x4_any __attribute__((aligned(1)));        // 16 bytes at any address (global memory)
typedef u32x2 u32x2_any __attribute__((aligned(1)));
typedef f32x4 f32x4_any __attribute__((aligned(1)));

// 128-bit logical right shift by 8 * bytes, 0 <= bytes < 16
__device__ __forceinline__ u32x4 shift_right_bytes(const u32x4 &v, int bytes)
{
    uint64_t lo = (uint64_t)v[0] | ((uint64_t)v[1] << 32), hi = (uint64_t)v[2] | ((uint64_t)v[3] << 32);
    if (bytes >= 8) { lo = hi; hi = 0; }
    const int s = 8 * (bytes & 7);
    if (s != 0) { lo = (lo >> s) | (hi << (64 - s)); hi >>= s; }
    return u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// Workgroup -> linear tile number: XCD x (workgroups are dealt to the eight XCDs in turn) takes the x-th eighth of `total`
// consecutive tiles, so neighbours in the numbering share an L2 and no XCD gets more than one tile more than another.
__device__ __forceinline__ int balanced_tile(int bid, int total)
{
    const int per = (total + 7) >> 3;
    const int t = (bid & 7) * per + (bid >> 3);
    return (bid >> 3) < per && t < total ? t : -1;
}

struct TiledRowsParams {
    const char *A;              // gather: [B,T,R] source; else dense [B,E,K,R] rows
    const char *W;              // [E,R,N] (W_TRANS) or [E,N,R]
    const void *Ind;            // gather only
    char *C;                    // [B,E,K,ldc] rows, element type or fp32
    const float *w_scale;       // [E,N] or nullptr
    const char *bias;           // [E,N] in the element type, or nullptr
    int64_t a_bytes, w_bytes;   // extents of A and W; tiled_rows_kernel: A and an expert's matrix are at least 16 bytes
    int64_t lda_b, lda_t;       // element strides of the source (gather)
    int32_t B, T, E, K, R, N, ldc;
    int32_t ind_dtype, gather, out_f32;
    int32_t m_tiles, n_tiles;
    int32_t act;                // Activation of the results (16-bit types)
    int32_t rows_major;         // numbering of the tiles: 1 = row tiles outermost (their source rows share an L2), 0 = experts outermost
};

// bytes of LDS: two stages of A and W tiles, or one
template <class TT, bool W_TRANS, int TN>
struct TiledLds {
    static constexpr int CH = 8, BKE = CH * TT::VEC;            // 128-byte row pieces per slab
    static constexpr int A = 64 * CH * 16;
    // [reduction][column] weight tiles.  16-bit: an odd number of 32-byte units per row and 128 more bytes every eight rows, so
    // that the 16 row pieces of a transpose read fall two deep on every bank; fp32: rows 4 banks apart modulo 16
    static constexpr int WROW = TT::ES == 2 ? 32 * (TN | 1) : (16 * TN + 4) * 4;
    static constexpr int W = W_TRANS ? (TT::ES == 2 ? BKE * WROW + (BKE / 8) * 128 : BKE * WROW) : 16 * TN * CH * 16;
    static constexpr int STAGE = A + W;
    static constexpr int BYTES = 2 * STAGE;
    static constexpr int RESULTS = 64 * (16 * TN + 4) * 4, ONE_STAGE = STAGE > RESULTS ? STAGE : RESULTS;
};

// 64 rows x 16 * TN columns per workgroup of four wavefronts, each 16 rows x all columns, two slabs in flight in registers.  What
// hides one workgroup's round trips is the others of its compute unit, so the registers are bounded for three or four.
// (128-row tiles of this kernel were level or slower at all of 42 small and ragged shapes but where they left fewer columns over;
// large 16-bit products are another matter, see rows_gemm_kernel.  Four slabs in flight gave 4% at R1000 and a few tiles, and cost
// occupancy elsewhere.)
// SLABS: how many, where they are few (at most four), or 0.  So short a reduction is a chain of round trips whatever is in flight under it, and the number of
// workgroups that a CU holds is what hides it: with the slabs written out there is nothing to request twice (the loop's requests past the end), one
// stage of LDS does (a barrier more for each slab), and 30 to 58, 48 to 96, 62 to 124 registers are enough for one, two, and three or four slabs instead of
// 76 to 156.  Products alone, us, loop / written out: f16 B70 T302 E52 K143 I32 J93 56 / 37, bf16 B114 T627 E44 K33 I64 J167 42 / 30, f32 B13 T243 E104
// K48 I49 J224 40 / 34, bf16 B81 T155 E72 K82 I192 J35 54 / 45; of 2200 with their sums 10 are more than 3 % slower.  The loop in one stage had to
// spill (73 -> 248 us at worst).
// The parameters: by value where the compiler then keeps a second slab's loads ahead (fp8 weights, 32 columns, the loop: 114 registers; by
// reference 92, and 1.014 of the time over 84 sizes, 9 of them more than 3 % slower), else by reference (by value 158 registers and not 126 with
// 96 columns).
template <int WES, int TN, int SLABS>
using TiledRowsBy = typename std::conditional<WES == 1 && TN == 2 && SLABS == 0, const TiledRowsParams, const TiledRowsParams &>::type;
template <class TT, int WES, bool W_TRANS, int TN, int SLABS = 0>
__device__ __forceinline__ void tiled_rows_body(TiledRowsBy<WES, TN, SLABS> p, const int block)
{
    constexpr int ES = TT::ES, VEC = TT::VEC;
    constexpr bool W_FP8 = WES == 1;
    typedef TiledLds<TT, W_TRANS, TN> L;
    constexpr int CH = L::CH, BKE = L::BKE, KSTEPS = CH / 4;
    constexpr int BM = 64, BN = 16 * TN;
    constexpr int NA = BM * CH / kThreads;                              // A chunks per thread and slab
    // W chunks (16 source bytes) per slab: W_TRANS rows of BN columns, else BN rows of CH chunks (fp8: half as many)
    constexpr int WPR = W_TRANS ? BN * WES / 16 : CH * WES / ES;        // chunks per source row
    constexpr int WCH = WPR * (W_TRANS ? BKE : BN);
    constexpr int NW = (WCH + kThreads - 1) / kThreads;
    constexpr int D = SLABS == 1 ? 1 : 2;                                      // slabs in flight in registers
    extern __shared__ __attribute__((aligned(16))) char smem_tiled[];

    const int total = p.E * p.m_tiles * p.n_tiles;
    const int lin = balanced_tile(block, total);
    if (lin < 0) return;
    int e, mt, nt;
    if (p.rows_major) { mt = lin / (p.E * p.n_tiles); const int r = lin - mt * p.E * p.n_tiles; e = r / p.n_tiles; nt = r - e * p.n_tiles; }
    else { e = lin / (p.m_tiles * p.n_tiles); const int r = lin - e * p.m_tiles * p.n_tiles; mt = r / p.n_tiles; nt = r - mt * p.n_tiles; }
    const int m0 = mt * BM, n0 = nt * BN;
    const int tid = (int)threadIdx.x;
    const int R = p.R, N = p.N, Me = p.B * p.K;
    const int nk = (R + BKE - 1) / BKE;

    // ---------------- this thread's rows of A (chunk tid % CH of rows tid / CH + i * (256 / CH)); the index words travel first
    const int ac = tid % CH;
    int64_t apick[NA];
    uint64_t iw[NA];
    int ab[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int m = min(m0 + tid / CH + i * (kThreads / CH), Me - 1);
        ab[i] = m / p.K;
        apick[i] = ((int64_t)ab[i] * p.E + e) * p.K + (m - ab[i] * p.K);
        iw[i] = 0;
    }
    if (p.gather) {
#pragma unroll
        for (int i = 0; i < NA; ++i) iw[i] = load_index_word(p.Ind, p.ind_dtype, apick[i]);
    }

    // ---------------- weight side: byte offsets from the expert's matrix.  A chunk may lie past the reduction length, past the last
    // column or past the matrix: those values are cleared, never stored, or read early (`w_last`: the last 16 bytes of W, which do
    // not start before this expert's matrix, see launch_tiled)
    const char *We = p.W + (int64_t)e * R * N * WES;
    const int64_t to_end = p.w_bytes - 16 - (int64_t)e * R * N * WES;
    const uint32_t w_last = to_end > 0xffffff00ll ? 0xffffff00u : (uint32_t)to_end;
    const uint32_t w_step = (uint32_t)BKE * (W_TRANS ? (uint32_t)N : 1u) * WES;
    uint32_t woff[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int v = min(tid + i * kThreads, WCH - 1);
        if constexpr (W_TRANS) woff[i] = ((uint32_t)(v / WPR) * (uint32_t)N + (uint32_t)n0) * WES + (uint32_t)(v % WPR) * 16u;
        else woff[i] = (uint32_t)min(n0 + v / WPR, N - 1) * (uint32_t)R * WES + (uint32_t)(v % WPR) * 16u;
    }
    u32x4 wreg[D][NW];
    auto issue_w = [&](int kt, u32x4 (&set)[NW]) {
#pragma unroll
        for (int i = 0; i < NW; ++i) set[i] = *reinterpret_cast<const u32x4_any *>(We + min(woff[i] + (uint32_t)kt * w_step, w_last));
    };
    int64_t arow[NA];           // byte offsets (always from p.A: the compiler then knows the loads are global ones)
    int alive = 0;
    const int64_t a_last = p.a_bytes - 16;
    u32x4 areg[D][NA];
    auto issue_a = [&](int kt, u32x4 (&set)[NA]) {
#pragma unroll
        for (int i = 0; i < NA; ++i) set[i] = *reinterpret_cast<const u32x4_any *>(p.A + min(arow[i] + kt * (CH * 16), a_last));
    };

    // slabs beyond the last are requested as the last one again: no load is conditional, so that the compiler can count the
    // outstanding ones and waits for one slab's only
#pragma unroll
    for (int d = 0; d < D; ++d) issue_w(min(d, nk - 1), wreg[d]);
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int m = m0 + tid / CH + i * (kThreads / CH);
        if (p.gather) {
            const int64_t t = decode_index_word(iw[i], p.Ind, p.ind_dtype, apick[i]);
            const bool ok = m < Me && t >= 0 && t < (int64_t)p.T;
            arow[i] = (ok ? ((int64_t)ab[i] * p.lda_b + t * p.lda_t) * ES : 0) + ac * 16;
            alive |= (int)ok << i;
        } else {
            arow[i] = apick[i] * R * ES + ac * 16;
            alive |= (int)(m < Me) << i;
        }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) issue_a(min(d, nk - 1), areg[d]);

    // ---------------- registers -> LDS.  `edge` (the last slab, and every slab of a matrix whose rows are shorter than a chunk):
    // chunks that were read early are shifted into place and what lies past the reduction length is cleared on both sides
    const bool short_rows = W_TRANS && (int64_t)N * WES < 16;
    auto w_off = [&](int r, int col_bytes) -> int {                     // byte offset in a [reduction][column] tile
        return ES == 2 ? r * L::WROW + (r >> 3) * 128 + col_bytes : r * L::WROW + col_bytes;
    };
    auto clear_past = [](u32x4 &v, int left) {                          // keeps the first `left` bytes
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const int nb = left - 4 * x;
            v[x] &= nb >= 4 ? 0xffffffffu : nb <= 0 ? 0u : 0xffffffffu >> (32 - 8 * nb);
        }
    };
    auto fix_edge = [&](u32x4 (&av)[NA], u32x4 (&wv)[NW], int kt) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int64_t past = arow[i] + kt * (CH * 16) - a_last;
            if (past > 0) av[i] = shift_right_bytes(av[i], (int)min(past, (int64_t)15));
            clear_past(av[i], R * ES - kt * (CH * 16) - ac * 16);
        }
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int v = min(tid + i * kThreads, WCH - 1);
            const uint32_t off = woff[i] + (uint32_t)kt * w_step;
            if (off > w_last) wv[i] = shift_right_bytes(wv[i], (int)min(off - w_last, 15u));
            if constexpr (W_TRANS) { if (kt * BKE + v / WPR >= R) wv[i] = u32x4{0u, 0u, 0u, 0u}; }
            else clear_past(wv[i], (R - kt * BKE) * WES - (v % WPR) * 16);
        }
    };
    auto commit = [&](u32x4 (&av)[NA], u32x4 (&wv)[NW], char *stage) {
        u32x4 *ta = reinterpret_cast<u32x4 *>(stage);
        char *tw = stage + L::A;
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const uint32_t keep = (alive >> i) & 1 ? 0xffffffffu : 0u;
            ta[tile_chunk_index<CH>(tid / CH + i * (kThreads / CH), ac)] = u32x4{av[i][0] & keep, av[i][1] & keep, av[i][2] & keep, av[i][3] & keep};
        }
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int v = tid + i * kThreads;
            if (WCH % kThreads != 0 && v >= WCH) continue;
            const u32x4 w = wv[i];
            const int r = v / WPR, c = v % WPR;
            if constexpr (W_TRANS && W_FP8) {
                *reinterpret_cast<u32x4 *>(tw + w_off(r, c * 32)) = fp8x8_to_bf16_chunk(w[0], w[1]);
                *reinterpret_cast<u32x4 *>(tw + w_off(r, c * 32) + 16) = fp8x8_to_bf16_chunk(w[2], w[3]);
            } else if constexpr (W_TRANS) {
                *reinterpret_cast<u32x4 *>(tw + w_off(r, c * 16)) = w;
            } else if constexpr (W_FP8) {
                reinterpret_cast<u32x4 *>(tw)[tile_chunk_index<CH>(r, 2 * c)] = fp8x8_to_bf16_chunk(w[0], w[1]);
                reinterpret_cast<u32x4 *>(tw)[tile_chunk_index<CH>(r, 2 * c + 1)] = fp8x8_to_bf16_chunk(w[2], w[3]);
            } else {
                reinterpret_cast<u32x4 *>(tw)[tile_chunk_index<CH>(r, c)] = w;
            }
        }
    };

    // ---------------- LDS -> matrix instructions
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = lane & 15, g = lane >> 4;
    const int wave_m0 = wave * 16;
    f32x4 acc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const char *stage, int left) {                   // `left`: reduction elements from this slab on
        const u32x4 *ta = reinterpret_cast<const u32x4 *>(stage);
        const char *tw = stage + L::A;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) {
            if (ks > 0 && ks * 4 * VEC >= left) break;
            const u32x4 mf = ta[tile_chunk_index<CH>(wave_m0 + a, ks * 4 + g)];
            u32x4 nf[TN];
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (!W_TRANS) {
                    nf[j] = reinterpret_cast<const u32x4 *>(tw)[tile_chunk_index<CH>(j * 16 + a, ks * 4 + g)];
                } else if constexpr (ES == 2) {
                    // transpose reads: lane (a, g) points at reduction row 32 ks + 8 g + 4 h + a / 4, columns 4 (a % 4) .. + 3
                    const char *at = tw + w_off(ks * 32 + g * 8 + (a >> 2), j * 32 + (a & 3) * 8);
                    const u32x2 lo = lds_read_tr16(at), hi = lds_read_tr16(at + 4 * L::WROW);
                    nf[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                } else {
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        nf[j][c] = *reinterpret_cast<const uint32_t *>(tw + w_off(ks * 16 + g * 4 + c, (j * 16 + a) * 4));
                }
            }
            if constexpr (ES == 2) {
#pragma unroll
                for (int j = 0; j < TN; ++j) mma_chunk<TT>(acc[j], nf[j], mf);
            } else {            // accumulators in turn: an fp32 matrix instruction then never waits for the one before it
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(bits_f32(nf[j][c]), bits_f32(mf[c]), acc[j], 0, 0, 0);
            }
        }
    };
    // One barrier per slab: a wavefront that writes slab kt + 1 has passed slab kt's barrier, before which every wavefront had
    // finished with slab kt - 1, the stage's previous content.  The rounds before the last request and consume without a condition,
    // so that the compiler can count the outstanding loads and waits for one slab's only; the last round requests nothing more.
    if constexpr (SLABS > 0) {
#pragma unroll
        for (int d = 0; d < SLABS; ++d) {
            constexpr int last = SLABS - 1;
            if (d > 0) __syncthreads();
            if (d == last || short_rows) fix_edge(areg[d % D], wreg[d % D], d);
            commit(areg[d % D], wreg[d % D], smem_tiled);
            if (d + D <= last) {
                issue_a(d + D, areg[d % D]);
                issue_w(d + D, wreg[d % D]);
            }
            __syncthreads();
            compute(smem_tiled, d < last ? BKE : R - d * BKE);
        }
    } else {
        static_assert(D % 2 == 0, "stage parity is static");
        int kt = 0;
        for (; kt + D < nk && !short_rows; kt += D) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                char *stage = smem_tiled + (d & 1) * L::STAGE;
                commit(areg[d], wreg[d], stage);
                issue_a(min(kt + d + D, nk - 1), areg[d]);
                issue_w(min(kt + d + D, nk - 1), wreg[d]);
                __syncthreads();
                compute(stage, BKE);
            }
        }
        for (;;) {
#pragma unroll
            for (int d = 0; d < D; ++d) {
                if (kt + d >= nk) break;
                char *stage = smem_tiled + (d & 1) * L::STAGE;
                if (kt + d == nk - 1 || short_rows) fix_edge(areg[d], wreg[d], kt + d);
                commit(areg[d], wreg[d], stage);
                __syncthreads();
                compute(stage, R - (kt + d) * BKE);
            }
            kt += D;
            if (kt >= nk) break;                                            // `short_rows` alone goes on: every slab is an edge
#pragma unroll
            for (int d = 0; d < D; ++d) {
                issue_a(min(kt + d, nk - 1), areg[d]);
                issue_w(min(kt + d, nk - 1), wreg[d]);
            }
        }
    }

    // ---------------- results.  Lane (a, g) holds columns 16 j + 4 g .. + 3 of row a of the wavefront's; they go through a piece of
    // LDS of its own and leave as whole row segments.  One short loop does everything else to a value: unrolled over the tile, the
    // activations alone were tens of KB of code, fetched anew by every launch.
    constexpr int ORS = BN + 4;                                         // floats per row
    static_assert(4 * 16 * ORS * 4 <= (SLABS > 0 ? L::ONE_STAGE : L::BYTES), "the slabs' LDS holds it");
    float *mine = reinterpret_cast<float *>(smem_tiled) + wave * 16 * ORS;
    auto as_float = [](const char *at) -> float {
        if constexpr (ES == 4) return *reinterpret_cast<const float *>(at);
        else return TT::ID == 2 ? bf16_bits_to_f32(*reinterpret_cast<const uint16_t *>(at)) : f16_bits_to_f32(*reinterpret_cast<const uint16_t *>(at));
    };
    const int orow = lane >> 3, ocol = (lane & 7) * 4;                  // eight lanes per row: rows orow and orow + 8, 32 columns at a time
    __syncthreads();
    int64_t crow[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int m = m0 + wave_m0 + h * 8 + orow, mm = min(m, Me - 1), b = mm / p.K;
        crow[h] = m < Me ? (((int64_t)b * p.E + e) * p.K + (mm - b * p.K)) * p.ldc : -1;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4 *>(mine + a * ORS + j * 16 + g * 4) = acc[j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll 1
    for (int c = ocol; c < BN && n0 + c < N; c += 32) {
        const int n = n0 + c;
        f32x4 v[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) v[h] = *reinterpret_cast<const f32x4 *>(mine + (h * 8 + orow) * ORS + c);
        if (p.w_scale != nullptr || p.bias != nullptr) {
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const int64_t at = (int64_t)e * N + min(n + x, N - 1);
                const float f = p.w_scale != nullptr ? p.w_scale[at] : 1.f, add = p.bias != nullptr ? as_float(p.bias + at * ES) : 0.f;
                v[0][x] = v[0][x] * f + add;
                v[1][x] = v[1][x] * f + add;
            }
        }
        if constexpr (WES == 2)
            apply_activation_of<TT>(p.act, [&](auto fn) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int x = 0; x < 4; ++x) v[h][x] = fn(v[h][x]);
            });
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (crow[h] < 0) continue;
            char *dst = p.C + (crow[h] + n) * (ES == 4 || p.out_f32 ? 4 : 2);
            if (n + 4 <= N) {
                if (ES == 4 || p.out_f32) *reinterpret_cast<f32x4_any *>(dst) = v[h];
                else *reinterpret_cast<u32x2_any *>(dst) = u32x2{pack2<TT>(v[h][0], v[h][1]), pack2<TT>(v[h][2], v[h][3])};
            } else {
                for (int x = 0; n + x < N; ++x) {
                    if (ES == 4 || p.out_f32) reinterpret_cast<float *>(dst)[x] = v[h][x];
                    else reinterpret_cast<uint16_t *>(dst)[x] = (uint16_t)f32_to_elem_bits<TT>(v[h][x]);
                }
            }
        }
    }
}

// Two slabs of fp32 rows times 80 columns of weights [N][R] take 104 registers: bound to the 96 of five wavefronts they put two away in memory (120 such
// gathers 1.011 of the time; two of them, of 46 us and more, 0.97).
template <class TT, int WES, bool W_TRANS, int TN, int SLABS>
__global__ __launch_bounds__(kThreads, SLABS == 1 ? 6 : SLABS == 2 && !(TT::ES == 4 && !W_TRANS && TN == 5) ? 5 : SLABS > 0 || TN <= 2 ? 4 : 3) void tiled_rows_kernel(TiledRowsParams p)
{
    tiled_rows_body<TT, WES, W_TRANS, TN, SLABS>(p, (int)blockIdx.x);
}

// Rows or experts of less than 16 bytes in all: one thread per product, element by element.
template <class TT, int WES, bool W_TRANS>
__global__ __launch_bounds__(kThreads) void tiny_rows_kernel(TiledRowsParams p)
{
    const int64_t total = (int64_t)p.B * p.E * p.K * p.N;
    auto elem = [](const char *at) -> float {
        if constexpr (TT::ES == 4) return *reinterpret_cast<const float *>(at);
        else return TT::ID == 2 ? bf16_bits_to_f32(*reinterpret_cast<const uint16_t *>(at)) : f16_bits_to_f32(*reinterpret_cast<const uint16_t *>(at));
    };
    for (int64_t at = (int64_t)blockIdx.x * kThreads + threadIdx.x; at < total; at += (int64_t)gridDim.x * kThreads) {
        const int64_t pick = at / p.N;
        const int n = (int)(at - pick * p.N), e = (int)(pick / p.K % p.E);
        const char *row = p.A + pick * p.R * TT::ES;
        if (p.gather) {
            const int32_t t = load_token(p.Ind, p.ind_dtype, pick, p.T);
            row = t < 0 ? nullptr : p.A + (pick / p.K / p.E * p.lda_b + (int64_t)t * p.lda_t) * TT::ES;
        }
        float v = 0.f;
        for (int r = 0; row != nullptr && r < p.R; ++r) {
            const int64_t w = (int64_t)e * p.R * p.N + (W_TRANS ? (int64_t)r * p.N + n : (int64_t)n * p.R + r);
            float wv;
            if constexpr (WES == 1) wv = __builtin_amdgcn_cvt_f32_fp8((int)(uint32_t)(uint8_t)p.W[w], 0);
            else wv = elem(p.W + w * TT::ES);
            v += elem(row + (int64_t)r * TT::ES) * wv;
        }
        if (p.w_scale != nullptr) v *= p.w_scale[(int64_t)e * p.N + n];
        if (p.bias != nullptr) v += elem(p.bias + ((int64_t)e * p.N + n) * TT::ES);
        if constexpr (TT::ES == 2) apply_activation_of<TT>(p.act, [&](auto fn) { v = fn(v); });
        if (TT::ES == 4 || p.out_f32) reinterpret_cast<float *>(p.C)[pick * p.ldc + n] = v;
        else reinterpret_cast<uint16_t *>(p.C)[pick * p.ldc + n] = (uint16_t)f32_to_elem_bits<TT>(v);
    }
}

// ------------------------------------------------------------------------------ weight gradient
struct TiledDwParams {
    const char *Xs;             // [B,T,I] rows, element strides (ldx_b, ldx_t, 1)
    const char *Ys;             // [B,E,K,J] dense
    const void *Ind;
    char *dW;                   // [E,I,J] or [E,J,I] in out_dtype; S > 1: fp32 [S] of them, in the same layout
    int64_t x_bytes, y_bytes;   // extents, at least 16
    int64_t ldx_b, ldx_t;
    int32_t B, T, E, K, I, J;
    int32_t ind_dtype, out_dtype, eji;
    int32_t i_tiles, j_tiles, S, picks_per_split;
    int32_t wide;               // tiled_dw_wide_kernel (S = 1)
    int32_t split32;            // fp32: tiled_dw_split_kernel (egs_split_f32.h); operands below 2 GiB
    int32_t edges;              // some row is not a whole number of chunks: chunks may have to be read early and shifted
};
// what a pick that does not exist reads instead of a row
static __device__ const u32x4 kZeroChunk = {0u, 0u, 0u, 0u};

template <class TT>
struct TiledDw {
    static constexpr int ES = TT::ES, TI = 32, TJ = ES == 2 ? 64 : 32;
    static constexpr int XB = TI * ES, YB = TJ * ES;                    // bytes of a pick's piece
    static constexpr int XS = ES == 2 ? XB : 192, YS = ES == 2 ? YB : 192;      // strides in the staging tile (fp32: padded)
    static constexpr int STAGE = 32 * (XS + YS);                        // one step of 32 picks
    static constexpr int TAB = 2 * 64 * 16;                             // byte offsets of both rows of two chunks of 64 picks
    static constexpr int RS = TJ + 4;                                   // floats per row of the exchange tile
    static constexpr int EXCHANGE = TI * RS * 4;
    static constexpr int PER_WAVE = (TAB + STAGE > EXCHANGE ? TAB + STAGE : EXCHANGE);
    static constexpr int BYTES = 4 * PER_WAVE;
};

// A workgroup owns a 32 x TJ tile of dW(e) for one split of the expert's picks; its four wavefronts take consecutive parts of
// them, two 32-pick steps of rows in flight each, and are summed through LDS in wavefront order (as in egs_dw_tile.h, whose
// swizzles the 16-bit staging tiles use; there the operands are aligned and read through buffer descriptors).
template <class TT>
__device__ __forceinline__ void tiled_dw_body(const TiledDwParams &p, const int block)
{
    typedef TiledDw<TT> L;
    constexpr int ES = TT::ES, VEC = TT::VEC, TJ = L::TJ, NWV = kThreads / 64;
    constexpr int XL = L::XB / 16, XN = 32 * XL / 64, YL = L::YB / 16, YN = 32 * YL / 64;
    constexpr int NY = TJ / 16;
    extern __shared__ __attribute__((aligned(16))) char smem_tiled_dw[];

    const int per_e = p.i_tiles * p.j_tiles * p.S;
    const int lin = balanced_tile(block, p.E * per_e);
    if (lin < 0) return;
    const int e = lin / per_e;
    int rest = lin - e * per_e;
    const int split = rest / (p.i_tiles * p.j_tiles);
    rest -= split * (p.i_tiles * p.j_tiles);
    const int i0 = (rest / p.j_tiles) * L::TI, j0 = (rest % p.j_tiles) * TJ;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = lane & 15, g = lane >> 4;
    const int Me = p.B * p.K;
    const int lo = split * p.picks_per_split, hi = min(Me, lo + p.picks_per_split);
    const int per_wave = ((hi - lo + NWV - 1) / NWV + 31) & ~31;
    const int w_begin = min(hi, lo + wave * per_wave), w_end = min(hi, w_begin + per_wave);
    const int nsteps = (w_end - w_begin + 31) >> 5;

    char *mine = smem_tiled_dw + wave * L::PER_WAVE;
    int64_t *tab = reinterpret_cast<int64_t *>(mine);                   // [2][x: 64 | y: 64], -1: no such pick
    char *stage = mine + L::TAB;

    const int xp = lane / XL, xcn = lane % XL, yp = lane / YL, ycn = lane % YL;
    const int xc = i0 + xcn * VEC, yc = j0 + ycn * VEC;
    const bool x_in = xc < p.I, y_in = yc < p.J;
    const int64_t x_last = p.x_bytes - 16, y_last = p.y_bytes - 16;

    uint64_t iw = 0;
    auto pick_of = [&](int c, int &m, int &b) -> int64_t {
        m = w_begin + c * 64 + lane;
        const int mm = min(m, Me - 1);
        b = mm / p.K;
        return ((int64_t)b * p.E + e) * p.K + (mm - b * p.K);
    };
    auto load_idx = [&](int c) { int m, b; iw = load_index_word(p.Ind, p.ind_dtype, pick_of(c, m, b)); };
    auto store_tab = [&](int c) {
        int m, b;
        const int64_t pick = pick_of(c, m, b);
        const int64_t t = decode_index_word(iw, p.Ind, p.ind_dtype, pick);
        const bool live = m < w_end && t >= 0 && t < (int64_t)p.T;
        int64_t *at = tab + (c & 1) * 128;
        at[lane] = live ? ((int64_t)b * p.ldx_b + t * p.ldx_t) * ES : -1;
        at[64 + lane] = live ? pick * p.J * ES : -1;
    };
    u32x4 rx[2][XN], ry[2][YN];
    int sx[2][XN], sy[2][YN];                                           // bytes by which a chunk was read early
    auto fetch = [&](const char *base, int64_t off, int col, bool in, int64_t last, int &early) -> u32x4 {
        // an offset from `base` in every case (also to the zeros): the compiler then knows the load is a global one
        int64_t at = off + (int64_t)col * ES;
        early = 0;
        if (p.edges && off >= 0 && at > last) { early = (int)(at - last); at = last; }
        if (off < 0 || !in) { at = reinterpret_cast<const char *>(&kZeroChunk) - base; early = 0; }
        return *reinterpret_cast<const u32x4_any *>(base + at);
    };
    auto issue = [&](int s, u32x4 (&x)[XN], u32x4 (&y)[YN], int (&ex)[XN], int (&ey)[YN]) {
        const int64_t *at = tab + ((s >> 1) & 1) * 128 + (s & 1) * 32;
#pragma unroll
        for (int h = 0; h < XN; ++h) x[h] = fetch(p.Xs, at[h * (64 / XL) + xp], xc, x_in, x_last, ex[h]);
#pragma unroll
        for (int h = 0; h < YN; ++h) y[h] = fetch(p.Ys, at[64 + h * (64 / YL) + yp], yc, y_in, y_last, ey[h]);
    };
    // see dw_tile_body for the 16-bit swizzles
    const int fr = a >> 2;
    const int xkey = ((fr >> 1) & 1) ^ (g & 1), ykey = (fr & 3) ^ g;
    const int at0 = ES == 2 ? (g * 8 + fr) * 64 + (a & 3) * 8 : g * L::XS + a * 4, at1 = at0 + 4 * 64;
    const int yat0 = ES == 2 ? (g * 8 + fr) * 128 + (a & 3) * 8 : g * L::YS + a * 4, yat1 = yat0 + 4 * 128;
    const int wr = ES == 2 ? xp * 64 + (((xcn >> 1) ^ ((xp >> 1) & 1) ^ ((xp >> 3) & 1)) << 5) + (xcn & 1) * 16 : xp * L::XS + xcn * 16;
    const int ywr = ES == 2 ? yp * 128 + (((ycn >> 1) ^ (yp & 3)) << 5) + (ycn & 1) * 16 : yp * L::YS + ycn * 16;
    constexpr int XT = 32 * L::XS;
    auto put = [&](u32x4 (&x)[XN], u32x4 (&y)[YN], const int (&ex)[XN], const int (&ey)[YN]) {
        if (p.edges) {
            int any = 0;
#pragma unroll
            for (int h = 0; h < XN; ++h) any |= ex[h];
#pragma unroll
            for (int h = 0; h < YN; ++h) any |= ey[h];
            if (__any(any)) {
#pragma unroll
                for (int h = 0; h < XN; ++h) x[h] = shift_right_bytes(x[h], ex[h]);
#pragma unroll
                for (int h = 0; h < YN; ++h) y[h] = shift_right_bytes(y[h], ey[h]);
            }
        }
#pragma unroll
        for (int h = 0; h < XN; ++h) *reinterpret_cast<u32x4 *>(stage + h * (64 / XL) * L::XS + wr) = x[h];
#pragma unroll
        for (int h = 0; h < YN; ++h)
            *reinterpret_cast<u32x4 *>(stage + XT + h * (64 / YL) * L::YS + (ES == 2 ? ywr ^ ((h & 3) << 5) : ywr)) = y[h];
    };
    struct Frag16 { u32x4 v; };
    struct Frag32 { float v[8]; };
    typedef typename std::conditional<ES == 2, Frag16, Frag32>::type Frag;
    f32x4 acc[2][NY];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto get = [&](Frag (&pf)[2], Frag (&qf)[NY]) {
        if constexpr (ES == 2) {
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const u32x2 l = lds_read_tr16(stage + at0 + ((x ^ xkey) << 5)), h = lds_read_tr16(stage + at1 + ((x ^ xkey) << 5));
                pf[x].v = u32x4{l[0], l[1], h[0], h[1]};
            }
#pragma unroll
            for (int y = 0; y < NY; ++y) {
                const u32x2 l = lds_read_tr16(stage + XT + yat0 + ((y ^ ykey) << 5)), h = lds_read_tr16(stage + XT + yat1 + ((y ^ ykey) << 5));
                qf[y].v = u32x4{l[0], l[1], h[0], h[1]};
            }
        } else {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int k = 0; k < 8; ++k) pf[x].v[k] = *reinterpret_cast<const float *>(stage + at0 + k * 4 * L::XS + x * 64);
#pragma unroll
            for (int y = 0; y < NY; ++y)
#pragma unroll
                for (int k = 0; k < 8; ++k) qf[y].v[k] = *reinterpret_cast<const float *>(stage + XT + yat0 + k * 4 * L::YS + y * 64);
        }
    };
    auto multiply = [&](const Frag (&pf)[2], const Frag (&qf)[NY]) {
        if constexpr (ES == 2) {
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < NY; ++y) mma_chunk<TT>(acc[x][y], qf[y].v, pf[x].v);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k)
#pragma unroll
                for (int x = 0; x < 2; ++x)
#pragma unroll
                    for (int y = 0; y < NY; ++y)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[y].v[k], pf[x].v[k], acc[x][y], 0, 0, 0);
        }
    };
    // Steps beyond the last read kZeroChunk; nothing in the loop is conditional on them, so the loads in flight stay countable.
    // Step s: its fragments out of the staging tile, step s + 1's rows into it (a wavefront's LDS accesses happen in order, so one
    // tile is enough), step s + 3's rows requested, then the matrix instructions of step s.
    if (nsteps > 0) {
        load_idx(0); store_tab(0);
        load_idx(1);
        issue(0, rx[0], ry[0], sx[0], sy[0]);
        issue(1, rx[1], ry[1], sx[1], sy[1]);
        store_tab(1);
        load_idx(2);
        put(rx[0], ry[0], sx[0], sy[0]);
        issue(2, rx[0], ry[0], sx[0], sy[0]);
        for (int s = 0; s < nsteps; s += 2) {
            Frag pf[2], qf[NY];
            get(pf, qf);
            __builtin_amdgcn_sched_barrier(0);
            put(rx[1], ry[1], sx[1], sy[1]);
            issue(s + 3, rx[1], ry[1], sx[1], sy[1]);
            __builtin_amdgcn_sched_barrier(0);
            multiply(pf, qf);
            get(pf, qf);
            __builtin_amdgcn_sched_barrier(0);
            put(rx[0], ry[0], sx[0], sy[0]);
            store_tab((s >> 1) + 2);
            load_idx((s >> 1) + 3);
            issue(s + 4, rx[0], ry[0], sx[0], sy[0]);
            __builtin_amdgcn_sched_barrier(0);
            multiply(pf, qf);
        }
    }
    __syncthreads();

    // lane (a, g) holds rows i0 + 16 x + a, columns j0 + 16 y + 4 g .. + 3 of its wavefront's share
    float *red = reinterpret_cast<float *>(smem_tiled_dw);
    constexpr int RS = L::RS, PW = L::PER_WAVE / 4;
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y)
            *reinterpret_cast<f32x4 *>(red + wave * PW + (x * 16 + a) * RS + y * 16 + g * 4) = acc[x][y];
    __syncthreads();
    const bool eji = p.eji != 0;
    const int out_dtype = p.S > 1 ? 0 : p.out_dtype;
    const int64_t base = p.S > 1 ? (int64_t)split * p.E * p.I * p.J : 0;
    for (int item = tid; item < 8 * TJ; item += kThreads) {
        const int gi_l = eji ? item & 31 : item / (TJ / 4), gj_l = (eji ? item >> 5 : item % (TJ / 4)) * 4;
        f32x4 v = *reinterpret_cast<const f32x4 *>(red + gi_l * RS + gj_l);
#pragma unroll
        for (int w = 1; w < NWV; ++w) {
            const f32x4 u = *reinterpret_cast<const f32x4 *>(red + w * PW + gi_l * RS + gj_l);
            v[0] += u[0]; v[1] += u[1]; v[2] += u[2]; v[3] += u[3];
        }
        const int gi = i0 + gi_l, gj = j0 + gj_l;
        if (gi >= p.I || gj >= p.J) continue;
        if (!eji && gj + 4 <= p.J) {
            const int64_t at = base + ((int64_t)e * p.I + gi) * p.J + gj;
            if (out_dtype == 0) *reinterpret_cast<f32x4_any *>(p.dW + at * 4) = v;
            else if (out_dtype == 1) *reinterpret_cast<u32x2_any *>(p.dW + at * 2) = u32x2{pack2<ElemF16>(v[0], v[1]), pack2<ElemF16>(v[2], v[3])};
            else *reinterpret_cast<u32x2_any *>(p.dW + at * 2) = u32x2{pack2<ElemBF16>(v[0], v[1]), pack2<ElemBF16>(v[2], v[3])};
        } else {
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                if (gj + x >= p.J) continue;
                const int64_t at = base + (eji ? ((int64_t)e * p.J + gj + x) * p.I + gi : ((int64_t)e * p.I + gi) * p.J + gj + x);
                if (out_dtype == 0) reinterpret_cast<float *>(p.dW)[at] = v[x];
                else reinterpret_cast<uint16_t *>(p.dW)[at] =
                         (uint16_t)((out_dtype == 1 ? pack2<ElemF16>(v[x], 0.f) : pack2<ElemBF16>(v[x], 0.f)) & 0xffffu);
            }
        }
    }
}

template <class TT>
__global__ __launch_bounds__(kThreads) void tiled_dw_kernel(TiledDwParams p) { tiled_dw_body<TT>(p, (int)blockIdx.x); }

// The same for experts of few picks, where dW itself is what takes the time: 64 rows x 256 bytes of columns per workgroup, a
// wavefront 16 rows x all columns, the picks in slabs of 32 that the four wavefronts share.  (Splitting the picks over wavefronts
// and adding four partial tiles up, as above, took 344 us for the 134 MB of fp32 dW at B1 E128 K4 I1024 J256; this way 46.)
template <class TT>
struct TiledDwWide {
    static constexpr int ES = TT::ES, TI = 64, TJ = 256 / ES, NJ = TJ / 16;
    // bytes of a pick's row in the tiles: an odd number of 32-byte units and 128 more bytes every eight rows for transpose reads
    // (see TiledLds), fp32 rows 4 banks apart modulo 16
    static constexpr int XROW = ES == 2 ? TI * 2 + 32 : (TI + 4) * 4, YROW = ES == 2 ? TJ * 2 + 32 : (TJ + 4) * 4;
    static constexpr int X = 32 * XROW + 512, Y = 32 * YROW + 512;
    static constexpr int STAGE = X + Y;
    static constexpr int RS = TJ + 4;                                   // floats per row of a wavefront's results
    static constexpr int TAB_AT = 2 * STAGE > 64 * RS * 4 ? 2 * STAGE : 64 * RS * 4;
    static constexpr int TAB = 256, BYTES = TAB_AT + 2 * TAB * 8;
};

template <class TT>
__device__ __forceinline__ void tiled_dw_wide_body(const TiledDwParams &p, const int block)
{
    typedef TiledDwWide<TT> L;
    constexpr int ES = TT::ES, VEC = TT::VEC, TI = L::TI, TJ = L::TJ, NJ = L::NJ;
    constexpr int XL = TI * ES / 16, YL = 16;                           // chunks per pick: 8 (fp32 16) of X, 16 of Y
    constexpr int XN = 32 * XL / kThreads, YN = 32 * YL / kThreads;
    extern __shared__ __attribute__((aligned(16))) char smem_tiled_dww[];
    const int per_e = p.i_tiles * p.j_tiles;
    const int lin = balanced_tile(block, p.E * per_e);
    if (lin < 0) return;
    const int e = lin / per_e, rest = lin - e * per_e;
    const int i0 = (rest / p.j_tiles) * TI, j0 = (rest % p.j_tiles) * TJ;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = lane & 15, g = lane >> 4;
    const int Me = p.B * p.K, nslabs = (Me + 31) >> 5;
    const int xp = tid / XL, xc = tid % XL, yp = tid / YL, yc = tid % YL;
    const bool x_in = i0 + xc * VEC < p.I, y_in = j0 + yc * VEC < p.J;
    const int64_t x_last = p.x_bytes - 16, y_last = p.y_bytes - 16;

    // byte offsets of the rows of kTab picks, -1: no such pick.  (Made slab by slab, the index words kept the rows' loads waiting.)
    constexpr int kTab = L::TAB;
    int64_t *tab = reinterpret_cast<int64_t *>(smem_tiled_dww + L::TAB_AT);       // [X: kTab | Y: kTab]
    auto make_tab = [&](int s) {                                        // from slab s on
#pragma unroll
        for (int at = tid; at < kTab; at += kThreads) {
            if (s * 32 + at - tid >= Me + 96) break;                    // (two slabs beyond the last are looked up)
            const int m = s * 32 + at, mm = min(m, Me - 1), b = mm / p.K;
            const int64_t pick = ((int64_t)b * p.E + e) * p.K + (mm - b * p.K);
            const int64_t t = decode_index_word(load_index_word(p.Ind, p.ind_dtype, pick), p.Ind, p.ind_dtype, pick);
            const bool ok = m < Me && t >= 0 && t < (int64_t)p.T;
            tab[at] = ok ? ((int64_t)b * p.ldx_b + t * p.ldx_t) * ES : -1;
            tab[kTab + at] = ok ? pick * p.J * ES : -1;
        }
    };
    u32x4 rx[2][XN], ry[2][YN];
    // no load is conditional: what must not count - picks that do not exist, columns past the matrix - is read somewhere in bounds and
    // cleared on the way into LDS; a chunk at the end of an operand is read early and shifted
    int shift_x[2][XN], shift_y[2][YN];
    auto issue = [&](int s, int q) {
        auto fetch = [&](const char *base, int64_t row, int at_in_row, bool in, int64_t last, int &shift) -> u32x4 {
            const bool ok = row >= 0 && in;
            const int64_t at = ok ? row + at_in_row : 0, from = min(at, last);
            shift = ok ? (int)(at - from) : 16;
            return *reinterpret_cast<const u32x4_any *>(base + from);
        };
        const int64_t *row = tab + s % (kTab / 32) * 32;
#pragma unroll
        for (int h = 0; h < XN; ++h) rx[q][h] = fetch(p.Xs, row[h * (kThreads / XL) + xp], i0 * ES + xc * 16, x_in, x_last, shift_x[q][h]);
#pragma unroll
        for (int h = 0; h < YN; ++h) ry[q][h] = fetch(p.Ys, row[kTab + h * (kThreads / YL) + yp], j0 * ES + yc * 16, y_in, y_last, shift_y[q][h]);
    };
    auto row_at = [&](int r, int stride) { return r * stride + (ES == 2 ? (r >> 3) * 128 : 0); };
    auto put = [&](char *stage, int q) {
        auto settle = [](u32x4 v, int shift) -> u32x4 {
            if (__any(shift & 15)) v = shift_right_bytes(v, shift & 15);            // (at an operand's end)
#pragma unroll
            for (int x = 0; x < 4; ++x) v[x] = shift >= 16 ? 0u : v[x];
            return v;
        };
#pragma unroll
        for (int h = 0; h < XN; ++h)
            *reinterpret_cast<u32x4 *>(stage + row_at(h * (kThreads / XL) + xp, L::XROW) + xc * 16) = settle(rx[q][h], shift_x[q][h]);
#pragma unroll
        for (int h = 0; h < YN; ++h)
            *reinterpret_cast<u32x4 *>(stage + L::X + row_at(h * (kThreads / YL) + yp, L::YROW) + yc * 16) = settle(ry[q][h], shift_y[q][h]);
    };
    f32x4 acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const char *stage) {
        const char *sy = stage + L::X;
        if constexpr (ES == 2) {
            // transpose reads: lane (a, g) points at pick 8 g + 4 h + a / 4, columns 4 (a % 4) .. + 3
            auto read = [&](const char *tile, int stride, int col) -> u32x4 {
                const char *at = tile + row_at(g * 8 + (a >> 2), stride) + col * 2 + (a & 3) * 8;
                const u32x2 lo = lds_read_tr16(at), hi = lds_read_tr16(at + 4 * stride);
                return u32x4{lo[0], lo[1], hi[0], hi[1]};
            };
            const u32x4 xf = read(stage, L::XROW, wave * 16);
#pragma unroll
            for (int j = 0; j < NJ; ++j) mma_chunk<TT>(acc[j], read(sy, L::YROW, j * 16), xf);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const float xv = *reinterpret_cast<const float *>(stage + (k * 4 + g) * L::XROW + (wave * 16 + a) * 4);
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(*reinterpret_cast<const float *>(sy + (k * 4 + g) * L::YROW + (j * 16 + a) * 4), xv,
                                                                  acc[j], 0, 0, 0);
            }
        }
    };
    // one barrier per slab, as in tiled_rows_kernel, two slabs in flight; those beyond the last are requested like any other
    make_tab(0);
    __syncthreads();
    issue(0, 0);
    issue(1, 1);
    for (int s0 = 0; s0 < nslabs; s0 += 2) {
        if ((s0 + 2) % (kTab / 32) == 0) { make_tab(s0 + 2); __syncthreads(); }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int s = s0 + q;
            if (s >= nslabs) break;
            char *stage = smem_tiled_dww + q * L::STAGE;
            put(stage, q);
            issue(s + 2, q);
            __syncthreads();
            multiply(stage);
        }
    }
    __syncthreads();

    // lane (a, g) holds row i0 + 16 wave + a, columns j0 + 16 j + 4 g .. + 3; through LDS, so that whole row (or, [E,J,I], column)
    // segments leave
    float *red = reinterpret_cast<float *>(smem_tiled_dww) + wave * 16 * L::RS;
#pragma unroll
    for (int j = 0; j < NJ; ++j) *reinterpret_cast<f32x4 *>(red + a * L::RS + j * 16 + g * 4) = acc[j];
    auto pack = [&](float x, float y) -> uint32_t { return p.out_dtype == 1 ? pack2<ElemF16>(x, y) : pack2<ElemBF16>(x, y); };
    const int oes = p.out_dtype == 0 ? 4 : 2;
    const bool eji = p.eji != 0;
    if (eji) __syncthreads();
    else __builtin_amdgcn_wave_barrier();
    // four values along the output's rows at a time: [E,I,J] a wavefront's own 16 rows, [E,J,I] all 64 of the workgroup's
#pragma unroll 1
    for (int v = lane; v < 4 * TJ; v += 64) {
        int gi, gj;
        f32x4 r;
        if (eji) {
            const int il = (v & 15) * 4, jl = wave * (TJ / 4) + (v >> 4);
            const float *at = reinterpret_cast<const float *>(smem_tiled_dww) + il * L::RS + jl;
            gi = i0 + il; gj = j0 + jl;
            r = f32x4{at[0], at[L::RS], at[2 * L::RS], at[3 * L::RS]};
        } else {
            const int il = v / (TJ / 4), jl = v % (TJ / 4) * 4;
            gi = i0 + wave * 16 + il; gj = j0 + jl;
            r = *reinterpret_cast<const f32x4 *>(red + il * L::RS + jl);
        }
        if (gi >= p.I || gj >= p.J) continue;
        const int live = min(4, eji ? p.I - gi : p.J - gj);
        char *dst = p.dW + (eji ? ((int64_t)e * p.J + gj) * p.I + gi : ((int64_t)e * p.I + gi) * p.J + gj) * oes;
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

template <class TT>
__global__ __launch_bounds__(kThreads, 3) void tiled_dw_wide_kernel(TiledDwParams p) { tiled_dw_wide_body<TT>(p, (int)blockIdx.x); }

// sums of S fp32 parts of n elements in increasing order, rounded once
static __global__ __launch_bounds__(kThreads) void tiled_dw_sum_kernel(const float *part, char *dW, int S, int64_t n, int out_dtype)
{
    const int64_t n4 = (n + 3) / 4;
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n4; i += (int64_t)gridDim.x * kThreads) {
        const int64_t at = i * 4 + 4 <= n ? i * 4 : n >= 4 ? n - 4 : 0;      // the last thread redoes a few sums rather than go element by element
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        const int live = n >= 4 ? 4 : (int)n;
        int s = 0;
        for (; live == 4 && s + 4 <= S; s += 4) {                            // four parts in flight
            f32x4 u[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) u[x] = *reinterpret_cast<const f32x4_any *>(part + (int64_t)(s + x) * n + at);
#pragma unroll
            for (int x = 0; x < 4; ++x) { v[0] += u[x][0]; v[1] += u[x][1]; v[2] += u[x][2]; v[3] += u[x][3]; }
        }
        for (; s < S; ++s) {
            const float *src = part + (int64_t)s * n + at;
            if (live == 4) { const f32x4 u = *reinterpret_cast<const f32x4_any *>(src); v[0] += u[0]; v[1] += u[1]; v[2] += u[2]; v[3] += u[3]; }
            else for (int x = 0; x < live; ++x) v[x] += src[x];
        }
        if (live == 4) {
            if (out_dtype == 0) *reinterpret_cast<f32x4_any *>(dW + at * 4) = v;
            else if (out_dtype == 1) *reinterpret_cast<u32x2_any *>(dW + at * 2) = u32x2{pack2<ElemF16>(v[0], v[1]), pack2<ElemF16>(v[2], v[3])};
            else *reinterpret_cast<u32x2_any *>(dW + at * 2) = u32x2{pack2<ElemBF16>(v[0], v[1]), pack2<ElemBF16>(v[2], v[3])};
        } else {
            for (int x = 0; x < live; ++x) {
                if (out_dtype == 0) reinterpret_cast<float *>(dW)[at + x] = v[x];
                else reinterpret_cast<uint16_t *>(dW)[at + x] =
                         (uint16_t)((out_dtype == 1 ? pack2<ElemF16>(v[x], 0.f) : pack2<ElemBF16>(v[x], 0.f)) & 0xffffu);
            }
        }
    }
}

// Operands of less than 16 bytes: one thread per element of dW, pick by pick, all picks (S = 1).
template <class TT>
__global__ __launch_bounds__(kThreads) void tiny_dw_kernel(TiledDwParams p)
{
    auto elem = [](const char *at) -> float {
        if constexpr (TT::ES == 4) return *reinterpret_cast<const float *>(at);
        else return TT::ID == 2 ? bf16_bits_to_f32(*reinterpret_cast<const uint16_t *>(at)) : f16_bits_to_f32(*reinterpret_cast<const uint16_t *>(at));
    };
    const int64_t total = (int64_t)p.E * p.I * p.J;
    for (int64_t w = (int64_t)blockIdx.x * kThreads + threadIdx.x; w < total; w += (int64_t)gridDim.x * kThreads) {
        const int e = (int)(w / ((int64_t)p.I * p.J));
        const int64_t ij = w - (int64_t)e * p.I * p.J;
        const int i = (int)(p.eji ? ij % p.I : ij / p.J), j = (int)(p.eji ? ij / p.I : ij % p.J);
        float v = 0.f;
        for (int m = 0; m < p.B * p.K; ++m) {
            const int b = m / p.K;
            const int64_t pick = ((int64_t)b * p.E + e) * p.K + (m - b * p.K);
            const int32_t t = load_token(p.Ind, p.ind_dtype, pick, p.T);
            if (t < 0) continue;
            v += elem(p.Xs + ((int64_t)b * p.ldx_b + (int64_t)t * p.ldx_t + i) * TT::ES) * elem(p.Ys + (pick * p.J + j) * TT::ES);
        }
        if (p.out_dtype == 0) reinterpret_cast<float *>(p.dW)[w] = v;
        else reinterpret_cast<uint16_t *>(p.dW)[w] =
                 (uint16_t)((p.out_dtype == 1 ? pack2<ElemF16>(v, 0.f) : pack2<ElemBF16>(v, 0.f)) & 0xffffu);
    }
}

}  // namespace egs
