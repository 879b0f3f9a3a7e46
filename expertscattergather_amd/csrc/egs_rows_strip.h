// Rows x weight products of mid-sized 16-bit experts, any well-formed reduction length, on the direct-to-LDS pipeline in tiles small enough
// to give every CU some.
//
// A workgroup of eight wavefronts owns 128 x 64 of one expert's results and goes through the reduction in slabs of 64: rows as
// [row][reduction], weights as they lie ([column][reduction] or, W_TRANS, [reduction][column], read back with the LDS transpose read), a
// slab of direct 16-byte loads in flight under the one being multiplied, one barrier per slab.  Chunks past the reduction length, rows
// that do not exist and columns past the last get an offset outside the buffer descriptors and arrive as zeros.
//
// What bounds such a product is a chain of round trips (index, with which the compiler waits for the first weights too, rows, slabs, results), so three workgroups share a CU: two stages of 24 KB
// (three stages and two workgroups: level where one round of those is enough, else slower, 27.7 us for 23.5 at R256 N136 Me2400 E40).
// 128 x 128 tiles took 1.8 times as long at R328 N136 Me900 E20, 64 x 64 tiles 1.2 times.  Against the general kernel's 64 rows through
// registers: R768 N64 Me2048 E32 (150 MB through the L2s instead of 200) 19.3 -> 13.8 us, R328 N136 Me900 E20 14 -> 10.
//
// Preconditions (checked by the host): R % 8 == 0, N % 8 == 0, 16-byte aligned rows, operands (of W: an expert's matrix) below 2 GiB.
#pragma once
#include "egs_rows_gemm_dl.h"
#include "egs_tiled.h"

namespace egs {

struct RowsStripParams {
    const char *A;              // gather: [B,T,R] source, strides (lda_b, lda_t, 1); else dense [B,E,K,R] rows
    const char *W;              // [E,R,N] (W_TRANS) or [E,N,R]
    const void *Ind;            // gather only
    char *C;                    // [B,E,K,ldc] rows, element type or fp32
    const char *bias;           // [E,N] in the element type, or nullptr
    int64_t lda_b, lda_t;
    uint32_t a_bytes;           // extent of A, below 2 GiB
    int32_t B, T, E, K, R, N, ldc;
    int32_t ind_dtype, gather, out_f32, act;
    int32_t m_tiles, n_tiles;
    int32_t rows_major;         // numbering of the tiles: 1 = row tiles outermost (their source rows share an L2), 0 = experts outermost
};

constexpr int kStripThreads = 512;

struct RowsStripLds {
    static constexpr int BM = 128, BN = 64, NST = 2;
    static constexpr int A = BM * 128, W = BN * 128, STAGE = A + W;     // bytes
    static constexpr int ORS = BN + 4;                                  // floats per row of the results
    static constexpr int BYTES = NST * STAGE + BM * 8;                  // (element offsets of the results' rows behind the stages)
    static_assert(BM * ORS * 4 <= NST * STAGE, "the results fit");
};

template <class TT, bool W_TRANS>
__global__ __launch_bounds__(kStripThreads, 6) void rows_strip_kernel(RowsStripParams p)
{
    static_assert(TT::ES == 2, "16-bit element types");
    typedef RowsStripLds L;
    constexpr int BM = L::BM, BN = L::BN, WM = 4, WN = 8 / WM, TM = BM / WM / 16, TN = BN / WN / 16;   // wavefront grid, 16 x 16 tiles of a wavefront
    constexpr int PL = BM / 64, QL = BN / 64;                           // loads (1 KB) per wavefront and slab: rows, weights
    extern __shared__ __attribute__((aligned(1024))) char smem_rows_strip[];

    const int lin = balanced_tile((int)blockIdx.x, p.E * p.m_tiles * p.n_tiles);
    if (lin < 0) return;
    int e, mt, nt;
    if (p.rows_major) { mt = lin / (p.E * p.n_tiles); const int r = lin - mt * p.E * p.n_tiles; e = r / p.n_tiles; nt = r - e * p.n_tiles; }
    else { e = lin / (p.m_tiles * p.n_tiles); const int r = lin - e * p.m_tiles * p.n_tiles; mt = r / p.n_tiles; nt = r - mt * p.n_tiles; }
    const int m0 = mt * BM, n0 = nt * BN;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = lane & 15, g = lane >> 4;
    const int R = p.R, N = p.N, Me = p.B * p.K, nk = (R + 63) / 64;
    auto pick_of = [&](int m, int &b) -> int64_t {
        b = m / p.K;
        return ((int64_t)b * p.E + e) * p.K + (m - b * p.K);
    };

    // ---------------- rows: a load covers eight 128-byte pieces; lane l lands on row 8 j + l / 8, chunk l % 8 and fetches chunk
    // (l % 8) ^ (row % 8), so that the 16 rows of a fragment read cover all banks
    const int ac = ((lane & 7) ^ (lane >> 3)) * 8;                      // reduction element of the lane's chunk
    uint64_t iw[PL];
    int64_t pick[PL];
    int pb[PL];
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        pick[j] = pick_of(min(m0 + (wave * PL + j) * 8 + (lane >> 3), Me - 1), pb[j]);
        iw[j] = 0;
    }
    if (p.gather) {
#pragma unroll
        for (int j = 0; j < PL; ++j) iw[j] = load_index_word(p.Ind, p.ind_dtype, pick[j]);
    }
    const u32x4 rs_w = make_rsrc(p.W + (size_t)e * R * N * 2, (uint32_t)((size_t)R * N * 2));
    uint32_t qv[QL];
    int qk[QL];                                                         // reduction element of the lane's chunk, or row
#pragma unroll
    for (int j = 0; j < QL; ++j) {
        if constexpr (!W_TRANS) {
            const int row = (wave * QL + j) * 8 + (lane >> 3);
            qk[j] = ac;
            qv[j] = n0 + row < N ? ((uint32_t)(n0 + row) * (uint32_t)R + ac) * 2 : kVoffInvalid;
        } else {
            const int at = (wave * QL + j) * 64 + lane, row = at / (BN / 8), pc = at % (BN / 8);
            const int n = n0 + ((((pc >> 1) ^ tr_key<BN>(row)) << 1) | (pc & 1)) * 8;
            qk[j] = row;
            qv[j] = n < N ? ((uint32_t)row * (uint32_t)N + n) * 2 : kVoffInvalid;
        }
    }
    auto issue_w = [&](int kt, int stage) {
        const uint32_t so = W_TRANS ? (uint32_t)kt * 128 * (uint32_t)N : (uint32_t)kt * 128;
        const int left = R - kt * 64;
#pragma unroll
        for (int j = 0; j < QL; ++j) direct_load16(rs_w, qk[j] < left ? qv[j] : kVoffInvalid, so, smem_rows_strip + stage * L::STAGE + L::A + (wave * QL + j) * 1024);
    };
    static_assert(L::NST == 2, "one slab on its way under the one being multiplied");
    if (nk > 0) issue_w(0, 0);
    const u32x4 rs_a = make_rsrc(p.A, p.a_bytes);
    uint32_t pv[PL];
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        bool ok = m0 + (wave * PL + j) * 8 + (lane >> 3) < Me;
        int64_t at = pick[j] * R;
        if (p.gather) {
            const int64_t t = decode_index_word(iw[j], p.Ind, p.ind_dtype, pick[j]);
            ok &= t >= 0 && t < (int64_t)p.T;
            at = (int64_t)pb[j] * p.lda_b + t * p.lda_t;
        }
        pv[j] = ok ? (uint32_t)((at + ac) * 2) : kVoffInvalid;
    }
    auto issue_a = [&](int kt, int stage) {
        const int left = R - kt * 64;
#pragma unroll
        for (int j = 0; j < PL; ++j) direct_load16(rs_a, ac < left ? pv[j] : kVoffInvalid, (uint32_t)kt * 128, smem_rows_strip + stage * L::STAGE + (wave * PL + j) * 1024);
    };
    if (nk > 0) issue_a(0, 0);
    int64_t *const c_row = reinterpret_cast<int64_t *>(smem_rows_strip + L::NST * L::STAGE);
    if (tid < BM) {
        int b;
        c_row[tid] = m0 + tid < Me ? pick_of(m0 + tid, b) * p.ldc : -1;
    }

    const int wm = wave / WN * (BM / WM), wn = wave % WN * (BN / WN);
    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    int stage = 0;
    for (int kt = 0; kt < nk; ++kt) {
        wait_vmem<0>();             // slab kt, the only one on its way
        __syncthreads();            // slab kt is everybody's; nobody reads the stage that is filled next
        if (kt + 1 < nk) {
            issue_a(kt + 1, stage ^ 1);
            issue_w(kt + 1, stage ^ 1);
        }
        const char *ta = smem_rows_strip + stage * L::STAGE, *tw = ta + L::A;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            u32x4 mf[TM], nf[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) mf[i] = *reinterpret_cast<const u32x4 *>(ta + (wm + i * 16 + a) * 128 + (((ks * 4 + g) ^ (a & 7)) << 4));
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                if constexpr (!W_TRANS) {
                    nf[j] = *reinterpret_cast<const u32x4 *>(tw + (wn + j * 16 + a) * 128 + (((ks * 4 + g) ^ (a & 7)) << 4));
                } else {
                    // lane (a, g) points at reduction row 32 ks + 8 g + 4 h + a / 4, columns 4 (a % 4) .. + 3 of the tile
                    const int row = ks * 32 + g * 8 + (a >> 2);
                    const u32x2 lo = lds_read_tr16(tw + row * (BN * 2) + (((wn >> 4) + j ^ tr_key<BN>(row)) << 5) + (a & 3) * 8);
                    const u32x2 hi = lds_read_tr16(tw + (row + 4) * (BN * 2) + (((wn >> 4) + j ^ tr_key<BN>(row + 4)) << 5) + (a & 3) * 8);
                    nf[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                }
            }
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) mma_chunk<TT>(acc[i][j], nf[j], mf[i]);
        }
        stage ^= 1;
    }

    // ---------------- results through LDS, out as whole row segments; lane (a, g) holds columns 4 g .. + 3 of row a of a tile
    __syncthreads();
    float *red = reinterpret_cast<float *>(smem_rows_strip);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) *reinterpret_cast<f32x4 *>(red + (wm + i * 16 + a) * L::ORS + wn + j * 16 + g * 4) = acc[i][j];
    __syncthreads();
    constexpr int CPR = BN / 4;                                         // four columns at a time
    const int c = (tid % CPR) * 4, n = n0 + c;
    if (n >= N) return;
    f32x4 add = {0.f, 0.f, 0.f, 0.f};
    if (p.bias != nullptr) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {                                   // N % 8 == 0: four columns are inside or outside
            const uint16_t h = reinterpret_cast<const uint16_t *>(p.bias)[(int64_t)e * N + n + x];
            add[x] = TT::ID == 2 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
        }
    }
#pragma unroll 1
    for (int r = tid / CPR; r < BM && m0 + r < Me; r += kStripThreads / CPR) {
        char *dst = p.C + (c_row[r] + n) * (p.out_f32 ? 4 : 2);
        f32x4 v = *reinterpret_cast<const f32x4 *>(red + r * L::ORS + c);
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] += add[x];
        apply_activation_of<TT>(p.act, [&](auto fn) {
#pragma unroll
            for (int x = 0; x < 4; ++x) v[x] = fn(v[x]);
        });
        if (p.out_f32) *reinterpret_cast<f32x4 *>(dst) = v;
        else *reinterpret_cast<u32x2 *>(dst) = u32x2{pack2<TT>(v[0], v[1]), pack2<TT>(v[2], v[3])};
    }
}

}  // namespace egs
