// Rows x weight products of experts with few rows: what takes the time is that every weight has to come from memory once.
//
// A workgroup of four wavefronts owns 16 MT rows (32 or 64) x 128 bytes of weight columns of one expert and goes through the whole
// reduction.  What bounds such a product is the number of bytes on their way: a request beyond the L2 takes about 4 us under load (3.9 at
// 4.9 TB/s), so 256 CUs move B / 4 us x 256 of weights for B bytes in flight on each.  tiled_rows_kernel keeps two slabs of two operands in
// registers, 24 KB a workgroup of which 8 KB fp8 weights.  Here slabs of 64 reduction elements (8 KB of weights and 4 KB
// of rows, at MT = 2) go from memory to LDS without passing through registers, three of them in flight and one being multiplied,
// three workgroups to a CU: 72 KB of weights.  Weight pieces are whole 128-byte lines.  A gather's first rows are requested once the first
// weights are there: the index words are the compiler's loads, and it waits for everything before it uses one, also what it does not count.
//
// 16-bit rows, 16-bit or (with [reduction][column] weights) fp8 weights, R a multiple of 64, 16-byte aligned rows, operands below 2 GiB.
#pragma once
#include "egs_rows_gemm.h"

namespace egs {

struct RowsStreamParams {
    const char *A;              // gather: [B,T,R] source, strides (lda_b, lda_t, 1); else dense [B,E,K,R] rows
    const char *W;              // [E,R,N] (W_TRANS) or [E,N,R]
    const void *Ind;            // gather only
    char *C;                    // [B,E,K,ldc] rows, element type or fp32
    const float *w_scale;       // [E,N] or nullptr
    const char *bias;           // [E,N] in the element type, or nullptr
    int64_t lda_b, lda_t;
    uint32_t a_bytes;           // extent of A, below 2 GiB
    int32_t B, T, E, K, R, N, ldc;
    int32_t ind_dtype, gather, out_f32, act;
    int32_t m_tiles, n_tiles;
};

template <int WES, int MT>
struct RowsStreamLds {
    static constexpr int STAGES = 4, BM = 16 * MT, BN = 128 / WES;
    static constexpr int A = BM * 128, W = 64 * 128, STAGE = A + W;     // bytes
    static constexpr int ORS = BN + 4;                                  // floats per row of the results
    static_assert(BM * ORS * 4 <= STAGES * STAGE, "the results fit");
    static constexpr int BYTES = STAGES * STAGE;
};

// ONCE: a single row tile, so that every weight is read once
template <class TT, int WES, bool W_TRANS, int MT, bool ONCE>
__global__ __launch_bounds__(kThreads) void rows_stream_kernel(RowsStreamParams p)
{
    static_assert(TT::ES == 2 && (WES == 2 || (W_TRANS && TT::ID == 2)), "16-bit rows; fp8 weights as stored, widened to bf16");
    typedef RowsStreamLds<WES, MT> L;
    constexpr int BM = L::BM, BN = L::BN, CT = BN / 64;                 // 16-column tiles per wavefront
    constexpr int PL = BM / 8 / 4, QL = 2, NL = PL + QL;                // loads (1 KB) per wavefront and slab: rows, weights
    extern __shared__ __attribute__((aligned(1024))) char smem_stream[];

    const int lin = balanced_tile((int)blockIdx.x, p.E * p.m_tiles * p.n_tiles);
    if (lin < 0) return;
    const int e = lin / (p.m_tiles * p.n_tiles), rest = lin - e * p.m_tiles * p.n_tiles;
    const int nt = rest / p.m_tiles, mt = rest - nt * p.m_tiles;        // the row tiles of the same weights are neighbours
    const int m0 = mt * BM, n0 = nt * BN;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a = lane & 15, g = lane >> 4;
    const int R = p.R, N = p.N, Me = p.B * p.K, nk = R / 64;
    auto pick_of = [&](int m, int &b) -> int64_t {
        b = m / p.K;
        return ((int64_t)b * p.E + e) * p.K + (m - b * p.K);
    };

    // ---------------- rows: a load covers eight 128-byte pieces; lane l lands on row 8 j + l / 8, chunk l % 8 and fetches chunk
    // (l % 8) ^ (row % 8), so that the 16 rows of a fragment read cover all banks
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
    // ---------------- weights: 128-byte pieces of 64 reduction rows (W_TRANS), or of 64 columns
    const u32x4 rs_w = make_rsrc(p.W + (size_t)e * R * N * WES, (uint32_t)((size_t)R * N * WES));
    uint32_t qv[QL];
#pragma unroll
    for (int j = 0; j < QL; ++j) {
        const int row = (wave * QL + j) * 8 + (lane >> 3), pc = lane & 7;
        if constexpr (!W_TRANS) {
            qv[j] = n0 + row < N ? (uint32_t)(n0 + row) * (uint32_t)R * 2 + ((pc ^ (row & 7)) << 4) : kVoffInvalid;
        } else if constexpr (WES == 1) {
            // 16-byte chunks (one 16-column tile each) XORed with (row / 2) % 8: the 32 rows of an 8-bit transpose read fall two deep on every bank
            const int n = n0 + ((pc ^ ((row >> 1) & 7)) << 4);
            qv[j] = n < N ? (uint32_t)row * (uint32_t)N + n : kVoffInvalid;
        } else {
            // 32-byte units XORed with bits 1 and 3 of the row: the 16 rows of a transpose read, two deep
            const int n = n0 + (((((pc >> 1) ^ (((row >> 1) & 1) | ((row >> 2) & 2))) << 1) | (pc & 1)) << 3);
            qv[j] = n < N ? ((uint32_t)row * (uint32_t)N + n) * 2 : kVoffInvalid;
        }
    }
    auto issue_w = [&](int kt, int stage) {
        const uint32_t so = W_TRANS ? (uint32_t)kt * 64 * (uint32_t)N * WES : (uint32_t)kt * 128;
#pragma unroll
        for (int j = 0; j < QL; ++j) direct_load16<ONCE>(rs_w, qv[j], so, smem_stream + stage * L::STAGE + L::A + (wave * QL + j) * 1024);
    };
    constexpr int AHEAD = L::STAGES - 1;
    for (int s = 0; s < min(AHEAD, nk); ++s) issue_w(s, s);
    const u32x4 rs_a = make_rsrc(p.A, p.a_bytes);
    uint32_t pv[PL];
#pragma unroll
    for (int j = 0; j < PL; ++j) {
        const int row = (wave * PL + j) * 8 + (lane >> 3);
        bool ok = m0 + row < Me;
        int64_t at = pick[j] * R;
        if (p.gather) {
            const int64_t t = decode_index_word(iw[j], p.Ind, p.ind_dtype, pick[j]);
            ok &= t >= 0 && t < (int64_t)p.T;
            at = (int64_t)pb[j] * p.lda_b + t * p.lda_t;
        }
        pv[j] = ok ? (uint32_t)(at * 2) + (((lane & 7) ^ (row & 7)) << 4) : kVoffInvalid;
    }
    auto issue_a = [&](int kt, int stage) {
#pragma unroll
        for (int j = 0; j < PL; ++j) direct_load16(rs_a, pv[j], (uint32_t)kt * 128, smem_stream + stage * L::STAGE + (wave * PL + j) * 1024);
    };
    for (int s = 0; s < min(AHEAD, nk); ++s) issue_a(s, s);

    f32x4 acc[MT][CT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    int stage = 0;
    for (int kt = 0; kt < nk; ++kt) {
        // what may still be on its way: the slabs requested after this one (of the first three the weights came before any rows)
        if (kt + AHEAD > nk) wait_vmem<0>();
        else if (kt == 0) wait_vmem<(AHEAD - 1) * PL>();
        else if (kt == 1) wait_vmem<(AHEAD - 2) * PL + NL>();
        else wait_vmem<(AHEAD - 1) * NL>();
        __syncthreads();            // slab kt is everybody's; nobody reads the stage that is filled next
        if (kt + AHEAD < nk) {
            const int fill = (stage + AHEAD) % L::STAGES;
            issue_a(kt + AHEAD, fill);
            issue_w(kt + AHEAD, fill);
        }
        const char *ta = smem_stream + stage * L::STAGE, *tw = ta + L::A;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            u32x4 mf[MT], nf[CT];
#pragma unroll
            for (int i = 0; i < MT; ++i) mf[i] = *reinterpret_cast<const u32x4 *>(ta + (i * 16 + a) * 128 + (((ks * 4 + g) ^ (a & 7)) << 4));
#pragma unroll
            for (int j = 0; j < CT; ++j) {
                if constexpr (!W_TRANS) {
                    const int row = (wave * CT + j) * 16 + a;
                    nf[j] = *reinterpret_cast<const u32x4 *>(tw + row * 128 + (((ks * 4 + g) ^ (a & 7)) << 4));
                } else if constexpr (WES == 1) {
                    const int row = ks * 32 + g * 8 + (a >> 1);
                    const u32x2 q8 = lds_read_tr8(tw + row * 128 + (((wave * CT + j) ^ ((row >> 1) & 7)) << 4) + (a & 1) * 8);
                    nf[j] = fp8x8_to_bf16_chunk(q8[0], q8[1]);
                } else {
                    const int row = ks * 32 + g * 8 + (a >> 2);
                    const char *at = tw + row * 128 + (((wave * CT + j) ^ (((row >> 1) & 1) | ((row >> 2) & 2))) << 5) + (a & 3) * 8;
                    const u32x2 lo = lds_read_tr16(at), hi = lds_read_tr16(at + 4 * 128);
                    nf[j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                }
            }
#pragma unroll
            for (int j = 0; j < CT; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) mma_chunk<TT>(acc[i][j], nf[j], mf[i]);
        }
        stage = (stage + 1) % L::STAGES;
    }

    // ---------------- results through LDS, out as whole row segments; lane (a, g) holds columns 4 g .. + 3 of row a of a tile
    __syncthreads();
    float *red = reinterpret_cast<float *>(smem_stream);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) *reinterpret_cast<f32x4 *>(red + (i * 16 + a) * L::ORS + (wave * CT + j) * 16 + g * 4) = acc[i][j];
    __syncthreads();
    constexpr int CPR = BN / 4;                                         // four columns at a time
    const int c = (tid % CPR) * 4, n = n0 + c;
    if (n >= N) return;
    f32x4 f = {1.f, 1.f, 1.f, 1.f}, add = {0.f, 0.f, 0.f, 0.f};
    const int64_t at = (int64_t)e * N + n;                              // N % 8 == 0: four columns are inside or outside
    if (p.w_scale != nullptr) f = f32x4{p.w_scale[at], p.w_scale[at + 1], p.w_scale[at + 2], p.w_scale[at + 3]};
    if (p.bias != nullptr) {
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const uint16_t h = reinterpret_cast<const uint16_t *>(p.bias)[at + x];
            add[x] = TT::ID == 2 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
        }
    }
#pragma unroll 1
    for (int r = tid / CPR; r < BM && m0 + r < Me; r += kThreads / CPR) {
        int b;
        char *dst = p.C + (pick_of(m0 + r, b) * p.ldc + n) * (p.out_f32 ? 4 : 2);
        f32x4 v = *reinterpret_cast<const f32x4 *>(red + r * L::ORS + c);
#pragma unroll
        for (int x = 0; x < 4; ++x) v[x] = v[x] * f[x] + add[x];
        if constexpr (WES == 2)
            apply_activation_of<TT>(p.act, [&](auto fn) {
#pragma unroll
                for (int x = 0; x < 4; ++x) v[x] = fn(v[x]);
            });
        if (p.out_f32) *reinterpret_cast<f32x4 *>(dst) = v;
        else *reinterpret_cast<u32x2 *>(dst) = u32x2{pack2<TT>(v[0], v[1]), pack2<TT>(v[2], v[3])};
    }
}

}  // namespace egs
