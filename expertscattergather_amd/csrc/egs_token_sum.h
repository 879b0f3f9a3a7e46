// Second half of the GEMM-scatter with product rows in memory, without a routing table: every workgroup finds the picks of its
// own few tokens in Ind, puts them in order and adds their product rows up.
//
//   out[b,t,:] = sum of P[b,q,:] over the picks q of batch element b with Ind[b,q] = t, in increasing q
//
// With the table built by a launch of its own (csr_count_kernel, 5 .. 15 us for a few hundred picks: one workgroup per batch
// element, a chain of phases) the table took as long as the sums.  Up to kTokenSumPicks picks per batch element (kTokenSumPicksFew for few tokens) it is cheaper
// that each workgroup reads all of the batch element's indices - a few KB out of the L2, all in flight at once - keeps those
// of its tokens, and sorts what is left, of which there is little.  The order of the additions is the order of the picks; where groups
// of threads share a token's picks (split_log2: few tokens to a workgroup), or all of them those of a token with more than kTokenSumHot each, in
// contiguous shares that are added in order: a function of Ind and the sizes alone, bitwise reproducible.
#pragma once
#include "egs_device.h"

namespace egs {

constexpr int kTokenSumPicks = 4096;        // most picks per batch element
constexpr int kTokenSumPicksFew = 8192;     // where there are few tokens, of short rows (token_sums_take)
constexpr int kTokenSumTokens = 32;         // most tokens per workgroup
constexpr int kTokenSumMany = 128;          // where they have few picks
constexpr int kTokenSumHot = 64;            // picks of a group's token; longer segments are shared by the whole workgroup
constexpr int kTokenSumOne = 32;            // a wavefront's only token: longer segments go sixteen rows at a time

struct TokenSumParams {
    const void *P;              // product rows [B, N, ldp], fp32 or the 16-bit element type
    const void *Ind;            // [B, N]
    char *out;                  // [B, T, I]
    int32_t B, T, N, I, ldp;
    int32_t ind_dtype;
    int32_t tb;                 // tokens per workgroup
    int32_t split_log2;         // groups of threads that share a token's picks
    int32_t tpr_log2;           // 2^tpr_log2 threads share a row (4 columns each)
    int32_t t_blocks, c_blocks; // workgroups per batch element: token blocks x column blocks of 4 << tpr_log2 columns
};

// bytes of LDS: picks of the workgroup's tokens as found, and in order; counters of four wavefronts
__host__ __device__ inline size_t token_sum_lds(int N, int most)
{
    const size_t list = (size_t)4 * (((N + 3) / 4 + 63) / 64 * 64);     // four wavefronts' shares
    return list * 8 + (4 * most + most + 4) * 4 + kThreads * 16;
}

// STREAM: as for segment_sum_body (B29 T216 E69 K40 I1280 J144, 410 MB of rows: the scatter 222 -> 194 us)
// WAVE: 2^tpr_log2 is 64.  (A kernel of its own: with both ways in one the other took 12.2 us instead of 11.1 at B53 T97 E29 K41 I111.)
// TBM: most tokens of a workgroup.  Where a row is less than a wavefront, and with many tokens of few picks, half as many rows on their way leave
// registers for eight workgroups per CU instead of five: bf16 B48 T3785 E11 K5 I64 J147 45 -> 36 us, f16 B95 T3445 E13 K17 I32 J20 63 -> 54.
template <class TT, class PT, bool WAVE, bool STREAM, int TBM, int PICKS = kTokenSumPicks>
__global__ __launch_bounds__(kThreads, PICKS > kTokenSumPicks ? 2 : WAVE && TBM == 32 ? 5 : 8) void token_sum_kernel(TokenSumParams p)
{
    extern __shared__ __attribute__((aligned(16))) char smem_token_sum[];
    const int N = p.N, T = p.T;
    const int share = ((N + 3) / 4 + 63) / 64 * 64;                     // picks a wavefront looks at
    f32x4 *part = reinterpret_cast<f32x4 *>(smem_token_sum);            // [256] partial sums of hot tokens
    int32_t *found = reinterpret_cast<int32_t *>(smem_token_sum + kThreads * 16);       // [4][share] pick | local token << 16, rank in the next
    int32_t *order = found + 4 * share;                                 // picks of the tokens, in order
    int32_t *hist = order + 4 * share;                                  // [4][TBM]
    int32_t *first = hist + 4 * TBM;                                    // [TBM + 1]

    int blk = (int)blockIdx.x;
    const int cb = blk % p.c_blocks;
    blk /= p.c_blocks;
    const int b = blk / p.t_blocks, t0 = (blk - b * p.t_blocks) * p.tb;
    const int tb = min(p.tb, T - t0);
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint64_t before = lane == 0 ? 0ull : (~0ull >> (64 - lane));

    // ---- the picks of this workgroup's tokens, in increasing order, wavefront by wavefront
    const int64_t base = (int64_t)b * N;
    const int q0 = wave * share;
    int have = 0;                                                       // found so far (uniform)
#pragma unroll
    for (int i = 0; i < TBM; i += 64)
        if (i + lane < TBM) hist[wave * TBM + i + lane] = 0;
    constexpr int U = 8;
    for (int c0 = 0; c0 < share; c0 += U * 64) {
        uint64_t w[U];
#pragma unroll
        for (int u = 0; u < U; ++u) w[u] = load_index_word(p.Ind, p.ind_dtype, base + min(q0 + c0 + u * 64 + lane, N - 1));
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int q = q0 + c0 + u * 64 + lane;
            const int64_t t = decode_index_word(w[u], p.Ind, p.ind_dtype, base + min(q, N - 1));
            const bool mine = c0 + u * 64 < share && q < N && t >= t0 && t < t0 + tb;
            const uint64_t who = __ballot(mine);
            if (mine) found[q0 + have + __popcll(who & before)] = q | ((int32_t)(t - t0) << 16);
            have += __popcll(who);
        }
    }
    __builtin_amdgcn_wave_barrier();
    // ---- rank of each among the wavefront's picks of the same token (a wavefront's LDS accesses happen in order)
    for (int c0 = 0; c0 < have; c0 += 64) {
        const int i = c0 + lane;
        const int ent = i < have ? found[q0 + i] : 0;
        const int tl = ent >> 16;
        uint64_t same = __ballot(i < have);
        if (i >= have) same = 0;
#pragma unroll
        for (int bit = 0; bit < (TBM == 32 ? 5 : 7); ++bit) {
            const uint64_t ones = __ballot((tl >> bit) & 1);
            same &= ((tl >> bit) & 1) ? ones : ~ones;
        }
        if (i < have) {
            const int rank = __popcll(same & before), start = hist[wave * TBM + tl];
            order[q0 + i] = start + rank;                               // parked; replaced below
            if ((same >> lane) == 1ull) hist[wave * TBM + tl] = start + __popcll(same);
        }
        __builtin_amdgcn_wave_barrier();
    }
    // ranks into registers before `order` gets its real contents
    constexpr int MAXR = PICKS / 4 / 64;
    int rk[MAXR];
#pragma unroll
    for (int c = 0; c < MAXR; ++c) rk[c] = c * 64 + lane < have ? order[q0 + c * 64 + lane] : 0;
    __syncthreads();
    if (wave == 0) {                                                    // counts -> starts: over wavefronts, then over tokens
        constexpr int PER = (TBM + 63) / 64;                            // tokens of a lane
        static_assert(TBM == 32 || TBM == 128, "");
        int n[PER][4], sum = 0;
        const bool has = lane * PER < TBM;
        if (has) {
#pragma unroll
            for (int i = 0; i < PER; ++i)
#pragma unroll
                for (int w = 0; w < 4; ++w) { n[i][w] = hist[w * TBM + lane * PER + i]; sum += n[i][w]; }
        }
        int incl = sum;
#pragma unroll
        for (int d = 1; d < TBM / PER; d <<= 1) {
            const int o = __shfl_up(incl, d);
            if (lane >= d) incl += o;
        }
        if (has) {
            int at = incl - sum;
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                first[lane * PER + i] = at;
#pragma unroll
                for (int w = 0; w < 4; ++w) { hist[w * TBM + lane * PER + i] = at; at += n[i][w]; }
            }
            if (lane == TBM / PER - 1) first[TBM] = incl;
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < MAXR; ++c)
        if (c * 64 + lane < have) {
            const int ent = found[q0 + c * 64 + lane];
            order[hist[wave * TBM + (ent >> 16)] + rk[c]] = ent & 0xffff;
        }
    __syncthreads();

    // ---- sums: 2^tpr_log2 threads per token, four columns each
    const int tpr = 1 << p.tpr_log2, groups = kThreads >> p.tpr_log2;
    const int grp = tid >> p.tpr_log2, ct = tid & (tpr - 1);
    const int col = (cb * tpr + ct) * 4;
    const bool live = col < p.I;
    const PT *Pb = reinterpret_cast<const PT *>(p.P) + base * p.ldp + (live ? col : 0);
    typedef typename std::conditional<sizeof(PT) == 4, f32x4, u32x2>::type vec_t;
    auto add = [&](f32x4 &acc, const vec_t &v) {
        if constexpr (sizeof(PT) == 4) {
#pragma unroll
            for (int x = 0; x < 4; ++x) acc[x] += v[x];
        } else {
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                const uint32_t h = (v[x >> 1] >> (16 * (x & 1))) & 0xffffu;
                acc[x] += TT::ID == 2 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
            }
        }
    };
    auto row = [&](int64_t q) -> vec_t {
        const vec_t *at = reinterpret_cast<const vec_t *>(Pb + q * p.ldp);
        if constexpr (STREAM) return __builtin_nontemporal_load(at);
        else return *at;
    };
    auto sum_of = [&](int s0, int s1, f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f}) -> f32x4 {
        constexpr int LB = (WAVE && TBM == 32) || PICKS > kTokenSumPicks ? 16 : 8, RB = 4;
        int s = s0;
        for (; s + LB <= s1; s += LB) {
            vec_t v[LB];
#pragma unroll
            for (int u = 0; u < LB; ++u) v[u] = row(order[s + u]);
#pragma unroll
            for (int u = 0; u < LB; ++u) add(acc, v[u]);
        }
        for (; s < s1; s += RB) {
            vec_t v[RB];
#pragma unroll
            for (int u = 0; u < RB; ++u) v[u] = row(order[min(s + u, s1 - 1)]);
#pragma unroll
            for (int u = 0; u < RB; ++u)
                if (s + u < s1) add(acc, v[u]);
        }
        return acc;
    };
    auto store = [&](int tl, const f32x4 &acc) {
        if (!live) return;
        char *dst = p.out + (((int64_t)b * T + t0 + tl) * p.I + col) * TT::ES;
        if (col + 4 <= p.I) {
            if constexpr (TT::ES == 4) *reinterpret_cast<f32x4 __attribute__((aligned(4))) *>(dst) = acc;
            else *reinterpret_cast<u32x2 __attribute__((aligned(2))) *>(dst) = u32x2{pack2<TT>(acc[0], acc[1]), pack2<TT>(acc[2], acc[3])};
        } else {
            for (int x = 0; col + x < p.I; ++x) {
                if constexpr (TT::ES == 4) reinterpret_cast<float *>(dst)[x] = acc[x];
                else reinterpret_cast<uint16_t *>(dst)[x] = (uint16_t)f32_to_elem_bits<TT>(acc[x]);
            }
        }
    };
    // Where a wavefront is a token's group it takes neighbouring tokens, whose picks follow one another, and has eight rows on their
    // way, whichever they are for; token by token, of two or three rows each, it waited for memory once for every token.  us, fp32 rows:
    // B5 T2250 E28 K24 I928 21.9 -> 14.7, B71 T1000 E12 K10 I160 23.6 -> 18.4, B62 T394 E31 K43 I386 37.5 -> 31.6, B4 T512 E256 K8 I2048
    // 20.0 -> 15.7, B6 T1100 E20 K150 I328 14.4 -> 12.5.  Not where a
    // wavefront has one token only, of more than kTokenSumOne picks, or two and one is hot: sixteen rows on their way are worth more there
    // (scatters under Zipf routing, one token at a time / in runs, B1 T315 E4 K44 I576 10.9 / 12.1, B10 T58 E7 K22 I672 14.9 / 15.6).  With more tokens
    // the hot ones are left out of the runs (B33 T3048 E4 K123 I192 39.3 -> 36.3).
    bool hot = false, some = false;
    if constexpr (WAVE)
        for (int i = lane; i < tb; i += 64) {
            const int len = first[i + 1] - first[i];
            hot = hot || len > kTokenSumHot;
            some = some || len > kTokenSumOne;
        }
    const bool runs = WAVE && p.split_log2 == 0 && (p.tb >= 4 * groups || __ballot(p.tb > groups ? hot : some) == 0);
    if (runs) {
        const int each = (tb + groups - 1) / groups, tl1 = min(tb, (wave + 1) * each), from = min(tb, wave * each);
        const int begins = first[min(from + lane, TBM)], ends = first[min(from + lane, TBM - 1) + 1];       // of token `from + lane`: at most 32 are this wavefront's
        const uint64_t hots = __ballot(from + lane < tl1 && ends - begins > kTokenSumHot);
        int tl = from;
        while (tl < tl1) {
            const uint64_t later = hots >> (tl - from);
            const int stop = later != 0 ? tl + (int)__builtin_ctzll(later) : tl1;       // the next hot token or the end
            int s = __builtin_amdgcn_readfirstlane(first[tl]);
            const int end = __builtin_amdgcn_readfirstlane(first[stop]);
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            int here = __builtin_amdgcn_readlane(ends, tl - from);
            auto next = [&]() {
                store(tl, acc);
                acc = f32x4{0.f, 0.f, 0.f, 0.f};
                ++tl;
                here = __builtin_amdgcn_readlane(ends, (tl - from) & 63);
            };
            constexpr int FB = 8;
            for (; s < end; s += FB) {
                const int q = order[min(s + (lane & (FB - 1)), end - 1)];
                vec_t v[FB];
#pragma unroll
                for (int u = 0; u < FB; ++u) v[u] = row(__builtin_amdgcn_readlane(q, u));
#pragma unroll
                for (int u = 0; u < FB; ++u) {
                    if (s + u >= end) break;
                    while (s + u >= here) next();
                    add(acc, v[u]);
                }
            }
            while (tl < stop) next();
            tl = stop + 1;
        }
        if (__ballot(hot) == 0) return;
    }
    const int hot_from = kTokenSumHot << p.split_log2;
    if (p.split_log2 > 0) {
        const int tl = grp >> p.split_log2, at = grp & ((1 << p.split_log2) - 1);
        const int s0 = first[min(tl, tb - 1)], len = tl < tb ? first[tl + 1] - s0 : 0;
        const int each = (len + (1 << p.split_log2) - 1) >> p.split_log2;
        if (len <= hot_from) part[tid] = sum_of(s0 + min(len, at * each), s0 + min(len, (at + 1) * each));
        __syncthreads();
        if (at == 0 && tl < tb && len <= hot_from) {
            f32x4 acc = part[tid];
            for (int gi = 1; gi < 1 << p.split_log2; ++gi) {
                const f32x4 v = part[(gi << p.tpr_log2) + tid];
                acc[0] += v[0]; acc[1] += v[1]; acc[2] += v[2]; acc[3] += v[3];
            }
            store(tl, acc);
        }
    } else if (!runs)
        for (int tl = grp; tl < tb; tl += groups) {
            const int s0 = first[tl], s1 = first[tl + 1];
            if (groups > 1 && s1 - s0 > kTokenSumHot) continue;
            store(tl, sum_of(s0, s1));
        }
    for (int tl = 0; tl < tb; ++tl) {                                   // hot tokens: a share of the segment per group
        const int s0 = first[tl], len = first[tl + 1] - s0;
        if (len <= hot_from) continue;                                  // uniform
        const int each = (len + groups - 1) / groups;
        __syncthreads();
        part[tid] = sum_of(s0 + min(len, grp * each), s0 + min(len, (grp + 1) * each));
        __syncthreads();
        if (grp == 0) {
            f32x4 acc = part[ct];
            for (int gi = 1; gi < groups; ++gi) {
                const f32x4 v = part[gi * tpr + ct];
                acc[0] += v[0]; acc[1] += v[1]; acc[2] += v[2]; acc[3] += v[3];
            }
            store(tl, acc);
        }
    }
}

}  // namespace egs
