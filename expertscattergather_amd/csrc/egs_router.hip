// Expert-choice router: softmax over the experts, then every expert's K tokens of highest affinity.
//
// The composed form (softmax, a transposed copy, top-K selection, a sort of the selected) is four to six launches that read and
// write the [B,T,E] affinities several times: 51 us at B64 T256 E32 K32, where the logits are 2 MB.  Here a workgroup takes one
// batch element and WV experts, WPE wavefronts each: it reads all of the batch element's logits (rows lie contiguous; the other
// workgroups of the batch element find them in the L2), keeps its experts' columns of the softmax in LDS, and finds the K-th
// largest value of each column bit by bit from the top (an affinity is a non-negative float: its bits order like the value),
// stopping as soon as exactly K values reach the candidate.  The selected are then ranked by counting.
//
// What bounds it is vector instructions and the latency of that chain, not bytes.  Every workgroup of a batch element computes all
// of its rows' exponentials, which is the cheaper way for small logits; for large ones router_stats_kernel leaves each row's maximum
// and sum in memory first.
#include "egs_host.h"

namespace egs {
namespace {

constexpr int kRouterMaxK = 512;
constexpr int kRouterRowLanes = 4;          // lanes that share a row of logits
// Where each workgroup computes the exponentials of all rows itself: as long as a batch element's take less than about 9 us (14
// vector instructions for each of T * E / 64, on the four units of a compute unit), the device's together no more, and a row's
// lanes can hold their values without giving up wavefronts.  Elsewhere another launch is cheaper (B1 T210 E83: 9.7 us with it, 12.3
// without; B128 T300 E64: 29 and 36; B64 T512 E32: 19 and 15).
constexpr int64_t kRouterOwnRows = 96 * 1024, kRouterOwnAll = 16 * 1024 * 1024;
constexpr int kRouterOwnE = 64;

struct RouterParams {
    const void *logits;         // [B,T,E]
    void *Ind;                  // [B,E,K]
    float *scores;              // [B,E,K]
    float2 *stats;              // [B,T] maximum and sum of exponentials, or nullptr: each workgroup's own
    int32_t B, T, E, K;
    int32_t ind_dtype, groups;  // groups of WV experts per batch element
};

__device__ __forceinline__ float logit(const float *p, int64_t i) { return p[i]; }
struct F16Ptr { const uint16_t *p; };
struct BF16Ptr { const uint16_t *p; };
__device__ __forceinline__ float logit(F16Ptr p, int64_t i) { return f16_bits_to_f32(p.p[i]); }
__device__ __forceinline__ float logit(BF16Ptr p, int64_t i) { return bf16_bits_to_f32(p.p[i]); }

// LDS: [WV][T] affinities (as bits; the columns of four experts start 16 banks apart), then per expert the K selected: their bits,
// their tokens; then the wavefronts' counts
__host__ __device__ constexpr int router_stride(int T) { return ((T + 63) & ~63) + 16; }
constexpr size_t kRouterCounts = 4 * 16 * 4;
size_t router_lds(int WV, int T, int K) { return (size_t)WV * router_stride(T) * 4 + (size_t)WV * (((size_t)K + 7) & ~(size_t)7) * 8 + kRouterCounts; }

// Each row's maximum and sum of exponentials: 16 lanes per row.  A NaN need not pass through the maximum: the sum has it.
template <class PT>
__global__ __launch_bounds__(256) void router_stats_kernel(RouterParams p, PT logits)
{
    const int rl = (int)threadIdx.x & 15;
    const int64_t row = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4), rows = (int64_t)p.B * p.T;
    const int64_t at = (row < rows ? row : rows - 1) * p.E;
    float v[8], m = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = logit(logits, at + min(rl + i * 16, p.E - 1));      // (the last again: no matter to a maximum)
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fmaxf(m, v[i]);
    for (int e = rl + 128; e < p.E; e += 16) m = fmaxf(m, logit(logits, at + e));
#pragma unroll
    for (int x = 8; x > 0; x /= 2) m = fmaxf(m, __shfl_xor(m, x));
    // the sum in torch's order (every 64th expert in turn, then pairwise, the furthest first), and so its bits
    float q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        q[i] = rl + i * 16 < p.E ? expf(v[i] - m) : 0.f;
        q[i] += rl + i * 16 + 64 < p.E ? expf(v[i + 4] - m) : 0.f;
        for (int e = rl + i * 16 + 128; e < p.E; e += 64) q[i] += expf(logit(logits, at + e) - m);
    }
    float s = (q[0] + q[2]) + (q[1] + q[3]);
#pragma unroll
    for (int x = 8; x > 0; x /= 2) s += __shfl_xor(s, x);
    if (rl == 0 && row < rows) p.stats[row] = float2{m, s};
}

// MAXI: experts per lane of a row (E <= 4 * MAXI), or 0: the rows' maxima and sums are in p.stats
template <class PT, int WV, int WPE, int MAXI>
__global__ __launch_bounds__(64 * WV * WPE) void router_kernel(RouterParams p, PT logits)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t smem_router[];
    const int T = p.T, E = p.E, K = p.K;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the workgroups of a batch element on one XCD: they read the same logits
    const int b = (int)(blockIdx.x & 7) + 8 * (int)(blockIdx.x / (8 * p.groups)), grp = (int)(blockIdx.x >> 3) % p.groups;
    if (b >= p.B) return;
    const int e0 = grp * WV;
    const int stride = router_stride(T), kpad = (K + 7) & ~7;
    const int64_t base = (int64_t)b * T * E;

    if constexpr (MAXI == 0) {
        for (int t = tid; t < T; t += 64 * WV * WPE) {
            const float2 ms = p.stats[(int64_t)b * T + t];
            float v[WV];
#pragma unroll
            for (int w = 0; w < WV; ++w) v[w] = logit(logits, base + (int64_t)t * E + min(e0 + w, E - 1));
#pragma unroll
            for (int w = 0; w < WV; ++w) smem_router[w * stride + t] = f32_bits(expf(v[w] - ms.x) / ms.y);
        }
    } else {
        // four lanes per row, several rows in flight.  An expert e is value e / 4 of lane e % 4: this workgroup's are
        // in one of them or WV / 4 in each.  A NaN need not pass through the maximum: the sum has it.
        constexpr int L = kRouterRowLanes, ROWS = 64 * WV * WPE / L, U = MAXI <= 8 ? 4 : 2;
        constexpr int OWN = WV < L ? 1 : WV / L;        // of this workgroup's experts, those in one lane
        const int rl = tid % L, rg = tid / L;
        auto reduce4 = [](float v, auto op) {           // every lane of the four gets the result (no LDS round trip)
            v = op(v, bits_f32(__builtin_amdgcn_update_dpp(0, (int)f32_bits(v), 0x4e, 0xf, 0xf, false)));       // quad_perm 2 3 0 1
            v = op(v, bits_f32(__builtin_amdgcn_update_dpp(0, (int)f32_bits(v), 0xb1, 0xf, 0xf, false)));       // quad_perm 1 0 3 2
            return v;
        };
        for (int t0 = 0; t0 < T; t0 += U * ROWS) {
            float v[U][MAXI];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < MAXI; ++i) {
                    const int t = min(t0 + u * ROWS + rg, T - 1), e = rl + i * L;
                    v[u][i] = logit(logits, base + (int64_t)t * E + min(e, E - 1));     // (the last again: no matter to a maximum)
                }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float m = v[u][0];
#pragma unroll
                for (int i = 1; i < MAXI; ++i) m = fmaxf(m, v[u][i]);
                m = reduce4(m, [](float x, float y) { return fmaxf(x, y); });
                float own[OWN];
#pragma unroll
                for (int i = 0; i < MAXI; ++i) {
                    float x = expf(v[u][i] - m);
                    v[u][i] = x = rl + i * L < E ? x : 0.f;
#pragma unroll
                    for (int w = 0; w < OWN; ++w) own[w] = i == 0 || e0 / L + w == i ? x : own[w];
                }
                // added pairwise, the furthest experts first: torch's order, and so its bits, and so the same picks
#pragma unroll
                for (int h = MAXI / 2; h > 0; h /= 2)
#pragma unroll
                    for (int i = 0; i < h; ++i) v[u][i] += v[u][i + h];
                const float s = reduce4(v[u][0], [](float x, float y) { return x + y; });
                const int t = t0 + u * ROWS + rg;
#pragma unroll
                for (int w = 0; w < OWN; ++w) {
                    const int at = w * L + rl - e0 % L;
                    if (t < T && (WV >= L || at == 0)) smem_router[at * stride + t] = f32_bits(own[w] / s);
                }
            }
        }
    }
    __syncthreads();
    const int slot = wave / WPE, part = wave % WPE, e = e0 + slot;
    if (WPE == 1 && e >= E) return;

    // ---- the K-th largest of this expert's column.  A NaN counts as larger than every number.  Each of the expert's wavefronts
    // counts in a run of chunks of 64 tokens: the first four of them or sixteen in registers, or none of a longer column
    uint32_t *col = smem_router + slot * stride;
    uint32_t key[16];
    const int chunks = (T + 63) >> 6, mine = (chunks + WPE - 1) / WPE, c0 = part * mine, c1 = min(c0 + mine, chunks);
    const bool held = mine <= 16;
#pragma unroll
    for (int i = 0; i < 16; ++i) key[i] = held && c0 + i < c1 && (c0 + i) * 64 + lane < T ? col[(c0 + i) * 64 + lane] & 0x7fffffffu : 0u;
    auto count = [&](uint32_t cand) -> int {            // of this wavefront's, values >= cand, cand > 0 (what pads a column is 0)
        int n = 0;
        if (!held) {
            for (int c = c0; c < c1; ++c) {
                const int t = c * 64 + lane;
                n += __popcll(__ballot(t < T && (col[min(t, T - 1)] & 0x7fffffffu) >= cand));
            }
            return n;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) n += __popcll(__ballot(key[i] >= cand));
        if (mine <= 4) return n;
#pragma unroll
        for (int i = 4; i < 16; ++i) n += __popcll(__ballot(key[i] >= cand));
        return n;
    };
    uint32_t *sel = smem_router + WV * stride + slot * kpad * 2, *sel_t = sel + kpad;
    int *shared_n = reinterpret_cast<int *>(smem_router + WV * stride + WV * kpad * 2);     // two sets in turn: one barrier per count
    uint32_t kth = 0;
    if constexpr (WPE == 1) {
        int above = T;                                  // values >= kth
        for (int bit = 30; bit >= 0 && above != K; --bit) {
            const int n = count(kth | (1u << bit));
            if (n >= K) { kth |= 1u << bit; above = n; }
        }
    } else {
        // a wavefront that has found its value goes on as one of those that wait: all leave the loop together
        static_assert(WV * WPE <= 16 && (WPE == 4 || WPE == 16), "room for the counts; they are added up in rows of 4 or 16 lanes");
        int above = e < E ? T : K;
        for (int bit = 30; bit >= 0; --bit) {
            int *set = shared_n + (bit & 1) * (WV * WPE);
            const bool found = above == K;
            const int n = found ? -1 : count(kth | (1u << bit));
            if (lane == 0) set[wave] = n;
            __syncthreads();
            int all = set[lane & (WV * WPE - 1)];
            if (__ballot(all >= 0) == 0) break;
            all += __builtin_amdgcn_update_dpp(0, all, 0xb1, 0xf, 0xf, false);              // quad_perm 1 0 3 2
            all += __builtin_amdgcn_update_dpp(0, all, 0x4e, 0xf, 0xf, false);              // quad_perm 2 3 0 1
            if constexpr (WPE == 16) {
                all += __builtin_amdgcn_update_dpp(0, all, 0x124, 0xf, 0xf, false);         // row_ror:4
                all += __builtin_amdgcn_update_dpp(0, all, 0x128, 0xf, 0xf, false);         // row_ror:8
            }
            const int sum = __builtin_amdgcn_readlane(all, slot * WPE);
            if (!found && sum >= K) { kth |= 1u << bit; above = sum; }
        }
    }
    // ---- how many are larger and how many equal, here and in the expert's wavefronts before this one.  Of the equal ones those of
    // the lowest tokens are taken.
    int larger = 0, equal = 0, larger_before = 0, equal_before = 0;
    for (int c = c0; c < c1; ++c) {
        const int t = c * 64 + lane;
        const uint32_t v = t < T ? col[t] & 0x7fffffffu : 0u;
        larger += __popcll(__ballot(t < T && v > kth));
        equal += __popcll(__ballot(t < T && v == kth));
    }
    if constexpr (WPE > 1) {
        int *set = shared_n + 2 * (WV * WPE);
        if (lane == 0) { set[wave] = larger; set[WV * WPE + wave] = equal; }
        __syncthreads();
        larger = 0;
#pragma unroll
        for (int w = 0; w < WPE; ++w) {
            const int l = set[slot * WPE + w], q = set[WV * WPE + slot * WPE + w];
            larger += l;
            larger_before += w < part ? l : 0;
            equal_before += w < part ? q : 0;
        }
    }
    const int take = K - larger;

    // ---- the selected, in token order
    if (part == 0 && lane < kpad - K) sel[K + lane] = 0u;               // never above anything, and behind everything it equals
    const uint64_t before = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int c = c0; c < c1 && e < E; ++c) {
        const int t = c * 64 + lane;
        const uint32_t v = t < T ? col[t] & 0x7fffffffu : 0u;
        const uint64_t gt = __ballot(t < T && v > kth), eq = __ballot(t < T && v == kth);
        const int eq_at = equal_before + __popcll(eq & before);
        if ((t < T && v > kth) || (t < T && v == kth && eq_at < take)) {
            const int at = larger_before + __popcll(gt & before) + min(eq_at, take);
            sel[at] = v; sel_t[at] = (uint32_t)t;
        }
        larger_before += __popcll(gt);
        equal_before += __popcll(eq);
    }
    if constexpr (WPE > 1) {
        __syncthreads();
        if (e >= E) return;
    } else __builtin_amdgcn_wave_barrier();
    // ---- ranked by counting, largest first, equal values in token order
    const int64_t out = ((int64_t)b * E + e) * K;
    for (int i0 = part * 64; i0 < K; i0 += 64 * WPE) {
        const int i = min(i0 + lane, K - 1);
        const uint32_t v = sel[i], t = sel_t[i];
        int rank = 0;
        auto against = [&](int from, int to, auto before) {             // eight values per round trip to LDS, broadcast to the lanes
            for (int j = from; j < to; j += 8) {
                const u32x4 lo = *reinterpret_cast<const u32x4 *>(sel + j), hi = *reinterpret_cast<const u32x4 *>(sel + j + 4);
#pragma unroll
                for (int x = 0; x < 4; ++x) rank += (before(lo[x], j + x) ? 1 : 0) + (before(hi[x], j + 4 + x) ? 1 : 0);
            }
        };
        against(0, i0, [&](uint32_t x, int) { return x >= v; });
        against(i0, min(i0 + 64, kpad), [&](uint32_t x, int j) { return x > v || (x == v && j < i); });
        against(i0 + 64, kpad, [&](uint32_t x, int) { return x > v; });
        if (i0 + lane < K) {
            p.scores[out + rank] = bits_f32(v);
            switch (p.ind_dtype) {
            case EGS_IND_I16: reinterpret_cast<int16_t *>(p.Ind)[out + rank] = (int16_t)t; break;
            case EGS_IND_I32: reinterpret_cast<int32_t *>(p.Ind)[out + rank] = (int32_t)t; break;
            case EGS_IND_U8: reinterpret_cast<uint8_t *>(p.Ind)[out + rank] = (uint8_t)t; break;
            default: reinterpret_cast<int64_t *>(p.Ind)[out + rank] = (int64_t)t; break;
            }
        }
    }
}

using namespace egs::host;

template <class PT, int WV, int WPE, int MAXI>
int launch_router_maxi(RouterParams &p, PT logits, hipStream_t s)
{
    static LdsGrant told;
    const size_t lds = router_lds(WV, p.T, p.K);
    const int rc = allow_large_lds((const void *)router_kernel<PT, WV, WPE, MAXI>, told, lds, "hipFuncSetAttribute(router_kernel)");
    if (rc != EGS_OK) return rc;
    p.groups = ceil_div(p.E, WV);
    const int64_t grid = (int64_t)8 * ceil_div(p.B, 8) * p.groups;
    if (grid > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    hipLaunchKernelGGL((router_kernel<PT, WV, WPE, MAXI>), dim3((unsigned)grid), dim3(64 * WV * WPE), lds, s, p, logits);
    EGS_CHECK_LAUNCH("router_kernel");
    return EGS_OK;
}

template <class PT, int WV, int WPE>
int launch_router(RouterParams &p, PT logits, hipStream_t s)
{
    if (p.stats != nullptr) {
        const int64_t grid = ((int64_t)p.B * p.T + 15) / 16;
        if (grid > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
        hipLaunchKernelGGL(router_stats_kernel<PT>, dim3((unsigned)grid), dim3(256), 0, s, p, logits);
        EGS_CHECK_LAUNCH("router_stats_kernel");
        return launch_router_maxi<PT, WV, WPE, 0>(p, logits, s);
    }
    if (p.E <= 16) return launch_router_maxi<PT, WV, WPE, 4>(p, logits, s);
    if (p.E <= 32) return launch_router_maxi<PT, WV, WPE, 8>(p, logits, s);
    return launch_router_maxi<PT, WV, WPE, 16>(p, logits, s);
}

template <class PT>
int launch_router_wv(RouterParams &p, PT logits, hipStream_t s)
{
    // One wavefront per expert holds a column of up to 1024 tokens in registers and needs no barrier: the way for a short column
    // and where there are workgroups enough (of eight experts: fewer read the same rows).  With few experts in all, several
    // wavefronts count a column and rank the selected, each expert on a compute unit of its own (B3 T667 E7 K229: 15 us, 26 with
    // one wavefront; B2 T2878 E10 K6: 16 us with sixteen, 19 with four); with many and long columns, four of each of four experts
    // (B8 T4096 E100 K128: 36 us, 50 with sixteen of one).
    if (router_lds(4, p.T, p.K) > 150 * 1024) return EGS_ERR_UNSUPPORTED;
    const int64_t experts = (int64_t)p.B * p.E;
    if (p.K <= 128 && (p.T <= 256 || (p.T <= 1024 && experts > 512)))
        return experts > 8 * 255 || p.T > 256 ? launch_router<PT, 8, 1>(p, logits, s) : launch_router<PT, 4, 1>(p, logits, s);
    if (p.T > 4096 || (p.T > 1024 && experts <= 512)) return launch_router<PT, 1, 16>(p, logits, s);
    return experts <= 512 ? launch_router<PT, 1, 4>(p, logits, s) : launch_router<PT, 4, 4>(p, logits, s);
}

}  // namespace
}  // namespace egs

extern "C" size_t egs_expert_choice_router_workspace_bytes(int32_t B, int32_t T, int32_t E)
{
    const int64_t rows = (int64_t)T * E, all = rows * B * ((E + 7) / 8);
    return rows <= egs::kRouterOwnRows && all <= egs::kRouterOwnAll && E <= egs::kRouterOwnE ? 0 : (size_t)B * T * sizeof(float2);
}

extern "C" int egs_expert_choice_router(const void *logits, void *Ind, float *scores, void *workspace, size_t workspace_bytes, int32_t B,
                                        int32_t T, int32_t E, int32_t K, int logits_dtype, int ind_dtype, void *stream)
{
    using namespace egs;
    if (B < 0 || T < 0 || E < 0 || K < 0 || K > T) return EGS_ERR_BAD_SHAPE;
    if (!(logits_dtype == EGS_F32 || logits_dtype == EGS_F16 || logits_dtype == EGS_BF16)) return EGS_ERR_BAD_DTYPE;
    if (ind_dtype < EGS_IND_I16 || ind_dtype > EGS_IND_U8) return EGS_ERR_BAD_DTYPE;
    if (B == 0 || E == 0 || K == 0) return EGS_OK;
    if (logits == nullptr || Ind == nullptr || scores == nullptr) return EGS_ERR_NULL_POINTER;
    const size_t need = egs_expert_choice_router_workspace_bytes(B, T, E);
    if (need > 0 && workspace == nullptr) return EGS_ERR_NULL_POINTER;
    if (need > workspace_bytes) return EGS_ERR_WORKSPACE;
    if (K > kRouterMaxK || router_lds(4, T, K) > 150 * 1024) return EGS_ERR_UNSUPPORTED;
    RouterParams p;
    memset(&p, 0, sizeof(p));
    p.logits = logits; p.Ind = Ind; p.scores = scores; p.stats = need > 0 ? (float2 *)workspace : nullptr;
    p.B = B; p.T = T; p.E = E; p.K = K; p.ind_dtype = ind_dtype;
    hipStream_t s = (hipStream_t)stream;
    if (logits_dtype == EGS_F32) return launch_router_wv<const float *>(p, (const float *)logits, s);
    if (logits_dtype == EGS_F16) return launch_router_wv<F16Ptr>(p, F16Ptr{(const uint16_t *)logits}, s);
    return launch_router_wv<BF16Ptr>(p, BF16Ptr{(const uint16_t *)logits}, s);
}
