// Expert-choice router in one kernel: softmax over the experts, then every expert's K tokens of highest affinity.
//
// The composed form (softmax, a transposed copy, top-K selection, a sort of the selected) is four to six launches that read and
// write the [B,T,E] affinities several times: 51 us at B64 T256 E32 K32, where the logits are 2 MB.  Here a workgroup takes one
// batch element and WV experts, one wavefront each: it reads all of the batch element's logits once (rows lie contiguous, so
// the loads are whole lines; the other workgroups of the batch element find them in the L2), keeps its experts' columns of
// the softmax in LDS, and each wavefront finds the K-th largest value of its column bit by bit from the top (an affinity is a
// non-negative float: its bits order like the value), stopping as soon as exactly K values reach the candidate.  The selected
// are then ranked by counting.  What bounds it is the latency of that chain, not bytes.
#include "egs_host.h"

namespace egs {
namespace {

constexpr int kRouterMaxK = 512;
constexpr int kRouterRowLanes = 16;         // lanes that share a row of logits

struct RouterParams {
    const void *logits;         // [B,T,E]
    void *Ind;                  // [B,E,K]
    float *scores;              // [B,E,K]
    int32_t B, T, E, K;
    int32_t ind_dtype, groups;  // groups of WV experts per batch element
};

__device__ __forceinline__ float logit(const float *p, int64_t i) { return p[i]; }
struct F16Ptr { const uint16_t *p; };
struct BF16Ptr { const uint16_t *p; };
__device__ __forceinline__ float logit(F16Ptr p, int64_t i) { return f16_bits_to_f32(p.p[i]); }
__device__ __forceinline__ float logit(BF16Ptr p, int64_t i) { return bf16_bits_to_f32(p.p[i]); }

// LDS: [WV][T] affinities (as bits), then per wavefront the K selected: their bits, their tokens
size_t router_lds(int WV, int T, int K) { return (size_t)WV * ((((size_t)T + 3) & ~(size_t)3) + 4) * 4 + (size_t)WV * (((size_t)K + 7) & ~(size_t)7) * 8; }

// MAXI: experts per lane of a row held in registers (E <= 16 * MAXI), or 4 and the row is read again
template <class PT, int WV, int MAXI>
__global__ __launch_bounds__(64 * WV) void router_kernel(RouterParams p, PT logits)
{
    extern __shared__ __attribute__((aligned(16))) uint32_t smem_router[];
    const int T = p.T, E = p.E, K = p.K;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the workgroups of a batch element on one XCD: they read the same logits
    const int b = (int)(blockIdx.x & 7) + 8 * (int)(blockIdx.x / (8 * p.groups)), grp = (int)(blockIdx.x >> 3) % p.groups;
    if (b >= p.B) return;
    const int e0 = grp * WV;
    const int stride = ((T + 3) & ~3) + 4, kpad = (K + 7) & ~7;

    // ---- softmax rows: 16 lanes per row, several rows in flight
    constexpr int L = kRouterRowLanes, ROWS = 64 * WV / L, U = 16 / MAXI;
    const int rl = tid % L, rg = tid / L;
    const int64_t base = (int64_t)b * T * E;
    // over the 16 lanes of a row, every lane gets the result: rotations inside a row of lanes (no LDS round trip)
    auto reduce16 = [](float v, auto op) {
        v = op(v, bits_f32(__builtin_amdgcn_update_dpp(0, (int)f32_bits(v), 0x128, 0xf, 0xf, false)));      // row_ror:8
        v = op(v, bits_f32(__builtin_amdgcn_update_dpp(0, (int)f32_bits(v), 0x124, 0xf, 0xf, false)));
        v = op(v, bits_f32(__builtin_amdgcn_update_dpp(0, (int)f32_bits(v), 0x122, 0xf, 0xf, false)));
        v = op(v, bits_f32(__builtin_amdgcn_update_dpp(0, (int)f32_bits(v), 0x121, 0xf, 0xf, false)));
        return v;
    };
    for (int t0 = 0; t0 < T; t0 += U * ROWS) {
        if (E <= L * MAXI) {                            // a row fits the registers of its lanes
            float v[U][MAXI];
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < MAXI; ++i) {
                    const int t = min(t0 + u * ROWS + rg, T - 1), e = rl + i * L;
                    v[u][i] = e < E ? logit(logits, base + (int64_t)t * E + e) : -INFINITY;
                }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                float m = v[u][0];
#pragma unroll
                for (int i = 1; i < MAXI; ++i) m = v[u][i] > m || v[u][i] != v[u][i] ? v[u][i] : m;
                m = reduce16(m, [](float x, float y) { return y > x || y != y ? y : x; });
                float s = 0.f;
#pragma unroll
                for (int i = 0; i < MAXI; ++i) { v[u][i] = rl + i * L < E ? expf(v[u][i] - m) : 0.f; s += v[u][i]; }
                s = reduce16(s, [](float x, float y) { return x + y; });
                const int t = t0 + u * ROWS + rg;
#pragma unroll
                for (int i = 0; i < MAXI; ++i) {
                    const int w = rl + i * L - e0;
                    if (t < T && w >= 0 && w < WV) smem_router[w * stride + t] = f32_bits(v[u][i] / s);
                }
            }
        } else {
            for (int u = 0; u < U; ++u) {
                const int t = t0 + u * ROWS + rg, tt = min(t, T - 1);
                float m = -INFINITY, s = 0.f;
                for (int e = rl; e < E; e += L) { const float x = logit(logits, base + (int64_t)tt * E + e); m = x > m || x != x ? x : m; }
                m = reduce16(m, [](float x, float y) { return y > x || y != y ? y : x; });
                for (int e = rl; e < E; e += L) s += expf(logit(logits, base + (int64_t)tt * E + e) - m);
                s = reduce16(s, [](float x, float y) { return x + y; });
                if (t < T && rl < WV && e0 + rl < E)
                    smem_router[rl * stride + t] = f32_bits(expf(logit(logits, base + (int64_t)t * E + e0 + rl) - m) / s);
            }
        }
    }
    __syncthreads();
    const int e = e0 + wave;
    if (e >= E) return;

    // ---- the K-th largest of this wavefront's column.  A NaN counts as larger than every number.
    uint32_t *col = smem_router + wave * stride;
    // values per lane held in registers: the first four chunks of 64 tokens, sixteen, or none of a longer column
    uint32_t key[16];
    const int chunks = (T + 63) >> 6;
#pragma unroll
    for (int i = 0; i < 16; ++i) key[i] = i < chunks && chunks <= 16 && i * 64 + lane < T ? col[i * 64 + lane] & 0x7fffffffu : 0u;
    auto count = [&](uint32_t cand) -> int {            // values >= cand, cand > 0 (what pads a column is 0)
        int n = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) n += __popcll(__ballot(key[i] >= cand));
        if (chunks <= 4) return n;
        if (chunks <= 16) {
#pragma unroll
            for (int i = 4; i < 16; ++i) n += __popcll(__ballot(key[i] >= cand));
            return n;
        }
        for (int c = 0; c < chunks; ++c) {
            const int t = c * 64 + lane;
            n += __popcll(__ballot(t < T && (col[min(t, T - 1)] & 0x7fffffffu) >= cand));
        }
        return n;
    };
    uint32_t kth = 0;
    int above = T;                                      // values >= kth
    for (int bit = 30; bit >= 0 && above != K; --bit) {
        const int n = count(kth | (1u << bit));
        if (n >= K) { kth |= 1u << bit; above = n; }
    }
    int ties = above - K;                               // of the values equal to kth, this many stay out: those of the highest tokens
    int equal = 0;
    if (ties > 0) equal = above - (kth == 0x7fffffffu ? 0 : count(kth + 1));

    // ---- the selected, in token order
    uint32_t *sel = smem_router + WV * stride + wave * kpad * 2, *sel_t = sel + kpad;
    if (lane < kpad - K) sel[K + lane] = 0u;            // never above anything, and behind everything it equals
    const uint64_t before = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    int have = 0, eq_seen = 0;
    for (int c = 0; c * 64 < T; ++c) {
        const int t = c * 64 + lane;
        const uint32_t v = t < T ? col[t] & 0x7fffffffu : 0u;
        bool in = t < T && v >= kth;
        if (ties > 0) {                                 // uniform
            const bool eq = t < T && v == kth;
            const uint64_t who = __ballot(eq);
            if (eq && eq_seen + __popcll(who & before) >= equal - ties) in = false;
            eq_seen += __popcll(who);
        }
        const uint64_t who = __ballot(in);
        if (in) {
            const int at = have + __popcll(who & before);
            sel[at] = v; sel_t[at] = (uint32_t)t;
        }
        have += __popcll(who);
    }
    __builtin_amdgcn_wave_barrier();
    // ---- ranked by counting, largest first, equal values in token order
    const int64_t out = ((int64_t)b * E + e) * K;
    for (int i0 = 0; i0 < K; i0 += 64) {
        const int i = min(i0 + lane, K - 1);
        const uint32_t v = sel[i], t = sel_t[i];
        int rank = 0;
        for (int j = 0; j < kpad; j += 8) {             // eight values per round trip to LDS, broadcast to the lanes
            const u32x4 lo = *reinterpret_cast<const u32x4 *>(sel + j), hi = *reinterpret_cast<const u32x4 *>(sel + j + 4);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                rank += lo[x] > v || (lo[x] == v && j + x < i) ? 1 : 0;
                rank += hi[x] > v || (hi[x] == v && j + 4 + x < i) ? 1 : 0;
            }
        }
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

template <class PT, int WV, int MAXI>
int launch_router_maxi(RouterParams &p, PT logits, hipStream_t s)
{
    static LdsGrant told;
    const size_t lds = router_lds(WV, p.T, p.K);
    const int rc = allow_large_lds((const void *)router_kernel<PT, WV, MAXI>, told, lds, "hipFuncSetAttribute(router_kernel)");
    if (rc != EGS_OK) return rc;
    p.groups = ceil_div(p.E, WV);
    const int64_t grid = (int64_t)8 * ceil_div(p.B, 8) * p.groups;
    if (grid > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    hipLaunchKernelGGL((router_kernel<PT, WV, MAXI>), dim3((unsigned)grid), dim3(64 * WV), lds, s, p, logits);
    EGS_CHECK_LAUNCH("router_kernel");
    return EGS_OK;
}

template <class PT, int WV>
int launch_router(RouterParams &p, PT logits, hipStream_t s)
{
    if (p.E <= 16) return launch_router_maxi<PT, WV, 1>(p, logits, s);
    return p.E <= 32 ? launch_router_maxi<PT, WV, 2>(p, logits, s) : launch_router_maxi<PT, WV, 4>(p, logits, s);
}

template <class PT>
int launch_router_wv(RouterParams &p, PT logits, hipStream_t s)
{
    // eight experts per workgroup while that gives every CU one; fewer for a small batch (more workgroups) or a long sequence
    // (the columns have to fit in LDS)
    const size_t budget = 150 * 1024;
    if (router_lds(8, p.T, p.K) <= budget && (int64_t)p.B * ceil_div(p.E, 8) >= 256) return launch_router<PT, 8>(p, logits, s);
    if (router_lds(4, p.T, p.K) <= budget) return launch_router<PT, 4>(p, logits, s);
    return EGS_ERR_UNSUPPORTED;
}

}  // namespace
}  // namespace egs

extern "C" int egs_expert_choice_router(const void *logits, void *Ind, float *scores, int32_t B, int32_t T, int32_t E, int32_t K,
                                        int logits_dtype, int ind_dtype, void *stream)
{
    using namespace egs;
    if (B < 0 || T < 0 || E < 0 || K < 0 || K > T) return EGS_ERR_BAD_SHAPE;
    if (!(logits_dtype == EGS_F32 || logits_dtype == EGS_F16 || logits_dtype == EGS_BF16)) return EGS_ERR_BAD_DTYPE;
    if (ind_dtype < EGS_IND_I16 || ind_dtype > EGS_IND_U8) return EGS_ERR_BAD_DTYPE;
    if (B == 0 || E == 0 || K == 0) return EGS_OK;
    if (logits == nullptr || Ind == nullptr || scores == nullptr) return EGS_ERR_NULL_POINTER;
    if (K > kRouterMaxK || router_lds(4, T, K) > 150 * 1024) return EGS_ERR_UNSUPPORTED;
    RouterParams p;
    memset(&p, 0, sizeof(p));
    p.logits = logits; p.Ind = Ind; p.scores = scores;
    p.B = B; p.T = T; p.E = E; p.K = K; p.ind_dtype = ind_dtype;
    hipStream_t s = (hipStream_t)stream;
    if (logits_dtype == EGS_F32) return launch_router_wv<const float *>(p, (const float *)logits, s);
    if (logits_dtype == EGS_F16) return launch_router_wv<F16Ptr>(p, F16Ptr{(const uint16_t *)logits}, s);
    return launch_router_wv<BF16Ptr>(p, BF16Ptr{(const uint16_t *)logits}, s);
}
