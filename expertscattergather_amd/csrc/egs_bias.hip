// Biases of the two modules and their gradients, for the launches that do not take them along (the tiled products of
// egs_tiled.h add a bias to what they store).
//
//   gather    Y[b,e,k,:] += bias[e,:]                          dbias[e,:] = sum over the expert's picks of dY[b,e,k,:]
//   scatter   out[b,t,:] += sum over the picks of t of bias[e]   dbias[e,:] = sum over the expert's picks of dOut[b,Ind[b,e,k],:]
//
// Composed from torch operations (a [B,T,E] count of picks filled by scatter_add, a matrix product with it, the broadcast add,
// and autograd's way back through them) these were about fifteen launches and 150 us of the 350 us that a B53 T97 E29 K41
// I111 J75 fp32 step took.  They are sums over small data: a launch each, bound by one pass over the rows they read.
#include "egs_host.h"

namespace egs {
namespace {

template <class TT> __device__ __forceinline__ float elem_at(const char *p, int64_t i)
{
    if constexpr (TT::ES == 4) return reinterpret_cast<const float *>(p)[i];
    else return TT::ID == 2 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p)[i]) : f16_bits_to_f32(reinterpret_cast<const uint16_t *>(p)[i]);
}
template <class TT> __device__ __forceinline__ void put_elem(char *p, int64_t i, float v)
{
    if constexpr (TT::ES == 4) reinterpret_cast<float *>(p)[i] = v;
    else reinterpret_cast<uint16_t *>(p)[i] = (uint16_t)f32_to_elem_bits<TT>(v);
}
// four consecutive elements of a row, `n` of them real
template <class TT> __device__ __forceinline__ f32x4 elems4(const char *p, int64_t at, int n)
{
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
    if (n >= 4) {
        if constexpr (TT::ES == 4) return *reinterpret_cast<const f32x4_any *>(p + at * 4);
        const u32x2 w = *reinterpret_cast<const u32x2_any *>(p + at * 2);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const uint32_t h = (w[x >> 1] >> (16 * (x & 1))) & 0xffffu;
            v[x] = TT::ID == 2 ? bf16_bits_to_f32(h) : f16_bits_to_f32(h);
        }
        return v;
    }
    for (int x = 0; x < n; ++x) v[x] = elem_at<TT>(p, at + x);
    return v;
}

struct BiasParams {
    const char *rows;           // gradient kernel: [B,T,N] source (gathered) or dense [B,E,K,N] rows
    const char *bias;           // [E,N]
    const void *Ind;
    char *out;                  // what is added to, or [E,N] gradients
    int64_t ld_b, ld_t;         // element strides of the gathered source
    int32_t B, T, E, K, N, ind_dtype, gathered;
    int32_t tb, ec;             // scatter: tokens per workgroup, experts counted at a time
};

template <class TT> __global__ __launch_bounds__(kThreads) void bias_rows_kernel(BiasParams p)
{
    const int64_t total = (int64_t)p.B * p.E * p.K * p.N;
    for (int64_t i = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * 4; i < total; i += (int64_t)gridDim.x * kThreads * 4) {
        const int n = (int)min((int64_t)4, total - i);
        const f32x4 v = elems4<TT>(p.out, i, n);
        int64_t pick = i / p.N;
        int col = (int)(i - pick * p.N);
        for (int x = 0; x < n; ++x) {
            put_elem<TT>(p.out, i + x, v[x] + elem_at<TT>(p.bias, (int64_t)(pick / p.K % p.E) * p.N + col));
            if (++col == p.N) { col = 0; ++pick; }
        }
    }
}

// A workgroup owns tb tokens of a batch element: it counts, in LDS, how often each expert picked each of them (integer
// additions: their order does not matter), then a wavefront per token adds the rows of the experts that did, in expert order.
// An output gets one fp32 sum and is rounded once: where the counters do not hold all experts, they are counted again, ec at a
// time, for every four tokens and 256 columns (E6400 K2 I40 otherwise came out rounded three times).
template <class TT> __global__ __launch_bounds__(kThreads) void bias_scatter_kernel(BiasParams p)
{
    extern __shared__ int32_t sh_picks[];               // [tb][ec]
    const int t_blocks = (p.T + p.tb - 1) / p.tb;
    const int b = (int)blockIdx.x / t_blocks, t0 = ((int)blockIdx.x - b * t_blocks) * p.tb;
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
    auto count = [&](int e0) {
        __syncthreads();
        for (int i = tid; i < p.tb * p.ec; i += kThreads) sh_picks[i] = 0;
        __syncthreads();
        const int64_t first = ((int64_t)b * p.E + e0) * p.K, n = (int64_t)min(p.ec, p.E - e0) * p.K;
        for (int64_t q0 = 0; q0 < n; q0 += 4 * kThreads) {
            uint64_t w[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) w[u] = load_index_word(p.Ind, p.ind_dtype, first + min(q0 + u * kThreads + tid, n - 1));
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t q = q0 + u * kThreads + tid;
                const int64_t t = decode_index_word(w[u], p.Ind, p.ind_dtype, first + min(q, n - 1));
                if (q < n && t >= t0 && t < min(t0 + p.tb, p.T)) atomicAdd(&sh_picks[(int)(t - t0) * p.ec + (int)(q / p.K)], 1);
            }
        }
        __syncthreads();
    };
    int counted = -1;                                   // first of the experts whose counts are in LDS
    for (int tl0 = 0; tl0 < p.tb; tl0 += kThreads / 64) {       // (tb is a multiple of the wavefronts)
        const int tl = tl0 + wave;
        const bool exists = t0 + tl < p.T;
        char *row = p.out + ((int64_t)b * p.T + t0 + tl) * p.N * TT::ES;
        for (int c0 = 0; c0 < p.N; c0 += 256) {
            const int col = c0 + lane * 4, live = min(4, p.N - col);
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            bool any = false;
            for (int e0 = 0; e0 < p.E; e0 += p.ec) {
                if (counted != e0) { count(e0); counted = e0; }
                const int ne = exists ? min(p.ec, p.E - e0) : 0;
                for (int i0 = 0; i0 < ne; i0 += 64) {
                    const int mine = i0 + lane < ne ? sh_picks[tl * p.ec + i0 + lane] : 0;
                    uint64_t who = __ballot(mine != 0);
                    any |= who != 0;
                    while (who != 0) {
                        const int l = __ffsll((unsigned long long)who) - 1;
                        who &= who - 1;
                        const float c = (float)__shfl(mine, l);
                        const f32x4 v = live > 0 ? elems4<TT>(p.bias, (int64_t)(e0 + i0 + l) * p.N + col, live) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int x = 0; x < 4; ++x) acc[x] += c * v[x];
                    }
                }
            }
            if (any && live > 0) {
                const f32x4 old = elems4<TT>(row, col, live);
                for (int x = 0; x < live; ++x) put_elem<TT>(row, col + x, old[x] + acc[x]);
            }
        }
    }
}

// Column sums of an expert's rows: a workgroup of 1024 threads per 32 columns, 32 rows side by side and eight of each in flight.
// The rows of 1024 picks at a time are looked up together, the next ones while these are summed, so that the index -> row
// chain is paid once per thousand picks; every load is unconditional (what does not exist reads row 0 and counts zero
// times).  Partial sums are added in a fixed order.
constexpr int kBiasGradThreads = 1024, kBiasGradCols = 32;
template <class TT> __global__ __launch_bounds__(kBiasGradThreads) void bias_grad_kernel(BiasParams p)
{
    constexpr int C = kBiasGradCols, G = kBiasGradThreads / C, U = 8;
    __shared__ float part[G][C + 1];
    __shared__ int64_t row_at[2][kBiasGradThreads];     // element offset of a pick's row, -1: none
    const int c_blocks = (p.N + C - 1) / C;
    const int e = (int)blockIdx.x / c_blocks, cb = (int)blockIdx.x - e * c_blocks;
    const int tid = (int)threadIdx.x, rg = tid / C;
    const int col = min(cb * C + tid % C, p.N - 1), Me = p.B * p.K;
    auto look_up = [&](int m0, int buf) {
        const int m = m0 + tid, mm = min(m, Me - 1), b = mm / p.K;
        const int64_t pick = ((int64_t)b * p.E + e) * p.K + (mm - b * p.K);
        int64_t at = pick * p.N;
        bool ok = m < Me;
        if (p.gathered) {
            const int32_t t = load_token(p.Ind, p.ind_dtype, pick, p.T);
            ok = ok && t >= 0;
            at = b * p.ld_b + (int64_t)t * p.ld_t;
        }
        row_at[buf][tid] = ok ? at : -1;
    };
    float acc = 0.f;
    if (Me > 0) {
        look_up(0, 0);
        for (int m0 = 0, buf = 0; m0 < Me; m0 += kBiasGradThreads, buf ^= 1) {
            __syncthreads();
            if (m0 + kBiasGradThreads < Me) look_up(m0 + kBiasGradThreads, buf ^ 1);
            for (int r0 = 0; r0 < kBiasGradThreads && m0 + r0 < Me; r0 += G * U) {
                float v[U], w[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int64_t at = row_at[buf][r0 + u * G + rg];
                    w[u] = at < 0 ? 0.f : 1.f;
                    v[u] = elem_at<TT>(p.rows, (at < 0 ? 0 : at) + col);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) acc += w[u] != 0.f ? v[u] : 0.f;
            }
        }
    }
    part[rg][tid % C] = acc;
    __syncthreads();
    if (tid < C && cb * C + tid < p.N) {
        float s = 0.f;
#pragma unroll
        for (int r = 0; r < G; ++r) s += part[r][tid];
        put_elem<TT>(p.out, (int64_t)e * p.N + cb * C + tid, s);
    }
}

}  // namespace

namespace host {

#define EGS_BY_TYPE(kernel, grid, threads, lds)                                                                                    \
    do {                                                                                                                           \
        if (act_dtype == EGS_F32) hipLaunchKernelGGL(kernel<ElemF32>, dim3((unsigned)(grid)), dim3(threads), lds, s, p);           \
        else if (act_dtype == EGS_F16) hipLaunchKernelGGL(kernel<ElemF16>, dim3((unsigned)(grid)), dim3(threads), lds, s, p);      \
        else hipLaunchKernelGGL(kernel<ElemBF16>, dim3((unsigned)(grid)), dim3(threads), lds, s, p);                               \
        EGS_CHECK_LAUNCH(#kernel);                                                                                                 \
    } while (0)

static BiasParams bias_params(const egs_dims *d, int N, int ind_dtype)
{
    BiasParams p;
    memset(&p, 0, sizeof(p));
    p.B = d->B; p.T = d->T; p.E = d->E; p.K = d->K; p.N = N; p.ind_dtype = ind_dtype;
    return p;
}

int bias_rows(void *Y, const void *bias, const egs_dims *d, int act_dtype, hipStream_t s)
{
    BiasParams p = bias_params(d, d->J, 0);
    p.out = (char *)Y; p.bias = (const char *)bias;
    const size_t total = (size_t)d->B * d->E * d->K * d->J;
    if (total == 0) return EGS_OK;
    EGS_BY_TYPE(bias_rows_kernel, grid_1d((total + 3) / 4), kThreads, 0);
    return EGS_OK;
}

int bias_scatter(void *Out, const void *bias, const void *Ind, const egs_dims *d, int act_dtype, int ind_dtype, hipStream_t s)
{
    BiasParams p = bias_params(d, d->I, ind_dtype);
    p.out = (char *)Out; p.bias = (const char *)bias; p.Ind = Ind;
    if ((size_t)d->B * d->T * d->I == 0 || (size_t)d->E * d->K == 0) return EGS_OK;
    // 48 KB of counters; more tokens per workgroup (each reads all indices of its batch element) once there are workgroups enough
    p.ec = d->E < 3072 ? d->E : 3072;
    p.tb = 4;
    while (p.tb < 32 && (int64_t)d->B * ceil_div(d->T, p.tb) > 1024 && p.tb * 2 * p.ec <= 12288) p.tb *= 2;
    const int64_t grid = (int64_t)d->B * ceil_div(d->T, p.tb);
    if (grid > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    EGS_BY_TYPE(bias_scatter_kernel, grid, kThreads, (size_t)p.tb * p.ec * 4);
    return EGS_OK;
}

static int bias_grad(BiasParams &p, int act_dtype, hipStream_t s)
{
    if (p.E == 0 || p.N == 0) return EGS_OK;
    const int64_t grid = (int64_t)p.E * ceil_div(p.N, kBiasGradCols);
    if (grid > INT32_MAX / 2) return EGS_ERR_BAD_SHAPE;
    EGS_BY_TYPE(bias_grad_kernel, grid, kBiasGradThreads, 0);
    return EGS_OK;
}

}  // namespace host
}  // namespace egs

using namespace egs;
using namespace egs::host;

static int check_bias_args(const void *rows, const void *Ind, const void *grad, const egs_dims *d, int N, int dtype, int ind_dtype)
{
    if (d == nullptr) return EGS_ERR_NULL_POINTER;
    if (d->B < 0 || d->T < 0 || d->E < 0 || d->K < 0 || N < 0 || (int64_t)d->B * d->K > INT32_MAX) return EGS_ERR_BAD_SHAPE;
    if (!(dtype == EGS_F32 || dtype == EGS_F16 || dtype == EGS_BF16) || ind_dtype < EGS_IND_I16 || ind_dtype > EGS_IND_U8) return EGS_ERR_BAD_DTYPE;
    if ((size_t)d->E * N == 0) return EGS_OK;
    if (grad == nullptr || ((size_t)d->B * d->K > 0 && (rows == nullptr || Ind == nullptr))) return EGS_ERR_NULL_POINTER;
    return EGS_OK;
}

extern "C" int egs_gather_bias_grad(const void *grad_Y, void *grad_bias, const egs_dims *d, int dtype, void *stream)
{
    const int rc = check_bias_args(grad_Y, grad_Y, grad_bias, d, d == nullptr ? 0 : d->J, dtype, EGS_IND_I64);
    if (rc != EGS_OK) return rc;
    BiasParams p = bias_params(d, d->J, 0);
    p.rows = (const char *)grad_Y; p.out = (char *)grad_bias;
    return bias_grad(p, dtype, (hipStream_t)stream);
}

extern "C" int egs_scatter_bias_grad(const void *grad_Out, const void *Ind, void *grad_bias, const egs_dims *d, int64_t ldg_b, int64_t ldg_t,
                                     int dtype, int ind_dtype, void *stream)
{
    const int rc = check_bias_args(grad_Out, Ind, grad_bias, d, d == nullptr ? 0 : d->I, dtype, ind_dtype);
    if (rc != EGS_OK) return rc;
    if (ldg_t < d->I || (d->B > 1 && ldg_b < 0)) return EGS_ERR_BAD_STRIDE;
    BiasParams p = bias_params(d, d->I, ind_dtype);
    p.rows = (const char *)grad_Out; p.Ind = Ind; p.out = (char *)grad_bias; p.gathered = 1; p.ld_b = ldg_b; p.ld_t = ldg_t;
    return bias_grad(p, dtype, (hipStream_t)stream);
}
