// Decoder-caller support outside the quantized matrix path: the fp32 ops the
// C++ Model runs between its quantized projections, with the reference's
// arithmetic (cpp/src/ops.cpp), so the device forward tracks the reference's
// CPU forward closely:
//   rmsnorm    ops.cpp:272-290  sum of squares in double, scale = 1/sqrt(float(ss/d) + eps), x * scale * w
//   silu, mul  ops.cpp:86-100   v / (1 + exp(-v)), then the product in float
//   attention  ops.cpp:206-270  causal, scores float(dot) * scale with the dot in double,
//                               float exp, double denominator, double sums of double(e) * inv * v
// rmsnorm and silu*mul take one workgroup per row. Attention runs on the fp64
// matrix cores for head sizes 32, 64, 96 and 128, else one workgroup per
// (query, head).
#include <hip/hip_runtime.h>

#include "nq_device.hpp"
#include "nq_internal.hpp"

namespace nq {
namespace {

constexpr int kOpsThreads = 256;

// Sum of a double over the workgroup, a fixed-order tree in LDS.
__device__ double block_sum_f64(double v, double* red) {
    const int tid = threadIdx.x;
    red[tid] = v;
    __syncthreads();
    for (int s = kOpsThreads / 2; s > 0; s >>= 1) {
        if (tid < s) red[tid] += red[tid + s];
        __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
}

__device__ float block_max_f32(float v, float* red) {
    const int tid = threadIdx.x;
    red[tid] = v;
    __syncthreads();
    for (int s = kOpsThreads / 2; s > 0; s >>= 1) {
        if (tid < s) red[tid] = red[tid + s] > red[tid] ? red[tid + s] : red[tid];
        __syncthreads();
    }
    const float r = red[0];
    __syncthreads();
    return r;
}

// One workgroup per row. With r: h = x + r is stored (the residual add that
// precedes the norm; h may be x) and the norm runs on h.
__global__ __launch_bounds__(kOpsThreads) void rmsnorm_f32_kernel(const float* x, const float* r, float* h,
                                                                  const float* __restrict__ w, float eps, int k,
                                                                  float* y) {
    __shared__ double red[kOpsThreads];
    const size_t off = static_cast<size_t>(blockIdx.x) * k;
    double ss = 0.0;
    for (int c = threadIdx.x; c < k; c += kOpsThreads) {
        float v = x[off + c];
        if (r) {
            v = v + r[off + c];
            h[off + c] = v;
        }
        ss += static_cast<double>(v) * static_cast<double>(v);
    }
    ss = block_sum_f64(ss, red);
    const float scale = __fdiv_rn(1.0f, __fsqrt_rn(static_cast<float>(ss / k) + eps));
    const float* src = r ? h : x;
    for (int c = threadIdx.x; c < k; c += kOpsThreads) y[off + c] = src[off + c] * scale * w[c];
}

__global__ __launch_bounds__(kOpsThreads) void silu_mul_f32_kernel(const float* __restrict__ g,
                                                                   const float* __restrict__ u, int64_t ld, int k,
                                                                   float* __restrict__ y) {
    const size_t in = static_cast<size_t>(blockIdx.x) * ld, out = static_cast<size_t>(blockIdx.x) * k;
    for (int c = threadIdx.x; c < k; c += kOpsThreads) {
        const float v = g[in + c];
        y[out + c] = __fdiv_rn(v, 1.0f + expf(-v)) * u[in + c];
    }
}

// One workgroup per (query i, head h): q [H, s, d], k / v [KV, s, d] head-major,
// out [s, H * d] token-major (the o_proj input). Scores of keys 0..i live in LDS.
__global__ __launch_bounds__(kOpsThreads) void attention_causal_f32_kernel(const float* __restrict__ q,
                                                                           const float* __restrict__ kk,
                                                                           const float* __restrict__ v, int heads,
                                                                           int n_rep, int s, int d,
                                                                           float* __restrict__ out) {
    extern __shared__ float sc[];
    __shared__ double red[kOpsThreads];
    __shared__ float redf[kOpsThreads];
    const int i = blockIdx.x, hh = blockIdx.y, kvh = hh / n_rep, tid = threadIdx.x;
    const float* qi = q + (static_cast<size_t>(hh) * s + i) * d;
    const float* kh = kk + static_cast<size_t>(kvh) * s * d;
    const float* vh = v + static_cast<size_t>(kvh) * s * d;
    const float scale = __fdiv_rn(1.0f, __fsqrt_rn(static_cast<float>(d)));
    float mx = -__builtin_inff();
    for (int j = tid; j <= i; j += kOpsThreads) {
        double dot = 0.0;
        for (int c = 0; c < d; ++c) dot = __builtin_fma(static_cast<double>(qi[c]), static_cast<double>(kh[static_cast<size_t>(j) * d + c]), dot);
        const float sj = static_cast<float>(dot) * scale;
        sc[j] = sj;
        mx = sj > mx ? sj : mx;
    }
    mx = block_max_f32(mx, redf);
    double den = 0.0;
    for (int j = tid; j <= i; j += kOpsThreads) {
        const float e = expf(sc[j] - mx);
        sc[j] = e;
        den += e;
    }
    den = block_sum_f64(den, red);
    const double inv = static_cast<double>(static_cast<float>(1.0 / den));
    for (int c = tid; c < d; c += kOpsThreads) {
        double acc = 0.0;
        for (int j = 0; j <= i; ++j) acc += static_cast<double>(sc[j]) * inv * static_cast<double>(vh[static_cast<size_t>(j) * d + c]);
        out[static_cast<size_t>(i) * heads * d + static_cast<size_t>(hh) * d + c] = static_cast<float>(acc);
    }
}

// ---- causal attention on the fp64 matrix cores --------------------------------------------
// The double sums of the reference as v_mfma_f64_16x16x4: one workgroup per 16
// queries of one head, its waves (eight, or four) taking the tiles of 16
// keys in turn. Scores are computed transposed, S^T = K Q^T: register v of lane (r = l %
// 16, g = l / 16) is then key 4v + g of query r, which is the B operand of step v
// of O^T = V^T P^T, so the probabilities go from one product to the next without
// leaving their lane. Both sums run in an order that lets a lane load its
// operands as whole 16-byte pieces: lane quarter g supplies the D / 4 consecutive
// columns from g * D / 4 of its K (Q) row, and lane r the D / 16 consecutive
// columns from r * D / 16 of its V rows.
// Two passes over the keys keep the reference's arithmetic: the first stores
// float(dot) * scale and the row maximum, the second forms expf(score - max),
// the double denominator and the double sums of e * v, which are scaled by
// double(float(1 / den)) at the end (once per output instead of once per term)
// and summed over the waves in a fixed tree. A lane reads back only the scores it
// wrote, 16 bytes per tile; SAVED holds them in LDS (1 KB per tile), otherwise
// (s > kAttSavedMax) the second pass repeats the products, whose bits are the same.
// Keys past the query (and rows past s, which are loaded as row s - 1) only occur
// in the last tile: they get e = 0, and where that tile's V holds an infinity or
// NaN it is summed by attention_tail instead of the MFMAs, as 0 * inf must not
// reach the earlier queries.
// Bound by fp64 MFMA issue (64 cycles each) and, on short prompts, the latency of
// the first loads. us against one workgroup per (query, head) with scalar double
// FMAs, which walked K a row per lane and V a key at a time: 14 heads of 64, s = 16
// 8.0 -> 5.8, s = 128 32.2 -> 7.4, s = 384 192 -> 19.4 (13.6 TFLOP/s), s = 1024
// 1519 -> 78 (24), s = 2048 6582 -> 233 (32); 12 heads of 128, s = 384 348 -> 32, s =
// 2048 11836 -> 365 (35). Without saved scores s = 2100 takes 320 (7092 before),
// which is why they are kept up to the 128 KB of 2048 keys.
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));  // four floats at any float's address
constexpr int kAttSavedMax = 2048;
// Waves per workgroup; four where eight left too few registers each.
template <int D, bool SAVED>
constexpr int att_waves() {
    return D == 128 && !SAVED ? 4 : 8;
}

template <int N>
__device__ __forceinline__ void load_floats(const float* p, float (&v)[N]) {
    static_assert(N % 2 == 0);
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
        const f4u t = *reinterpret_cast<const f4u*>(p + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * i + e] = t[e];
    }
#pragma unroll
    for (int i = N / 4 * 4; i < N; ++i) v[i] = p[i];
}

// The last tile of a workgroup, key by key: acc += e * v over the keys that the
// lane's query sees. acc[t][v'] is column r(4v' + g) * D / 16 + t of O.
template <int D>
__device__ void attention_tail(const float* vh, int key0, int query, int s, const float (&e)[4], int lane,
                               d4 (&acc)[D / 16]) {
    const int r = lane & 15, g = lane >> 4;
    for (int kk = 0; kk < 16; ++kk) {
        float ek = 0.0f;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float t = __shfl(e[v], (kk & 3) * 16 + r);
            ek = (kk >> 2) == v ? t : ek;
        }
        const int key = key0 + kk;
        if (key > query || key >= s) continue;
        const float* row = vh + static_cast<size_t>(key) * D;
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                acc[t][v] += static_cast<double>(ek) * static_cast<double>(row[(4 * v + g) * (D / 16) + t]);
            __builtin_amdgcn_sched_barrier(0);  // a rare path: no registers for its loads
        }
    }
}

template <int D, bool SAVED>
__global__ __launch_bounds__((att_waves<D, SAVED>() * 64)) void attention_causal_f64mfma_kernel(
    const float* __restrict__ q, const float* __restrict__ kk, const float* __restrict__ v, int heads, int n_rep,
    int s, float* __restrict__ out) {
    constexpr int QL = D / 4, T = D / 16, kAttWaves = att_waves<D, SAVED>();
    extern __shared__ __attribute__((aligned(16))) char att_lds[];
    __shared__ float redm[kAttWaves][16];
    __shared__ double redd[kAttWaves][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
    const int qt = static_cast<int>(gridDim.x - 1 - blockIdx.x);  // the longest rows of keys first
    const int hh = blockIdx.y, kvh = hh / n_rep, q0 = qt * 16, query = q0 + r;
    const float* kh = kk + static_cast<size_t>(kvh) * s * D;
    const float* vh = v + static_cast<size_t>(kvh) * s * D;
    const float scale = __fdiv_rn(1.0f, __fsqrt_rn(static_cast<float>(D)));
    f4* saved = reinterpret_cast<f4*>(att_lds);

    float qf[QL];
    load_floats<QL>(q + (static_cast<size_t>(hh) * s + min(query, s - 1)) * D + g * QL, qf);
    // Scores of key tile jt. The second pass without saved scores takes K in two
    // halves and keeps Q as floats between the tiles (registers at D = 128).
    auto scores = [&](int jt) {
        constexpr int P = SAVED ? QL : QL / 2;
        const float* row = kh + static_cast<size_t>(min(jt * 16 + r, s - 1)) * D + g * QL;
        d4 c = {0, 0, 0, 0};
#pragma unroll
        for (int p = 0; p < QL; p += P) {
            float kf[P];
            load_floats<P>(row + p, kf);
#pragma unroll
            for (int t = 0; t < P; ++t) {
                if constexpr (!SAVED) asm volatile("" : "+v"(qf[p + t]));
                c = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(kf[t]), static_cast<double>(qf[p + t]), c, 0,
                                                         0, 0);
            }
            if constexpr (!SAVED) __builtin_amdgcn_sched_barrier(0);
        }
        f4 sc;
#pragma unroll
        for (int i = 0; i < 4; ++i) sc[i] = static_cast<float>(c[i]) * scale;
        return sc;
    };

    float mx = -__builtin_inff();
    for (int jt = wave; jt <= qt; jt += kAttWaves) {
        const f4 sc = scores(jt);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (jt * 16 + 4 * i + g <= query) mx = sc[i] > mx ? sc[i] : mx;
        if constexpr (SAVED) saved[jt * 64 + lane] = sc;
    }
    {
        float o = __shfl_xor(mx, 16);
        mx = o > mx ? o : mx;
        o = __shfl_xor(mx, 32);
        mx = o > mx ? o : mx;
        if (g == 0) redm[wave][r] = mx;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kAttWaves; ++w) mx = redm[w][r] > mx ? redm[w][r] : mx;
    }

    double den = 0.0;
    d4 acc[T];
#pragma unroll
    for (int t = 0; t < T; ++t) acc[t] = d4{0, 0, 0, 0};
    for (int jt = wave; jt <= qt; jt += kAttWaves) {
        float vf[4][T];
        auto load_v = [&] {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                load_floats<T>(vh + static_cast<size_t>(min(jt * 16 + 4 * i + g, s - 1)) * D + r * T, vf[i]);
        };
        f4 sc;
        if constexpr (SAVED) {
            load_v();
            sc = saved[jt * 64 + lane];
        } else {
            sc = scores(jt);
            load_v();
        }
        float e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            e[i] = jt * 16 + 4 * i + g <= query ? expf(sc[i] - mx) : 0.0f;
            den += static_cast<double>(e[i]);
        }
        if (jt == qt) {
            float big = 0.0f;  // NaN or infinite where any of the tile's values is
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int t = 0; t < T; ++t) big += vf[i][t] * 0.0f;
            if (__any(!(big == 0.0f))) {
                attention_tail<D>(vh, jt * 16, query, s, e, lane, acc);
                continue;
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int t = 0; t < T; ++t)
                acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(static_cast<double>(vf[i][t]), static_cast<double>(e[i]),
                                                              acc[t], 0, 0, 0);
            if constexpr (!SAVED) __builtin_amdgcn_sched_barrier(0);
        }
    }
    den += __shfl_xor(den, 16);
    den += __shfl_xor(den, 32);
    if (g == 0) redd[wave][r] = den;
    // O over the waves: the upper half hands its sums to the lower half, three times.
    d4* part = reinterpret_cast<d4*>(att_lds);
    for (int half = kAttWaves / 2; half > 0; half >>= 1) {
        __syncthreads();  // the scores (or the last round's sums) have been read
        if (wave >= half && wave < 2 * half)
#pragma unroll
            for (int t = 0; t < T; ++t) part[((wave - half) * T + t) * 64 + lane] = acc[t];
        __syncthreads();
        if (wave < half)
#pragma unroll
            for (int t = 0; t < T; ++t) acc[t] += part[(wave * T + t) * 64 + lane];
    }
    if (wave != 0 || query >= s) return;
    den = redd[0][r];
#pragma unroll
    for (int w = 1; w < kAttWaves; ++w) den += redd[w][r];
    const double inv = static_cast<double>(static_cast<float>(1.0 / den));
    float* o = out + (static_cast<size_t>(query) * heads + hh) * D;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < T; ++t) o[(4 * i + g) * T + t] = static_cast<float>(acc[t][i] * inv);
}

// LDS of the sums that the waves hand over.
template <int D, bool SAVED>
constexpr size_t sums_of() {
    return size_t(att_waves<D, SAVED>() / 2) * (D / 16) * 64 * sizeof(d4);
}

template <int D>
nq_status launch_attention_f64(const float* q, const float* k, const float* v, int heads, int n_rep, int s, float* out,
                               hipStream_t st) {
    const size_t saved = static_cast<size_t>((s + 15) / 16) * 64 * sizeof(f4);
    const dim3 grid(static_cast<unsigned>((s + 15) / 16), static_cast<unsigned>(heads));
    if (s <= kAttSavedMax) {
        constexpr size_t sums = sums_of<D, true>();
        const size_t lds = saved > sums ? saved : sums;
        auto* fn = attention_causal_f64mfma_kernel<D, true>;
        constexpr size_t most = size_t(kAttSavedMax / 16) * 64 * sizeof(f4);  // the limit is set once, for every s
        static_assert(most >= sums, "scores outgrow the sums");
        if (nq_status e = set_dynamic_lds(reinterpret_cast<const void*>(fn), most, "attention_causal_f32")) return e;
        fn<<<grid, att_waves<D, true>() * 64, lds, st>>>(q, k, v, heads, n_rep, s, out);
    } else {
        constexpr size_t sums = sums_of<D, false>();
        auto* fn = attention_causal_f64mfma_kernel<D, false>;
        if (nq_status e = set_dynamic_lds(reinterpret_cast<const void*>(fn), sums, "attention_causal_f32")) return e;
        fn<<<grid, att_waves<D, false>() * 64, sums, st>>>(q, k, v, heads, n_rep, s, out);
    }
    return launch_status("attention_causal_f64mfma_kernel");
}

}  // namespace
}  // namespace nq

using namespace nq;

extern "C" nq_status nq_rmsnorm_f32(const float* x, const float* r, float* h, const float* w, float eps, int64_t m,
                                    int64_t k, float* y, void* stream) {
    NQ_REQUIRE(m >= 0 && k >= 0 && m <= kMaxIndex && k <= kMaxIndex, NQ_BAD_SHAPE, "rmsnorm_f32: bad shape");
    if (m == 0 || k == 0) return NQ_OK;
    NQ_REQUIRE(x && w && y && (!r || h), NQ_BAD_ARG, "rmsnorm_f32: null pointer");
    NQ_REQUIRE(aligned(x, 4) && aligned(w, 4) && aligned(y, 4) && aligned(r, 4) && aligned(h, 4), NQ_BAD_ALIGN,
               "rmsnorm_f32: misaligned pointer");
    rmsnorm_f32_kernel<<<static_cast<unsigned>(m), kOpsThreads, 0, as_stream(stream)>>>(x, r, h, w, eps,
                                                                                         static_cast<int>(k), y);
    return launch_status("rmsnorm_f32_kernel");
}

extern "C" nq_status nq_silu_mul_f32(const float* gate, const float* up, int64_t ld, int64_t m, int64_t k, float* y,
                                     void* stream) {
    NQ_REQUIRE(m >= 0 && k >= 0 && ld >= k && m <= kMaxIndex && k <= kMaxIndex, NQ_BAD_SHAPE,
               "silu_mul_f32: bad shape");
    if (m == 0 || k == 0) return NQ_OK;
    NQ_REQUIRE(gate && up && y, NQ_BAD_ARG, "silu_mul_f32: null pointer");
    silu_mul_f32_kernel<<<static_cast<unsigned>(m), kOpsThreads, 0, as_stream(stream)>>>(gate, up, ld,
                                                                                          static_cast<int>(k), y);
    return launch_status("silu_mul_f32_kernel");
}

extern "C" nq_status nq_attention_causal_f32(const float* q, const float* k, const float* v, int64_t heads,
                                             int64_t kv_heads, int64_t s, int64_t head_dim, float* out,
                                             void* stream) {
    NQ_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && s >= 0 && head_dim > 0 && s <= 16384 &&
                   heads <= 65535 && head_dim <= 1024,
               NQ_BAD_SHAPE, "attention_causal_f32: bad shape (heads %% kv_heads == 0, s <= 16384)");
    if (s == 0) return NQ_OK;
    NQ_REQUIRE(q && k && v && out, NQ_BAD_ARG, "attention_causal_f32: null pointer");
    const int nh = static_cast<int>(heads), rep = static_cast<int>(heads / kv_heads), si = static_cast<int>(s);
    switch (head_dim) {
        case 32: return launch_attention_f64<32>(q, k, v, nh, rep, si, out, as_stream(stream));
        case 64: return launch_attention_f64<64>(q, k, v, nh, rep, si, out, as_stream(stream));
        case 96: return launch_attention_f64<96>(q, k, v, nh, rep, si, out, as_stream(stream));
        case 128: return launch_attention_f64<128>(q, k, v, nh, rep, si, out, as_stream(stream));
        default: break;
    }
    const size_t lds = static_cast<size_t>(s) * sizeof(float);
    if (nq_status st = set_dynamic_lds(reinterpret_cast<const void*>(attention_causal_f32_kernel), lds,
                                       "attention_causal_f32"))
        return st;
    const dim3 grid(static_cast<unsigned>(s), static_cast<unsigned>(heads));
    attention_causal_f32_kernel<<<grid, kOpsThreads, lds, as_stream(stream)>>>(
        q, k, v, nh, rep, si, static_cast<int>(head_dim), out);
    return launch_status("attention_causal_f32_kernel");
}
