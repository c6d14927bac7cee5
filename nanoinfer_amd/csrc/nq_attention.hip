// Causal grouped-query attention on fp16 heads, the step between the RoPE and the
// output projection of a decoder layer (ops.cpp:206-270 with fp16 activations): scores
// and softmax in fp32, the weights exp(s - max) in fp16 for the second product, fp32 sums.
//
// One workgroup per 16 queries of one head, its four waves taking every fourth tile of
// 32 keys with a running maximum each, merged through LDS at the end. Scores are computed
// transposed, S^T = K Q^T, so a lane ends with 8 weights of its own query, and these are
// already the B operand of O^T = V^T P^T when V's rows are taken in the same order
// (position (g, e) of lane quarter g is key 4 g + e of the tile's first half for e < 4,
// of its second half otherwise). K and Q rows are read in 16-byte pieces, lane quarter g the
// D / 4 columns from g * D / 4 of its row; of V lane r reads the D / 16 columns from r * D / 16 of
// its 8 keys, whose transpose, a few byte permutes in its own registers, is the A
// operand of D / 16 tiles (tile c: column r * D / 16 + c). So nothing passes through LDS
// but the merge.
//
// Keys past the query weigh 0. They only share a tile with counted ones in the last tile of
// a workgroup, where an infinity or NaN of V takes that tile through attention_tail (0 *
// inf would reach the earlier queries).
// Bound by the latency of a few tiles per wave up to some 500 tokens, then by the re-reads of
// K and V, 16 queries to each. us against torch's fused attention: 12 heads of 128 (2 of K
// and V), s = 24 9.2 -> 4.3, s = 128 14.2 -> 5.2, s = 512 30.9 -> 13.7, s = 2048 97.7 -> 85;
// 14 heads of 64, s = 512 21.7 -> 9.1, s = 1024 31.6 -> 26.4, s = 2048 51.9 against 59.0 (its
// caller keeps torch's there).
#include <hip/hip_runtime.h>

#include "nq_device.hpp"
#include "nq_internal.hpp"

namespace nq {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
constexpr int kHeadWaves = 4;

template <int N>  // N halves as N / 2 dwords
__device__ __forceinline__ void load_dwords(const _Float16* p, int (&v)[N / 2]) {
    __builtin_memcpy(v, __builtin_assume_aligned(p, 2 * N < 16 ? 2 * N : 16), 2 * N);
}

// One tile key by key: acc += weight * V over the keys the lane's query sees.
template <int C>
__device__ void attention_tail(const _Float16* vh, int key0, int query, const float (&p)[8], int lane, f4 (&acc)[C]) {
    constexpr int D = 16 * C;
    const int r = lane & 15, g = lane >> 4;
    for (int kk = 0; kk < 32; ++kk) {
        float pk = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float t = __shfl(p[e], ((kk & 15) >> 2) * 16 + r);
            pk = ((kk >> 4) * 4 + (kk & 3)) == e ? t : pk;
        }
        if (key0 + kk > query) continue;
        const _Float16* row = vh + static_cast<size_t>(key0 + kk) * D;
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[c][v] = __builtin_fmaf(pk, static_cast<float>(row[(4 * g + v) * C + c]), acc[c][v]);
    }
}

template <int D>
__global__ __launch_bounds__(kHeadWaves * 64) void attention_causal_f16_kernel(
    const _Float16* __restrict__ q, const _Float16* __restrict__ kk, const _Float16* __restrict__ v, int n_rep, int s,
    _Float16* __restrict__ out) {
    constexpr int C = D / 16, T = D / 32, QL = D / 4;  // V tiles, MFMA steps, columns of a K row per lane
    __shared__ float red[2][kHeadWaves][16];
    __shared__ __attribute__((aligned(16))) float part[kHeadWaves][16][D + 4];
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qt = static_cast<int>(gridDim.x - 1 - blockIdx.x);  // the longest rows of keys first
    const int hh = blockIdx.y, kvh = hh / n_rep, q0 = qt * 16, query = min(q0 + r, s - 1);
    const _Float16* kh = kk + static_cast<size_t>(kvh) * s * D;
    const _Float16* vh = v + static_cast<size_t>(kvh) * s * D;
    // exp(x / sqrt(D)) as 2^(x * c)
    const float c2 = 1.44269504088896f / __builtin_sqrtf(static_cast<float>(D));

    int qf[T][4];
#pragma unroll
    for (int t = 0; t < T; ++t) load_dwords<8>(q + (static_cast<size_t>(hh) * s + query) * D + g * QL + 8 * t, qf[t]);
    f4 acc[C];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] = f4{0, 0, 0, 0};
    float mx = -__builtin_inff(), den = 0.0f;
    const int last = (q0 + 15) / 32;  // the tile that holds the last query's key
    for (int jt = wave; jt <= last; jt += kHeadWaves) {
        const int key0 = jt * 32;
        int kf[2][T][4], vf[8][C / 2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int t = 0; t < T; ++t)
                load_dwords<8>(kh + static_cast<size_t>(min(key0 + 16 * b + r, s - 1)) * D + g * QL + 8 * t, kf[b][t]);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            load_dwords<C>(vh + static_cast<size_t>(min(key0 + (e >> 2) * 16 + 4 * g + (e & 3), s - 1)) * D + r * C, vf[e]);
        float sc[8];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            f4 d = {0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < T; ++t)
                d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, *reinterpret_cast<const v4i*>(kf[b][t])),
                                                           __builtin_bit_cast(h8, *reinterpret_cast<const v4i*>(qf[t])), d, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) sc[4 * b + i] = key0 + 16 * b + 4 * g + i <= query ? d[i] * c2 : -__builtin_inff();
        }
        float m1 = mx;
#pragma unroll
        for (int e = 0; e < 8; ++e) m1 = sc[e] > m1 ? sc[e] : m1;
        {
            float o = __uint_as_float(swap_partner<16>(__float_as_uint(m1), lane));
            m1 = o > m1 ? o : m1;
            o = __uint_as_float(swap_partner<32>(__float_as_uint(m1), lane));
            m1 = o > m1 ? o : m1;
        }
        // Rescale by 2^(old - new maximum); 1 while neither is above -inf.
        const float corr = m1 == mx ? 1.0f : __builtin_amdgcn_exp2f(mx - m1);
        mx = m1;
        float p[8];
        den *= corr;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            p[e] = sc[e] == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(sc[e] - mx);
            den += p[e];
        }
        if (__any(corr != 1.0f)) {
#pragma unroll
            for (int c = 0; c < C; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[c][i] *= corr;
        }
        if (jt == last) {
            float bad = 0.0f;  // NaN where the tile holds an infinity or NaN
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int i = 0; i < C / 2; ++i) {
                    const h2 t = __builtin_bit_cast(h2, vf[e][i]);
                    bad += (static_cast<float>(t[0]) + static_cast<float>(t[1])) * 0.0f;
                }
            if (__any(!(bad == 0.0f))) {
                attention_tail<C>(vh, key0, query, p, lane, acc);
                continue;
            }
        }
        h8 pb;
#pragma unroll
        for (int e = 0; e < 8; ++e) pb[e] = static_cast<_Float16>(p[e]);
#pragma unroll
        for (int c = 0; c < C; ++c) {
            v4i a;  // column c of the 8 x C block
#pragma unroll
            for (int j = 0; j < 4; ++j)
                a[j] = static_cast<int>(__builtin_amdgcn_perm(static_cast<unsigned>(vf[2 * j + 1][c / 2]), static_cast<unsigned>(vf[2 * j][c / 2]),
                                                              c % 2 ? 0x07060302u : 0x05040100u));
            acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, a), pb, acc[c], 0, 0, 0);
        }
    }
    den += __uint_as_float(swap_partner<16>(__float_as_uint(den), lane));
    den += __uint_as_float(swap_partner<32>(__float_as_uint(den), lane));
    if (g == 0) {
        red[0][wave][r] = mx;
        red[1][wave][r] = den;
    }
    __syncthreads();
    float m = red[0][0][r];
#pragma unroll
    for (int w = 1; w < kHeadWaves; ++w) m = red[0][w][r] > m ? red[0][w][r] : m;
    // a wave without a tile weighs 0; where every score is -inf, or NaN, the sums are NaN
    const float mine = mx == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(mx - m);
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[wave][r][(4 * g + i) * C + c] = acc[c][i] * mine;
    __syncthreads();
    // thread t: D / 16 consecutive columns of query t / 16
    const int row = threadIdx.x >> 4, col = (threadIdx.x & 15) * C;
    if (q0 + row >= s) return;
    float mr = red[0][0][row], dsum = 0.0f;
#pragma unroll
    for (int w = 1; w < kHeadWaves; ++w) mr = red[0][w][row] > mr ? red[0][w][row] : mr;
#pragma unroll
    for (int w = 0; w < kHeadWaves; ++w)
        dsum += red[1][w][row] * (red[0][w][row] == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(red[0][w][row] - mr));
    const float inv = __fdiv_rn(1.0f, dsum);
    _Float16 o[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        float t = part[0][row][col + c];
#pragma unroll
        for (int w = 1; w < kHeadWaves; ++w) t += part[w][row][col + c];
        o[c] = from_f32<_Float16>(t * inv);
    }
    __builtin_memcpy(__builtin_assume_aligned(out + (static_cast<size_t>(hh) * s + q0 + row) * D + col, 2 * C), o, 2 * C);
}

}  // namespace
}  // namespace nq

using namespace nq;

extern "C" nq_status nq_attention_causal_f16(const void* q, const void* k, const void* v, int64_t heads, int64_t kv_heads,
                                             int64_t s, int64_t head_dim, void* out, void* stream) {
    NQ_REQUIRE(heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && heads <= 65535 && s >= 0 && s <= (int64_t(1) << 30) &&
                   (head_dim == 64 || head_dim == 128),
               NQ_BAD_SHAPE, "attention_causal_f16: bad shape (heads %% kv_heads == 0, head_dim 64 or 128)");
    if (s == 0) return NQ_OK;
    NQ_REQUIRE(q && k && v && out, NQ_BAD_ARG, "attention_causal_f16: null pointer");
    NQ_REQUIRE(aligned(q, 16) && aligned(k, 16) && aligned(v, 16) && aligned(out, 16), NQ_BAD_ALIGN,
               "attention_causal_f16: 16-byte alignment required");
    const dim3 grid(static_cast<unsigned>((s + 15) / 16), static_cast<unsigned>(heads));
    auto go = [&](auto* fn) {
        fn<<<grid, kHeadWaves * 64, 0, as_stream(stream)>>>(static_cast<const _Float16*>(q), static_cast<const _Float16*>(k),
                                                            static_cast<const _Float16*>(v), static_cast<int>(heads / kv_heads),
                                                            static_cast<int>(s), static_cast<_Float16*>(out));
    };
    if (head_dim == 64) go(attention_causal_f16_kernel<64>);
    else go(attention_causal_f16_kernel<128>);
    return launch_status("attention_causal_f16_kernel");
}
