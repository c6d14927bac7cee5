// GEMVs (up to 8 activation rows) over any k and any row alignment: the operands that
// the 16-byte GEMVs cannot take (k % 16, k % 32 for int4, unaligned pointers, one
// int4 group per row of such a k), which ran a column per lane (int4: a group per
// lane) and one activation row after the other.
//
// A wave owns R weight rows and all M activation rows; its lanes take whole pieces of
// PC columns (16-byte loads at any byte address) over K, which KW waves of the
// workgroup share when the weight is too narrow to fill the GPU with rows. A piece is
// summed by fp32 FMAs, the pieces of a lane and then of the wave, in a fixed tree, in
// fp64 (in fp32 they were off by 7.3e-8 where the element kernel's groups of 256 were by
// 5.4e-8, k = 1003, fp16; now 2.6e-8); int8 activations in int32 by v_dot4. The columns of
// the last, partial piece go one to a lane, so nothing past a row is touched.
//
// Bound by latency on small weights and by the activation re-reads (one per R weight
// rows) at 8 rows. us, element kernel -> this: Q8 fp32 x, n = 1001, k = 1003 m = 7 15.4 ->
// 5.5; n = 1536, k = 8955 m = 1 37 -> 6.5, m = 8 272 -> 13; n = k = 9001 m = 2 146 -> 26
// (3.1 TB/s); Q4G m = 1, n = 17920, k = 1531 83 -> 9.0; one int4 group per row, m = 8, n =
// 1536, k = 8955 7029 -> 13; W8A8 m = 2, n = k = 9001 135 -> 17 (4.7 TB/s).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "nq_device.hpp"
#include "nq_internal.hpp"
#include "nq_tile_gemm.hpp"

namespace nq {
namespace {

enum class WF { Q8, Q4Row, Q4G };

struct AnyArgs {
    const void* x;
    const uint8_t* w;
    const void* scale;
    const float* a_scale;
    const float* bias;
    void* y;
    int m, n, k, groups, cpg;
    unsigned cpg_magic;  // chunk / cpg == umulhi(chunk, magic)
    int kw, scale_f16, y_kind;
};

template <int N>
__device__ __forceinline__ void load_x(const float* p, float (&v)[N]) {
    __builtin_memcpy(v, p, 4 * N);
}
template <int N>
__device__ __forceinline__ void load_x(const _Float16* p, float (&v)[N]) {
    _Float16 t[N];
    __builtin_memcpy(t, p, 2 * N);
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = static_cast<float>(t[e]);
}
__device__ __forceinline__ float scale_at(const AnyArgs& a, size_t i) {
    return a.scale_f16 ? static_cast<float>(static_cast<const _Float16*>(a.scale)[i]) : static_cast<const float*>(a.scale)[i];
}

template <typename XT, WF F, int M, int R>
__global__ __launch_bounds__(256) void gemv_any_kernel(AnyArgs a) {
    constexpr bool I8 = sizeof(XT) == 1, Q4 = F != WF::Q8;
    constexpr int PC = I8 || M <= 2 ? 16 : 8;  // columns per piece: 8 keeps M rows of x in registers
    constexpr int WD = PC / (Q4 ? 8 : 4);      // dwords of a weight piece
    constexpr int NV = M * R;
    using Acc = std::conditional_t<I8, int, double>;
    __shared__ Acc part[4][NV];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int k = a.k, m = a.m, n = a.n, rb = Q4 ? (k + 1) / 2 : k;
    const int kw = a.kw, wk = wave % kw;
    const int row0 = (blockIdx.x * (4 / kw) + wave / kw) * R;
    const uint8_t* wr[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wr[r] = a.w + static_cast<size_t>(min(row0 + r, n - 1)) * rb;
    const XT* xr[M];
#pragma unroll
    for (int i = 0; i < M; ++i) xr[i] = static_cast<const XT*>(a.x) + static_cast<size_t>(min(i, m - 1)) * k;

    Acc acc[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[v] = 0;
    auto scales = [&](int c, float (&sc)[R]) {
        if constexpr (F == WF::Q4G) {
            const int chunk = c >> 5, g = a.cpg == 1 ? chunk : static_cast<int>(__umulhi(static_cast<unsigned>(chunk), a.cpg_magic));
#pragma unroll
            for (int r = 0; r < R; ++r) sc[r] = scale_at(a, static_cast<size_t>(min(row0 + r, n - 1)) * a.groups + g);
        }
    };
    auto code = [&](const int (&w)[WD], int e) -> float {
        if constexpr (Q4) return static_cast<float>((static_cast<unsigned>(w[e / 8]) >> (4 * (e % 8))) & 15u) - 8.0f;
        else return static_cast<float>((w[e / 4] << (24 - 8 * (e % 4))) >> 24);
    };
    auto add = [&](const int (&w)[R][WD], const float (&sc)[R], int i, const auto& xv) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (I8) {
#pragma unroll
                for (int d = 0; d < WD; ++d) acc[i * R + r] = __builtin_amdgcn_sdot4(w[r][d], xv[d], acc[i * R + r], false);
            } else {
                float p = 0.0f;
#pragma unroll
                for (int e = 0; e < PC; ++e) p = __builtin_fmaf(xv[e], code(w[r], e), p);
                if constexpr (F == WF::Q4G) acc[i * R + r] = __builtin_fma(static_cast<double>(p), static_cast<double>(sc[r]), acc[i * R + r]);
                else acc[i * R + r] += p;
            }
        }
    };
    const int whole = k / PC;
    for (int u = wk * 64 + lane; u < whole; u += 64 * kw) {
        const int c = u * PC;
        int w[R][WD];
#pragma unroll
        for (int r = 0; r < R; ++r) __builtin_memcpy(w[r], wr[r] + (Q4 ? c >> 1 : c), 4 * WD);
        float sc[R];
        scales(c, sc);
#pragma unroll
        for (int i = 0; i < M; ++i) {
            if constexpr (I8) {
                int xv[4];
                __builtin_memcpy(xv, xr[i] + c, 16);
                add(w, sc, i, xv);
            } else {
                float xv[PC];
                load_x<PC>(xr[i] + c, xv);
                add(w, sc, i, xv);
            }
        }
    }
    if (wk == 0 && lane < k - whole * PC) {  // the partial piece, a column per lane
        const int c = whole * PC + lane;
        float sc[R];
        scales(c, sc);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int b = Q4 ? wr[r][c >> 1] : wr[r][c];
            const int q = Q4 ? (c & 1 ? b >> 4 : b & 15) - 8 : static_cast<int8_t>(b);
#pragma unroll
            for (int i = 0; i < M; ++i) {
                if constexpr (I8) acc[i * R + r] += q * static_cast<int>(xr[i][c]);
                else acc[i * R + r] += static_cast<double>(xr[i][c]) * q * (F == WF::Q4G ? sc[r] : 1.0f);
            }
        }
    }
    // Lane l ends with the wave's sum of value l / (64 / NV). Doubles without the LDS: m = 7, n =
    // 1001, k = 1003 6.1 -> 5.5 us, m = 8, n = 1536, k = 8955 13.7 -> 13.1.
    if constexpr (I8) wave_reduce_stage_bperm<NV, 32>(acc, lane);
    else wave_reduce_stage<NV, 32>(acc, lane);
    Acc sum = acc[0];
    constexpr int G = 64 / NV;
    if (kw > 1) {
        if (lane % G == 0) part[wave][lane / G] = sum;
        __syncthreads();
        if (wk != 0) return;
        for (int s = 1; s < kw; ++s) sum += part[wave + s][lane / G];
    }
    const int v = lane / G, i = v / R, row = row0 + v % R;
    if (lane % G != 0 || i >= m || row >= n) return;
    const size_t o = static_cast<size_t>(i) * n + row;
    if constexpr (I8) {
        if (a.y_kind == kTileI32) {
            static_cast<int32_t*>(a.y)[o] = sum;
            return;
        }
    }
    const float b = a.bias ? a.bias[row] : 0.0f;
    float t;
    if constexpr (I8) t = w8a8_epilogue(sum, a.a_scale[i], scale_at(a, row), b);
    else t = static_cast<float>(F == WF::Q4G ? sum + b : sum * scale_at(a, row) + b);
    if (a.y_kind == kTileF16) static_cast<_Float16*>(a.y)[o] = from_f32<_Float16>(t);
    else static_cast<float*>(a.y)[o] = t;
}

template <typename XT, WF F, int M>
void launch_any(AnyArgs a, hipStream_t s) {
    // Two weight rows per wave; four from 8192 rows, which leave waves enough for half the
    // activation re-reads.
    const int R = a.n >= 8192 ? 4 : 2;
    // K over 2 or 4 waves while rows alone leave under 4096 waves, with at least 1024 columns
    // each: 64 pieces of 16, or 128 of 8.
    const int waves = (a.n + R - 1) / R;
    a.kw = a.k >= 4096 && waves < 2048 ? 4 : a.k >= 2048 && waves < 4096 ? 2 : 1;
    const int rows = R * 4 / a.kw;
    const unsigned grid = static_cast<unsigned>((a.n + rows - 1) / rows);
    if (R == 4) gemv_any_kernel<XT, F, M, 4><<<grid, 256, 0, s>>>(a);
    else gemv_any_kernel<XT, F, M, 2><<<grid, 256, 0, s>>>(a);
}

template <typename XT, WF F>
nq_status launch_any_m(const AnyArgs& a, hipStream_t s) {
    if (a.m == 1) launch_any<XT, F, 1>(a, s);
    else if (a.m == 2) launch_any<XT, F, 2>(a, s);
    else if (a.m <= 4) launch_any<XT, F, 4>(a, s);
    else launch_any<XT, F, 8>(a, s);
    return launch_status("gemv_any_kernel");
}

}  // namespace

nq_status gemv_any(const TileCall& c, hipStream_t s) {
    const bool row = c.q4 && c.group >= c.k, grouped = c.q4 && !row;
    AnyArgs a{};
    a.x = c.x;
    a.w = c.w;
    a.scale = c.scale;
    a.a_scale = c.a_scale;
    a.bias = c.bias;
    a.y = c.y;
    a.m = static_cast<int>(c.m);
    a.n = static_cast<int>(c.n);
    a.k = static_cast<int>(c.k);
    a.cpg = grouped ? static_cast<int>(c.group / 32) : 1;
    a.groups = grouped ? static_cast<int>((c.k + c.group - 1) / c.group) : 1;
    a.cpg_magic = a.cpg > 1 ? static_cast<unsigned>(((uint64_t(1) << 32) + a.cpg - 1) / a.cpg) : 0;
    a.scale_f16 = c.scale_f16;
    a.y_kind = c.yt;
    if (c.xt == TileX::I8) return launch_any_m<int8_t, WF::Q8>(a, s);
    if (c.xt == TileX::F32) {
        if (!c.q4) return launch_any_m<float, WF::Q8>(a, s);
        return row ? launch_any_m<float, WF::Q4Row>(a, s) : launch_any_m<float, WF::Q4G>(a, s);
    }
    if (!c.q4) return launch_any_m<_Float16, WF::Q8>(a, s);
    return row ? launch_any_m<_Float16, WF::Q4Row>(a, s) : launch_any_m<_Float16, WF::Q4G>(a, s);
}

}  // namespace nq
