// Linears over any K, any row alignment and any group of whole 32-column chunks:
// the shapes whose rows the LDS-DMA and raw-buffer kernels cannot take (k not a
// multiple of 16, 64 or 128, group sizes that are no power of two times 32, one
// group per row), and fp32 activations over prompts, where splitting the
// activations once per tile instead of once per wave pays.
//
// Tile GEMM. A workgroup owns a BM x BN output tile over one range of K. K advances in
// slabs of SK columns through two LDS buffers: a thread loads its pieces of the
// activation and weight rows (8 or 16 columns, 16-byte loads at any byte address)
// two slabs ahead into registers, converts them once for the whole workgroup
// (fp32 activations into three bf16 parts that sum to them exactly, codes into bf16 or
// fp16 exactly, int8 as it is) and writes them to LDS in the MFMA operand layout,
// 16-byte chunks swizzled as in the LDS-DMA kernels. The per-wave kernels convert
// inside the K loop, so each weight fragment is converted by every wave along m and
// each activation fragment split by every wave along n.
//
// Nothing is read past a row's last column: a K that is no whole number of slabs
// has its tail slab loaded element by element with clamped addresses, activations
// past k as zeros, and that slab goes first, so that its latency hides behind the
// first whole slabs. Rows past m or n are loaded as the last row and not stored.
//
// Results: products are exact in fp32; sums over up to 256 columns are fp32, and those
// of K fp64 or fp32 (int32 for int8), see PART and FINE. With K split over gridDim.y
// each range stores its raw sums into its own plane, in fp32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "nq_device.hpp"
#include "nq_internal.hpp"
#include "nq_tile_gemm.hpp"

namespace nq {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef double d4 __attribute__((ext_vector_type(4)));

// Weight formats: int8 codes (Q8Fine: sums as for int4, see tile_gemm_kernel), int4
// codes with one scale per row, int4 in groups of 32 columns, int4 in groups of a
// larger multiple of 32.
enum class WF { Q8, Q8Fine, Q4Row, Q4G32, Q4G };
constexpr bool is_q4(WF f) { return f != WF::Q8 && f != WF::Q8Fine; }
constexpr bool is_grouped(WF f) { return f == WF::Q4G32 || f == WF::Q4G; }

// n bytes at any address (global memory takes unaligned vector loads).
__device__ __forceinline__ v4i load16(const void* p) {
    v4i v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

__device__ __forceinline__ unsigned bits(float f) { return __builtin_bit_cast(unsigned, f); }
__device__ __forceinline__ float top16(float f) { return __builtin_bit_cast(float, bits(f) & 0xFFFF0000u); }
// Two fp32 values whose low halves are dropped, as a bf16 pair.
__device__ __forceinline__ int bf16_pair(float a, float b) {
    return static_cast<int>(__builtin_amdgcn_perm(bits(b), bits(a), 0x07060302u));
}

// Eight fp32 values as three bf16 parts whose sum is exact (|v| >= 2^-110): the top 8
// significant bits, the next 8, the rest. An infinity keeps itself in the first
// part and zeros in the others (inf - inf would be NaN). No branch here: the
// conversions share a basic block with the MFMAs that they hide behind.
// FINE: `lost` collects the bits that the parts drop, those of a smaller |v| and of a NaN
// that has bits in its low half only.
template <bool FINE>
__device__ __forceinline__ void split3(const float (&v)[8], v4i& hi, v4i& mid, v4i& lo, unsigned& lost) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float m[2], l[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const float f = v[2 * i + e];
            float r = f - top16(f);
            r = r == r ? r : FINE ? __builtin_bit_cast(float, bits(f) & 0xFFFFu) : 0.0f;
            m[e] = r;
            l[e] = r - top16(r);
            if constexpr (FINE) lost |= bits(l[e]) & 0xFFFFu;
        }
        hi[i] = bf16_pair(v[2 * i], v[2 * i + 1]);
        mid[i] = bf16_pair(m[0], m[1]);
        lo[i] = bf16_pair(l[0], l[1]);
    }
}

// Eight codes in column order as eight bf16 or fp16 values (exact).
template <bool BF>
__device__ __forceinline__ v4i codes_q8(int w0, int w1) {
    v4i r;
    if constexpr (BF) {
        const unsigned u0 = static_cast<unsigned>(w0) ^ 0x80808080u, u1 = static_cast<unsigned>(w1) ^ 0x80808080u;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            r[i] = bf16_pair(static_cast<float>((u0 >> (16 * i)) & 0xFFu) - 128.0f,
                             static_cast<float>((u0 >> (16 * i + 8)) & 0xFFu) - 128.0f);
            r[2 + i] = bf16_pair(static_cast<float>((u1 >> (16 * i)) & 0xFFu) - 128.0f,
                                 static_cast<float>((u1 >> (16 * i + 8)) & 0xFFu) - 128.0f);
        }
    } else {
        // bytes (2t, 2t + 1) into two halves; XOR 0x6480 is the fp16 value 1024 + (code + 128)
        const h2 off = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const unsigned sel = 0x0C000C00u | static_cast<unsigned>(2 * t) | (static_cast<unsigned>(2 * t + 1) << 16);
            const unsigned b = __builtin_amdgcn_perm(static_cast<unsigned>(w1), static_cast<unsigned>(w0), sel);
            r[t] = __builtin_bit_cast(int, __builtin_bit_cast(h2, b ^ 0x64806480u) + off);
        }
    }
    return r;
}
template <bool BF>
__device__ __forceinline__ v4i codes_q4(int w) {
    const unsigned lo = static_cast<unsigned>(w) & 0x0F0F0F0Fu, hi = (static_cast<unsigned>(w) >> 4) & 0x0F0F0F0Fu;
    v4i r;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        if constexpr (BF) {
            r[t] = bf16_pair(static_cast<float>((lo >> (8 * t)) & 0xFFu) - 8.0f,
                             static_cast<float>((hi >> (8 * t)) & 0xFFu) - 8.0f);
        } else {
            const h2 off = {static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-1032.0f)};
            const unsigned sel = 0x0C000C00u | static_cast<unsigned>(t) | (static_cast<unsigned>(4 + t) << 16);
            const unsigned b = __builtin_amdgcn_perm(hi, lo, sel) | 0x64006400u;  // 1024 + nibble
            r[t] = __builtin_bit_cast(int, __builtin_bit_cast(h2, b) + off);
        }
    }
    return r;
}

// The pieces a thread stages: 8 fp32 columns, 8 fp16 or 16 int8.
template <typename XT>
struct XPiece;
template <>
struct XPiece<float> {
    static constexpr int kCols = 8, kPlanes = 3, kElem = 2;
    float v[8];
    __device__ __forceinline__ void load(const float* p) {
        const f4 a = __builtin_bit_cast(f4, load16(p)), b = __builtin_bit_cast(f4, load16(p + 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] = a[e];
            v[4 + e] = b[e];
        }
    }
    __device__ __forceinline__ void load_tail(const float* row, int c, int k) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float f = row[min(c + e, k - 1)];
            v[e] = c + e < k ? f : 0.0f;
        }
    }
    template <bool FINE>
    __device__ __forceinline__ void store(int8_t* dst, int plane, unsigned& lost) const {
        v4i h, m, l;
        split3<FINE>(v, h, m, l, lost);
        *reinterpret_cast<v4i*>(dst) = h;
        *reinterpret_cast<v4i*>(dst + plane) = m;
        *reinterpret_cast<v4i*>(dst + 2 * plane) = l;
    }
};
template <>
struct XPiece<_Float16> {
    static constexpr int kCols = 8, kPlanes = 1, kElem = 2;
    v4i v;
    __device__ __forceinline__ void load(const _Float16* p) { v = load16(p); }
    __device__ __forceinline__ void load_tail(const _Float16* row, int c, int k) {
        h8 t;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const _Float16 f = row[min(c + e, k - 1)];
            t[e] = c + e < k ? f : static_cast<_Float16>(0.0f);
        }
        v = __builtin_bit_cast(v4i, t);
    }
    template <bool>
    __device__ __forceinline__ void store(int8_t* dst, int, unsigned&) const { *reinterpret_cast<v4i*>(dst) = v; }
};
template <>
struct XPiece<int8_t> {
    static constexpr int kCols = 16, kPlanes = 1, kElem = 1;
    v4i v;
    __device__ __forceinline__ void load(const int8_t* p) { v = load16(p); }
    __device__ __forceinline__ void load_tail(const int8_t* row, int c, int k) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            unsigned u = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int cc = c + 4 * d + e;
                const unsigned b = static_cast<uint8_t>(row[min(cc, k - 1)]);
                u |= (cc < k ? b : 0u) << (8 * e);
            }
            v[d] = static_cast<int>(u);
        }
    }
    template <bool>
    __device__ __forceinline__ void store(int8_t* dst, int, unsigned&) const { *reinterpret_cast<v4i*>(dst) = v; }
};

// PC (8 or 16) weight columns of one row. Columns past k keep whatever code the
// row's last byte holds: the activations there are zeros.
template <bool Q4, int PC>
struct WPiece {
    static constexpr int kDwords = PC / (Q4 ? 8 : 4);
    int v[kDwords];
    __device__ __forceinline__ void load(const uint8_t* row, int c) { __builtin_memcpy(v, row + (Q4 ? c >> 1 : c), 4 * kDwords); }
    __device__ __forceinline__ void load_tail(const uint8_t* row, int c, int rb) {
#pragma unroll
        for (int d = 0; d < kDwords; ++d) {
            unsigned u = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                u |= static_cast<unsigned>(row[min((Q4 ? c >> 1 : c) + 4 * d + e, rb - 1)]) << (8 * e);
            v[d] = static_cast<int>(u);
        }
    }
    // columns 8h..8h+7 as eight bf16 or fp16
    template <bool BF>
    __device__ __forceinline__ v4i codes(int h) const {
        if constexpr (Q4) return codes_q4<BF>(v[h]);
        else return codes_q8<BF>(v[2 * h], v[2 * h + 1]);
    }
};

template <int C>
__device__ __forceinline__ int tile_swz(int r) {  // slot XOR of row r, C 16-byte chunks per row
    return (r >> 1) & (C - 1);
}

template <typename XT, WF F, int WM, int WN, int FM, int FN, int SK>
struct TileShape {
    using XP = XPiece<XT>;
    static constexpr int kThreads = WM * WN * 64, kBM = WM * FM * 16, kBN = WN * FN * 16;
    static constexpr int kRow = SK * XP::kElem, kC = kRow / 16;    // LDS bytes and chunks per row
    static constexpr int kStep = 64 / XP::kElem, kT = SK / kStep;  // columns per MFMA, MFMA steps per slab
    static constexpr int kPlane = kBM * kRow, kWOff = kPlane * XP::kPlanes, kSOff = kWOff + kBN * kRow;
    static constexpr int kScales = is_grouped(F) ? kT * kBN : 0;
    static constexpr int kBuf = kSOff + kScales * 4;
    static constexpr int kXCpr = SK / XP::kCols, kXU = kBM * kXCpr, kNX = (kXU + kThreads - 1) / kThreads;
    static constexpr int kPC = SK == 32 ? 8 : 16, kWCpr = SK / kPC, kWU = kBN * kWCpr, kNW = (kWU + kThreads - 1) / kThreads;
    static constexpr int kNS = (kScales + kThreads - 1) / kThreads;
    static constexpr size_t kLds = 2 * size_t(kBuf);
    static_assert(kC == 4 || kC == 8, "swizzle");
    static_assert(kLds <= 160 * 1024, "LDS");
};

struct TileArgs {
    const void* x;
    const uint8_t* w;
    const void* scale;   // Q8 / Q4Row: per row; Q4G*: [n, groups]
    const float* a_scale;  // int8 activations: per row of x
    const float* bias;
    void* y;
    void* planes;  // raw sums [splits][m][n], fp32 (int32 for int8 activations), when K is split
    int m, n, k, groups, cpg;  // cpg: 32-column chunks per group
    unsigned cpg_magic;        // ceil(2^32 / cpg): chunk / cpg == umulhi(chunk, magic)
    int tiles_m, tiles_n, gm, per;  // gm: row tiles per group of the tile order; per: slabs per K range
    int scale_f16, y_kind;      // y_kind: 0 fp32, 1 fp16, 2 int32 accumulators
};

__device__ __forceinline__ int chunk_group(const TileArgs& a, int chunk) {
    return a.cpg == 1 ? chunk : static_cast<int>(__umulhi(static_cast<unsigned>(chunk), a.cpg_magic));
}
__device__ __forceinline__ float tile_scale(const TileArgs& a, size_t i) {
    return a.scale_f16 ? static_cast<float>(static_cast<const _Float16*>(a.scale)[i]) : static_cast<const float*>(a.scale)[i];
}

template <typename XT, WF F, int WM, int WN, int FM, int FN, int SK>
__global__ __launch_bounds__((WM * WN * 64)) void tile_gemm_kernel(TileArgs a) {
    using S = TileShape<XT, F, WM, WN, FM, FN, SK>;
    using XP = XPiece<XT>;
    constexpr bool I8 = sizeof(XT) == 1, BF = sizeof(XT) == 4, Q4 = is_q4(F), GROUPED = is_grouped(F);
    constexpr int NT = S::kThreads, T = S::kT, C = S::kC;
    constexpr bool FINE = F != WF::Q8;  // never for int8 activations, whose sums are exact
    using Acc = std::conditional_t<I8, v4i, f4>;
    using Sum = std::conditional_t<FINE, d4, Acc>;
    extern __shared__ __attribute__((aligned(16))) int8_t tile_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WN, wn = wave % WN, fr = lane & 15, fq = lane >> 4;
    // Consecutive workgroups go round-robin over the 8 XCDs: each takes a contiguous
    // range of the tiles, which are ordered in groups of `gm` row tiles, row tile
    // fastest, column tiles next: an XCD's L2 then keeps the group's activation rows.
    const int total = a.tiles_m * a.tiles_n;
    const int per = (total + 7) / 8, xcd = blockIdx.x % 8, idx = blockIdx.x / 8;
    const int full = total - 8 * (per - 1);
    const int lin = xcd < full ? xcd * per + idx : full * per + (xcd - full) * (per - 1) + idx;
    const int grp = lin / (a.gm * a.tiles_n), in = lin - grp * a.gm * a.tiles_n, rows = min(a.gm, a.tiles_m - grp * a.gm);
    const int m0 = (grp * a.gm + in % rows) * S::kBM, n0 = in / rows * S::kBN;
    const int m = a.m, n = a.n, k = a.k, rb = Q4 ? (k + 1) / 2 : k;

    // This range: whole slabs [s0, s1), and the tail slab if it is the last range's.
    const int whole = k / SK, slabs = (k + SK - 1) / SK;
    const int s0 = static_cast<int>(blockIdx.y) * a.per, end = min(slabs, s0 + a.per), s1 = min(whole, end);
    const int tail = end > whole ? 1 : 0, nk = end - s0;

    const XT* xr[S::kNX];
    const uint8_t* wr[S::kNW];
#pragma unroll
    for (int u = 0; u < S::kNX; ++u)
        xr[u] = static_cast<const XT*>(a.x) + static_cast<size_t>(min(m0 + (tid + u * NT) / S::kXCpr, m - 1)) * k;
#pragma unroll
    for (int u = 0; u < S::kNW; ++u)
        wr[u] = a.w + static_cast<size_t>(min(n0 + (tid + u * NT) / S::kWCpr, n - 1)) * rb;

    struct Stage {
        XP x[S::kNX];
        WPiece<Q4, S::kPC> w[S::kNW];
        float s[S::kNS > 0 ? S::kNS : 1];
    };
    auto load_scales = [&](int slab, Stage& st) {
        if constexpr (GROUPED) {
#pragma unroll
            for (int u = 0; u < S::kNS; ++u) {
                const int i = tid + u * NT, row = min(n0 + i % S::kBN, n - 1);
                const int chunk = slab * T + min(i / S::kBN, T - 1);  // int4 slabs: one chunk per MFMA step
                const int g = min(chunk_group(a, chunk), a.groups - 1);
                st.s[u] = tile_scale(a, static_cast<size_t>(row) * a.groups + g);
            }
        }
    };
    auto load = [&](int slab, Stage& st) {  // a whole slab
#pragma unroll
        for (int u = 0; u < S::kNX; ++u) st.x[u].load(xr[u] + slab * SK + (tid + u * NT) % S::kXCpr * XP::kCols);
#pragma unroll
        for (int u = 0; u < S::kNW; ++u) st.w[u].load(wr[u], slab * SK + (tid + u * NT) % S::kWCpr * S::kPC);
        load_scales(slab, st);
    };
    auto load_tail = [&](Stage& st) {
#pragma unroll
        for (int u = 0; u < S::kNX; ++u)
            st.x[u].load_tail(xr[u], whole * SK + (tid + u * NT) % S::kXCpr * XP::kCols, k);
#pragma unroll
        for (int u = 0; u < S::kNW; ++u) st.w[u].load_tail(wr[u], whole * SK + (tid + u * NT) % S::kWCpr * S::kPC, rb);
        load_scales(whole, st);
    };
    unsigned lost[S::kNX] = {};
    auto store = [&](const Stage& st, int8_t* buf) {
#pragma unroll
        for (int u = 0; u < S::kNX; ++u) {
            const int i = tid + u * NT, r = i / S::kXCpr, c = i % S::kXCpr;
            if (S::kXU % NT == 0 || i < S::kXU) st.x[u].template store<FINE>(buf + r * S::kRow + ((c ^ tile_swz<C>(r)) << 4), S::kPlane, lost[u]);
        }
#pragma unroll
        for (int u = 0; u < S::kNW; ++u) {
            const int i = tid + u * NT, r = i / S::kWCpr, c = i % S::kWCpr;
            if (S::kWU % NT == 0 || i < S::kWU) {
                int8_t* row = buf + S::kWOff + r * S::kRow;
                if constexpr (I8) {
                    v4i t;
                    __builtin_memcpy(&t, st.w[u].v, 16);
                    *reinterpret_cast<v4i*>(row + ((c ^ tile_swz<C>(r)) << 4)) = t;
                } else {
#pragma unroll
                    for (int h = 0; h < S::kPC / 8; ++h)
                        *reinterpret_cast<v4i*>(row + (((S::kPC / 8 * c + h) ^ tile_swz<C>(r)) << 4)) = st.w[u].template codes<BF>(h);
                }
            }
        }
        if constexpr (GROUPED) {
#pragma unroll
            for (int u = 0; u < S::kNS; ++u) {
                const int i = tid + u * NT;
                if (S::kScales % NT == 0 || i < S::kScales) reinterpret_cast<float*>(buf + S::kSOff)[i] = st.s[u];
            }
        }
    };

    // Sums in two levels, as one chain over all of K rounds its running sum once per MFMA:
    // `part` holds the sums of 256 columns, and fp32 activations start each chunk's three
    // products from zero, largest part first. (Smallest first is as good on one linear
    // but leaves a mean error: the MFMA cuts the low bits of the sum it is given when
    // larger products join, always downwards, m = 384, n = 896, k = 4864 -7.7e-8 of the rms
    // against -1e-9, and a decoder's attention averages over such a shift without
    // shrinking it: 2 layers, 384 tokens, int4 logits 6.5e-7 off and not 3.6e-7. Adding
    // the largest part's product separately costs 5%.)
    // Q8 on 16-byte rows of whole chunks stands for kernels of one chain: its larger
    // fp32 tiles add each chunk to the sum itself, as `part` costs them the second
    // workgroup of a CU (m = 333, n = 1536, k = 8960 47 -> 54 us).
    // FINE, all others, stands for kernels that summed K in 64 lanes and a tree: it adds
    // the parts in fp64 and sums again in fp64 what three bf16 parts cannot hold. Errors
    // against 64 bits, those kernels / fp32 sums of the parts / this: one int4 group per
    // row, fp32, m = 333, n = 9000, k = 8960 1.1e-7 / 2.3e-7 / 0.9e-7; groups of 64, fp16, k =
    // 9000 7.5e-8 / 15e-8 / 4e-8; int8, fp32, k = 1003 1.02e-7 / 1.30e-7 / 0.94e-7. us, fp32
    // sums -> this: int4 fp32, m = 333, n = 1536, k = 8960 groups of 32 61 -> 66, one group
    // 51 -> 63; m = 1500, n = 6768, k = 2160 int8 fp32 182 -> 216, fp16 98 -> 102.
    constexpr bool PART = !I8 && (FINE || !BF || FN * FM <= 4);
    constexpr int kPart = FINE && !BF && !GROUPED ? 128 : 256;  // columns of a part
    Sum acc[FN][FM];
    Acc part[PART ? FN : 1][PART ? FM : 1];
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) {
            acc[i][j] = Sum{0, 0, 0, 0};
            if constexpr (PART) part[i][j] = Acc{0, 0, 0, 0};
        }
    const int xrow = wm * FM * 16 + fr, wrow = wn * FN * 16 + fr;
    const int xsw = tile_swz<C>(xrow), wsw = tile_swz<C>(wrow);  // a 16-row step keeps the swizzle
    // The MFMAs of a slab in LDS; flush(t): whether step t closes a part.
    auto compute = [&](const int8_t* buf, auto flush) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            v4i xa[XP::kPlanes][FM], wb[FN];
            const int8_t* px = buf + xrow * S::kRow + (((t * 4 + fq) ^ xsw) << 4);
            const int8_t* pw = buf + S::kWOff + wrow * S::kRow + (((t * 4 + fq) ^ wsw) << 4);
#pragma unroll
            for (int i = 0; i < FN; ++i) wb[i] = *reinterpret_cast<const v4i*>(pw + i * 16 * S::kRow);
#pragma unroll
            for (int p = 0; p < XP::kPlanes; ++p)
#pragma unroll
                for (int j = 0; j < FM; ++j) xa[p][j] = *reinterpret_cast<const v4i*>(px + p * S::kPlane + j * 16 * S::kRow);
            float sc[GROUPED ? FN : 1];
            if constexpr (GROUPED) {
#pragma unroll
                for (int i = 0; i < FN; ++i)
                    sc[i] = reinterpret_cast<const float*>(buf + S::kSOff)[t * S::kBN + wrow + i * 16];
            }
            const bool close = PART && flush(t);
#pragma unroll
            for (int i = 0; i < FN; ++i) {
#pragma unroll
                for (int j = 0; j < FM; ++j) {
                    if constexpr (I8) {
                        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(xa[0][j], wb[i], acc[i][j], 0, 0, 0);
                    } else {
                        Acc d = Acc{0, 0, 0, 0};
                        if constexpr (BF) {
#pragma unroll
                            for (int p = 0; p < 3; ++p)
                                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8, xa[p][j]),
                                                                            __builtin_bit_cast(b8, wb[i]), d, 0, 0, 0);
                        } else {
                            if constexpr (PART && F != WF::Q4G32) d = part[i][j];
                            d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8, xa[0][j]),
                                                                       __builtin_bit_cast(h8, wb[i]), d, 0, 0, 0);
                        }
                        if constexpr (F == WF::Q4G32) {
#pragma unroll
                            for (int v = 0; v < 4; ++v) part[i][j][v] = __builtin_fmaf(d[v], sc[i], part[i][j][v]);
                        } else if constexpr (PART && BF) {
#pragma unroll
                            for (int v = 0; v < 4; ++v) part[i][j][v] += d[v];
                        } else if constexpr (PART) {
                            part[i][j] = d;
                        } else {
#pragma unroll
                            for (int v = 0; v < 4; ++v) acc[i][j][v] += d[v];
                        }
                    }
                }
                if constexpr (F == WF::Q4G32 && FN * FM >= 16) __builtin_amdgcn_sched_barrier(0);  // registers
            }
            if constexpr (F == WF::Q4G32 && FN * FM < 16) __builtin_amdgcn_sched_barrier(0);  // one step's sums at a time
            if constexpr (PART) {
                if (close) {
#pragma unroll
                    for (int i = 0; i < FN; ++i)
#pragma unroll
                        for (int j = 0; j < FM; ++j) {
#pragma unroll
                            for (int v = 0; v < 4; ++v) {
                                // Q4G closes a part with its group's scale; the others add it as it is.
                                if constexpr (F == WF::Q4G)
                                    acc[i][j][v] = __builtin_fma(static_cast<double>(part[i][j][v]), static_cast<double>(sc[i]), acc[i][j][v]);
                                else
                                    acc[i][j][v] += part[i][j][v];
                            }
                            part[i][j] = Acc{0, 0, 0, 0};
                        }
                }
            }
        }
    };

    // Slab i of the range: the tail first, then the whole slabs in order. Loads run
    // two slabs ahead; past the end they repeat the last whole slab, as a branch
    // around them would make the compiler wait for all loads at its end.
    if (s1 > s0) {
        Stage st[2];
        int8_t *cur = tile_lds, *nxt = tile_lds + S::kBuf;
        // position of the next computed chunk in its group (Q4G)
        int pos = 0;
        if constexpr (F == WF::Q4G)
            pos = s0 * T - static_cast<int>(__umulhi(static_cast<unsigned>(s0 * T), a.cpg_magic)) * a.cpg;
        const int first = tail ? s0 - 1 : s0;  // slab i (i >= 1, or i >= 0 without a tail) is first + i
        if (tail) load_tail(st[0]);
        else load(s0, st[0]);
        load(min(first + 1, s1 - 1), st[1]);
        store(st[0], cur);
        __syncthreads();
        auto body = [&](int i, Stage& a0, Stage& a1) {  // a0 free, a1 = slab i + 1
            load(min(first + i + 2, s1 - 1), a0);
            __builtin_amdgcn_sched_barrier(0);  // the loads stay two slabs ahead: left alone they sank to the barrier
            const bool is_tail = tail && i == 0, full = i == nk - 1 || i % (kPart / SK) == 0;
            compute(cur, [&](int t) {
                if constexpr (F == WF::Q4G) {
                    if (is_tail) return true;
                    const bool end_of_group = ++pos == a.cpg;
                    if (end_of_group) pos = 0;
                    return end_of_group || (full && t == T - 1);
                } else {
                    return full && t == T - 1;
                }
            });
            store(a1, nxt);  // past the last slab: a repeat nobody reads
            // The next slab's conversions between this slab's MFMAs: 2 VALU to one MFMA
            // (fp32 Q8, m = 333, n = 1536, k = 8960 47.6 -> 45.2 us; m = 2048, n = 8960, k =
            // 1536 189 -> 178).
            __builtin_amdgcn_sched_group_barrier(0x100, FN + FM * XP::kPlanes, 0);
#pragma unroll
            for (int q = 0; q < FN * FM * T * XP::kPlanes; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
                if (T > 1 && q % 4 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
            }
            int8_t* const t = cur;
            cur = nxt;
            nxt = t;
            __syncthreads();
        };
        int i = 0;
        for (; i + 2 <= nk; i += 2) {
            body(i, st[0], st[1]);
            body(i + 1, st[1], st[0]);
        }
        if (i < nk) body(i, st[0], st[1]);
    } else if (tail) {  // k (or the last range) holds no whole slab
        Stage st;
        load_tail(st);
        store(st, tile_lds);
        __syncthreads();
        compute(tile_lds, [&](int) { return true; });
    }

    const size_t plane = static_cast<size_t>(blockIdx.y) * m * n;
    auto put = [&](int row, int col, float ws, float b, auto sum) {
        const size_t o = static_cast<size_t>(row) * n + col;
        float r;
        if constexpr (I8) {
            if (a.planes) {
                static_cast<int32_t*>(a.planes)[plane + o] = sum;
                return;
            }
            if (a.y_kind == 2) {
                static_cast<int32_t*>(a.y)[o] = sum;
                return;
            }
            r = w8a8_epilogue(sum, a.a_scale[row], ws, b);
        } else {
            if (a.planes) {
                static_cast<float*>(a.planes)[plane + o] = static_cast<float>(sum);
                return;
            }
            r = static_cast<float>(GROUPED ? sum + b : sum * ws + b);
        }
        if (a.y_kind == 1) static_cast<_Float16*>(a.y)[o] = from_f32<_Float16>(r);
        else static_cast<float*>(a.y)[o] = r;
    };
    const bool scaled = !a.planes && a.y_kind != 2;

    // FINE fp32: an output of a row that dropped bits (less than 2^-133 of each value, so
    // 2^-126 of each product with a code) is summed again in fp64 where these are over
    // 2^-27 of it, that is where the whole row is tiny, or where it is no number.
    unsigned* redo = reinterpret_cast<unsigned*>(tile_lds);  // a bit per output of the tile
    __shared__ unsigned lost_rows[(S::kBM + 31) / 32];
    unsigned any_lost = 0;
    double least[FN] = {};
    if constexpr (FINE && BF) {
        constexpr int words = (S::kBM + 31) / 32;
        if (tid < words) lost_rows[tid] = 0;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < S::kNX; ++u) {
            const int r = (tid + u * NT) / S::kXCpr;
            if (lost[u]) atomicOr(&lost_rows[r >> 5], 1u << (r & 31));
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < words; ++i) any_lost |= lost_rows[i];
        if (any_lost) {
            for (int i = tid; i < S::kBM * S::kBN / 32; i += NT) redo[i] = 0;
#pragma unroll
            for (int i = 0; i < FN; ++i) {
                float top = GROUPED ? 0.0f : 1.0f;
                if constexpr (GROUPED)
                    for (int g = 0; g < a.groups; ++g)
                        top = fmaxf(top, fabsf(tile_scale(a, static_cast<size_t>(min(n0 + wrow + i * 16, n - 1)) * a.groups + g)));
                least[i] = 0x1p-99 * (nk * SK) * top;
            }
            __syncthreads();
        }
    }
    // Lane l holds, of fragment (i, j), rows 4 * (l / 16) + v of column l % 16.
#pragma unroll
    for (int i = 0; i < FN; ++i) {
        const int col = n0 + wrow + i * 16;
        if (col >= n) continue;
        const float ws = scaled && !GROUPED ? tile_scale(a, col) : 1.0f, b = scaled && a.bias ? a.bias[col] : 0.0f;
#pragma unroll
        for (int j = 0; j < FM; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = wm * FM * 16 + j * 16 + 4 * fq + v;
                if (m0 + r >= m) continue;
                if constexpr (FINE && BF) {
                    const double t = fabs(acc[i][j][v]);
                    if (any_lost && (lost_rows[r >> 5] >> (r & 31) & 1) && !(t >= least[i] && t < __builtin_inf())) {
                        const int e = r * S::kBN + col - n0;
                        atomicOr(&redo[e >> 5], 1u << (e & 31));
                        continue;
                    }
                }
                put(m0 + r, col, ws, b, acc[i][j][v]);
            }
    }
    if constexpr (FINE && BF) {
        if (!any_lost) return;
        __syncthreads();
        for (int e = tid; e < S::kBM * S::kBN; e += NT) {
            if (!(redo[e >> 5] >> (e & 31) & 1)) continue;
            const int row = m0 + e / S::kBN, col = n0 + e % S::kBN;
            const XT* xp = static_cast<const XT*>(a.x) + static_cast<size_t>(row) * k;
            const uint8_t* wp = a.w + static_cast<size_t>(col) * rb;
            double sum = 0.0;
            for (int c = s0 * SK; c < min(k, end * SK); ++c) {
                const int q = Q4 ? ((wp[c >> 1] >> (4 * (c & 1))) & 15) - 8 : static_cast<int8_t>(wp[c]);
                double t = static_cast<double>(xp[c]) * q;
                if constexpr (GROUPED) t *= tile_scale(a, static_cast<size_t>(col) * a.groups + chunk_group(a, c >> 5));
                sum += t;
            }
            put(row, col, scaled && !GROUPED ? tile_scale(a, col) : 1.0f, scaled && a.bias ? a.bias[col] : 0.0f, sum);
        }
    }
}

// Sums the raw planes [splits][m][n] in plane order, then scales and adds as the
// unsplit epilogue does. All of an output's loads are issued before the first add.
constexpr int kTileMaxSplits = 16;
template <bool I8>
__global__ __launch_bounds__(256) void tile_reduce_kernel(TileArgs a, int splits, int row_scale) {
    const size_t mn = static_cast<size_t>(a.m) * a.n, i = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= mn) return;
    using V = std::conditional_t<I8, int32_t, float>;
    const V* part = static_cast<const V*>(a.planes);
    V v[kTileMaxSplits];
#pragma unroll
    for (int sp = 0; sp < kTileMaxSplits; ++sp)
        if (sp < splits) v[sp] = part[sp * mn + i];
    std::conditional_t<I8, int32_t, double> t = v[0];
#pragma unroll
    for (int sp = 1; sp < kTileMaxSplits; ++sp)
        if (sp < splits) t += v[sp];
    if constexpr (I8) {
        if (a.y_kind == 2) {
            static_cast<int32_t*>(a.y)[i] = t;
            return;
        }
    }
    const int col = static_cast<int>(i % a.n);
    const float ws = row_scale ? tile_scale(a, col) : 1.0f;
    const float b = a.bias ? a.bias[col] : 0.0f;
    float r;
    if constexpr (I8) r = w8a8_epilogue(t, a.a_scale[i / a.n], ws, b);
    else r = static_cast<float>(t * ws + b);
    if (a.y_kind == 1) static_cast<_Float16*>(a.y)[i] = from_f32<_Float16>(r);
    else static_cast<float*>(a.y)[i] = r;
}

// ---- plan ------------------------------------------------------------------------------
// Tiles by falling area. A tile's time per slab is `alone` us with its CU to itself and
// `shared` us times the workgroups of its CU once they fill it, over `extra` slabs more
// than it has (first loads, stores); a split adds a launch and the planes' traffic.
// Least-squares fit to the measured (shape, tile, split) points of 5400 shapes (m
// 5..2048, n 128..18432, k 1..9216): the pick is 1.5% slower than the measured best on
// average, 5% at the 90th percentile. The points of the fine sums' rows are int4 groups with
// fp32 sums of the parts; with fp64 ones the larger tiles take up to a fifth longer.
struct TileCost {
    float extra, alone, shared;
};
struct TileModel {
    float launch, reduce, plane_tbs;  // us, us, TB/s
    TileCost t[5];
};
struct TileDim {
    int bm, bn;
};
constexpr int kTileCount = 5;
constexpr TileDim kTiles[kTileCount] = {{128, 128}, {64, 128}, {64, 64}, {32, 64}, {16, 64}};
constexpr TileModel kTileModels[] = {
    // fp32 activations; the same with fine sums; fp16; with fine sums; int8
    {4.5f, 1.1f, 2.9f, {{3.1f, 0.898f, 0.657f}, {3.5f, 0.7f, 0.422f}, {2.8f, 0.462f, 0.288f}, {1.1f, 0.476f, 0.209f}, {0.4f, 0.362f, 0.164f}}},
    {4.5f, 1.2f, 2.8f, {{3.1f, 0.982f, 0.921f}, {3.3f, 0.756f, 0.477f}, {2.4f, 0.513f, 0.322f}, {1.f, 0.463f, 0.269f}, {0.f, 0.397f, 0.243f}}},
    {4.1f, 1.4f, 4.f, {{7.7f, 0.843f, 0.574f}, {6.2f, 0.576f, 0.371f}, {5.f, 0.364f, 0.234f}, {2.7f, 0.252f, 0.17f}, {1.1f, 0.258f, 0.162f}}},
    {3.7f, 1.5f, 3.9f, {{6.6f, 1.02f, 0.781f}, {5.5f, 0.681f, 0.457f}, {4.4f, 0.455f, 0.292f}, {2.2f, 0.381f, 0.237f}, {1.f, 0.367f, 0.232f}}},
    {4.1f, 1.6f, 5.9f, {{10.7f, 0.762f, 0.561f}, {8.6f, 0.492f, 0.382f}, {6.7f, 0.328f, 0.258f}, {4.1f, 0.245f, 0.201f}, {2.6f, 0.23f, 0.179f}}},
};
constexpr int64_t kTilePlanesMax = int64_t(64) << 20;  // bytes of split-K planes

struct TilePlan {
    int cfg, splits;
    double us;  // modelled time
};
TilePlan model_plan(TileX xt, bool fine, int64_t m, int64_t n, int64_t k, int64_t ws_bytes) {
    const TileModel& mod = kTileModels[xt == TileX::I8 ? 4 : (xt == TileX::F16 ? 2 : 0) + (fine ? 1 : 0)];
    const int64_t sk = xt == TileX::F32 ? 32 : xt == TileX::F16 ? 64 : 128, slabs = (k + sk - 1) / sk;
    const double mn = static_cast<double>(m) * n;
    TilePlan best{kTileCount - 1, 1, 0};
    for (int c = 0; c < kTileCount; ++c) {
        // never the best: rows of a tile mostly empty, or tens of tiles along m
        if (c < kTileCount - 1 && (kTiles[c].bm >= 4 * m || (c > 1 && m > 32 * kTiles[c].bm))) continue;
        const int64_t tiles = ((m + kTiles[c].bm - 1) / kTiles[c].bm) * ((n + kTiles[c].bn - 1) / kTiles[c].bn);
        for (int want : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (want > 1 && (slabs < 2 * want || tiles * want > 2048)) break;
            const int64_t per = (slabs + want - 1) / want, splits = (slabs + per - 1) / per;
            if (want > 1 && (splits < 2 || per < 2 || splits * mn * 4 > std::min(ws_bytes, kTilePlanesMax))) continue;
            const double q = static_cast<double>((tiles * splits + 255) / 256);
            double t = mod.launch + (per + mod.t[c].extra) * std::max<double>(mod.t[c].alone, q * mod.t[c].shared);
            // the second launch costs its caller 1.5 us more than the GPU
            if (splits > 1) t += 1.5 + mod.reduce + (splits + 1) * mn * 4e-6 / mod.plane_tbs;
            if (best.us == 0 || t < best.us) best = {c, static_cast<int>(splits), t};
        }
    }
    return best;
}

// The plan of a shape, modelled once per thread while it stays among the last seen: a call
// asks for up to six plans (each type's workspace, the route, the launch), 0.3 to 1 us each.
TilePlan plan_tile(TileX xt, bool fine, int64_t m, int64_t n, int64_t k, int64_t ws_bytes) {
    struct Seen {
        int64_t m, n, k, ws;
        int kind;
        TilePlan plan;
    };
    constexpr unsigned kSeen = 64;
    static thread_local Seen seen[kSeen];  // m = 0: empty
    const int kind = static_cast<int>(xt) * 2 + (fine ? 1 : 0);
    const uint64_t h = (static_cast<uint64_t>(m) * 0x9E3779B97F4A7C15u) ^ (static_cast<uint64_t>(n) * 0xC2B2AE3D27D4EB4Fu) ^
                       (static_cast<uint64_t>(k) * 0x165667B19E3779F9u) ^ (static_cast<uint64_t>(ws_bytes) * 0xD6E8FEB86659FD93u) ^
                       (static_cast<uint64_t>(kind) << 58);
    Seen& e = seen[h >> 58];
    if (e.m != m || e.n != n || e.k != k || e.ws != ws_bytes || e.kind != kind)
        e = {m, n, k, ws_bytes, kind, model_plan(xt, fine, m, n, k, ws_bytes)};
    return e.plan;
}

template <typename XT, WF F, int WM, int WN, int FM, int FN>
nq_status launch_tile(TileArgs a, int splits, hipStream_t s) {
    constexpr int SK = sizeof(XT) == 4 ? 32 : sizeof(XT) == 2 ? 64 : 128;
    using S = TileShape<XT, F, WM, WN, FM, FN, SK>;
    auto* fn = tile_gemm_kernel<XT, F, WM, WN, FM, FN, SK>;
    if (nq_status st = set_dynamic_lds(reinterpret_cast<const void*>(fn), S::kLds, "tile_gemm")) return st;
    a.tiles_m = (a.m + S::kBM - 1) / S::kBM;
    a.tiles_n = (a.n + S::kBN - 1) / S::kBN;
    const int slabs = (a.k + SK - 1) / SK;
    if (!a.planes) splits = 1;
    a.per = (slabs + splits - 1) / splits;
    // Row tiles per group of the tile order: about 1 MB of activations, a quarter of an
    // XCD's L2 (m = 2048, n = 8960, k = 1536, all 32 row tiles of 64 against 8: fp16
    // 100.8 -> 90.3 us, int8 64.4 -> 59.5; fp32 196 -> 181), and at least 4.
    a.gm = std::max<int64_t>(4, (int64_t(1) << 20) / (int64_t(S::kBM) * a.per * SK * int64_t(sizeof(XT))));
    a.gm = std::min(a.gm, a.tiles_m);
    splits = (slabs + a.per - 1) / a.per;  // no empty range
    if (splits <= 1) a.planes = nullptr;
    fn<<<dim3(static_cast<unsigned>(a.tiles_m) * a.tiles_n, splits), S::kThreads, S::kLds, s>>>(a);
    if (nq_status st = launch_status("tile_gemm_kernel")) return st;
    if (splits <= 1) return NQ_OK;
    const size_t mn = static_cast<size_t>(a.m) * a.n;
    tile_reduce_kernel<sizeof(XT) == 1><<<static_cast<unsigned>((mn + 255) / 256), 256, 0, s>>>(a, splits, !is_grouped(F));
    return launch_status("tile_reduce_kernel");
}

template <typename XT, WF F>
nq_status launch_tile_cfg(const TileArgs& a, int cfg, int splits, hipStream_t s) {
    switch (cfg) {
        case 0:
            // fp32 activations and fp64 sums: eight waves, as three planes of fragments (the
            // sums) per wave of four leave too few registers
            if constexpr (sizeof(XT) == 4 || F != WF::Q8) return launch_tile<XT, F, 4, 2, 2, 4>(a, splits, s);
            else return launch_tile<XT, F, 2, 2, 4, 4>(a, splits, s);
        case 1: return launch_tile<XT, F, 2, 2, 2, 4>(a, splits, s);
        case 2: return launch_tile<XT, F, 2, 2, 2, 2>(a, splits, s);
        case 3: return launch_tile<XT, F, 1, 4, 2, 1>(a, splits, s);
        default: return launch_tile<XT, F, 1, 4, 1, 1>(a, splits, s);
    }
}

template <typename XT>
nq_status launch_tile_fmt(const TileArgs& a, WF f, int cfg, int splits, hipStream_t s) {
    switch (f) {
        case WF::Q8: return launch_tile_cfg<XT, WF::Q8>(a, cfg, splits, s);
        case WF::Q4G32: return launch_tile_cfg<XT, WF::Q4G32>(a, cfg, splits, s);
        case WF::Q8Fine: return launch_tile_cfg<XT, WF::Q8Fine>(a, cfg, splits, s);
        case WF::Q4Row: return launch_tile_cfg<XT, WF::Q4Row>(a, cfg, splits, s);
        default: return launch_tile_cfg<XT, WF::Q4G>(a, cfg, splits, s);
    }
}

}  // namespace

bool tile_gemm_ok(bool q4, int64_t m, int64_t n, int64_t k, int64_t group) {
    if (m < 1 || n < 1 || k < 1 || m > kMaxIndex || n > kMaxIndex || k > (int64_t(1) << 20)) return false;
    if (q4 && group < k && group % 32 != 0) return false;
    return ((m + 15) / 16) * ((n + 63) / 64) <= (int64_t(1) << 24);  // tiles, and chunks * cpg, in 32 bits
}

size_t tile_gemm_ws_bytes(TileX xt, bool fine, int64_t m, int64_t n, int64_t k) {
    const TilePlan p = plan_tile(xt, fine, m, n, k, kTilePlanesMax);
    return p.splits > 1 ? round_up(static_cast<size_t>(p.splits) * m * n * 4, 256) : 0;
}

bool tile_gemm_split_fits(TileX xt, bool fine, int64_t m, int64_t n, int64_t k, size_t ws_bytes) {
    const TilePlan best = plan_tile(xt, fine, m, n, k, kTilePlanesMax);
    if (best.splits < 2 || static_cast<size_t>(best.splits) * m * n * 4 <= ws_bytes) return true;
    return plan_tile(xt, fine, m, n, k, static_cast<int64_t>(ws_bytes)).us <= (xt == TileX::F32 ? 1.15 : 1.05) * best.us;
}

nq_status tile_gemm(const TileCall& c, void* ws, size_t ws_bytes, hipStream_t s) {
    const bool row = c.q4 && c.group >= c.k, grouped = c.q4 && !row;
    const TilePlan p = plan_tile(c.xt, c.q4 || c.fine, c.m, c.n, c.k, ws ? static_cast<int64_t>(std::min<size_t>(ws_bytes, kTilePlanesMax)) : 0);
    TileArgs a{};
    a.x = c.x;
    a.w = c.w;
    a.scale = c.scale;
    a.a_scale = c.a_scale;
    a.bias = c.bias;
    a.y = c.y;
    a.planes = p.splits > 1 ? ws : nullptr;
    a.m = static_cast<int>(c.m);
    a.n = static_cast<int>(c.n);
    a.k = static_cast<int>(c.k);
    a.scale_f16 = c.scale_f16;
    a.y_kind = c.yt;
    a.cpg = grouped ? static_cast<int>(c.group / 32) : 1;
    a.groups = grouped ? static_cast<int>((c.k + c.group - 1) / c.group) : 1;
    a.cpg_magic = a.cpg > 1 ? static_cast<unsigned>(((uint64_t(1) << 32) + a.cpg - 1) / a.cpg) : 0;
    const WF f = !c.q4 ? c.fine ? WF::Q8Fine : WF::Q8 : row ? WF::Q4Row : c.group == 32 ? WF::Q4G32 : WF::Q4G;
    if (c.xt == TileX::F32) return launch_tile_fmt<float>(a, f, p.cfg, p.splits, s);
    if (c.xt == TileX::F16) return launch_tile_fmt<_Float16>(a, f, p.cfg, p.splits, s);
    return launch_tile_cfg<int8_t, WF::Q8>(a, p.cfg, p.splits, s);
}

}  // namespace nq
