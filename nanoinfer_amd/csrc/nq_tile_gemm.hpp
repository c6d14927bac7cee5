// Linears over any K, row alignment and group of whole 32-column chunks (nq_tile_gemm.hip).
#pragma once

#include "nq_internal.hpp"

namespace nq {

enum class TileX { F32, F16, I8 };        // activations; I8: codes with a_scale per row
enum TileY { kTileF32, kTileF16, kTileI32 };  // results; I32: raw accumulators (I8 only)

struct TileCall {
    TileX xt;
    const void* x;
    const uint8_t* w;
    bool q4;              // nibbles in groups of `group` columns (one group per row when group >= k), else int8
    const void* scale;    // per weight row, or [n, ceil(k / group)]; unused for I32
    bool scale_f16;
    int64_t group;
    const float* a_scale;
    const float* bias;
    void* y;
    TileY yt;
    int64_t m, n, k;
    bool fine;  // int8 codes, F32 / F16: sums no coarser than 64 lanes and a tree (int4: always)
};

// Whether the tile GEMM takes these operands: any pointer alignment, any k up to 2^20.
bool tile_gemm_ok(bool q4, int64_t m, int64_t n, int64_t k, int64_t group);
// Workspace its split-K planes take at this shape (0: no split); less or none is accepted
// and splits less. fine: int4 codes, or TileCall::fine.
size_t tile_gemm_ws_bytes(TileX xt, bool fine, int64_t m, int64_t n, int64_t k);
// Whether the plan within ws_bytes comes near the unlimited one: within 15% (F32) or 5%, as
// past that the kernels with planes of their own are the faster ones on average.
bool tile_gemm_split_fits(TileX xt, bool fine, int64_t m, int64_t n, int64_t k, size_t ws_bytes);
nq_status tile_gemm(const TileCall& c, void* ws, size_t ws_bytes, hipStream_t s);

// The same operands at m <= 8 (nq_gemv_any.hip); no workspace.
nq_status gemv_any(const TileCall& c, hipStream_t s);

}  // namespace nq
