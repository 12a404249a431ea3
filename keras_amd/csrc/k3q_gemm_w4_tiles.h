// Launch of the int4 tile kernel (k3q_gemm_w4_tiles.hip) for the entry points in k3q_gemv_w4.hip.
#pragma once

#include "k3q_common.h"

namespace k3q {

// How the nibbles become bfloat16: 136 + q and 24 + w (an offset, taken out again with the sums of x), or the integers
// w - zero themselves.
constexpr int kW4Form136 = 0, kW4Form24 = 1, kW4FormPlain = 2;

struct W4TilePlan {
    int mb;      // blocks of 32 rows per tile: 1, 2 or 4
    int bn;      // columns per tile: 128 (K in two slices), or 256 with mb = 4
    int ks;      // workgroups that share K
    int steps;   // of a workgroup, each kq() units of K: ks and steps cover K with this plan's own bn only
    int kq() const { return 256 / bn; }
};

struct W4TileCall {
    const uint16_t* x;    // [parts * rows, K] bfloat16, K % 128 == 0; part h of row m is row h * rows + m
    int64_t rows, K, N;   // N % 32 == 0: the columns of the copy
    int parts;            // 1, or 2 or 3 bfloat16 rows per row
    const void* w;        // strip-linear copy
    int form;
    bool grouped;         // groups of 128 with scales [K / 128, N] and zero points; else one scale per column
    bool f32;             // scales, bias and result are float32
    const void* scale;
    const int8_t* zero;
    const v2u* sx;        // [K / 128, parts * rows]: sums of x over groups of 128, as three bfloat16 parts (form 136 and 24)
    const void* bias;
    int64_t bias_stride;
    void* y;              // [rows, n_out], n_out <= N; not written when the plan splits K or parts == 3
    int64_t n_out;
    float* part;          // [ks][parts * rows][N]: the raw sums in that case
};

// Whether a call's result comes from the tile kernel itself (otherwise a second pass adds the partial sums).
inline bool w4_tile_direct(const W4TilePlan& pl, int parts) { return pl.ks == 1 && parts < 3; }

// Whether the kernel's 32-bit lane offsets reach every operand.
bool w4_tile_fits(int64_t rows, int parts, int64_t K, int64_t N);
W4TilePlan w4_tile_plan(int64_t rows, int parts, int64_t K, int64_t N);
int w4_tile_launch(const W4TileCall& c, const W4TilePlan& pl, hipStream_t s);

}  // namespace k3q
