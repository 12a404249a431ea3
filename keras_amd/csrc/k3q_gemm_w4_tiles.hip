// int4 matmul for more rows than the decode kernels take: tiles on the decode kernels' strip-linear copy of the kernel
// (k3q_w4s_pack), nothing de-quantised in memory; the result is written here unless K is split over workgroups.
//
// Eight waves, each 32 columns x 32 kMB rows: kNS of them side by side along N, kKQ slices of K (every kKQ-th unit of 128), whose
// sums meet in LDS at the end -- 4 x 2 in tiles of 128 columns, 8 x 1 in tiles of 256.  The tile kernel before this one (k3q_gemv_w4.hip, which keeps the other group lengths) filled
// the chip by splitting K over workgroups: at 96 rows of 4096 x 14336 four splits wrote and read 44 MB of partial sums
// beside 29 MB of kernel, 13 of its 34 us.  Slices inside a workgroup need none of that, and narrow tiles of few rows (64 x
// 128) fill the chip at 96 rows without a split.  A lane's products are one column of the kernel, so that a unit's scale is one
// value, and each nibble is converted by one wave of the tile (by two before).
//
// A round is 64 of K per slice: the rows of x as they lie, 128 bytes each (32-byte pieces, which the copy's half units had
// asked for, load at 0.74 of the rate: 37 against 50 bytes a ns and CU), the kernel bytes of a unit in whole 1 KiB blocks.  All
// of it arrives by LDS-DMA; the next step's operands are read and converted beside the products of a step, and a unit's sums
// are folded (tot += scale acc) beside the next unit's first products.
//
// What bounds it: at 512 rows and more the matrix cores (128 x 256 tiles: 1.23 PFLOP/s in the loop, the library's large
// products on this card 1.26), below that the starts of ring and launch and the rate of the requests (64 x 128: 39 bytes a ns
// and CU).  Graph nodes, groups of 128, us, before -> now: 32 rows of 4096 x 14336 21.7 -> 17.2, 96 32.0 -> 27.3, 512 86.2 ->
// 68.9; 128 rows of 4096 x 4096 23.6 -> 17.3, 512 37.8 -> 28.7; 128 of 14336 x 4096 34.3 -> 29.0; 256 of 8192 x 8192 54.8 ->
// 47.8.  Tried and slower: the sums of x in this kernel, from the rows in LDS (saves 2.8 us of launch, costs 0.1 us a round: 512
// rows of 4096 x 14336 76.9); a block's four products in turn instead of a step's four blocks (80.9, the sums depend on each
// other); an explicit wait for a step's operands ahead of the next reads (no gain).
#include "k3q_gemm_w4_tiles.h"
#include "k3q_nibbles.h"

namespace k3q {
namespace {

constexpr int kTThreads = 512;  // 8 waves: kNS along N (32 columns each) x kKQ along K

struct TileParams {
    const char* x;
    const char* w;
    const char* scale;
    const char* zero;
    const char* sx;
    const void* bias;
    void* y;
    float* part;
    int64_t rows, N, n_out, bias_stride;
    int64_t row_bytes;   // of x
    int units;           // K / 128
    int steps;           // units of K per split, kKQ at a time
    int m_tiles, n_tiles, splits;
    int parts;
    int direct;          // y is written here (else part)
    int wide;            // four results of a row of y are one store
};

__device__ __forceinline__ v8bf tile_bf(const v4u& v) { return __builtin_bit_cast(v8bf, v); }
__device__ __forceinline__ int tile_swz(int row) { return (row & 6) | ((row ^ (row >> 3)) & 1); }
constexpr int tile_vmcnt(int n) { return (n & 0xF) | ((n >> 4) << 14) | 0x0F70; }
constexpr int kTileLgkm0 = ~0x0F00;  // and lgkmcnt 0

__device__ __forceinline__ void tile_barrier() {
    // no fence: a fence would drain the requests in flight
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <bool kF32>
__device__ __forceinline__ float tile_load(const void* p, int64_t i) {
    return kF32 ? ((const float*)p)[i] : bf16_bits_to_f32(((const uint16_t*)p)[i]);
}

// kKQ: slices of K in a workgroup (of units, in turn); kMB: blocks of 32 rows.
template <bool kF32, int kMB, int kKQ>
struct TileLds {
    static constexpr int kNS = 8 / kKQ;             // waves along N
    static constexpr int kBN = 32 * kNS;
    static constexpr int kXRing = kMB == 4 ? (kKQ == 2 ? 3 : 5) : kMB == 2 ? 5 : 6;
    static constexpr int kWRing = kXRing / 2 + 1, kParRing = (kXRing + 1) / 2 + 1;
    static constexpr int kXSlot = kKQ * kMB * 4096;  // slices of K x 32 kMB rows x 128 bytes
    static constexpr int kWSlot = 16384;             // 16 strips of units, 1 KiB each
    static constexpr int kScaleOps = kBN * (kF32 ? 4 : 2) / 256;  // requests of 256 bytes per slice
    static constexpr int kScale = kKQ * kMB * 256;   // sums of x first: rows x 8 bytes per slice
    static constexpr int kZero = kScale + kKQ * kScaleOps * 256;
    static constexpr int kSpare = kZero + 256;
    static constexpr int kParSlot = kSpare + 256;
    static constexpr int kW = kXRing * kXSlot, kPar = kW + kWRing * kWSlot;
    static constexpr int kPitch = kBN * 4 + 16;
    static constexpr int kRing = kPar + kParRing * kParSlot, kSums = kKQ * kMB * 32 * kPitch;
    static constexpr int kBytes = kRing > kSums ? kRing : kSums;
};

template <bool kGrouped, bool kF32, int kMB, int kKQ, int kForm>
__global__ __launch_bounds__(kTThreads) void gemm_w4_tiles(TileParams p) {
    typedef TileLds<kF32, kMB, kKQ> L;
    constexpr int kXRing = L::kXRing, kNS = L::kNS, kBN = L::kBN;
    constexpr int kXOps = kMB * 4 / kNS, kOps = kXOps + 2;  // requests of a wave per round
    static_assert(kXOps >= 1, "every wave fetches rows");
    extern __shared__ __attribute__((aligned(1024))) char tile_lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % kNS, kq = wave / kNS;
    const int i = lane & 31, g = lane >> 5;

    const int total = p.m_tiles * p.n_tiles * p.splits, per_xcd = (total + 7) >> 3;
    const int item = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
    if (item >= total || (int)(blockIdx.x >> 3) >= per_xcd) return;
    const int sp = item % p.splits, tile = item / p.splits;
    const int tile_m = tile % p.m_tiles;
    const int64_t n0 = (int64_t)(tile / p.m_tiles) * kBN;
    // two parts of a row sit in neighbouring blocks of 32 rows: one lane ends up with both sums
    const bool two = p.parts == 2;
    const int64_t m0 = (int64_t)tile_m * (two ? 16 * kMB : 32 * kMB);
    const int64_t xrows = p.rows * p.parts;
    const int64_t limit = two ? p.rows : xrows;
    auto x_row = [&](const int r) -> int64_t {  // row of x of row r of the tile
        const int64_t real = m0 + (two ? ((r >> 6) << 5) + (r & 31) : r);
        return (real < limit ? real : limit - 1) + (two && (r & 32) ? p.rows : 0);
    };
    const int u_begin = sp * kKQ * p.steps;
    const int u_end = u_begin + kKQ * p.steps < p.units ? u_begin + kKQ * p.steps : p.units;
    const int steps = (u_end - u_begin + kKQ - 1) / kKQ;
    const int rounds = 2 * steps;

    // ---- request sources: wave-uniform bases and 32-bit lane offsets (w4_tile_launch has checked the sizes) ----
    const char* x_base = p.x + m0 * p.row_bytes;
    u32 x_off[kXOps];
#pragma unroll
    for (int j = 0; j < kXOps; ++j) {
        const int row = (wn * kXOps + j) * 8 + (lane >> 3);
        x_off[j] = (u32)((x_row(row) - m0) * p.row_bytes) + (((lane & 7) ^ tile_swz(row)) << 4);
    }
    const char* w_base[2];
    const char* par_base[2];
    u32 par_off[2], par_step[2];
    int par_slice[2], par_dst[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
        const int pi = hf * 8 + wave;
        int64_t strip = n0 / 16 + pi % (kBN / 16);
        const int64_t last = p.N / 16 - 1;
        if (strip > last) strip = last;
        w_base[hf] = p.w + strip * p.units * 1024;
        constexpr int el = kF32 ? 4 : 2, kCols = 256 / el;
        if (kGrouped && pi >= 8 && pi < 8 + kKQ * L::kScaleOps) {
            int64_t n = n0 + (pi - 8) % L::kScaleOps * kCols + lane * (4 / el);
            if (n > p.N - 4 / el) n = p.N - 4 / el;
            par_base[hf] = p.scale;
            par_off[hf] = (u32)n * el;
            par_slice[hf] = (pi - 8) / L::kScaleOps;
            par_step[hf] = (u32)(p.N * el);
            par_dst[hf] = L::kScale + (pi - 8) * 256;
        } else if (kGrouped && pi == 12) {
            int64_t n = n0 + (lane & (kBN / 4 - 1)) * 4;
            if (n > p.N - 4) n = p.N - 4;
            par_base[hf] = p.zero;
            par_off[hf] = (u32)n;
            par_slice[hf] = 0;  // (two slices: the upper half of the lanes fetches the second one's, issue_w)
            par_step[hf] = (u32)p.N;
            par_dst[hf] = L::kZero;
        } else {
            const bool sums = pi < kKQ * kMB;
            const int at = sums ? pi : 0;
            par_base[hf] = p.sx;
            par_off[hf] = (u32)x_row((at % kMB) * 32 + (lane >> 1)) * 8 + (lane & 1) * 4;
            par_slice[hf] = at / kMB;
            par_step[hf] = (u32)(xrows * 8);
            par_dst[hf] = sums ? pi * 256 : L::kSpare;
        }
    }
    static_assert(kKQ * kMB <= 8 && kKQ * L::kScaleOps <= 4, "sixteen parameter requests");
    auto lds_dma16 = [&](const char* base, const u32 off, int at) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + off),
                                         (__attribute__((address_space(3))) void*)(tile_lds + at), 16, 0, 0);
    };
    auto lds_dma4 = [&](const char* base, const u32 off, int at) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + off),
                                         (__attribute__((address_space(3))) void*)(tile_lds + at), 4, 0, 0);
    };
    auto clamp_unit = [&](int u) { return u < u_end ? u : u_end - 1; };
    // Half hf of the kernel bytes (op 0) and parameters (op 1) of step j.
    auto issue_w = [&](const int j, const int hf, const int op) {
        const int u0 = u_begin + kKQ * j;
        if (op == 0) {
            lds_dma16(w_base[hf] + (int64_t)clamp_unit(u0 + (hf * 8 + wave) / (kBN / 16)) * 1024, (u32)lane * 16,
                      L::kW + (j % L::kWRing) * L::kWSlot + (hf * 8 + wave) * 1024);
        } else {
            u32 off = par_off[hf] + (u32)clamp_unit(u0 + par_slice[hf]) * par_step[hf];
            if (kGrouped && kKQ == 2 && hf == 1) {  // (the zero points' request, wave 4: both slices)
                const u32 second = par_off[hf] + (u32)clamp_unit(u0 + 1) * par_step[hf];
                if (wave == 4 && g) off = second;
            }
            lds_dma4(par_base[hf], off, L::kPar + (j % L::kParRing) * L::kParSlot + par_dst[hf]);
        }
    };
    // Request `op` of group r: the x rows of round r, and the half of a step's kernel bytes whose turn it is -- a step is
    // whole when its first round's group is.
    auto issue = [&](const int r, const int op) {
        if (op < kXOps) {
            const int64_t at = (int64_t)clamp_unit(u_begin + kKQ * (r >> 1) + kq) * 256 + (r & 1) * 128;
            lds_dma16(x_base + at, x_off[op], (r % kXRing) * L::kXSlot + (kq * 4 * kMB + wn * kXOps + op) * 1024);
        } else {
            issue_w((r + 1) >> 1, (r & 1) ^ 1, op - kXOps);
        }
    };
    auto wait_groups_behind = [&](const int behind) {
        // (this wave's own LDS reads have come, too: the slot they were from is filled again behind the meeting)
        if (kXRing >= 6 && behind >= 4) __builtin_amdgcn_s_waitcnt(tile_vmcnt(kXRing >= 6 ? 4 * kOps : 0) & kTileLgkm0);
        else if (kXRing >= 5 && behind >= 3) __builtin_amdgcn_s_waitcnt(tile_vmcnt(kXRing >= 5 ? 3 * kOps : 0) & kTileLgkm0);
        else if (kXRing >= 4 && behind >= 2) __builtin_amdgcn_s_waitcnt(tile_vmcnt(kXRing >= 4 ? 2 * kOps : 0) & kTileLgkm0);
        else if (behind >= 1) __builtin_amdgcn_s_waitcnt(tile_vmcnt(kOps) & kTileLgkm0);
        else __builtin_amdgcn_s_waitcnt(tile_vmcnt(0) & kTileLgkm0);
    };
    static_assert(kXRing >= 3 && kXRing <= 6, "wait_groups_behind");

    // ---- operands ----
    v16f acc[kMB], tot[kMB], zero16;
#pragma unroll
    for (int r = 0; r < 16; ++r) zero16[r] = 0.f;
#pragma unroll
    for (int mb = 0; mb < kMB; ++mb) acc[mb] = tot[mb] = zero16;
    v4u xa[2][kMB], wq[2], wb[2];
    float off = 8.f, sc = 0.f;
    const int x_at = kq * kMB * 4096 + i * 128 + ((g ^ tile_swz(i)) << 4);
    const int w_at = L::kW + kq * (kBN * 64) + (2 * wn + (i >> 4)) * 1024 + ((i & 15) + 16 * g) * 16;
    const int col = wn * 32 + i;
    auto read_x = [&](const int buf, const int slot, const int t) {
        const char* at = tile_lds + slot * L::kXSlot + (x_at ^ (t << 5));
#pragma unroll
        for (int mb = 0; mb < kMB; ++mb) xa[buf][mb] = *(const v4u*)(at + mb * 4096);
    };
    auto read_w = [&](const int j) {
        const char* at = tile_lds + w_at + (j % L::kWRing) * L::kWSlot;
        wq[0] = *(const v4u*)at;
        wq[1] = *(const v4u*)(at + 512);
        if (kForm == kW4FormPlain && kGrouped)
            off = 8.f + (float)*(const int8_t*)(tile_lds + L::kPar + (j % L::kParRing) * L::kParSlot + L::kZero + kq * kBN + col);
    };
    auto convert = [&](const u32 d) {
        if constexpr (kForm == kW4FormPlain) return plain_nibbles(d, off);
        v4u o;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            o[q] = kForm == kW4Form24 ? ((q ? d >> (4 * q - 3) : d << 3) & 0x00780078u) ^ 0x41C041C0u
                                      : ((d >> (4 * q)) & 0x000F000Fu) ^ 0x43084308u;
        return o;
    };
    // A unit's end: acc -= (136 + zero) sum(x) as one more product per block (kernel side: -128, or -16, at k = 0 ... 2 and
    // -(8 + zero) at k = 3 ... 5, x side: the three bfloat16 parts of the sum twice; every product is exact in float32),
    // then tot += scale acc, which waits for the next unit's first products to be in front of (below).
    v2u raw_sum[kMB];
    int raw_zero = 0;
    float raw_scale = 1.f;
    auto read_params = [&](const int j) {
        const char* par = tile_lds + L::kPar + (j % L::kParRing) * L::kParSlot;
        if (kGrouped) {
            if (kForm != kW4FormPlain) raw_zero = *(const int8_t*)(par + L::kZero + kq * kBN + col);
            raw_scale = kF32 ? *(const float*)(par + L::kScale + (kq * kBN + col) * 4)
                             : bf16_bits_to_f32(*(const uint16_t*)(par + L::kScale + (kq * kBN + col) * 2));
        }
        if (kForm != kW4FormPlain) {
#pragma unroll
            for (int mb = 0; mb < kMB; ++mb) raw_sum[mb] = *(const v2u*)(par + (kq * kMB + mb) * 256 + i * 8);
        }
    };
    auto take_out_offset = [&]() {
        if constexpr (kForm != kW4FormPlain) {
            const u32 cz = __float_as_uint(-(float)(8 + raw_zero)) >> 16;
            constexpr u32 kBase = kForm == kW4Form24 ? 0xC180u : 0xC300u;  // -16, -128
            const v4u wz = {kBase | (kBase << 16), kBase | (cz << 16), cz | (cz << 16), 0u};
#pragma unroll
            for (int mb = 0; mb < kMB; ++mb) {
                const u32 a = g ? 0u : raw_sum[mb][0], b = g ? 0u : raw_sum[mb][1];
                const v4u xs = {a, (b & 0xffffu) | (a << 16), (a >> 16) | (b << 16), 0u};
                acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tile_bf(xs), tile_bf(wz), acc[mb], 0, 0, 0);
            }
        }
        sc = raw_scale;
    };
    auto fold = [&](const int mb) {
#pragma unroll
        for (int e = 0; e < 16; ++e) tot[mb][e] = __builtin_fmaf(sc, acc[mb][e], tot[mb][e]);
        asm volatile("" : "+v"(tot[mb]));  // here, and not where the compiler would sink it to: behind the next sums
    };

    // ---- start: the first step's first half, then kXRing groups ----
    issue_w(0, 0, 0);
    issue_w(0, 0, 1);
#pragma unroll
    for (int r = 0; r < kXRing; ++r)
        if (r < rounds) {
#pragma unroll
            for (int op = 0; op < kOps; ++op) issue(r, op);
        }
    if (rounds >= kXRing) __builtin_amdgcn_s_waitcnt(tile_vmcnt(kOps * (kXRing - 1)));
    else __builtin_amdgcn_s_waitcnt(tile_vmcnt(0));
    tile_barrier();
    read_w(0);
    read_x(0, 0, 0);
    wb[0] = convert(wq[0][0]);

    int slot = 0;
#pragma clang loop unroll(disable)
    for (int j = 0; j < steps; ++j) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r = 2 * j + h;
            const int next_slot = slot == kXRing - 1 ? 0 : slot + 1;
            constexpr int kPerStep = (kOps - 1 + 2) / 3;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                constexpr int kFirst = kMB / 2;  // products of the last step ahead of the meeting
                auto product = [&](const int mb) {
                    acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(tile_bf(xa[t & 1][mb]), tile_bf(wb[t & 1]),
                                                                      (h == 0 && t == 0) ? zero16 : acc[mb], 0, 0, 0);
                };
                __builtin_amdgcn_sched_barrier(0);
                if (t < 3) {
                    read_x((t + 1) & 1, slot, t + 1);
                    if (r > 0 && r - 1 + kXRing < rounds) {
#pragma unroll
                        for (int o = 0; o < kPerStep; ++o)
                            if (1 + t * kPerStep + o < kOps) issue(r - 1 + kXRing, 1 + t * kPerStep + o);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    const int s = 2 * h + ((t + 1) >> 1);
                    if (h == 0 && t == 0) {
                        // the unit before: its last sums are folded block by block, each ahead of the product that
                        // overwrites them and behind the product of the block before
#pragma unroll
                        for (int mb = 0; mb < kMB; ++mb) {
                            fold(mb);
                            __builtin_amdgcn_sched_barrier(0);
                            product(mb);
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        wb[1] = convert(wq[1][s]);
                    } else {
#pragma unroll
                        for (int mb = 0; mb < kMB; ++mb) product(mb);
                        wb[(t + 1) & 1] = convert(wq[(t + 1) & 1][s]);
#pragma unroll
                        for (int q = 0; q < kMB; ++q) {
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, 8 / kMB, 0);
                        }
                    }
                } else {
#pragma unroll
                    for (int mb = 0; mb < kFirst; ++mb) product(mb);
                    __builtin_amdgcn_sched_barrier(0);
                    if (h == 1) read_params(j);
                    if (r + 1 < rounds) {
                        wait_groups_behind(rounds - 2 - r);
                        tile_barrier();
                        if (r + kXRing < rounds) issue(r + kXRing, 0);
                        if (h == 1) read_w(j + 1);
                        read_x(0, next_slot, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int mb = kFirst; mb < kMB; ++mb) product(mb);
                    if (h == 1) take_out_offset();
                    wb[0] = convert(h == 0 ? wq[0][2] : wq[0][0]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            slot = next_slot;
        }
    }
    // (where the units end inside a step, the slices behind them have multiplied the last unit once more)
    if (u_begin + kKQ * (steps - 1) + kq < u_end) {
#pragma unroll
        for (int mb = 0; mb < kMB; ++mb) fold(mb);
    }

    // ---- the slices' sums, through LDS, and the result ----
    __syncthreads();
    constexpr int kRows = 32 * kMB;
#pragma unroll
    for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const int row = mb * 32 + 8 * (e >> 2) + 4 * g + (e & 3);
            *(float*)(tile_lds + (kq * kRows + row) * L::kPitch + (wn * 32 + i) * 4) = tot[mb][e];
        }
    __syncthreads();
    constexpr int kPieces = kBN / 4;  // of four columns
    const int c4 = (tid % kPieces) * 4;
    const int64_t n = n0 + c4;
    if (n >= p.N) return;
    auto sum_of = [&](const int row) {
        const char* at = tile_lds + row * L::kPitch + c4 * 4;
        v4f v = *(const v4f*)at;
        if (kKQ == 2) v += *(const v4f*)(at + kRows * L::kPitch);
        return v;
    };
    if (!p.direct) {
#pragma unroll 2
        for (int row = tid / kPieces; row < kRows; row += kTThreads / kPieces) {
            const int64_t real = m0 + (two ? ((row >> 6) << 5) + (row & 31) : row);
            if (real >= limit) continue;
            *(v4f*)(p.part + ((int64_t)sp * xrows + x_row(row)) * p.N + n) = sum_of(row);
        }
        return;
    }
    if (n >= p.n_out) return;  // (a column of the copy past the last of y)
    float sb[4], bv[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int64_t c = n + e < p.n_out ? n + e : p.n_out - 1;
        sb[e] = kGrouped ? 1.f : tile_load<kF32>(p.scale, c);
        if (p.bias && p.bias_stride == 0) bv[e] = tile_load<kF32>(p.bias, c);
    }
#pragma unroll 2
    for (int rr = tid / kPieces; rr < (two ? kRows / 2 : kRows); rr += kTThreads / kPieces) {
        const int64_t m = m0 + rr;
        if (m >= limit) continue;
        v4f v;
        if (two) {
            const int row = ((rr >> 5) << 6) + (rr & 31);
            const v4f lo = sum_of(row + 32);
            v = lo + sum_of(row);
        } else {
            v = sum_of(rr);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (!kF32) v[e] = round_bf16(v[e]);
            if (!kGrouped) {
                v[e] = v[e] / sb[e];
                if (!kF32) v[e] = round_bf16(v[e]);
            }
            if (p.bias) {
                float b = bv[e];
                if (p.bias_stride != 0 && n + e < p.n_out) b = tile_load<kF32>(p.bias, m * p.bias_stride + n + e);
                v[e] = v[e] + b;
            }
        }
        if (p.wide) {
            if (kF32) *(v4f*)((float*)p.y + m * p.n_out + n) = v;
            else *(v2u*)((uint16_t*)p.y + m * p.n_out + n) = v2u{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (n + e >= p.n_out) break;
                if (kF32) ((float*)p.y)[m * p.n_out + n + e] = v[e];
                else ((uint16_t*)p.y)[m * p.n_out + n + e] = (uint16_t)f32_to_bf16_bits(v[e]);
            }
        }
    }
}

typedef void (*TileKernel)(TileParams);

template <bool kGrouped, bool kF32, int kMB, int kKQ, int kForm>
TileKernel raised(int* lds) {
    typedef TileLds<kF32, kMB, kKQ> L;
    static_assert(L::kBytes <= 160 * 1024, "LDS");
    static const bool ok = hipFuncSetAttribute((const void*)gemm_w4_tiles<kGrouped, kF32, kMB, kKQ, kForm>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, L::kBytes) == hipSuccess;
    *lds = L::kBytes;
    return ok ? gemm_w4_tiles<kGrouped, kF32, kMB, kKQ, kForm> : nullptr;
}

template <bool kGrouped, bool kF32, int kForm>
TileKernel pick_rows(const W4TilePlan& pl, int* lds) {
    if (pl.bn == 256) return raised<kGrouped, kF32, 4, 1, kForm>(lds);
    return pl.mb == 4   ? raised<kGrouped, kF32, 4, 2, kForm>(lds)
           : pl.mb == 2 ? raised<kGrouped, kF32, 2, 2, kForm>(lds)
                        : raised<kGrouped, kF32, 1, 2, kForm>(lds);
}

template <bool kGrouped, bool kF32>
TileKernel pick_form(int form, const W4TilePlan& pl, int* lds) {
    if constexpr (!kF32)
        if (form == kW4Form136) return pick_rows<kGrouped, kF32, kW4Form136>(pl, lds);
    return form == kW4Form24 ? pick_rows<kGrouped, kF32, kW4Form24>(pl, lds) : pick_rows<kGrouped, kF32, kW4FormPlain>(pl, lds);
}

}  // namespace

bool w4_tile_fits(int64_t rows, int parts, int64_t K, int64_t N) {
    const int64_t most = (int64_t)1 << 32, units = K / 128;
    return ((parts == 2 ? rows : 0) + 128) * K * 2 < most && units * 4 * N < most && units * 8 * rows * parts < most;
}

// Tile shape and split of K from a model of the time (ns) fitted to a sweep of every shape and split (1469 calls of 17 ... 1024
// rows, K = 768 ... 14336, N = 768 ... 14336; what it chooses takes 0.4 % more than the best measured one in the mean, 5.4 % in 99
// of 100): a workgroup its rounds at the shape's rate, 7.5 % slower with all CUs at it than with one, which the start of its ring
// and its sums' way through LDS come on top of, 256 of them at a time; partial sums a launch, something per split, and their
// bytes out and in at 7.2 TB/s.  (A first fit, on fewer shapes and with splits dearer, left 1.0 % and 12 %, and more than the old
// kernel took in places: 65 rows of 5120 x 11008 32.9 us, old kernel 29.5, now 29.5.)
W4TilePlan w4_tile_plan(int64_t rows, int parts, int64_t K, int64_t N) {
    struct Shape {
        int mb, bn, round_ns, start_ns;
    };
    static const Shape shapes[] = {{1, 128, 460, 2220}, {2, 128, 600, 3370}, {4, 128, 880, 5410}, {4, 256, 820, 6560}};
    const int64_t xrows = rows * parts, units = K / 128;
    W4TilePlan best{};
    int64_t best_ns = -1;
    for (const Shape& sh : shapes) {
        if (parts == 2 && sh.mb == 1) continue;  // (both parts of a row in one tile)
        const int64_t tiles = ((xrows + 32 * sh.mb - 1) / (32 * sh.mb)) * ((N + sh.bn - 1) / sh.bn);
        const int kq = W4TilePlan{sh.mb, sh.bn, 1, 1}.kq();
        const int64_t all = (units + kq - 1) / kq;
        for (int64_t want = 1; want <= 8; ++want) {
            const int64_t steps = (all + want - 1) / want;
            const int64_t ks = (all + steps - 1) / steps;
            if (want > 1 && (steps < 4 || tiles * want > 256)) break;
            if (ks != want) continue;
            const int64_t turns = (tiles * ks + 255) / 256, rounds = 2 * steps * sh.round_ns;
            int64_t ns = turns * (rounds + sh.start_ns) + rounds * 75 * tiles * ks / 256000;
            if (ks > 1 || parts == 3) ns += 1010 + 252 * ks + ks * xrows * N * 8 / 7170;
            if (best_ns < 0 || ns < best_ns) {
                best_ns = ns;
                best.mb = sh.mb;
                best.bn = sh.bn;
                best.ks = (int)ks;
                best.steps = (int)steps;
            }
        }
    }
    return best;
}

int w4_tile_launch(const W4TileCall& c, const W4TilePlan& pl, hipStream_t s) {
    TileParams p{};
    p.x = (const char*)c.x;
    p.w = (const char*)c.w;
    p.scale = (const char*)c.scale;
    p.zero = (const char*)c.zero;
    p.sx = (const char*)c.sx;
    p.bias = c.bias;
    p.y = c.y;
    p.part = c.part;
    p.rows = c.rows;
    p.N = c.N;
    p.n_out = c.n_out;
    p.bias_stride = c.bias_stride;
    p.row_bytes = c.K * 2;
    p.units = (int)(c.K / 128);
    p.steps = pl.steps;
    p.parts = c.parts;
    p.splits = pl.ks;
    const int64_t xrows = c.rows * c.parts, tile_rows = c.parts == 2 ? 16 * pl.mb : 32 * pl.mb;
    p.m_tiles = (int)(((c.parts == 2 ? c.rows : xrows) + tile_rows - 1) / tile_rows);
    p.n_tiles = (int)((c.N + pl.bn - 1) / pl.bn);
    p.direct = w4_tile_direct(pl, c.parts) ? 1 : 0;
    p.wide = c.n_out % 4 == 0 && aligned_to(c.y, c.f32 ? 16 : 8) ? 1 : 0;
    const int64_t total = (int64_t)p.m_tiles * p.n_tiles * p.splits;
    // (a plan that leaves a part of K out is not launched)
    if (total > (1 << 28) || !w4_tile_fits(c.rows, c.parts, c.K, c.N) || (int64_t)pl.ks * pl.steps * pl.kq() < p.units)
        return K3Q_ERR_SHAPE;
    int lds = 0;
    const TileKernel k = c.grouped ? (c.f32 ? pick_form<true, true>(c.form, pl, &lds) : pick_form<true, false>(c.form, pl, &lds))
                                   : (c.f32 ? pick_form<false, true>(c.form, pl, &lds) : pick_form<false, false>(c.form, pl, &lds));
    if (!k) return K3Q_ERR_LAUNCH;
    k<<<(unsigned)((total + 7) / 8 * 8), kTThreads, (size_t)lds, s>>>(p);
    return launch_status();
}

}  // namespace k3q
