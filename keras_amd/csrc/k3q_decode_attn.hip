// One new position of causal self-attention against a key / value cache, bfloat16, head
// width 128: rotate the new query and key (rotate-half RoPE, tables indexed by the position),
// write the new key and value rows into the cache at the position, attend over rows
// 0 ... position.  One launch where the decoder step otherwise runs a dozen small ones.
//
// One workgroup per (sequence, head), 8 waves.  A wave instruction covers 4 cache rows
// (16 lanes x 16 bytes per 256-byte row), waves take blocks of 4 rows round-robin; scores go
// through LDS (one float per cache row), softmax in float32, the value sum is reduced over
// the 4 row slots of a wave by lane exchange and over the waves through LDS.
// The position is read from device memory, so a captured graph replays with a new one.
// Two dependent rounds of loads: the position with the new query / key / value rows, then the
// rotation's table entries with the cached rows below the position; the new rows are used from
// LDS, so nothing waits for their stores into the cache to be acknowledged.
#include "k3q_common.h"

namespace k3q {
namespace {

constexpr int kHd = 128;
constexpr int kAW = 8;           // waves per workgroup
constexpr int kAT = 64 * kAW;

struct AttnParams {
    const uint16_t *q, *k, *v;      // [B, H, 128] bfloat16 (one position)
    const uint16_t *cos_t, *sin_t;  // [max_len, 128] bfloat16
    const int64_t* pos;             // device: the position of this step
    uint16_t *kc, *vc;              // [B, H, max_len, 128]
    uint16_t* out;                  // [B, H, 128]
    int* oob;                       // device flag, may be null: set to 1 when the position is outside the cache
    int H, max_len;
    float scale;
};

// every lane of a row of 16 gets the row's sum: x ^ 1, x ^ 2, then the other quad of the half row,
// then the other half (the same pairs, in the same order, as a butterfly over 1, 2, 4, 8)
__device__ __forceinline__ float row16_sum(float v) {
    v += dpp_move<0xB1, 0xf>(v);   // quad_perm [1,0,3,2]
    v += dpp_move<0x4E, 0xf>(v);   // quad_perm [2,3,0,1]
    v += dpp_move<0x141, 0xf>(v);  // row_half_mirror
    v += dpp_move<0x140, 0xf>(v);  // row_mirror
    return v;
}

__global__ __launch_bounds__(kAT) void decode_attention(AttnParams p) {
    extern __shared__ __attribute__((aligned(16))) float attn_lds[];
    float* qs = attn_lds;                   // [128] rotated query, pre-scaled
    float* red = qs + kHd;                  // [2 * kAW]
    float* oacc = red + 2 * kAW;            // [kAW][128]
    uint16_t* knew = (uint16_t*)(oacc + kAW * kHd);  // [128] the new key row as it goes into the cache
    uint16_t* vnew = knew + kHd;            // [128] the new value row
    float* sc = (float*)(vnew + kHd);       // [max_len]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int bh = blockIdx.x;
    // The loads that do not depend on the position go out together with the position itself:
    // the new query / key elements (with their rotate-half partners) and the new value row.
    const int d = tid & (kHd - 1);
    float x = 0.f, sw = 0.f;
    v4u vrow = {0u, 0u, 0u, 0u};
    if (tid < 2 * kHd) {
        const uint16_t* src = (tid < kHd ? p.q : p.k) + (int64_t)bh * kHd;
        x = bf16_bits_to_f32(src[d]);
        sw = bf16_bits_to_f32(src[d ^ (kHd / 2)]);
    } else if (tid < 2 * kHd + 16) {
        vrow = ((const v4u*)(p.v + (int64_t)bh * kHd))[tid - 2 * kHd];
    }
    // A position outside the cache (the torch ops this stands for raise there): nothing is written
    // to the caches, the output rows are zero and the caller's flag is raised.  Every thread reads
    // the same position, so the whole workgroup leaves here before its first barrier.
    const int64_t pos64 = p.pos[0];
    if (pos64 < 0 || pos64 >= p.max_len) {
        if (tid < kHd) p.out[(int64_t)bh * kHd + tid] = 0;
        if (tid == 0 && p.oob) p.oob[0] = 1;
        return;
    }
    const int pos = (int)pos64;
    const int64_t row0 = (int64_t)bh * p.max_len;  // first cache row of this (sequence, head)

    // ---- second round of loads: the rotation's table entries and the cached rows ----
    // Rows 0 ... pos-1 are in the cache already, so their loads need not wait for the new row to be
    // written: row pos itself is taken from LDS below.  Blocks of 4 cache rows go to the waves
    // round-robin; a wave asks for kU blocks of keys at once and -- for its first kU blocks -- for
    // the value rows too, before the softmax, so that the weighted sum finds them in registers
    // (the value rows do not depend on the scores).
    float cs = 0.f, sn = 0.f;
    if (tid < 2 * kHd) {
        cs = bf16_bits_to_f32(p.cos_t[(int64_t)pos * kHd + d]);
        sn = bf16_bits_to_f32(p.sin_t[(int64_t)pos * kHd + d]);
    }
    const int n = pos + 1;
    const int nblk = (n + 3) >> 2;
    const int sub = lane >> 4, dl = (lane & 15) * 8;
    const int last_old = pos > 0 ? pos - 1 : 0;  // a row that is safe to read for lanes without a cached row
    constexpr int kU = 8;
    v4u kk0[kU], vv0[kU];
    if (wave < nblk) {
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int j = 4 * (wave + u * kAW) + sub;
            kk0[u] = *(const v4u*)(p.kc + (row0 + (j < pos ? j : last_old)) * kHd + dl);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int j = 4 * (wave + u * kAW) + sub;
            vv0[u] = *(const v4u*)(p.vc + (row0 + (j < pos ? j : last_old)) * kHd + dl);
        }
    }

    // ---- rotate q and k; the new rows go to the cache and, for this launch, to LDS ----
    if (tid < 2 * kHd) {
        // the rounding steps of x * cos + swapped * sin evaluated in bfloat16
        const float r = round_bf16(round_bf16(x * cs) + round_bf16(sw * sn));
        if (tid < kHd) {
            qs[d] = r * p.scale;
        } else {
            const uint16_t bits = (uint16_t)f32_to_bf16_bits(r);
            knew[d] = bits;
            p.kc[(row0 + pos) * kHd + d] = bits;
        }
    } else if (tid < 2 * kHd + 16) {
        const int c = tid - 2 * kHd;
        ((v4u*)vnew)[c] = vrow;
        ((v4u*)(p.vc + (row0 + pos) * kHd))[c] = vrow;
    }
    __syncthreads();

    // ---- scores ----
    float qv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) qv[e] = qs[dl + e];
    float mx = -INFINITY;
    for (int kb0 = wave; kb0 < nblk; kb0 += kAW * kU) {
        v4u kk[kU];
        if (kb0 == wave) {
#pragma unroll
            for (int u = 0; u < kU; ++u) kk[u] = kk0[u];
        } else {
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int j = 4 * (kb0 + u * kAW) + sub;
                kk[u] = *(const v4u*)(p.kc + (row0 + (j < pos ? j : last_old)) * kHd + dl);
            }
        }
        float dot[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int j = 4 * (kb0 + u * kAW) + sub;
            if (j == pos) kk[u] = *(const v4u*)(knew + dl);
            dot[u] = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                dot[u] += qv[2 * e] * __uint_as_float(kk[u][e] << 16);
                dot[u] += qv[2 * e + 1] * __uint_as_float(kk[u][e] & 0xffff0000u);
            }
        }
        // sum over the 16 lanes of a row, as lane exchanges inside the vector unit (through LDS
        // permutes the kU dependent chains of four exchanges took 2 us of the launch's 8)
#pragma unroll
        for (int u = 0; u < kU; ++u) dot[u] = row16_sum(dot[u]);
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int j = 4 * (kb0 + u * kAW) + sub;
            if (j < n) {
                mx = fmaxf(mx, dot[u]);
                if ((lane & 15) == 0) sc[j] = dot[u];
            }
        }
    }
    mx = wave_max(mx);
    if (lane == 0) red[wave] = mx;
    __syncthreads();
    float gmx = red[0];
#pragma unroll
    for (int w = 1; w < kAW; ++w) gmx = fmaxf(gmx, red[w]);

    // ---- softmax numerators ----
    float part = 0.f;
    for (int j = tid; j < n; j += kAT) {
        const float e = __expf(sc[j] - gmx);
        sc[j] = e;
        part += e;
    }
    part = wave_sum(part);
    if (lane == 0) red[kAW + wave] = part;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < kAW; ++w) total += red[kAW + w];

    // ---- weighted sum of the value rows ----
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    auto add_row = [&](const v4u& vv, const float w) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            acc[2 * e] += w * __uint_as_float(vv[e] << 16);
            acc[2 * e + 1] += w * __uint_as_float(vv[e] & 0xffff0000u);
        }
    };
    if (wave < nblk) {
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int j = 4 * (wave + u * kAW) + sub;
            if (j == pos) vv0[u] = *(const v4u*)(vnew + dl);
            add_row(vv0[u], j < n ? sc[j] : 0.f);
        }
    }
    for (int kb0 = wave + kAW * kU; kb0 < nblk; kb0 += kAW * kU) {
        v4u vv[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int j = 4 * (kb0 + u * kAW) + sub;
            vv[u] = *(const v4u*)(p.vc + (row0 + (j < pos ? j : last_old)) * kHd + dl);
        }
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const int j = 4 * (kb0 + u * kAW) + sub;
            if (j == pos) vv[u] = *(const v4u*)(vnew + dl);
            add_row(vv[u], j < n ? sc[j] : 0.f);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        acc[e] += __shfl_xor(acc[e], 16, kWave);
        acc[e] += __shfl_xor(acc[e], 32, kWave);
    }
    if (lane < 16) {
#pragma unroll
        for (int e = 0; e < 8; ++e) oacc[wave * kHd + dl + e] = acc[e];
    }
    __syncthreads();
    if (tid < kHd) {
        float o = 0.f;
#pragma unroll
        for (int w = 0; w < kAW; ++w) o += oacc[w * kHd + tid];
        p.out[(int64_t)bh * kHd + tid] = (uint16_t)f32_to_bf16_bits(o / total);
    }
}

// ---- several positions: the prompt's rotation and cache update -------------------------------------------------
// out = rotated q, the cache rows at pos[t] = rotated k and v, with the roundings of the torch sequence
// (bf16(x cos) + bf16(swapped sin), rounded), which cost eight passes over q and k (cat, swap, two products, sum, two
// index copies): 104 us per block of 8 x 128 tokens of 32 heads.  Here every value is read and written once.
// Bound by memory: a thread takes pieces c and c + 8 (16 bytes each) of a head's 128 values of q, k and v, so that it
// holds both halves of a rotation and eight threads read and write whole 128-byte lines.
struct RopeParams {
    const uint16_t *q, *k, *v;      // [B, T, H, 128]
    const uint16_t *cos_t, *sin_t;  // [max_len, 128]
    const int64_t* pos;             // device [T]
    uint16_t *kc, *vc;              // [B, H, max_len, 128]
    uint16_t* out;                  // [B, T, H, 128]
    int* oob;                       // device flag, may be null: 1 when a position is outside the cache (not written)
    int64_t heads;                  // B T H
    int T, H, max_len;
};

// x cos + swapped sin for one 16-byte piece, each step rounded to bfloat16
__device__ __forceinline__ v4u rotate_piece(const v4u& x, const v4u& swapped, const v4u& cs, const v4u& sn) {
    v4u o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float lo = round_bf16(__uint_as_float(x[e] << 16) * __uint_as_float(cs[e] << 16)) +
                         round_bf16(__uint_as_float(swapped[e] << 16) * __uint_as_float(sn[e] << 16));
        const float hi = round_bf16(__uint_as_float(x[e] & 0xffff0000u) * __uint_as_float(cs[e] & 0xffff0000u)) +
                         round_bf16(__uint_as_float(swapped[e] & 0xffff0000u) * __uint_as_float(sn[e] & 0xffff0000u));
        o[e] = f32_to_bf16_bits(lo) | (f32_to_bf16_bits(hi) << 16);
    }
    return o;
}

__global__ __launch_bounds__(256) void rope_cache_rows(RopeParams p) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t row = i >> 3;  // (b, t, h)
    const int c = (int)(i & 7);
    if (row >= p.heads) return;
    const int h = (int)(row % p.H);
    const int64_t bt = row / p.H;
    const int t = (int)(bt % p.T);
    const int64_t b = bt / p.T;
    const v4u* q = (const v4u*)(p.q + row * kHd);
    const v4u* k = (const v4u*)(p.k + row * kHd);
    const v4u* v = (const v4u*)(p.v + row * kHd);
    const v4u q0 = q[c], q1 = q[c + 8], k0 = k[c], k1 = k[c + 8], v0 = v[c], v1 = v[c + 8];
    const int64_t pos = p.pos[t];
    const bool inside = pos >= 0 && pos < p.max_len;
    const int64_t at = inside ? pos : 0;
    const v4u* cs = (const v4u*)(p.cos_t + at * kHd);
    const v4u* sn = (const v4u*)(p.sin_t + at * kHd);
    const v4u c0 = cs[c], c1 = cs[c + 8], s0 = sn[c], s1 = sn[c + 8];
    v4u* o = (v4u*)(p.out + row * kHd);
    o[c] = rotate_piece(q0, q1, c0, s0);
    o[c + 8] = rotate_piece(q1, q0, c1, s1);
    if (!inside) {
        if (p.oob) p.oob[0] = 1;
        return;
    }
    const int64_t crow = ((b * p.H + h) * p.max_len + pos) * kHd;
    v4u* kc = (v4u*)(p.kc + crow);
    v4u* vc = (v4u*)(p.vc + crow);
    kc[c] = rotate_piece(k0, k1, c0, s0);
    kc[c + 8] = rotate_piece(k1, k0, c1, s1);
    vc[c] = v0;
    vc[c + 8] = v1;
}

// ---- several positions: a prompt's attention over the cache -------------------------------------------------------
// out[b, t, h] = softmax(q k^T / sqrt(128) + mask[t]) v over the cache rows, the mask added as it is.  A workgroup takes 64
// positions of a (sequence, head), a wave 16 of them, and walks the cache in blocks of 64 rows, running maximum and sum per
// position; blocks that the mask closes for all 64 positions (an additive -inf) are not read.  Products on the matrix cores, keys
// as the rows: a lane then holds scores of ONE position (its column), four keys of each 16, and these are, as they lie, the
// operand of the product with the values -- whose other operand takes its keys in the same order, from a transposed tile in
// LDS.  Scores and sums are float32; a probability goes into its product as two bfloat16 parts (2^-17), not one.
// 8 x 128 positions of 32 heads, cache of 256: bound by the chain of a block (mask, keys, scores, values) beside its 32 MB; 49
// us in the library's kernel behind transposed views, 16 here (dispatches in a kernel trace).
constexpr int kPKeys = 64, kPRows = 64;             // cache rows per block, positions per workgroup
constexpr int kPKPitch = kHd * 2 + 16;              // LDS bytes per key row
constexpr int kPVPitch = kPKeys * 2 + 24;           // and per value column (of the transposed tile)
// Scores below this leave float32's range when they are taken to base 2: closed, as in the library (a mask of the type's
// lowest value closes a row whose keys it all names, and does not make it the mean of all values).
constexpr float kPLowest = -2.3586498e38f;
struct PromptParams {
    const uint16_t* q;      // [B, T, H, 128]
    const uint16_t *kc, *vc;  // [B, H, max_len, 128]
    const uint16_t* mask;   // [T, max_len] bfloat16
    uint16_t* out;          // [B, T, H, 128]
    int T, H, max_len;
    float scale;
};

// The walk over the cache: this lane's sums o (columns 16 d + 4 g + e of its position) and its keys' share l of the
// probabilities.  kTwo: a probability as two parts; one: where a value is no number.
template <bool kTwo>
__device__ __forceinline__ void prompt_walk(const PromptParams& p, char* ks, char* vs, const int tid, const v4u (&qf)[4],
                                            const uint16_t* mrow, const uint16_t* kb, const uint16_t* vb, v4f (&o)[8],
                                            float& l) {
    const int lane = tid & 63, i = lane & 15, g = lane >> 4;
#pragma unroll
    for (int d = 0; d < 8; ++d) o[d] = v4f{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY;
    l = 0.f;
    const int blocks = (p.max_len + kPKeys - 1) / kPKeys;
    // the mask of keys 16 kt + 4 g ... + 3 of a block (max_len % 4 == 0: four keys are inside or outside together)
    auto load_mask = [&](v2u (&mk)[4], const int blk) {
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            const int j = blk * kPKeys + kt * 16 + 4 * g;
            mk[kt] = j < p.max_len ? *(const v2u*)(mrow + j) : v2u{0xFF80FF80u, 0xFF80FF80u};  // -inf
        }
    };
    v2u mk[4], mk_next[4];
    load_mask(mk_next, 0);
    for (int blk = 0; blk < blocks; ++blk) {
        u32 open = 0;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            mk[kt] = mk_next[kt];
#pragma unroll
            for (int e = 0; e < 2; ++e) open |= (mk[kt][e] ^ 0xFF80FF80u);
        }
        if (blk + 1 < blocks) load_mask(mk_next, blk + 1);
        // (the barrier also ends the reads of the block before)
        if (!__syncthreads_or(open != 0)) continue;
        // ---- keys as they lie, values transposed, into LDS; rows past the cache repeat its last ----
        {
            const int c = tid & 15, a = tid >> 4;
            v4u kk[4], vv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int64_t j = blk * kPKeys + 4 * a + r;
                const int64_t at = (j < p.max_len ? j : p.max_len - 1) * kHd + 8 * c;
                kk[r] = *(const v4u*)(kb + at);
                vv[r] = *(const v4u*)(vb + at);
                if (!kTwo && j >= p.max_len) vv[r] = v4u{0u, 0u, 0u, 0u};  // (nothing, not 0 times what the last row holds)
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) *(v4u*)(ks + (4 * a + r) * kPKPitch + 16 * c) = kk[r];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const u32 sel = e & 1 ? 0x07060302u : 0x05040100u;
                const v2u w = {byte_perm(vv[1][e >> 1], vv[0][e >> 1], sel), byte_perm(vv[3][e >> 1], vv[2][e >> 1], sel)};
                *(v2u*)(vs + (8 * c + e) * kPVPitch + 8 * a) = w;
            }
        }
        __syncthreads();
        // ---- scores ----
        float x[4][4];
        float top = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const v4u kf = *(const v4u*)(ks + (kt * 16 + i) * kPKPitch + 64 * s + 16 * g);
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, kf), __builtin_bit_cast(v8bf, qf[s]), acc,
                                                              0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const u32 w = mk[kt][e >> 1];
                const float v = acc[e] * p.scale + __uint_as_float(e & 1 ? w & 0xffff0000u : w << 16);
                x[kt][e] = v < kPLowest ? -INFINITY : v;
                top = fmaxf(top, x[kt][e]);
            }
        }
        top = fmaxf(top, __shfl_xor(top, 16, kWave));
        top = fmaxf(top, __shfl_xor(top, 32, kWave));
        const float m_new = fmaxf(m, top);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;  // (nothing open yet: every term below is zero)
        const float shrink = __builtin_amdgcn_exp2f((m - m_use) * 1.44269504f);
        m = m_new;
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[kt][e] = __builtin_amdgcn_exp2f((x[kt][e] - m_use) * 1.44269504f);
                sum += x[kt][e];
            }
        l = l * shrink + sum;  // (this lane's keys; the four lanes of a position meet at the end)
#pragma unroll
        for (int d = 0; d < 8; ++d)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[d][e] *= shrink;
        // ---- values: 32 keys per product, slot 8 g + e of it key 16 (2 pr) + 4 g + e, slots e >= 4 the next 16's ----
#pragma unroll
        for (int pr = 0; pr < 2; ++pr) {
            v4u hi, lo;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v0 = x[2 * pr + (e >> 1)][2 * (e & 1)], v1 = x[2 * pr + (e >> 1)][2 * (e & 1) + 1];
                hi[e] = pack_bf16x2(v0, v1);
                lo[e] = pack_bf16x2(v0 - __uint_as_float(hi[e] << 16), v1 - __uint_as_float(hi[e] & 0xffff0000u));
            }
#pragma unroll
            for (int d = 0; d < 8; ++d) {
                const char* at = vs + (16 * d + i) * kPVPitch + (32 * pr + 4 * g) * 2;
                const v2u v0 = *(const v2u*)at, v1 = *(const v2u*)(at + 32);
                const v8bf vf = __builtin_bit_cast(v8bf, (v4u{v0[0], v0[1], v1[0], v1[1]}));
                if (kTwo) o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(v8bf, lo), o[d], 0, 0, 0);
                o[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(v8bf, hi), o[d], 0, 0, 0);
            }
        }
    }
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
}

// (the bound keeps three waves a SIMD, as one walk alone has; two cost 0.3 % of a prompt of 8 x 128 positions)
__global__ __launch_bounds__(256, 3) void prompt_attention(PromptParams p) {
    __shared__ __attribute__((aligned(16))) char ks[kPKeys * kPKPitch];
    __shared__ __attribute__((aligned(16))) char vs[kHd * kPVPitch];
    const int tid = threadIdx.x, lane = tid & 63, i = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t bh = blockIdx.x;
    const int64_t b = bh / p.H;
    const int h = (int)(bh - b * p.H);
    const int t0 = (int)blockIdx.y * kPRows + wave * 16;
    const int t = t0 + i < p.T ? t0 + i : p.T - 1;  // this lane's position (past the end: a copy of the last, not stored)
    const int64_t qrow = ((b * p.T + t) * p.H + h) * kHd;
    v4u qf[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[s] = *(const v4u*)(p.q + qrow + 32 * s + 8 * g);
    const uint16_t* mrow = p.mask + (int64_t)t * p.max_len;
    const uint16_t* kb = p.kc + bh * p.max_len * kHd;
    const uint16_t* vb = p.vc + bh * p.max_len * kHd;
    v4f o[8];
    float l;
    prompt_walk<true>(p, ks, vs, tid, qf, mrow, kb, vb, o, l);
    const bool live = t0 + i < p.T;
    // (a position with no open row has no probabilities: zeros, as the library gives)
    auto value = [&](const int d, const int e) { return l == 0.f ? 0.f : o[d][e] / l; };
    u32 odd = 0;  // this lane's results that are no numbers
#pragma unroll
    for (int d = 0; d < 8; ++d) {
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            y[e] = value(d, e);
            if (!(fabsf(y[e]) < INFINITY)) odd |= 1u << (4 * d + e);
        }
        if (live) *(v2u*)(p.out + qrow + 16 * d + 4 * g) = v2u{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
    }
    // The low part of a probability may be zero or negative, so that an infinite value makes a NaN of an infinity: such
    // results are worked out again with one part.
    if (!__syncthreads_or(live && odd)) return;
    prompt_walk<false>(p, ks, vs, tid, qf, mrow, kb, vb, o, l);
#pragma unroll
    for (int d = 0; d < 8; ++d)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (live && ((odd >> (4 * d + e)) & 1)) p.out[qrow + 16 * d + 4 * g + e] = (uint16_t)f32_to_bf16_bits(value(d, e));
}


}  // namespace
}  // namespace k3q

using namespace k3q;

extern "C" int k3q_prompt_attention(const void* q, int dtype, int64_t B, int64_t T, int64_t H, int64_t head_dim,
                                    int64_t max_len, const void* k_cache, const void* v_cache, const void* mask,
                                    void* out, void* stream) {
    if (dtype != K3Q_BF16) return K3Q_ERR_DTYPE;
    if (B < 0 || T < 0 || H <= 0 || head_dim != kHd || max_len <= 0 || (max_len % 4) != 0 || max_len >= (1 << 30) ||
        T > 65535 * kPRows || H >= (1 << 20))
        return K3Q_ERR_SHAPE;
    if (B == 0 || T == 0) return K3Q_OK;
    if (B >= (int64_t(1) << 31) / H) return K3Q_ERR_SHAPE;
    if (!q || !k_cache || !v_cache || !mask || !out) return K3Q_ERR_NULL;
    if (!aligned_to(q, 16) || !aligned_to(k_cache, 16) || !aligned_to(v_cache, 16) || !aligned_to(mask, 8) ||
        !aligned_to(out, 8))
        return K3Q_ERR_ALIGN;
    PromptParams p;
    p.q = (const uint16_t*)q;
    p.kc = (const uint16_t*)k_cache;
    p.vc = (const uint16_t*)v_cache;
    p.mask = (const uint16_t*)mask;
    p.out = (uint16_t*)out;
    p.T = (int)T;
    p.H = (int)H;
    p.max_len = (int)max_len;
    p.scale = 0.08838834764831845f;  // 1 / sqrt(128)
    prompt_attention<<<dim3((unsigned)(B * H), (unsigned)((T + kPRows - 1) / kPRows)), 256, 0, (hipStream_t)stream>>>(p);
    return launch_status();
}

extern "C" int k3q_rope_cache(const void* q, const void* k, const void* v, int dtype, int64_t B, int64_t T, int64_t H,
                              int64_t head_dim, int64_t max_len, const void* cos_table, const void* sin_table,
                              const int64_t* pos, void* k_cache, void* v_cache, void* q_out, int* oob_flag,
                              void* stream) {
    if (dtype != K3Q_BF16) return K3Q_ERR_DTYPE;
    if (B < 0 || T < 0 || H <= 0 || head_dim != kHd || max_len <= 0 || max_len >= (1 << 30) || T >= (1 << 30) ||
        H >= (1 << 20))
        return K3Q_ERR_SHAPE;
    if (B == 0 || T == 0) return K3Q_OK;
    if (B > (int64_t(1) << 33) / T / H) return K3Q_ERR_SHAPE;
    if (!q || !k || !v || !cos_table || !sin_table || !pos || !k_cache || !v_cache || !q_out) return K3Q_ERR_NULL;
    if (!aligned_to(q, 16) || !aligned_to(k, 16) || !aligned_to(v, 16) || !aligned_to(cos_table, 16) ||
        !aligned_to(sin_table, 16) || !aligned_to(pos, 8) || !aligned_to(k_cache, 16) || !aligned_to(v_cache, 16) ||
        !aligned_to(q_out, 16))
        return K3Q_ERR_ALIGN;
    RopeParams p;
    p.q = (const uint16_t*)q;
    p.k = (const uint16_t*)k;
    p.v = (const uint16_t*)v;
    p.cos_t = (const uint16_t*)cos_table;
    p.sin_t = (const uint16_t*)sin_table;
    p.pos = pos;
    p.kc = (uint16_t*)k_cache;
    p.vc = (uint16_t*)v_cache;
    p.out = (uint16_t*)q_out;
    p.oob = oob_flag;
    p.heads = B * T * H;
    p.T = (int)T;
    p.H = (int)H;
    p.max_len = (int)max_len;
    rope_cache_rows<<<(unsigned)((p.heads * 8 + 255) / 256), 256, 0, (hipStream_t)stream>>>(p);
    return launch_status();
}

extern "C" int k3q_decode_attention(const void* q, const void* k, const void* v, int dtype, int64_t B,
                                    int64_t H, int64_t head_dim, int64_t max_len, const void* cos_table,
                                    const void* sin_table, const int64_t* pos, void* k_cache,
                                    void* v_cache, void* out, int* oob_flag, void* stream) {
    if (dtype != K3Q_BF16) return K3Q_ERR_DTYPE;
    if (B < 0 || H <= 0 || head_dim != kHd || max_len <= 0 || max_len > 32768 || B * H >= (1 << 30))
        return K3Q_ERR_SHAPE;
    if (B == 0) return K3Q_OK;
    if (!q || !k || !v || !cos_table || !sin_table || !pos || !k_cache || !v_cache || !out) return K3Q_ERR_NULL;
    if (!aligned_to(v, 16) || !aligned_to(k_cache, 16) || !aligned_to(v_cache, 16) || !aligned_to(pos, 8))
        return K3Q_ERR_ALIGN;
    AttnParams p;
    p.q = (const uint16_t*)q;
    p.k = (const uint16_t*)k;
    p.v = (const uint16_t*)v;
    p.cos_t = (const uint16_t*)cos_table;
    p.sin_t = (const uint16_t*)sin_table;
    p.pos = pos;
    p.kc = (uint16_t*)k_cache;
    p.vc = (uint16_t*)v_cache;
    p.out = (uint16_t*)out;
    p.oob = oob_flag;
    p.H = (int)H;
    p.max_len = (int)max_len;
    p.scale = 0.08838834764831845f;  // 1 / sqrt(128)
    const size_t lds = (size_t)(kHd + 2 * kAW + kAW * kHd + kHd + max_len) * sizeof(float);  // as laid out in the kernel
    if (lds > 64 * 1024) {
        static const bool raised = hipFuncSetAttribute((const void*)decode_attention,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       160 * 1024) == hipSuccess;
        if (!raised) return K3Q_ERR_LAUNCH;
    }
    decode_attention<<<(unsigned)(B * H), kAT, lds, (hipStream_t)stream>>>(p);
    return launch_status();
}
