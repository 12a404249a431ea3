// Weight quantizers for kernels that already live on the device: the float32 arithmetic of the
// reference's numpy (`to_numpy=True`) paths, step for step, so that the integers, scales and zero
// points are the bits numpy produces on the host.
//
//   absmax_reduce   abs-max over a run of axes that is not trailing: x [outer, R, inner], one scale
//                   per (outer, inner) -- Dense kernels (axis 0: outer 1, R = input_dim, inner =
//                   units) and EinsumDense kernels (keras/src/quantizers/quantizers.py:95-109)
//   grouped_zp      groups of `block` rows of a [K, N] kernel, per (group, column) scale and zero
//                   point from the group's min / max (quantizers.py:182-234)
//
// What makes the bits equal: every step is one IEEE float32 operation in numpy and here (compiled
// with -ffp-contract=off, `/` is the correctly rounded division, rintf rounds half to even as
// np.round does); bfloat16 inputs are widened first, as the reference's conversion to numpy does.
// The abs-max form reads x twice (a column's maximum needs all of the column before the first integer).
// It is bound by memory where there are workgroups enough: a thread has kWqDeep rows in flight, and a
// kernel that would make fewer than 1024 workgroups is cut into shorter chunks of rows -- down to 64, and
// to 32 below 512 workgroups, since every chunk costs an atomic a column (6400 x 1600: 24 us in chunks of
// 64, 30 of 32).  One row at a time in chunks of 256 -> now, float32 / bfloat16, us: 768 x 768 27 / 28 -> 8 / 8,
// 1600 x 6400 46 / 45 -> 19 / 15, 4096 x 4096 45 / 52 -> 29 / 24, 4096 x 14336 111 / 84 -> 87 / 53, 8192 x 8192
// 116 / 95 -> 113 / 59.  Pass 2 goes from the end of x to its start and stores past the caches (with ordinary stores
// 4096 x 14336 takes 97).
//  Groups of up to 128 rows keep
// their rows in registers between the min / max and the integers (grouped_zp_held: one read); larger
// groups take the generic two-pass kernel.
#include <type_traits>

#include "k3q_common.h"

namespace k3q {
namespace {

constexpr int kWqX = 64;   // threads along the columns
constexpr int kWqY = 4;    // threads along the reduced rows
constexpr int kWqT = kWqX * kWqY;
constexpr int kWqDeep = 8;     // rows that a thread of the abs-max passes has in flight

// kV values as they lie in memory, and as floats
template <bool kBF16, int kV>
struct RawVals {
    typedef typename std::conditional<kBF16, v2u, v4u>::type Four;
    typename std::conditional<kV == 4, Four, u32>::type raw;
    __device__ __forceinline__ void load(const void* x, int64_t idx) {
        if constexpr (kV == 4) raw = *(const Four*)((const char*)x + idx * (kBF16 ? 2 : 4));
        else raw = load_raw<kBF16>(x, idx);
    }
    __device__ __forceinline__ void values(float* f) const {
        if constexpr (kV != 4) {
            f[0] = raw_to_f32<kBF16>(raw);
        } else if constexpr (kBF16) {
            f[0] = __uint_as_float(raw[0] << 16);
            f[1] = __uint_as_float(raw[0] & 0xffff0000u);
            f[2] = __uint_as_float(raw[1] << 16);
            f[3] = __uint_as_float(raw[1] & 0xffff0000u);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = __uint_as_float(raw[e]);
        }
    }
};

template <bool kBF16, int kV>
__device__ __forceinline__ void load_vals(const void* x, int64_t idx, float* f) {
    RawVals<kBF16, kV> v;
    v.load(x, idx);
    v.values(f);
}

// kStream: past the caches, which keep more of the input then
template <int kV, bool kStream = false>
__device__ __forceinline__ void store_q(int8_t* q, int64_t idx, const int* v) {
    if (kV == 4) {
        const u32 w = (u32)(v[0] & 0xff) | ((u32)(v[1] & 0xff) << 8) | ((u32)(v[2] & 0xff) << 16) |
                      ((u32)(v[3] & 0xff) << 24);
        if (kStream) __builtin_nontemporal_store(w, (u32*)(q + idx));
        else *(u32*)(q + idx) = w;
    } else {
        q[idx] = (int8_t)v[0];
    }
}

template <bool kBF16>
__device__ __forceinline__ void store_scale(void* s, int64_t idx, float v) {
    if (kBF16) ((uint16_t*)s)[idx] = (uint16_t)f32_to_bf16_bits(v);
    else ((float*)s)[idx] = v;
}

struct ReduceParams {
    const void* x;
    int8_t* q;
    void* scale;
    u32* amax;  // [outer * inner] bit patterns of the running max of |x| (zeroed by the entry point)
    int64_t R, inner;
    int chunk;  // rows of R per workgroup
    float eps, qlo, qhi;
};

// pass 1: |x| maxima of a chunk of rows, merged into `amax` with an unsigned max of the bit patterns
// (non-negative floats order like their bits)
template <bool kBF16, int kV>
__global__ __launch_bounds__(kWqT) void absmax_reduce_max(ReduceParams p) {
    __shared__ float part[kWqY][kWqX * 4];
    const int tx = threadIdx.x % kWqX, ty = threadIdx.x / kWqX;
    const int64_t col = ((int64_t)blockIdx.x * kWqX + tx) * kV;
    const int64_t o = blockIdx.z;
    const int64_t r0 = (int64_t)blockIdx.y * p.chunk;
    const int64_t r1 = r0 + p.chunk < p.R ? r0 + p.chunk : p.R;
    float m[kV];
#pragma unroll
    for (int e = 0; e < kV; ++e) m[e] = 0.f;
    if (col < p.inner) {
        for (int64_t r = r0 + ty; r < r1; r += kWqY * kWqDeep) {
            RawVals<kBF16, kV> raw[kWqDeep];  // (a row past the chunk's last counts as that one again)
#pragma unroll
            for (int j = 0; j < kWqDeep; ++j)
                raw[j].load(p.x, (o * p.R + (r + j * kWqY < r1 ? r + j * kWqY : r1 - 1)) * p.inner + col);
#pragma unroll
            for (int j = 0; j < kWqDeep; ++j) {
                float f[kV];
                raw[j].values(f);
#pragma unroll
                for (int e = 0; e < kV; ++e) m[e] = fmaxf(m[e], fabsf(f[e]));
            }
        }
    }
#pragma unroll
    for (int e = 0; e < kV; ++e) part[ty][tx * 4 + e] = m[e];
    __syncthreads();
    if (ty == 0 && col < p.inner) {
#pragma unroll
        for (int e = 0; e < kV; ++e) {
            float v = part[0][tx * 4 + e];
#pragma unroll
            for (int y = 1; y < kWqY; ++y) v = fmaxf(v, part[y][tx * 4 + e]);
            atomicMax(p.amax + o * p.inner + col + e, __float_as_uint(v));
        }
    }
}

// pass 2: scale = hi / (amax + eps), q = clip(rint(x * scale)); from the end of x to its start, so that what pass 1 read last
// comes out of the caches
template <bool kBF16, int kV>
__global__ __launch_bounds__(kWqT) void absmax_reduce_quantize(ReduceParams p) {
    const int tx = threadIdx.x % kWqX, ty = threadIdx.x / kWqX;
    const int64_t col = ((int64_t)(gridDim.x - 1 - blockIdx.x) * kWqX + tx) * kV;
    if (col >= p.inner) return;
    const int64_t o = gridDim.z - 1 - blockIdx.z;
    const int64_t r0 = (int64_t)(gridDim.y - 1 - blockIdx.y) * p.chunk;
    const int64_t r1 = r0 + p.chunk < p.R ? r0 + p.chunk : p.R;
    float s[kV];
#pragma unroll
    for (int e = 0; e < kV; ++e) s[e] = p.qhi / (__uint_as_float(p.amax[o * p.inner + col + e]) + p.eps);
    if (blockIdx.y == 0 && ty == 0) {
#pragma unroll
        for (int e = 0; e < kV; ++e) store_scale<kBF16>(p.scale, o * p.inner + col + e, s[e]);
    }
    for (int64_t r = r0 + ty; r < r1; r += kWqY * kWqDeep) {
        RawVals<kBF16, kV> raw[kWqDeep];
#pragma unroll
        for (int j = 0; j < kWqDeep; ++j)
            raw[j].load(p.x, (o * p.R + (r + j * kWqY < r1 ? r + j * kWqY : r1 - 1)) * p.inner + col);
#pragma unroll
        for (int j = 0; j < kWqDeep; ++j) {
            if (r + j * kWqY >= r1) break;
            float f[kV];
            int v[kV];
            raw[j].values(f);
#pragma unroll
            for (int e = 0; e < kV; ++e) v[e] = (int)fminf(fmaxf(rintf(f[e] * s[e]), p.qlo), p.qhi);
            store_q<kV, true>(p.q, (o * p.R + r + j * kWqY) * p.inner + col, v);
        }
    }
}

struct GroupedParams {
    const void* x;
    int8_t* q;
    void* scale;
    int8_t* zero;
    int64_t K, N;
    int block;
    float eps, qmin, qmax, levels;  // levels = qmax - qmin
};

// one workgroup per (column tile, group): min / max of the group's rows (rows past K count as the
// zeros the reference pads with), then scale, zero point and the integers
template <bool kBF16, int kV>
__global__ __launch_bounds__(kWqT) void grouped_zp(GroupedParams p) {
    __shared__ float lo_s[kWqY][kWqX * 4], hi_s[kWqY][kWqX * 4];
    const int tx = threadIdx.x % kWqX, ty = threadIdx.x / kWqX;
    const int64_t col = ((int64_t)blockIdx.x * kWqX + tx) * kV;
    const int64_t g = blockIdx.y;
    const int64_t r0 = g * p.block;
    const bool live = col < p.N;
    float lo[kV], hi[kV];
#pragma unroll
    for (int e = 0; e < kV; ++e) {
        lo[e] = INFINITY;
        hi[e] = -INFINITY;
    }
    if (live) {
        for (int i = ty; i < p.block; i += kWqY) {
            float f[kV];
            if (r0 + i < p.K) {
                load_vals<kBF16, kV>(p.x, (r0 + i) * p.N + col, f);
            } else {
#pragma unroll
                for (int e = 0; e < kV; ++e) f[e] = 0.f;
            }
#pragma unroll
            for (int e = 0; e < kV; ++e) {
                lo[e] = fminf(lo[e], f[e]);
                hi[e] = fmaxf(hi[e], f[e]);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < kV; ++e) {
        lo_s[ty][tx * 4 + e] = lo[e];
        hi_s[ty][tx * 4 + e] = hi[e];
    }
    __syncthreads();
    if (!live) return;
    float scale[kV], zero[kV];
#pragma unroll
    for (int e = 0; e < kV; ++e) {
        float l = lo_s[0][tx * 4 + e], h = hi_s[0][tx * 4 + e];
#pragma unroll
        for (int y = 1; y < kWqY; ++y) {
            l = fminf(l, lo_s[y][tx * 4 + e]);
            h = fmaxf(h, hi_s[y][tx * 4 + e]);
        }
        scale[e] = ((h - l) + p.eps) / p.levels;
        zero[e] = fminf(fmaxf(rintf(-l / scale[e]) + p.qmin, p.qmin), p.qmax);
    }
    if (ty == 0) {
#pragma unroll
        for (int e = 0; e < kV; ++e) {
            store_scale<kBF16>(p.scale, g * p.N + col + e, scale[e]);
            p.zero[g * p.N + col + e] = (int8_t)(int)zero[e];
        }
    }
    for (int i = ty; i < p.block && r0 + i < p.K; i += kWqY) {
        const int64_t idx = (r0 + i) * p.N + col;
        float f[kV];
        load_vals<kBF16, kV>(p.x, idx, f);
        int v[kV];
#pragma unroll
        for (int e = 0; e < kV; ++e)
            v[e] = (int)fminf(fmaxf(rintf(f[e] / scale[e]) + zero[e], p.qmin), p.qmax);
        store_q<kV>(p.q, idx, v);
    }
}

// rintf(x / s) with the division's own rounding, for a column scale s > 0 whose reciprocal
// (correctly rounded) is at hand.  r = x * (1 / s) lies within 3 * 2^-24 |r| of the correctly rounded
// quotient t, so rint(t) = rint(r) unless r is that close to a half-integer; there (and for
// anything that is not a number) the division is done.  The margin used is 2^-20 |r|.
// Four columns of a row share one branch (a value in 2^15 takes it; the quotient is right for all of them).
__device__ __forceinline__ void rint_quotients(const float (&x)[4], const float (&s)[4], const float (&inv_s)[4],
                                               float (&n)[4]) {
    bool safe = true;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float r = x[e] * inv_s[e];
        n[e] = rintf(r);
        safe &= 0.5f - fabsf(r - n[e]) > fabsf(r) * 0x1p-20f;
    }
    if (!safe) {
#pragma unroll
        for (int e = 0; e < 4; ++e) n[e] = rintf(x[e] / s[e]);
    }
}

// The same for groups of up to kHeldY * kHeldRows rows with N a multiple of 4.  A thread keeps its rows of a work item (column
// tile, group) in registers between the two passes, so memory sees x once; the integers come from rint_quotients.  A
// workgroup walks the items at a stride of the grid, and a row's registers take the next item's row as soon as the row's
// integers are out: loads run through the whole of the vector work, and a workgroup holds the registers of one item only.
// Every load of an item is unconditional, at a row and a column held inside x (what a repeated row holds is not used): with a
// condition on each, the compiler waited for every load before the next.  4096 x 14336 float32 to int4, groups of 128:
// 73.3 -> 51.8 us, where reading x and writing the result takes 52 at the rate of a large copy (8192 x 8192: 79.0 -> 57.9,
// 1600 x 6400, whose last group is short: 22.1 -> 18.7).
// kFull: every group has kHeldY * kHeldRows rows, all of them in x; no condition is left between the loads and stores, and 96
// registers let two workgroups share a CU.  kPacked: the integers leave as int4 pairs along N (k3q_pack_int4's bytes; q is
// [K, N / 2], the range fits four bits): half a byte written per weight instead of one byte written, read again and packed.
constexpr int kHeldY = 8, kHeldRows = 16;
// kRows: rows of a group that a thread holds, the smallest of 2, 4, 8 and 16 that takes the group.  With 16 for all of them a
// thread loaded its last row again up to fourteen times: 4096 x 14336 float32, groups of 8, 16, 32 and 64, conditional loads /
// 16 rows / now: 262 / 295 / 150, 155 / 168 / 97, 104 / 101 / 64, 77 / 70 / 51 us.
template <int kRows, bool kFull, bool kBF16, bool kPacked>
__global__ __launch_bounds__(kWqX * kHeldY, kFull || kRows < kHeldRows ? 4 : 2) void grouped_zp_held(GroupedParams p, int col_tiles,
                                                                                                     int items) {
    __shared__ float lo_s[2][kHeldY][kWqX * 4], hi_s[2][kHeldY][kWqX * 4];
    const int tx = threadIdx.x % kWqX, ty = __builtin_amdgcn_readfirstlane(threadIdx.x / kWqX);
    RawVals<kBF16, 4> rows[kRows];
    auto fetch = [&](const int item, const int j) {
        const int g = item / col_tiles;
        const int64_t col = ((int64_t)(item - g * col_tiles) * kWqX + tx) * 4, r0 = (int64_t)g * p.block;
        const int i = ty + j * kHeldY;
        int64_t r = r0 + (i < p.block ? i : p.block - 1);
        r = r < p.K ? r : p.K - 1;
        rows[j].load(p.x, r * p.N + (col < p.N ? col : p.N - 4));
    };
    auto work = [&](auto more, const int item, const int next, const int par) {
        constexpr bool kMore = decltype(more)::value;  // (there is a next item)
        const int g = item / col_tiles;
        const int64_t col = ((int64_t)(item - g * col_tiles) * kWqX + tx) * 4, r0 = (int64_t)g * p.block;
        float lo[4], hi[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            lo[e] = INFINITY;
            hi[e] = -INFINITY;
        }
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
            const int i = ty + j * kHeldY;
            if (!kFull && i >= p.block) break;
            float f[4];
            rows[j].values(f);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = kFull || r0 + i < p.K ? f[e] : 0.f;  // (rows past K count as zeros)
                lo[e] = fminf(lo[e], v);
                hi[e] = fmaxf(hi[e], v);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            lo_s[par][ty][tx * 4 + e] = lo[e];
            hi_s[par][ty][tx * 4 + e] = hi[e];
        }
        __syncthreads();  // (the buffers alternate, so the item after the next may overwrite this one's)
        float scale[4], inv[4], zero[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float l = lo_s[par][0][tx * 4 + e], h = hi_s[par][0][tx * 4 + e];
#pragma unroll
            for (int y = 1; y < kHeldY; ++y) {
                l = fminf(l, lo_s[par][y][tx * 4 + e]);
                h = fmaxf(h, hi_s[par][y][tx * 4 + e]);
            }
            scale[e] = ((h - l) + p.eps) / p.levels;
            inv[e] = 1.0f / scale[e];
            zero[e] = fminf(fmaxf(rintf(-l / scale[e]) + p.qmin, p.qmin), p.qmax);
        }
        const bool live = col < p.N;
        if (ty == 0 && live) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                store_scale<kBF16>(p.scale, g * p.N + col + e, scale[e]);
                p.zero[g * p.N + col + e] = (int8_t)(int)zero[e];
            }
        }
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
            const int i = ty + j * kHeldY;
            if (kFull || (i < p.block && r0 + i < p.K)) {
                float f[4], n[4];
                int v[4];
                rows[j].values(f);
                rint_quotients(f, scale, inv, n);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = (int)__builtin_amdgcn_fmed3f(n[e] + zero[e], p.qmin, p.qmax);
                if (live) {
                    if (kPacked)
                        *(uint16_t*)(p.q + ((r0 + i) * p.N + col) / 2) = (uint16_t)(
                            (v[0] & 0xf) | ((v[1] & 0xf) << 4) | ((v[2] & 0xf) << 8) | ((v[3] & 0xf) << 12));
                    else
                        store_q<4>(p.q, (r0 + i) * p.N + col, v);
                }
            }
            if (kMore) fetch(next, j);
        }
    };
    const int step = gridDim.x;
    int item = blockIdx.x;
#pragma unroll
    for (int j = 0; j < kRows; ++j) fetch(item, j);
    int par = 0;
#pragma clang loop unroll(disable)
    for (; item + step < items; item += step, par ^= 1)  // (uniform over the workgroup: every thread meets every barrier)
        work(std::true_type{}, item, item + step, par);
    work(std::false_type{}, item, item, par);
}

template <int kRows, bool kFull>
void (*held_kernel(const bool bf, const bool packed))(GroupedParams, int, int) {
    return bf ? (packed ? grouped_zp_held<kRows, kFull, true, true> : grouped_zp_held<kRows, kFull, true, false>)
              : (packed ? grouped_zp_held<kRows, kFull, false, true> : grouped_zp_held<kRows, kFull, false, false>);
}

__global__ void clear_u32(u32* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

}  // namespace
}  // namespace k3q

using namespace k3q;

extern "C" int k3q_weight_absmax_quantize(const void* x, int x_dtype, int64_t outer, int64_t R, int64_t inner,
                                          float epsilon, float range_lo, float range_hi, int8_t* q,
                                          void* scale, void* amax_workspace, void* stream) {
    if (x_dtype != K3Q_F32 && x_dtype != K3Q_BF16) return K3Q_ERR_DTYPE;
    if (outer < 0 || R < 0 || inner < 0 || outer > 65535) return K3Q_ERR_SHAPE;
    if (range_lo < -128.f || range_hi > 127.f || range_lo > range_hi) return K3Q_ERR_RANGE;
    if (outer == 0 || inner == 0) return K3Q_OK;
    if (R == 0) return K3Q_ERR_SHAPE;  // the maximum of nothing
    if (!x || !q || !scale || !amax_workspace) return K3Q_ERR_NULL;
    if ((R + 255) / 256 > 65535) return K3Q_ERR_SHAPE;
    hipStream_t s = (hipStream_t)stream;
    ReduceParams p;
    p.x = x;
    p.q = q;
    p.scale = scale;
    p.amax = (u32*)amax_workspace;
    p.R = R;
    p.inner = inner;
    p.eps = epsilon;
    p.qlo = range_lo;
    p.qhi = range_hi;
    const int64_t cells = outer * inner;
    clear_u32<<<(unsigned)((cells + 255) / 256), 256, 0, s>>>(p.amax, cells);
    const bool bf = x_dtype == K3Q_BF16;
    const bool vec = (inner % 4) == 0 && aligned_to(x, bf ? 8 : 16) && aligned_to(q, 4);
    const int v = vec ? 4 : 1;
    const int64_t col_tiles = (inner + (int64_t)kWqX * v - 1) / ((int64_t)kWqX * v);
    p.chunk = 256;  // (the reasons stand at the top)
    const int64_t across = col_tiles * outer;
    while (p.chunk > 32 && across * ((R + p.chunk - 1) / p.chunk) < (p.chunk > 64 ? 1024 : 512)) p.chunk /= 2;
    dim3 grid((unsigned)col_tiles, (unsigned)((R + p.chunk - 1) / p.chunk), (unsigned)outer);
    if (bf && vec) {
        absmax_reduce_max<true, 4><<<grid, kWqT, 0, s>>>(p);
        absmax_reduce_quantize<true, 4><<<grid, kWqT, 0, s>>>(p);
    } else if (bf) {
        absmax_reduce_max<true, 1><<<grid, kWqT, 0, s>>>(p);
        absmax_reduce_quantize<true, 1><<<grid, kWqT, 0, s>>>(p);
    } else if (vec) {
        absmax_reduce_max<false, 4><<<grid, kWqT, 0, s>>>(p);
        absmax_reduce_quantize<false, 4><<<grid, kWqT, 0, s>>>(p);
    } else {
        absmax_reduce_max<false, 1><<<grid, kWqT, 0, s>>>(p);
        absmax_reduce_quantize<false, 1><<<grid, kWqT, 0, s>>>(p);
    }
    return launch_status();
}

static int run_weight_quantize_grouped(const void* x, int x_dtype, int64_t K, int64_t N, int64_t block_size,
                                       float epsilon, float range_lo, float range_hi, int8_t* q, bool packed,
                                       void* scale, int8_t* zero, void* stream) {
    if (x_dtype != K3Q_F32 && x_dtype != K3Q_BF16) return K3Q_ERR_DTYPE;
    if (K < 0 || N < 0 || block_size <= 0 || block_size > (1 << 20)) return K3Q_ERR_SHAPE;
    if (range_lo < -128.f || range_hi > 127.f || range_lo >= range_hi) return K3Q_ERR_RANGE;
    if (K == 0 || N == 0) return K3Q_OK;
    if (!x || !q || !scale || !zero) return K3Q_ERR_NULL;
    const int64_t groups = (K + block_size - 1) / block_size;
    if (groups > 65535) return K3Q_ERR_SHAPE;
    GroupedParams p;
    p.x = x;
    p.q = q;
    p.scale = scale;
    p.zero = zero;
    p.K = K;
    p.N = N;
    p.block = (int)block_size;
    p.eps = epsilon;
    p.qmin = range_lo;
    p.qmax = range_hi;
    p.levels = range_hi - range_lo;
    const bool bf = x_dtype == K3Q_BF16;
    const bool vec = (N % 4) == 0 && aligned_to(x, bf ? 8 : 16) && aligned_to(q, 4);
    const int v = vec ? 4 : 1;
    dim3 grid((unsigned)((N + (int64_t)kWqX * v - 1) / ((int64_t)kWqX * v)), (unsigned)groups);
    hipStream_t s = (hipStream_t)stream;
    // the held form's quotient needs a finite positive scale and its reciprocal: an epsilon > 0 gives
    // both for any finite kernel
    const int64_t col_tiles = grid.x, items = col_tiles * groups;
    const bool held = vec && block_size <= (int64_t)kHeldY * kHeldRows && epsilon > 0.f && items < (1ll << 30);
    if (held) {
        // two workgroups per CU where the registers allow it; 256, 768 and 1024 of them, and one per item, take 54.6, 56.6,
        // 52.9 and 52.9 us where this takes 51.8 (4096 x 14336)
        const unsigned blocks = (unsigned)(items < 512 ? items : 512);
        const bool full = block_size == kHeldY * kHeldRows && K % block_size == 0;
        void (*kernel)(GroupedParams, int, int) =
            full                         ? held_kernel<kHeldRows, true>(bf, packed)
            : block_size <= 2 * kHeldY ? held_kernel<2, false>(bf, packed)
            : block_size <= 4 * kHeldY ? held_kernel<4, false>(bf, packed)
            : block_size <= 8 * kHeldY ? held_kernel<8, false>(bf, packed)
                                         : held_kernel<kHeldRows, false>(bf, packed);
        kernel<<<blocks, kWqX * kHeldY, 0, s>>>(p, (int)col_tiles, (int)items);
        return launch_status();
    }
    if (packed) return K3Q_ERR_SHAPE;
    if (bf && vec) grouped_zp<true, 4><<<grid, kWqT, 0, s>>>(p);
    else if (bf) grouped_zp<true, 1><<<grid, kWqT, 0, s>>>(p);
    else if (vec) grouped_zp<false, 4><<<grid, kWqT, 0, s>>>(p);
    else grouped_zp<false, 1><<<grid, kWqT, 0, s>>>(p);
    return launch_status();
}

extern "C" int k3q_weight_quantize_grouped(const void* x, int x_dtype, int64_t K, int64_t N, int64_t block_size,
                                           float epsilon, float range_lo, float range_hi, int8_t* q,
                                           void* scale, int8_t* zero, void* stream) {
    return run_weight_quantize_grouped(x, x_dtype, K, N, block_size, epsilon, range_lo, range_hi, q, false, scale, zero,
                                       stream);
}

extern "C" int k3q_weight_quantize_grouped_int4(const void* x, int x_dtype, int64_t K, int64_t N, int64_t block_size,
                                                float epsilon, int8_t* packed, void* scale, int8_t* zero,
                                                void* stream) {
    return run_weight_quantize_grouped(x, x_dtype, K, N, block_size, epsilon, -8.f, 7.f, packed, true, scale, zero,
                                       stream);
}
