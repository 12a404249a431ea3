// Conversion of a strip-linear int4 copy's nibbles that leaves no offset in the weights.
#pragma once

#include "k3q_common.h"

namespace k3q {

// The eight nibbles of a dword of a strip-linear int4 copy (value 2t of a lane's k at bits [4t, 4t + 4), 2t + 1 at
// [16 + 4t, ...)) as bfloat16 pairs of what they stand for: w - zero, off = 8 + zero.  Every such integer is below 2^8
// and exact.  About twice the operations of a conversion that leaves an offset in the values, and nothing to take out of
// the sums afterwards.
__device__ __forceinline__ v4u plain_nibbles(const u32 d, float off) {
    const u32 u = d ^ 0x88888888u;
    u32 lo = u & 0x0F0F0F0Fu, hi = (u >> 4) & 0x0F0F0F0Fu;
    v4u out;
    // (hidden from the compiler, which would fetch every nibble on its own and subtract integers: a conversion of a byte
    // and a subtraction per value here, four operations there)
    asm("" : "+v"(off), "+v"(lo), "+v"(hi));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const u32 v = (t & 1) ? hi : lo;
        const float even = (float)((v >> (8 * (t >> 1))) & 0xffu) - off;
        const float odd = (float)((v >> (16 + 8 * (t >> 1))) & 0xffu) - off;
        out[t] = byte_perm(__float_as_uint(odd), __float_as_uint(even), 0x07060302u);
    }
    return out;
}

}  // namespace k3q
