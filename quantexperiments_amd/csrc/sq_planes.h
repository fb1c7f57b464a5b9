// Columns ("planes") of a codebook of 65,536 codewords of width 8.
#pragma once
#include "sq_common.h"

namespace sq {

constexpr int PLANE = 65536;                 // codewords, and elements of a plane

// element e of eight chunks, chunk after chunk
__device__ __forceinline__ u32x4 plane_of(const u32x4 (&v)[8], int e) {
    u32x4 o;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        const uint32_t lo = v[2 * w][e / 2], hi = v[2 * w + 1][e / 2];
        o[w] = e & 1 ? (lo >> 16) | (hi & 0xFFFF0000u) : (lo & 0xFFFFu) | (hi << 16);
    }
    return o;
}

}  // namespace sq
