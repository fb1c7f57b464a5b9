// The sum of a product's K slices.
#pragma once
#include "sq_common.h"

namespace sq {

// y[t, y_off + r] = row_scale[r] * sum over the slices (in their order, at most eight) of part[slice][t][r], four rows of one token
// per thread.  Latency is what it costs: all slices' loads are on their way at once (one after the other, eight slices of 77 x
// 3584 sums took 5.8 us, now 4.4), and four 16-bit results leave together where they may.
template <class Args>
__global__ __launch_bounds__(256) void slice_sum_kernel(Args a) {
    int pi = 0;
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    while (pi < a.n && i >= (int64_t)a.T * ((a.p[pi].m.R + 3) / 4)) i -= (int64_t)a.T * ((a.p[pi].m.R + 3) / 4), ++pi;
    if (pi >= a.n) return;
    const sq_matrix& m = a.p[pi].m;
    const int q = (m.R + 3) / 4, t = (int)(i / q), r = (int)(i - (int64_t)t * q) * 4;
    const float* p = a.p[pi].part + (int64_t)t * m.R + r;
    const int64_t step = (int64_t)a.T * m.R, o = (int64_t)t * a.ldy + m.y_off + r;
    float sc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) sc[e] = h2f(m.row_scale[min(r + e, m.R - 1)]);
    float4v v = {0.f, 0.f, 0.f, 0.f};
    if (m.R % 4 == 0) {
        float4v s[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) s[k] = *reinterpret_cast<const float4v*>(p + min(k, a.ks - 1) * step);
#pragma unroll
        for (int k = 0; k < 8; ++k) if (k < a.ks) v += s[k];
        if (a.y_dtype != SQ_F32 && ((o | (int64_t)((uintptr_t)a.y >> 1)) & 3) == 0) {
            *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(a.y) + o) =
                a.y_dtype == SQ_BF16 ? u32x2{f2bf_x2(v[0] * sc[0], v[1] * sc[1]), f2bf_x2(v[2] * sc[2], v[3] * sc[3])}
                                     : u32x2{f2h_x2(v[0] * sc[0], v[1] * sc[1]), f2h_x2(v[2] * sc[2], v[3] * sc[3])};
            return;
        }
    } else {
        for (int k = 0; k < a.ks; ++k)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += r + e < m.R ? p[k * step + e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (r + e < m.R) store_y(a.y, a.y_dtype, o + e, v[e] * sc[e]);
}

}  // namespace sq
