// The sum of a product's K slices.
#pragma once
#include <algorithm>
#include "sq_common.h"

namespace sq {

struct SlicePiece {
    const float* part;           // fp32 [ks, T, ld]
    const uint16_t* row_scale;
    int R, ld, y_off;
    uint32_t end;                // quads of this piece and those before it
};
struct SliceArgs {
    SlicePiece p[MID_PIECES];
    void* y;
    int64_t ldy;
    int n, T, ks, y_dtype;
};

// y[t, y_off + r] = row_scale[r] * sum over the slices (in their order) of part[slice][t][r], four rows of one token
// per thread.  Latency is what it costs: eight slices' loads are on their way at once (one after the other, eight slices of 77 x
// 3584 sums took 5.8 us, five of 8 x 3584 4.2), four 16-bit results leave together where they may, and a workgroup is one wave, so
// that the few of a decode step's sums spread over the chip.
static __global__ __launch_bounds__(64) void slice_sum_kernel(SliceArgs a) {
    uint32_t i = blockIdx.x * 64 + threadIdx.x, before = 0;
    int pi = 0;
    while (pi < a.n && i >= a.p[pi].end) before = a.p[pi++].end;
    if (pi >= a.n) return;
    const SlicePiece& m = a.p[pi];
    i -= before;
    const uint32_t q = (uint32_t)(m.R + 3) / 4, t = i / q;
    const int r = (int)(i - t * q) * 4;
    const float* p = m.part + (int64_t)t * m.ld + r;
    const int64_t step = (int64_t)a.T * m.ld, o = (int64_t)t * a.ldy + m.y_off + r;
    float sc[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) sc[e] = h2f(m.row_scale[min(r + e, m.R - 1)]);
    float4v v = {0.f, 0.f, 0.f, 0.f};
    if (m.ld % 4 == 0 && ((uintptr_t)m.part & 15) == 0) {
        for (int k0 = 0; k0 < a.ks; k0 += 8) {
            float4v s[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) s[k] = *reinterpret_cast<const float4v*>(p + min(k0 + k, a.ks - 1) * step);
#pragma unroll
            for (int k = 0; k < 8; ++k) if (k0 + k < a.ks) v += s[k];
        }
        if (a.y_dtype != SQ_F32 && r + 4 <= m.R && ((o | (int64_t)((uintptr_t)a.y >> 1)) & 3) == 0) {
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

// Pieces: {.m, .part}, n of them; whole_quads: rows of sums are whole quads of them, whatever R is
template <class Piece>
int launch_slice_sum(const Piece* pieces, int n, int ks, int T, void* y, int y_dtype, int64_t ldy, hipStream_t s, bool whole_quads = false) {
    SliceArgs a{};
    a.y = y; a.ldy = ldy; a.n = n; a.T = T; a.ks = ks; a.y_dtype = y_dtype;
    uint32_t quads = 0;
    for (int i = 0; i < n; ++i) {
        const sq_matrix& m = pieces[i].m;
        quads += (uint32_t)T * (uint32_t)((m.R + 3) / 4);
        a.p[i] = {pieces[i].part, m.row_scale, m.R, whole_quads ? (m.R + 3) / 4 * 4 : m.R, m.y_off, quads};
    }
    hipLaunchKernelGGL(slice_sum_kernel, dim3((quads + 63) / 64), dim3(64), 0, s, a);
    return check_launch("sum of K slices");
}

}  // namespace sq
