// Dense fp16 decode of 16-bit tags of width 8 for the tile GEMM, a column of the codebook ("plane") at a time.
//
// A whole codebook of 65,536 codewords is 1 MB: gathered a codeword at a time it comes out of L2, 64 bytes for 16.  One of its eight
// columns is 128 KB, which LDS holds.  A workgroup stages plane e and looks up element e of every tag of its rows; chunks that are
// neighbours in a row then have neighbouring results in plane order,
//     out[r, e * n + j] = table[tag[r, j]][e]        (n = C / 8 chunks)
// so stretches of C / 4 bytes leave, whole lines where C is a multiple of 512.  The activations are copied into the same order of columns and the product does not notice: its sum over
// columns is the same sum in another order.
#include <algorithm>
#include "sq_planes.h"

namespace sq {

constexpr int NT = 512, U = 8;               // planes_kernel's threads, and units of a thread in flight

// Rows of n chunks of 8 elements into plane order, 8 chunks (128 bytes in, a 16-byte piece of each plane out) per thread: the codebooks of
// the pieces as one row each, then the activations, which become fp16.
struct PlaneOrderArgs {
    const uint16_t* table[GEMM256_PIECES];
    uint16_t* planes;                        // 8 x PLANE per piece
    int pieces;
    const uint16_t* x;
    uint16_t* xout;
    int64_t ldx, units;                      // units of 64 elements of x (0: no copy)
    int C, bf16;
};

__global__ __launch_bounds__(256) void plane_order_kernel(PlaneOrderArgs a) {
    constexpr int PER = PLANE / 8;           // units of a codebook
    int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const uint16_t* src;
    uint16_t* dst;
    int n;
    bool convert = false;
    if (u < (int64_t)a.pieces * PER) {
        const int piece = (int)(u / PER), at = (int)(u - piece * PER);
        const uint16_t* table = a.table[0];
#pragma unroll
        for (int i = 1; i < GEMM256_PIECES; ++i) table = i == piece ? a.table[i] : table;
        src = table + (int64_t)at * 64;
        dst = a.planes + (int64_t)piece * 8 * PLANE + at * 8;
        n = PLANE;
    } else {
        u -= (int64_t)a.pieces * PER;
        if (u >= a.units) return;
        const int per_row = a.C / 64, t = (int)(u / per_row), at = (int)(u - (int64_t)t * per_row);
        src = a.x + (int64_t)t * a.ldx + at * 64;
        dst = a.xout + (int64_t)t * a.C + at * 8;
        n = a.C / 8;
        convert = a.bf16;
    }
    u32x4 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const u32x4*>(src + i * 8);
    if (convert) {
#pragma unroll
        for (int i = 0; i < 8; ++i) { v[i].x = bf2h_x2(v[i].x); v[i].y = bf2h_x2(v[i].y); v[i].z = bf2h_x2(v[i].z); v[i].w = bf2h_x2(v[i].w); }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) *reinterpret_cast<u32x4*>(dst + (int64_t)e * n) = plane_of(v, e);
}

struct PlanesArgs {
    const u32x4* tags[GEMM256_PIECES];
    uint16_t* out[GEMM256_PIECES];
    int rows[GEMM256_PIECES];
    int g0[GEMM256_PIECES + 1];              // first group of eight workgroups of each piece
    const uint16_t* planes;
    int n, C;
};

// A group of eight workgroups, one per plane, shares the tags of its rows; it sits on one XCD, whose L2 then reads them once.
// A thread has eight tags (16 bytes) in, eight look-ups and 16 bytes out per unit, U units at a time with the next U's tags on their way.
// 37888 x 3584 (272 MB written) takes 66 us, 27 without the stores: look-ups keep the LDS busy half of the time, 70 % of that bank conflicts, the stores
// reach 4.1 TB/s (kernels that write whole rows 5.5), and with one workgroup per CU the two take turns in part.  1024 threads with 4 units 76, with 8 69; 512 with 6 or 12 71 and 75.  Stores that bypass the caches take 52, but the product that reads them next then takes as much
// longer, and with small matrices more: 3584 x 3584 at 2048 rows 63 us in all and 73.
// A codeword at a time out of L2 (sq_dequant.hip) the decode takes 122 us: product of 2048 rows 514, now 474 with the 10 us of plane_order_kernel.
__global__ __launch_bounds__(NT) void planes_kernel(PlanesArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint16_t plane[];
    const int b = (int)blockIdx.x, tid = (int)threadIdx.x, slot = b >> 3, e = slot & 7, group = (slot >> 3) * 8 + (b & 7);
    int pi = 0;
#pragma unroll
    for (int i = 1; i < GEMM256_PIECES; ++i) pi += i < a.n && group >= a.g0[i];
    const int np = a.C / 64, per_row = a.C / 8;                  // units of eight chunks, and chunks, of a row
    const int total = a.rows[pi] * np, step = (a.g0[pi + 1] - a.g0[pi]) * NT, dr = step / np, dp = step - dr * np;
    const u32x4* tags = a.tags[pi];
    int u = (group - a.g0[pi]) * NT + tid, r = u / np, p = u - r * np;
    auto load = [&](int64_t at) { return tags[at < total ? at : total - 1]; };
    u32x4 t[U];
#pragma unroll
    for (int k = 0; k < U; ++k) t[k] = load((int64_t)u + (int64_t)k * step);
    const u32x4* src = reinterpret_cast<const u32x4*>(a.planes + ((int64_t)pi * 8 + e) * PLANE);
#pragma unroll
    for (int i = 0; i < PLANE / 8 / NT; ++i) reinterpret_cast<u32x4*>(plane)[i * NT + tid] = src[i * NT + tid];
    __syncthreads();
    uint16_t* out = a.out[pi] + e * per_row;
    auto look_up = [&](u32x4 tag) {
        u32x4 o;
#pragma unroll
        for (int w = 0; w < 4; ++w) o[w] = (uint32_t)plane[tag[w] & 0xFFFFu] | ((uint32_t)plane[tag[w] >> 16] << 16);
        return o;
    };
    auto place = [&]() {                                         // of the present unit; r and p move on
        uint16_t* at = out + (int64_t)r * a.C + p * 8;
        r += dr; p += dp;
        if (p >= np) { p -= np; ++r; }
        return at;
    };
    while ((int64_t)u + (U - 1) * (int64_t)step < total) {
        u32x4 next[U];
#pragma unroll
        for (int k = 0; k < U; ++k) next[k] = load((int64_t)u + (int64_t)(U + k) * step);
#pragma unroll
        for (int k = 0; k < U; ++k) *reinterpret_cast<u32x4*>(place()) = look_up(t[k]);
#pragma unroll
        for (int k = 0; k < U; ++k) t[k] = next[k];
        u += U * step;
    }
#pragma unroll
    for (int k = 0; k < U - 1; ++k) {
        if ((int64_t)u + (int64_t)k * step >= total) break;
        *reinterpret_cast<u32x4*>(place()) = look_up(t[k]);
    }
}

bool planes_ok(const sq_matrix* mats, int n) {
    if (n < 1 || n > GEMM256_PIECES || device_cus() < 64) return false;
    const int C = mats[0].C;
    for (int i = 0; i < n; ++i) {
        const sq_matrix& m = mats[i];
        if (!m.tags || m.R <= 0 || m.C != C || C % 64 || m.d != 8 || m.bits != 16 || m.G != 1 || m.row_book || m.perms || m.W != C / 16) return false;
        if (((uintptr_t)m.tags & 15) || ((uintptr_t)m.table & 15)) return false;
        if ((int64_t)m.R * (C / 64) >= (int64_t)1 << 30) return false;
    }
    return true;
}

size_t planes_bytes(int n) { return (size_t)n * 8 * PLANE * sizeof(uint16_t); }

// The pieces (planes_ok) one behind the other at out, rows of C, and x (bf16 or fp16, 16-byte aligned rows; NULL: no copy) as fp16
// [T, C] at xout, both in plane order; `planes`: planes_bytes(n) of workspace.
int launch_planes(const sq_matrix* mats, int n, uint16_t* out, uint16_t* planes, const void* x, int x_dtype, int64_t ldx, int T, uint16_t* xout,
                  hipStream_t s) {
    const int C = mats[0].C;
    PlaneOrderArgs o{};
    o.planes = planes; o.pieces = n; o.C = C; o.bf16 = x_dtype == SQ_BF16;
    o.x = (const uint16_t*)x; o.ldx = ldx; o.xout = xout; o.units = x ? (int64_t)T * (C / 64) : 0;
    PlanesArgs a{};
    a.planes = planes; a.n = n; a.C = C;
    int groups[GEMM256_PIECES];
    for (int i = 0; i < n; ++i) {
        o.table[i] = mats[i].table;
        a.tags[i] = (const u32x4*)mats[i].tags;
        a.out[i] = out;
        a.rows[i] = mats[i].R;
        out += (size_t)mats[i].R * C;
        groups[i] = 1;
    }
    // a CU has room for one workgroup; the groups, a multiple of eight so that one stays on its XCD, go to where the most rows per group are
    const int all = device_cus() / 64 * 8;
    for (int left = all - n; left > 0; --left) {
        int most = 0;
        for (int i = 1; i < n; ++i)
            if ((int64_t)a.rows[i] * groups[most] > (int64_t)a.rows[most] * groups[i]) most = i;
        ++groups[most];
    }
    for (int i = 0; i < n; ++i) a.g0[i + 1] = a.g0[i] + groups[i];
    for (int i = n; i < GEMM256_PIECES; ++i) a.g0[i + 1] = all;
    const int64_t wgs = ((int64_t)n * (PLANE / 8) + o.units + 255) / 256;
    if (wgs >= ((int64_t)1 << 31)) return fail(SQ_EINVAL, "sq_linear_gemm: %lld workgroups", (long long)wgs);
    hipLaunchKernelGGL(plane_order_kernel, dim3((unsigned)wgs), dim3(256), 0, s, o);
    if (const int rc = check_launch("sq_linear_gemm(plane order)")) return rc;
    static bool raised = false;
    if (!raised) {
        (void)hipFuncSetAttribute((const void*)planes_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, PLANE * 2);
        (void)hipGetLastError();
        raised = true;
    }
    hipLaunchKernelGGL(planes_kernel, dim3((unsigned)(all * 8)), dim3(NT), PLANE * 2, s, a);
    return check_launch("sq_linear_gemm(planes)");
}

}  // namespace sq

// For tests: the decode by itself.  planes: planes_bytes(n); out: the pieces' rows; SQ_EUNSUPPORTED where the pieces do not take it.
extern "C" __attribute__((visibility("default"))) int32_t sq_planes_for_tests(const sq_matrix* mats, int32_t n, void* out, void* planes, const void* x, int32_t x_dtype,
                                                                              int64_t ldx, int32_t T, void* xout, void* stream) {
    if (!sq::planes_ok(mats, n)) return SQ_EUNSUPPORTED;
    return sq::launch_planes(mats, n, (uint16_t*)out, (uint16_t*)planes, x, x_dtype, ldx, T, (uint16_t*)xout, (hipStream_t)stream);
}
