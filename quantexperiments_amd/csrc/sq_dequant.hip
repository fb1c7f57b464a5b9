// Dense decode of a packed codebook matrix: one thread per chunk.
//   out[r, perm[mask[r]][j*d + k]] = rn_T( f32(table[book[r]*K + tag[r, j]][k]) * f32(row_scale[r]) )
// The fp32 product of two fp16 values is exact, so T = fp32 reproduces the CPU decode bit
// for bit and T = fp16 / bf16 differ from it by exactly one round-to-nearest-even.
#include <algorithm>
#include "sq_stream.h"

namespace sq {

template <int DT, int D>   // D = 0: any chunk width (scalar path)
__global__ __launch_bounds__(256) void dequant_kernel(sq_matrix m, typename store_as<DT>::type* __restrict__ out,
                                                      int64_t ld_out, int r0, int r1, int raw) {
    typedef typename store_as<DT>::type T;
    const int d = D ? D : m.d;
    const int nch = m.C / d;
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (int64_t)(r1 - r0) * nch) return;
    const int rr = (int)(idx / nch), j = (int)(idx - (int64_t)rr * nch);
    const int r = r0 + rr;
    const uint32_t* row = reinterpret_cast<const uint32_t*>(m.tags) + (int64_t)r * m.W;
    uint32_t tag = tag_at(row, m.W, m.bits, j);
    if (m.row_book) tag += (uint32_t)m.row_book[r] << m.bits;
    const float s = raw ? 1.f : h2f(m.row_scale[r]);     // raw: unscaled codewords (exact in fp16)
    const uint16_t* cw = m.table + (int64_t)tag * d;
    T* o = out + (int64_t)rr * ld_out;
    // a perms array without row_mask is one matrix-wide column order
    const int32_t* pm = m.perms ? m.perms + (int64_t)(m.row_mask ? m.row_mask[r] : 0) * m.C : nullptr;
    if (D == 8 && !pm) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(cw);
        T t[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            t[2 * k] = store_as<DT>::cvt(h2f((uint16_t)(v[k] & 0xFFFFu)) * s);
            t[2 * k + 1] = store_as<DT>::cvt(h2f((uint16_t)(v[k] >> 16)) * s);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) o[j * 8 + k] = t[k];
        return;
    }
    if (D == 4 && !pm) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(cw);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            o[j * 4 + 2 * k] = store_as<DT>::cvt(h2f((uint16_t)(v[k] & 0xFFFFu)) * s);
            o[j * 4 + 2 * k + 1] = store_as<DT>::cvt(h2f((uint16_t)(v[k] >> 16)) * s);
        }
        return;
    }
    for (int k = 0; k < d; ++k) {
        const int c = j * d + k;
        o[pm ? pm[c] : c] = store_as<DT>::cvt(h2f(cw[k]) * s);
    }
}

// d = 8 without column orders: four chunks per thread, 256 chunks apart, so that a thread has four tag loads and then
// four 16-byte table gathers in flight instead of one (the decode is bound by the rate and latency of those gathers,
// which hit L2, not HBM).  Same arithmetic as dequant_kernel; `vec`: 16-byte aligned rows of a 16-bit type, stored
// as one 16-byte piece per chunk; raw fp16 output copies the codeword's bits.
template <int DT>
__device__ __forceinline__ void dequant8x4_block(const sq_matrix& m, typename store_as<DT>::type* __restrict__ out, int64_t ld_out,
                                                 int r0, int r1, int raw, int vec, int block) {
    typedef typename store_as<DT>::type T;
    const int nch = m.C / 8;
    const int total = (r1 - r0) * nch;                          // < 2^31, checked by the launcher
    const int base = block * 1024 + (int)threadIdx.x;
    int rr[4], j[4];
    bool ok[4];
    uint32_t tag[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        int idx = base + k * 256;
        ok[k] = idx < total;
        idx = min(idx, total - 1);
        rr[k] = idx / nch;
        j[k] = idx - rr[k] * nch;
        const uint32_t* row = reinterpret_cast<const uint32_t*>(m.tags) + (int64_t)(r0 + rr[k]) * m.W;
        tag[k] = tag_at(row, m.W, m.bits, j[k]);
    }
    if (m.row_book) {
#pragma unroll
        for (int k = 0; k < 4; ++k) tag[k] += (uint32_t)m.row_book[r0 + rr[k]] << m.bits;
    }
    u32x4 cw[4];
    float s[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        cw[k] = *reinterpret_cast<const u32x4*>(m.table + (int64_t)tag[k] * 8);
        s[k] = raw ? 1.f : h2f(m.row_scale[r0 + rr[k]]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (!ok[k]) continue;
        T* o = out + (int64_t)rr[k] * ld_out + j[k] * 8;
        if (DT == SQ_F16 && raw && vec) {
            *reinterpret_cast<u32x4*>(o) = cw[k];
            continue;
        }
        T t[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            t[2 * e] = store_as<DT>::cvt(h2f((uint16_t)(cw[k][e] & 0xFFFFu)) * s[k]);
            t[2 * e + 1] = store_as<DT>::cvt(h2f((uint16_t)(cw[k][e] >> 16)) * s[k]);
        }
        if (DT != SQ_F32 && vec) {
            u32x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (uint32_t)t[2 * e] | ((uint32_t)t[2 * e + 1] << 16);
            *reinterpret_cast<u32x4*>(o) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = t[e];
        }
    }
}

template <int DT>
__global__ __launch_bounds__(256) void dequant8x4_kernel(sq_matrix m, typename store_as<DT>::type* __restrict__ out,
                                                         int64_t ld_out, int r0, int r1, int raw, int vec) {
    dequant8x4_block<DT>(m, out, ld_out, r0, r1, raw, vec, (int)blockIdx.x);
}

// The raw fp16 decode of a whole matrix and the fp16 copy of a bf16 activation matrix in one launch: the decode is
// bound by table gathers out of L2, the copy by HBM, so the copy's `nc` workgroups (8 elements per thread) are dealt
// evenly among the decode's `nd` and the two overlap instead of running one after the other.
__global__ __launch_bounds__(256) void dequant8x4_cvt_kernel(sq_matrix m, uint16_t* __restrict__ out, int64_t ld_out,
                                                             const uint16_t* __restrict__ x, int64_t ldx, int T, int C,
                                                             uint16_t* __restrict__ xout, int nd, int nc) {
    const int64_t b = blockIdx.x, total = (int64_t)nd + nc;
    const int cb = (int)(b * nc / total);                       // copy workgroups before this one
    if ((int)((b + 1) * nc / total) == cb) {
        dequant8x4_block<SQ_F16>(m, out, ld_out, 0, m.R, 1, 1, (int)b - cb);
        return;
    }
    const int64_t i = ((int64_t)cb * 256 + threadIdx.x) * 8;
    if (i >= (int64_t)T * C) return;
    const int t = (int)(i / C), c = (int)(i - (int64_t)t * C);
    u32x4 v = *reinterpret_cast<const u32x4*>(x + (int64_t)t * ldx + c);
    v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w);
    *reinterpret_cast<u32x4*>(xout + i) = v;
}

// d = 4 without column orders, codebooks that fit LDS: persistent workgroups stage their piece's codebook in LDS and decode two
// neighbouring chunks per lane and step, 16 bytes of 16-bit output (32 of fp32) stored in whole 16-byte pieces, so a wave
// writes 1 KB of consecutive bytes per instruction.  Four steps are in flight per thread: tags of all four, then the gathers,
// then the stores.  What bounds it is the write of the dense copy (37888 x 3584 with the copy of 1024 activation rows: 279 MB written
// and 64 read in 62 us, 5.5 TB/s, what a large copy reaches; LDS is busy 12 % of the time).  One thread per chunk with 2-byte stores
// and its codeword gathered from L2 took 75 us for 18944 x 3584 (136 MB written), this takes 31.  Up to GEMM256_PIECES stacked pieces share a
// launch (each gets workgroups by its rows), and a bf16 activation matrix that the product needs as fp16 rides along.
struct Dequant4Args {
    sq_matrix m[GEMM256_PIECES];
    void* out[GEMM256_PIECES];
    int wg0[GEMM256_PIECES + 1];             // first workgroup of each piece; behind the last piece's: workgroups of the copy
    int n, r0, raw;                          // r0: first row of the (single) piece that is decoded, its rows end at m.R
    int64_t ld_out;
    const uint16_t* x;                       // bf16 [T, C] -> xout fp16 (NULL: no copy)
    uint16_t* xout;
    int64_t ldx;
    int T, C;
};

template <int DT, int NT>
__global__ __launch_bounds__(NT) void dequant4_lds_kernel(Dequant4Args a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char dequant4_lds[];
    const int wg = (int)blockIdx.x, tid = (int)threadIdx.x;
    if (wg >= a.wg0[a.n]) {                  // fp16 copy of the activations, 8 elements per thread and step
        const int64_t total = (int64_t)a.T * a.C / 8, step = (int64_t)(gridDim.x - a.wg0[a.n]) * NT;
        for (int64_t i = (int64_t)(wg - a.wg0[a.n]) * NT + tid; i < total; i += step) {
            const int t = (int)(i * 8 / a.C), c = (int)(i * 8 - (int64_t)t * a.C);
            u32x4 v = *reinterpret_cast<const u32x4*>(a.x + (int64_t)t * a.ldx + c);
            v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w);
            *reinterpret_cast<u32x4*>(a.xout + i * 8) = v;
        }
        return;
    }
    int pi = 0;
#pragma unroll
    for (int i = 1; i < GEMM256_PIECES; ++i) pi += i < a.n && wg >= a.wg0[i];
    const sq_matrix& m = a.m[pi];
    const int tab16 = (m.G << m.bits) / 2;                      // 16-byte pieces of the codebook
    for (int i = tid; i < tab16; i += NT)
        reinterpret_cast<u32x4*>(dequant4_lds)[i] = reinterpret_cast<const u32x4*>(m.table)[i];
    __syncthreads();
    const int np = m.C / 8, rows = m.R - a.r0;                  // chunk pairs per row
    const int nwg = a.wg0[pi + 1] - a.wg0[pi], step = nwg * NT, dr = step / np, dp = step - dr * np;
    const int first = (wg - a.wg0[pi]) * NT + tid;
    int r = first / np, p = first - r * np;
    const uint32_t mask = (1u << m.bits) - 1u;
    typedef typename store_as<DT>::type OT;
    OT* out = reinterpret_cast<OT*>(a.out[pi]);
    while (r < rows) {
        int rr[4], pp[4];
        uint64_t w[4];
        uint32_t book[4];
        float sc[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            rr[k] = r; pp[k] = p;
            const int rc = min(r, rows - 1) + a.r0, pos = p * 2 * m.bits, at = pos >> 5;
            const uint32_t* row = reinterpret_cast<const uint32_t*>(m.tags) + (int64_t)rc * m.W;
            w[k] = (((uint64_t)row[min(at + 1, m.W - 1)] << 32) | row[at]) >> (pos & 31);
            book[k] = m.row_book ? (uint32_t)m.row_book[rc] << m.bits : 0u;
            sc[k] = a.raw ? 1.f : h2f(m.row_scale[rc]);
            r += dr; p += dp;
            if (p >= np) { p -= np; ++r; }
        }
        u32x2 c[4][2];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            c[k][0] = *reinterpret_cast<const u32x2*>(dequant4_lds + (size_t)(((uint32_t)w[k] & mask) + book[k]) * 8);
            c[k][1] = *reinterpret_cast<const u32x2*>(dequant4_lds + (size_t)(((uint32_t)(w[k] >> m.bits) & mask) + book[k]) * 8);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (rr[k] >= rows) continue;
            OT* o = out + (int64_t)rr[k] * a.ld_out + pp[k] * 8;
            if (DT == SQ_F16 && a.raw) {
                *reinterpret_cast<u32x4*>(o) = u32x4{c[k][0].x, c[k][0].y, c[k][1].x, c[k][1].y};
                continue;
            }
            float v[8];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t d = c[k][e >> 1][e & 1];
                v[2 * e] = h2f((uint16_t)(d & 0xFFFFu)) * sc[k];
                v[2 * e + 1] = h2f((uint16_t)(d >> 16)) * sc[k];
            }
            if constexpr (DT == SQ_F32) {
                *reinterpret_cast<float4v*>(o) = float4v{v[0], v[1], v[2], v[3]};
                *reinterpret_cast<float4v*>(o + 4) = float4v{v[4], v[5], v[6], v[7]};
            } else if constexpr (DT == SQ_F16) {
                *reinterpret_cast<u32x4*>(o) = u32x4{f2h_x2(v[0], v[1]), f2h_x2(v[2], v[3]), f2h_x2(v[4], v[5]), f2h_x2(v[6], v[7])};
            } else {
                *reinterpret_cast<u32x4*>(o) = u32x4{f2bf_x2(v[0], v[1]), f2bf_x2(v[2], v[3]), f2bf_x2(v[4], v[5]), f2bf_x2(v[6], v[7])};
            }
        }
    }
}

static bool dequant4_ok(const sq_matrix& m, const void* out, int64_t ld_out, int esize) {
    return m.tags && m.d == 4 && !m.perms && m.C % 8 == 0 && ((int64_t)m.G << m.bits) >= 2 && ((int64_t)m.G << m.bits) * 8 <= 128 * 1024 &&
           ((uintptr_t)m.table & 15) == 0 && ((uintptr_t)out & 15) == 0 && ld_out * esize % 16 == 0 && (int64_t)m.R * (m.C / 8) < ((int64_t)1 << 30);
}

// a.m, a.out, a.n, a.r0, a.raw, a.ld_out and the copy are set; the workgroups are dealt here: enough for two codebooks of 64 KB
// or four of 32 KB per CU, one of 1024 threads where a codebook fills LDS.
template <int DT>
static int launch_dequant4(Dequant4Args& a, hipStream_t s) {
    size_t tab = 0;
    int64_t pairs = 0;
    for (int i = 0; i < a.n; ++i) {
        tab = std::max(tab, (size_t)((int64_t)a.m[i].G << a.m[i].bits) * 8);
        pairs += (int64_t)(a.m[i].R - a.r0) * (a.m[i].C / 8);
    }
    const bool large = tab > 64 * 1024;
    const int nt = large ? 1024 : 512, per_cu = large ? 1 : (int)std::min<size_t>(4, 160 * 1024 / std::max<size_t>(tab, 1));
    const int slots = device_cus() * per_cu;
    int wg = 0;
    for (int i = 0; i < a.n; ++i) {
        const int64_t mine = (int64_t)(a.m[i].R - a.r0) * (a.m[i].C / 8);
        const int64_t most = (mine + 4 * nt - 1) / (4 * nt);     // four pairs per thread at least
        a.wg0[i] = wg;
        wg += (int)std::max<int64_t>(1, std::min<int64_t>(most, slots * mine / std::max<int64_t>(pairs, 1)));
    }
    for (int i = a.n; i <= GEMM256_PIECES; ++i) a.wg0[i] = wg;
    if (a.x) wg += (int)std::min<int64_t>(slots, ((int64_t)a.T * a.C / 8 + nt - 1) / nt);
    if (large) {
        static bool raised = false;
        if (!raised) {
            (void)hipFuncSetAttribute((const void*)dequant4_lds_kernel<DT, 1024>, hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024);
            (void)hipGetLastError();
            raised = true;
        }
        hipLaunchKernelGGL((dequant4_lds_kernel<DT, 1024>), dim3((unsigned)wg), dim3(1024), tab, s, a);
    } else {
        hipLaunchKernelGGL((dequant4_lds_kernel<DT, 512>), dim3((unsigned)wg), dim3(512), tab, s, a);
    }
    return check_launch("sq_dequant");
}

// Matrices with column orders: scattering 2-byte values straight to HBM costs 4x the plain decode, so a workgroup decodes RB rows
// into LDS at their permuted positions (ds_write of one element each) and then writes them out in 16-byte pieces.
// What bounds it is L2: a gathered codeword moves 64 bytes, the order 32 per chunk of eight, 13.5 TB/s reach the CUs.  The rows of a
// workgroup are neighbours in the file's row_order (rows sorted by order), so a thread reads the positions of its chunk once for
// all of them and again only where the order changes.
// Stacked pieces share a launch, with the fp16 copy of a bf16 activation matrix behind them: 5120, 1024 and 1024 rows of 5120 with
// 16-bit tags and the copy of 1024 activation rows take 35 us; in a launch each 25 + 9 + 9 + 13.
struct OrdersArgs {
    sq_matrix m[GEMM256_PIECES];
    void* out[GEMM256_PIECES];
    int wg0[GEMM256_PIECES + 1];             // first workgroup of each piece; behind the last piece's: workgroups of the copy
    int n, r0, raw, vec_out;                 // r0: first row of the (single) piece that is decoded, its rows end at m.R
    int64_t ld_out;
    const uint16_t* x;                       // bf16 [T, C] -> xout fp16 (NULL: no copy)
    uint16_t* xout;
    int64_t ldx;
    int T, C;
};

template <int DT, int D, int RB>   // D = 8 or 4; RB = 2 or 1
__global__ __launch_bounds__(512) void dequant_orders_kernel(OrdersArgs a) {
    typedef typename store_as<DT>::type T;
    extern __shared__ __attribute__((aligned(16))) unsigned char row_smem[];
    T* row_lds = reinterpret_cast<T*>(row_smem);
    const int wg = (int)blockIdx.x, tid = (int)threadIdx.x, nt = (int)blockDim.x;
    if (wg >= a.wg0[a.n]) {
        const int64_t total = (int64_t)a.T * a.C / 8, step = (int64_t)(gridDim.x - a.wg0[a.n]) * nt;
        for (int64_t i = (int64_t)(wg - a.wg0[a.n]) * nt + tid; i < total; i += step) {
            const int t = (int)(i * 8 / a.C), c = (int)(i * 8 - (int64_t)t * a.C);
            u32x4 v = *reinterpret_cast<const u32x4*>(a.x + (int64_t)t * a.ldx + c);
            v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w);
            *reinterpret_cast<u32x4*>(a.xout + i * 8) = v;
        }
        return;
    }
    int pi = 0;
#pragma unroll
    for (int i = 1; i < GEMM256_PIECES; ++i) pi += i < a.n && wg >= a.wg0[i];
    const sq_matrix& m = a.m[pi];
    const int C = m.C, nch = C / D, k0 = a.r0 + (wg - a.wg0[pi]) * RB, cnt = min(RB, m.R - k0);
    int r[RB], mask[RB];
    uint32_t boff[RB];
    float sc[RB];
#pragma unroll
    for (int q = 0; q < RB; ++q) {
        const int k = k0 + min(q, cnt - 1);
        r[q] = m.row_order ? m.row_order[k] : k;
        mask[q] = m.row_mask ? m.row_mask[r[q]] : 0;
        boff[q] = m.row_book ? (uint32_t)m.row_book[r[q]] << m.bits : 0u;
        sc[q] = a.raw ? 1.f : h2f(m.row_scale[r[q]]);
    }
    constexpr int V = 16 / (int)sizeof(T);                      // elements per 16-byte store
    for (int j = tid; j < nch; j += nt) {
        uint32_t tag[RB], v[RB][D / 2];
        int32_t p[D];
        auto order = [&](int q) {
            const int32_t* pm = m.perms + (int64_t)mask[q] * C + j * D;
#pragma unroll
            for (int h = 0; h < D / 4; ++h) {
                const u32x4 t = *reinterpret_cast<const u32x4*>(pm + h * 4);
#pragma unroll
                for (int k = 0; k < 4; ++k) p[h * 4 + k] = (int32_t)t[k];
            }
        };
#pragma unroll
        for (int q = 0; q < RB; ++q)
            tag[q] = tag_at(reinterpret_cast<const uint32_t*>(m.tags) + (int64_t)r[q] * m.W, m.W, m.bits, j) + boff[q];
        order(0);
#pragma unroll
        for (int q = 0; q < RB; ++q) {
            const uint16_t* cw = m.table + (int64_t)tag[q] * D;
            if constexpr (D == 8) {
                const u32x4 t = *reinterpret_cast<const u32x4*>(cw);
                v[q][0] = t[0]; v[q][1] = t[1]; v[q][2] = t[2]; v[q][3] = t[3];
            } else {
                const u32x2 t = *reinterpret_cast<const u32x2*>(cw);
                v[q][0] = t[0]; v[q][1] = t[1];
            }
        }
#pragma unroll
        for (int q = 0; q < RB; ++q) {
            if (q && mask[q] != mask[q - 1]) order(q);
            T* row = row_lds + (size_t)q * C;
#pragma unroll
            for (int k = 0; k < D / 2; ++k) {
                row[p[2 * k]] = store_as<DT>::cvt(h2f((uint16_t)(v[q][k] & 0xFFFFu)) * sc[q]);
                row[p[2 * k + 1]] = store_as<DT>::cvt(h2f((uint16_t)(v[q][k] >> 16)) * sc[q]);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < RB; ++q) {
        if (q >= cnt) break;
        T* o = reinterpret_cast<T*>(a.out[pi]) + (int64_t)(r[q] - a.r0) * a.ld_out;
        const T* row = row_lds + (size_t)q * C;
        if (a.vec_out) {
            for (int c = tid * V; c < C; c += nt * V) *reinterpret_cast<u32x4*>(o + c) = *reinterpret_cast<const u32x4*>(row + c);
        } else {
            for (int c = tid; c < C; c += nt) o[c] = row[c];
        }
    }
}

static bool orders_ok(const sq_matrix& m, size_t esize) {
    return m.tags && m.perms && (m.d == 8 || m.d == 4) && (size_t)m.C * esize <= 65536 && ((uintptr_t)m.perms & 15) == 0 &&
           ((uintptr_t)m.table & 15) == 0 && m.C % 4 == 0;
}

// a.m (one d, one C), a.out, a.n, a.r0, a.raw, a.ld_out, a.vec_out and the copy are set.
// Two rows per workgroup where they are short and many (us with two rows, with one; 16-bit tags and output): 7168 x 5120 31.6, 33.3;
// 2048 x 5120 12.3, 13.1; 512 x 5120 5.9, 5.3 (two workgroups on a CU hide less); 4096 x 8192 29.4, 29.8; 4096 x 12288 43.5, 42.2;
// 3584 x 18944 75, 60 (two workgroups' LDS fill a CU); and with rows in no order 35.8, 35.6 at 4096 x 10240.  Four rows: 33.3 at 7168 x 5120.
template <int DT>
static int launch_orders(OrdersArgs& a, hipStream_t s) {
    const int C = a.m[0].C, nch = C / a.m[0].d;
    const size_t row_bytes = (size_t)C * sizeof(typename store_as<DT>::type);
    // threads: as few rounds of at most 320 as the chunks need, all rounds nearly full
    const int rounds = (nch + 319) / 320, nt = std::max(64, ((nch + rounds - 1) / rounds + 63) & ~63);
    int64_t rows = 0, wg = 0;
    for (int i = 0; i < a.n; ++i) rows += a.m[i].R - a.r0;
    const int rb = a.m[0].row_order && row_bytes <= 16384 && rows >= 8 * device_cus() ? 2 : 1;
    for (int i = 0; i < a.n; ++i) {
        a.wg0[i] = (int)wg;
        wg += (a.m[i].R - a.r0 + rb - 1) / rb;
    }
    for (int i = a.n; i <= GEMM256_PIECES; ++i) a.wg0[i] = (int)wg;
    if (a.x) wg += std::min<int64_t>(device_cus() * 4, ((int64_t)a.T * a.C / 8 + nt - 1) / nt);
    if (wg >= ((int64_t)1 << 31)) return fail(SQ_EINVAL, "sq_dequant: %lld workgroups", (long long)wg);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)wg), dim3((unsigned)nt), row_bytes * rb, s, a); };
    if (a.m[0].d == 8) { if (rb > 1) go(dequant_orders_kernel<DT, 8, 2>); else go(dequant_orders_kernel<DT, 8, 1>); }
    else { if (rb > 1) go(dequant_orders_kernel<DT, 4, 2>); else go(dequant_orders_kernel<DT, 4, 1>); }
    return check_launch("sq_dequant");
}

static bool dequant8x4_ok(const sq_matrix& m, int64_t n) {
    return m.d == 8 && !m.perms && n > 0 && n < ((int64_t)1 << 31) - 1024 && ((uintptr_t)m.table & 15) == 0;
}

template <int DT>
static int launch_dt(const sq_matrix& m, void* out, int64_t ld_out, int r0, int r1, hipStream_t s, int raw) {
    typedef typename store_as<DT>::type T;
    const int64_t n = (int64_t)(r1 - r0) * (m.C / m.d);
    if (n == 0) return SQ_OK;
    if (orders_ok(m, sizeof(T))) {
        constexpr int V = 16 / (int)sizeof(T);
        OrdersArgs a{};
        a.m[0] = m; a.m[0].R = r1; a.out[0] = out; a.n = 1; a.r0 = r0; a.raw = raw; a.ld_out = ld_out;
        if (r0 > 0 || r1 < m.R) a.m[0].row_order = nullptr;     // part of the rows: taken as they lie
        a.vec_out = ((uintptr_t)out & 15) == 0 && ld_out % V == 0 && m.C % V == 0;
        return launch_orders<DT>(a, s);
    }
    if (dequant8x4_ok(m, n)) {
        const int vec = sizeof(T) == 2 && ((uintptr_t)out & 15) == 0 && ld_out % 8 == 0;
        hipLaunchKernelGGL((dequant8x4_kernel<DT>), dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, s, m, (T*)out, ld_out, r0, r1, raw, vec);
        return check_launch("sq_dequant");
    }
    if (dequant4_ok(m, out, ld_out, (int)sizeof(T))) {
        Dequant4Args a{};
        a.m[0] = m; a.m[0].R = r1; a.out[0] = out; a.n = 1; a.r0 = r0; a.raw = raw; a.ld_out = ld_out;
        return launch_dequant4<DT>(a, s);
    }
    const unsigned grid = (unsigned)((n + 255) / 256);
    if (m.d == 8) hipLaunchKernelGGL((dequant_kernel<DT, 8>), dim3(grid), dim3(256), 0, s, m, (T*)out, ld_out, r0, r1, raw);
    else if (m.d == 4) hipLaunchKernelGGL((dequant_kernel<DT, 4>), dim3(grid), dim3(256), 0, s, m, (T*)out, ld_out, r0, r1, raw);
    else hipLaunchKernelGGL((dequant_kernel<DT, 0>), dim3(grid), dim3(256), 0, s, m, (T*)out, ld_out, r0, r1, raw);
    return check_launch("sq_dequant");
}

// Raw fp16 decode of every row of `m` into out[r * ld_out + c] together with the fp16 copy of the bf16 matrix x
// [T, C] (row stride ldx, 16-byte aligned rows, C % 8 == 0) into xout [T, C].  Returns 1 without launching
// anything when the matrix does not take the four-chunk kernel; the caller then launches the two steps itself.
int launch_dequant_with_cvt(const sq_matrix& m, void* out, int64_t ld_out, const uint16_t* x, int64_t ldx, int T, int C,
                            uint16_t* xout, hipStream_t s) {
    const int64_t n = (int64_t)m.R * (m.C / (m.d ? m.d : 1)), ne = (int64_t)T * C;
    if (!m.tags || !dequant8x4_ok(m, n) || ((uintptr_t)out & 15) || ld_out % 8 || ne <= 0 || ne >= ((int64_t)1 << 40)) return 1;
    const int64_t nd = (n + 1023) / 1024, nc = (ne / 8 + 255) / 256;
    if (nd + nc >= ((int64_t)1 << 31)) return 1;
    hipLaunchKernelGGL(dequant8x4_cvt_kernel, dim3((unsigned)(nd + nc)), dim3(256), 0, s, m, (uint16_t*)out, ld_out, x, ldx, T, C, xout,
                       (int)nd, (int)nc);
    return check_launch("sq_linear_gemm(decode + fp16 copy)");
}

// fp16 decode (raw: without the row scales) of up to GEMM256_PIECES pieces, one behind the other at out (rows of C elements), with
// the fp16 copy of x as above (x NULL: none).  Returns 1 without launching anything when the pieces do not all take one of the two
// LDS kernels.
int launch_dequant_stack(const sq_matrix* mats, int n, void* out, int raw, const uint16_t* x, int64_t ldx, int T, int C, uint16_t* xout, hipStream_t s) {
    if (n < 1 || n > GEMM256_PIECES || ((uintptr_t)out & 15) || C % 8) return 1;
    auto fill = [&](auto& a, auto ok) -> bool {
        uint16_t* o = (uint16_t*)out;
        for (int i = 0; i < n; ++i) {
            if (mats[i].R <= 0 || !ok(mats[i], o)) return false;
            a.m[i] = mats[i];
            a.out[i] = o;
            o += (size_t)mats[i].R * C;
        }
        a.n = n; a.raw = raw; a.ld_out = C; a.x = x; a.xout = xout; a.ldx = ldx; a.T = T; a.C = C;
        return true;
    };
    if (mats[0].perms) {
        OrdersArgs a{};
        if (!fill(a, [&](const sq_matrix& m, uint16_t*) { return orders_ok(m, 2) && m.d == mats[0].d; })) return 1;
        a.vec_out = 1;
        return launch_orders<SQ_F16>(a, s);
    }
    Dequant4Args a{};
    if (!fill(a, [&](const sq_matrix& m, uint16_t* o) { return dequant4_ok(m, o, C, 2); })) return 1;
    return launch_dequant4<SQ_F16>(a, s);
}

int launch_dequant(const sq_matrix& m, void* out, int out_dtype, int64_t ld_out, int r0, int r1, hipStream_t s, bool raw) {
    if (!m.tags) return launch_stream_dequant(m, out, out_dtype, ld_out, r0, r1, s, raw);    // one-copy residency
    switch (out_dtype) {
        case SQ_F32: return launch_dt<SQ_F32>(m, out, ld_out, r0, r1, s, raw ? 1 : 0);
        case SQ_F16: return launch_dt<SQ_F16>(m, out, ld_out, r0, r1, s, raw ? 1 : 0);
        case SQ_BF16: return launch_dt<SQ_BF16>(m, out, ld_out, r0, r1, s, raw ? 1 : 0);
    }
    return fail(SQ_EINVAL, "sq_dequant: out_dtype %d", out_dtype);
}

}  // namespace sq
