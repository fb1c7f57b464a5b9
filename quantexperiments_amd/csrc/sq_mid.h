// Codebook product for more activation rows than a decode step has: T = 33 .. 256 (384 for large d = 4 matrices), and more of them for
// matrices that are small enough.
//
// Decoding the matrix to fp16 first writes and reads eight times its bytes and then multiplies tiles of 256 rows; passes of 32
// rows through the decode-time kernel gather every codeword once per pass.  Here every codeword is gathered once for a block of up to 256
// rows, which are fewer where a launch would leave CUs idle otherwise: what a small product takes is the length of a workgroup's loop (512 x 512
// at 228 rows 15.7 us in four workgroups, 4.8 in 120; 896 x 896 with 16-bit tags 38 and 8).
// v_mfma_f32_16x16x32_f16 takes the weights as its A operand (lane l: row l % 16, 8 consecutive k), which are two d = 4
// codewords (LDS) or one d = 8 codeword (L2), so a lane gathers its operand straight into registers and uses it for all NT
// tiles of 16 activation rows; the activations are the B operand and come from LDS.
//
// Bound: d = 8 by the gathers up to about 128 rows (one L2 request each, 16 bytes used of the 64 that come: 178 G a second for
// 18944 x 2 x 3584 at 77 rows, which take 96 us; the matrix cores are busy 15 % of the time).  d = 4 by no pipe
// alone: with 12-bit tags at 128 rows the matrix cores are busy 47 % of a CU's time and LDS 51 % (every wave reads all the
// activations for its 32 weight rows; 29 % of it bank conflicts of the codeword reads), taking turns.  In passes of 32 rows or decoded
// first, at 33 / 77 / 128 / 256 rows: d = 8, 18944 x 2 x 3584: 172 / 205 / 205 / 209 us, here 86 / 91 / 103 / 188 (sq_plane_product.hip, which takes it up to 96 rows:
// 54 / 78; sq_fused.h: 103 at 256); 12-bit: 41 / 68 / 102 / 165, here 25 / 34 / 53 / 105 (sq_fused.h: 80).
//
//   workgroup   NW waves, two per SIMD or more so that one gathers while the other multiplies (4 waves: a third slower, and the choice
//               where they spread better or a CU takes several); each has TW tiles of 16 weight rows x NT x 16 activation rows
//               (accumulators TW x NT x 4 registers)
//   K           in rounds of 4 lane units (UK columns of tags each, as in sq_rows_mfma.h), rounds in stages of S matrix steps;
//               step j of lane group g is columns (4 round + g) UK + 8 j .. + 7
//   X           stages of NT x 16 rows x 4 x S x 16 bytes, double buffered in LDS; loaded to registers two stages ahead
//               (converted bf16 -> fp16 on the way to LDS), one barrier per stage
//   tags        two rounds ahead; codewords PD steps ahead (one from LDS, three from L2 where the steps are short)
//   grid        blocks of weight rows x blocks of activation rows x ks slices of the rounds; with ks > 1 fp32 partial sums, added by
//               slice_sum_kernel
//
// D = 0: weights already decoded to fp16 (column orders, formats whose rows are not whole lane units).  The A operand is loaded
// from there, up to seven steps ahead; step j of lane group g is columns 256 round + 32 j + 8 g .. + 7, so that the four lane groups
// of a row read 64 neighbouring bytes.
//
// WIDE: bf16 activations keep their range and bits, for matrices that come here decoded because the vector kernel, which multiplies in
// fp32, takes them four rows at a time.  A token's values go to LDS times a power of two chosen by the largest of its columns so far, 1 as long as
// that is an ordinary one (2^-4 .. 65,504), else what makes it 2^12 .. 2^13; where the power changes the sums so far follow, at the end
// they are divided by it.  Without branches, on whose account loads would be waited for (18944 x 3584, decode included, at 3 / 32 rows 71.4 / 74.7
// us without, 72.4 / 75.9 so, 79.5 / 82 with a branch around what ordinary values can do without).
//
// An X row of a stage is 4 S pieces of 16 bytes; piece c of row t sits at slot c ^ h(t), with h such that the 16 lanes of an
// LDS clock (rows 0-3, 12-15 of one lane group with rows 4-11 of the next, and so on) fall into 16 different groups of four
// banks.
#pragma once
#include <iterator>
#include <utility>
#include <type_traits>
#include "sq_rows_mfma.h"

namespace sq {

struct MidPiece {
    sq_matrix m;
    const void* w;               // D = 0: the decoded weights [R, C]; else the tile-major copy of the tags or NULL
    float* part;                 // ks > 1: fp32 [ks, T, R]
    int wg0;
};

struct MidArgs {
    MidPiece p[MID_PIECES];
    int n;
    const uint16_t* x;
    int64_t ldx;
    void* y;
    int64_t ldy;
    int T, x_dtype, y_dtype;
    int U, ks, tbs, table_bytes; // tbs: blocks of 16 NT activation rows
    int wide;                    // 1: bf16 activations keep their range (WIDE; decoded weights, up to 48 activation rows)
};

template <int S> __device__ __forceinline__ int mid_swizzle(int t) {
    const int b = ((t >> 2) ^ (t >> 3)) & 1;         // rows 4 .. 11
    if (S == 4) return (t & 1) | (b ^ 1) << 1 | ((t >> 1) & 1) << 2 | ((t >> 3) & 1) << 3;
    return b | ((t >> 1) & 1) << 1 | ((t >> 3) & 1) << 2;
}

constexpr int mid_stage_bytes(int NT, int S) { return NT * 16 * S * 64; }
constexpr int mid_x_bytes(int NT, int S, bool wide) { return 2 * (mid_stage_bytes(NT, S) + (wide ? NT * 64 : 0)); }     // (WIDE: the stages' powers behind)

template <int BITS, int D, int NT, int TW, int S, int NW, bool BF, bool WIDE = false>
__global__ __launch_bounds__(64 * NW, 2) void mid_kernel(MidArgs a) {
    constexpr bool DENSE = D == 0;
    constexpr int UD = DENSE ? 1 : unit_of<DENSE ? 16 : BITS>::UD, TPU = DENSE ? 1 : UD * 32 / (DENSE ? 1 : BITS);
    constexpr int SPR = DENSE ? 8 : TPU / (8 / (DENSE ? 1 : D)), UK = DENSE ? 8 : TPU * D, UPR = DENSE ? 4 * SPR : 4, NST = SPR / S;
    constexpr int GC = DENSE ? 8 : UK, JC = DENSE ? 32 : 8, UPS = DENSE ? 4 * S : 0;   // columns from lane group to group, from step to step; units per stage
    constexpr int ROWB = S * 64, STAGE = mid_stage_bytes(NT, S), NTH = 64 * NW, PCS = (NT * 64 * S + NTH - 1) / NTH;
    constexpr int PD = DENSE ? (NT * TW <= 16 ? 7 : 3) : D == 8 && NT * TW < 24 ? 3 : 1, XB = NT <= 8 ? 2 : 1;   // steps that codewords and activations are fetched ahead of
    static_assert(SPR % S == 0 && SPR % (PD + 1) == 0 && (NST == 1 || NST % 2 == 0), "steps per round");
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (D == 4 && (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem != 0u) return;   // (gathers count from LDS address 0)
    int pi = 0;
    while (pi + 1 < a.n && (int)blockIdx.x >= a.p[pi + 1].wg0) ++pi;
    const MidPiece& P = a.p[pi];
    const sq_matrix& m = P.m;
    int blk = (int)blockIdx.x - P.wg0, slice = 0, tok0 = 0;                          // blocks of weight rows, of activation rows in them, slices in those
    if (a.ks > 1) { const int w = blk; blk = (int)((uint32_t)w / (uint32_t)a.ks); slice = w - blk * a.ks; }
    if (a.tbs > 1) { const int w = blk; blk = (int)((uint32_t)w / (uint32_t)a.tbs); tok0 = (w - blk * a.tbs) * (16 * NT); }
    const int NR = (a.U + UPR - 1) / UPR, NP = (NR + 1) >> 1;                       // rounds, and pairs of them: slices are whole pairs
    const int r0 = 2 * (int)((uint32_t)(NP * slice) / (uint32_t)a.ks), r1 = min(NR, 2 * (int)((uint32_t)(NP * (slice + 1)) / (uint32_t)a.ks));
    unsigned char* xbuf = smem + a.table_bytes;

    // ---- this wave's tiles (tiles past the last row repeat the last one and are not stored)
    const int ntiles = (m.R + 15) >> 4, tile0 = (blk * NW + wave) * TW;
    // (byte offsets from a uniform base: one address register per load)
    const bool tiled = !DENSE && P.w;
    const uint32_t us = (tiled ? 16 * UD : UD) * 4;                          // bytes between two units of a row
    const char* tags = reinterpret_cast<const char*>(P.w ? P.w : m.tags);
    uint32_t to[TW], bo[TW];
#pragma unroll
    for (int i = 0; i < TW; ++i) {
        const int tile = min(tile0 + i, ntiles - 1), row = min(tile * 16 + li, m.R - 1);
        to[i] = DENSE ? (uint32_t)row * (uint32_t)m.C * 2u : tiled ? ((uint32_t)tile * (uint32_t)a.U * 16u + (uint32_t)li) * (UD * 4) : (uint32_t)row * (uint32_t)m.W * 4u;
        bo[i] = !DENSE && m.row_book ? (uint32_t)m.row_book[row] << (BITS + (D == 8 ? 4 : 3)) : 0u;
    }
    auto load_tags = [&](int round, dwords<UD>* t) {
        if (DENSE) return;
        const uint32_t u = (uint32_t)min(4 * round + lg, a.U - 1) * us;
#pragma unroll
        for (int i = 0; i < TW; ++i) t[i] = load_unit<UD>(reinterpret_cast<const uint32_t*>(tags + (to[i] + u)));
    };

    // ---- activations: thread's pieces q = tid + NTH k of a stage, row q / (4 S), piece q % (4 S) = lane group * S + step
    uint32_t xo[PCS], xl[PCS];
    int xg[PCS];
#pragma unroll
    for (int k = 0; k < PCS; ++k) {
        const int q = min(tid + NTH * k, NT * 64 * S - 1), t = q / (4 * S), c = q - t * (4 * S), g = c / S, j = c - g * S;
        xg[k] = DENSE ? j * 4 + g : g;
        xo[k] = ((uint32_t)min(tok0 + t, a.T - 1) * (uint32_t)a.ldx + (uint32_t)(g * GC + j * JC)) * 2u;
        xl[k] = (uint32_t)(t * ROWB + ((c ^ mid_swizzle<S>(t & 15)) << 4));
    }
    // columns past the row's end (the last round's missing units, rounds past the slice) are zeros; what is read in their
    // place is the row's last unit
    auto load_x = [&](u32x4* px, int round, int st) {
        int left = a.U - 1 - UPR * min(round, NR - 1) - st * UPS;            // the stage's last unit; D = 0: < 0 if it is past the row
        const char* base = reinterpret_cast<const char*>(a.x) + (int64_t)min(round, NR - 1) * (2 * UPR * UK) + st * (S * JC * 2);
        if (DENSE && left < 0) base += left * (2 * UK), left = 0;
#pragma unroll
        for (int k = 0; k < PCS; ++k) px[k] = *reinterpret_cast<const u32x4*>(base + (xo[k] - (uint32_t)(max(xg[k] - left, 0) * (UK * 2))));
    };
    static_assert(!WIDE || (BF && 4 * S == 16), "a token's pieces of a stage are those of a row of 16 lanes");
    int* xpow = reinterpret_cast<int*>(xbuf + 2 * STAGE);                    // [2][NT * 16]
    float top[PCS] = {};                                                     // WIDE: the largest magnitude of the piece's token so far
    auto store_x = [&](const u32x4* px, int buf, int round, int st) {
        const int units = round < r1 ? a.U - UPR * round - st * UPS : 0;
#pragma unroll
        for (int k = 0; k < PCS; ++k) {
            u32x4 v = px[k];
            if constexpr (WIDE) {
                float f[8], mag = 0.f;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (xg[k] >= units) v[e] = 0u;
                    f[2 * e] = bf2f((uint16_t)(v[e] & 0xFFFFu)); f[2 * e + 1] = bf2f((uint16_t)(v[e] >> 16));
                    mag = fmaxf(mag, fmaxf(fabsf(f[2 * e]), fabsf(f[2 * e + 1])));
                }
                mag = fmaxf(mag, row_rotated<8>(mag)); mag = fmaxf(mag, row_rotated<4>(mag));
                mag = fmaxf(mag, row_rotated<2>(mag)); mag = fmaxf(mag, row_rotated<1>(mag));
                top[k] = fmaxf(top[k], mag);
                const int exponent = (int)min(__builtin_bit_cast(uint32_t, top[k]) >> 23, 254u) - 127, power = exponent >= -4 && exponent <= 15 ? 0 : max(exponent - 12, -64);
                const float by = __builtin_bit_cast(float, (uint32_t)(127 - power) << 23);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = f2h_x2(f[2 * e] * by, f[2 * e + 1] * by);
                if ((tid & 15) == 0 && ((NT * 64 * S) % NTH == 0 || tid + NTH * k < NT * 64 * S)) xpow[buf * (NT * 16) + (tid + NTH * k) / 16] = power;
            } else if constexpr (BF) { v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w); }
            const uint32_t keep = xg[k] < units ? 0xFFFFFFFFu : 0u;
            v.x &= keep; v.y &= keep; v.z &= keep; v.w &= keep;
            if ((NT * 64 * S) % NTH == 0 || tid + NTH * k < NT * 64 * S) *reinterpret_cast<u32x4*>(xbuf + buf * STAGE + xl[k]) = v;
        }
    };
    const uint32_t xbase = (uint32_t)(li * ROWB + (((lg * S) ^ mid_swizzle<S>(li)) << 4));

    // ---- codewords of one step.  In units past the row's end, whose X is zeros, a codeword that is not finite would make NaN of them: from
    // memory these read zeros (an offset past the end of the buffer); from LDS the row's last unit again, as in sq_rows_mfma.h (a choice
    // per codeword costs 4 to 9 % at 33 to 128 rows, 18944 x 2 x 3584 with 12-bit tags).
    const __amdgpu_buffer_rsrc_t words = __builtin_amdgcn_make_buffer_rsrc((void*)(DENSE ? (const void*)tags : (const void*)m.table), 0,
                                                                           DENSE ? (uint32_t)m.R * (uint32_t)m.C * 2u : D == 8 ? (uint32_t)m.G << (BITS + 4) : 0u, 0x00027000);
    auto gather = [&](u32x4* f, const dwords<UD>* t, int round, int step) {
        const int col = round * (UPR * UK) + step * JC + lg * GC;
        const bool past = DENSE ? col >= m.C : 4 * round + lg >= a.U;
#pragma unroll
        for (int i = 0; i < TW; ++i) {
            if constexpr (D != 4) {
                const uint32_t at = DENSE ? to[i] + (uint32_t)col * 2u : (unit_tag<DENSE ? 16 : BITS, UD>(t[i], step) << 4) + bo[i];
                f[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(words, past ? 0xFFFFFFF0u : at, 0, 0));
            } else {
                const u32x2 lo = *(const mma_lds_u32x2*)(uintptr_t)unit_lds_offset<BITS, UD, 3>(t[i], step * 2, bo[i]);
                const u32x2 hi = *(const mma_lds_u32x2*)(uintptr_t)unit_lds_offset<BITS, UD, 3>(t[i], step * 2 + 1, bo[i]);
                f[i] = u32x4{lo.x, lo.y, hi.x, hi.y};
            }
        }
    };

    float4v acc[TW][NT];
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[i][n] = float4v{0.f, 0.f, 0.f, 0.f};
    int power[NT] = {};                                                      // WIDE: of this lane's activation rows
    auto times = [&](int n, int by) {
#pragma unroll
        for (int i = 0; i < TW; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][n][e] = __builtin_ldexpf(acc[i][n][e], by);
    };

    // Two of everything that is on its way: tags of this round and the next, activations of the next stage and the one after.
    // A pair's members swap by the parity of the round (the loop is unrolled twice), never by moving registers, which would
    // wait for the loads.
    dwords<UD> tag[2][TW];
    u32x4 px[2][PCS], wf[PD + 1][TW];
    load_tags(r0, tag[0]);
    load_x(px[0], r0, 0);
    load_tags(r0 + 1, tag[1]);
    load_x(px[1], NST > 1 ? r0 : r0 + 1, NST > 1 ? 1 : 0);
    if (D == 4) stage_table(m.table, a.table_bytes, smem);
    store_x(px[0], 0, r0, 0);
    __syncthreads();
#pragma unroll
    for (int s = 0; s < PD; ++s) gather(wf[s], tag[0], r0, s);
    auto do_round = [&](auto parity, int round) {
        constexpr int P = decltype(parity)::value;
#pragma unroll
        for (int st = 0; st < NST; ++st) {
            constexpr int B0 = NST == 1 ? P : 0;                             // LDS buffer and register set of the round's first stage
            const int q = (B0 + st) & 1;
            load_x(px[q], round + (st + 2) / NST, (st + 2) % NST);
            half8v xf[XB][NT];
            auto read_x = [&](half8v* f, int j) {
                const unsigned char* xs = xbuf + q * STAGE + (xbase ^ (uint32_t)(j << 4));
#pragma unroll
                for (int n = 0; n < NT; ++n) f[n] = *reinterpret_cast<const half8v*>(xs + n * (16 * ROWB));
            };
            int now[NT] = {};
            if constexpr (WIDE) {
#pragma unroll
                for (int n = 0; n < NT; ++n) now[n] = xpow[q * (NT * 16) + n * 16 + li];
            }
            if (XB == 2) read_x(xf[0], 0);
            if constexpr (WIDE) {
                bool same = true;
#pragma unroll
                for (int n = 0; n < NT; ++n) same = same && now[n] == power[n];
                if (__builtin_expect(!__all((int)same), 0)) {
#pragma unroll
                    for (int n = 0; n < NT; ++n) { times(n, power[n] - now[n]); power[n] = now[n]; }
                }
            }
#pragma unroll
            for (int j = 0; j < S; ++j) {
                const int s = st * S + j;
                __builtin_amdgcn_sched_barrier(0);
                if (s + PD < SPR) gather(wf[(s + PD) % (PD + 1)], tag[P], round, s + PD);
                else gather(wf[(s + PD) % (PD + 1)], tag[P ^ 1], round + 1, s + PD - SPR);
                if (s + PD == SPR - 1) load_tags(round + 2, tag[P]);         // this round's tags have all been used
                if (XB == 1) read_x(xf[0], j);
                else if (j + 1 < S) read_x(xf[(j + 1) & (XB - 1)], j + 1);
                // the next stage's activations, in the middle of this one, where the other wave of the SIMD multiplies
                if (j == S / 2 - 1) store_x(px[q ^ 1], q ^ 1, round + (st + 1) / NST, (st + 1) % NST);
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int i = 0; i < TW; ++i)
                        acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8v, wf[s % (PD + 1)][i]), xf[j & (XB - 1)][n], acc[i][n], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
        }
    };
    for (int round = r0; round < r1; round += 2) {                           // (a partner past the slice's end multiplies zeros)
        do_round(std::integral_constant<int, 0>{}, round);
        do_round(std::integral_constant<int, 1>{}, round + 1);
    }

    // ---- lane: activation row 16 n + li, weight rows 16 tile + 4 lg .. + 3
    if constexpr (WIDE) {
#pragma unroll
        for (int n = 0; n < NT; ++n) times(n, power[n]);
    }
    const bool vec = m.R % 4 == 0;
#pragma unroll
    for (int i = 0; i < TW; ++i) {
        const int r = (tile0 + i) * 16 + lg * 4;
        if (r >= m.R) continue;
        float sc[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[e] = h2f(m.row_scale[min(r + e, m.R - 1)]);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int t = tok0 + n * 16 + li;
            if (t >= a.T) continue;
            if (a.ks > 1) {
                float* o = P.part + ((int64_t)slice * a.T + t) * m.R + r;
                if (vec) {
                    *reinterpret_cast<float4v*>(o) = acc[i][n];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) if (r + e < m.R) o[e] = acc[i][n][e];
                }
                continue;
            }
            const int64_t o = (int64_t)t * a.ldy + m.y_off + r;
            if (a.y_dtype != SQ_F32 && r + 4 <= m.R && ((o | (int64_t)((uintptr_t)a.y >> 1)) & 3) == 0) {
                const float4v v = acc[i][n];
                *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(a.y) + o) =
                    a.y_dtype == SQ_BF16 ? u32x2{f2bf_x2(v[0] * sc[0], v[1] * sc[1]), f2bf_x2(v[2] * sc[2], v[3] * sc[3])}
                                         : u32x2{f2h_x2(v[0] * sc[0], v[1] * sc[1]), f2h_x2(v[2] * sc[2], v[3] * sc[3])};
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) if (r + e < m.R) store_y(a.y, a.y_dtype, o + e, acc[i][n][e] * sc[e]);
            }
        }
    }
}

template <int BITS, int D, int NT, int TW, int S, int NW, bool BF, bool WIDE = false>
int launch_mid_dtype(const MidArgs& a, int grid, hipStream_t s) {
    static bool raised = false;
    if (!raised) {
        (void)hipFuncSetAttribute((const void*)mid_kernel<BITS, D, NT, TW, S, NW, BF, WIDE>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
        raised = true;
    }
    hipLaunchKernelGGL((mid_kernel<BITS, D, NT, TW, S, NW, BF, WIDE>), dim3((unsigned)grid), dim3(64 * NW), (size_t)a.table_bytes + mid_x_bytes(NT, S, WIDE), s, a);
    return check_launch("sq_linear_gemm(mid)");
}

template <int BITS, int D, int NT, int TW, int S, int NW>
int launch_mid_as(const MidArgs& a, int grid, hipStream_t s) {
    if constexpr (D == 0 && NT <= 3 && TW == 1) {
        if (a.wide && a.x_dtype == SQ_BF16) return launch_mid_dtype<BITS, D, NT, TW, S, NW, true, true>(a, grid, s);
    }
    return a.x_dtype == SQ_BF16 ? launch_mid_dtype<BITS, D, NT, TW, S, NW, true>(a, grid, s) : launch_mid_dtype<BITS, D, NT, TW, S, NW, false>(a, grid, s);
}

// The variants there are, each a kernel per format and type of x: the plans of sq_mid.hip choose among them, the launch finds its kernel in the same list.
struct MidVariant { int8_t nt, tw, nw, st; };
inline constexpr MidVariant MID4[] = {{1, 1, 4, 4}, {2, 1, 4, 4}, {3, 1, 4, 4}, {4, 1, 4, 4}, {5, 1, 4, 4}, {1, 1, 8, 4}, {2, 1, 8, 4}, {3, 1, 8, 4}, {4, 1, 8, 4},
                                      {5, 1, 8, 4}, {8, 1, 8, 4}, {3, 2, 8, 4}, {4, 2, 8, 4}, {5, 2, 8, 4}, {8, 2, 8, 4}, {3, 1, 10, 4}, {3, 1, 12, 4}, {5, 1, 10, 4},
                                      {5, 1, 12, 4}, {5, 1, 8, 2}, {8, 1, 8, 2}, {5, 2, 8, 2}, {8, 2, 8, 2}};
inline constexpr MidVariant MID8[] = {{1, 1, 4, 4}, {2, 1, 4, 4}, {3, 1, 4, 4}, {4, 1, 4, 4}, {5, 1, 4, 4}, {3, 1, 8, 4}, {4, 1, 8, 4}, {5, 1, 8, 4}, {8, 1, 8, 4},
                                      {12, 1, 8, 2}, {16, 1, 8, 2}, {3, 1, 10, 4}, {3, 1, 12, 4}, {5, 1, 10, 4}, {5, 1, 12, 4}, {8, 1, 12, 4}, {12, 1, 12, 2}, {5, 2, 8, 4},
                                      {8, 2, 8, 4}, {12, 2, 8, 2}, {16, 2, 8, 2}};
inline constexpr MidVariant MID_DENSE[] = {{1, 1, 8, 4}, {3, 1, 8, 4}, {5, 1, 8, 4}, {8, 1, 8, 4}, {12, 1, 8, 2}, {16, 1, 8, 2}};
template <int D> constexpr const auto& mid_variants() {
    if constexpr (D == 4) return MID4;
    else if constexpr (D == 8) return MID8;
    else return MID_DENSE;
}

template <int BITS, int D, size_t... I>
int launch_mid_variant(std::index_sequence<I...>, const MidArgs& a, int nt, int tw, int st, int nw, int grid, hipStream_t s) {
    constexpr const auto& v = mid_variants<D>();
    int rc = SQ_EUNSUPPORTED;
    (void)((nt == v[I].nt && tw == v[I].tw && nw == v[I].nw && st == v[I].st && (rc = launch_mid_as<BITS, D, v[I].nt, v[I].tw, v[I].st, v[I].nw>(a, grid, s), true)) || ...);
    return rc;
}
template <int BITS, int D>
int launch_mid_format(const MidArgs& a, int nt, int tw, int st, int nw, int grid, hipStream_t s) {
    return launch_mid_variant<BITS, D>(std::make_index_sequence<std::size(mid_variants<D>())>(), a, nt, tw, st, nw, grid, s);
}

#define SQ_MID_FORMAT(BITS, D)                                                                                             \
    int launch_mid_b##BITS##d##D(const MidArgs& a, int nt, int tw, int st, int nw, int grid, hipStream_t s) {                     \
        return launch_mid_format<BITS, D>(a, nt, tw, st, nw, grid, s);                                                         \
    }

}  // namespace sq
