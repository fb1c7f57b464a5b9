// Codebook product for more activation rows than a few tiles and fewer than a long prefill (129 .. 768): tiles of up to 384 tokens x
// 160 weight rows whose weights are gathered from the codebook on their way into LDS, so that no decoded copy of the matrix goes
// through memory (its write and the gathers do not overlap: a 16-bit decode of 18944 x 3584 takes 42 us without its stores, 31
// without its gathers, 66 with both).
//
//   workgroup   8 waves, 4 token quarters x 2 row halves, two per SIMD; a wave has NW tiles of 16 tokens x TW of 16 weight rows of
//               v_mfma_f32_16x16x32_f16 accumulators (weights are the A operand: lane l row l % 16, 8 consecutive k)
//   K           rounds of four lane units, as in sq_rows_mfma.h; stages of S steps of 32 columns, NB stages in LDS
//   weights     a fragment (16 rows x 32 columns) is 1 KB in the order of the lanes that will hold it, written and read without bank
//               conflicts.  d = 8: one global_load_lds per fragment with a codeword's address per lane.  d = 4: two ds_read_b64
//               from the codebook in LDS and a ds_write_b128.  Wave w makes tiles w and w + 8 for all eight.
//   X           turned into the same 1 KB fragments by a kernel of its own (5 us for 333 x 3584), copied with global_load_lds
//   tags        a round's units of a tile go to LDS too: a load into registers inside the loop would make the compiler wait for
//               every copy in flight
//   barrier     one per stage, two slots of products before its end: every wave has then read the stage to its end, so its buffer
//               takes the stage NB further on at once, and the next stage's first fragments come in under the last products
//
// Bound, d = 8: what L2 gives, about 13.5 TB/s over the chip: 64 bytes per codeword and the activations once per workgroup (18944 x 2
// x 3584 at 333 rows: 1.09 + 0.65 GB, 119 us with everything; decoded and multiplied in tiles 243; 256 rows 108, in one pass over the tags 188).
// d = 4: matrix cores and LDS (reads of fragments, codewords 1.7 clocks apart by bank conflicts) in turn, 43 and 48 percent of
// the time at 256 rows: 82 us with 10-bit tags, 110 in one pass over the tags; 333 rows 103 and 153.  Reading all fragments a whole step ahead, the
// barrier a stage early, and all LDS operations dealt out between the products changed nothing (80 to 84); eight token tiles a
// wave spill.
#pragma once
#include <type_traits>
#include "sq_rows_mfma.h"

namespace sq {

constexpr int FUSED_TN = 4, FUSED_RN = 2;    // waves of a workgroup: token quarters x row halves, two per SIMD

// 16 bytes per lane from offset `at` of a buffer to LDS, 16 bytes apart; zeros where the offset lies past its end
__device__ __forceinline__ void buffer_to_lds16(__amdgpu_buffer_rsrc_t buffer, uint32_t at, __attribute__((address_space(3))) void* to) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer, to, 16, at, 0, 0, 0);
}

struct FusedPiece {
    sq_matrix m;
    const void* w;               // tile-major copy of the tags, or NULL
    float* part;                 // ks > 1: fp32 [ks, T, R]
    int wg0;
};

struct FusedArgs {
    FusedPiece p[MID_PIECES];
    int n;
    const unsigned char* x;      // activations in fragment order (fused_x_kernel)
    void* y;
    int64_t ldy;
    int T, y_dtype;
    int U, ks, table_bytes, per_tb, k32;     // units of a row, K slices, workgroups per token block, steps of 32 columns
};

// s_waitcnt immediate: at most n vector-memory operations outstanding, all LDS reads and writes done (vmcnt in bits 3:0 and 15:14,
// expcnt 6:4, lgkmcnt 11:8)
constexpr int fused_wait(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

// Stages of S steps of 32 columns, NB of them in LDS.  With 192 tokens two steps, or the barrier comes too often.
constexpr int fused_steps(int NW) { return NW == 3 ? 2 : 1; }
constexpr int fused_slots(int D, int NW) { return NW == 3 ? 2 : D == 8 ? 4 : 3; }
constexpr int fused_stage_bytes(int NW, int TW, int S) { return S * (FUSED_RN * TW + FUSED_TN * NW) * 1024; }
// LDS that a tile's tags of one round take: a unit per lane, 16 bytes apart (a 12-byte load to LDS leaves its lanes 16 bytes apart
// too), the fifth dwords of 20-byte units behind them
constexpr int fused_tag_bytes(int bits) { return bits == 10 ? 1280 : 1024; }
// d = 4: eight zero bytes behind the stages for the units past a row's end.  With two books of 12-bit tags this variant fills LDS to the last
// byte without them: there the codewords read are replaced by zeros (which costs other variants up to 4 percent).
constexpr bool fused_zero_word(int bits, int NW, int TW) { return !(bits == 12 && NW == 3 && TW == 4); }
constexpr int fused_lds(int bits, int table_bytes, int NW, int TW, int S, int NB) {
    return table_bytes + 2 * FUSED_RN * TW * fused_tag_bytes(bits) + NB * fused_stage_bytes(NW, TW, S) + (table_bytes && fused_zero_word(bits, NW, TW) ? 8 : 0);
}

template <int BITS, int D, int NW, int TW, int S, int NB>
__global__ __launch_bounds__(512, 2) void fused_kernel(FusedArgs a) {
    constexpr int UD = unit_of<BITS>::UD, TPU = UD * 32 / BITS, SPR = TPU / (8 / D), NST = SPR / S, TB = fused_tag_bytes(BITS);
    constexpr int RT = FUSED_RN * TW, NT = FUSED_TN * NW, WB = S * RT * 1024, STAGE = fused_stage_bytes(NW, TW, S);
    constexpr int PT = (RT + 7) / 8, XI = NW * S / 2, Q = S * NW;          // weight tiles a wave fetches (at most); its copies of X; slots of a stage
    static_assert(SPR % S == 0 && SPR % 2 == 0 && NB <= NST && NW * S % 2 == 0 && Q >= 3, "stages of a round");
    constexpr int CNT = XI + (D == 8 ? S : 0);                             // memory operations of a stage and wave, with one weight tile
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), tn = wave & 3, rn = wave >> 2;
    if (D == 4 && (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem != 0u) return;   // (gathers count from LDS address 0)
    const int tb = (int)blockIdx.x / a.per_tb, wg = (int)blockIdx.x - tb * a.per_tb;
    int pi = 0;
    while (pi + 1 < a.n && wg >= a.p[pi + 1].wg0) ++pi;
    const FusedPiece& P = a.p[pi];
    const sq_matrix& m = P.m;
    const int w = wg - P.wg0, slice = w % a.ks, blk = w / a.ks;
    const int NR = a.k32 / SPR, r0 = (int)((int64_t)NR * slice / a.ks), r1 = (int)((int64_t)NR * (slice + 1) / a.ks);
    unsigned char* ring = smem + a.table_bytes + 2 * RT * TB;

    // ---- weights: wave w fetches tiles w and w + 8 of the workgroup's
    const int ntiles = (m.R + 15) >> 4, tile0 = blk * RT;
    const bool tiled = P.w != nullptr;
    const uint32_t us = (tiled ? 16 * UD : UD) * 4;
    const char* tags = reinterpret_cast<const char*>(P.w ? P.w : m.tags);
    uint32_t to[PT], bo[PT];
    const bool mine = wave < RT, both = wave + 8 < RT;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int tile = min(tile0 + min(wave + 8 * i, RT - 1), ntiles - 1), row = min(tile * 16 + li, m.R - 1);
        to[i] = tiled ? ((uint32_t)tile * (uint32_t)a.U * 16u + (uint32_t)li) * (UD * 4) : (uint32_t)row * (uint32_t)m.W * 4u;
        bo[i] = m.row_book ? (uint32_t)m.row_book[row] << (BITS + (D == 8 ? 4 : 3)) : 0u;
    }
    typedef const __attribute__((address_space(1))) void* gptr_t;
    typedef __attribute__((address_space(3))) void* lptr_t;
    // the lanes' units of a round, straight into LDS (nobody but this wave reads them)
    unsigned char* tagbuf = smem + a.table_bytes + wave * TB;
    auto load_tags = [&](int round, int set) {
        const uint32_t u = (uint32_t)min(4 * round + lg, a.U - 1) * us;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            if (!(i ? both : mine)) continue;
            unsigned char* at = tagbuf + (set * RT + 8 * i) * TB;
            const char* from = tags + (to[i] + u);
            if constexpr (UD == 3) __builtin_amdgcn_global_load_lds((gptr_t)from, (lptr_t)at, 12, 0, 0);
            else __builtin_amdgcn_global_load_lds((gptr_t)from, (lptr_t)at, 16, 0, 0);
            if constexpr (UD == 5) __builtin_amdgcn_global_load_lds((gptr_t)(from + 16), (lptr_t)(at + 1024), 4, 0, 0);
        }
    };
    // the dwords of a unit that hold a step's tags, taken out of LDS a stage before they are used
    dwords<UD> held[S][PT];
    auto hold = [&](int set, int step0) {
#pragma unroll
        for (int jj = 0; jj < S; ++jj)
#pragma unroll
            for (int i = 0; i < PT; ++i) {
                const unsigned char* at = tagbuf + (set * RT + 8 * i) * TB;
                const int bit = (step0 + jj) * (8 / D) * BITS;
#pragma unroll
                for (int k = 0; k < UD; ++k)
                    if (k * 32 < bit + 8 / D * BITS && k * 32 + 32 > bit)
                        held[jj][i].v[k] = *reinterpret_cast<const uint32_t*>(UD == 5 && k == 4 ? at + 1024 + lane * 4 : at + lane * 16 + k * 4);
            }
    };
    // the held tags' codewords into the stage buffer at `buf`, 1 KB a tile and step in the lanes' order.  d = 8: from L2, straight
    // into LDS.  d = 4: out of the codebook in LDS to registers (gather_w), from there into the buffer (put_w).
    u32x4 word[S][PT];
    // A round's units past the row's end are zeros (products of the row's last unit with the zeros of X would be NaN where one of its
    // codewords is not finite): d = 8, an offset past the end of the codebooks, which reads as zeros; d = 4, zeros in LDS.
    constexpr bool ZW = fused_zero_word(BITS, NW, TW);
    const __amdgpu_buffer_rsrc_t words = __builtin_amdgcn_make_buffer_rsrc((void*)m.table, 0, D == 8 ? (uint32_t)m.G << (BITS + 4) : 0u, 0x00027000);
    const uint32_t wzero = (uint32_t)(a.table_bytes + 2 * RT * TB + NB * STAGE);
    auto gather_w = [&](int round, int step0, unsigned char* buf) {
        const bool past = 4 * round + lg >= a.U;
        const uint32_t mask = ZW && past ? 0u : ((1u << BITS) - 1u) << 3;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            if (D == 8 && !(i ? both : mine)) continue;
#pragma unroll
            for (int jj = 0; jj < S; ++jj) {
                const int step = step0 + jj;
                if constexpr (D == 8) {
                    buffer_to_lds16(words, (unit_tag<BITS, UD>(held[jj][i], step) << 4) | (past ? 0xFFFFFFF0u : bo[i]), (lptr_t)(buf + (jj * RT + wave + 8 * i) * 1024));
                } else {
                    const u32x2 lo = *(const mma_lds_u32x2*)(uintptr_t)unit_lds_offset<BITS, UD, 3>(held[jj][i], step * 2, ZW && past ? wzero : bo[i], mask);
                    const u32x2 hi = *(const mma_lds_u32x2*)(uintptr_t)unit_lds_offset<BITS, UD, 3>(held[jj][i], step * 2 + 1, ZW && past ? wzero : bo[i], mask);
                    word[jj][i] = !ZW && past ? u32x4{0u, 0u, 0u, 0u} : u32x4{lo.x, lo.y, hi.x, hi.y};
                }
            }
        }
    };
    auto put_w = [&](unsigned char* buf) {
        if (D == 8) return;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            if (!(i ? both : mine)) continue;
#pragma unroll
            for (int jj = 0; jj < S; ++jj) *reinterpret_cast<u32x4*>(buf + (jj * RT + wave + 8 * i) * 1024 + lane * 16) = word[jj][i];
        }
    };
    const unsigned char* xsrc = a.x + (int64_t)tb * a.k32 * (NT * 1024) + wave * (XI * 1024);
    const uint32_t xlane = (uint32_t)lane * 16u;
    auto copy_x = [&](int k32, unsigned char* buf) {
        const unsigned char* from = xsrc + (uint32_t)min(k32, a.k32 - S) * (uint32_t)(NT * 1024);
#pragma unroll
        for (int i = 0; i < XI; ++i)
            __builtin_amdgcn_global_load_lds((gptr_t)(from + i * 1024 + xlane), (lptr_t)(buf + WB + wave * (XI * 1024) + i * 1024), 16, 0, 0);
    };

    float4v acc[TW][NW];
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int n = 0; n < NW; ++n) acc[i][n] = float4v{0.f, 0.f, 0.f, 0.f};

    load_tags(r0, r0 & 1);
    load_tags(r0 + 1, (r0 + 1) & 1);
    if (D == 4) {
        stage_table(m.table, a.table_bytes, smem);
        if (ZW && tid == 0) *reinterpret_cast<u32x2*>(smem + wzero) = u32x2{0u, 0u};
        __syncthreads();
    }
    __builtin_amdgcn_s_waitcnt(fused_wait(0));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        hold(r0 & 1, q * S);
        gather_w(r0, q * S, ring + q * STAGE);
        put_w(ring + q * STAGE);
        copy_x(r0 * SPR + q * S, ring + q * STAGE);
    }
    hold((r0 + NB / NST) & 1, NB % NST * S);
    if (NB == NST) load_tags(r0 + 2, r0 & 1);
    // what waits for all but the copies of the `stages` newest stages: by a wave without a weight tile, with one, with two
    auto wait_stage = [&](auto stages) {
        constexpr int N = decltype(stages)::value;
        if (D == 8 && !mine) __builtin_amdgcn_s_waitcnt(fused_wait(N * XI));
        else if (D == 8 && both) __builtin_amdgcn_s_waitcnt(fused_wait(N * (CNT + S)));
        else __builtin_amdgcn_s_waitcnt(fused_wait(N * CNT));
    };
    wait_stage(std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0); __builtin_amdgcn_s_barrier(); __builtin_amdgcn_sched_barrier(0);

    half8v fa[2][TW], b0, b1, b2;                                          // weights of this step and the next, activations of three slots
    const uint32_t la = (uint32_t)(rn * TW * 1024 + lane * 16), lb = (uint32_t)(WB + tn * NW * 1024 + lane * 16);
    auto read_a = [&](int set, int i, const unsigned char* buf, int j) { fa[set][i] = *reinterpret_cast<const half8v*>(buf + la + (j * RT + i) * 1024); };
    auto read_b = [&](int q, const unsigned char* buf) { return *reinterpret_cast<const half8v*>(buf + lb + ((q / NW) * NT + q % NW) * 1024); };
#pragma unroll
    for (int i = 0; i < TW; ++i) read_a(0, i, ring, 0);
    b0 = read_b(0, ring); b1 = read_b(1, ring);
    int cur = 0;                                                           // ring slot of the stage being multiplied
#pragma unroll 1
    for (int round = r0; round < r1; ++round) {
#pragma unroll
        for (int h = 0; h < NST; ++h) {
            const int ph = h * S;                                          // steps of the round before this stage
            unsigned char* buf = ring + cur * STAGE;
            cur = cur + 1 == NB ? 0 : cur + 1;
            unsigned char* next = ring + cur * STAGE;
            const int ahead = h + NB, pr = ahead / NST, ps = ahead % NST;   // the stage that is fetched: its round from `round`, its place in it
#pragma unroll
            for (int q = 0; q < Q; ++q) {
                const int j = q / NW, n = q % NW;
                if (q == 1) put_w(ring + (cur < 2 ? cur + NB - 2 : cur - 2) * STAGE);   // (gathered two slots before this stage, for the buffer in front of this one)
                if (q == Q - 2) {
                    // every wave's part of the next stage is there, and every wave has read this one to the end
                    wait_stage(std::integral_constant<int, NB - 2>{});
                    __builtin_amdgcn_sched_barrier(0); __builtin_amdgcn_s_barrier(); __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int i = 0; i < TW; ++i) read_a((ph + S) & 1, i, next, 0);
                }
                if (q + 2 < Q) {
                    b2 = read_b(q + 2, buf);
                    if (j + 1 < S && n < TW) read_a((ph + j + 1) & 1, n, buf, j + 1);
                    if (j + 1 < S && n == NW - 1)
#pragma unroll
                        for (int i = NW; i < TW; ++i) read_a((ph + j + 1) & 1, i, buf, j + 1);
                } else {
                    b2 = read_b(q + 2 - Q, next);
                }
                if (q == Q - 2) {
                    // this stage's buffer is free: the stage NB further on goes there
                    gather_w(round + pr, ps * S, buf);
                    copy_x((round + pr) * SPR + ps * S, buf);
                    if (ps + 1 < NST) hold((round + pr) & 1, (ps + 1) * S);
                    else { hold((round + pr + 1) & 1, 0); load_tags(round + pr + 2, (round + pr) & 1); }
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < TW; ++i)
                    acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa[(ph + j) & 1][i], b0, acc[i][n], 0, 0, 0);
                b0 = b1; b1 = b2;
            }
        }
    }
    __builtin_amdgcn_s_waitcnt(fused_wait(0));
    __syncthreads();

    // ---- results: lane: token 16 n + li, weight rows 16 tile + 4 lg .. + 3.  16 tokens at a time through LDS, from where they
    // leave in pieces of eight rows of a token.
    constexpr int PITCH = TW * 64 + 16;
    unsigned char* my = smem + wave * (16 * PITCH);
    const int rw0 = (tile0 + rn * TW) * 16, tw0 = tb * NT * 16 + tn * NW * 16;
    const bool vec = a.y_dtype != SQ_F32 && (a.ldy & 7) == 0 && (m.y_off & 7) == 0 && ((uintptr_t)a.y & 15) == 0;
    // 16-bit results whose rows allow no 16-byte stores leave in pairs, so that a wave's stores are whole lines (row after row of eight, us, before / so:
    // 333 rows of 2 x 18945 x 3584 134 / 125, 170 of 15000 | 3751 | 3751 x 1024 28.4 / 24.1)
    const bool pairs = a.y_dtype != SQ_F32 && a.ks == 1 && !vec, whole = (a.ldy & 1) == 0 && (m.y_off & 1) == 0 && ((uintptr_t)a.y & 3) == 0;
    float sc[TW][4];
#pragma unroll
    for (int i = 0; i < TW; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) sc[i][e] = a.ks > 1 ? 1.f : h2f(m.row_scale[min(rw0 + i * 16 + lg * 4 + e, m.R - 1)]);
#pragma unroll
    for (int n = 0; n < NW; ++n) {
#pragma unroll
        for (int i = 0; i < TW; ++i) {
            const float4v v = acc[i][n];
            *reinterpret_cast<float4v*>(my + li * PITCH + (i * 16 + lg * 4) * 4) = float4v{v[0] * sc[i][0], v[1] * sc[i][1], v[2] * sc[i][2], v[3] * sc[i][3]};
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (pairs) {
#pragma unroll 1
            for (int k = lane; k < 16 * TW * 8; k += 64) {
                const int tl = k / (TW * 8), pc = k - tl * (TW * 8), t = tw0 + n * 16 + tl, r = rw0 + pc * 2;
                const float* v = reinterpret_cast<const float*>(my + tl * PITCH + pc * 8);
                if (t < a.T) store_pair(reinterpret_cast<uint16_t*>(a.y) + (int64_t)t * a.ldy + m.y_off + r, a.y_dtype == SQ_BF16 ? f2bf_x2(v[0], v[1]) : f2h_x2(v[0], v[1]), r - m.R, whole);
            }
        } else
#pragma unroll 1
        for (int k = lane; k < 16 * TW * 2; k += 64) {
            const int tl = k / (TW * 2), pc = k - tl * (TW * 2), t = tw0 + n * 16 + tl, r = rw0 + pc * 8;
            if (t >= a.T || r >= m.R) continue;
            const float4v lo = *reinterpret_cast<const float4v*>(my + tl * PITCH + pc * 32), hi = *reinterpret_cast<const float4v*>(my + tl * PITCH + pc * 32 + 16);
            const int64_t o = (int64_t)t * a.ldy + m.y_off + r;
            if (a.ks > 1) {
                float* p = P.part + ((int64_t)slice * a.T + t) * m.R + r;
                if (m.R % 8 == 0) {
                    *reinterpret_cast<float4v*>(p) = lo;
                    *reinterpret_cast<float4v*>(p + 4) = hi;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) if (r + e < m.R) p[e] = e < 4 ? lo[e & 3] : hi[e & 3];
                }
            } else if (vec && r + 8 <= m.R) {
                *reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(a.y) + o) =
                    a.y_dtype == SQ_BF16 ? u32x4{f2bf_x2(lo[0], lo[1]), f2bf_x2(lo[2], lo[3]), f2bf_x2(hi[0], hi[1]), f2bf_x2(hi[2], hi[3])}
                                         : u32x4{f2h_x2(lo[0], lo[1]), f2h_x2(lo[2], lo[3]), f2h_x2(hi[0], hi[1]), f2h_x2(hi[2], hi[3])};
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) if (r + e < m.R) store_y(a.y, a.y_dtype, o + e, e < 4 ? lo[e & 3] : hi[e & 3]);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

template <int BITS, int D, int NW, int TW, int S, int NB>
int launch_fused_as(const FusedArgs& a, int grid, hipStream_t s) {
    static bool raised = false;
    if (!raised) {
        (void)hipFuncSetAttribute((const void*)fused_kernel<BITS, D, NW, TW, S, NB>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
        raised = true;
    }
    hipLaunchKernelGGL((fused_kernel<BITS, D, NW, TW, S, NB>), dim3((unsigned)grid), dim3(512), (size_t)fused_lds(BITS, a.table_bytes, NW, TW, S, NB), s, a);
    return check_launch("sq_linear_gemm(fused)");
}

// a variant per number of token and weight tiles of a wave
#define SQ_FUSED_CASE(NW_, TW_) if (nw == NW_ && tw == TW_) return launch_fused_as<BITS, D, NW_, TW_, fused_steps(NW_), fused_slots(D, NW_)>(a, grid, s);
template <int BITS, int D>
int launch_fused_format(const FusedArgs& a, int nw, int tw, int grid, hipStream_t s) {
    SQ_FUSED_CASE(3, 2) SQ_FUSED_CASE(3, 3) SQ_FUSED_CASE(3, 4) SQ_FUSED_CASE(3, 5) SQ_FUSED_CASE(4, 2) SQ_FUSED_CASE(4, 3) SQ_FUSED_CASE(4, 4)
    SQ_FUSED_CASE(4, 5) SQ_FUSED_CASE(6, 2) SQ_FUSED_CASE(6, 3) SQ_FUSED_CASE(6, 4) SQ_FUSED_CASE(6, 5)
    if constexpr (D == 8) { SQ_FUSED_CASE(4, 1) }
    return SQ_EUNSUPPORTED;
}

#define SQ_FUSED_FORMAT(BITS, D)                                                                                          \
    int launch_fused_b##BITS##d##D(const FusedArgs& a, int nw, int tw, int grid, hipStream_t s) {                         \
        return launch_fused_format<BITS, D>(a, nw, tw, grid, s);                                                           \
    }

}  // namespace sq
