// Decode-time codebook product on the matrix cores, B = 1..32 activation rows, for gfx950.
//
// v_mfma_f32_16x16x32_f16 multiplies a 16 x 32 tile of weights (A) by 32 x 16 activations (B):
//   A: lane l supplies row l % 16, 8 consecutive k starting at 8 * (l / 16)
//   B: lane l supplies activation row (token) l % 16, the same 8 k
//   D: lane l holds token l % 16, weight rows 4 * (l / 16) .. + 3
// Eight consecutive k of one weight row are exactly two d = 4 codewords or one d = 8 codeword, so a
// lane builds its A operand by gathering raw fp16 codewords (from LDS when the codebook fits) with no
// arithmetic at all, the sum over k happens inside the accumulator, and the cost of a tile does not
// depend on how many of the 16 activation rows are real.  The row scale multiplies the fp32 result.
//
// Work split.  A wave owns a slice of the columns for its whole life, so its B operands (the
// activations of that slice, converted bf16 -> fp16 once) are loaded once and stay in registers; it
// walks over 16-row tiles with the tags of the next tiles in flight (one tile ahead when the codewords come
// through the cache, which is then the bound; two or three tiles when the codebook sits in LDS).
// The tag stream is read in lane units (UD dwords = TPU whole tags = UK columns): in round n the four
// lane groups g = 0..3 of a row read units 4n + g, one wide load each, and the round's SPU matrix
// instructions consume the units chunk pair by chunk pair.  The KW waves of a workgroup split the
// columns of a tile; their accumulators are added through LDS by one wave per tile (round robin): after
// every MMA_TT tiles when the codebook is read through the cache, after all the tiles of the workgroup (as
// many as LDS holds accumulators for: MmaArgs.tg) when it sits in LDS, so that the waves of a launch of the
// 7B shapes meet once.  Rows longer than KW * RW rounds are split over `ks` workgroups whose
// partial sums go to a workspace and are added, in slice order, by slice_sum_kernel.
#pragma once
#include <mutex>
#include <unordered_map>
#include "sq_gemv_kernel.h"

namespace sq {

struct MmaPiece {
    sq_matrix m;
    const uint32_t* tiled; // tile-major copy of the tags (sq_matrix.stream of a d = 4 format) or NULL (rows of whole units only)
    float* part;          // ks > 1: fp32 [ks, B, R] unscaled partial sums of this piece
    int wg_begin;         // first workgroup of this piece
    int wg_count;         // nshare * ks workgroups
};

struct MmaArgs {
    MmaPiece p[GEMV_MAX_PIECES];
    int n;
    const uint16_t* x;
    int64_t ldx;
    void* y;
    int64_t ldy;
    int B;
    int x_dtype, y_dtype;
    int U;                // lane units per row
    int ks;               // workgroup-level column slices
    int table_bytes;      // bytes of codebook staged in LDS (0 = read through cache)
    int tg;               // codebook in LDS: 16-row tiles whose accumulators LDS holds between two barriers (a multiple of mma_group())
    int xt;               // tokens of a staging area: 16, or 8 (one token tile)
    int broken;           // 1: the rows end within a unit (codebook in LDS, tile-major copies, no act)
    int act;              // 1: the two pieces are a gate and an up projection, y receives SiLU(gate) * up (16-bit)
};

constexpr int MMA_TT = 4;     // 16-row tiles multiplied between two workgroup barriers (codebook read through the cache)
// codebook in LDS: tiles of tags in flight per lane (two where a third one's registers would cost a wave per SIMD; 2 to 5 tiles
// in flight measure alike on the 7B shapes)
constexpr int mma_pft(int RW, int NT) { return RW >= 8 || (RW >= 4 && NT == 1) ? 2 : 3; }
constexpr int mma_group(int RW, int NT, bool act) { return act && mma_pft(RW, NT) % 2 ? 2 * mma_pft(RW, NT) : mma_pft(RW, NT); }     // ACT: whole pairs
// LDS per wave in which a round's activations (`tokens` x 4 lane units of UK columns, fp16) pass from whole-line loads to the lanes
// that use them; it lies where the accumulators are added afterwards.  16 tokens at a time, or 8 (MmaArgs.xt): enough for up to
// 8 rows, and what lets twice the waves start next to 128 KB of codebooks.
constexpr int mma_x_stage_bytes(int UK, int tokens) { return tokens * (4 * UK * 2 + 16); }
constexpr int mma_x_tokens_min(int NT) { return NT == 1 ? 8 : 16; }

// Optional timeline of the first wave of every workgroup (debug builds define SQ_TRACE_POINT).
#ifndef SQ_TRACE_POINT
#define SQ_TRACE_POINT(k)
#endif

// LDS byte offset of the codeword of tag t of a unit, counted from the start of the dynamic LDS: the tag times 2^SH (the
// codeword size) plus `bo`, the byte offset of the row's codebook, whose bits lie above the tag's: one shift (or
// v_alignbit_b32 for a tag that straddles two dwords, which starts past bit SH) and one v_and_or_b32
// (mask: the tag's bits where they end up, or 0: the offset is then `bo` itself)
template <int BITS, int UD, int SH>
__device__ __forceinline__ uint32_t unit_lds_offset(const dwords<UD>& u, int t, uint32_t bo, uint32_t mask = ((1u << BITS) - 1u) << SH) {
    const int p = t * BITS, w = p >> 5, s = p & 31;
    uint32_t v;
    if (s + BITS <= 32) v = s >= SH ? u.v[w] >> (s - SH) : u.v[w] << (SH - s);
    else v = __builtin_amdgcn_alignbit(u.v[w + 1 < UD ? w + 1 : w], u.v[w], s - SH);
    return (v & mask) | bo;
}
typedef __attribute__((address_space(3))) u32x2 mma_lds_u32x2;
typedef __attribute__((address_space(3))) u32x4 mma_lds_u32x4;

// two packed bf16 -> two packed fp16: round to nearest even like every other kernel of the library (exact for every
// fp16-normal value, +-inf beyond 65,504; a round-toward-zero conversion would clamp to 65,504 instead and make this
// kernel differ from the batch-1 one on the same input)
__device__ __forceinline__ uint32_t bf2h_pk(uint32_t v) { return bf2h_x2(v); }

// Waves per workgroup beside a codebook in LDS: 16 (four per SIMD) for the variants whose lanes hold at most 8 activation operands (32
// registers), 12 for those with 16; 8 otherwise.
constexpr int mma_waves_max(int x_operands, bool lds_tab) { return !lds_tab ? 8 : x_operands <= 8 ? 16 : x_operands <= 16 ? 12 : 8; }

// ACT (codebooks in LDS): p[0] is a gate and p[1] an up projection of one shape, both codebooks are staged, a workgroup walks the
// two pieces' tiles in turn (virtual tile i: tile i / 2 of piece i % 2), and the wave that adds up a pair of tiles writes SiLU(gate) * up,
// with the same roundings as the product followed by silu_mul_kernel.  It saves that launch and the trip of gate and up through memory
// (2 x 18944 x 3584, 12-bit tags, 8 rows: 20.4 us, now 17.6).
// BROKEN (codebooks in LDS, tile-major copies): the row's last unit has columns past the row's end.  Their codewords, and those of the units
// behind it, are read from 16 zero bytes behind the codebook (a choice per codeword, which whole rows do without).
template <int BITS, int D, int RW, int NT, bool LDS_TAB, bool ACT = false, int XT = 16, bool BROKEN = false>
__global__ __launch_bounds__(64 * mma_waves_max(RW * ((unit_of<BITS>::UD * 32 / BITS) / (8 / D)) * NT, LDS_TAB))
void rows_mfma_kernel(MmaArgs a) {
    constexpr int UD = unit_of<BITS>::UD;
    constexpr int TPU = UD * 32 / BITS;      // tags per lane unit
    constexpr int CPS = 8 / D;               // codewords a lane feeds into one matrix instruction
    constexpr int SPU = TPU / CPS;           // matrix instructions per round
    constexpr int UK = TPU * D;              // columns per lane unit
    constexpr int ESZ = D * 2;               // bytes per codeword
    constexpr int TT = MMA_TT;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), KW = blockDim.x >> 6;
    int pi = 0;
    while (pi + 1 < a.n && (int)blockIdx.x >= a.p[pi + 1].wg_begin) ++pi;
    const MmaPiece& P = a.p[pi];
    const sq_matrix& m = P.m;
    const int w = blockIdx.x - P.wg_begin, slice = w % a.ks, share = w / a.ks, nshare = P.wg_count / a.ks;
    const int ntiles = (m.R + 15) >> 4;
    const int t0 = (int)((int64_t)ntiles * share / nshare), t1 = (int)((int64_t)ntiles * (share + 1) / nshare);
    SQ_TRACE_POINT(0);

    // LDS: [codebook][16 bytes: zeros if BROKEN][reduction buffer: TT tiles x KW waves x 64 lanes x NT x 16 bytes]
    // (the codeword gathers form LDS addresses as numbers counted from the start of the dynamic LDS, which is address 0 in a
    // kernel without static LDS; a build in which it is not leaves y unwritten, which no test survives)
    if (LDS_TAB && (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem != 0u) return;
    float4v* red = reinterpret_cast<float4v*>(smem + a.table_bytes + 16);

    // ---- this wave's rounds
    const int rbase = (slice * KW + wave) * RW;
    bool live[RW];
    bool lane_live = true;
    uint32_t uoff[RW];
    int cols[RW];                            // columns of the row from this lane's unit on
#pragma unroll
    for (int n = 0; n < RW; ++n) {
        const int u = 4 * (rbase + n) + lg;
        live[n] = u < a.U;
        cols[n] = m.C - u * UK;
        lane_live = lane_live && live[n];
        const int uc = live[n] ? u : a.U - 1;
        uoff[n] = (uint32_t)uc * UD;
    }
    // Units past the row's end (only in waves that cover the tail of the columns) contribute exact zeros: their
    // activation operands are zero, and what they multiply with is the row's own last unit again (with the codebook in
    // LDS; a codeword that is not finite is already part of the row's sum) or a zeroed operand (without).
    const bool all_live = __builtin_amdgcn_readfirstlane(__all(lane_live) ? 1 : 0) != 0;
    const uint32_t* tags = reinterpret_cast<const uint32_t*>(m.tags);
    const unsigned char* table = reinterpret_cast<const unsigned char*>(m.table);

    // ---- a tile's memory: tags of this lane's row, its codebook offset, the scales of its four output rows
    // (book: the byte of row_book as loaded; without codebook ids a byte of valid memory that `bkmask` turns into 0 where it is
    // used: a branch around the load, or a use right behind it, would make every wait of the loop a wait for all loads)
    struct Tile { dwords<UD> t[RW]; uint32_t book; };
    const uint8_t* bkp = m.row_book ? m.row_book : reinterpret_cast<const uint8_t*>(m.row_scale);
    const uint32_t bkmask = m.row_book ? 0xFFu : 0u;
    auto fetch = [&](int t, Tile& T, float (&sc)[4]) {
        const int row0 = t << 4;
        const int r = row0 + li < m.R ? row0 + li : m.R - 1;
        T.book = bkp[r];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int ro = row0 + 4 * lg + v;
            sc[v] = h2f(m.row_scale[ro < m.R ? ro : m.R - 1]);
        }
        if (P.tiled) {           // unit u of the tile's 16 rows: 16 * UD consecutive dwords
            const uint32_t* tp = P.tiled + ((size_t)t * a.U * 16 + li) * UD;
#pragma unroll
            for (int n = 0; n < RW; ++n) T.t[n] = load_unit<UD>(tp + (size_t)uoff[n] * 16);
        } else {
            const uint32_t* rp = tags + (size_t)r * m.W;
#pragma unroll
            for (int n = 0; n < RW; ++n) T.t[n] = load_unit<UD>(rp + uoff[n]);
        }
        if (!LDS_TAB && !all_live) {
#pragma unroll
            for (int n = 0; n < RW; ++n)
#pragma unroll
                for (int i = 0; i < UD; ++i) T.t[n].v[i] = live[n] ? T.t[n].v[i] : 0u;
        }
    };

    // ---- start-up: every load the first products need is requested before anything waits, in the order in which it
    // can come back (a wave's loads return in the order of their issue): the activations of this wave's columns, which
    // the cache holds; the tags of the first tiles, which come from memory; then, once the activations have been handed
    // to the lanes (a wait for them alone), the codebook.
    Tile tA, tB;
    float sc[TT + 1][4];                                      // [TT]: first tile of the next group, fetched early
    const bool table_dma = LDS_TAB && (a.table_bytes & 1023) == 0;
    // The activations.  In the matrix instruction a lane supplies one token's 8 columns, so loading the operands where
    // they are used makes every load instruction touch 64 different cache lines (16 tokens x 4 lane units, 16 bytes of
    // each).  Instead the wave fetches the columns of a round, 16 tokens x XRB contiguous bytes, with whole-line loads
    // (1 KB per instruction: 8 lines), and the lanes pick their operands out of LDS: a staging area per wave that lies
    // where the accumulators are added later, which nobody writes before the barrier below.
    constexpr int XRB = 4 * UK * 2;                          // bytes of one token's columns in one round of a wave
    constexpr int XROW = XRB + 16;                           // a token's row in the staging area (the 16 tokens' reads spread over the banks)
    constexpr int XTPI = 1024 / XRB;                         // tokens per load instruction
    static_assert(16 / XTPI == SPU, "a round's activations are SPU loads per token tile");
    constexpr int F = ACT ? 2 : 1;                           // pieces whose tiles a workgroup walks
    const MmaPiece& P1 = a.p[F - 1];
    unsigned char* xst = smem + a.table_bytes + 16 + wave * mma_x_stage_bytes(UK, XT);
    const int xtl = lane / (XRB / 16), xob = (lane % (XRB / 16)) * 16;    // this lane's token (within an instruction) and byte in the round
    u32x4 xraw[RW][NT][SPU];
#pragma unroll
    for (int n = 0; n < RW; ++n)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int j = 0; j < SPU; ++j) {
                const int tok = nt * 16 + j * XTPI + xtl;
                int col = 4 * (rbase + n) * UK + (xob >> 1);
                col = col < m.C ? col : m.C - 8;             // (columns past the row's end: any valid address, the operand is zeroed)
                xraw[n][nt][j] = *reinterpret_cast<const u32x4*>(a.x + (int64_t)(tok < a.B ? tok : a.B - 1) * a.ldx + col);
            }
    if constexpr (!ACT) fetch(t0 < t1 ? t0 : ntiles - 1, tA, sc[0]);     // (no branch around the loads; a workgroup without tiles reads the last one)
    // (codebook in LDS: the tags of the first tiles in flight, without a branch around the loads so that the waits count
    // them exactly: the two layouts differ in a base and a stride, chosen once)
    constexpr int PFT = LDS_TAB ? mma_pft(RW, NT) : 1;
    const bool til = P.tiled != nullptr;
    const uint32_t* fbase = til ? P.tiled + li * UD : tags;
    const uint32_t* fbase1 = ACT ? (til ? P1.tiled + li * UD : reinterpret_cast<const uint32_t*>(P1.m.tags)) : fbase;
    const uint8_t* bkp1 = !ACT ? bkp : P1.m.row_book ? P1.m.row_book : reinterpret_cast<const uint8_t*>(P1.m.row_scale);
    uint32_t fo[RW];
#pragma unroll
    for (int n = 0; n < RW; ++n) fo[n] = til ? uoff[n] * 16u : uoff[n];
    auto fetch_tags = [&](int i, Tile& T) {
        const int t = i / F, row0 = t << 4;
        const int r = row0 + li < m.R ? row0 + li : m.R - 1;
        const bool second = ACT && (i & 1);
        const uint32_t* bp = (second ? fbase1 : fbase) + (til ? (size_t)t * a.U * 16 * UD : (size_t)r * m.W);
        T.book = (second ? bkp1 : bkp)[r];                                  // (first: loads return in order, the tags' waits then cover it)
#pragma unroll
        for (int n = 0; n < RW; ++n) T.t[n] = load_unit<UD>(bp + fo[n]);
    };
    Tile ring[PFT];
    const int i0 = t0 * F, i1 = t1 * F;                      // this workgroup's (virtual) tiles
    if constexpr (LDS_TAB) {
        if constexpr (!ACT) ring[0] = tA;
#pragma unroll
        for (int q = ACT ? 0 : 1; q < PFT; ++q) fetch_tags(min(i0 + q, max(i1 - 1, i0)), ring[q]);
    }
    // the B operands: this wave's activations as fp16, in registers for the whole kernel
    constexpr bool WHOLE = XT == 16;                             // else tokens 0 .. 7 first, then 8 .. 15 in the same place
    static_assert(WHOLE || (XT == 8 && NT == 1), "one token tile in parts of 8");
    half8v xb[RW][SPU][NT];
    auto stage = [&](u32x4 v, int row) {
        if (a.x_dtype == SQ_BF16) { v.x = bf2h_pk(v.x); v.y = bf2h_pk(v.y); v.z = bf2h_pk(v.z); v.w = bf2h_pk(v.w); }
        *reinterpret_cast<u32x4*>(xst + row * XROW + xob) = v;
    };
    // (the lanes of a wave exchange data here: its LDS instructions run in order, the fences keep the compiler from
    // moving a lane's reads before its writes)
    auto exchange = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const unsigned char* xmine = xst + (WHOLE ? li : li & 7) * XROW + lg * (UK * 2);
#pragma unroll
    for (int n = 0; n < RW; ++n)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
            constexpr int HALF = 8 / XTPI;
#pragma unroll
            for (int j = 0; j < HALF; ++j) stage(xraw[n][nt][j], j * XTPI + xtl);
            if (WHOLE)
#pragma unroll
                for (int j = HALF; j < SPU; ++j) stage(xraw[n][nt][j], j * XTPI + xtl);
            exchange();
            const bool mine = live[n] && nt * 16 + li < a.B;
            auto real = [&](int s) { return mine && (!BROKEN || s * 8 < cols[n]); };
#pragma unroll
            for (int s = 0; s < SPU; ++s) {
                u32x4 v = *reinterpret_cast<const u32x4*>(xmine + s * 16);
                if (!(real(s) && (WHOLE || li < 8))) v = u32x4{0u, 0u, 0u, 0u};
                xb[n][s][nt] = __builtin_bit_cast(half8v, v);
            }
            exchange();
            if (!WHOLE && a.B > 8) {
#pragma unroll
                for (int j = HALF; j < SPU; ++j) stage(xraw[n][nt][j], j * XTPI + xtl - 8);
                exchange();
#pragma unroll
                for (int s = 0; s < SPU; ++s) {
                    const u32x4 v = *reinterpret_cast<const u32x4*>(xmine + s * 16);
                    if (real(s) && li >= 8) xb[n][s][nt] = __builtin_bit_cast(half8v, v);
                }
                exchange();
            }
        }
    // (a codebook of whole KB goes memory -> LDS without passing through registers, a wave instruction per KB)
    if (table_dma) {
        typedef const __attribute__((address_space(1))) void* gptr_t;
        typedef __attribute__((address_space(3))) void* lptr_t;
        const int half = a.table_bytes >> 11;
        for (int c = wave; c < (a.table_bytes >> 10); c += KW) {
            const unsigned char* from = table + (size_t)c * 1024;
            if (ACT && c >= half) from = reinterpret_cast<const unsigned char*>(P1.m.table) + (size_t)(c - half) * 1024;
            __builtin_amdgcn_global_load_lds((gptr_t)(from + lane * 16), (lptr_t)(smem + c * 1024), 16, 0, 0);
        }
    } else if (LDS_TAB) {
        stage_table(m.table, a.table_bytes, smem);
    }
    if (BROKEN && tid < 4) reinterpret_cast<uint32_t*>(smem + a.table_bytes)[tid] = 0u;
    // BROKEN: such rows ran on the vector kernel, which multiplies bf16 in fp32: a token's bf16 activations whose fp16 values would not be
    // theirs (beyond 65,504), or would lose bits that matter (a mean square below 2^-13, of which values below 2^-17 are no longer a
    // negligible part), are taken again here, straight into the operands, times a power of two that the sums are divided by.  (The sum of
    // squares of the fp16 values says which: a dot product per pair of them, while the codebook is on its way; 5120 x 2064 at 2 / 16 / 32 rows
    // 6.8 / 7.4 / 10.4 us without, 7.0 / 7.6 / 11.0 so.)
    int xexp[NT];
    bool scaled = false;
    if constexpr (BROKEN) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) xexp[nt] = 0;
        if (a.x_dtype == SQ_BF16) {
            const float least = (float)min(RW * 4 * UK, m.C - 4 * rbase * UK) * 0x1p-13f;      // (not positive: a wave without columns)
            bool odd = false;
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                float part[4] = {};                              // (a chain each)
#pragma unroll
                for (int n = 0; n < RW; ++n)
#pragma unroll
                    for (int s = 0; s < SPU; ++s)
#pragma unroll
                        for (int e = 0; e < 8; e += 2) {
                            const half2v h = {xb[n][s][nt][e], xb[n][s][nt][e + 1]};
                            part[e >> 1] = __builtin_amdgcn_fdot2(h, h, part[e >> 1], false);
                        }
                __builtin_amdgcn_sched_barrier(0);
                const float sq = lane_groups_sum((part[0] + part[1]) + (part[2] + part[3]));
                odd = odd || (nt * 16 + li < a.B && least > 0.f && !(sq >= least && sq < __builtin_inff()));
            }
            scaled = __any((int)odd) != 0;
        }
        if (__builtin_expect(scaled, 0)) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) {
                const uint16_t* xr = a.x + (int64_t)min(nt * 16 + li, a.B - 1) * a.ldx;
                int first = 4 * rbase * UK + lg * UK;
                auto raw = [&](int n, int s) {
                    const bool real = live[n] && s * 8 < cols[n] && nt * 16 + li < a.B;
                    const u32x4 v = *reinterpret_cast<const u32x4*>(xr + (real ? first + 4 * n * UK + s * 8 : 0));
                    return real ? v : u32x4{0u, 0u, 0u, 0u};
                };
                uint32_t top = 0u;                               // the largest magnitude of this token's columns, as bf16 bits
#pragma unroll
                for (int n = 0; n < RW; ++n)
#pragma unroll 1
                    for (int s = 0; s < SPU; ++s) {
                        const u32x4 v = raw(n, s);
#pragma unroll
                        for (int e = 0; e < 4; ++e) top = max(top, max(v[e] & 0x7FFFu, (v[e] >> 16) & 0x7FFFu));
                    }
                top = max(top, (uint32_t)__shfl_xor((int)top, 16, 64));
                top = max(top, (uint32_t)__shfl_xor((int)top, 32, 64));
                // the largest one to 2^12 .. 2^13 (what is 2^-29 of it and more keeps all its bits); infinities and NaN stay what they are
                xexp[nt] = max((int)min(top >> 7, 254u) - (127 + 12), -64);
                const float by = __builtin_bit_cast(float, (uint32_t)(127 - xexp[nt]) << 23);
#pragma unroll
                for (int n = 0; n < RW; ++n)
#pragma unroll
                    for (int s = 0; s < SPU; ++s) {
                        const u32x4 v = raw(n, s);
                        u32x4 h;
#pragma unroll
                        for (int e = 0; e < 4; ++e) h[e] = f2h_x2(bf2f((uint16_t)(v[e] & 0xFFFFu)) * by, bf2f((uint16_t)(v[e] >> 16)) * by);
                        xb[n][s][nt] = __builtin_bit_cast(half8v, h);
                        asm volatile("" : "+v"(first) : "v"(h));  // (one load at a time: there are no registers for more)
                    }
            }
        }
    }
    SQ_TRACE_POINT(1);
    // every wave has taken its operands out of the staging area (and, with the codebook in LDS, the codebook has landed
    // and the first tile's tags with it)
    __builtin_amdgcn_s_waitcnt(0);
    if (LDS_TAB || KW > 1) __syncthreads();
    SQ_TRACE_POINT(2);

    // One tile: NS = RW * SPU matrix instructions.  The codeword gathers run PD instructions ahead of the
    // matrix instruction that consumes them, so LDS latency overlaps the multiplies of earlier steps.
    constexpr int NS = RW * SPU, PD = NS < 6 ? NS : 6;
    // (tab: byte offset of the piece's codebooks in LDS)
    auto multiply = [&](const Tile& cur, float4v (&acc)[NT], uint32_t tab = 0) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) acc[nt] = float4v{0.f, 0.f, 0.f, 0.f};
        u32x4 av[NS];
        auto gather = [&](int k) {
            const int n = k / SPU, s = k - n * SPU;
            const bool dead = !all_live && !live[n];
            const uint32_t bo = ((cur.book & bkmask) << BITS) * ESZ + tab;      // byte offset of the row's codebook
            if (D == 8) {
                if (LDS_TAB) {
                    av[k] = *reinterpret_cast<const mma_lds_u32x4*>((uintptr_t)unit_lds_offset<BITS, UD, 4>(cur.t[n], s, bo));
                } else {
                    const uint32_t tag = unit_tag<BITS, UD>(cur.t[n], s);
                    av[k] = *reinterpret_cast<const u32x4*>(table + ((size_t)tag * ESZ + bo));
                }
            } else {
                u32x2 c0, c1;
                if (LDS_TAB) {
                    uint32_t o0 = unit_lds_offset<BITS, UD, 3>(cur.t[n], 2 * s, bo), o1 = unit_lds_offset<BITS, UD, 3>(cur.t[n], 2 * s + 1, bo);
                    if (BROKEN && s * 8 >= cols[n]) o0 = o1 = (uint32_t)a.table_bytes;
                    c0 = *reinterpret_cast<const mma_lds_u32x2*>((uintptr_t)o0);
                    c1 = *reinterpret_cast<const mma_lds_u32x2*>((uintptr_t)o1);
                } else {
                    const uint32_t g0 = unit_tag<BITS, UD>(cur.t[n], 2 * s);
                    const uint32_t g1 = unit_tag<BITS, UD>(cur.t[n], 2 * s + 1);
                    c0 = *reinterpret_cast<const u32x2*>(table + ((size_t)g0 * ESZ + bo));
                    c1 = *reinterpret_cast<const u32x2*>(table + ((size_t)g1 * ESZ + bo));
                }
                av[k] = u32x4{c0.x, c0.y, c1.x, c1.y};
            }
            if (!LDS_TAB && dead) av[k] = u32x4{0u, 0u, 0u, 0u};
        };
#pragma unroll
        for (int k = 0; k < PD; ++k) gather(k);
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            if (k + PD < NS) gather(k + PD);
            __builtin_amdgcn_sched_barrier(0);          // keep the gathers ahead of the multiply they are not for
            const int n = k / SPU, s = k - n * SPU;
            const half8v af = __builtin_bit_cast(half8v, av[k]);
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
                acc[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af, xb[n][s][nt], acc[nt], 0, 0, 0);
        }
        if (BROKEN && __builtin_expect(scaled, 0)) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[nt][v] = __builtin_ldexpf(acc[nt][v], xexp[nt]);
        }
    };

    if constexpr (LDS_TAB) {
        // ---- codebook in LDS.  Nothing here waits for the cache, so what bounds the kernel is how many bytes of tags it
        // keeps in flight and how often its waves meet: every lane holds mma_pft(RW) tiles of tags (a tile's registers are
        // refilled as soon as its last codeword has been gathered), a tile's accumulator goes straight to its place in
        // LDS, and the waves meet once per a.tg tiles (once per launch when the workgroup's tiles all fit), after which
        // each tile is added up by one wave (round robin), scaled and stored.
        if (t0 >= t1) return;                                 // (uniform in the workgroup; the launcher gives every one a tile)
        auto tab_of = [&](int i) { return ACT && (i & 1) ? (uint32_t)a.table_bytes / 2 : 0u; };
        auto tile_done = [&](int tl, const float4v (&acc)[NT]) {
#pragma unroll
            for (int nt = 0; nt < NT; ++nt) red[((tl * KW + wave) * 64 + lane) * NT + nt] = acc[nt];
        };
        for (int tg = i0; tg < i1; tg += a.tg) {
            const int te = min(tg + a.tg, i1);
            if (tg > i0) __syncthreads();                     // the previous group's sums have been read
            int t = tg;
            for (; t + PFT <= te; t += PFT) {
#pragma unroll
                for (int q = 0; q < PFT; ++q) {
                    float4v acc[NT];
                    multiply(ring[q], acc, tab_of(t + q));
                    __builtin_amdgcn_sched_barrier(0);
                    fetch_tags(min(t + q + PFT, i1 - 1), ring[q]);
                    __builtin_amdgcn_sched_barrier(0);
                    tile_done(t + q - tg, acc);
                }
            }
#pragma unroll
            for (int q = 0; q < PFT; ++q)
                if (t + q < te) {                             // (the last group's last tiles: nothing left to fetch)
                    float4v acc[NT];
                    multiply(ring[q], acc, tab_of(t + q));
                    tile_done(t + q - tg, acc);
                }
            __syncthreads();
            auto sum_of = [&](int tl, int nt) {
                float4v s4 = red[((tl * KW) * 64 + lane) * NT + nt];
                for (int k = 1; k < KW; ++k) {
                    const float4v o = red[((tl * KW + k) * 64 + lane) * NT + nt];
                    s4.x += o.x; s4.y += o.y; s4.z += o.z; s4.w += o.w;
                }
                return s4;
            };
            if constexpr (ACT) {
                for (int tl = 2 * wave; tl < te - tg; tl += 2 * KW) {
                    const int row0 = ((tg + tl) >> 1) << 4;
#pragma unroll
                    for (int nt = 0; nt < NT; ++nt) {
                        const float4v g4 = sum_of(tl, nt), u4 = sum_of(tl + 1, nt);
                        const int tok = nt * 16 + li;
                        if (tok >= a.B) continue;
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            const int r = row0 + 4 * lg + v;
                            if (r >= m.R) continue;
                            reinterpret_cast<uint16_t*>(a.y)[(int64_t)tok * a.ldy + r] =
                                silu_mul_one(round16(g4[v] * h2f(m.row_scale[r]), a.y_dtype), round16(u4[v] * h2f(P1.m.row_scale[r]), a.y_dtype), a.y_dtype);
                        }
                    }
                }
                continue;
            }
            for (int tl = wave; tl < te - tg; tl += KW) {
                const int row0 = (tg + tl) << 4;
                float scl[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int ro = row0 + 4 * lg + v;
                    scl[v] = h2f(m.row_scale[ro < m.R ? ro : m.R - 1]);
                }
#pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const float4v s4 = sum_of(tl, nt);
                    const int tok = nt * 16 + li;
                    if (tok >= a.B) continue;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int r = row0 + 4 * lg + v;
                        if (r >= m.R) continue;
                        if (a.ks > 1) P.part[((int64_t)slice * a.B + tok) * m.R + r] = s4[v];
                        else store_y(a.y, a.y_dtype, (int64_t)tok * a.ldy + m.y_off + r, s4[v] * scl[v]);
                    }
                }
            }
        }
    } else {
        // ---- groups of TT tiles: multiply them one after the other (the next tile's tags load meanwhile), then
        // add the KW waves' accumulators through LDS, each tile of the group by a different wave
        for (int tg = t0, grp = 0; tg < t1; tg += TT, ++grp) {
            float4v acc[TT][NT];
            if (grp > 0) {
    #pragma unroll
                for (int v = 0; v < 4; ++v) sc[0][v] = sc[TT][v];
            }
    #pragma unroll
            for (int tt = 0; tt < TT; tt += 2) {
                if (tg + tt < t1) {
                    if (tg + tt + 1 < t1) fetch(tg + tt + 1, tB, sc[tt + 1]);
                    multiply(tA, acc[tt]);
                }
                if (tg + tt + 1 < t1) {
                    if (tg + tt + 2 < t1) fetch(tg + tt + 2, tA, sc[tt + 2]);
                    multiply(tB, acc[tt + 1]);
                }
            }
            SQ_TRACE_POINT(3 + 3 * (grp < 4 ? grp : 4));
            if (KW > 1) {
                if (grp > 0) __syncthreads();                     // the previous group's reducers are done reading
    #pragma unroll
                for (int tt = 0; tt < TT; ++tt)
    #pragma unroll
                    for (int nt = 0; nt < NT; ++nt) red[((tt * KW + wave) * 64 + lane) * NT + nt] = acc[tt][nt];
                __syncthreads();
            }
            SQ_TRACE_POINT(4 + 3 * (grp < 4 ? grp : 4));
    #pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
                const int t = tg + tt;
                if (t >= t1) continue;
                if (KW > 1 && wave != (tt + grp) % KW) continue;   // this tile's reducer
                float4v tot[NT];
    #pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    if (KW > 1) {
                        float4v s4 = red[((tt * KW) * 64 + lane) * NT + nt];
                        for (int k = 1; k < KW; ++k) {
                            const float4v o = red[((tt * KW + k) * 64 + lane) * NT + nt];
                            s4.x += o.x; s4.y += o.y; s4.z += o.z; s4.w += o.w;
                        }
                        tot[nt] = s4;
                    } else tot[nt] = acc[tt][nt];
                }
                const int row0 = t << 4;
    #pragma unroll
                for (int nt = 0; nt < NT; ++nt) {
                    const int tok = nt * 16 + li;
                    if (tok >= a.B) continue;
    #pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int r = row0 + 4 * lg + v;
                        if (r >= m.R) continue;
                        if (a.ks > 1) P.part[((int64_t)slice * a.B + tok) * m.R + r] = tot[nt][v];
                        else store_y(a.y, a.y_dtype, (int64_t)tok * a.ldy + m.y_off + r, tot[nt][v] * sc[tt][v]);
                    }
                }
            }
            SQ_TRACE_POINT(5 + 3 * (grp < 4 ? grp : 4));
        }
    }
    SQ_TRACE_POINT(19);
}

// op 0: launch; op 1: workgroups of `threads` threads and `smem` bytes of LDS that fit on one CU
template <int BITS, int D, int RW, int NT>
static inline int mma_inst(int op, const MmaArgs& a, int grid, int threads, size_t smem, hipStream_t s) {
    // (the widest variant with codebooks in LDS is for rows that only it takes in one launch, which have no fused SiLU: see mma_whole_row)
    constexpr bool LDS = D == 4, WIDEST = NT == 1 && RW * ((unit_of<BITS>::UD * 32 / BITS) / (8 / D)) > 16;
    void (*k)(MmaArgs) = rows_mfma_kernel<BITS, D, RW, NT, false>;
    if constexpr (LDS) {
        if (a.table_bytes) k = rows_mfma_kernel<BITS, D, RW, NT, true>;
        if constexpr (NT == 1)
            if (a.xt == 8 && a.table_bytes) k = rows_mfma_kernel<BITS, D, RW, NT, true, false, 8>;
        if (a.table_bytes && a.broken) k = rows_mfma_kernel<BITS, D, RW, NT, true, false, 16, true>;
        if constexpr (NT == 1)
            if (a.xt == 8 && a.table_bytes && a.broken) k = rows_mfma_kernel<BITS, D, RW, NT, true, false, 8, true>;
        if constexpr (!WIDEST) {
            if (a.table_bytes && a.act) k = rows_mfma_kernel<BITS, D, RW, NT, true, true>;
            if constexpr (NT == 1)
                if (a.xt == 8 && a.table_bytes && a.act) k = rows_mfma_kernel<BITS, D, RW, NT, true, true, 8>;
        }
    }
    if (a.broken && !(LDS && a.table_bytes)) return fail(SQ_EUNSUPPORTED, "sq_linear_small: rows that end within a lane unit need their codebook in LDS");
    if (a.table_bytes && (!LDS || (WIDEST && a.act)))
        return fail(SQ_EUNSUPPORTED, "sq_linear_small: no matrix-core kernel for %d rounds and codebooks in LDS", RW);
    if (op == 1) {
        static std::mutex mu;
        static std::unordered_map<uint64_t, int> cache;
        const uint64_t key = ((uint64_t)threads << 40) | ((uint64_t)(a.table_bytes != 0) << 39) | ((uint64_t)a.act << 38) | ((uint64_t)(a.xt == 8) << 37) | ((uint64_t)a.broken << 36) | (uint64_t)smem;
        std::lock_guard<std::mutex> lock(mu);
        auto it = cache.find(key);
        if (it != cache.end()) return it->second;
        if (smem > 64 * 1024) {      // allow the 160 KB of a gfx950 CU
            (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            (void)hipGetLastError();
        }
        hipFuncAttributes fa;
        int n = 1;
        if (hipFuncGetAttributes(&fa, (const void*)k) == hipSuccess && fa.numRegs > 0) {
            int wps = 512 / ((fa.numRegs + 7) / 8 * 8);     // 512 VGPRs per SIMD lane, granules of 8
            if (wps > 8) wps = 8;
            n = 4 * wps / (threads / 64);
        } else {
            (void)hipGetLastError();
        }
        if (smem && (size_t)n * smem > 160 * 1024) n = (int)(160 * 1024 / smem);
        if (n < 1) n = 1;
        cache[key] = n;
        return n;
    }
    hipLaunchKernelGGL(k, dim3(grid), dim3(threads), smem, s, a);
    return check_launch("sq_linear_small(mfma)");
}

// (RW, NT) pairs built per format: RW * SPU * NT <= 32 activation operands (128 registers) per lane
template <int BITS, int D>
static inline int mma_dispatch(int op, const MmaArgs& a, int RW, int NT, int grid, int threads, size_t smem, hipStream_t s) {
    constexpr int SPU = (unit_of<BITS>::UD * 32 / BITS) / (8 / D);
    constexpr int R1 = 32 / SPU;          // most rounds per wave with 16 activation rows
#define SQ_MMA(RW_, NT_) if (RW == RW_ && NT == NT_) return mma_inst<BITS, D, RW_, NT_>(op, a, grid, threads, smem, s)
    SQ_MMA(R1, 1);
    SQ_MMA(R1 / 2, 1);
    SQ_MMA(R1 / 2, 2);
    if constexpr (R1 >= 4) {
        SQ_MMA(R1 / 4, 1);
        SQ_MMA(R1 / 4, 2);
    }
#undef SQ_MMA
    return fail(SQ_EUNSUPPORTED, "sq_linear_small: no matrix-core kernel for %d rounds, %d token tiles", RW, NT);
}

#define SQ_MMA_FORMAT(BI, DD)                                                                               \
    int launch_mma_b##BI##d##DD(int op, const MmaArgs& a, int RW, int NT, int grid, int threads, size_t smem, \
                                hipStream_t s) {                                                            \
        return mma_dispatch<BI, DD>(op, a, RW, NT, grid, threads, smem, s);                                 \
    }

}  // namespace sq
