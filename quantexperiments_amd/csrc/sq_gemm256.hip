// Large-tile fp16 GEMM for prefill: Y[T, R] = X[T, C] . W[R, C]^T, fp32 accumulate, optional row scale.
//
// Workgroup tile 256, 192 or 128 tokens x 256 weight rows (64 MT x 256, chosen by gemm256_plan), 4 waves in 2 x 2, each a
// 32 MT x 128 tile of v_mfma_f32_16x16x32_f16 accumulators (MT = 4: all 256 accumulator registers), one wave per SIMD.  Both
// operands are K-contiguous fp16 in memory.  The K loop moves in slabs of 64 columns; a slab of ONE operand (rows of 128 bytes,
// whole 128-byte lines: half-line requests get 10.5 TB/s out of L2 over the chip, whole lines 15.2 TB/s) is copied from global
// memory straight into LDS (buffer_load_dwordx4 ... lds: no staging registers) into a ring of slots of that operand.
//
// Bound: the chip's power.  Matrix instructions alone, on normally distributed operands held in registers, reach 1.69 PFLOP/s as
// 32x32x16 and 1.95 as 16x16x32 (2.42 both on zeros, where the clock stays at its limit): the accumulators a product reads
// and writes cost power, and 16x16x32 has half of them per operation.  What else takes power or clocks in the loop counts the same way:
//   * the products are written out as instructions: of the builtin's 128 accumulators the compiler moves some away and back in every
//     step (0.9 vector instructions a product; in that form 16x16x32 was slower than 32x32x16, 1.26 and 1.29 PFLOP/s on 8192^3);
//   * a slab's 128 products of a wave share the loop with 32 LDS reads, 16 copies and about 30 other instructions: four copies
//     share an LDS base, pieces past a row's end change the copies' offsets once, in front of the last slab, and the ring's offsets
//     are worked out between products.  With an offset chosen per copy and bases per copy: 74 instead of 80 % of the matrix
//     cores' time;
//   * a product's neighbours share an operand (rows of blocks walked to and fro: 0.4 %).
// 8192^3 / 2048 x 37888 x 3584, in turn on one machine: 835 / 472 us as 32x32x16, 758 / 437 as 16x16x32, 727 / 415 with the lean loop
// (1.51 PFLOP/s).
//
// What a lone wave per SIMD needs is that nothing in its instruction stream waits:
//   * X blocks are read in place, a row of products behind their last use, the weights' blocks one 32-column step ahead;
//   * one barrier per slab, eight products into the slab's last step, when its last fragments have arrived: it
//     frees the slab's two slots and says that the next slab is complete;
//   * the slots it frees take one operand's slab behind the barrier, among the reads of the next slab's first fragments, and a slab
//     of the other during the next slab's first step.
// MT = 4 and 3: three W slots, two X slots: W, which comes from memory where X stays in L2, has one to two slabs' time to
// arrive.  MT = 2, whose slabs take half as long: three W and four X slots, two to three slabs' time (with two and three:
// 333 x 3584 x 18944 in four 89 us, now 77; 1024 x 7168 x 5120 91 and 81).  Eight waves of 128 x 64 (two per SIMD) ran at 1.15
// PFLOP/s on 8192^3, in one schedule or as two groups taking turns at matrix and memory phases.
//
// LDS rows are 128 bytes; the 16-byte piece c of row r is stored at slot c ^ ((r >> 1) & 7).  A ds_read_b128
// serves 16 lanes per clock from 64 banks (256 bytes), rows 0-3 and 12-15 of one piece with rows 4-11 of the next; they fall on
// 16 different 16-byte bank groups ((r & 1) * 8 + slot), so the operand reads are conflict free.
//
// Operand layout of v_mfma_f32_16x16x32_f16, lane l: A row / B column l % 16, k = 8 * (l / 16) .. + 7;
// D[v], v = 0..3: row 4 * (l / 16) + v, column l % 16.  Rows of D are weight rows, columns are tokens,
// so a lane holds 4 consecutive outputs of one token in a row of registers.
#include <algorithm>
#include <climits>
#include <type_traits>
#include <utility>
#include "sq_common.h"

namespace sq {

constexpr int G_BN = 256, G_BK = 64, G_WAVES = 4;
constexpr int G_W_SLOT = G_BN * G_BK * 2;
constexpr int gemm256_tokens(int mt) { return 64 * mt; }                           // token rows of a tile
constexpr int gemm256_x_slots(int mt) { return mt == 2 ? 4 : 2; }
constexpr int gemm256_w_slots(int) { return 3; }
constexpr int gemm256_lds(int mt) { return gemm256_x_slots(mt) * gemm256_tokens(mt) * G_BK * 2 + gemm256_w_slots(mt) * G_W_SLOT; }     // 160, 144, 160 KB
constexpr int gemm256_super(int mt) { return 32 / mt; }       // token tiles (about 2048 rows) that are walked together, see below

struct Gemm256Args {
    const uint16_t* x;        // fp16 [T, C], row stride ldx
    const uint16_t* w;        // fp16 [R, C], row stride ldw
    Gemm256Scales sc;         // row scales of the pieces the R rows consist of
    void* y;
    int64_t ldx, ldw, ldy;
    int T, R, C, y_off, y_dtype;
    int y_align;              // alignment of the rows of 16-bit results: 16 bytes, 4 or 2
    int tiles_t, tiles_r;     // token / weight-row tiles (for the workgroup -> tile mapping)
    // The last round of tiles rarely fills the chip (592 tiles on 256 CUs: 2 full rounds and 80 tiles).  Tiles
    // [0, main_tiles) are multiplied whole; each of the remaining tail tiles is split over kt workgroups, each
    // taking the slabs [kz nk / kt, (kz + 1) nk / kt) and leaving an unscaled fp32 partial tile in
    // part[(tail tile * kt + kz)][token rows of a tile][256] for gemm256_reduce_kernel.
    int main_tiles, kt;
    float* part;
};

// Tile numbers walk super-columns of up to `super` token tiles, weight tile after weight tile: consecutive tiles, which
// run on one XCD at the same time, then share both operands' slabs in its L2 (8192^3, 32 token tiles: 990 us in one column,
// 900 us in columns of 8).
__host__ __device__ __forceinline__ void gemm256_tile(int tile, int tiles_t, int tiles_r, int super, int* bt, int* br) {
    const int full = tiles_r * super, g = tile / full, l = tile - g * full;
    const int w = tiles_t - g * super < super ? tiles_t - g * super : super;
    *bt = g * super + l % w;
    *br = l / w;
}

// scale of weight row r as fp16 bits (1 without scales).  FLAT: tested against all eight pieces, without a loop, which the tile kernel with all its
// accumulators alive has no registers for (136 bytes of scratch per lane); else against as many as there are (the reduction, four
// look-ups a thread, takes 2 us less of 333 x 37888 x 3584 that way).
template <bool FLAT>
__device__ __forceinline__ uint16_t gemm256_scale(const Gemm256Scales& s, int r) {
    if (s.n == 0) return 0x3C00;
    const uint16_t* p = s.p[0];
    int at = r;
    auto test = [&](int i) { if (r >= s.end[i - 1]) { p = s.p[i]; at = r - s.end[i - 1]; } };
    if constexpr (FLAT) {
#pragma unroll
        for (int i = 1; i < GEMM256_PIECES; ++i) if (i < s.n) test(i);
    } else {
#pragma unroll 1
        for (int i = 1; i < s.n; ++i) test(i);
    }
    return p[at];
}

// s_waitcnt immediate that waits until at most n vector-memory operations are outstanding (gfx9 encoding: vmcnt in bits 3:0 and
// 15:14, expcnt 6:4, lgkmcnt 11:8) and leaves the other counters alone, or also until every LDS read of the wave has arrived
constexpr int vmcnt_only(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }
constexpr int vmcnt_and_lds(int n) { return vmcnt_only(n) & ~(15 << 8); }

// The accumulators are named registers, a[4 (8 i + j)] .. + 3 for token block i and weight-row block j, which no value of the compiler's
// lives in (tests/test_abi.py): written as variables, 256 of 256 registers live over a loop with branches, they spill.
template <int R> __device__ __forceinline__ void acc_product(half8v w, half8v x) {
    asm volatile("v_mfma_f32_16x16x32_f16 a[%0:%1], %2, %3, a[%0:%1]" :: "n"(R), "n"(R + 3), "v"(w), "v"(x));
}
template <int R> __device__ __forceinline__ void acc_clear16(half8v z) {       // sixteen of them, as a product of zeros
    asm volatile("v_mfma_f32_32x32x16_f16 a[%0:%1], %2, %2, 0" :: "n"(R), "n"(R + 15), "v"(z));
}
template <int R> __device__ __forceinline__ float4v acc_read() {
    float4v v;
    asm volatile("v_accvgpr_read_b32 %0, a[%4]\n\tv_accvgpr_read_b32 %1, a[%5]\n\tv_accvgpr_read_b32 %2, a[%6]\n\tv_accvgpr_read_b32 %3, a[%7]"
                 : "=v"(v[0]), "=v"(v[1]), "=v"(v[2]), "=v"(v[3]) : "n"(R), "n"(R + 1), "n"(R + 2), "n"(R + 3));
    return v;
}
template <int N> __device__ __forceinline__ void acc_claim() {                 // the kernel needs the first N of them
    if constexpr (N == 128) asm volatile("" ::: "a127");
    if constexpr (N == 192) asm volatile("" ::: "a191");
    if constexpr (N == 256) asm volatile("" ::: "a255");
}

// calls f with the numbers 0 .. N - 1 as types
template <class F, int... I> __device__ __forceinline__ void each(F f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F> __device__ __forceinline__ void each(F f) { each(f, std::make_integer_sequence<int, N>{}); }

#define SQ_INLINE __attribute__((always_inline))
#define SQ_SB() __builtin_amdgcn_sched_barrier(0)

// What both kernels share: the sizes of a tile of 64 MT rows and the rings' waits ...
template <int MT> struct Gemm256Shape {
    // XC: copies a wave makes of an X slab (of a W slab: 8); TB: its blocks of 16 tokens; NM: products of a step
    static constexpr int BM = gemm256_tokens(MT), XC = 2 * MT, X_SLOT = BM * G_BK * 2, TB = 2 * MT, NM = 8 * TB;
    static constexpr bool XE = gemm256_x_slots(MT) > gemm256_w_slots(MT);        // X is the early operand, the one of E slots; the late one has L
    static constexpr int E = XE ? gemm256_x_slots(MT) : gemm256_w_slots(MT), L = E - 1, EC = XE ? XC : 8, LC = XE ? 8 : XC;
    static_assert(L == (XE ? gemm256_w_slots(MT) : gemm256_x_slots(MT)), "the waits count on it");
    static constexpr int W_AT = gemm256_x_slots(MT) * X_SLOT;
    static constexpr int ES = XE ? X_SLOT : G_W_SLOT, LS = XE ? G_W_SLOT : X_SLOT;       // the slots' sizes
    static constexpr int AHEAD = (E - 2) * EC + (L - 2) * LC;                    // copies that may be on their way when slab s + 1 has to be there
};

// ... copy j of an operand's slab to LDS (four copies share an LDS base: the instruction's own offset, 1024 (j % 4), counts for LDS and memory, so
// the lanes' offsets hold that much less, and bases that start 3072 bytes early keep them positive); an offset of G_PAST is past the buffer's
// end and puts zeros there ...
constexpr uint32_t G_PAST = 0xFFFF0000u;
__device__ __forceinline__ void gemm256_copy(const char* base, uint32_t off, int at, unsigned char* to, int j) {
    typedef __attribute__((address_space(3))) void* lptr_t;
    const __amdgpu_buffer_rsrc_t buf = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, G_PAST, 0x00027000);
    const lptr_t lds = (lptr_t)to;
    if ((j & 3) == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, lds, 16, off, at, 0, 0);
    if ((j & 3) == 1) __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, lds, 16, off, at, 1024, 0);
    if ((j & 3) == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, lds, 16, off, at, 2048, 0);
    if ((j & 3) == 3) __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, lds, 16, off, at, 3072, 0);
}

// ... the slots (byte offsets) of the slab being multiplied (early and late operand), of the next one, and the one the early copies go to ...
template <int MT> struct Gemm256Slots { int ce = 0, cl = 0, ne = 0, nl = 0, to = (Gemm256Shape<MT>::E - 1) * Gemm256Shape<MT>::ES; };

// ... and the schedule of a slab, two steps of 32 columns.  mma(step, n): product n of a step, token block n / 8, weight-row block n % 8, to and
// fro; read_x(kk, slot, i) and read_w(set, kk, slot, j): fragments of step kk; copy_early, copy_late(slot, j); ready(): the wait for this wave's
// copies of slab s + 1 (those of later slabs stay in flight) and its reads of slab s; next(): on to the next slab to copy.  The slots are
// worked out between the products, a little at a time: a scalar instruction in front of them takes four clocks of the matrix core's time.
template <int MT, class Mma, class ReadX, class ReadW, class Early, class Late, class Ready, class Next>
__device__ __forceinline__ void gemm256_slab(Gemm256Slots<MT>& p, Mma mma, ReadX read_x, ReadW read_w, Early copy_early, Late copy_late, Ready ready, Next next) {
    typedef Gemm256Shape<MT> S;
    constexpr bool XE = S::XE;
    constexpr int TB = S::TB, NM = S::NM, GAP = MT == 2 ? 2 : 4;
    // first step: its last X blocks, the second step's fragments, the early copies of slab s + L
    each<NM>([&](auto nn) SQ_INLINE {
        constexpr int n = decltype(nn)::value;
        mma(std::integral_constant<int, 0>{}, nn); SQ_SB();
        if (n < 2) read_x(0, XE ? p.ce : p.cl, TB - 1 - n);
        if (n >= 2 && n <= 16 && n % 2 == 0) read_w(1, 1, XE ? p.cl : p.ce, n / 2 - 1);
        if (n % 8 == 1 && n > 8 && n < NM - 8) read_x(1, XE ? p.ce : p.cl, n / 8 - 1);
        if (n % 4 == 3 && n / 4 < S::EC) copy_early(p.to, n / 4);
        if (n == NM - 6) { p.ne = p.ce + S::ES; SQ_SB(); }
        if (n == NM - 5) { p.ne = p.ne == S::E * S::ES ? 0 : p.ne; SQ_SB(); }
        if (n == NM - 4) { p.nl = p.cl + S::LS; SQ_SB(); }
        if (n == NM - 3) { p.nl = p.nl == S::L * S::LS ? 0 : p.nl; SQ_SB(); }
        if (n == NM - 2) { p.to = p.ce; SQ_SB(); }
        SQ_SB();
    });
    // second step: this wave's copies of slab s + 1 and its reads of slab s, whose slots the copies behind the barrier overwrite, are waited
    // for; then the barrier: everybody's copies have landed and everybody has read slab s to the end.  (Six products behind the last of
    // those reads their wait costs little.)
    each<NM>([&](auto nn) SQ_INLINE {
        constexpr int n = decltype(nn)::value;
        mma(std::integral_constant<int, 1>{}, nn); SQ_SB();
        if (n < 2) read_x(1, XE ? p.ce : p.cl, TB - 1 - n);
        if (n == 7) { ready(); SQ_SB(); __builtin_amdgcn_s_barrier(); SQ_SB(); }
        if (n >= 8 && n <= 22 && n % 2 == 0) read_w(0, 0, XE ? p.nl : p.ne, n / 2 - 4);
        if (n % 8 == 1 && n > 8 && n < NM - 8) read_x(0, XE ? p.ne : p.nl, n / 8 - 1);
        if (n >= 11 && (n - 11) % GAP == 0 && (n - 11) / GAP < S::LC) copy_late(p.cl, (n - 11) / GAP);
        if (n == NM - 4) { next(); SQ_SB(); }
        if (n == NM - 3) { p.ce = p.ne; p.cl = p.nl; SQ_SB(); }
        SQ_SB();
    });
}

// What a workgroup multiplies: a whole tile, or one of the parts of a tail tile.
struct Gemm256Item { int tile, kz, nparts, t0, r0, k_begin, nk; };

// EP: SQ_F16 / SQ_BF16 = results of that type, SQ_F32 = fp32 ones, element by element.  Rows of 16-bit results that allow no 16-byte stores leave in
// pieces of 4 bytes, or 2, a token's 128 by one wave (element by element,
// straight from the accumulators: 496 rows of 666 x 512 with their decode 26.4 us, 19.0 so, 2048 of 18945 x 3584 345 / 303, 2000 of 2 x 18946 x 1024
// 361 / 204, 1024 of 2 x 4098 x 2048 76.6 / 55.9).
// MT: blocks of 32 token rows a wave holds, 64 MT rows a tile
//
// A workgroup per CU takes tile after tile: the copies run L slabs ahead of the products over the end of a tile, so the next
// tile's first slabs arrive while the last products run and the results leave, and the stores of the results have two slabs of
// the next tile to get through.  A workgroup per tile spent 9 us a round of tiles beyond its slabs, 4 to 5 of them on the stores;
// the power limit takes part of that back: gate|up of 2048 rows with its decode (2 x 18944 x 3584, five rounds) 536 -> 523 us, a
// layer of 2048 rows 980 -> 968, 8192^3 with its decode 809 -> 802, products of one round level.
template <int EP, int MT>
__global__ __launch_bounds__(G_WAVES * 64, 1) void gemm256_kernel(Gemm256Args a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroups are dealt round-robin to the 8 XCDs (each with its own L2), so XCD x = blockIdx % 8 takes one
    // contiguous run of whole tiles (a weight tile is then fetched by one L2 only) and, after those, one
    // contiguous run of tail parts; its workgroups take them in turn.
    const int ntiles = a.tiles_t * a.tiles_r, xcd = (int)(blockIdx.x & 7), stride = (int)(gridDim.x >> 3);
    const int main_per = (a.main_tiles + 7) >> 3, parts = (ntiles - a.main_tiles) * a.kt, parts_per = (parts + 7) >> 3;
    const int main_mine = min(main_per, a.main_tiles - xcd * main_per), items = main_per + max(0, min(parts_per, parts - xcd * parts_per));
    typedef Gemm256Shape<MT> S;
    constexpr int BM = S::BM, XC = S::XC, X_SLOT = S::X_SLOT, TB = S::TB, L = S::L, EC = S::EC, LC = S::LC, ES = S::ES, LS = S::LS, W_AT = S::W_AT, AHEAD = S::AHEAD;
    constexpr bool XE = S::XE;
    const int nk_all = (a.C + G_BK - 1) / G_BK;
    auto valid = [&](int j) SQ_INLINE {                // this item, or the workgroup's next one where the XCD's run of tiles is shorter than others'
        while (j >= main_mine && j < main_per) j += stride;
        return j;
    };
    auto item = [&](int j) SQ_INLINE {
        Gemm256Item it;
        it.tile = xcd * main_per + j; it.kz = 0; it.nparts = 1;
        if (j >= main_per) {
            const unsigned p = (unsigned)(xcd * parts_per + (j - main_per)), kt = (unsigned)a.kt;
            it.tile = a.main_tiles + (int)(p / kt);
            it.kz = (int)(p % kt);
            it.nparts = a.kt;
        }
        int bt, br;
        gemm256_tile(it.tile, a.tiles_t, a.tiles_r, gemm256_super(MT), &bt, &br);
        it.t0 = bt * BM; it.r0 = br * G_BN;
        it.k_begin = (int)((unsigned)it.kz * (unsigned)nk_all / (unsigned)it.nparts);
        it.nk = (int)((unsigned)(it.kz + 1) * (unsigned)nk_all / (unsigned)it.nparts) - it.k_begin;
        // (the same for all lanes, but the divisions are vector code)
        it.tile = __builtin_amdgcn_readfirstlane(it.tile); it.kz = __builtin_amdgcn_readfirstlane(it.kz);
        it.t0 = __builtin_amdgcn_readfirstlane(it.t0); it.r0 = __builtin_amdgcn_readfirstlane(it.r0);
        it.nparts = __builtin_amdgcn_readfirstlane(it.nparts); it.k_begin = __builtin_amdgcn_readfirstlane(it.k_begin); it.nk = __builtin_amdgcn_readfirstlane(it.nk);
        return it;
    };
    int jm = valid((int)(blockIdx.x >> 3));  // the item being multiplied, and the one being copied
    if (jm >= items) return;
    int jc = jm;
    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * 128;

    acc_claim<32 * TB>();

    // Copies.  One buffer_load_dwordx4 to LDS fills 1 KB = 8 LDS rows in lane order, so lane s lands in row
    // s >> 3, slot s & 7 of its block and therefore fetches the piece the swizzle puts there.  Wave w copies
    // rows 64 w .. 64 w + 63 of a W slab (8 instructions) and a quarter of the X slab's rows.  Global addresses are a
    // uniform base, a uniform column (advanced per slab) and per-lane 32-bit byte offsets computed once a tile; rows past the matrix
    // edge re-read the last row (their outputs are never stored).  One operand is early (E slots, the copies of slab s + L go out
    // during the first step of slab s), the other late (L = E - 1 slots, the copies go out behind the barrier of slab s); behind the
    // last item's last slab that one is read again.  The pieces of a row's last slab that lie past its end (C % 64 != 0) are asked
    // for past the end of the buffer, which puts zeros into LDS, for both operands (global_load_lds instead of the buffers, for whole
    // slabs: level; rows of broken slabs ran in the 128 x 128 kernel: 5120 x 2080 at 400 / 1500 rows 80-120 / 126-194 us, now 38-43 / 47-53).
    const int lrow = lane >> 3, slot = lane & 7;
    bool past[2];                            // this lane's piece of a row's last slab lies past its end, in even and odd copies (whose rows' swizzles differ by 4)
#pragma unroll
    for (int h = 0; h < 2; ++h) past[h] = (slot ^ (h * 4 + (lrow >> 1))) * 8 >= a.C - (nk_all - 1) * G_BK;
    uint32_t xo[XC], wo[8];
    const char *xt, *wt;
    int at, left, step;                      // the copied slab's first column in bytes, the item's slabs from it on, bytes to the next slab
    int last;                                // 1 in an item that ends with a slab that the row does not fill, until that is the next
    auto row_end = [&]() SQ_INLINE {
#pragma unroll
        for (int j = 0; j < XC; ++j) xo[j] = past[j & 1] ? G_PAST : xo[j];
#pragma unroll
        for (int j = 0; j < 8; ++j) wo[j] = past[j & 1] ? G_PAST : wo[j];
    };
    auto copy_from = [&](int j) SQ_INLINE {
        const Gemm256Item it = item(j);
        int lc = lane;
        asm volatile("" : "+v"(lc));         // (or what depends on the lane alone is worked out in front of the loop and kept in registers that it lacks)
        const int row0 = lc >> 3, piece0 = ((lc & 7) ^ (row0 >> 1)) * 16;
#pragma unroll
        for (int j = 0; j < XC; ++j) {       // (rows 8 j on: their swizzle is that of rows 0 or 8)
            const int t = min(wave * (BM / 4) + j * 8 + row0, a.T - 1 - it.t0);
            xo[j] = (uint32_t)(t * (int)a.ldx * 2 + (piece0 ^ ((j & 1) << 6))) + (uint32_t)(3 - (j & 3)) * 1024u;
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int r = min(wave * 64 + j * 8 + row0, a.R - 1 - it.r0);
            wo[j] = (uint32_t)(r * (int)a.ldw * 2 + (piece0 ^ ((j & 1) << 6))) + (uint32_t)(3 - (j & 3)) * 1024u;
        }
        xt = reinterpret_cast<const char*>(a.x + (int64_t)it.t0 * a.ldx + (int64_t)it.k_begin * G_BK) - 3072;
        wt = reinterpret_cast<const char*>(a.w + (int64_t)it.r0 * a.ldw + (int64_t)it.k_begin * G_BK) - 3072;
        at = 0; left = it.nk; step = G_BK * 2;
        last = a.C % G_BK != 0 && it.kz == it.nparts - 1 ? 1 : 0;
        if (left == last) { row_end(); last = 0; }
    };
    auto next_slab = [&]() SQ_INLINE {
        at += step;
        if (__builtin_expect(--left > last, 1)) return;
        if (left == 1) { row_end(); last = 0; return; }
        jc = valid(jc + stride);
        if (jc < items) copy_from(jc);
        else { at -= step; step = 0; left = INT_MAX; }
    };
    // `to`: the slot's offset
    auto copy_x = [&](int to, int j) SQ_INLINE { gemm256_copy(xt, xo[j], at, smem + to + wave * (X_SLOT / 4) + (j & ~3) * 1024, j); };
    auto copy_w = [&](int to, int j) SQ_INLINE { gemm256_copy(wt, wo[j], at, smem + to + W_AT + wave * 8192 + (j & ~3) * 1024, j); };
    auto copy_early = [&](int to, int j) SQ_INLINE { if constexpr (XE) copy_x(to, j); else copy_w(to, j); };
    auto copy_late = [&](int to, int j) SQ_INLINE { if constexpr (XE) copy_w(to, j); else copy_x(to, j); };

    // Fragments.  A lane reads row (lane & 15) + 16 i of its wave's rows, piece 4 kk + (lane >> 4); the swizzle term depends on the
    // row modulo 16 only and the column step kk only flips bit 6 of the offset, so one offset plus compile-time multiples of
    // 16 rows (2048 bytes) covers all reads of a slab.
    half8v fx[TB], fw[2][8];
    const uint32_t foff = (uint32_t)((lane & 15) * 128 + (((lane >> 4) ^ ((lane >> 1) & 7)) << 4));
    auto read_x = [&](int kk, int at, int i) SQ_INLINE {
        fx[i] = *reinterpret_cast<const half8v*>(smem + at + wm * 128 + i * 2048 + (foff ^ (uint32_t)(kk << 6)));
    };
    auto read_w = [&](int set, int kk, int at, int j) SQ_INLINE {
        fw[set][j] = *reinterpret_cast<const half8v*>(smem + W_AT + at + wn * 128 + j * 2048 + (foff ^ (uint32_t)(kk << 6)));
    };
    auto mma = [&](auto set, auto n) SQ_INLINE {
        constexpr int N = decltype(n)::value, i = N >> 3, j = i & 1 ? 7 - (N & 7) : N & 7;
        acc_product<4 * (8 * i + j)>(fw[decltype(set)::value][j], fx[i]);
    };
    // (the waits of both directions are written out: the compiler does not know what is in the accumulators)
    auto clear = [&]() SQ_INLINE {
        asm volatile("s_nop 15\n\ts_nop 15");
        each<2 * TB>([&](auto q) SQ_INLINE { acc_clear16<16 * decltype(q)::value>(half8v{}); });
        asm volatile("s_nop 15\n\ts_nop 15");
    };

    copy_from(jc);
#pragma unroll 1
    for (int q = 0; q < L; ++q) {
#pragma unroll
        for (int j = 0; j < EC; ++j) copy_early(q * ES, j);
#pragma unroll
        for (int j = 0; j < LC; ++j) copy_late(q * LS, j);
        next_slab();
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only((L - 1) * (EC + LC)));
    SQ_SB(); __builtin_amdgcn_s_barrier(); SQ_SB();
#pragma unroll
    for (int i = 0; i < TB - 2; ++i) read_x(0, 0, i);
#pragma unroll
    for (int j = 0; j < 8; ++j) read_w(0, 0, 0, j);
    Gemm256Slots<MT> slots;
    // the 16-byte stores a wave makes of a whole tile's results, which the next tile's first slab need not wait for
    constexpr int STORES = 8 * MT;
    static_assert(AHEAD + STORES < 64, "what the counter holds");
    Gemm256Item it = item(jm);
    int togo = it.nk;                        // slabs to the item's end
    int stores = 0;                          // 1: the item before this one left in STORES stores and this is the first slab behind them
    // EVENT: a slab that may be an item's first or last one or the last one before the copies go on to another item (or come to a
    // row's broken end); the others have no branches
    auto slab = [&](auto event) SQ_INLINE {
        constexpr bool EVENT = decltype(event)::value;
        gemm256_slab<MT>(slots, mma, read_x, read_w, copy_early, copy_late,
            // (the stores of the item before went out behind slab s + 1's copies where s is an item's first slab: they stay in flight too)
            [&]() SQ_INLINE {
                if (!EVENT || !stores) __builtin_amdgcn_s_waitcnt(vmcnt_and_lds(AHEAD));
                else __builtin_amdgcn_s_waitcnt(vmcnt_and_lds(AHEAD + STORES));
            },
            [&]() SQ_INLINE { if constexpr (EVENT) next_slab(); else at += step; });
    };
    uint32_t scale[2] = {};                  // of weight rows lane and 64 + lane of this wave's 128, fp16
    clear();
    while (true) {
        const int plain = stores ? 0 : min(togo, left - last) - 1;
#pragma unroll 1
        for (int s = 0; s < plain; ++s) slab(std::false_type{});
        if (plain > 0) { togo -= plain; left -= plain; }
        // (asked for a slab ahead: behind the loop their latency would be the tile's)
        if (togo == 1) {
#pragma unroll
            for (int h = 0; h < 2; ++h) scale[h] = gemm256_scale<true>(a.sc, min(it.r0 + wn + h * 64 + lane, a.R - 1));
        }
        slab(std::true_type{});
        stores = 0;
        if (--togo > 0) continue;
        asm volatile("s_nop 15\n\ts_nop 15");    // the last products' results are there before they are read

        // Results leave block of 16 tokens after block.  A split tile's go to its partial tile as they are.  16-bit ones go
        // through LDS, two blocks (MT = 2: one) at a time: every wave lays them out token-major, 256 bytes a token, in its quarter of
        // the early operand's slot of the slab that everybody has read to the end (the quarter that it copies into next itself),
        // 16-byte piece c of token t at slot c ^ (t % 16), and stores them in 16-byte pieces, 256 contiguous bytes per token
        // (2-byte stores straight from the accumulators cost 49 us of a 376 us product of a 2048 x 18944 output).
        int le = lane;
        const int64_t ldy = a.ldy;
        asm volatile("" : "+v"(le));             // (nothing of what follows is worked out in front of the loop and kept in registers that it lacks)
        const int quad = le >> 4, tok = le & 15;
        const int split = it.nparts - 1;
        stores = __builtin_amdgcn_readfirstlane(EP != SQ_F32 && a.y_align == 16 && split == 0 && it.t0 + BM <= a.T && it.r0 + G_BN <= a.R ? 1 : 0);
        float* part = a.part + ((int64_t)(it.tile - a.main_tiles) * a.kt + it.kz) * (BM * G_BN);
        float4v sc[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) sc[j][e] = h2f((uint16_t)__builtin_amdgcn_ds_bpermute(((j & 3) * 16 + 4 * quad + e) * 4, (int)scale[j >> 2]));
        constexpr int TBP = ES / 4 / 4096;
        static_assert(TB % TBP == 0, "whole passes");
        unsigned char* my = smem + (XE ? 0 : W_AT) + slots.to + wave * (ES / 4);
        uint16_t* dst = reinterpret_cast<uint16_t*>(a.y) + (int64_t)(it.t0 + wm) * ldy + a.y_off + it.r0 + wn + (quad * ldy + tok * 8);
        each<TB / TBP>([&](auto pp) SQ_INLINE {
            constexpr int p = decltype(pp)::value;
            auto block = [&](auto q, auto use) SQ_INLINE {
                constexpr int b = decltype(q)::value / 8, j = decltype(q)::value % 8;
                use(b, j, acc_read<4 * (8 * (p * TBP + b) + j)>());
            };
            if (split) {
                each<8 * TBP>([&](auto q) SQ_INLINE {
                    block(q, [&](int b, int j, float4v val) {
                        *reinterpret_cast<float4v*>(part + (wm + (p * TBP + b) * 16 + tok) * G_BN + wn + j * 16 + 4 * quad) = val;
                    });
                });
                return;
            }
            if constexpr (EP == SQ_F32) {
                each<8 * TBP>([&](auto q) SQ_INLINE {
                    block(q, [&](int b, int j, float4v val) {
                        const int t = it.t0 + wm + (p * TBP + b) * 16 + tok, r = it.r0 + wn + j * 16 + 4 * quad;
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (t < a.T && r + e < a.R) store_y(a.y, a.y_dtype, (int64_t)t * ldy + a.y_off + r + e, val[e] * sc[j][e]);
                    });
                });
                return;
            }
            each<8 * TBP>([&](auto q) SQ_INLINE {
                block(q, [&](int b, int j, float4v val) {
                    const float4v o = val * sc[j];
                    *reinterpret_cast<u32x2*>(my + (b * 16 + tok) * 256 + (((2 * j + (quad >> 1)) ^ tok) * 16) + (quad & 1) * 8) =
                        EP == SQ_BF16 ? u32x2{f2bf_x2(o[0], o[1]), f2bf_x2(o[2], o[3])} : u32x2{f2h_x2(o[0], o[1]), f2h_x2(o[2], o[3])};
                });
            });
            if (a.y_align != 16) {
                const int over = it.r0 + wn + 2 * le - a.R;      // (-2 and less: both are rows of W)
                uint16_t* pair = reinterpret_cast<uint16_t*>(a.y) + (int64_t)(it.t0 + wm + p * TBP * 16) * ldy + a.y_off + it.r0 + wn + 2 * le;
#pragma unroll 4
                for (int k = 0; k < 16 * TBP; ++k, pair += ldy) {
                    const uint32_t v2 = *reinterpret_cast<const uint32_t*>(my + k * 256 + (((le >> 2) ^ (k & 15)) * 16) + (le & 3) * 4);
                    if (it.t0 + wm + p * TBP * 16 + k < a.T) store_pair(pair, v2, over, a.y_align == 4);
                }
                return;
            }
            u32x4 v[4 * TBP];
#pragma unroll
            for (int k = 0; k < 4 * TBP; ++k) v[k] = *reinterpret_cast<const u32x4*>(my + (k * 4 + quad) * 256 + ((tok ^ ((k * 4 + quad) & 15)) * 16));
            if (stores) {
#pragma unroll
                for (int k = 0; k < 4 * TBP; ++k) { *reinterpret_cast<u32x4*>(dst) = v[k]; dst += 4 * ldy; }
                return;
            }
#pragma unroll
            for (int k = 0; k < 4 * TBP; ++k) {
                const int t = it.t0 + wm + p * TBP * 16 + k * 4 + quad, over = it.r0 + wn + tok * 8 - a.R;     // (-8 and less: all eight are rows of W)
                if (t < a.T && over <= -8) {
                    *reinterpret_cast<u32x4*>(dst) = v[k];
                } else if (t < a.T) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (e + over < 0) dst[e] = (uint16_t)(v[k][e >> 1] >> (16 * (e & 1)));
                }
                dst += 4 * ldy;
            }
        });
        jm = valid(jm + stride);
        if (jm >= items) break;
        it = item(jm);
        togo = it.nk;
        clear();
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(0));       // no copy is on its way into LDS that is another workgroup's by then
}

constexpr int G_EP_PITCH = 128 * 2 + 16;     // bytes per token row of a wave's 32 MT x 128 output tile in LDS

__device__ __forceinline__ void product(float4v& sums, half8v w, half8v x) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(sums) : "v"(w), "v"(x));
}

// The product of at most a tile (or a part of one) per workgroup: what a workgroup needs to go from tile to tile, products that know about events,
// accumulators it names, addresses in front of every tile, is longer than the slabs of a small product.  us, the kernel above / this one:
// 264 x 576 x 576 16.0 / 12.4, x 2176 20.0 / 18.9, 264 x 4352 x 576 14.5 / 13.5, 1024 x 7168 x 5120 level; of two rounds and more the one above is
// the faster (see there).
template <int EP, int MT>
__global__ __launch_bounds__(G_WAVES * 64, 1) void gemm256_one_kernel(Gemm256Args a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroups are dealt round-robin to the 8 XCDs (each with its own L2), so XCD x = blockIdx % 8 takes one
    // contiguous run of whole tiles (a weight tile is then fetched by one L2 only) and, after those, one
    // contiguous run of tail parts.  The grid is padded; surplus workgroups leave.
    const int ntiles = a.tiles_t * a.tiles_r;
    const int xcd = (int)(blockIdx.x & 7), jx = (int)(blockIdx.x >> 3);
    const int main_per = (a.main_tiles + 7) >> 3, parts = (ntiles - a.main_tiles) * a.kt, parts_per = (parts + 7) >> 3;
    int tile, kz = 0, nparts = 1;
    if (jx < main_per) {
        tile = xcd * main_per + jx;
        if (tile >= a.main_tiles) return;
    } else {
        const int pidx = xcd * parts_per + (jx - main_per);
        if (jx - main_per >= parts_per || pidx >= parts) return;
        tile = a.main_tiles + pidx / a.kt;
        kz = pidx - (pidx / a.kt) * a.kt;
        nparts = a.kt;
    }
    int bt, br;
    gemm256_tile(tile, a.tiles_t, a.tiles_r, gemm256_super(MT), &bt, &br);
    typedef Gemm256Shape<MT> S;
    constexpr int BM = S::BM, XC = S::XC, X_SLOT = S::X_SLOT, TB = S::TB, E = S::E, L = S::L, EC = S::EC, LC = S::LC, ES = S::ES, LS = S::LS, W_AT = S::W_AT, AHEAD = S::AHEAD;
    constexpr bool XE = S::XE;
    const int t0 = bt * BM, r0 = br * G_BN;
    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * 128;

    float4v acc[TB][8];                      // [token block][weight-row block]
#pragma unroll
    for (int i = 0; i < TB; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = float4v{0.f, 0.f, 0.f, 0.f};

    // Copies, as above; slabs past the last one re-read the last.
    const int lrow = lane >> 3, slot = lane & 7;
    uint32_t xo[XC], wo[8];
#pragma unroll
    for (int j = 0; j < XC; ++j) {
        const int row = wave * (BM / 4) + j * 8 + lrow;
        const int t = t0 + row < a.T ? row : a.T - 1 - t0;
        xo[j] = (uint32_t)(t * (int)a.ldx + (slot ^ ((row >> 1) & 7)) * 8) * 2u + (uint32_t)(3 - (j & 3)) * 1024u;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int row = wave * 64 + j * 8 + lrow;
        const int r = r0 + row < a.R ? row : a.R - 1 - r0;
        wo[j] = (uint32_t)(r * (int)a.ldw + (slot ^ ((row >> 1) & 7)) * 8) * 2u + (uint32_t)(3 - (j & 3)) * 1024u;
    }
    const int nk_all = (a.C + G_BK - 1) / G_BK, k_begin = (int)((int64_t)kz * nk_all / nparts);
    const int nk = (int)((int64_t)(kz + 1) * nk_all / nparts) - k_begin;
    const char* xt = reinterpret_cast<const char*>(a.x + (int64_t)t0 * a.ldx + (int64_t)k_begin * G_BK) - 3072;
    const char* wt = reinterpret_cast<const char*>(a.w + (int64_t)r0 * a.ldw + (int64_t)k_begin * G_BK) - 3072;
    const int lastk = nk_all - 1 - k_begin;  // the row's last slab, counted from this part's first
    bool past[2];                            // this lane's piece of it lies past the row's end, in even and odd copies (whose rows' swizzles differ by 4)
#pragma unroll
    for (int h = 0; h < 2; ++h) past[h] = (slot ^ (h * 4 + (lrow >> 1))) * 8 >= a.C - (nk_all - 1) * G_BK;
    // `at`: the slab's first column in bytes, `to`: its slot's offset
    auto copy_x = [&](int at, int to, int j) { gemm256_copy(xt, xo[j], at, smem + to + wave * (X_SLOT / 4) + (j & ~3) * 1024, j); };
    auto copy_w = [&](int at, int to, int j) { gemm256_copy(wt, wo[j], at, smem + to + W_AT + wave * 8192 + (j & ~3) * 1024, j); };
    auto copy_early = [&](int at, int to, int j) { if constexpr (XE) copy_x(at, to, j); else copy_w(at, to, j); };
    auto copy_late = [&](int at, int to, int j) { if constexpr (XE) copy_w(at, to, j); else copy_x(at, to, j); };
    // from the row's last slab on the pieces past its end are asked for past the buffer's end
    const int plast = lastk < nk && a.C % G_BK != 0 ? lastk : INT_MAX;
    auto end_early = [&](int q) {
        if (q < plast) return;
#pragma unroll
        for (int j = 0; j < EC; ++j) { uint32_t& o = XE ? xo[j] : wo[j]; o = past[j & 1] ? G_PAST : o; }
    };
    auto end_late = [&](int q) {
        if (q < plast) return;
#pragma unroll
        for (int j = 0; j < LC; ++j) { uint32_t& o = XE ? wo[j] : xo[j]; o = past[j & 1] ? G_PAST : o; }
    };
    auto column = [&](int q) { return (q < nk ? q : nk - 1) * (G_BK * 2); };

    // Fragments, as above
    half8v fx[TB], fw[2][8];
    const uint32_t foff = (uint32_t)((lane & 15) * 128 + (((lane >> 4) ^ ((lane >> 1) & 7)) << 4));
    auto read_x = [&](int kk, int at, int i) {
        fx[i] = *reinterpret_cast<const half8v*>(smem + at + wm * 128 + i * 2048 + (foff ^ (uint32_t)(kk << 6)));
    };
    auto read_w = [&](int set, int kk, int at, int j) {
        fw[set][j] = *reinterpret_cast<const half8v*>(smem + W_AT + at + wn * 128 + j * 2048 + (foff ^ (uint32_t)(kk << 6)));
    };
    auto mma = [&](auto set, auto n) SQ_INLINE {
        constexpr int N = decltype(n)::value, i = N >> 3, j = i & 1 ? 7 - (N & 7) : N & 7;
        product(acc[i][j], fw[decltype(set)::value][j], fx[i]);
    };
    // the accumulators stay in their registers before and behind the loop (without this the compiler copies all 256 into the
    // other half of the register file at the loop's end, spills, and a launch that needs scratch memory takes 7 us longer)
#define SQ_PIN() _Pragma("unroll") for (int i = 0; i < TB; ++i) { asm volatile("" : "+a"(acc[i][0]), "+a"(acc[i][1]), "+a"(acc[i][2]), "+a"(acc[i][3]), "+a"(acc[i][4]), "+a"(acc[i][5]), "+a"(acc[i][6]), "+a"(acc[i][7])); }

#pragma unroll
    for (int q = 0; q < E - 1; ++q) {
        end_early(q);
#pragma unroll
        for (int j = 0; j < EC; ++j) copy_early(column(q), q * ES, j);
        if (q == L - 1) break;
        end_late(q);
#pragma unroll
        for (int j = 0; j < LC; ++j) copy_late(column(q), q * LS, j);
    }
    __builtin_amdgcn_s_waitcnt(vmcnt_only(AHEAD));
    SQ_SB(); __builtin_amdgcn_s_barrier(); SQ_SB();
#pragma unroll
    for (int i = 0; i < TB - 2; ++i) read_x(0, 0, i);
#pragma unroll
    for (int j = 0; j < 8; ++j) read_w(0, 0, 0, j);
    end_late(L - 1);
#pragma unroll
    for (int j = 0; j < LC; ++j) copy_late(column(L - 1), (L - 1) * LS, j);
    Gemm256Slots<MT> slots;
    int at = column(L);                      // of the slab that is copied
    SQ_PIN();
    asm volatile("s_nop 7");                 // (no wait of the compiler's between the zeroed accumulators and a written-out product)
#pragma unroll 1
    for (int s = 0; s < nk; ++s) {
        if (s + L >= plast) { end_early(s + L); end_late(s + L); }
        gemm256_slab<MT>(slots, mma, read_x, read_w, [&](int to, int j) SQ_INLINE { copy_early(at, to, j); }, [&](int to, int j) SQ_INLINE { copy_late(at, to, j); },
                         [&]() SQ_INLINE { __builtin_amdgcn_s_waitcnt(vmcnt_and_lds(AHEAD)); }, [&]() SQ_INLINE { at = column(s + 1 + L); });
    }
    asm volatile("s_nop 15\n\ts_nop 15");    // the last products' results are behind the loop before they are read
    SQ_PIN();
#undef SQ_PIN
    __builtin_amdgcn_s_waitcnt(vmcnt_and_lds(0));
    __syncthreads();                         // every wave is done with the operand ring, and no copy is on its way into it

    // Results leave column of registers after column of registers.  A split tile's go to its partial tile as they are.  16-bit
    // ones go through LDS: every wave lays its 32 MT x 128 tile out token-major (8 bytes per write) and stores it in 16-byte
    // pieces, 256 contiguous bytes per token (2-byte stores straight from the accumulators cost 49 us of a 376 us product of
    // a 2048 x 18944 output).
    const int quad4 = 4 * (lane >> 4), tok = lane & 15;
    float* scales = reinterpret_cast<float*>(smem + 2 * BM * G_EP_PITCH);        // behind the four waves' tiles
    scales[tid] = h2f(gemm256_scale<true>(a.sc, r0 + tid < a.R ? r0 + tid : a.R - 1));
    __syncthreads();
    float* part = a.part + ((int64_t)(tile - a.main_tiles) * a.kt + kz) * (BM * G_BN);
    unsigned char* my = smem + wave * (BM / 2 * G_EP_PITCH);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int rl = j * 16 + quad4;
        const float4v sc = *reinterpret_cast<const float4v*>(scales + wn + rl);
#pragma unroll
        for (int i = 0; i < TB; ++i) {
            const int tl = i * 16 + tok;
            const float4v val = acc[i][j];
            if (nparts > 1) {
                *reinterpret_cast<float4v*>(part + (wm + tl) * G_BN + wn + rl) = val;
            } else if constexpr (EP != SQ_F32) {
                const float4v o = val * sc;
                *reinterpret_cast<u32x2*>(my + tl * G_EP_PITCH + rl * 2) =
                    EP == SQ_BF16 ? u32x2{f2bf_x2(o[0], o[1]), f2bf_x2(o[2], o[3])} : u32x2{f2h_x2(o[0], o[1]), f2h_x2(o[2], o[3])};
            } else {
                const int t = t0 + wm + tl, r = r0 + wn + rl;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (t < a.T && r + e < a.R) store_y(a.y, a.y_dtype, (int64_t)t * a.ldy + a.y_off + r + e, val[e] * sc[e]);
            }
            if (i & 1) __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (EP == SQ_F32 || nparts > 1) return;
    uint16_t* yb = reinterpret_cast<uint16_t*>(a.y);
    if (a.y_align != 16) {
        uint16_t* pair = yb + (int64_t)(t0 + wm) * a.ldy + a.y_off + r0 + wn + 2 * lane;
#pragma unroll 4
        for (int k = 0; k < BM / 2; ++k, pair += a.ldy)
            if (t0 + wm + k < a.T) store_pair(pair, *reinterpret_cast<const uint32_t*>(my + k * G_EP_PITCH + lane * 4), r0 + wn + 2 * lane - a.R, a.y_align == 4);
        return;
    }
#pragma unroll 4
    for (int k = 0; k < 8 * MT; ++k) {
        const int idx = k * 64 + lane, tl = idx >> 4, piece = idx & 15;
        const int t = t0 + wm + tl, r = r0 + wn + piece * 8;
        if (t >= a.T || r >= a.R) continue;
        const u32x4 v = *reinterpret_cast<const u32x4*>(my + tl * G_EP_PITCH + piece * 16);
        uint16_t* dst = yb + (int64_t)t * a.ldy + a.y_off + r;
        if (r + 8 <= a.R) {
            *reinterpret_cast<u32x4*>(dst) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (r + e < a.R) dst[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
        }
    }
}

// fp16 copy of a bf16 activation matrix (round to nearest even; exact for every fp16-normal value)
__global__ __launch_bounds__(256) void bf16_to_f16_kernel(const uint16_t* __restrict__ x, int64_t ldx, int T, int C,
                                                          uint16_t* __restrict__ out) {
    const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 8;       // 8 elements per thread
    if (i >= (int64_t)T * C) return;
    const int t = (int)(i / C), c = (int)(i - (int64_t)t * C);
    u32x4 v = *reinterpret_cast<const u32x4*>(x + (int64_t)t * ldx + c);
    v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w);
    *reinterpret_cast<u32x4*>(out + i) = v;
}

// tail tiles: y[t, y_off + r] = scale of r * sum over kz of part[(tail tile * kt + kz)][t - t0][r - r0]
__global__ __launch_bounds__(256) void gemm256_reduce_kernel(const float* __restrict__ part, int mt, int main_tiles, int kt,
                                                             int tiles_t, int tiles_r, int T, int R, Gemm256Scales sc, void* y, int64_t ldy,
                                                             int y_off, int y_dtype) {
    const int size = gemm256_tokens(mt) * G_BN, blocks = size / 1024;            // 1024 elements of a tail tile a workgroup
    const int tail = (int)blockIdx.x / blocks, e = ((int)blockIdx.x - tail * blocks) * 1024 + (int)threadIdx.x * 4;
    int bt, br;
    gemm256_tile(main_tiles + tail, tiles_t, tiles_r, gemm256_super(mt), &bt, &br);
    const int t = bt * gemm256_tokens(mt) + e / G_BN, r = br * G_BN + e % G_BN;
    if (t >= T) return;
    const float* p = part + (int64_t)tail * kt * size + e;
    float4v sum = *reinterpret_cast<const float4v*>(p);
    for (int kz = 1; kz < kt; ++kz) sum += *reinterpret_cast<const float4v*>(p + (int64_t)kz * size);
#pragma unroll
    for (int q = 0; q < 4; ++q)
        if (r + q < R) store_y(y, y_dtype, (int64_t)t * ldy + y_off + r + q, sum[q] * h2f(gemm256_scale<false>(sc, r + q)));
}

// How a T x R output is cut: tiles of 64 mt token rows; whole rounds of whole tiles over the `cus` CUs, and the tiles of
// the last, partial round split over kt workgroups each (kt = 1: no split) while a part keeps at least 16 slabs.
struct Gemm256Plan { int mt, main_tiles, tail_tiles, kt; float us; };

// Tiles of 256 rows read least per product and are the ones for products of many rounds (8192^3: 880 us, 963 with 192 rows,
// 1019 with 128); where few tiles leave CUs idle, or most of a tile's rows are past the end, smaller ones win.  The plan with the
// least estimated time is taken.  A slab takes G_SLAB + G_SLAB_BUSY * (share of the CUs at work, squared) microseconds (the chip's power
// and its L2 set the pace when it is full), a round G_ENDS at its ends, and a split adds the partial tiles written and read back.  Fitted to every height in up
// to eight parts for 153 products of 260 to 2048 x 1500 to 38000 x 512 to 18944 (6 %), and then for the choice: what is taken is 0.4 % slower than the best of them in the
// mean.  With the times of an earlier kernel it was 1.0 %, up to 23: 902 x 1780 x 4416 36.7 us, now 29.8; 334 x 10325 x 4608 53.3 and 46.2; 372 x 5262 x 5248 39.3, 34.3;
// 1070 x 7033 x 15488 227, 201; 1382 x 3722 x 4480 60.2, 55.7; none of them slower.
// Up to eight parts, for few tiles of long rows (with up to four, now): 333 x 3584 x 18944 83, 71.  Parts of 8 slabs would gain 2
// us on short rows (520 x 1024 x 2048 22.5, 20.6) for twice the workspace.
constexpr double G_SLAB[5] = {0, 0, 0.449, 0.723, 0.979}, G_SLAB_BUSY[5] = {0, 0, 0.375, 0.404, 0.503}, G_ENDS = 9.8;

static Gemm256Plan gemm256_plan(int T, int R, int C, int cus, bool split) {
    const int slabs = (C + G_BK - 1) / G_BK;
    const bool rounds = cus >= 8 && cus % 8 == 0;
    const int n = rounds ? cus : 256;
    Gemm256Plan best{4, 0, 0, 1, 0.f};
    double best_t = 1e30;
    for (int mt = 4; mt >= 2; --mt) {
        const int64_t tiles = (int64_t)((T + gemm256_tokens(mt) - 1) / gemm256_tokens(mt)) * ((R + G_BN - 1) / G_BN);
        const int main = (int)(tiles / n) * n, tail = (int)(tiles - main);
        const double slab = G_SLAB[mt] + G_SLAB_BUSY[mt];
        for (int kt = 1; kt <= (split && rounds && tail ? 8 : 1); ++kt) {
            if (kt > 1 && slabs / kt < 16) break;
            const int wgs = tail * kt, of = (slabs + kt - 1) / kt;
            const double share = (double)(wgs % n) / n;
            double t = 2.5 + (double)(main / n) * (slabs * slab + G_ENDS) + (wgs / n) * (of * slab + G_ENDS);
            if (wgs % n) t += of * (G_SLAB[mt] + G_SLAB_BUSY[mt] * share * share) + G_ENDS;
            if (kt > 1) t += 0.1 + wgs * mt * 0.0124;
            if (t < best_t - 1e-9) {
                best_t = t;
                best = kt > 1 ? Gemm256Plan{mt, main, tail, kt, (float)t} : Gemm256Plan{mt, (int)tiles, 0, 1, (float)t};
            }
        }
    }
    return best;
}

size_t gemm256_part_bytes(int T, int R, int C, int cus) {
    const Gemm256Plan p = gemm256_plan(T, R, C, cus, true);
    return ((size_t)p.tail_tiles * p.kt * gemm256_tokens(p.mt) * G_BN * 4 + 255) & ~(size_t)255;
}

float gemm256_us(int T, int R, int C, int cus) { return gemm256_plan(T, R, C, cus, true).us; }     // (as estimated, see there)

bool gemm256_ok(int C, int64_t ldx, int64_t ldw, const void* x, const void* w) {
    return C % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0;
}

// x and w fp16.  `part` (gemm256_part_bytes) enables the split of the last round; NULL = no split.
int launch_gemm256(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, const Gemm256Scales& sc, void* y,
                   int y_dtype, int64_t ldy, int y_off, int T, int R, int C, float* part, int cus, hipStream_t s) {
    typedef void (*kernel_t)(Gemm256Args);
#define SQ_MT(MT) {{gemm256_kernel<SQ_F16, MT>, gemm256_kernel<SQ_BF16, MT>, gemm256_kernel<SQ_F32, MT>}, \
                   {gemm256_one_kernel<SQ_F16, MT>, gemm256_one_kernel<SQ_BF16, MT>, gemm256_one_kernel<SQ_F32, MT>}}
    static constexpr kernel_t kernels[3][2][3] = {SQ_MT(2), SQ_MT(3), SQ_MT(4)};
#undef SQ_MT
    static bool raised = false;
    if (!raised) {
        for (const auto& mt : kernels)
            for (const auto& one : mt)
                for (kernel_t k : one) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
        raised = true;
    }
    Gemm256Args a;
    a.x = x; a.w = w; a.sc = sc; a.y = y; a.ldx = ldx; a.ldw = ldw; a.ldy = ldy;
    a.T = T; a.R = R; a.C = C; a.y_off = y_off; a.y_dtype = y_dtype;
    const Gemm256Plan pl = gemm256_plan(T, R, C, cus, part != nullptr);
    a.tiles_t = (T + gemm256_tokens(pl.mt) - 1) / gemm256_tokens(pl.mt);
    a.tiles_r = (R + G_BN - 1) / G_BN;
    a.main_tiles = pl.main_tiles;
    a.kt = pl.kt;
    a.part = part;
    a.y_align = ((uintptr_t)y & 15) == 0 && ldy % 8 == 0 && y_off % 8 == 0 ? 16 : ((uintptr_t)y & 3) == 0 && ldy % 2 == 0 && y_off % 2 == 0 ? 4 : 2;
    const int per = (pl.main_tiles + 7) / 8 + (pl.tail_tiles * pl.kt + 7) / 8;       // an XCD's tiles and parts
    const int most = std::max(1, device_cus() / 8);
    const unsigned grid = (unsigned)(8 * std::min(per, most));
    hipLaunchKernelGGL(kernels[pl.mt - 2][per <= most][y_dtype == SQ_F32 ? 2 : y_dtype == SQ_BF16 ? 1 : 0], dim3(grid), dim3(G_WAVES * 64), gemm256_lds(pl.mt), s, a);
    int rc = check_launch("sq_linear_gemm(gemm256)");
    if (rc || pl.tail_tiles == 0) return rc;
    const unsigned blocks = (unsigned)(pl.tail_tiles * (gemm256_tokens(pl.mt) * G_BN / 1024));
    hipLaunchKernelGGL(gemm256_reduce_kernel, dim3(blocks), dim3(256), 0, s, part, pl.mt, pl.main_tiles, pl.kt,
                       a.tiles_t, a.tiles_r, T, R, sc, y, ldy, y_off, y_dtype);
    return check_launch("sq_linear_gemm(gemm256 reduce)");
}

int launch_bf16_to_f16(const uint16_t* x, int64_t ldx, int T, int C, uint16_t* out, hipStream_t s) {
    const int64_t n = ((int64_t)T * C + 7) / 8;
    hipLaunchKernelGGL(bf16_to_f16_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, ldx, T, C, out);
    return check_launch("sq_linear_gemm(bf16_to_f16)");
}

}  // namespace sq
