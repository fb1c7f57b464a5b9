// Host side of the product for 33 and more activation rows, and d = 4 from 17 on (kernel: sq_mid.h): which stacks it takes, and how the work
// is cut.
#include <algorithm>
#include "sq_mid.h"
#include "sq_slices.h"

namespace sq {

int launch_mid_b16d8(const MidArgs&, int, int, int, int, int, hipStream_t);
int launch_mid_b12d4(const MidArgs&, int, int, int, int, int, hipStream_t);
int launch_mid_b10d4(const MidArgs&, int, int, int, int, int, hipStream_t);
int launch_mid_b8d4(const MidArgs&, int, int, int, int, int, hipStream_t);
int launch_mid_dense(const MidArgs&, int, int, int, int, int, hipStream_t);

static int mid_units(const sq_matrix& m) { return m.W / (m.bits == 12 ? 3 : m.bits == 10 ? 5 : 4); }

// The variants: workgroups of NW waves, each with TW tiles of 16 weight rows x NT tiles of 16 activation rows, those of a stack cut into
// blocks of NT; and K slices, whose sums cost a launch.  Which one is taken is estimated from what a workgroup's matrix steps cost its CU
// (products, reads of activations by every wave, codewords, activations on their way into LDS) and how long a step takes that waits for nothing
// but itself, as the constants below say; d = 8 also from the rate at which L2 serves the whole chip's codewords.  They are fitted to 1852 products
// of 200 .. 30000 rows of 512 .. 18944 columns at 33 .. 2048 activation rows in 10 to 130 cuts each, to 10 %
// (single tiles take 14 % longer than they say); the cut that is taken then is 2 % slower than the best one in the mean, in one case of ten by 9 % (d = 4),
// 6 % (d = 8).  In one block of all activation rows and eight waves,
// the cut of before, and so, us (77 / 228 / 700 activation rows, beyond 256 decoded and in tiles before):
//   rows x columns   12-bit tags, d = 4                              16-bit tags, d = 8
//   512 x 512        8.4 / 15.7 / 15.4     4.7 / 4.8 / 5.4           9.0 / 15.6 / 14.7     5.3 / 5.9 / 7.0
//   1024 x 896      11.2 / 23.6 / 19.9     5.7 / 5.8 / 8.2          12.0 / 23.0 / 19.2     7.3 / 8.3 / 12.5
//   4096 x 1024     12.3 / 23.4 / 23.6     6.6 / 8.8 / 13.7         13.8 / 24.0 / 25.0    10.0 / 17.2 / 23.7
//   3584 x 3584     15.8 / 30.5 / 45.0    13.3 / 18.8 / 30.9        21.6 / 36.1 / 46.8    21.8 / 36.3 / 68.6 (not taken)
//   8000 x 2048     17.6 / 35.1 / 40.4    11.3 / 16.5 / 35.7
// us: a launch; staged codebooks per KB and round of workgroups; per matrix step of a workgroup: a wave's product, its read of a tile of
// activations, a tile of codewords, a tile of activations staged; a step by itself, per tile, and per tile that a wave stages; slices: their launch, and per million sums;
// per million results; per tile of codewords over the chip
struct MidCost { float launch, table, product, read, words, stage, wait, wait_tile, wait_stage, slices, sums, results, chip; };
static constexpr MidCost MID_COST4 = {4.04f, 0.0179f, 0.00132f, 0.00139f, 0.00346f, 0.00832f, 0.0385f, 0.0083f, 0.0362f, 3.14f, 3.16f, 1.86f, 2.1e-5f};
static constexpr MidCost MID_COST8 = {3.49f, 0.f, 0.00198f, 0.00198f, 0.0168f, 0.0109f, 0.0121f, 0.f, 0.f, 3.38f, 2.87f, 1.09f, 2.74e-4f};

static int64_t mid_blocks(const sq_matrix* mats, int n, int rows) {       // of `rows` weight rows
    int64_t w = 0;
    for (int i = 0; i < n; ++i) w += (uint32_t)(mats[i].R + rows - 1) / (uint32_t)rows;
    return w;
}
static int mid_lds(const MidVariant& v, int table) { return table + 2 * mid_stage_bytes(v.nt, v.st); }

static size_t mid_part_bytes(const sq_matrix& m, int T, int ks) { return ks > 1 ? (((size_t)ks * T * m.R * 4) + 255) & ~(size_t)255 : 0; }
static size_t mid_sums_bytes(const sq_matrix* mats, int n, int T, int ks) {
    size_t need = 0;
    for (int i = 0; i < n; ++i) need += mid_part_bytes(mats[i], T, ks);
    return need;
}

// What the estimate needs of a variant alone
struct MidTerms { float step, wait, chip; int beside, rows; };          // rows: of a workgroup's weights, as a place in mid_cut's list of blocks
template <size_t N> struct MidTermsOf { MidTerms t[N]; };
template <size_t N>
static constexpr MidTermsOf<N> mid_terms(const MidVariant (&vs)[N], const MidCost& c) {
    MidTermsOf<N> r{};
    for (size_t k = 0; k < N; ++k) {
        const MidVariant v = vs[k];
        r.t[k].step = (v.nw + 3) / 4 * 4 * v.tw * (c.product * v.nt + c.words) + c.read * v.nw * v.nt + c.stage * v.nt;      // (ten waves: three on a SIMD)
        r.t[k].wait = c.wait + c.wait_tile * v.nt * v.tw + c.wait_stage * v.nt / v.nw;
        r.t[k].chip = v.nw * v.tw * c.chip;
        r.t[k].beside = std::max(1, std::min(4 * (512 / (40 + 6 * v.nt + 4 * v.nt * v.tw)) / v.nw, 32 / v.nw));              // workgroups that a CU's registers hold side by side
        r.t[k].rows = v.tw == 2 ? 4 : v.nw == 4 ? 0 : v.nw == 8 ? 1 : v.nw == 10 ? 2 : 3;
    }
    return r;
}
static constexpr auto MID_TERMS4 = mid_terms(MID4, MID_COST4);
static constexpr auto MID_TERMS8 = mid_terms(MID8, MID_COST8);

// The cut with the least estimated time whose sums of slices take at most `room` bytes.  (Every call plans; what the matrix steps alone, spread evenly, rule
// out is not looked at any further.)
static MidPlan mid_cut(const sq_matrix* mats, int n, int T, size_t room) {
    const bool d4 = mats[0].d == 4;
    const int cus = device_cus(), table = d4 ? (mats[0].G << mats[0].bits) * 8 : 0, pairs = ((mid_units(mats[0]) + 3) / 4 + 1) / 2;   // of rounds
    const MidCost& c = d4 ? MID_COST4 : MID_COST8;
    const MidVariant* vs = d4 ? MID4 : MID8;
    const MidTerms* terms = d4 ? MID_TERMS4.t : MID_TERMS8.t;
    const int count = d4 ? (int)std::size(MID4) : (int)std::size(MID8);
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += mats[i].R;
    const float results = (float)rows * T * 1e-6f, pair_steps = mats[0].bits == 12 ? 8.f : 16.f, fixed = c.launch + c.results * results;
    const float even = pair_steps * pairs / cus;                          // matrix steps of a workgroup whose row is one slice, per CU
    // blocks of weight rows, and of activation rows by tiles
    const int64_t blocks[5] = {mid_blocks(mats, n, 64), mid_blocks(mats, n, 128), mid_blocks(mats, n, 160), mid_blocks(mats, n, 192), mid_blocks(mats, n, 256)};
    auto over = [](int64_t a, int b) { return a >> 32 ? a / b : (int64_t)((uint32_t)a / (uint32_t)b); };
    MidPlan best{0, 1, 8, 4, 1, 1e30f};
    for (int k = 0; k < count; ++k) {
        const MidVariant& v = vs[k];
        const MidTerms& t = terms[k];
        const int64_t whole = blocks[t.rows] * (int64_t)((uint32_t)(T + 16 * v.nt - 1) / (uint32_t)(16 * v.nt));
        if (fixed + whole * even * t.step * 0.9999f >= best.us) continue;
        const int lds = mid_lds(v, table);
        if (lds > 160 * 1024 || (v.st == 2 && v.nt <= 8 && mid_lds({v.nt, v.tw, v.nw, 4}, table) <= 160 * 1024)) continue;
        if (v.nt > 3 && v.nt * 16 >= 2 * T) continue;                     // (more than half of it past the last row)
        if (!d4 && v.tw == 2 && whole < cus) continue;                    // (bound by its codewords, two tiles of which a wave cannot fetch far enough ahead)
        const int beside = std::max(1, std::min(160 * 1024 / lds, t.beside)), most = whole > cus ? 1 : std::min({cus / (int)whole, 8, pairs});
        for (int cut = 0; cut < 3; ++cut) {
            const int ks = cut == 0 ? 1 : cut == 1 ? most : most / 2;
            if (cut && ks < 2) continue;
            const int64_t wgs = whole * ks, rounds = over(wgs + cus - 1, cus);
            const float s = pair_steps * ((pairs + ks - 1) / ks), work = rounds * s * t.step, sums = ks > 1 ? c.slices + c.sums * ks * results : 0.f;
            if (fixed + work + sums >= best.us) continue;
            const int64_t waits = over(rounds + beside - 1, beside);
            const float wait = waits * s * t.wait, chip = wgs * s * t.chip;
            const float us = fixed + c.table * (table >> 10) * waits + (v.nt == 1 ? 1.14f : 1.f) * __builtin_sqrtf(work * work + wait * wait + chip * chip) + sums;
            if (us < best.us && (ks == 1 || mid_sums_bytes(mats, n, T, ks) <= room)) best = {v.nt, v.tw, v.nw, v.st, ks, us};
        }
    }
    return best;
}

// the pieces share format, row length and codebook size, and the kernel takes them
static bool mid_shape(const sq_matrix* mats, int n, int T) {
    if (n < 1 || n > MID_PIECES || T < 1) return false;
    for (int i = 0; i < n; ++i) {
        const sq_matrix &m = mats[i], &m0 = mats[0];
        if (!mma_shape(m) || m.R <= 0 || m.d != m0.d || m.bits != m0.bits || m.W != m0.W || m.G != m0.G) return false;
        if (m.d == 4 && ((int64_t)m.G << m.bits) * 8 > 128 * 1024) return false;
        if (((int64_t)m.R + 16) * m.W * 4 >= ((int64_t)1 << 32)) return false;                 // 32-bit offsets
        if (m.d == 8 && ((int64_t)m.G << m.bits) * 16 > ((int64_t)1 << 31)) return false;
    }
    return true;
}

// Activation rows that always run here: 256, and 384 of large d = 4 matrices.
static int mid_limit(const sq_matrix* mats, int n) {
    int64_t weights = 0;
    for (int i = 0; i < n; ++i) weights += (int64_t)mats[i].R * mats[i].C;
    return mats[0].d == 4 && weights >= (int64_t)1 << 26 ? 384 : 256;
}

bool mid_ok(const sq_matrix* mats, int n, int T) { return T > SQ_SMALL_BMAX && mid_shape(mats, n, T) && T <= mid_limit(mats, n); }

// What a workspace has to hold up to there: the sums of as many slices as the kernel took when a launch had one block of all activation
// rows (or half of them).  Cuts that need more than there is are passed over.
size_t mid_least(const sq_matrix* mats, int n, int T) {
    const int cus = device_cus(), table = mats[0].d == 4 ? (mats[0].G << mats[0].bits) * 8 : 0;
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += mats[i].R;
    for (int parts = 1; parts <= 2; ++parts) {
        const int t = parts == 1 ? T : (T + 31) / 32 * 16, nt = t <= 48 ? 3 : t <= 80 ? 5 : t <= 128 ? 8 : t <= 192 ? 12 : 16;
        int nw = 8, tw = 1;
        if (t > 256 || table + 2 * mid_stage_bytes(nt, 2) > 160 * 1024) continue;
        if (nt == 16 ? rows >= (int64_t)cus / 2 * 32 * 8 : mid_blocks(mats, n, 16 * 8) > cus) {
            if (nt <= 5 && mid_blocks(mats, n, 16 * 10) <= cus) nw = 10;
            else if (nt <= 12 && !(nt == 8 && mats[0].d == 4) && mid_blocks(mats, n, 16 * 12) <= cus) nw = 12;
            else tw = 2;
        }
        if (mats[0].d == 4 && nt == 16 && tw == 2) continue;
        const int64_t blocks = (rows + 16 * nw * tw - 1) / (16 * nw * tw);
        const int ks = (int)std::max<int64_t>(1, std::min<int64_t>({cus / std::max<int64_t>(blocks, 1), 8, mats[0].C / 512}));
        return mid_sums_bytes(mats, n, t, ks);
    }
    return 0;
}

// (a decode step's sums are those that sq_linear_small_noalloc has room for)
static size_t mid_room(int T, size_t room) { return T <= SQ_SMALL_BMAX ? std::min(room, SMALL_ROOM) : room; }

MidPlan mid_plan(const sq_matrix* mats, int n, int T, size_t room) {
    return mid_shape(mats, n, T) ? mid_cut(mats, n, T, mid_room(T, room)) : MidPlan{0, 1, 8, 4, 1, 1e30f};
}

size_t mid_workspace(const sq_matrix* mats, int n, int T, const MidPlan* planned) {
    const size_t need = mid_sums_bytes(mats, n, T, planned && planned->nt ? planned->ks : mid_plan(mats, n, T).ks);
    return T > SQ_SMALL_BMAX && T <= mid_limit(mats, n) ? std::max(need, mid_least(mats, n, T)) : need;
}

// For tests: the cut that a stack takes at T rows, as token tiles | weight tiles << 8 | waves << 16 | K slices << 24; 0: the kernel does not take it.
extern "C" __attribute__((visibility("default"))) int32_t sq_mid_variant_for_tests(const sq_matrix* mats, int32_t n, int32_t T) {
    const MidPlan p = mid_plan(mats, n, T);
    return p.nt ? p.nt | p.tw << 8 | p.nw << 16 | p.ks << 24 : 0;
}

static int launch_mid_rows(const sq_matrix* mats, int n, const MidPlan& pl, const void* const* dense, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype,
                           int64_t ldy, int T, void* ws, hipStream_t s, bool wide = false) {
    MidArgs a{};
    const sq_matrix& m0 = mats[0];
    a.n = n;
    a.x = (const uint16_t*)x; a.ldx = ldx; a.y = y; a.ldy = ldy; a.T = T; a.x_dtype = x_dtype; a.y_dtype = y_dtype;
    a.U = dense ? m0.C / 8 : mid_units(m0); a.ks = pl.ks; a.tbs = (T + 16 * pl.nt - 1) / (16 * pl.nt);
    a.wide = wide;
    a.table_bytes = !dense && m0.d == 4 ? (m0.G << m0.bits) * 8 : 0;
    int wg = 0;
    char* part = (char*)ws;
    for (int i = 0; i < n; ++i) {
        MidPiece& P = a.p[i];
        const sq_matrix& m = mats[i];
        P.m = m;
        P.w = dense ? dense[i] : m.stream && tiled_format_ok(m.R, m.W, m.C, m.d, m.bits) && ((uintptr_t)m.stream & 15) == 0 ? (const void*)m.stream : nullptr;
        P.part = (float*)part;
        part += mid_part_bytes(m, T, pl.ks);
        P.wg0 = wg;
        wg += ((m.R + 16 * pl.nw * pl.tw - 1) / (16 * pl.nw * pl.tw)) * pl.ks * a.tbs;
    }
    int rc = SQ_EUNSUPPORTED;
    if (dense) rc = launch_mid_dense(a, pl.nt, pl.tw, pl.st, pl.nw, wg, s);
    else if (m0.d == 8) rc = launch_mid_b16d8(a, pl.nt, pl.tw, pl.st, pl.nw, wg, s);
    else if (m0.bits == 12) rc = launch_mid_b12d4(a, pl.nt, pl.tw, pl.st, pl.nw, wg, s);
    else if (m0.bits == 10) rc = launch_mid_b10d4(a, pl.nt, pl.tw, pl.st, pl.nw, wg, s);
    else if (m0.bits == 8) rc = launch_mid_b8d4(a, pl.nt, pl.tw, pl.st, pl.nw, wg, s);
    if (rc || pl.ks == 1) return rc;
    return launch_slice_sum(a.p, n, a.ks, T, y, y_dtype, ldy, s);
}

// For decoded weights: one tile of rows per wave, so that small stacks spread (593 x 1984 at 16 rows: 17 us with the decode, 22
// with two), K slices of 256 columns at least, up to eight (3584 x 18944 at 64 rows: 99 us with the decode, 119 in four slices,
// 111 in nine).
static MidPlan mid_dense_plan(const sq_matrix* mats, int n, int T, int cus) {
    MidPlan p{0, 1, 8, 4, 1, 0.f};
    for (const MidVariant& v : MID_DENSE) if (T <= v.nt * 16) { p.nt = v.nt; p.st = v.st; break; }
    int64_t blocks = 0;
    for (int i = 0; i < n; ++i) blocks += (mats[i].R + 16 * 8 - 1) / (16 * 8);
    p.ks = (int)std::max<int64_t>(1, std::min<int64_t>({cus / std::max<int64_t>(blocks, 1), 8, mats[0].C / 256}));
    return p;
}

bool mid_dense_ok(const sq_matrix* mats, int n, int T) {
    if (n < 1 || n > MID_PIECES || T < 1 || T > 256) return false;
    for (int i = 0; i < n; ++i)
        if (mats[i].R <= 0 || mats[i].C != mats[0].C || mats[i].C % 8 || ((int64_t)mats[i].R + 16) * mats[i].C * 2 >= ((int64_t)1 << 32)) return false;
    return true;
}

size_t mid_dense_workspace(const sq_matrix* mats, int n, int T) { return mid_sums_bytes(mats, n, T, mid_dense_plan(mats, n, T, device_cus()).ks); }

int launch_mid_decoded(const sq_matrix* mats, int n, const void* const* w, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T,
                       void* ws, hipStream_t s, bool wide) {
    return launch_mid_rows(mats, n, mid_dense_plan(mats, n, T, device_cus()), w, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, s, wide);
}

int launch_mid(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws,
               size_t ws_bytes, hipStream_t s, const MidPlan* planned) {
    const bool kept = planned && planned->nt && (planned->ks == 1 || mid_sums_bytes(mats, n, T, planned->ks) <= ws_bytes);
    return launch_mid_rows(mats, n, kept ? *planned : mid_plan(mats, n, T, ws_bytes), nullptr, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, s);
}

}  // namespace sq
