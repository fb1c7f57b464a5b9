// Host side of the product for 33 to 256 (384) activation rows (kernel: sq_mid.h): which stacks it takes, and how the work
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

struct MidPlan { int nt, tw, st, ks, nw; };

static int mid_units(const sq_matrix& m) { return m.W / (m.bits == 12 ? 3 : m.bits == 10 ? 5 : 4); }

// Variants: NT tiles of 16 activation rows (up to 256 rows; a 24-tile variant ran at half the rate), stages of four matrix steps
// or, where they do not fit beside the codebook, two.  A workgroup is 8 waves of a tile of weight rows, which a CU takes two of no
// faster than one after the other; where that is more workgroups than CUs, ten or twelve waves if one round is then enough, else
// two tiles per wave, which halves the activations' way through LDS.  18944 x 2 rows in 148 workgroups of 8 x 2 tiles / 237 of ten
// (198 of twelve at 128 and 192 activation rows), us, at 40 / 77 / 128 / 192: 10-bit tags 31 / 42 / 55 / 78 and 27 / 37 / 57 (not
// taken) / 71, 16-bit ones of width 8 100 / 109 / 115 / 142 and 90 / 96 / 105 / 135.  Fewer rows are cut along K until there is about one
// workgroup per CU, in slices of at least 512 columns (3584 x 3584 at 77 rows, 28 blocks: 28 us whole, 18 in seven).
static MidPlan mid_plan(const sq_matrix* mats, int n, int T, int cus) {
    MidPlan p{0, 1, 4, 1, 8};
    const int sizes[] = {3, 5, 8, 12, 16};
    for (int nt : sizes) if (T <= nt * 16) { p.nt = nt; break; }
    if (p.nt == 0) return p;
    const int tab = mats[0].d == 4 ? (mats[0].G << mats[0].bits) * 8 : 0;
    if (p.nt > 8 || tab + 2 * mid_stage_bytes(p.nt, 4) > 160 * 1024) p.st = 2;
    if (tab + 2 * mid_stage_bytes(p.nt, p.st) > 160 * 1024) { p.nt = 0; return p; }
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += mats[i].R;
    auto workgroups = [&](int nw) {
        int64_t w = 0;
        for (int i = 0; i < n; ++i) w += (mats[i].R + 16 * nw - 1) / (16 * nw);
        return w;
    };
    if (p.nt == 16 ? rows >= (int64_t)cus / 2 * 32 * 8 : workgroups(8) > cus) {
        if (p.nt <= 5 && workgroups(10) <= cus) p.nw = 10;
        else if (p.nt <= 12 && !(p.nt == 8 && mats[0].d == 4) && workgroups(12) <= cus) p.nw = 12;
        else p.tw = 2;
    }
    const int64_t blocks = (rows + 16 * p.nw * p.tw - 1) / (16 * p.nw * p.tw);
    p.ks = (int)std::max<int64_t>(1, std::min<int64_t>({cus / std::max<int64_t>(blocks, 1), 8, mats[0].C / 512}));
    return p;
}

// Activation rows one launch takes: all T, or half of them (whole tiles) where T is more than fits beside the codebook and where
// sixteen tiles of activations and two of weights need more registers than leave room to fetch ahead (18944 x 2 rows at 256
// activation rows, 12-bit tags: 133 us at once, 108 us in two; d = 8, bound by its gathers, 188 against 224).
static int mid_rows(const sq_matrix* mats, int n, int T) {
    for (int parts = 1; parts <= 2; ++parts) {
        const int rows = parts == 1 ? T : (T + 31) / 32 * 16;
        const MidPlan p = mid_plan(mats, n, rows, device_cus());
        if (p.nt && !(mats[0].d == 4 && p.nt == 16 && p.tw == 2)) return rows;
    }
    return 0;
}

// Activation rows up to which this is the faster way.  Decode + tile GEMM costs the decode once and a tile of 256 rows whatever is
// in it, so it is level at 256 rows (d = 8, 18944 x 2: 188 us here, 205 there) and ahead above, except for large d = 4 matrices,
// whose decode is the longest part (18944 x 2 rows at 384: 162 us here, 206 there; 3584 x 18944: 109 and 127; 3584 x 3584: 56
// and 49).
static int mid_limit(const sq_matrix* mats, int n) {
    int64_t weights = 0;
    for (int i = 0; i < n; ++i) weights += (int64_t)mats[i].R * mats[i].C;
    return mats[0].d == 4 && weights >= (int64_t)1 << 26 ? 384 : 256;
}

static size_t mid_part_bytes(const sq_matrix& m, int T, int ks) { return ks > 1 ? (((size_t)ks * T * m.R * 4) + 255) & ~(size_t)255 : 0; }

// the pieces share format, row length and codebook size, and the kernel takes them at T rows
bool mid_ok(const sq_matrix* mats, int n, int T) {
    if (n < 1 || n > MID_PIECES || T <= SQ_SMALL_BMAX) return false;
    for (int i = 0; i < n; ++i) {
        const sq_matrix &m = mats[i], &m0 = mats[0];
        if (!mma_shape(m) || m.R <= 0 || m.d != m0.d || m.bits != m0.bits || m.W != m0.W || m.G != m0.G) return false;
        if (m.d == 4 && ((int64_t)m.G << m.bits) * 8 > 128 * 1024) return false;
        if (((int64_t)m.R + 16) * m.W * 4 >= ((int64_t)1 << 32)) return false;                 // 32-bit offsets
        if (m.d == 8 && ((int64_t)m.G << m.bits) * 16 > ((int64_t)1 << 31)) return false;
    }
    return T <= mid_limit(mats, n) && mid_rows(mats, n, T) != 0;
}

size_t mid_workspace(const sq_matrix* mats, int n, int T) {
    const MidPlan p = mid_plan(mats, n, mid_rows(mats, n, T), device_cus());
    size_t need = 0;
    for (int i = 0; i < n; ++i) need += mid_part_bytes(mats[i], mid_rows(mats, n, T), p.ks);
    return need;
}

static int launch_mid_rows(const sq_matrix* mats, int n, const MidPlan& pl, const void* const* dense, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype,
                           int64_t ldy, int T, void* ws, hipStream_t s, bool wide = false) {
    MidArgs a{};
    const sq_matrix& m0 = mats[0];
    a.n = n;
    a.x = (const uint16_t*)x; a.ldx = ldx; a.y = y; a.ldy = ldy; a.T = T; a.x_dtype = x_dtype; a.y_dtype = y_dtype;
    a.U = dense ? m0.C / 8 : mid_units(m0); a.ks = pl.ks;
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
        wg += ((m.R + 16 * pl.nw * pl.tw - 1) / (16 * pl.nw * pl.tw)) * pl.ks;
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
    MidPlan p{0, 1, 4, 1, 8};
    const int sizes[] = {1, 3, 5, 8, 12, 16};
    for (int nt : sizes) if (T <= nt * 16) { p.nt = nt; break; }
    if (p.nt > 8) p.st = 2;
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

size_t mid_dense_workspace(const sq_matrix* mats, int n, int T) {
    const MidPlan p = mid_dense_plan(mats, n, T, device_cus());
    size_t need = 0;
    for (int i = 0; i < n; ++i) need += mid_part_bytes(mats[i], T, p.ks);
    return need;
}

int launch_mid_decoded(const sq_matrix* mats, int n, const void* const* w, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T,
                       void* ws, hipStream_t s, bool wide) {
    return launch_mid_rows(mats, n, mid_dense_plan(mats, n, T, device_cus()), w, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, s, wide);
}

int launch_mid(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws,
               size_t ws_bytes, hipStream_t s) {
    if (mid_workspace(mats, n, T) > ws_bytes) return fail(SQ_EWORKSPACE, "sq_linear_gemm: workspace %zu < %zu", ws_bytes, mid_workspace(mats, n, T));
    const int rows = mid_rows(mats, n, T);
    const MidPlan pl = mid_plan(mats, n, rows, device_cus());
    for (int t = 0; t < T; t += rows) {
        const int rc = launch_mid_rows(mats, n, pl, nullptr, (const char*)x + (size_t)t * ldx * 2, x_dtype, ldx,
                                       (char*)y + (size_t)t * ldy * (y_dtype == SQ_F32 ? 4 : 2), y_dtype, ldy, std::min(rows, T - t), ws, s);
        if (rc) return rc;
    }
    return SQ_OK;
}

}  // namespace sq
