// Prefill product Y[T, R] = X[T, C] . W^T on fp16 MFMA (v_mfma_f32_32x32x16_f16), fp32 accumulate.
//
// The MFMA's B operand wants, per lane, 8 consecutive k of one weight row: exactly one d = 8
// codeword (or two d = 4 codewords), so a weight tile is "dequantised" by gathering raw fp16
// codewords into an LDS tile; the row scale multiplies the fp32 accumulator in the epilogue,
// which keeps the tile exact.  bf16 activations are converted to fp16 while they are staged
// (exact for every fp16-normal value); fp16 MFMA runs at the bf16 rate on gfx950 and keeps the
// codewords' 11-bit significands, which bf16 tiles would cut to 8.
//
// Operand layout of v_mfma_f32_32x32x16_f16 (A: 32 x 16, B: 16 x 32, D: 32 x 32), lane l:
//   A: row l % 32, k = 8 * (l / 32) .. + 7        (tokens)
//   B: col l % 32, k = 8 * (l / 32) .. + 7        (weight rows)
//   D[v], v = 0..15: row 8 * (v / 4) + 4 * (l / 32) + v % 4, col l % 32
#include <algorithm>
#include <cmath>
#include "sq_common.h"

namespace sq {

constexpr int BM = 128, BN = 128, BK = 32, LDT = BK + 8;   // LDT: padded LDS row stride (halves)

struct GemmArgs {
    sq_matrix m;          // codebook piece (fused) ...
    const uint16_t* wd;   // ... or dense weight [R, C] with row stride ldw (m.R, m.C, m.y_off still valid)
    int64_t ldw;
    const uint16_t* x;
    int64_t ldx;
    void* y;
    int64_t ldy;
    int T;
    int x_dtype, y_dtype, w_dtype;   // w_dtype: element type of wd
};

// 8 consecutive halves of activation row t starting at column k (zeros outside the matrix)
__device__ __forceinline__ u32x4 load_x8(const GemmArgs& a, int t, int k) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (t < a.T && k < a.m.C) {
        v = *reinterpret_cast<const u32x4*>(a.x + (int64_t)t * a.ldx + k);
        if (a.x_dtype == SQ_BF16) { v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w); }
    }
    return v;
}

// 8 consecutive raw weights (unscaled codewords, or dense halves) of row r starting at column k
template <int D, bool DENSE>
__device__ __forceinline__ u32x4 load_w8(const GemmArgs& a, int r, int k) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (r >= a.m.R || k >= a.m.C) return v;
    if (DENSE) {
        v = *reinterpret_cast<const u32x4*>(a.wd + (int64_t)r * a.ldw + k);
        if (a.w_dtype == SQ_BF16) { v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w); }
        return v;
    }
    const sq_matrix& m = a.m;
    const uint32_t* row = reinterpret_cast<const uint32_t*>(m.tags) + (int64_t)r * m.W;
    const uint32_t boff = m.row_book ? (uint32_t)m.row_book[r] << m.bits : 0u;
    if (D == 8) {
        const uint32_t tag = tag_at(row, m.W, m.bits, k >> 3) + boff;
        v = *reinterpret_cast<const u32x4*>(m.table + (size_t)tag * 8);
    } else {
        const uint32_t t0 = tag_at(row, m.W, m.bits, k >> 2) + boff;
        const uint32_t t1 = tag_at(row, m.W, m.bits, (k >> 2) + 1) + boff;
        const u32x2 c0 = *reinterpret_cast<const u32x2*>(m.table + (size_t)t0 * 4);
        const u32x2 c1 = *reinterpret_cast<const u32x2*>(m.table + (size_t)t1 * 4);
        v.x = c0.x; v.y = c0.y; v.z = c1.x; v.w = c1.y;
    }
    return v;
}

template <int D, bool DENSE>
__global__ __launch_bounds__(256) void gemm_kernel(GemmArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t sx[BM * LDT];
    __shared__ __attribute__((aligned(16))) uint16_t sw[BN * LDT];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t0 = blockIdx.y * BM, r0 = blockIdx.x * BN;
    const int wm = (wave >> 1) * 64, wn = (wave & 1) * 64;     // wave tile origin inside the block tile
    float16v acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    // staging assignment: 512 16-byte pieces per tile, two per thread
    const int sr0 = tid >> 2, sk = (tid & 3) * 8;              // rows sr0 and sr0 + 64, columns sk .. sk + 7
    u32x4 px[2], pw[2];
    px[0] = load_x8(a, t0 + sr0, sk);
    px[1] = load_x8(a, t0 + sr0 + 64, sk);
    pw[0] = load_w8<D, DENSE>(a, r0 + sr0, sk);
    pw[1] = load_w8<D, DENSE>(a, r0 + sr0 + 64, sk);

    for (int k0 = 0; k0 < a.m.C; k0 += BK) {
        __syncthreads();
        *reinterpret_cast<u32x4*>(sx + sr0 * LDT + sk) = px[0];
        *reinterpret_cast<u32x4*>(sx + (sr0 + 64) * LDT + sk) = px[1];
        *reinterpret_cast<u32x4*>(sw + sr0 * LDT + sk) = pw[0];
        *reinterpret_cast<u32x4*>(sw + (sr0 + 64) * LDT + sk) = pw[1];
        __syncthreads();
        if (k0 + BK < a.m.C) {                                  // next tile's loads fly during the MFMAs
            px[0] = load_x8(a, t0 + sr0, k0 + BK + sk);
            px[1] = load_x8(a, t0 + sr0 + 64, k0 + BK + sk);
            pw[0] = load_w8<D, DENSE>(a, r0 + sr0, k0 + BK + sk);
            pw[1] = load_w8<D, DENSE>(a, r0 + sr0 + 64, k0 + BK + sk);
        }
#pragma unroll
        for (int kk = 0; kk < BK; kk += 16) {
            half8v fa[2], fb[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
                fa[i] = *reinterpret_cast<const half8v*>(sx + (wm + i * 32 + (lane & 31)) * LDT + kk + (lane >> 5) * 8);
#pragma unroll
            for (int j = 0; j < 2; ++j)
                fb[j] = *reinterpret_cast<const half8v*>(sw + (wn + j * 32 + (lane & 31)) * LDT + kk + (lane >> 5) * 8);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], fb[j], acc[i][j], 0, 0, 0);
        }
    }

    // epilogue: row scale on the accumulator, one rounding to the output type
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int r = r0 + wn + j * 32 + (lane & 31);
        if (r >= a.m.R) continue;
        const float sc = a.m.row_scale ? h2f(a.m.row_scale[r]) : 1.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int t = t0 + wm + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                if (t >= a.T) continue;
                const float val = acc[i][j][v] * sc;
                const int64_t o = (int64_t)t * a.ldy + a.m.y_off + r;
                if (a.y_dtype == SQ_BF16) reinterpret_cast<uint16_t*>(a.y)[o] = f2bf(val);
                else if (a.y_dtype == SQ_F16) reinterpret_cast<uint16_t*>(a.y)[o] = f2h(val);
                else reinterpret_cast<float*>(a.y)[o] = val;
            }
    }
}

// ------------------------------------------------------------------------------------------ host

int launch_small_generic(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y,
                         int y_dtype, int64_t ldy, int B, hipStream_t s);

bool gemm256_ok(int C, int64_t ldx, int64_t ldw, const void* x, const void* w);
size_t gemm256_part_bytes(int T, int R, int C, int cus);
float gemm256_us(int T, int R, int C, int cus);
int launch_gemm256(const uint16_t* x, int64_t ldx, const uint16_t* w, int64_t ldw, const Gemm256Scales& sc, void* y,
                   int y_dtype, int64_t ldy, int y_off, int T, int R, int C, float* part, int cus, hipStream_t s);
int launch_dequant_with_cvt(const sq_matrix& m, void* out, int64_t ld_out, const uint16_t* x, int64_t ldx, int T, int C,
                            uint16_t* xout, hipStream_t s);

static bool x_vec_ok(const void* x, int64_t ldx, int C) { return C % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x & 15) == 0; }
// Activation rows from which the large-tile route (decode each piece once into the workspace as raw fp16
// codewords, then the 256 x 256 tile GEMM with the row scale in its epilogue) replaces the fused 128 x 128
// kernel, which re-gathers every codeword once per 128 activation rows.  It also wins below 256 rows (7B layer,
// 64 rows: 0.60 ms against 1.90 ms on the fused kernel, whose grid is then a few dozen workgroups), so it is
// used from the first row count sq_linear_small does not take.
constexpr int GEMM256_MIN_T = SQ_SMALL_BMAX + 1;
static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
static bool fused_ok(const sq_matrix& m) { return m.tags && (m.d == 8 || m.d == 4) && !m.perms && ((uintptr_t)m.table & 15) == 0; }
static size_t dense_bytes(const sq_matrix& m) { return (((size_t)m.R * m.C * 2) + 255) & ~(size_t)255; }

// The decode + 256 x 256 tile route: from GEMM256_MIN_T rows, and for stacks with column orders at any row count
// (their decode-time kernel is the slow one: 27B-shaped layer with 16 orders, 880 us at 16 rows and 1746 us at 32
// against 625 us here).  Rows that end within a slab of 64 columns take it from BROKEN_DECODED_T on, up to where they are decoded in steps
// of bounded workspace (5120 x 2080: 34-38 us there at 200 rows, 38-44 here at 400; in the 128 x 128 kernel 80-120).
constexpr int BROKEN_DECODED_T = 256;
bool has_orders(const sq_matrix* mats, int n) {
    for (int i = 0; i < n; ++i)
        if (mats[i].perms) return true;
    return false;
}

static bool big_route(const sq_matrix* mats, int n, int T) {
    if (mats[0].C % 64) return mats[0].C % 8 == 0 && T > BROKEN_DECODED_T;
    return T >= GEMM256_MIN_T || has_orders(mats, n);
}

// Pieces that are neighbours in Y are decoded one behind the other and multiplied in ONE tile GEMM over all their
// rows: a 512-row k or v projection alone is 2 tiles of 256 rows, a
// launch that leaves the chip idle (7B q|k|v at 64-255 rows: 139 us as three products, the o projection of q's
// size: 62 us; 8 pieces of 1024 x 3584 at 333 / 1024 / 2048 rows, 16-bit tags of width 8: 257 / 267 / 304 us one by one,
// 90 / 106 / 148 in one).
constexpr size_t STACK_MAX_BYTES = (size_t)1 << 30;
static bool stacked_route(const sq_matrix* mats, int n) {
    if (n < 2) return false;
    size_t tot = 0;
    for (int i = 0; i < n; ++i) {
        if (mats[i].R <= 0) return false;
        if (i + 1 < n && mats[i + 1].y_off != mats[i].y_off + mats[i].R) return false;
        tot += dense_bytes(mats[i]);
    }
    return tot <= STACK_MAX_BYTES;
}
static int stacked_rows(const sq_matrix* mats, int n) {
    int r = 0;
    for (int i = 0; i < n; ++i) r += mats[i].R;
    return r;
}
static size_t stacked_bytes(const sq_matrix* mats, int n) {
    size_t b = 0;
    for (int i = 0; i < n; ++i) b += dense_bytes(mats[i]);
    return b;
}

// Up to 256 activation rows of what cannot go in one pass over the tags (sq_mid.h): column orders, formats whose rows are not
// whole lane units, codebooks too large for it.  Rows are decoded and multiplied straight from there, as many at a time as
// DECODED_BYTES of workspace hold, evenly cut and across the ends of pieces.  192 MB: what has just been decoded is then still in
// the 256 MB last-level cache when it is multiplied, and the stacks and matrices below it, whose K is cut less the fewer rows a
// step has, stay in one (37888 rows of 3592 columns in two steps instead of one at 40 / 128 / 256 rows 156 / 173 / 254 us instead
// of 215 / 239 / 319, in three 177 / 199 / 275; 34816 x 5128 198 / 230 / 342 instead of 303 / 333 / 435; 5120 x 17416 whole 91 /
// 102 / 133, in two 117 / 136 / 188).
constexpr size_t DECODED_BYTES = (size_t)192 << 20;
struct DecodedRows { sq_matrix m[MID_PIECES]; const sq_matrix* of[MID_PIECES]; int r0[MID_PIECES], n; size_t bytes; };

static int decoded_step_rows(const sq_matrix* mats, int n) {
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += mats[i].R;
    const int64_t bytes = rows * mats[0].C * 2, steps = std::max<int64_t>(1, (bytes + DECODED_BYTES - 1) / DECODED_BYTES);
    return (int)std::max<int64_t>(128, (rows + steps * 128 - 1) / (steps * 128) * 128);     // (also where all pieces are empty)
}

// The step that begins at row r0 of piece i, each of its parts as a piece of its own to the kernel (which reads the scales and
// the place in Y of decoded rows, not their tags); i and r0 move behind it.
static DecodedRows decoded_step(const sq_matrix* mats, int n, int& i, int& r0) {
    DecodedRows d;
    d.n = 0; d.bytes = 0;
    int left = decoded_step_rows(mats, n);
    while (i < n && d.n < MID_PIECES && left > 0) {
        const int R = std::min(mats[i].R - r0, left);
        if (R > 0) {
            sq_matrix& m = d.m[d.n] = mats[i];
            m.R = R; m.row_scale += r0; m.y_off += r0;
            d.of[d.n] = mats + i;
            d.r0[d.n++] = r0;
            d.bytes += dense_bytes(m);
        }
        left -= R;
        r0 += R;
        if (r0 >= mats[i].R) ++i, r0 = 0;
    }
    return d;
}

// Where the tile GEMM, whose workgroups read less, is the faster one behind the same decode: with more rows than half the CUs'
// worth of 256-row tiles, and from 129 activation rows for 24 M weights and more (there and here, us: 37888 x 3584 at 64 rows 216
// and 248; 30000 x 3584 at 128 / 200 / 256 rows 164 / 154 / 153 and 138 / 169 / 173, 18944 x 3584 96 / 107 / 108 and 103 / 128 /
// 127, 3584 x 18944 107 / 116 / 120 and 112 / 131 / 134, 4608 x 3584 44 / 46 / 47 and 40 / 46 / 49, 593 x 1984 41 / 41 / 41 and
// 26 / 32 / 34).
static bool decoded_route(const sq_matrix* mats, int n, int T) {
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) {
        rows += mats[i].R;
        if (mats[i].R > 0 && (!mats[i].tags || !mid_dense_ok(mats + i, 1, T))) return false;
    }
    if (mats[0].C % 64) return true;
    return rows < (int64_t)128 * device_cus() && (T <= 128 || rows * mats[0].C < (int64_t)24 << 20);
}

size_t decoded_workspace(const sq_matrix* mats, int n, int T) {
    size_t need = 0;
    for (int i = 0, r0 = 0; i < n;) {
        const DecodedRows d = decoded_step(mats, n, i, r0);
        if (d.n) need = std::max(need, d.bytes + mid_dense_workspace(d.m, d.n, T));
    }
    return need;
}

int launch_decoded(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws, hipStream_t s, bool wide) {
    int rows = T;                                                // activation rows at a time: all, unless they span 4 GB
    while (rows > 1 && !mid_x_ok(ldx, rows)) rows = (rows + 1) / 2;
    for (int i = 0, r0 = 0; i < n;) {
        const DecodedRows d = decoded_step(mats, n, i, r0);
        const void* w[MID_PIECES];
        char* next = (char*)ws;
        for (int j = 0; j < d.n; ++j) {
            w[j] = next;
            if (const int rc = launch_dequant(*d.of[j], next, SQ_F16, mats[0].C, d.r0[j], d.r0[j] + d.m[j].R, s, /*raw=*/true)) return rc;
            next += dense_bytes(d.m[j]);
        }
        for (int t = 0; d.n && t < T; t += rows)
            if (const int rc = launch_mid_decoded(d.m, d.n, w, (const char*)x + (size_t)t * ldx * 2, x_dtype, rows > 1 ? ldx : mats[0].C,
                                                  (char*)y + (size_t)t * ldy * (y_dtype == SQ_F32 ? 4 : 2), y_dtype, ldy, std::min(rows, T - t), next, s, wide))
                return rc;
    }
    return SQ_OK;
}

// Activation rows from which a stack with column orders is decoded and multiplied instead of reading x through its orders:
// where the rows have tag streams, whose kernel takes up to eight rows at once, 11, or 17 if the decode is long (8 / 10 / 11 rows
// there and here: 4608 x 3584 46 / 89 us and 43, 37888 x 3584 81 / 118 and 237).  Without, each four rows cost as much again,
// twice that on long rows (4 / 5 / 8 rows there, and any of them here: 593 x 1984 15 / 23 / 28 us and 18, 16000 x 3584 54 / 91 /
// 103 and 78, 3584 x 18944 193 / 242 / 384 and 95, at 2 rows 97; 37888 x 3584 at 8 / 9 rows 194 / 272 and 237 in the tile GEMM).
static bool masked_gemm(const sq_matrix* mats, int n, int B) {
    if (!has_orders(mats, n)) return false;
    if (small_uses_sums(mats, n)) return decoded_route(mats, n, B) ? B >= 11 : B >= 17 && mats[0].C % 64 == 0;
    if (decoded_route(mats, n, B)) return B >= (mats[0].C > 8192 ? 3 : 5);
    return B >= 9 && mats[0].C % 64 == 0;
}

bool small_takes_gemm_route(const sq_matrix* mats, int n, int B, const void* x, int64_t ldx) {
    return masked_gemm(mats, n, B) && x_vec_ok(x, ldx, mats[0].C);
}

size_t small_gemm_route_workspace(const sq_matrix* mats, int n, int B) {
    return masked_gemm(mats, n, B) ? gemm_workspace(mats, n, B) : 0;
}

// What a piece takes on the vector kernel, in microseconds: columns one behind the other in a lane, and weights over the chip, both per pass of
// four rows and slower the less the caches near a CU hold of the codebook.  Fitted to 27 eager calls of 256, 2048 and 16384 rows of 512 to
// 1544 columns, 6-, 14- and 16-bit tags, at 3 to 6 activation rows (most within 15 %).
static double vector_us(const sq_matrix& m, int B) {
    const double columns = m.C * 1e-3, weights = m.R * columns * 1e-3, table = ((double)m.G * m.d * 2) * ((int64_t)1 << m.bits);
    const int passes = (B + 3) / 4;
    if (table <= 32 * 1024) return 4.5 + std::hypot((1.25 * B + 3.1 * (passes - 1)) * columns, 2.2 * passes * weights);
    return (table > 512 * 1024 ? 7.5 : 5.5) + std::hypot((2.2 * B + 2.4 * (passes - 1)) * columns, 4.2 * passes * weights);
}

// Without orders: how many pieces, the first one on, are decoded and multiplied from there at B rows because the decode-time product would
// run them on the vector kernel (tags of other widths; rows that end within a lane unit with 16-bit tags, codebooks beyond LDS or no tile-major copy), which
// takes every few rows as long again: from VECTOR_DECODED_B rows, where the decode, a product and a sum of slices take less (vector
// kernel / decoded, us at 3 / 4 / 5 rows: 5120 x 2080, 16-bit tags, 58 / 66 / 107 and 24 at any; 300 x 2080 21 / 25 / 36, 14; 512 x 1024,
// 14-bit tags of width 4, 10.8 / 12.5 / 18.2, 17.7; 4864 x 896, 6-bit, 13.8 / 15.8 / 21.5, 20; 2048 x 512, 6-bit, 7.9 / 8.0 / 9.7, 17; 16384 x
// 512 23 / 27 / 36, 20).  Their neighbours in the stack keep their kernels, which read tags.
constexpr int VECTOR_DECODED_B = 3;
int vector_decoded(const sq_matrix* mats, int n, int B) {
    if (B < VECTOR_DECODED_B) return 0;
    int k = 0;
    double vector = 0.0, decoded = 0.0;
    for (; k < n; ++k) {
        const sq_matrix& m = mats[k];
        if (m.R == 0) continue;
        if (!small_vector(m, B) || !mid_dense_ok(&m, 1, B)) break;
        vector += vector_us(m, B);
        decoded += (decoded > 0.0 ? 3.0 : m.d == 8 ? 13.5 : 16.5) + 0.7e-6 * m.R * m.C;
    }
    return vector > decoded ? k : 0;
}

static size_t gemm_workspace_beyond_small(const sq_matrix* mats, int n, int T);

// What decoding in plane order (sq_planes.hip) saves a product in the tile GEMM, in microseconds: 0.24 per million weights, and a launch per
// piece beyond the first, less a launch that brings the codebooks and the activations into that order, which fp16 activations would otherwise not
// pay for.  Fitted to 56 products of 3 M to 136 M weights at 1100 and 2048 rows (before / now, us: 2 x 18944 x 3584 at 1024 / 2048 rows 338 / 514 and
// 301 / 474, 15000 x 4992 at 1100 200 and 183, 3000 + 3000 x 3584 70 and 65; where it is not taken, 3584 x 3584 at 2048 62.2 and 63.3, 3000 x 1024 27 and 32).
static float planes_gain(const sq_matrix* mats, int n, int T, int x_dtype) {
    if (n > 1 && !stacked_route(mats, n)) return 0.f;
    float weights = 0.f;
    for (int i = 0; i < n; i += GEMM256_PIECES)
        if (!planes_ok(mats + i, std::min(n - i, GEMM256_PIECES))) return 0.f;
    for (int i = 0; i < n; ++i) weights += (float)mats[i].R * mats[i].C * 1e-6f;
    const float x = (float)T * mats[0].C * 1e-6f;
    return 0.24f * weights + 3.5f * (n - 1) - 5.5f * ((n + GEMM256_PIECES - 1) / GEMM256_PIECES) - (x_dtype == SQ_F16 ? 1.f + 0.35f * x : 0.f);
}
bool planes_route(const sq_matrix* mats, int n, int T, int x_dtype) { return big_route(mats, n, T) && planes_gain(mats, n, T, x_dtype) > 0.5f; }

// What decode and tile GEMM take, in microseconds, fitted to 722 products (8 %)
static float tiles_us(const sq_matrix* mats, int n, int T, int x_dtype) {
    float us = 3.2f, weights = 0.f;
    int rows = 0;
    for (int i = 0; i < n; ++i) weights += (float)mats[i].R * mats[i].C * 1e-6f, rows += mats[i].R;
    us += 1.13f * gemm256_us(T, rows, mats[0].C, device_cus()) + (mats[0].d == 8 ? 0.77f : 0.51f) * weights;
    if (mats[0].d == 8) us -= 0.6f * std::max(0.f, planes_gain(mats, n, T, x_dtype));     // (1500 x 4032 in three pieces: 260 rows 31.3 there, 32.0 decoded, 500 42.0 and 39.9)
    return us;
}

// The same for the d = 8 products of two blocks of tokens that fused_us knows, fitted to 226 of them with activations of either type (7 %): a million weights costs
// seven times as much from about where the 256 MB last-level cache no longer holds their fp16 copy beside what the product reads and writes.  (Whether the
// codebooks go in columns makes no difference beyond that error.)
static float tiles_us_two_blocks(const sq_matrix* mats, int n, int T) {
    float weights = 0.f;
    int rows = 0;
    for (int i = 0; i < n; ++i) weights += (float)mats[i].R * mats[i].C * 1e-6f, rows += mats[i].R;
    return 9.4f + 1.225f * gemm256_us(T, rows, mats[0].C, device_cus()) + 0.0765f * weights + 0.51f * std::max(0.f, weights - 90.f);
}

// Which kernel takes a product, in one place: what one of them gives up is taken by the one that it was compared with.
//
// Products that the fused kernel has a cut for (129 to 768 rows) run there, unless
//   d = 4   the kernel of sq_mid.h, in blocks of activation rows, is estimated to take at most 85 % of the time and 80 us (a long product runs at a lower clock than both
//           estimates know: 26000 x 5600, 10-bit tags, at 237 rows 95 us there, 104 here).  It does for most of them: 11600 x 3800, 10-bit, at 259 rows 68 us there, 42
//           here; 18900 x 1900, 8-bit, at 201 42 / 29; 7704 x 8192 in four books of 10-bit tags at 262 75 / 59, 12257 x 6592, 10-bit, at 391 101 / 78; not for 29600 x
//           2300, 10-bit, at 370 72 / 90, or 15500 x 1200 at 470 37 / 38.  Rows below 512 columns, a launch's length either way, were not measured and stay.  From 50 us on that
//           kernel also has to be estimated at 73 % of the tiles, which gain most where the rows are just beyond two of theirs: of 47 products of 50 to 80 us
//           at 260 to 738 rows those below 73 % took 0.58 to 0.98 of the tiles' time (0.55 to 0.94 of this kernel's), those above 0.88 to 1.12, the
//           tiles 0.73 to 0.88 of this kernel's (18549 x 1920, 10-bit, at 541 rows 81 here, 69 there, 62 in tiles).
//   d = 8   they are two blocks of tokens in one round of workgroups and decode and tiles are estimated to take less.  They do for most of 226 such products
//           of 192 to 14000 columns, us here and there: 18944 x 3584 at 450 / 700 rows 118 / 135 and 97 / 117, 2 x 9313 x 2048 at 533 90 / 67, 3977 x 8896
//           at 712 117 / 88; not for short rows (7749 + 2 x 1937 x 448 at 483 25 / 32, 2 x 9394 x 576 at 498 39 / 44) and some long ones whose copy
//           the last-level cache does not hold (10009 x 13568 twice at 490 382 / 394).  What is taken is 0.6 % slower than the faster one in the mean, by more than 5 % for eight of them
//           (2 x 6081 x 12992 at 510, in tiles, 244 / 297; 12436 + 2 x 3109 x 576 at 700, here, 49 / 43).  In two rounds, 37888 x 3584 at 450 / 600 / 768, 205 / 230 / 238 here and 206 /
//           252 / 240.
//
// Without such a cut, beyond the row counts that always take it, the kernel of sq_mid.h is the faster way for small products: where its estimated
// time is below 50 us (longer ones run at a lower clock) and 90 % of what decode and tile GEMM take.  There and here, us (700 / 1000 / 1600
// rows): 1024 x 896, 12-bit tags, 19.9 / 19.6 / 20.2 and 8.2 / 8.5 / 11.0, 3584 x 3584 45.0 / 47.7 / 55.2 and 30.9 / 33.9 / 54.3, 18000 x 1024 43 /
// 58 / 76 and 45 / 57 / 87; 16-bit, 1024 x 896, 19.2 / 19.1 / 19.8 and 12.5 / 14.9 / 17.9, 3584 x 3584 47 / 51 / 58 and 69 / 80 / 116.
// (44 products on whose way this and an older estimate of the tile GEMM disagree take 0.94 of the time in the mean,
// none of them longer: 1078 + 1078 x 1408, 16-bit, at 610 rows 37.5 and 24.8, 8310 x 960, 8-bit, at 616 31.6 and 23.4.)
constexpr int FUSED_MID_C = 512;
GemmRoute gemm_route(const sq_matrix* mats, int n, int T, int x_dtype) {
    GemmRoute r{GEMM_FUSED, fused_plan(mats, n, T), {}, {}};
    float most = 50.f;                                           // us that the kernel of sq_mid.h may take beyond mid_ok
    if (r.fused.nw && mats[0].d == 8) {
        if (!fused_two_blocks(r.fused, mats, n) || tiles_us_two_blocks(mats, n, T) >= fused_us(r.fused, mats, n)) return r;
    } else if (r.fused.nw) {
        if (mats[0].C < FUSED_MID_C) return r;
        most = 80.f;
        r.mid = mid_plan(mats, n, T);
        if (r.mid.us > most || r.mid.us > 0.85f * fused_us(r.fused, mats, n)) return r;
    }
    if (T > SQ_SMALL_BMAX) {
        if (!r.mid.nt) r.mid = mid_plan(mats, n, T);
        if (plane_product_group(mats, n, T, r.columns, &r.mid) == n) { r.kernel = GEMM_COLUMNS; return r; }
        if (r.mid.nt && (mid_ok(mats, n, T) || (r.mid.us < most && r.mid.us < (r.mid.us < 50.f ? 0.9f : 0.73f) * tiles_us(mats, n, T, x_dtype)))) { r.kernel = GEMM_MID; return r; }
        if (T <= small_pass_limit(mats, n)) { r.kernel = GEMM_PASSES; return r; }
    }
    r.kernel = decoded_route(mats, n, T) ? GEMM_DECODED : GEMM_TILES;
    return r;
}

// For tests: that kernel (7: the tile GEMM behind a decode in plane order), and what the first one, the kernel of sq_mid.h and the tiles are estimated to take, in
// microseconds (1e30: not for these pieces).
extern "C" __attribute__((visibility("default"))) int32_t sq_gemm_kernel_for_tests(const sq_matrix* mats, int32_t n, int32_t T, int32_t x_dtype, float* us) {
    const FusedPlan fused = fused_plan(mats, n, T);
    const bool two = mats[0].d == 8 && fused.nw && fused_two_blocks(fused, mats, n);
    us[0] = two || (fused.nw && mats[0].d == 4) ? fused_us(fused, mats, n) : 1e30f;
    us[1] = mid_plan(mats, n, T).us;
    us[2] = two ? tiles_us_two_blocks(mats, n, T) : tiles_us(mats, n, T, x_dtype);
    const GemmKernel k = gemm_route(mats, n, T, x_dtype).kernel;
    return k == GEMM_TILES && planes_route(mats, n, T, x_dtype) ? 7 : k;
}

size_t gemm_workspace(const sq_matrix* mats, int n, int T) {
    // up to SQ_SMALL_BMAX rows sq_linear_gemm is sq_linear_small, unless the stack goes the other way (see above);
    // which of the two runs then depends on the alignment of x, so the workspace covers both
    if (T > SQ_SMALL_BMAX) return gemm_workspace_beyond_small(mats, n, T);
    const size_t small = small_workspace(mats, n, T);
    return masked_gemm(mats, n, T) ? std::max(small, gemm_workspace_beyond_small(mats, n, T)) : small;
}

static size_t gemm_workspace_beyond_small(const sq_matrix* mats, int n, int T) {
    // (covers the other routes too: the size is asked for without knowing x; up to SQ_SMALL_BMAX rows the only one is the
    // decode-time kernel, which the caller adds)
    if (T <= SQ_SMALL_BMAX && decoded_route(mats, n, T)) return decoded_workspace(mats, n, T);
    const size_t tiles = gemm_workspace_without_mid(mats, n, T) + (planes_route(mats, n, T, SQ_BF16) ? planes_bytes(std::min(n, GEMM256_PIECES)) : (size_t)0);
    // (the kernel of small products takes some with fp16 activations that go through the tiles, which are counted above, with bf16 ones; else x's type makes no difference)
    const GemmRoute r = gemm_route(mats, n, T, SQ_F16);
    switch (r.kernel) {
    case GEMM_FUSED: return std::max({tiles, fused_workspace(r.fused, mats, n, T), mid_ok(mats, n, T) ? mid_workspace(mats, n, T, &r.mid) : (size_t)0});
    case GEMM_COLUMNS: return std::max({tiles, mid_workspace(mats, n, T, &r.mid), plane_product_workspace(mats, n, T, &r.columns)});
    case GEMM_MID: return std::max(tiles, mid_workspace(mats, n, T, &r.mid));
    case GEMM_DECODED: return std::max(tiles, decoded_workspace(mats, n, T));
    default: return tiles;
    }
}

size_t gemm_workspace_without_mid(const sq_matrix* mats, int n, int T) {
    if (T > SQ_SMALL_BMAX && T <= small_pass_limit(mats, n)) {
        // full passes and the last, shorter one may run different kernels with different needs
        const size_t full = small_workspace(mats, n, SQ_SMALL_BMAX);
        const size_t last = T % SQ_SMALL_BMAX ? small_workspace(mats, n, T % SQ_SMALL_BMAX) : 0;
        return std::max(full, last);
    }
    size_t need = 0;
    const bool big = big_route(mats, n, T);
    if (big && stacked_route(mats, n)) {
        for (int i = 0; i < n; i += GEMM256_PIECES) {
            const int k = std::min(n - i, GEMM256_PIECES);
            need = std::max(need, stacked_bytes(mats + i, k) + gemm256_part_bytes(T, stacked_rows(mats + i, k), mats[0].C, device_cus()));
        }
        return need + align256((size_t)T * mats[0].C * 2);
    }
    for (int i = 0; i < n; ++i)
        if ((big || !fused_ok(mats[i])) && dense_bytes(mats[i]) > need) need = dense_bytes(mats[i]);
    if (big) {
        need += align256((size_t)T * mats[0].C * 2);            // fp16 copy of bf16 activations
        size_t part = 0;                                        // fp32 partial products of a K split
        for (int i = 0; i < n; ++i) part = std::max(part, gemm256_part_bytes(T, mats[i].R, mats[i].C, device_cus()));
        need += part;
    }
    return need;
}

static size_t gathered_workspace(const sq_matrix* mats, int n) {
    size_t need = 0;
    for (int i = 0; i < n; ++i)
        if (!fused_ok(mats[i])) need = std::max(need, dense_bytes(mats[i]));
    return need;
}

static int run(const GemmArgs& a, int d, bool dense, hipStream_t s) {
    const dim3 grid((a.m.R + BN - 1) / BN, (a.T + BM - 1) / BM);
    if (dense) hipLaunchKernelGGL((gemm_kernel<8, true>), grid, dim3(256), 0, s, a);
    else if (d == 8) hipLaunchKernelGGL((gemm_kernel<8, false>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((gemm_kernel<4, false>), grid, dim3(256), 0, s, a);
    return check_launch("sq_linear_gemm");
}

size_t gemm_dense_workspace(int R, int C, int T) {
    return (T >= GEMM256_MIN_T && C % 64 == 0) ? gemm256_part_bytes(T, R, C, device_cus()) : 0;
}

int launch_gemm_dense(const void* w, int w_dtype, int64_t ldw, int R, int C, const void* x, int x_dtype, int64_t ldx,
                      void* y, int y_dtype, int64_t ldy, int T, hipStream_t s, void* ws, size_t ws_bytes) {
    if (!x_vec_ok(x, ldx, C) || !x_vec_ok(w, ldw, C))
        return fail(SQ_EUNSUPPORTED, "sq_gemm_dense: C, ldx, ldw must be multiples of 8 and pointers 16-byte aligned");
    if (x_dtype == SQ_F16 && w_dtype == SQ_F16 && T >= GEMM256_MIN_T && gemm256_ok(C, ldx, ldw, x, w)) {
        const size_t part = gemm_dense_workspace(R, C, T);      // (none is asked for where the last slab is broken)
        const bool split = ws && part && ws_bytes >= part;
        return launch_gemm256((const uint16_t*)x, ldx, (const uint16_t*)w, ldw, Gemm256Scales{}, y, y_dtype, ldy, 0, T, R, C,
                              split ? (float*)ws : nullptr, split ? device_cus() : 0, s);
    }
    GemmArgs a{};
    a.m.R = R; a.m.C = C; a.m.y_off = 0;
    a.wd = (const uint16_t*)w; a.ldw = ldw;
    a.x = (const uint16_t*)x; a.ldx = ldx; a.y = y; a.ldy = ldy; a.T = T; a.x_dtype = x_dtype; a.y_dtype = y_dtype;
    a.w_dtype = w_dtype;
    return run(a, 8, true, s);
}

int launch_gemm(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype,
                int64_t ldy, int T, void* ws, size_t ws_bytes, void* sums, hipStream_t s) {
    if (T <= SQ_SMALL_BMAX && !small_takes_gemm_route(mats, n, T, x, ldx))
        return launch_small(mats, n, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, ws_bytes, sums, s);
    if (T > SQ_SMALL_BMAX && x_vec_ok(x, ldx, mats[0].C)) {
        const GemmRoute r = gemm_route(mats, n, T, x_dtype);
        if (r.kernel == GEMM_COLUMNS && plane_product_workspace(mats, n, T, &r.columns) <= ws_bytes)
            return launch_plane_product(mats, n, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, ws_bytes, s, &r.columns);
        // (the fused kernel's cuts also serve where a workspace or the span of x does not let the others in)
        const bool mid = mid_x_ok(ldx, T) && (mid_ok(mats, n, T) ? mid_least(mats, n, T) <= ws_bytes : r.kernel == GEMM_MID && gemm_workspace_without_mid(mats, n, T) <= ws_bytes);
        if (r.fused.nw && (r.kernel == GEMM_FUSED || !mid) && fused_workspace(r.fused, mats, n, T) <= ws_bytes && (r.kernel != GEMM_TILES || gemm_workspace_without_mid(mats, n, T) > ws_bytes))
            return launch_fused(r.fused, mats, n, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, s);
        if (mid) return launch_mid(mats, n, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, ws_bytes, s, &r.mid);
        if (mid_x_ok(ldx, T) && mid_ok(mats, n, T)) return fail(SQ_EWORKSPACE, "sq_linear_gemm: workspace %zu < %zu", ws_bytes, gemm_workspace(mats, n, T));
    }
    if (T > SQ_SMALL_BMAX && T <= small_pass_limit(mats, n) && x_vec_ok(x, ldx, mats[0].C)) {
        // stacks that cannot go in one pass (pieces of different formats): a few passes of the decode-time kernel read the packed
        // tags a few times; decoding to fp16 first (below) writes and reads 8 to 16 times as many bytes once
        const size_t ys = y_dtype == SQ_F32 ? 4 : 2;
        for (int t = 0; t < T; t += SQ_SMALL_BMAX) {
            const int nb = T - t < SQ_SMALL_BMAX ? T - t : SQ_SMALL_BMAX;
            int rc = launch_small(mats, n, (const char*)x + (size_t)t * ldx * 2, x_dtype, ldx, (char*)y + (size_t)t * ldy * ys,
                                  y_dtype, ldy, nb, ws, ws_bytes, sums, s);
            if (rc) return rc;
        }
        return SQ_OK;
    }
    if (!x_vec_ok(x, ldx, mats[0].C)) {
        for (int i = 0; i < n; ++i)
            if (!mats[i].tags) return fail(SQ_EUNSUPPORTED, "sq_linear_gemm: a matrix held as its tag stream only needs 16-byte aligned x with ldx %% 8 == 0");
        // odd strides: the any-shape kernel, SQ_SMALL_BMAX activation rows at a time
        for (int t = 0; t < T; t += SQ_SMALL_BMAX) {
            const int nb = T - t < SQ_SMALL_BMAX ? T - t : SQ_SMALL_BMAX;
            const size_t es = 2, ys = y_dtype == SQ_F32 ? 4 : 2;
            int rc = launch_small_generic(mats, n, (const char*)x + (size_t)t * ldx * es, x_dtype, ldx,
                                          (char*)y + (size_t)t * ldy * ys, y_dtype, ldy, nb, s);
            if (rc) return rc;
        }
        return SQ_OK;
    }
    if (decoded_route(mats, n, T) && decoded_workspace(mats, n, T) <= ws_bytes)
        return launch_decoded(mats, n, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, s);
    const bool room = gemm_workspace_without_mid(mats, n, T) <= ws_bytes;
    // (rows of a broken slab run in 128 x 128 tiles where the workspace holds less: what that kernel cannot gather itself)
    if (!room && (mats[0].C % 64 == 0 || gathered_workspace(mats, n) > ws_bytes))
        return fail(SQ_EWORKSPACE, "sq_linear_gemm: workspace %zu < %zu", ws_bytes, gemm_workspace(mats, n, T));
    if (room && big_route(mats, n, T)) {
        const int C = mats[0].C;
        const uint16_t* xh = (const uint16_t*)x;
        int64_t ldxh = ldx;
        char* wd = (char*)ws;
        // bf16 activations are copied to fp16 once; the copy rides along with the first decode when that takes
        // the four-chunk kernel (the two overlap in one launch), else it is a launch of its own.  A decode in plane order
        // (given the workspace) needs activations of either type in that order.
        const size_t plane_bytes = planes_route(mats, n, T, x_dtype) ? planes_bytes(std::min(n, GEMM256_PIECES)) : 0;
        const bool planes = plane_bytes && gemm_workspace_without_mid(mats, n, T) + plane_bytes <= ws_bytes;
        bool copy_pending = planes || x_dtype == SQ_BF16;
        if (copy_pending) {
            xh = (const uint16_t*)ws;
            ldxh = C;
        }
        wd += align256((size_t)T * C * 2);
        uint16_t* plane_tables = (uint16_t*)wd;
        if (planes) wd += plane_bytes;
        auto decode_stack = [&](const sq_matrix* ms, int k, void* w) -> int {
            const void* xs = copy_pending ? x : nullptr;
            const int rc = planes ? launch_planes(ms, k, (uint16_t*)w, plane_tables, xs, x_dtype, ldx, T, (uint16_t*)ws, s)
                                  : launch_dequant_stack(ms, k, w, 1, (const uint16_t*)xs, ldx, T, C, (uint16_t*)ws, s);
            if (rc == 0) copy_pending = false;
            return rc;
        };
        auto decode = [&](const sq_matrix& m, void* w) -> int {
            if (const int rc = decode_stack(&m, 1, w); rc <= 0) return rc;
            if (copy_pending) {
                copy_pending = false;
                const int rc = launch_dequant_with_cvt(m, w, C, (const uint16_t*)x, ldx, T, C, (uint16_t*)ws, s);
                if (rc <= 0) return rc;
                const int rc2 = launch_bf16_to_f16((const uint16_t*)x, ldx, T, C, (uint16_t*)ws, s);
                if (rc2) return rc2;
            }
            return launch_dequant(m, w, SQ_F16, C, 0, m.R, s, /*raw=*/true);
        };
        const int cus0 = device_cus();
        if (stacked_route(mats, n)) {
            for (int i0 = 0; i0 < n; i0 += GEMM256_PIECES) {
                const sq_matrix* ms = mats + i0;
                const int k = std::min(n - i0, GEMM256_PIECES), R = stacked_rows(ms, k);
                float* part = (float*)(wd + stacked_bytes(ms, k));
                char* w = wd;
                Gemm256Scales sc{};
                int r0 = 0;
                const int whole = decode_stack(ms, k, w);       // all pieces in one launch, or (1) piece by piece
                if (whole < 0) return whole;
                for (int i = 0; i < k; ++i) {
                    const sq_matrix& m = ms[i];
                    if (whole == 1)
                        if (int rc = decode(m, w)) return rc;
                    w += (size_t)m.R * C * 2;                   // rows follow each other without gaps
                    r0 += m.R;
                    sc.p[i] = m.row_scale;
                    sc.end[i] = r0;
                }
                sc.n = k;
                if (int rc = launch_gemm256(xh, ldxh, (const uint16_t*)wd, C, sc, y, y_dtype, ldy, ms[0].y_off, T, R, C,
                                            gemm256_part_bytes(T, R, C, cus0) ? part : nullptr, cus0, s))
                    return rc;
            }
            return SQ_OK;
        }
        size_t dense = 0;
        for (int i = 0; i < n; ++i) dense = std::max(dense, dense_bytes(mats[i]));
        float* part = (float*)(wd + dense);
        const int cus = device_cus();
        for (int i = 0; i < n; ++i) {
            const sq_matrix& m = mats[i];
            if (m.R == 0) continue;
            int rc = decode(m, wd);
            if (rc) return rc;
            rc = launch_gemm256(xh, ldxh, (const uint16_t*)wd, C, Gemm256Scales{{m.row_scale}, {m.R}, 1}, y, y_dtype, ldy, m.y_off, T, m.R, C,
                                gemm256_part_bytes(T, m.R, C, cus) ? part : nullptr, cus, s);
            if (rc) return rc;
        }
        return SQ_OK;
    }
    for (int i = 0; i < n; ++i) {
        const sq_matrix& m = mats[i];
        if (m.R == 0) continue;
        GemmArgs a{};
        a.m = m;
        a.x = (const uint16_t*)x; a.ldx = ldx; a.y = y; a.ldy = ldy; a.T = T; a.x_dtype = x_dtype; a.y_dtype = y_dtype;
        int rc;
        if (fused_ok(m)) {
            rc = run(a, m.d, false, s);
        } else {
            // column orders or an unusual chunk width: gather the raw codewords (with the column
            // scatter) into the workspace as fp16, which is exact, and multiply from there with the row scale
            // applied to the accumulator as in the fused kernel; the stream orders the two kernels and the next piece
            rc = launch_dequant(m, ws, SQ_F16, m.C, 0, m.R, s, /*raw=*/true);
            if (rc) return rc;
            a.wd = (const uint16_t*)ws; a.ldw = m.C; a.w_dtype = SQ_F16;
            rc = run(a, 8, true, s);
        }
        if (rc) return rc;
    }
    return SQ_OK;
}

// ---- the 8-bit block-32 head above SQ_SMALL_BMAX activation rows: row chunks decoded to fp16 (scale folded
// in, one rounding, as the reference's chunked route does: shapequant/vllm_ext/core.py:548-555, 587-591) and
// multiplied by the dense tile GEMM.  A chunk is as large as Q8_CHUNK_BYTES of fp16 allows so that one GEMM
// launch has enough tiles for the whole chip.
constexpr size_t Q8_CHUNK_BYTES = (size_t)256 << 20;

static int q8_chunk_rows(int V, int C) {
    int64_t rows = (int64_t)(Q8_CHUNK_BYTES / ((size_t)C * 2)) / 256 * 256;
    if (rows < 256) rows = 256;
    return rows < V ? (int)rows : V;
}

static bool q8_big(int T, int C) { return T >= GEMM256_MIN_T && C % 8 == 0; }

size_t q8_workspace(int V, int C, int T) {
    if (T <= SQ_SMALL_BMAX || V <= 0) return 0;
    const int chunk = q8_chunk_rows(V, C);
    size_t need = align256((size_t)chunk * C * 2);
    if (q8_big(T, C)) {
        const int last = V % chunk;                             // the split of a launch depends on its tile count
        const size_t part = std::max(gemm256_part_bytes(T, chunk, C, device_cus()),
                                     last ? gemm256_part_bytes(T, last, C, device_cus()) : (size_t)0);
        need += align256((size_t)T * C * 2) + part;
    }
    return need;
}

int launch_q8_large(const int8_t* q, const uint16_t* sc, int V, int C, const void* x, int x_dtype, int64_t ldx, void* y,
                    int y_dtype, int64_t ldy, int T, void* ws, size_t ws_bytes, hipStream_t s) {
    if (q8_workspace(V, C, T) > ws_bytes)
        return fail(SQ_EWORKSPACE, "sq_q8_linear: workspace %zu < %zu", ws_bytes, q8_workspace(V, C, T));
    if (!x_vec_ok(x, ldx, C))
        return fail(SQ_EUNSUPPORTED, "sq_q8_linear: more than %d rows need ldx %% 8 == 0 and 16-byte aligned x", SQ_SMALL_BMAX);
    const int chunk = q8_chunk_rows(V, C);
    const size_t ys = y_dtype == SQ_F32 ? 4 : 2;
    char* wd = (char*)ws;
    const bool big = q8_big(T, C);
    const uint16_t* xh = (const uint16_t*)x;
    int64_t ldxh = ldx;
    float* part = nullptr;
    const int cus = device_cus();
    if (big) {
        if (x_dtype == SQ_BF16) {
            int rc = launch_bf16_to_f16((const uint16_t*)x, ldx, T, C, (uint16_t*)ws, s);
            if (rc) return rc;
            xh = (const uint16_t*)ws;
            ldxh = C;
        }
        wd += align256((size_t)T * C * 2);
        part = (float*)(wd + align256((size_t)chunk * C * 2));
    }
    for (int r0 = 0; r0 < V; r0 += chunk) {
        const int r1 = r0 + chunk < V ? r0 + chunk : V;
        int rc = launch_q8_dequant(q, sc, C, wd, SQ_F16, C, r0, r1, s);
        if (rc) return rc;
        void* yc = (char*)y + (size_t)r0 * ys;
        if (big && gemm256_ok(C, ldxh, C, xh, wd))
            rc = launch_gemm256(xh, ldxh, (const uint16_t*)wd, C, Gemm256Scales{}, yc, y_dtype, ldy, 0, T, r1 - r0, C,
                                gemm256_part_bytes(T, r1 - r0, C, cus) ? part : nullptr, cus, s);
        else
            rc = launch_gemm_dense(wd, SQ_F16, C, r1 - r0, C, x, x_dtype, ldx, yc, y_dtype, ldy, T, s);
        if (rc) return rc;
    }
    return SQ_OK;
}

}  // namespace sq
