// Host side of the decode-time product: picks the team geometry per shape, fuses stacked pieces
// into one persistent launch, prepares permuted activations for pieces with column orders.
#include "sq_rows_mfma.h"
#include "sq_slices.h"
#include "sq_stream.h"

namespace sq {

int launch_gemv_b16d8(int, const GemvArgs&, int, int, int, int, size_t, hipStream_t);
int launch_gemv_b12d4(int, const GemvArgs&, int, int, int, int, size_t, hipStream_t);
int launch_gemv_b10d4(int, const GemvArgs&, int, int, int, int, size_t, hipStream_t);
int launch_gemv_b8d4(int, const GemvArgs&, int, int, int, int, size_t, hipStream_t);
int launch_mma_b16d8(int, const MmaArgs&, int, int, int, int, size_t, hipStream_t);
int launch_mma_b12d4(int, const MmaArgs&, int, int, int, int, size_t, hipStream_t);
int launch_mma_b10d4(int, const MmaArgs&, int, int, int, int, size_t, hipStream_t);
int launch_mma_b8d4(int, const MmaArgs&, int, int, int, int, size_t, hipStream_t);

// xp[m, b, c] = fp16(x[b, perms[m, c]])
__global__ __launch_bounds__(256) void permute_x_kernel(const uint16_t* __restrict__ x, int64_t ldx, int x_dtype,
                                                        const int32_t* __restrict__ perms, int M, int B, int C,
                                                        uint16_t* __restrict__ xp) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)M * B * C) return;
    const int c = (int)(i % C);
    const int b = (int)((i / C) % B);
    const int mk = (int)(i / ((int64_t)C * B));
    const uint16_t v = x[(int64_t)b * ldx + perms[(int64_t)mk * C + c]];
    xp[i] = x_dtype == SQ_BF16 ? __builtin_bit_cast(uint16_t, bf2h(v)) : v;
}

// ------------------------------------------------------------------------------------------ host

int launch_small_generic(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y,
                         int y_dtype, int64_t ldy, int B, hipStream_t s);

int unit_dwords(int bits) { return bits == 12 ? 3 : bits == 10 ? 5 : 4; }
int row_units(int C, int d, int bits) { const int tags = unit_dwords(bits) * 32 / bits; return (C / d + tags - 1) / tags; }

bool whole_units(const sq_matrix& m) { return m.W % unit_dwords(m.bits) == 0 && (int64_t)(m.C / m.d) * m.bits == (int64_t)m.W * 32; }

static bool fast_shape(const sq_matrix& m) {
    if (!m.tags) return false;                                   // held as its tag stream only
    const bool fmt = (m.d == 8 && m.bits == 16) || (m.d == 4 && (m.bits == 12 || m.bits == 10 || m.bits == 8));
    if (!fmt) return false;
    if (((uintptr_t)m.tags & 15) || ((uintptr_t)m.table & 15)) return false;
    return whole_units(m);
}

// ---- tile-major copy of the tags for the matrix-core decode kernel (d = 4 formats, whose codebooks live in
// LDS and which have no slice stream).  In the file's row-major layout the 16 lanes of a quarter wave read 16
// different rows, 48 bytes each; in the copy the units of a 16-row tile are stored unit by unit,
//     tiled[((t * U + u) * 16 + i) * UD + w] = tags[(16 t + i) * W + u * UD + w]      (rows past R: zeros)
// so the same 16 lanes read 16 * UD consecutive dwords and a wave load covers one contiguous piece.  Rows that end within a
// unit (of whole pieces of 8 columns) have it filled up with zeros: in the copy every unit is whole, so these rows take the matrix-core
// kernel too (5120 x 2064, 12-bit tags, at 2 / 16 / 32 rows on the vector kernel 27 / 134 / 264 us; now 6.5 / 7 / 10.5).
bool tiled_format_ok(int R, int W, int C, int d, int bits) {
    if (!(d == 4 && (bits == 12 || bits == 10 || bits == 8))) return false;
    if (R <= 0 || C <= 0 || C % 8) return false;
    return ((int64_t)(C / d) * bits + 31) / 32 == W;
}

size_t tiled_bytes(int R, int C, int bits) { return (size_t)((R + 15) / 16) * 16 * row_units(C, 4, bits) * unit_dwords(bits) * 4; }

void tiled_build(const uint32_t* tags, int R, int W, int C, int bits, uint32_t* out) {
    const int ud = unit_dwords(bits), U = row_units(C, 4, bits), ntiles = (R + 15) / 16;
    for (int t = 0; t < ntiles; ++t)
        for (int u = 0; u < U; ++u)
            for (int i = 0; i < 16; ++i) {
                uint32_t* dst = out + (((size_t)t * U + u) * 16 + i) * ud;
                const int r = t * 16 + i;
                for (int w = 0; w < ud; ++w) dst[w] = r < R && u * ud + w < W ? tags[(size_t)r * W + u * ud + w] : 0u;
            }
}

static size_t xp_bytes(const sq_matrix& m, int B) {
    return (((size_t)(m.M > 1 ? m.M : 1) * B * m.C * 2) + 255) & ~(size_t)255;
}

struct Plan { int TS, S, nwaves; };

// Host mirror of gemv_cfg<>::XW / OK / LB.
static int cfg_xw(int bits, int d, int S, int NB) {
    const int ud = unit_dwords(bits);
    return NB * S * (ud * 32 / bits * d / 2);
}
static int cfg_lb(int bits, int d, int S, int NB) { return cfg_xw(bits, d, S, NB) < 64 ? 512 : 256; }

// Team size / slots for U units per row: fewest idle lanes, then fewest slots.
static Plan plan_for(int U, int bits, int d) {
    Plan best{0, 0, 0};
    double best_eff = -1.0;
    const int cands[] = {16, 32, 64, 128, 192, 256, 320, 384, 448, 512, 640, 768, 1024};
    const int slots[] = {1, 2, 3, 5};
    for (int ts : cands)
        for (int s : slots) {
            if (ts * s < U) continue;
            if (cfg_xw(bits, d, s, 1) > 192) break;
            if (ts > cfg_lb(bits, d, s, 1)) break;
            const double eff = (double)U / (ts * s) - 0.02 * (s - 1) - (ts > 64 ? 0.05 : 0.0);   // barriers cost
            if (eff > best_eff + 1e-9) { best_eff = eff; best.TS = ts; best.S = s; }
            break;
        }
    if (best.TS == 0) return best;
    // 4 waves per workgroup (several workgroups per CU) unless a row needs more waves than that
    const int wpr = best.TS > 64 ? best.TS / 64 : 1;
    best.nwaves = wpr * (4 / wpr > 0 ? 4 / wpr : 1);
    return best;
}

// The tag-stream kernel multiplies up to 8 activation rows per pass (every codeword gathered once, one x gather
// per row).  With column orders (where the alternative is the VALU kernel) it is used for any B <= 32.  Without,
// it wins over the matrix-core kernel's single L2 gather per tag up to 4 rows on every shape, and up to 8 rows
// when a row's part of x is short enough for several rows per pass.  Measured on the 7B layer (microseconds,
// stream / matrix-core kernel): q|k|v 13.8 / 26.7 at 2 rows, 14.5 / 27.1 at 4, 18.6 / 26.8 at 8; o 12.5 / 15.0, 13.7 /
// 14.9, 17.6 / 15.4; gate|up 24.7 / (85 at any row count), 33.5, 62.8; down (rows of 2368 chunks) 18.3, 33.4 / (52 at
// any row count), 63.2.
static bool stream_rows(const sq_matrix& m, int B) {
    if (!stream_shape(m)) return false;
    if (!m.tags) return true;                                    // one-copy residency: the stream is all there is
    return B <= 4 || m.perms != nullptr || (B <= 8 && m.C / m.d <= 1024);
}

// ---- matrix-core path (pieces without column orders)
struct MmaPlan { int RW, NT, KW, ks; };

bool mma_shape(const sq_matrix& m) { return fast_shape(m) && !m.perms; }

// the tile-major copy of a piece's tags, NULL if it has none
static const uint32_t* tiled_piece(const sq_matrix& m) {
    return m.stream && !m.perms && tiled_format_ok(m.R, m.W, m.C, m.d, m.bits) && ((uintptr_t)m.stream & 15) == 0 ? (const uint32_t*)m.stream : nullptr;
}

// what the decode-time kernel takes: those shapes, and rows that end within a unit where they have a tile-major copy
static bool mma_rows(const sq_matrix& m) {
    return mma_shape(m) || (m.tags && !m.perms && ((uintptr_t)m.table & 15) == 0 && tiled_piece(m) && !whole_units(m) && ((int64_t)m.G << m.bits) * m.d * 2 <= 128 * 1024);
}

bool small_vector(const sq_matrix& m, int B) { return m.R > 0 && m.tags && !m.perms && !stream_rows(m, B) && !mma_rows(m); }

// bytes of codebook the matrix-core kernel stages in LDS (0: gathers go through the cache)
static size_t mma_table_bytes(const sq_matrix& m) {
    const size_t tab = (size_t)m.G * ((size_t)1 << m.bits) * m.d * 2;
    return tab <= 128 * 1024 ? tab : 0;
}

// Rounds per wave, waves per workgroup and workgroup-level column slices that cover ceil(U / 4) rounds.
// Gathers from L2 (d = 8 and codebooks beyond LDS): the fewest idle rounds (ties: more rounds per wave, fewer waves to add up).
// Codebooks in LDS: a tile is a chain of LDS round trips in every wave, so few waves leave the LDS idle, and a wave with all the
// rounds its registers hold spends 5 us on fetching its activations; from 7 waves on the gathers' bank conflicts are the bound.
// Extra column slices cost a launch that adds them up.  us at 4 rows, fewest idle rounds / this rule: 2 x 17408 x 5120, 12-bit tags
// 25.1 (5 waves of 8 rounds) / 18.4 (10 of 4), with 4 books 27.4 / 24.8; 5120 x 17408 19.6 / 15.8; 2 x 14336 x 4096, 10-bit 18.0 / 13.5;
// 4864 x 896, 8-bit 7.5 (1 wave) / 4.8 (4); 2 x 2048 x 2048, 4 books 9.4 / 6.3; 7 waves of 4 against 14 of 2 are alike (28 rounds).  With two
// token tiles the sums to add are twice as long and 3 waves are enough (6 waves of 1 round: 15.8, 3 of 2: 11.9, 2 x 8960 x 1536).
static MmaPlan mma_plan(const sq_matrix& m, int B) {
    const int ud = unit_dwords(m.bits), tpu = ud * 32 / m.bits, spu = tpu / (8 / m.d);
    const int rounds = (row_units(m.C, m.d, m.bits) + 3) / 4, r1 = 32 / spu;
    MmaPlan best{0, 0, 0, 0};
    double best_cost = 1e30;
    const int NT = B > 16 ? 2 : 1;
    // waves per workgroup: mma_waves_max, or as many as leave room in the CU's 160 KB of LDS, next to a codebook that is staged there
    // (4 books of 4096 d = 4 entries fill 128 KB), for their accumulators of the tiles in flight and their activation staging areas.
    // Long rows then take more, shorter column slices: 7B down, 148 rounds, at 4 rows: 15.1 us with 15 waves x 2 rounds x 5 slices
    // against 18.4 with 7 x 8 x 3, reduction launch included.
    const size_t tab = mma_table_bytes(m);
    for (int rw = NT == 1 && !tab ? r1 : r1 / 2; rw >= 1 && rw >= r1 / 4; rw /= 2) {
        const int need = (rounds + rw - 1) / rw;
        int mk = 8;
        if (tab) {
            const size_t room = 160 * 1024 - tab - 16;
            const size_t per_wave = std::max((size_t)64 * NT * 16 * mma_pft(rw, NT), (size_t)mma_x_stage_bytes(tpu * m.d, mma_x_tokens_min(NT)));
            mk = (int)std::min<size_t>(mma_waves_max(rw * spu * NT, true), room / per_wave);
            if (mk < 1) continue;
        }
        const int ks = (need + mk - 1) / mk, kw = (need + ks - 1) / ks;
        const double idle = (double)rw * kw * ks / rounds;
        double cost = idle + 0.03 * (ks - 1) + 0.002 * kw;
        if (tab) {
            const double few = std::min(kw, NT == 1 ? 7 : 3);
            cost = idle + 5.5 / (few * few) + 0.004 * kw + (ks > 1 ? 0.2 + 0.018 * (ks - 1) : 0.0);
        }
        if (cost < best_cost - 1e-9) { best_cost = cost; best = MmaPlan{rw, NT, kw, ks}; }
    }
    return best;
}

// The widest variant, whose waves hold all the rounds their registers can, where it takes a row in one launch and mma_plan's does not
// (KW = 0: it does not): up to 8192 columns, from 6145 or, beside 128 KB of codebooks, 5633.
static MmaPlan mma_whole_row(const sq_matrix& m, int B) {
    const MmaPlan none{0, 0, 0, 0};
    const size_t tab = mma_table_bytes(m);
    if (!tab || B > 16 || m.d != 4 || mma_plan(m, B).ks == 1) return none;
    const int ud = unit_dwords(m.bits), tpu = ud * 32 / m.bits, spu = tpu / (8 / m.d), rw = 32 / spu;
    const int need = ((row_units(m.C, m.d, m.bits) + 3) / 4 + rw - 1) / rw;
    const size_t per_wave = std::max((size_t)64 * 16 * mma_pft(rw, 1), (size_t)mma_x_stage_bytes(tpu * m.d, mma_x_tokens_min(1)));
    if (need > (int)std::min<size_t>(mma_waves_max(rw * spu, true), (160 * 1024 - tab - 16) / per_wave)) return none;
    return MmaPlan{rw, 1, need, 1};
}

// Such a launch is slow to begin (its waves fetch all their activations first), column slices cost a reduction launch for every piece
// and the sums' way through memory, three of them share few rows' tiles badly.  us, slices / one launch, 8 rows: one piece of 8192 x 8192 with 8-, 10- and 12-bit
// tags 11.8 / 11.9, 12.0 / 13.5, 12.1 / 13.5, of 14336 rows 14.6 / 15.2, 15.9 / 17.5, 15.3 / 17.6, of 20480 17.9 / 16.7, 19.4 / 19.4, 19.0 / 19.5,
// of 28672 21.6 / 19.9, 23.5 / 23.1, 23.2 / 23.0; two of 4096 rows 13.9 / 12.1, 14.7 / 13.5, 14.3 / 13.5, two of 18944 29.8 / 25.6, 32.0 / 29.5,
// 31.3 / 29.8; four books of 12-bit tags in three slices, 8192 x 6272 14.4 / 13.0, two of 8192 rows 23.5 / 16.7.
static bool mma_whole_row_pays(const sq_matrix& m0, int cnt, const MmaPlan& slices) { return cnt > 1 || m0.R >= 20000 || slices.ks > 2; }

// For pieces that cannot share one pass (formats or lengths differ), and for the workspace of those that can: passes of 32 rows
// through the matrix-core decode kernel against decode + tile GEMM (7B layer): 77 us per pass
// against 600-640 us when the codebook sits in LDS (d = 4), 201 us per pass when its gathers go to L2.  A
// codebook that fills most of LDS leaves room for fewer waves per workgroup and doubles the cost of a pass
// (27B layer, 4 books of 4096: 246 us per pass against 800 us).
int small_pass_limit(const sq_matrix* mats, int n) {
    int limit = 224;
    for (int i = 0; i < n; ++i) {
        if (!mma_shape(mats[i])) return 0;
        const size_t tab = mma_table_bytes(mats[i]);
        const int li = tab == 0 ? 64 : tab > 64 * 1024 ? 96 : 224;
        if (li < limit) limit = li;
    }
    return n > 0 ? limit : 0;
}

static size_t mma_part_bytes(const sq_matrix& m, int B) {
    const MmaPlan pl = mma_plan(m, B);
    return pl.ks > 1 ? ((((size_t)pl.ks * B * m.R * 4) + 255) & ~(size_t)255) : 0;
}

// Rows that end within a unit ran without a workspace before they had a copy: where it has no room for partial sums that only slices
// of such a row need, they still do, on the vector kernels.
static bool mma_without_room(const sq_matrix& m, int B) { return !whole_units(m) && mma_plan(m, B).ks > 1 && !mma_whole_row(m, B).KW; }

// How many pieces, the first one on, run on the kernel of sq_sieve.hip: none that has tag streams for these rows
static int sieve_len(const sq_matrix* mats, int n, int B) {
    int k = 0;
    while (k < n && mma_rows(mats[k]) && !stream_rows(mats[k], B)) ++k;
    return sieve_group(mats, k, B);
}

// The same for the kernel of sq_plane_product.hip
static int plane_product_len(const sq_matrix* mats, int n, int B, PlanePlan& planned) {
    if (B < PLANE_PRODUCT_MIN_T) return 0;
    int k = 0;
    while (k < n && mma_rows(mats[k]) && !stream_rows(mats[k], B)) ++k;
    return plane_product_group(mats, k, B, planned);
}

// SiLU(gate) * up written by the matrix-core kernel: the two pieces' codebooks (one format, one shape) fit LDS side by side next to the
// accumulators of a group of tiles, the rows are not split over workgroups (same plan, so the same sums, as without), and the product
// by itself would run on this kernel: two activation rows or more.  us, the two launches / this one, 8 rows: 2 x 18944 x 3584 with 12-bit tags
// 20.4 / 17.6, 8-bit 18.7 / 15.2; 17408 x 5120, 12-bit 28.7 / 25.0, 10-bit in 4 books 26.3 / 24.0; 8960 x 1536, 12-bit 11.8 / 10.1;
// 1024 x 512, 8-bit 7.6 / 6.6.  But 4864 x 896 (two waves a workgroup) with 64 KB of codebooks 11.7 / 12.0, with 128 KB 13.7 / 17.5: a
// workgroup's waves fetch the codebooks, at most 24 KB each here.
static bool mma_silu_shape(const sq_matrix* mats, int n, int B) {
    if (n != 2 || B < 2 || B > SQ_SMALL_BMAX) return false;
    const sq_matrix &g = mats[0], &u = mats[1];
    if (g.d != 4 || !mma_shape(g) || !mma_shape(u) || g.R <= 0 || g.R != u.R || g.bits != u.bits || g.d != u.d || g.W != u.W || g.G != u.G) return false;
    if (tiled_piece(g) == nullptr != (tiled_piece(u) == nullptr)) return false;
    const size_t tab = mma_table_bytes(g);
    if (tab == 0 || tab > 64 * 1024) return false;               // (beyond 64 KB two rows take the row-segment kernel)
    const MmaPlan pl = mma_plan(g, B);
    const int tpu = unit_dwords(g.bits) * 32 / g.bits;
    return pl.ks == 1 && 2 * tab <= (size_t)pl.KW * 24 * 1024 && 2 * tab + 16 + std::max((size_t)pl.KW * mma_x_stage_bytes(tpu * g.d, mma_x_tokens_min(pl.NT)), (size_t)mma_group(pl.RW, pl.NT, true) * pl.KW * 64 * pl.NT * 16) <= 160 * 1024;
}
static bool mma_fuses_silu(const sq_matrix* mats, int n, int B, const void* x, int64_t ldx) {
    return mma_silu_shape(mats, n, B) && ldx % 8 == 0 && ((uintptr_t)x & 15) == 0 && !small_takes_gemm_route(mats, n, B, x, ldx);
}

// Estimated microseconds of that kernel for d = 4 pieces that share a launch at 17 to 32 rows, fitted to 400 products (9 %): weights (and more of them
// where codebooks leave a CU few waves), column slices and their sums, waves and rounds of a wave, results.
static float mma_us(const sq_matrix* mats, int n, int B) {
    const MmaPlan pl = mma_plan(mats[0], B);
    float rows = 0.f;
    for (int i = 0; i < n; ++i) rows += (float)mats[i].R * 1e-6f;
    return 4.86f + 0.106f * rows * mats[0].C * (mma_table_bytes(mats[0]) > 64 * 1024 ? 1.43f : 1.f) + (pl.ks > 1 ? 2.8f + 1.58f * pl.ks * B * rows : 0.f) +
           0.29f * pl.KW + 0.69f * pl.RW + 2.9f * B * rows;
}

// How many d = 4 pieces, the first one on, take the kernel of sq_mid.h at 17 to SQ_SMALL_BMAX rows; room: bytes for its sums.  With two tiles of activation rows
// the decode-time kernel's waves are few and add long sums (most where codebooks of 128 KB leave it five, which splits rows); there every wave has its own rows.
// Taken where it is estimated 8 % faster, as both estimates err by that much: of 400 products of 256 to 19000 rows and 512 to 10000 columns a third, at 0.86 of the
// time in the mean.  us, decode-time kernel / that one, at 17 / 32 rows: 2 x 18944 x 3584 with four books of 12-bit tags 39.9 / 42.0 and 29.9 / 27.9, 24074 x 1152 so
// 12.4 / 12.4 and 10.8 / 10.7; 4864 x 896, 8-bit, 7.9 / 8.0 and 5.6 / 5.5; 16546 x 832, 10-bit, 10.1 / 10.4 and 8.1 / 8.3; not 2570 x 2304, 12-bit in two books,
// 8.9 / 9.1 and 11.3 / 10.5.  At 16 rows it is the slower one for most (18944 x 3584 in four books twice, at 12: 21.5, 32.6).  A gate|up pair that
// mma_silu_shape takes stays, so that with and without SiLU it has the same sums.
// (Products below 2 M weights are a launch's length either way, and stay: 464 x 512, 12-bit, 6.4 and 7.4.  Rows below 512 columns were not measured.)
constexpr int MID_SMALL_T = 17, MID_SMALL_C = 512, MID_SMALL_WEIGHTS = 2 << 20;
static int mid_len(const sq_matrix* mats, int n, int B, size_t room, MidPlan& planned) {
    const sq_matrix& m0 = mats[0];
    if (B < MID_SMALL_T || B > SQ_SMALL_BMAX || m0.d != 4 || m0.C < MID_SMALL_C || mma_silu_shape(mats, n, B)) return 0;
    int k = 0;
    int64_t weights = 0;
    while (k < n && k < MID_PIECES && mma_shape(mats[k]) && mats[k].R > 0 && !stream_rows(mats[k], B) && mats[k].d == 4 && mats[k].bits == m0.bits &&
           mats[k].W == m0.W && mats[k].G == m0.G) weights += (int64_t)mats[k++].R * m0.C;
    if (weights < MID_SMALL_WEIGHTS || !mma_table_bytes(m0)) return 0;
    planned = mid_plan(mats, k, B, room);
    return planned.us < 0.92f * mma_us(mats, k, B) ? k : 0;
}
// For tests: that number where the workspace holds whatever sums there are.
extern "C" __attribute__((visibility("default"))) int32_t sq_mid_pieces_for_tests(const sq_matrix* mats, int32_t n, int32_t B) {
    MidPlan planned;
    return mid_len(mats, n, B, SIZE_MAX, planned);
}

// What the pieces' kernels keep side by side; not what a launch has from the workspace's first byte on for itself (small_workspace).
// tight: the pieces that can run without partial sums do
static size_t small_need(const sq_matrix* mats, int n, int B, bool tight) {
    size_t tot = 0;
    for (int i = 0; i < n; ++i) {
        if (stream_rows(mats[i], B)) continue;                   // its partial sums live in the workspace header
        if (mma_rows(mats[i])) tot += tight && (mma_whole_row(mats[i], B).KW || mma_without_room(mats[i], B)) ? 0 : mma_part_bytes(mats[i], B);
        else if (mats[i].perms && fast_shape(mats[i])) tot += xp_bytes(mats[i], B);
    }
    return tot;
}

size_t small_workspace(const sq_matrix* mats, int n, int B) {
    size_t need = small_need(mats, n, B, false);
    const bool orders = has_orders(mats, n);
    PlanePlan plane;
    MidPlan mid;
    for (int i = 0; i < n; ++i) {
        if (const int k = orders ? 0 : vector_decoded(mats + i, n - i, B); k > 0) {
            need = std::max(need, decoded_workspace(mats + i, k, B));
            i += k - 1;
        } else if (const int k = plane_product_len(mats + i, n - i, B, plane); k > 0) {
            need = std::max(need, plane_product_workspace(mats + i, k, B, &plane));
            i += k - 1;
        } else if (const int k = sieve_len(mats + i, n - i, B); k > 0) {
            need = std::max(need, sieve_workspace(mats + i, k, B));
            i += k - 1;
        } else if (const int k = mid_len(mats + i, n - i, B, SIZE_MAX, mid); k > 0) {
            need = std::max(need, mid_workspace(mats + i, k, B, &mid));
            i += k - 1;
        }
    }
    return need;
}
size_t small_workspace_least(const sq_matrix* mats, int n, int B) { return small_need(mats, n, B, true); }

bool small_uses_sums(const sq_matrix* mats, int n) {
    for (int i = 0; i < n; ++i)
        if (mats[i].R > 0 && stream_shape(mats[i])) return true;
    return false;
}

// Pieces [0, cnt) share format and row length: one persistent launch (+ one reduction per piece if ks > 1).  act: mma_fuses_silu
// holds for them.  whole: the workspace has no room for partial sums that mma_whole_row can do without.
static int launch_mma_group(const sq_matrix* mats, int cnt, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype,
                            int64_t ldy, int B, char* ws, size_t& ws_off, int cus, hipStream_t s, bool act = false, bool whole = false) {
    const sq_matrix& m0 = mats[0];
    MmaPlan pl = mma_plan(m0, B);
    if (pl.ks > 1 && !act && (whole || mma_whole_row_pays(m0, cnt, pl))) {
        const MmaPlan one = mma_whole_row(m0, B);
        if (one.KW) pl = one;
    }
    MmaArgs a;
    a.n = cnt;
    a.x = (const uint16_t*)x; a.ldx = ldx; a.y = y; a.ldy = ldy; a.B = B; a.x_dtype = x_dtype; a.y_dtype = y_dtype;
    a.U = row_units(m0.C, m0.d, m0.bits);
    a.ks = pl.ks;
    a.act = act;
    a.broken = !whole_units(m0);
    const int per = act ? 2 : 1;                                 // pieces whose tiles a workgroup walks in turn
    a.table_bytes = (int)mma_table_bytes(m0) * per;
    const int threads = pl.KW * 64;
    // LDS behind the codebook: the waves' accumulators of the tiles between two barriers (MMA_TT tiles when the codebook
    // is read through the cache; with the codebook in LDS as many as the workgroup walks, if they fit: sized below)
    const size_t red_tile = (size_t)pl.KW * 64 * pl.NT * 16;
    const int pft = mma_group(pl.RW, pl.NT, act);
    a.tg = a.table_bytes ? pft : 0;
    const int tpu = unit_dwords(m0.bits) * 32 / m0.bits;
    // 9 to 16 rows go through the staging areas at once where 16 tokens fit (7 waves of 12-bit tags: 7.6 us, in two parts 8.4)
    a.xt = !a.table_bytes || (B > 8 && (size_t)a.table_bytes + 16 + (size_t)pl.KW * mma_x_stage_bytes(tpu * m0.d, 16) <= 160 * 1024) ? 16 : mma_x_tokens_min(pl.NT);
    const size_t xstage = (size_t)pl.KW * mma_x_stage_bytes(tpu * m0.d, a.xt);      // the waves' activation staging areas (same LDS)
    size_t smem = (size_t)a.table_bytes + 16 + std::max(xstage, a.table_bytes ? (size_t)a.tg * red_tile : pl.KW > 1 ? (size_t)MMA_TT * red_tile : 0);
    int rc = SQ_EUNSUPPORTED;
#define SQ_CASE(BI, DD) if (m0.bits == BI && m0.d == DD) rc = launch_mma_b##BI##d##DD(OP, a, pl.RW, pl.NT, GRID, threads, smem, s)
#define OP 1
#define GRID 0
    SQ_CASE(16, 8); SQ_CASE(12, 4); SQ_CASE(10, 4); SQ_CASE(8, 4);
#undef OP
#undef GRID
    if (rc < 1) return rc < 0 ? rc : fail(SQ_ELAUNCH, "sq_linear_small: kernel does not fit a CU");
    const int slots = cus * rc;                                  // workgroups resident at once
    int64_t rows_total = 0;
    for (int k = 0; k < cnt; ++k) rows_total += mats[k].R;
    int wg = 0;
    for (int k = 0; k < cnt; ++k) {
        MmaPiece& P = a.p[k];
        P.m = mats[k];
        const sq_matrix& mk = mats[k];
        P.tiled = tiled_piece(mk);
        P.part = nullptr;
        if (pl.ks > 1) {
            P.part = (float*)(ws + ws_off);
            ws_off += mma_part_bytes(mats[k], B);
        }
        const int ntiles = (mats[k].R + 15) / 16;
        int nshare = (int)((mats[k].R * per * (int64_t)slots / rows_total) / pl.ks);
        if (nshare > ntiles) nshare = ntiles;
        if (nshare < 1) nshare = 1;
        P.wg_begin = wg;
        P.wg_count = nshare * pl.ks;
        if (!act || k) wg += P.wg_count;
    }
    if (act) a.n = 1;                                            // (every workgroup begins with piece 0)
    for (int k = cnt; k < GEMV_MAX_PIECES; ++k) a.p[k] = a.p[0];
    if (a.table_bytes) {
        int most = 1;                                            // most tiles one workgroup walks
        for (int k = 0; k < cnt; ++k) {
            const int ntiles = (mats[k].R + 15) / 16, nshare = a.p[k].wg_count / pl.ks;
            most = std::max(most, (ntiles + nshare - 1) / nshare * per);
        }
        const size_t room = (size_t)(160 * 1024) / rc - a.table_bytes - 16;
        int fit = (int)(room / red_tile) / pft * pft;
        a.tg = std::min((most + pft - 1) / pft * pft, std::max(fit, pft));
        smem = (size_t)a.table_bytes + 16 + std::max(xstage, (size_t)a.tg * red_tile);
    }
#define OP 0
#define GRID wg
    rc = SQ_EUNSUPPORTED;
    SQ_CASE(16, 8); SQ_CASE(12, 4); SQ_CASE(10, 4); SQ_CASE(8, 4);
#undef OP
#undef GRID
#undef SQ_CASE
    if (rc) return rc;
    return pl.ks > 1 ? launch_slice_sum(a.p, cnt, pl.ks, B, y, y_dtype, ldy, s) : SQ_OK;
}

// (Pieces with column orders would gather the producer's three operands through every order of a run from memory:
// measured 39.9 against 21.4 us for the stand-alone add + norm followed by the product on the masked 27B q|k|v stack,
// 43.5 against 30.6 us on gate|up.  They take the two launches.)
bool small_fuses_producer(const sq_matrix* mats, int n, int B) {
    if (B != 1 || n < 1 || n > GEMV_MAX_PIECES_STREAM) return false;
    for (int i = 0; i < n; ++i)
        if (mats[i].R <= 0 || !stream_rows(mats[i], 1) || mats[i].bits != mats[0].bits || mats[i].G != mats[0].G || mats[i].perms) return false;
    return true;
}

// SiLU(gate) * up written by the product itself: the two pieces are a gate and an up projection of one shape on the
// tag-stream kernel (no column orders, cut into the same runs), at most 8 activation rows (one pass)
bool small_fuses_silu(const sq_matrix* mats, int n, int B) {
    if (n != 2 || B < 1 || B > 8) return false;
    const sq_matrix &g = mats[0], &u = mats[1];
    if (g.R <= 0 || g.R != u.R || g.C != u.C || g.bits != u.bits || g.G != u.G || g.perms || u.perms) return false;
    // (the same cut into runs; the other fields of stream_runs describe each piece's own buffer and may differ)
    if (!stream_rows(g, B) || !stream_rows(u, B) || stream_runs_of(g) != stream_runs_of(u) || stream_run_max_of(g) != stream_run_max_of(u) ||
        g.stream_groups != u.stream_groups)
        return false;
    if (stream_geom_of(g).NV > 16 || stream_group_len(mats, 2) != 2) return false;
    return stream_pass_rows(B) >= B;
}

int launch_small_silu(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* act, int64_t ld_act, int B,
                      void* sums, hipStream_t s, const sq_producer* from) {
    const bool x_ok = (B == 1 || ldx % 8 == 0) && (((uintptr_t)x & 15) == 0);
    const char *xb = (const char*)x, *xe = xb + ((int64_t)(B - 1) * ldx + mats[0].C) * 2, *ob = (const char*)act, *oe = ob + ((int64_t)(B - 1) * ld_act + mats[0].R) * 2;
    if (!from && mma_fuses_silu(mats, n, B, x, ldx) && (oe <= xb || xe <= ob)) {     // (act written over x: the two launches)
        size_t off = 0;
        return launch_mma_group(mats, 2, x, x_dtype, ldx, act, x_dtype, ld_act, B, nullptr, off, device_cus(), s, true);
    }
    if (!small_fuses_silu(mats, n, B) || !(x_ok || from) || (from && !small_fuses_producer(mats, n, B)))
        return fail(SQ_EUNSUPPORTED, "sq_linear_small_silu: no fused kernel for this stack (run sq_linear_small, then sq_silu_mul)");
    if (!sums) return fail(SQ_EWORKSPACE, "sq_linear_small_silu: these pieces need a workspace (its header holds their partial sums)");
    return launch_stream_group(mats, 2, x, x_dtype, ldx, nullptr, x_dtype, 0, B, (char*)sums, s, from, act, ld_act);
}

int launch_small(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype,
                 int64_t ldy, int B, void* ws, size_t ws_bytes, void* sums, hipStream_t s, const sq_producer* from) {
    if (from && !small_fuses_producer(mats, n, B)) return fail(SQ_EUNSUPPORTED, "sq_linear_small_from: no fused kernel for this stack");
    const bool tight = small_need(mats, n, B, false) > ws_bytes, orders = has_orders(mats, n);
    if (tight && small_workspace_least(mats, n, B) > ws_bytes)
        return fail(SQ_EWORKSPACE, "sq_linear_small: workspace %zu < %zu", ws_bytes, small_workspace(mats, n, B));
    const int cus = device_cus();
    const bool x_ok = (B == 1 || ldx % 8 == 0) && (((uintptr_t)x & 15) == 0);   // 16-byte activation loads
    size_t ws_off = 0;
    PlanePlan plane;
    MidPlan mid;
    int i = 0;
    while (i < n) {
        const sq_matrix& m0 = mats[i];
        if (m0.R == 0) { ++i; continue; }
        const int ud = unit_dwords(m0.bits);
        if (stream_rows(m0, B) && (x_ok || from)) {
            if (!sums) return fail(SQ_EWORKSPACE, "sq_linear_small: these pieces need a workspace (its header holds their partial sums)");
            int j = i + 1;
            while (j < n && j - i < GEMV_MAX_PIECES_STREAM && stream_rows(mats[j], B) && mats[j].bits == m0.bits && mats[j].G == m0.G && mats[j].R > 0) ++j;
            j = i + stream_group_len(mats + i, j - i);
            int rc = launch_stream_group(mats + i, j - i, x, x_dtype, ldx, y, y_dtype, ldy, B, (char*)sums, s, from);
            if (rc) return rc;
            i = j;
            continue;
        }
        if (const int k = orders || !x_ok ? 0 : vector_decoded(mats + i, n - i, B); k > 0 && decoded_workspace(mats + i, k, B) <= ws_bytes) {
            if (const int rc = launch_decoded(mats + i, k, x, x_dtype, ldx, y, y_dtype, ldy, B, ws, s, /*wide=*/true)) return rc;
            i += k;
            continue;
        }
        if (const int k = !x_ok ? 0 : plane_product_len(mats + i, n - i, B, plane); k > 0 && plane_product_workspace_least(mats + i, k, B, &plane) <= ws_bytes) {
            if (const int rc = launch_plane_product(mats + i, k, x, x_dtype, ldx, y, y_dtype, ldy, B, ws, ws_bytes, s, &plane)) return rc;
            ws_off += small_need(mats + i, k, B, tight);
            i += k;
            continue;
        }
        if (const int k = !x_ok ? 0 : sieve_len(mats + i, n - i, B); k > 0 && sieve_workspace_least(mats + i, k, B) <= ws_bytes) {
            if (const int rc = launch_sieve(mats + i, k, x, x_dtype, ldx, y, y_dtype, ldy, B, ws, ws_bytes, s)) return rc;
            ws_off += small_need(mats + i, k, B, tight);         // (what was counted for them)
            i += k;
            continue;
        }
        if (const int k = !x_ok || !mid_x_ok(ldx, B) ? 0 : mid_len(mats + i, n - i, B, ws_bytes, mid); k > 0) {
            if (const int rc = launch_mid(mats + i, k, x, x_dtype, ldx, y, y_dtype, ldy, B, ws, ws_bytes, s, &mid)) return rc;
            ws_off += small_need(mats + i, k, B, tight);
            i += k;
            continue;
        }
        if (B <= 2 && x_ok && segs_shape(m0) && (B == 1 || mma_table_bytes(m0) > 64 * 1024)) {
            // d = 4 rows of whole segments at one activation row, and at two when the codebooks leave a CU room for one
            // workgroup only: the row-segment kernel (7B-shaped layer, 12-bit tags: 41.7 us at one row against 50 on the
            // matrix-core kernel, 52.4 against 49.8 at two; four codebooks of 4096: 71-73 against 78-83 at two)
            int j = i + 1;
            while (j < n && j - i < 4 && segs_shape(mats[j]) && mats[j].W == m0.W && mats[j].G == m0.G) ++j;
            if (segs_fits(mats + i, j - i, B, cus)) {
                int rc = launch_segs_group(mats + i, j - i, x, x_dtype, ldx, y, y_dtype, ldy, B, cus, s);
                if (rc) return rc;
                ws_off += small_need(mats + i, j - i, B, tight);     // (what was counted for them)
                i = j;
                continue;
            }
        }
        if (mma_rows(m0) && x_ok && !(tight && mma_without_room(m0, B))) {
            int j = i + 1;
            while (j < n && j - i < GEMV_MAX_PIECES && mma_rows(mats[j]) && mats[j].bits == m0.bits && mats[j].d == m0.d &&
                   mats[j].W == m0.W && mats[j].G == m0.G && mats[j].R > 0)
                ++j;
            int rc = launch_mma_group(mats + i, j - i, x, x_dtype, ldx, y, y_dtype, ldy, B, (char*)ws, ws_off, cus, s, false, tight);
            if (rc) return rc;
            i = j;
            continue;
        }
        const Plan pl = (fast_shape(m0) && x_ok) ? plan_for(m0.W / ud, m0.bits, m0.d) : Plan{0, 0, 0};
        if (pl.TS == 0 && !m0.tags)
            return fail(SQ_EUNSUPPORTED, "sq_linear_small: a matrix held as its tag stream only needs 16-byte aligned x with ldx %% 8 == 0");
        if (pl.TS == 0) {
            int rc = launch_small_generic(mats + i, 1, x, x_dtype, ldx, y, y_dtype, ldy, B, s);
            if (rc) return rc;
            ws_off += small_need(mats + i, 1, B, tight);
            ++i;
            continue;
        }
        // pieces i .. j-1 share one launch when their format, geometry and codebook size agree
        const int U = m0.W / ud;
        const size_t tab0 = (size_t)m0.G * ((size_t)1 << m0.bits) * m0.d * 2;
        int j = i + 1;
        while (j < n && j - i < GEMV_MAX_PIECES && fast_shape(mats[j]) && mats[j].bits == m0.bits && mats[j].d == m0.d &&
               mats[j].W == m0.W && mats[j].G == m0.G && mats[j].R > 0)
            ++j;
        GemvArgs a;
        a.n = j - i;
        a.x = (const uint16_t*)x; a.ldx = ldx; a.y = y; a.ldy = ldy; a.B = B;
        a.x_dtype = x_dtype; a.y_dtype = y_dtype; a.TS = pl.TS;
        a.table_bytes = tab0 <= 128 * 1024 ? (int)tab0 : 0;
        const int wpr = pl.TS > 64 ? pl.TS / 64 : 1;
        int64_t rows_total = 0;
        for (int k = i; k < j; ++k) rows_total += mats[k].R;
        for (int k = i; k < j; ++k) {
            GemvPiece& P = a.p[k - i];
            P.m = mats[k];
            P.U = U;
            P.xp = nullptr;
            if (mats[k].perms) {
                uint16_t* xp = (uint16_t*)((char*)ws + ws_off);
                ws_off += xp_bytes(mats[k], B);
                const int Mx = mats[k].M > 1 ? mats[k].M : 1;
                const int64_t tot = (int64_t)Mx * B * mats[k].C;
                hipLaunchKernelGGL(permute_x_kernel, dim3((unsigned)((tot + 255) / 256)), dim3(256), 0, s,
                                   (const uint16_t*)x, ldx, x_dtype, mats[k].perms, Mx, B, mats[k].C, xp);
                int rc = check_launch("sq_linear_small(permute_x)");
                if (rc) return rc;
                P.xp = xp;
            }
        }
        for (int k = j - i; k < GEMV_MAX_PIECES; ++k) a.p[k] = a.p[0];
        for (int b0 = 0; b0 < B;) {
            const int left = B - b0;
            int nbt = left >= 3 ? 4 : left;                          // (three rows: 16 us as four, 20 as two and one, 2048 x 2048)
            // fewer activation rows per pass when the registers or the workgroup width do not allow more
            while (nbt > 1 && (cfg_xw(m0.bits, m0.d, pl.S, nbt) > 192 || cfg_lb(m0.bits, m0.d, pl.S, nbt) < wpr * 64)) nbt >>= 1;
            const int lb = cfg_lb(m0.bits, m0.d, pl.S, nbt);
            int nwaves = pl.nwaves;
            // a codebook that leaves room for one workgroup per CU: make that workgroup as wide as allowed
            if (nwaves * 64 > lb || a.table_bytes > 80 * 1024) nwaves = (lb / 64) / wpr * wpr;
            const int ngrp = pl.TS > 64 ? nwaves / wpr : nwaves * (64 / pl.TS);
            const size_t smem = (size_t)a.table_bytes + (wpr > 1 ? (size_t)GEMV_PF * ngrp * wpr * nbt * sizeof(float) : 0);
            // persistent grid: workgroups per CU bounded by LDS and wave slots, split over the pieces by rows
            int rc = SQ_EUNSUPPORTED;
#define SQ_CASE(BI, DD) if (m0.bits == BI && m0.d == DD) rc = launch_gemv_b##BI##d##DD(OP, a, pl.S, nbt, GRID, nwaves * 64, smem, s)
#define OP 1
#define GRID 0
            SQ_CASE(16, 8); SQ_CASE(12, 4); SQ_CASE(10, 4); SQ_CASE(8, 4);      // workgroups that fit on a CU
#undef OP
#undef GRID
            if (rc < 1) return rc < 0 ? rc : fail(SQ_ELAUNCH, "sq_linear_small: kernel does not fit a CU");
            const int per_cu = rc;
            const int64_t row_quant = (int64_t)ngrp * GEMV_PF;
            const int grid_target = cus * per_cu;
            int wg_begin = 0;
            for (int k = i; k < j; ++k) {
                GemvPiece& P = a.p[k - i];
                int cnt = (int)((mats[k].R * (int64_t)grid_target + rows_total - 1) / rows_total);
                const int most = (int)((mats[k].R + row_quant - 1) / row_quant);
                if (cnt > most) cnt = most;
                if (cnt < 1) cnt = 1;
                P.wg_begin = wg_begin;
                P.wg_count = cnt;
                wg_begin += cnt;
            }
            a.b0 = b0;
            rc = SQ_EUNSUPPORTED;
#define OP 0
#define GRID wg_begin
            SQ_CASE(16, 8); SQ_CASE(12, 4); SQ_CASE(10, 4); SQ_CASE(8, 4);
#undef OP
#undef GRID
#undef SQ_CASE
            if (rc) return rc;
            b0 += nbt;
        }
        i = j;
    }
    return SQ_OK;
}

}  // namespace sq
