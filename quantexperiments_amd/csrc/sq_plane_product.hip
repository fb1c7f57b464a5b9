// Codebook product for 17 to 128 activation rows, d = 8 with 16-bit tags, a column of the codebook ("plane", sq_planes.hip) at a time.
//
// What gathers codewords from L2 is bound by its requests, 64 bytes moved for 16: 2 x 18944 x 3584 takes 88 us at 17 rows and 91 at 64.
// LDS holds one of the codebook's eight columns.  A workgroup stages column e, looks element e of its rows' tags up and multiplies with
// the same elements of the activations: an eighth of the sum over columns, so nothing is multiplied in vain (the sieve of sq_sieve.hip, which
// serves up to 16 rows, multiplies eight times as much).  The eight workgroups of a set of rows sit on one XCD, whose L2 reads the tags once; slice_sum_kernel
// adds their fp32 sums.  Where those are many, a workgroup takes two columns one after the other, which halves them.
//
//   workgroup   8 waves, each with up to TW tiles of 16 weight rows x NT of 16 activation rows at a time, in rounds
//   K           pairs of steps, 64 chunks: step s of lane group g is chunks 64 pair + 16 g + 8 s .. + 7 of the column
//   tags        128 bytes of a row per pair.  The lanes of a matrix operand are different rows, and a request of 16 bytes a row and lane costs the
//               address unit a clock each; so lanes 2 i and 2 i + 1 ask for 32 bytes of the same row, first of row 2 i, then of 2 i + 1, and exchange
//               halves (55 -> 48 us at 16 rows, 75 -> 67 at 64).  A tile's tags are asked for as soon as the last ones have been used
//   X           in the order of the operands (pp_order_kernel), 1 KB a step and token tile, straight to registers
//
// Bound: LDS look-ups, two thirds of a CU's time (2 x 18944 x 3584 at 24 / 64 rows 69 and 64 %, 72 % of that bank conflicts of 64 random two-byte elements),
// then the way of tags, activations and columns, which a workgroup that fills a CU does not overlap; and the sums (4 or 8 T R fp32 written and read: the
// launch that adds them takes 9 us of 60 at 64 rows).  us at 24 / 48 / 64 / 96 rows before and now: 2 x 18944 x 3584 89 / 88 / 91 / 99 -> 53 / 56 / 60 / 82, 18944 x 3584 49 / 54 / 56 / 60 ->
// 34 / 38 / 41 / 47, 3584 x 18944 54 / 56 / 58 / 63 -> 34 / 37 / 40 / 48, q|k|v of 7168 x 5120 35 / 33 / 36 / 45 -> 28 / 30 / 31 / 36.
#include <algorithm>
#include "sq_planes.h"
#include "sq_slices.h"

namespace sq {

constexpr int PP_WAVES = 8, PP_MAX_NT = 8;
constexpr int PP_TILES[PP_MAX_NT + 1] = {0, 0, 5, 5, 5, 4, 3, 2, 2};     // most tiles of a wave at once, by token tiles: what 256 registers hold
typedef __attribute__((address_space(3))) void* pp_lptr_t;

// Codebooks in plane order, and the activations as fp16 operands of the matrix instruction: 1 KB per plane, pair of steps (64 chunks),
// step and token tile, [lane][8]: token 16 tile + lane % 16, chunks 64 pair + 16 (lane / 16) + 8 step .. + 7; zeros past the last token and chunk.
struct PpOrderArgs {
    const uint16_t* table[MID_PIECES];
    uint16_t* planes;
    const uint16_t* x;
    unsigned char* xf;
    int64_t ldx;
    int pieces, T, NT, n, pairs, bf;
};

__global__ __launch_bounds__(64) void pp_order_kernel(PpOrderArgs a) {
    constexpr int PER = PLANE / 8;
    int u = (int)blockIdx.x * 64 + (int)threadIdx.x;
    u32x4 v[8];
    unsigned char* dst;
    int64_t step;                            // bytes from plane to plane
    if (u < a.pieces * PER) {
        const int piece = u / PER, at = u - piece * PER;
        const uint16_t* table = a.table[0];
#pragma unroll
        for (int i = 1; i < MID_PIECES; ++i) table = i == piece ? a.table[i] : table;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = *reinterpret_cast<const u32x4*>(table + (int64_t)at * 64 + i * 8);
        dst = reinterpret_cast<unsigned char*>(a.planes + (int64_t)piece * 8 * PLANE + at * 8);
        step = PLANE * 2;
    } else {
        u -= a.pieces * PER;
        const int groups = a.pairs * 8, t = u / groups, g = u - t * groups;      // token, group of eight chunks
        if (t >= a.NT * 16) return;
        const bool real = t < a.T && g * 8 < a.n;
        const uint16_t* src = a.x + (int64_t)(real ? t : 0) * a.ldx + (real ? g : 0) * 64;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = *reinterpret_cast<const u32x4*>(src + i * 8);
            if (a.bf) { v[i].x = bf2h_x2(v[i].x); v[i].y = bf2h_x2(v[i].y); v[i].z = bf2h_x2(v[i].z); v[i].w = bf2h_x2(v[i].w); }
            if (!real) v[i] = u32x4{0u, 0u, 0u, 0u};
        }
        const int pair = g >> 3, lane = (t & 15) + 16 * ((g & 7) >> 1), s = g & 1;
        dst = a.xf + (((int64_t)pair * 2 + s) * a.NT + (t >> 4)) * 1024 + lane * 16;
        step = (int64_t)a.pairs * 2 * a.NT * 1024;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) *reinterpret_cast<u32x4*>(dst + e * step) = plane_of(v, e);
}

struct PpPiece {
    sq_matrix m;
    const uint16_t* planes;                  // of its codebook
    float* part;                             // fp32 [8 / pl, T, R rounded up to 4]
    int job0, parts;                         // first job; parts of the rows, a job each
};
struct PpArgs {
    PpPiece p[MID_PIECES];
    const unsigned char* xf;
    int n, T, chunks, pairs, jobs, pl;       // pl: planes of a workgroup, one after the other
};

template <int TW, int NT>
__global__ __launch_bounds__(64 * PP_WAVES) void plane_product_kernel(PpArgs a) {
    constexpr int PF = 2;                    // products that look-ups run ahead (1 and 3: the same)
    extern __shared__ __attribute__((aligned(16))) unsigned char pp_lds[];
    const int tid = (int)threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pgs = 8 / a.pl, slot = (int)blockIdx.x >> 3, pg = slot % pgs, job = slot / pgs * 8 + ((int)blockIdx.x & 7);
    if (job >= a.jobs) return;
    int pi = 0;
    while (pi + 1 < a.n && job >= a.p[pi + 1].job0) ++pi;
    const PpPiece& P = a.p[pi];
    const sq_matrix& m = P.m;
    const int part = job - P.job0;
    const int ntiles = (m.R + 15) >> 4, w0 = (int)((int64_t)ntiles * part / P.parts), wn = (int)((int64_t)ntiles * (part + 1) / P.parts) - w0;
    const int mine0 = w0 + wn * wave / PP_WAVES, mine1 = w0 + wn * (wave + 1) / PP_WAVES;      // this wave's tiles
    const int rounds = ((wn + PP_WAVES - 1) / PP_WAVES + TW - 1) / TW;
    const char* tags = reinterpret_cast<const char*>(m.tags);
    const uint32_t end = (uint32_t)a.chunks * 2 - 16;                                        // the last eight tags' place in a row
    const uint32_t row_bytes = (uint32_t)m.W * 4u, last_row = (uint32_t)(m.R - 1) * row_bytes;
    const unsigned char* xf = a.xf + lane * 16;

    for (int round = 0; round < rounds; ++round) {
        const int tile0 = mine0 + round * TW;
        const bool work = tile0 < mine1;
        uint32_t to[TW];                                         // the even row of this lane's pair
#pragma unroll
        for (int i = 0; i < TW; ++i) to[i] = (uint32_t)min(min(tile0 + i, ntiles - 1) * 16 + (li & 14), m.R - 1) * (uint32_t)m.W * 4u;
        float4v acc[TW][NT];
#pragma unroll
        for (int i = 0; i < TW; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[i][t] = float4v{0.f, 0.f, 0.f, 0.f};
        for (int q = 0; q < a.pl; ++q) {
            const int e = pg * a.pl + q;
            if (round == 0 || a.pl > 1) {
                if (round > 0 || q > 0) __syncthreads();         // the plane before it has been read
                const uint16_t* src = P.planes + (int64_t)e * PLANE;
                const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)src, 0, PLANE * 2, 0x00027000);
#pragma unroll
                for (int k = 0; k < PLANE * 2 / (64 * PP_WAVES * 16); ++k)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (pp_lptr_t)(pp_lds + (k * PP_WAVES + wave) * 1024), 16, tid * 16, k * PP_WAVES * 1024, 0, 0);
            }
            u32x4 tg[TW][2];
            half8v xb[2][NT];
            auto load_tags = [&](int pair, int i) {
#pragma unroll
                for (int s = 0; s < 2; ++s) tg[i][s] = *reinterpret_cast<const u32x4*>(tags + (min(to[i] + s * row_bytes, last_row) + min((uint32_t)(pair * 128 + lg * 32 + (li & 1) * 16), end)));
            };
            auto load_x = [&](int pair, int s) {
                const unsigned char* from = xf + (((int64_t)e * a.pairs + pair) * 2 + s) * (NT * 1024);
#pragma unroll
                for (int t = 0; t < NT; ++t) xb[s][t] = *reinterpret_cast<const half8v*>(from + t * 1024);
            };
            if (work) {
#pragma unroll
                for (int i = 0; i < TW; ++i) load_tags(0, i);
                load_x(0, 0);
                load_x(0, 1);
            }
            if (round == 0 || a.pl > 1) {
                __builtin_amdgcn_s_waitcnt(0);                   // this wave's part of the plane has landed
                __syncthreads();
            }
            if (!work) continue;
            const uint16_t* plane = reinterpret_cast<const uint16_t*>(pp_lds);
            for (int pair = 0; pair < a.pairs; ++pair) {
                const int next = min(pair + 1, a.pairs - 1);
                uint32_t sel[2];                                 // bytes of two looked-up elements, or zeros past the row's last chunk
#pragma unroll
                for (int s = 0; s < 2; ++s) sel[s] = pair * 64 + lg * 16 + s * 8 < a.chunks ? 0x05040100u : 0x0C0C0C0Cu;
                auto look_up = [&](int z) {
                    u32x4 t;
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        const uint32_t own = tg[z % TW][z / TW][w], other = tg[z % TW][1 - z / TW][w];
                        const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)other, 0xB1, 0xF, 0xF, true);      // of lane ^ 1
                        t[w] = (li & 1) == z / TW ? own : got;
                    }
                    u32x4 o;
#pragma unroll
                    for (int w = 0; w < 4; ++w) o[w] = __builtin_amdgcn_perm((uint32_t)plane[t[w] >> 16], (uint32_t)plane[t[w] & 0xFFFFu], sel[z / TW]);
                    return __builtin_bit_cast(half8v, o);
                };
                half8v wf[PF + 1];
#pragma unroll
                for (int z = 0; z < PF && z < 2 * TW; ++z) wf[z] = look_up(z);
#pragma unroll
                for (int z = 0; z < 2 * TW; ++z) {
                    if (z + PF < 2 * TW) wf[(z + PF) % (PF + 1)] = look_up(z + PF);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[z % TW][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[z % (PF + 1)], xb[z / TW][t], acc[z % TW][t], 0, 0, 0);
                    if (z == TW - 1) load_x(next, 0);
                    if (z >= TW) load_tags(next, z - TW);
                }
                load_x(next, 1);
            }
        }
        if (!work) continue;
        // ---- lane: token 16 t + li, weight rows 16 tile + 4 lg .. + 3
        const int ld = (m.R + 3) & ~3;
        float* out = P.part + (int64_t)pg * a.T * ld;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if (t * 16 + li >= a.T) continue;
#pragma unroll
            for (int i = 0; i < TW; ++i) {
                const int r = (tile0 + i) * 16 + lg * 4;
                if (tile0 + i < mine1 && r < m.R) *reinterpret_cast<float4v*>(out + (int64_t)(t * 16 + li) * ld + r) = acc[i][t];
            }
        }
    }
}

// ------------------------------------------------------------------------------------------ host

static bool pp_shape(const sq_matrix& m) {
    return m.R > 0 && m.tags && m.d == 8 && m.bits == 16 && m.G == 1 && !m.row_book && !m.perms && m.C % 64 == 0 && m.W == m.C / 16 &&
           (((uintptr_t)m.tags | (uintptr_t)m.table) & 15) == 0 && (int64_t)m.R * m.W < ((int64_t)1 << 30);
}

// Parts of the rows so that every CU has a workgroup, tiles of a wave in as few rounds as registers allow, evenly; one plane a workgroup or
// two, whichever is estimated to take less.  Microseconds, fitted to 203 products (6 %): launches and activations; staging; look-ups and
// products; activations to registers; sums.  (planes: that many a workgroup, if it is given)
static PlanePlan pp_plan(const sq_matrix* mats, int n, int T, int planes = 0) {
    const int cus = device_cus();
    int64_t tiles = 0, rows = 0;
    for (int i = 0; i < n; ++i) tiles += (mats[i].R + 15) / 16, rows += mats[i].R;
    PlanePlan best{};
    for (int pl = planes ? planes : 1; pl <= (planes ? planes : 2); ++pl) {
        PlanePlan p{};
        p.nt = (T + 15) / 16; p.pl = pl;
        int64_t per = 0;                     // most tiles of a part
        for (int i = 0; i < n; ++i) {
            const int64_t mine = (mats[i].R + 15) / 16;
            p.parts[i] = (int)std::max<int64_t>(1, std::min<int64_t>(mine, cus * pl / 8 * mine / tiles));
            per = std::max(per, (mine + p.parts[i] - 1) / p.parts[i]);
        }
        const int64_t wave = (per + PP_WAVES - 1) / PP_WAVES, rounds = (wave + PP_TILES[p.nt] - 1) / PP_TILES[p.nt];
        p.tw = (int)((wave + rounds - 1) / rounds);
        const double steps = (double)((mats[0].C / 8 + 63) / 64) * rounds * pl;
        p.us = 10.3 + 1.3 * n + 5.75e-6 * T * mats[0].C + 1.7 * (pl > 1 ? pl * rounds : 1) + steps * (p.tw * (0.36 + 0.016 * p.nt) + 0.0103 * p.nt) + 11.6e-6 / pl * T * rows;
        if (!best.pl || p.us < best.us) best = p;
    }
    return best;
}

static size_t pp_align(size_t n) { return (n + 255) & ~(size_t)255; }
static size_t pp_x_bytes(const sq_matrix* mats, int nt) { return (size_t)8 * ((mats[0].C / 8 + 63) / 64) * 2 * nt * 1024; }
static size_t pp_part_bytes(int R, int T, int pl) { return pp_align((size_t)(8 / pl) * T * ((R + 3) / 4 * 4) * 4); }

// how many of the pieces, the first one on, have a shape that the kernel takes
static int pp_fit(const sq_matrix* mats, int n, int T) {
    if (T < PLANE_PRODUCT_MIN_T || T > 16 * PP_MAX_NT || device_cus() < 64) return 0;
    int k = 0;
    while (k < n && k < MID_PIECES && pp_shape(mats[k]) && mats[k].C == mats[0].C) ++k;
    return k;
}

// What a launch keeps besides the sums, and the sums of so many rows in n pieces
static size_t pp_fixed_bytes(const sq_matrix* mats, int n, int nt) { return planes_bytes(n) + pp_x_bytes(mats, nt); }
static size_t pp_sums_bytes(int64_t rows, int n, int T, int pl) { return (size_t)(8 / pl) * T * 4 * (rows + 4 * n) + 256 * n; }

// The gathers from L2 take 8 us and 4.75 more per million tags up to 32 rows (fitted to 12 products: 10 %), and then what mid_plan says; here has
// to be estimated a seventh faster (8000 x 2048 at 32 / 64 rows 17.3 / 18.7 there, 20.8 / 25 here; 3584 x 3584 16.8 / 19.0, 17.7 / 21.7).  A decode step's
// products also need room for a fair part of their rows' sums in what sq_linear_small_noalloc has.
constexpr int PP_PART_ROWS = 4096;
int plane_product_group(const sq_matrix* mats, int n, int T, PlanePlan& p, const MidPlan* mid) {
    const int k = pp_fit(mats, n, T);
    double tags = 0.0;
    for (int i = 0; i < k; ++i) tags += (double)mats[i].R * mats[i].C / 8e6;
    if (tags < 2.0) return 0;                // (no product of that size gains; the estimates cost the host a microsecond)
    p = pp_plan(mats, k, T);
    if (T <= SQ_SMALL_BMAX && pp_fixed_bytes(mats, k, p.nt) + pp_sums_bytes(PP_PART_ROWS, k, T, p.pl) > SMALL_ROOM) return 0;
    return p.us < 0.85 * (T <= SQ_SMALL_BMAX ? 8.0 + 4.75 * tags : (double)(mid && k == n ? *mid : mid_plan(mats, k, T)).us) ? k : 0;
}

size_t plane_product_workspace(const sq_matrix* mats, int n, int T, const PlanePlan* planned) {
    const PlanePlan p = planned ? *planned : pp_plan(mats, n, T);
    size_t need = pp_fixed_bytes(mats, n, p.nt);
    for (int i = 0; i < n; ++i) need += pp_part_bytes(mats[i].R, T, p.pl);
    return need;
}
size_t plane_product_workspace_least(const sq_matrix* mats, int n, int T, const PlanePlan* planned) { return std::min(plane_product_workspace(mats, n, T, planned), SMALL_ROOM); }

typedef void (*pp_kernel_t)(PpArgs);
template <int TW, int NT>
static constexpr pp_kernel_t pp_kernel() {
    if constexpr (TW <= PP_TILES[NT]) return plane_product_kernel<TW, NT>;
    else return nullptr;
}

// Rows of all pieces, or, where their sums do not fit the workspace (plane_product_workspace_least: up to SQ_SMALL_BMAX activation rows), as many at a time as do, evenly
// cut.  A row's sums depend on the planes a workgroup takes alone, which are those of the whole product: the results are the same bits either way.
int launch_plane_product(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws, size_t ws_bytes,
                         hipStream_t s, const PlanePlan* planned) {
    const PlanePlan whole = planned ? *planned : pp_plan(mats, n, T);
    const size_t fixed = pp_fixed_bytes(mats, n, whole.nt);
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += mats[i].R;
    int64_t most = rows;                     // weight rows of a launch
    if (plane_product_workspace(mats, n, T, &whole) > ws_bytes) {
        const size_t none = fixed + pp_sums_bytes(0, n, T, whole.pl);
        const int64_t fit = ws_bytes > none ? (int64_t)((ws_bytes - none) / ((size_t)(8 / whole.pl) * T * 4)) / 16 * 16 : 0;
        if (fit < 16) return fail(SQ_EWORKSPACE, "plane product: workspace %zu < %zu", ws_bytes, plane_product_workspace(mats, n, T));
        const int64_t launches = (rows + fit - 1) / fit;
        most = std::min(fit, ((rows + launches - 1) / launches + 15) / 16 * 16);
    }
    PpOrderArgs o{};
    o.planes = (uint16_t*)ws; o.x = (const uint16_t*)x; o.ldx = ldx; o.pieces = n; o.T = T; o.NT = whole.nt; o.n = mats[0].C / 8; o.pairs = (o.n + 63) / 64;
    o.bf = x_dtype == SQ_BF16;
    o.xf = (unsigned char*)ws + planes_bytes(n);
    for (int i = 0; i < n; ++i) o.table[i] = mats[i].table;
    const int64_t units = (int64_t)n * (PLANE / 8) + (int64_t)whole.nt * 16 * o.pairs * 8;
    hipLaunchKernelGGL(pp_order_kernel, dim3((unsigned)((units + 63) / 64)), dim3(64), 0, s, o);
    if (const int rc = check_launch("plane order")) return rc;
#define SQ_NT(NT) {pp_kernel<1, NT>(), pp_kernel<2, NT>(), pp_kernel<3, NT>(), pp_kernel<4, NT>(), pp_kernel<5, NT>()}
    static constexpr pp_kernel_t kernels[PP_MAX_NT - 1][5] = {SQ_NT(2), SQ_NT(3), SQ_NT(4), SQ_NT(5), SQ_NT(6), SQ_NT(7), SQ_NT(8)};
#undef SQ_NT
    static const bool raised = [] {
        for (const auto& nt : kernels)
            for (pp_kernel_t k : nt)
                if (k) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, PLANE * 2);
        (void)hipGetLastError();
        return true;
    }();
    (void)raised;
    for (int i = 0, r0 = 0; i < n;) {
        sq_matrix part[MID_PIECES];
        PpArgs a{};
        a.xf = o.xf; a.T = T; a.chunks = o.n; a.pairs = o.pairs; a.pl = whole.pl;
        for (int64_t left = most; i < n && left > 0;) {
            const int R = (int)std::min<int64_t>(mats[i].R - r0, left);
            sq_matrix& m = part[a.n] = mats[i];
            m.R = R; m.tags += (int64_t)r0 * m.W; m.row_scale += r0; m.y_off += r0;
            a.p[a.n++].planes = o.planes + (int64_t)i * 8 * PLANE;
            left -= R;
            r0 += R;
            if (r0 >= mats[i].R) ++i, r0 = 0;
        }
        const PlanePlan p = most == rows ? whole : pp_plan(part, a.n, T, whole.pl);
        char* sums = (char*)ws + fixed;
        for (int j = 0; j < a.n; ++j) {
            a.p[j].m = part[j]; a.p[j].part = (float*)sums; a.p[j].job0 = a.jobs; a.p[j].parts = p.parts[j];
            sums += pp_part_bytes(part[j].R, T, p.pl);
            a.jobs += p.parts[j];
        }
        hipLaunchKernelGGL(kernels[p.nt - 2][p.tw - 1], dim3((unsigned)((a.jobs + 7) / 8 * 8 * (8 / p.pl))), dim3(64 * PP_WAVES), PLANE * 2, s, a);
        if (const int rc = check_launch("plane product")) return rc;
        if (const int rc = launch_slice_sum(a.p, a.n, 8 / p.pl, T, y, y_dtype, ldy, s, /*whole_quads=*/true)) return rc;
    }
    return SQ_OK;
}

}  // namespace sq

// For tests: the kernel whatever its estimate says; workspace: what it needs, or with ws the call.  Negative: pieces or rows that it does not take.
extern "C" __attribute__((visibility("default"))) int64_t sq_plane_product_for_tests(const sq_matrix* mats, int32_t n, const void* x, int32_t x_dtype, int64_t ldx, void* y,
                                                                                     int32_t y_dtype, int64_t ldy, int32_t T, void* ws, void* stream) {
    if (n < 1 || sq::pp_fit(mats, n, T) != n) return SQ_EUNSUPPORTED;
    if (!ws) return (int64_t)sq::plane_product_workspace(mats, n, T);
    return sq::launch_plane_product(mats, n, x, x_dtype, ldx, y, y_dtype, ldy, T, ws, sq::plane_product_workspace(mats, n, T), (hipStream_t)stream);
}
