// Host side of the product of sq_fused.h: which stacks take it, how the work is cut, and the activations in fragment order.
#include <algorithm>
#include "sq_fused.h"
#include "sq_slices.h"

namespace sq {

int launch_fused_b16d8(const FusedArgs&, int, int, int, hipStream_t);
int launch_fused_b12d4(const FusedArgs&, int, int, int, hipStream_t);
int launch_fused_b10d4(const FusedArgs&, int, int, int, hipStream_t);
int launch_fused_b8d4(const FusedArgs&, int, int, int, hipStream_t);

// The activations as the kernel's matrix instructions take them: 1 KB blocks of 16 tokens x 32 columns in fp16, block
// [token block][step][tile of 16 tokens], in it lane l's 16 bytes: token l % 16, columns (4 round + l / 16) UK + 8 j .. + 7 of step
// j of a round.  Zeros past the last token and column.  A workgroup turns 16 tokens x one round (4 UK columns, read in whole
// lines) round in LDS, whose blocks lie 1040 bytes apart so that neighbouring steps' pieces fall on different banks.
template <int SPR>
__global__ __launch_bounds__(256) void fused_x_kernel(const uint16_t* __restrict__ x, int64_t ldx, int x_dtype, int T, int C, int NT, int k32,
                                                      unsigned char* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) unsigned char turn[SPR * 1040];
    constexpr int PCS = 4 * SPR;                                          // 16-byte pieces of a token
    const int round = (int)blockIdx.x, tile = (int)blockIdx.y, tb = tile / NT, n = tile - tb * NT;
    for (int i = threadIdx.x; i < 16 * PCS; i += 256) {
        const int tl = i / PCS, c = i - tl * PCS, t = tile * 16 + tl, col = (round * PCS + c) * 8;
        u32x4 v = u32x4{0u, 0u, 0u, 0u};
        if (t < T && col < C) {
            v = *reinterpret_cast<const u32x4*>(x + (int64_t)t * ldx + col);
            if (x_dtype == SQ_BF16) { v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w); }
        }
        *reinterpret_cast<u32x4*>(turn + (c % SPR) * 1040 + ((c / SPR) * 16 + tl) * 16) = v;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * PCS; i += 256) {
        const int j = i >> 6, l = i & 63;
        *reinterpret_cast<u32x4*>(out + (((int64_t)tb * k32 + round * SPR + j) * NT + n) * 1024 + l * 16) = *reinterpret_cast<const u32x4*>(turn + j * 1040 + l * 16);
    }
}

static int fused_unit_dwords(int bits) { return bits == 12 ? 3 : bits == 10 ? 5 : 4; }
static int fused_round_steps(const sq_matrix& m) { return fused_unit_dwords(m.bits) * 32 / m.bits / (8 / m.d); }
static int fused_rounds(const sq_matrix& m) { return (m.W / fused_unit_dwords(m.bits) + 3) / 4; }

// How a product is cut, nw = 0 where the others were the faster ones when this kernel was cut (which products with a cut run here: gemm_route, sq_gemm.hip).  Up to 768 rows, in blocks of up to 384 tokens; rows of
// the weights in tiles of 32 tw, where a launch should fill the CUs once: what a workgroup takes hardly depends on how many run
// beside it.  A tile of 64 / 96 / 128 / 160 rows x 333 tokens x 3584 columns takes 66 / 83 / 104 / 123 us with 16-bit tags of
// width 8 (the weights below), 62 / 73 / 85 / 103 with 10-bit ones of width 4.  Decoded and multiplied in tiles, or in one pass over the tags where
// that is the faster one (sq_mid.h), against here, us (d = 8, then d = 4):
//   rows x columns    200 tokens                333                       512                       768
//   12000 x 3584      75 / 57    58 / 46        79 / 66    71 / 62        79 / 77    69 / 60        92 / 89    84 / 80
//   18944 x 3584      95 / 72    72 / 55        97 / 83   113 / 72       112 / 111   98 / 83       133 / 127  121 / 109
//   25000 x 3584     105 / 83    75 / 63       126 / 96  115 / 81       143 / 186  124 / 149     210 / 225  180 / 192
//   37888 x 3584     177 / 106  104 / 79       234 / 130  154 / 102      263 / 216  209 / 164      301 / 246  245 / 206
//   3584 x 18944      96 / 72    67 / 59       132 / 90   109 / 77       143 / 137  136 / 102      173 / 162  152 / 136
// so two blocks of tokens need the last round of workgroups nearly full; a second round is for the widest tiles, where the other way
// is longer than two of them (d = 8 from 193 tokens, d = 4 from 257); and rows of 8192 columns and more are cut into K slices of
// 2048 at least where there are too few tiles (in shorter rows the slices' sums cost what they gain: 4608 x 3584 at 333 tokens 51 us
// in three, 53 there).  At 1000 tokens 191 / 225 for 18944 rows, 371 / 353 for 37888.
static FusedPlan fused_cut(const sq_matrix* mats, int n, int T, int cus) {
    const FusedPlan none{0, 0, 1, 1, 0};
    if (T < 129 || T > 768) return none;
    const int tbs = T <= 384 ? 1 : 2, per = (T + tbs - 1) / tbs, nw = per <= 192 ? 3 : per <= 256 ? 4 : 6;
    const int table = mats[0].d == 4 ? (mats[0].G << mats[0].bits) * 8 : 0, weight[6] = {0, 0, 17, 21, 27, 32};
    auto fits = [&](int tw) { return fused_lds(mats[0].bits, table, nw, tw, fused_steps(nw), fused_slots(mats[0].d, nw)) <= 160 * 1024; };
    auto tiles = [&](int tw) {
        int64_t b = 0;
        for (int i = 0; i < n; ++i) b += (mats[i].R + 32 * tw - 1) / (32 * tw);
        return b * tbs;
    };
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += mats[i].R;
    int tw = 0;
    int64_t rounds = 0;
    for (int w = 2; w <= 5; ++w) {
        const int64_t r = (tiles(w) + cus - 1) / cus;
        if (fits(w) && (!tw || r * weight[w] < rounds * weight[tw])) tw = w, rounds = r;
    }
    if (!tw) return none;
    const int64_t used = rows * tbs * 100, room = rounds * cus * 32 * tw;     // percent of the weight rows that the rounds have room for
    const bool whole = tbs == 1 ? used >= 66 * room : used >= 85 * room && tw >= 3;
    if (whole && (rounds == 1 || (tw == 5 && (tbs == 2 || nw == 6 || (nw == 4 && mats[0].d == 8))))) return {nw, tw, 1, tbs, T};
    if (mats[0].d == 8 && nw == 4 && tbs == 1 && tiles(1) <= cus && used >= 70 * cus * 32) return {nw, 1, 1, tbs, T};   // (6000 x 3584 at 200 tokens: 43 us, 49 there)
    const int64_t t3 = tiles(3);
    const int ks = (int)std::min<int64_t>({8, cus / t3, mats[0].C / 2048});
    if (fits(3) && mats[0].C >= 8192 && ks > 1 && t3 * ks * 4 >= cus * 3) return {nw, 3, ks, tbs, T};
    return none;
}

static int64_t fused_workgroups(const FusedPlan& p, const sq_matrix* mats, int n) {
    int64_t w = 0;
    for (int i = 0; i < n; ++i) w += (mats[i].R + 32 * p.tw - 1) / (32 * p.tw);
    return w * p.ks * p.tbs;
}

bool fused_two_blocks(const FusedPlan& p, const sq_matrix* mats, int n) { return p.tbs == 2 && fused_workgroups(p, mats, n) <= device_cus(); }

// What a product takes in such a cut, in microseconds.  d = 4: a launch of the activations and one of the product, 20 between rounds of workgroups; fitted to
// 76 of 1700 to 54000 rows at 130 to 768 tokens (9 %).  d = 8, two blocks of tokens in one round (fused_two_blocks): fitted to 226 of 1500 to 23000 rows of 192 to 14000
// columns (7 %; the more workgroups, the longer L2 takes for each one's codewords), with the sums of K slices per million.
float fused_us(const FusedPlan& p, const sq_matrix* mats, int n) {
    const int cus = device_cus();
    const int64_t w = fused_workgroups(p, mats, n), rounds = (w + cus - 1) / cus;
    const float columns = mats[0].C * 1e-3f / p.ks;
    if (mats[0].d == 4) return -4.5f + rounds * (19.6f + columns * (0.163f * p.tw + 0.809f * p.nw * p.tw + 0.707f * p.nw - 0.217f));
    float sums = 0.f;
    for (int i = 0; i < n && p.ks > 1; ++i) sums += (float)mats[i].R * p.t * p.ks * 1e-6f;
    return 19.7f + columns * (5.89f * p.tw + 2.22f * p.nw + 6.63f * w / cus - 16.1f) + 4.19f * sums;
}

static size_t fused_x_bytes(const sq_matrix* mats, const FusedPlan& p) {
    return (size_t)p.tbs * fused_rounds(mats[0]) * fused_round_steps(mats[0]) * FUSED_TN * p.nw * 1024;
}
static size_t fused_part_bytes(const sq_matrix& m, int T, int ks) { return ks > 1 ? (((size_t)ks * T * m.R * 4) + 255) & ~(size_t)255 : 0; }

FusedPlan fused_plan(const sq_matrix* mats, int n, int T) {
    const FusedPlan none{0, 0, 1, 1, 0};
    if (n < 1 || n > MID_PIECES) return none;
    for (int i = 0; i < n; ++i) {
        const sq_matrix &m = mats[i], &m0 = mats[0];
        if (!mma_shape(m) || m.R <= 0 || m.d != m0.d || m.bits != m0.bits || m.W != m0.W || m.G != m0.G) return none;
        if (((int64_t)m.R + 16) * m.W * 4 >= ((int64_t)1 << 32)) return none;                  // 32-bit offsets
        if (m.d == 8 && ((int64_t)m.G << m.bits) * 16 > ((int64_t)1 << 31)) return none;
        if (m.d == 4 && ((int64_t)m.G << m.bits) * 8 > 128 * 1024) return none;
    }
    return fused_cut(mats, n, T, device_cus());
}

// For tests: the variant that a stack takes at T rows, as token tiles | weight tiles << 8 | K slices << 16 | token blocks << 24; 0: another kernel.
extern "C" __attribute__((visibility("default"))) int32_t sq_fused_variant_for_tests(const sq_matrix* mats, int32_t n, int32_t T) {
    const GemmRoute r = gemm_route(mats, n, T, SQ_BF16);
    if (r.kernel != GEMM_FUSED) return 0;
    const FusedPlan& p = r.fused;
    return p.nw | p.tw << 8 | p.ks << 16 | p.tbs << 24;
}

size_t fused_workspace(const FusedPlan& p, const sq_matrix* mats, int n, int T) {
    size_t need = fused_x_bytes(mats, p);
    for (int i = 0; i < n; ++i) need += fused_part_bytes(mats[i], T, p.ks);
    return need;
}

int launch_fused(const FusedPlan& p, const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws, hipStream_t s) {
    const sq_matrix& m0 = mats[0];
    FusedArgs a{};
    a.n = n; a.y = y; a.ldy = ldy; a.T = T; a.y_dtype = y_dtype; a.ks = p.ks;
    a.U = m0.W / fused_unit_dwords(m0.bits);
    a.table_bytes = m0.d == 4 ? (m0.G << m0.bits) * 8 : 0;
    const int rounds = fused_rounds(m0), spr = fused_round_steps(m0), NT = FUSED_TN * p.nw;
    a.k32 = rounds * spr;
    a.x = (const unsigned char*)ws;
    char* part = (char*)ws + fused_x_bytes(mats, p);
    for (int i = 0; i < n; ++i) {
        FusedPiece& P = a.p[i];
        const sq_matrix& m = mats[i];
        P.m = m;
        P.w = m.stream && tiled_format_ok(m.R, m.W, m.C, m.d, m.bits) && ((uintptr_t)m.stream & 15) == 0 ? (const void*)m.stream : nullptr;
        P.part = (float*)part;
        part += fused_part_bytes(m, T, p.ks);
        P.wg0 = a.per_tb;
        a.per_tb += (m.R + 32 * p.tw - 1) / (32 * p.tw) * p.ks;
    }
    const dim3 xgrid((unsigned)rounds, (unsigned)(p.tbs * NT));
    if (spr == 8) hipLaunchKernelGGL(fused_x_kernel<8>, xgrid, dim3(256), 0, s, (const uint16_t*)x, ldx, x_dtype, T, m0.C, NT, a.k32, (unsigned char*)ws);
    else hipLaunchKernelGGL(fused_x_kernel<4>, xgrid, dim3(256), 0, s, (const uint16_t*)x, ldx, x_dtype, T, m0.C, NT, a.k32, (unsigned char*)ws);
    int rc = check_launch("sq_linear_gemm(fused, activations)");
    if (rc) return rc;
    const int grid = a.per_tb * p.tbs;
    if (m0.d == 8) rc = launch_fused_b16d8(a, p.nw, p.tw, grid, s);
    else if (m0.bits == 12) rc = launch_fused_b12d4(a, p.nw, p.tw, grid, s);
    else if (m0.bits == 10) rc = launch_fused_b10d4(a, p.nw, p.tw, grid, s);
    else rc = launch_fused_b8d4(a, p.nw, p.tw, grid, s);
    if (rc || p.ks == 1) return rc;
    return launch_slice_sum(a.p, n, a.ks, T, y, y_dtype, ldy, s);
}

}  // namespace sq
