// Codebook product for up to 16 activation rows, d = 8 with 16-bit tags, where no tag streams serve them: a codebook of 65,536
// codewords, 1 MB, eight times what LDS holds beside its activations.
//
// What gathers codewords from L2 is bound by its requests, one per tag, 64 bytes moved for the 16 that are used, 150 to 180 G a second
// however few activation rows there are; the tag streams, which gather from LDS, multiply on the vector ALU, row by row.  Here a
// workgroup holds one slice of the codebook, 8192 codewords, and walks ALL tags of its rows: a tag of its slice gathers its
// codeword from LDS, any other one a codeword of zeros, and v_mfma_f32_16x16x32_f16 multiplies them alike.  Every tag is looked at by
// eight workgroups, whose fp32 sums slice_sum_kernel adds up.
//
// Bound: what LDS returns, 1 KB per 64 tags and slice (12 clocks a read with its share of the tags' way from L2, 8 at best; seven lanes
// of eight read the one zero codeword, so bank conflicts are few), matrix cores and vector ALU a third of the time each (counters of 2 x 18944 x 3584
// at 16 rows: 13 clocks of a CU per gather from the launch's first to its last, LDS busy 45 % of them, 7 with conflicts, matrix cores 31 %, vector
// ALU 38 %).  Microseconds
// at 9 / 16 rows with the gathers from L2 and here: 2 x 18944 x 3584 82 / 83, now 55 / 58; 3584 x 18944 50 / 50, 36 / 36; 28672 x 4096 75 / 75, 47 / 50;
// 14336 x 4096 40 / 40, 29 / 31; 5120 x 5120 28 / 28, 21 / 23; a 7B layer of 16 rows 191, now 147, of 8 157, now 143.  From 17 rows the second
// tile's products fill the matrix cores, which multiply eight times as much as they must (2 x 18944 x 3584 at 32 rows 90 us either way).
//
//   workgroup   16 waves, four per SIMD (eight with twice the tiles: 15 % slower), each with TW tiles of 16 weight rows x 16 activation
//               rows; slice s of the codebook
//   grid        jobs (blocks of 256 TW rows x ks slices of K) x 8 codebook slices; the eight of a job on one XCD (workgroups go to the
//               XCDs in turn), whose L2 then reads the job's tags once
//   K           in rounds of 4 units of 64 columns (8 tags, 16 bytes); step j of lane group g is columns (4 round + g) 64 + 8 j ..
//               + 7, so a lane's operand of a step is one codeword; rounds in pairs, the second one past the end multiplies zeros
//   X           a round's 16 rows x 32 pieces of 16 bytes, double buffered in LDS, loaded to registers two rounds ahead
//   tags        two rounds ahead; codewords PF products ahead, in a ring of RING
//
// Zero codewords times activations that are not finite would be NaN where the product is infinite: a workgroup that has staged such an
// activation multiplies its share again, tag by tag on the vector ALU, without the zeros.
#include <algorithm>
#include <type_traits>
#include "sq_slices.h"

namespace sq {

constexpr int SIEVE_MAX_T = 16, SIEVE_TW = 5;
constexpr int SIEVE_CODEWORDS = 8192, SIEVE_SLICES = 8, SIEVE_TAB = SIEVE_CODEWORDS * 16, SIEVE_ODD = SIEVE_TAB + 16, SIEVE_X = SIEVE_TAB + 32, SIEVE_WAVES = 16, SIEVE_ROWS = 16 * SIEVE_WAVES;     // (weight rows per TW)
typedef __attribute__((address_space(3))) void* sieve_lptr_t;
typedef const __attribute__((address_space(3))) u32x4 sieve_lds_u32x4;
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

struct SievePiece {
    sq_matrix m;
    float* part;                 // fp32 [8 ks, T, R]
    int job0;                    // first job
};
struct SieveArgs {
    SievePiece p[MID_PIECES];
    const uint16_t* x;
    int64_t ldx;
    int n, T, U, ks, jobs, bf;   // U: units of a row
};

// An X row of a stage (a round) is 32 pieces of 16 bytes, lane group by lane group; piece c of row t sits at slot c ^ this.  The 16 lanes of
// an LDS clock are rows 0-3 and 12-15 of one lane group with rows 4-11 of the next; they fall into 16 different groups of four banks.
__device__ __forceinline__ int sieve_swizzle(int t) { return (t & 3) | ((t >> 3) & 1) << 2; }
constexpr int SIEVE_STAGE = 16 * 512;

// s_waitcnt immediate that waits until at most n vector-memory operations are outstanding (gfx9 encoding: vmcnt in bits 3:0 and 15:14)
constexpr int sieve_vmcnt_only(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }

template <int TW>
__global__ __launch_bounds__(64 * SIEVE_WAVES) void sieve_kernel(SieveArgs a) {
    constexpr int NTH = 64 * SIEVE_WAVES;
    constexpr int RING = 4, PF = 3;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if ((uint32_t)(uintptr_t)(sieve_lptr_t)smem != 0u) return;               // (gathers count from LDS address 0)
    const int job = (int)(blockIdx.x >> 6) * 8 + (int)(blockIdx.x & 7), cs = (int)(blockIdx.x >> 3) & 7;
    if (job >= a.jobs) return;
    int pi = 0;
    while (pi + 1 < a.n && job >= a.p[pi + 1].job0) ++pi;
    const SievePiece& P = a.p[pi];
    const sq_matrix& m = P.m;
    const int slice = (job - P.job0) % a.ks, blk = (job - P.job0) / a.ks;
    const int NR = (a.U + 3) / 4, NP = (NR + 1) >> 1;
    const int r0 = 2 * (int)((unsigned)NP * (unsigned)slice / (unsigned)a.ks), r1 = min(NR, 2 * (int)((unsigned)NP * (unsigned)(slice + 1) / (unsigned)a.ks));
    unsigned char* xbuf = smem + SIEVE_X;

    // ---- the codebook slice and the zero codeword behind it
    const __amdgpu_buffer_rsrc_t table = __builtin_amdgcn_make_buffer_rsrc((void*)(reinterpret_cast<const unsigned char*>(m.table) + (size_t)cs * SIEVE_TAB), 0, SIEVE_TAB, 0x00027000);
#pragma unroll
    for (int k = 0; k < SIEVE_TAB / (NTH * 16); ++k)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(table, (sieve_lptr_t)(smem + (k * NTH + wave * 64) * 16), 16, tid * 16, k * NTH * 16, 0, 0);
    if (tid < 8) reinterpret_cast<uint32_t*>(smem + SIEVE_TAB)[tid] = 0u;       // (and the flag behind it)
    __builtin_amdgcn_sched_barrier(0);       // (the wait for the slice counts the loads behind it)

    // ---- this wave's tiles (tiles past the last row repeat the last one and are not stored; waves without a tile only stage)
    const int ntiles = (m.R + 15) >> 4, tile0 = (blk * SIEVE_WAVES + wave) * TW;
    const bool work = tile0 < ntiles;
    uint32_t to[TW];
#pragma unroll
    for (int i = 0; i < TW; ++i) to[i] = (uint32_t)min(min(tile0 + i, ntiles - 1) * 16 + li, m.R - 1) * (uint32_t)m.W * 4u;
    const char* tags = reinterpret_cast<const char*>(m.tags);
    auto load_tags = [&](int round, u32x4* t) {
        const uint32_t u = (uint32_t)min(4 * round + lg, a.U - 1) * 16u;
#pragma unroll
        for (int i = 0; i < TW; ++i) t[i] = *reinterpret_cast<const u32x4*>(tags + (to[i] + u));
    };
    // tags of this slice as their places in it, all others (and those of units past the row's end, whose activations are zeros, and
    // whose codewords may not be finite) as that of the zero codeword
    const uint16_t first = (uint16_t)(cs * SIEVE_CODEWORDS);
    auto place_tags = [&](int round, u32x4* t) {
        const bool past = 4 * round + lg >= a.U;
#pragma unroll
        for (int i = 0; i < TW; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t w = t[i][k];      // (by itself: the bit cast of a vector's element is that of its first one)
                const u16x2 d = __builtin_elementwise_min(__builtin_bit_cast(u16x2, w) - u16x2{first, first}, u16x2{SIEVE_CODEWORDS, SIEVE_CODEWORDS});
                t[i][k] = past ? (uint32_t)(SIEVE_CODEWORDS | SIEVE_CODEWORDS << 16) : __builtin_bit_cast(uint32_t, d);
            }
    };
    auto gather = [&](uint32_t w, int half) {
        const uint32_t at = (half ? w >> 12 : w << 4) & 0xFFFF0u;
        return __builtin_bit_cast(half8v, *(sieve_lds_u32x4*)(uintptr_t)at);
    };

    // ---- activations: thread tid < 512 stages piece tid % 32 = lane group * 8 + step of row tid / 32
    const int xt = (tid >> 5) & 15, xg = (tid >> 3) & 3;
    const char* xrow = reinterpret_cast<const char*>(a.x + (int64_t)min(xt, a.T - 1) * a.ldx) + (tid & 7) * 16;
    const uint32_t xl = (uint32_t)(xt * 512 + (((tid & 31) ^ sieve_swizzle(xt)) << 4));
    // (columns past the row's end are zeros; what is read in their place is the row's last unit)
    auto load_x = [&](int round) { return *reinterpret_cast<const u32x4*>(xrow + (int64_t)min(4 * round + xg, a.U - 1) * 128); };
    uint32_t odd = 0;                        // not zero: this thread has staged an activation that is not finite
    auto store_x = [&](u32x4 v, int buf, int round) {
        if (tid >= 512) return;
        if (a.bf) { v.x = bf2h_x2(v.x); v.y = bf2h_x2(v.y); v.z = bf2h_x2(v.z); v.w = bf2h_x2(v.w); }
        const uint32_t keep = round < r1 && 4 * round + xg < a.U ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            v[e] &= keep;
            // exponents of all ones carry into the sign's place, which the mask has cleared
            odd |= ((v[e] & 0x7FFF7FFFu) + 0x04000400u) & 0x80008000u;
        }
        *reinterpret_cast<u32x4*>(xbuf + buf * SIEVE_STAGE + xl) = v;
    };
    const uint32_t xbase = (uint32_t)(li * 512 + (((lg * 8) ^ sieve_swizzle(li)) << 4));

    float4v acc[TW];
#pragma unroll
    for (int i = 0; i < TW; ++i) acc[i] = float4v{0.f, 0.f, 0.f, 0.f};

    u32x4 tag[2][TW], px[2];
    half8v wf[RING];
    load_tags(r0, tag[0]);
    px[0] = load_x(r0);
    load_tags(r0 + 1, tag[1]);
    px[1] = load_x(r0 + 1);
    store_x(px[0], 0, r0);
    place_tags(r0, tag[0]);
    // every wave gathers what others have copied, and no barrier waits for copies: this wave's part of the slice has landed once no more
    // operations are on their way than it has issued behind it for the second round, TW of tags and one of activations
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(sieve_vmcnt_only(TW + 1));
    __syncthreads();
    if (work) {
#pragma unroll
        for (int q = 0; q < PF; ++q) wf[q] = gather(tag[0][q % TW][q / TW >> 1], q / TW & 1);
    }
    auto do_round = [&](auto parity, int round) {
        constexpr int Q = decltype(parity)::value;
        const unsigned char* xs = xbuf + Q * SIEVE_STAGE;
        auto read_x = [&](int j) { return *reinterpret_cast<const half8v*>(xs + (xbase ^ (uint32_t)(j << 4))); };
        px[Q] = load_x(round + 2);
        half8v xf[2];
        if (work) xf[0] = read_x(0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            if (j == 4) store_x(px[Q ^ 1], Q ^ 1, round + 1);
            if (j == (8 * TW - PF) / TW) place_tags(round + 1, tag[Q ^ 1]);  // (the step whose gathers go over into that round)
            if (!work) continue;
            if (j < 7) xf[(j + 1) & 1] = read_x(j + 1);
#pragma unroll
            for (int i = 0; i < TW; ++i) {
                const int q = j * TW + i, z = q + PF, zj = z / TW;
                __builtin_amdgcn_sched_barrier(0);
                if (z < 8 * TW) wf[z % RING] = gather(tag[Q][z % TW][zj >> 1], zj & 1);
                else wf[z % RING] = gather(tag[Q ^ 1][z % TW][(zj - 8) >> 1], zj & 1);
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[q % RING], xf[j & 1], acc[i], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        load_tags(round + 2, tag[Q]);                                        // (this round's have all been used)
        __syncthreads();
    };
    for (int round = r0; round < r1; round += 2) {                           // (a partner past the slice's end multiplies zeros)
        do_round(std::integral_constant<int, 0>{}, round);
        do_round(std::integral_constant<int, 1>{}, round + 1);
    }

    float* part = P.part + (int64_t)(cs * a.ks + slice) * a.T * m.R;
    volatile uint32_t* flag = reinterpret_cast<volatile uint32_t*>(smem + SIEVE_ODD);
    if (odd) *flag = 1u;
    __syncthreads();
    if (*flag) {
        // a thread per weight row: all its tags of the slice, an activation row at a time
        for (int r = blk * (SIEVE_ROWS * TW) + tid; r < min(m.R, (blk + 1) * (SIEVE_ROWS * TW)); r += NTH)
            for (int t = 0; t < a.T; ++t) {
                float sum = 0.f;
                const uint16_t *row = reinterpret_cast<const uint16_t*>(tags + (size_t)r * m.W * 4), *x = a.x + (int64_t)t * a.ldx;
#pragma unroll 1
                for (int c = 32 * r0; c < min(32 * r1, 8 * a.U); ++c) {
                    const int at = (int)row[c] - cs * SIEVE_CODEWORDS;
                    if (at < 0 || at >= SIEVE_CODEWORDS) continue;
                    const uint16_t* w = reinterpret_cast<const uint16_t*>(smem + at * 16);
#pragma unroll 1
                    for (int e = 0; e < 8; ++e) sum = __builtin_fmaf(h2f(w[e]), a.bf ? (float)bf2h(x[c * 8 + e]) : h2f(x[c * 8 + e]), sum);
                }
                part[(int64_t)t * m.R + r] = sum;
            }
        return;
    }
    if (!work) return;
    // ---- lane: activation row li, weight rows 16 tile + 4 lg .. + 3
    if (li >= a.T) return;
    const bool vec = m.R % 4 == 0;
#pragma unroll
    for (int i = 0; i < TW; ++i) {
        const int r = (tile0 + i) * 16 + lg * 4;
        if (r >= m.R) continue;
        float* o = part + (int64_t)li * m.R + r;
        if (vec) {
            *reinterpret_cast<float4v*>(o) = acc[i];
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) if (r + e < m.R) o[e] = acc[i][e];
        }
    }
}

// ------------------------------------------------------------------------------------------ host

static bool sieve_shape(const sq_matrix& m) {
    return m.R > 0 && m.tags && m.d == 8 && m.bits == 16 && m.G == 1 && !m.row_book && !m.perms && m.C % 64 == 0 && m.W == m.C / 16 &&
           (((uintptr_t)m.tags | (uintptr_t)m.table) & 15) == 0 && (int64_t)m.R * m.W < ((int64_t)1 << 30);
}

struct SievePlan { int tw, ks; double us; };

static int sieve_jobs(const sq_matrix* mats, int n, int tw) {
    int jobs = 0;
    for (int i = 0; i < n; ++i) jobs += (mats[i].R + SIEVE_ROWS * tw - 1) / (SIEVE_ROWS * tw);
    return jobs;
}

// The plan of least estimated time, in microseconds: rounds of workgroups over the CUs, each the slice's way to LDS and its steps, and
// the partial sums, written and read back.  Fitted to 25 plans of the products above (within 10 %); the best of them fill the
// chip once with the fewest K slices.  (slices: the number of K slices, if it is given)
static SievePlan sieve_plan(const sq_matrix* mats, int n, int T, int cus, int slices = 0) {
    const int NP = ((mats[0].C / 64 + 3) / 4 + 1) / 2;                       // pairs of rounds
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += mats[i].R;
    SievePlan best{2, 1, 1e30};
    for (int tw = 2; tw <= SIEVE_TW; ++tw)                                   // (one tile a wave: next to never the best of what pays)
        for (int ks = slices ? slices : 1; ks <= (slices ? slices : std::min(NP, 8)); ++ks) {
            const int64_t jobs = (int64_t)sieve_jobs(mats, n, tw) * ks, rounds = (jobs * SIEVE_SLICES + cus - 1) / cus;
            const int steps = (NP + ks - 1) / ks * 16;
            const double us = 3.2 + rounds * (4.4 + steps * (0.02 + 0.07 * tw)) + 32.0 * ks * T * rows / 2.74e6;
            if (us < best.us) best = {tw, ks, us};
        }
    return best;
}

static size_t sieve_part_bytes(int R, int T, int ks) { return ((size_t)SIEVE_SLICES * ks * T * R * 4 + 255) & ~(size_t)255; }

size_t sieve_workspace(const sq_matrix* mats, int n, int T) {
    const SievePlan pl = sieve_plan(mats, n, T, device_cus());
    size_t need = 0;
    for (int i = 0; i < n; ++i) need += sieve_part_bytes(mats[i].R, T, pl.ks);
    return need;
}
size_t sieve_workspace_least(const sq_matrix* mats, int n, int T) { return std::min(sieve_workspace(mats, n, T), SMALL_ROOM); }

// How many of the n pieces, the first one on, the kernel takes in one launch, 0 where the gathers from L2 are the faster way: they
// take 4.6 us per million tags and 4 more, 1.1 to 1.3 times that for rows of more than 8192 columns (4096 x 4096 at 9 / 16 rows 15.5 /
// 15.6 us, here 17 / 19; 8192 x 4096 23.5 / 23.8, 21 / 21).
int sieve_group(const sq_matrix* mats, int n, int T) {
    if (T < 1 || T > SIEVE_MAX_T) return 0;
    int k = 0;
    double tags = 0.0;
    for (; k < n && k < MID_PIECES && sieve_shape(mats[k]) && mats[k].C == mats[0].C; ++k) tags += (double)mats[k].R * mats[k].C / 8e6;
    return k && sieve_plan(mats, k, T, device_cus()).us < 0.92 * (4.0 + 4.6 * tags) ? k : 0;
}

// Rows of all pieces, or, where their partial sums do not fit the workspace, as many at a time as do, evenly cut (2 x 18944 x 3584 at 16
// rows in two launches 75 us, in one 58, through the gathers from L2 85; 60001 x 4160, which fills the chip anyway, level).  A row's sums depend on the K slices alone, which are those of the whole product: the results are the
// same bits either way.
int launch_sieve(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws, size_t ws_bytes, hipStream_t s) {
    typedef void (*kernel_t)(SieveArgs);
    static constexpr kernel_t kernels[SIEVE_TW - 1] = {sieve_kernel<2>, sieve_kernel<3>, sieve_kernel<4>, sieve_kernel<5>};
    static const bool raised = [] {
        for (kernel_t k : kernels) (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipGetLastError();
        return true;
    }();
    (void)raised;
    const SievePlan whole = sieve_plan(mats, n, T, device_cus());
    int64_t rows = 0;
    for (int i = 0; i < n; ++i) rows += mats[i].R;
    int64_t most = rows;                     // rows of a launch
    if (sieve_workspace(mats, n, T) > ws_bytes) {
        const int64_t fit = (int64_t)((ws_bytes - std::min(ws_bytes, (size_t)256 * n)) / ((size_t)SIEVE_SLICES * whole.ks * T * 4)) / 16 * 16;
        const int64_t launches = (rows + fit - 1) / fit;
        most = std::min(fit, ((rows + launches - 1) / launches + 15) / 16 * 16);
    }
    for (int i = 0, r0 = 0; i < n;) {
        sq_matrix part[MID_PIECES];
        int k = 0;
        for (int64_t left = most; i < n && left > 0;) {
            const int R = (int)std::min<int64_t>(mats[i].R - r0, left);
            sq_matrix& m = part[k++] = mats[i];
            m.R = R; m.tags += (int64_t)r0 * m.W; m.row_scale += r0; m.y_off += r0;
            left -= R;
            r0 += R;
            if (r0 >= mats[i].R) ++i, r0 = 0;
        }
        const SievePlan pl = most == rows ? whole : sieve_plan(part, k, T, device_cus(), whole.ks);
        SieveArgs a{};
        a.x = (const uint16_t*)x; a.ldx = ldx; a.n = k; a.T = T; a.U = mats[0].C / 64; a.ks = pl.ks; a.bf = x_dtype == SQ_BF16;
        char* sums = (char*)ws;
        for (int j = 0; j < k; ++j) {
            a.p[j] = {part[j], (float*)sums, a.jobs};
            sums += sieve_part_bytes(part[j].R, T, pl.ks);
            a.jobs += (part[j].R + SIEVE_ROWS * pl.tw - 1) / (SIEVE_ROWS * pl.tw) * pl.ks;
        }
        hipLaunchKernelGGL(kernels[pl.tw - 2], dim3((unsigned)((a.jobs + 7) / 8 * 64)), dim3(64 * SIEVE_WAVES), (size_t)SIEVE_X + 2 * SIEVE_STAGE, s, a);
        if (const int rc = check_launch("sq_linear_small(sieve)")) return rc;
        if (const int rc = launch_slice_sum(a.p, k, SIEVE_SLICES * pl.ks, T, y, y_dtype, ldy, s)) return rc;
    }
    return SQ_OK;
}

}  // namespace sq
