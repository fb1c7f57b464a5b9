// The packed file's two block-32 side formats on the device:
//   8-bit output head   q int8  [V, C],   scale fp16 [V, C/32]:  w[v, c] = q[v, c] * scale[v, c/32]
//   4-bit embedding     q uint8 [V, C/2], scale fp16 [V, C/32]:  w[v, 2k]   = ((q[v, k] & 15) - 8) * scale[v, 2k/32]
//                                                                w[v, 2k+1] = ((q[v, k] >> 4) - 8) * scale[v, (2k+1)/32]
// (reference shapequant/packed.py:30-40, 134-159).  The head product Y[b, v] = sum_c X[b, c] * w[v, c] is pure
// weight streaming for a handful of activation rows: every byte of q is read once from HBM and nothing is
// reused, so the kernel is built around full-line loads (one wave load = 1 KB of one weight row), many loads in
// flight per wave, and as few VALU operations per weight byte as the fp16 dot-product instruction allows.
#include <type_traits>
#include "sq_common.h"

namespace sq {

constexpr int Q8_WAVE_ROWS = 8;                 // weight rows a wave carries at once (loads in flight, x reuse)
constexpr int Q8_WG_WAVES = 4;
constexpr int Q8_TASK_ROWS = Q8_WAVE_ROWS * Q8_WG_WAVES;
constexpr int Q8_LDS_HALVES = 32768;            // fp16 activations a workgroup stages (64 KB)

struct Q8Args {
    const int8_t* q;
    const uint16_t* sc;
    const uint16_t* x;
    void* y;
    int64_t ldx, ldy;
    int V, C, B, x_dtype, y_dtype, tasks, x_vec;
};

// Four int8 -> two half2, exactly: flip the sign bit (q + 128 as a byte), put the byte under the exponent of
// 1024 (0x6400 | u = 1024 + u) and subtract 1152.
__device__ __forceinline__ void i8x4_to_h2(uint32_t w, half2v& lo, half2v& hi) {
    const uint32_t u = w ^ 0x80808080u;
    const half2v bias = {(half_t)1152.f, (half_t)1152.f};
    // v_perm_b32: selector bytes 0..3 pick from the second operand, 4..7 from the first
    lo = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) - bias;
    hi = __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) - bias;
}

// Sums N per-lane values over the 64 lanes with N - 1 + log2(64 / N) exchanges instead of 6 N: each halving step
// trades half of the values with the lane `o` away.  Afterwards lane l holds the total of value l >> (6 - log2 N)
// (in v[0]).
template <int N>
__device__ __forceinline__ void wave_sum_many(float (&v)[N], int lane) {
    int o = 32;
#pragma unroll
    for (int n = N; n > 1; n >>= 1, o >>= 1) {
        // bitwise select on a lane mask: a ?: on the array elements is turned into a select of the INDEX,
        // i.e. dynamic indexing of a register array
        const uint32_t up = (lane & o) ? 0xFFFFFFFFu : 0u;
#pragma unroll
        for (int i = 0; i < n / 2; ++i) {
            const uint32_t a = __builtin_bit_cast(uint32_t, v[i]), b = __builtin_bit_cast(uint32_t, v[i + n / 2]);
            const float give = __builtin_bit_cast(float, (a & up) | (b & ~up));
            const float keep = __builtin_bit_cast(float, (b & up) | (a & ~up));
            v[i] = keep + __shfl_xor(give, o, 64);
        }
    }
#pragma unroll
    for (; o > 0; o >>= 1) v[0] += __shfl_xor(v[0], o, 64);
}

template <int N> struct log2_of { static constexpr int value = 1 + log2_of<N / 2>::value; };
template <> struct log2_of<1> { static constexpr int value = 0; };

struct Q8Regs {
    u32x4 w[Q8_WAVE_ROWS];
    uint16_t s[Q8_WAVE_ROWS];
};

// One wave load per row: 16 bytes per lane at column step*1024 + lane*16 (clamped inside the row), and the
// scale of that lane's block.  Uniform row base + 32-bit lane offset keeps the addresses in few registers.
__device__ __forceinline__ void q8_load(Q8Regs& r, const Q8Args& a, int row0, int col) {
    const int nblk = a.C >> 5;
#pragma unroll
    for (int i = 0; i < Q8_WAVE_ROWS; ++i) {
        const int row = min(row0 + i, a.V - 1);
        const int8_t* base = a.q + (int64_t)row * a.C;
        r.w[i] = *reinterpret_cast<const u32x4*>(base + col);
        r.s[i] = a.sc[(int64_t)row * nblk + (col >> 5)];
    }
}

// Persistent workgroups of 4 waves; a task is 32 consecutive rows (8 per wave).  The NB activation rows sit in LDS
// as fp16 for the whole launch.  Each wave walks its rows' columns 1 KB at a time with the next step's loads
// (possibly the next task's first step) issued before the current step is multiplied.
template <int NB>
__global__ __launch_bounds__(256, 2) void q8_gemv_kernel(Q8Args a) {
    extern __shared__ __attribute__((aligned(16))) uint16_t xs[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int C = a.C;
    if (a.x_vec) {
        for (int i = tid * 8; i < NB * C; i += 256 * 8) {
            const int nb = i / C, c = i - nb * C;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (nb < a.B) {
                v = *reinterpret_cast<const u32x4*>(a.x + nb * a.ldx + c);
                if (a.x_dtype == SQ_BF16) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) v[k] = bf2h_x2(v[k]);
                }
            }
            *reinterpret_cast<u32x4*>(xs + i) = v;
        }
    } else {
        for (int i = tid; i < NB * C; i += 256) {
            const int nb = i / C, c = i - nb * C;
            uint16_t v = 0;
            if (nb < a.B) {
                v = a.x[nb * a.ldx + c];
                if (a.x_dtype == SQ_BF16) v = __builtin_bit_cast(uint16_t, bf2h(v));
            }
            xs[i] = v;
        }
    }
    __syncthreads();

    const int nsteps = (C + 1023) >> 10;
    int task = blockIdx.x, step = 0;
    if (task >= a.tasks) return;
    float acc[Q8_WAVE_ROWS * NB];
#pragma unroll
    for (int i = 0; i < Q8_WAVE_ROWS * NB; ++i) acc[i] = 0.f;
    Q8Regs cur, nxt;
    {
        const int col = lane * 16;
        q8_load(cur, a, task * Q8_TASK_ROWS + wave * Q8_WAVE_ROWS, col < C ? col : C - 16);
    }
    nxt = cur;
    while (task < a.tasks) {
        int ntask = task, nstep = step + 1;
        if (nstep == nsteps) { nstep = 0; ntask += gridDim.x; }
        if (ntask < a.tasks) {
            const int col = nstep * 1024 + lane * 16;
            q8_load(nxt, a, ntask * Q8_TASK_ROWS + wave * Q8_WAVE_ROWS, col < C ? col : C - 16);
        }
        {
            const int col = step * 1024 + lane * 16;
            const bool live = col < C;
            const int cc = live ? col : C - 16;
            half2v xf[NB][8];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const u32x4 lo = *reinterpret_cast<const u32x4*>(xs + nb * C + cc);
                const u32x4 hi = *reinterpret_cast<const u32x4*>(xs + nb * C + cc + 8);
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t l = lo[k], h = hi[k];
                    xf[nb][k] = __builtin_bit_cast(half2v, l);
                    xf[nb][4 + k] = __builtin_bit_cast(half2v, h);
                }
            }
#pragma unroll
            for (int i = 0; i < Q8_WAVE_ROWS; ++i) {
                half2v wh[8];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t wk = cur.w[i][k];
                    i8x4_to_h2(wk, wh[2 * k], wh[2 * k + 1]);
                }
                const float sc = live ? h2f(cur.s[i]) : 0.f;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    float d = 0.f;
#pragma unroll
                    for (int k = 0; k < 8; ++k) d = __builtin_amdgcn_fdot2(wh[k], xf[nb][k], d, false);
                    acc[i * NB + nb] += d * sc;
                }
            }
        }
        if (nstep == 0) {
            wave_sum_many<Q8_WAVE_ROWS * NB>(acc, lane);
            constexpr int SH = 6 - log2_of<Q8_WAVE_ROWS * NB>::value;
            const int idx = lane >> SH;
            const int i = idx / NB, nb = idx - i * NB;
            const int row = task * Q8_TASK_ROWS + wave * Q8_WAVE_ROWS + i;
            if ((lane & ((1 << SH) - 1)) == 0 && row < a.V && nb < a.B) store_y(a.y, a.y_dtype, nb * a.ldy + row, acc[0]);
#pragma unroll
            for (int k = 0; k < Q8_WAVE_ROWS * NB; ++k) acc[k] = 0.f;
        }
        cur = nxt;
        task = ntask;
        step = nstep;
    }
}

// ---- 3 .. Q8_MFMA_MAX_ROWS activation rows: fp16 MFMA, 16, 32 or 64 activation rows per pass.
// v_mfma_f32_16x16x32_f16 operand layout: A: lane l supplies weight row l % 16, k = 8 * (l / 16) .. + 7; B: token
// l % 16, the same k; D: lane l holds token l % 16, weight rows 4 * (l / 16) .. + 3.  Weights are the A operand and a
// wave owns 16 rows.  The rows reach the wave through LDS: global_load_lds (no registers in between) fetches them in
// lane order ALONG the row, one instruction = 8 rows x 128 bytes, whole cache lines with 8 consecutive lanes per
// line, into a private ring of Q8_RING steps per wave (a step = 16 rows x 128 columns = 2 KB); the wave reads its
// fragments back in the operand layout (lane (r, g) takes pieces 2 g and 2 g + 1 of row r, 32 bytes per step), so
// the weights need no barrier, only counted waits.  Rows are XOR-swizzled in 16-byte pieces (piece p of row r at
// slot p ^ ((r >> 1) & 7), applied through the source addresses of the copy), so the 16 lanes of an LDS read clock
// hit 16 different bank groups.  Block scales travel the same way (a 4-byte copy per lane: 16 bytes per row and
// chunk of 256 columns).  Each 16-byte piece feeds two MFMAs per block of 16 tokens; the k index of MFMA m of piece
// j is column 128 s + 16 (2 g + j) + 8 m + e, and the activations (B operand) are read with the same mapping from
// LDS, where the workgroup keeps the current 256-column chunk of the fp16 activations (global_load_lds, double
// buffered, one barrier per chunk).  The block scale is folded into the fp16 weight (one rounding, as the
// reference's tile kernel does, shapequant/kernels/batched_runs.py:442-447): all 16 weights of a piece sit in one
// block.  What bounds a pass: HBM up to 32 rows of a large head; beyond that, and in small heads, LDS reads (18 KB of fragments per tile and
// step at 64 rows, an eighth of them weights), conversions and matrix instructions of the waves of a CU, which barely overlap (64 rows of 8,000 x
// 3,584: 29 us, without the products 27, without what is in LDS read at all 18; two tiles of weights per fragment of x 44, each fragment read
// a step's start ahead 32).  A first form loaded the operand layout straight from memory (lane = row, 16 bytes per lane): every
// quarter wave then touches 16 different cache lines, and it stayed at 4.1-4.4 TB/s where this one reaches
// 5.2-5.5 TB/s (the one-row kernel: 5.7); 32 rows per wave on the 32x32x16 instruction was slower still.
constexpr int Q8_MFMA_MAX_ROWS = 320;           // up to here passes of 64 beat decode + tile GEMM (152,064 x 3,584: 151 us per pass,
                                                // 5 passes 755 us against ~880; 8 passes 1208 against 961 at 512 rows)

// x [B, C] (fp16 or bf16, any stride) -> fp16 [B, C] contiguous.
__global__ __launch_bounds__(256) void q8_x_kernel(const uint16_t* __restrict__ x, int64_t ldx, int B, int C, int x_dtype,
                                                   uint16_t* __restrict__ out) {
    const int64_t n = (int64_t)B * C;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int b = (int)(i / C), c = (int)(i - (int64_t)b * C);
        const uint16_t v = x[b * ldx + c];
        out[i] = x_dtype == SQ_BF16 ? __builtin_bit_cast(uint16_t, bf2h(v)) : v;
    }
}

struct Q8MfmaArgs {
    const int8_t* q;
    const uint16_t* sc;
    const uint16_t* xh;     // fp16, or bf16 where the kernel converts it, [B, ldxh], rows 16-byte aligned
    void* y;
    int64_t ldy;
    int ldxh;
    int V, C, B, y_dtype, tasks;
    int groups;             // groups of 16 NBLK tokens, each in workgroups of its own
    int vec_y;              // y rows allow 8-byte stores of 16-bit results (y 8-byte aligned, ldy % 4 == 0)
};

constexpr int q8_vmcnt(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }   // wait on vmcnt only

constexpr int Q8_RING = 3;                      // steps: one being multiplied, two in flight
// weights ring + scales of two chunks
enum { Q8_CHUNKS, Q8_PAIRS, Q8_ODD };       // rows of whole 256-column chunks, of whole pairs of blocks, of an odd number of blocks
constexpr int q8l_scale_bytes(int rows) { return rows == Q8_ODD ? 512 : 256; }
constexpr int q8l_wave_bytes(int rows) { return Q8_RING * 2048 + 2 * q8l_scale_bytes(rows); }
constexpr int q8l_lds_bytes(int nblk, int waves, int xs, int rows) { return 2 * nblk * 16 * xs * 256 + waves * q8l_wave_bytes(rows); }

// NBLK 16-token blocks, WAVES waves per workgroup,
// x chunks of XS steps (128 XS columns; a copy moves 4 / XS tokens, so the first 4 NBLK XS waves make one of every chunk, or all
// waves XI of them)
// ROWS: Q8_PAIRS (C % 64 == 0) and Q8_ODD are rows that end within a chunk.  The steps behind the row's end copy its last pieces again and
// multiply nothing.  Such rows ran on the exact-product kernel, so their block scales stay out of the fp16 weights: a matrix instruction takes
// the 32 columns of one block (lane group g: columns 8 g .. 8 g + 7) and its sums, fp32, are multiplied by the block's scales.
// Scales come in 4-byte pairs; every other row of an odd number of blocks begins within one, so there each comes by itself (a 2-byte copy per
// lane, which leaves them 4 bytes apart; twice the copies).
// CVT: x is bf16 and becomes fp16 on its way into LDS: its pieces are loaded into registers where they would be copied, converted and written
// behind the last product of the chunk (a launch that converted x first took 3 us of an eager call, 5 of the product's time on the device).
// The load is written out, and waited for by count like the copies beside it: the compiler would wait for all of those.  Its registers are
// named, above all that a kernel needs (106), since a compiler moves values that it believes to be there already.
template <int I> using int_c = std::integral_constant<int, I>;
constexpr int Q8_XR = 112;                      // 4 of them a piece
template <int I>
__device__ __forceinline__ void q8_x_load(const uint16_t* src) {
    asm volatile("global_load_dwordx4 v[%1:%2], %0, off" ::"v"(src), "n"(Q8_XR + 4 * I), "n"(Q8_XR + 4 * I + 3)
                 : "memory", "v112", "v113", "v114", "v115", "v116", "v117", "v118", "v119", "v120", "v121", "v122", "v123", "v124", "v125", "v126", "v127");
}
template <int I, int NEWER>                     // piece I, once all but the wave's NEWER last operations are done
__device__ __forceinline__ u32x4 q8_x_take() {
    uint32_t v[4];
    asm volatile("s_waitcnt vmcnt(%4)\n\tv_mov_b32 %0, v[%5]\n\tv_mov_b32 %1, v[%6]\n\tv_mov_b32 %2, v[%7]\n\tv_mov_b32 %3, v[%8]"
                 : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
                 : "n"(NEWER), "n"(Q8_XR + 4 * I), "n"(Q8_XR + 4 * I + 1), "n"(Q8_XR + 4 * I + 2), "n"(Q8_XR + 4 * I + 3) : "memory");
    return u32x4{v[0], v[1], v[2], v[3]};
}
constexpr int q8l_x_copies(int nblk, int waves, int xs) { return 4 * nblk * xs > waves ? 4 * nblk * xs / waves : 1; }
template <int NBLK, int WAVES, int XS, int ROWS, bool CVT, int XI = q8l_x_copies(NBLK, WAVES, XS)>
__global__ __launch_bounds__(WAVES * 64, WAVES == 8 ? 2 : 1) void q8_mfma_kernel(Q8MfmaArgs a) {
    static_assert(Q8_RING == 3 && (XS == 1 || XS == 2) && XI <= 4, "wait counts below are written out for these");
    constexpr bool ANY_C = ROWS != Q8_CHUNKS;
    constexpr int Q8L_WAVE_BYTES = q8l_wave_bytes(ROWS), SB = q8l_scale_bytes(ROWS), SC = SB / 256;      // SC: copies of a chunk's scales
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char* xs = smem;                                   // [2][16 NBLK tokens][256 XS bytes]
    constexpr int XPITCH = XS * 256, XBUF = NBLK * 16 * XPITCH;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    unsigned char* wl = smem + 2 * XBUF + wave * Q8L_WAVE_BYTES;  // this wave's ring
    unsigned char* sl_ = wl + Q8_RING * 2048;                      // this wave's scales: [2][16 rows][SB / 16 bytes]
    // the workgroups of the same weights are 8 apart: on one die, whose L2 the second finds them in
    const int tgroup = (blockIdx.x >> 3) % a.groups;
    const int task_raw = (int)((blockIdx.x >> 3) / a.groups * 8 + (blockIdx.x & 7)) * (int)(blockDim.x >> 6) + wave;
    if (task_raw - wave >= a.tasks) return;                     // (all waves of the workgroup)
    const uint16_t* xh = a.xh + (int64_t)tgroup * (NBLK * 16) * a.ldxh;
    const int nrows = min(a.B - tgroup * (NBLK * 16), NBLK * 16);
    const bool active = task_raw < a.tasks;
    const int task = active ? task_raw : a.tasks - 1;
    const int r = lane & 15, g = lane >> 4;
    const int C = a.C, nblk = C >> 5, nsteps = ANY_C ? ((C + 255) >> 8) * 2 : C >> 7, nchunks = nsteps / XS;

    typedef const __attribute__((address_space(1))) void* gptr_t;
    typedef __attribute__((address_space(3))) void* lptr_t;
    // activations: one copy instruction moves 1 KB = 4 / XS tokens of a chunk; the 16-byte piece p of token t is kept
    // at slot p ^ (t % 16), so the 16 lanes of a read clock (16 tokens, one piece) spread over 16 bank groups
    constexpr int TPI = 4 / XS, LPT = 64 / TPI;                 // tokens per instruction, lanes (= pieces) per token
    uint32_t xsrc[XI];
    int xcol[XI];                                               // this lane's column in a chunk
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const int rowx = (wave * XI + i) * TPI + lane / LPT;
        const int piece = (lane % LPT) ^ (rowx & 15);
        xcol[i] = piece * 8;
        xsrc[i] = (uint32_t)(min(rowx, nrows - 1) * a.ldxh + (ANY_C ? 0 : xcol[i]));
    }
    const bool xo = wave * XI * TPI < 16 * NBLK;                // this wave takes part in the x copies
    auto copy_x = [&](int c) __attribute__((always_inline)) {
        if (!xo) return;
        auto piece = [&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            if constexpr (i < XI) {
                const uint32_t at = ANY_C ? (uint32_t)min(c * (XS * 128) + xcol[i], C - 8) : (uint32_t)(c * (XS * 128));
                const uint16_t* src = xh + at + xsrc[i];
                if constexpr (CVT) q8_x_load<i>(src);
                else __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(xs + (c & 1) * XBUF + (wave * XI + i) * TPI * XPITCH), 16, 0, 0);
            }
        };
        piece(int_c<0>()); piece(int_c<1>()); piece(int_c<2>()); piece(int_c<3>());
    };
    // CVT: chunk c, once all but the wave's `newer` last operations are done
    auto put_x = [&](int c, auto newer) __attribute__((always_inline)) {
        if (!xo) return;
        auto piece = [&](auto i_) __attribute__((always_inline)) {
            constexpr int i = decltype(i_)::value;
            if constexpr (i < XI) {
                const u32x4 v = q8_x_take<i, decltype(newer)::value>();
                *reinterpret_cast<u32x4*>(xs + (c & 1) * XBUF + (wave * XI + i) * TPI * XPITCH + lane * 16) = u32x4{bf2h_x2(v.x), bf2h_x2(v.y), bf2h_x2(v.z), bf2h_x2(v.w)};
            }
        };
        piece(int_c<0>()); piece(int_c<1>()); piece(int_c<2>()); piece(int_c<3>());
    };
    // weights: instruction n of a step fills rows 8 n .. 8 n + 7; lane i lands in row 8 n + i / 8, slot i % 8 and
    // fetches the piece the swizzle keeps there
    const int8_t* wsrc[2];
    int wcol[2];                                                // this lane's column in a step
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const int rw = 8 * n + (lane >> 3);
        const int piece = (lane & 7) ^ ((rw >> 1) & 7);
        wcol[n] = piece * 16;
        wsrc[n] = a.q + (int64_t)min(task * 16 + rw, a.V - 1) * C + (ANY_C ? 0 : wcol[n]);
    }
    auto copy_w = [&](int s) {
#pragma unroll
        for (int n = 0; n < 2; ++n)
            __builtin_amdgcn_global_load_lds((gptr_t)(wsrc[n] + (ANY_C ? min(s * 128 + wcol[n], C - 16) : s * 128)), (lptr_t)(wl + (s % Q8_RING) * 2048 + n * 1024), 16, 0, 0);
    };
    // scales of chunk c: lane i fetches dword i % 4 of row i / 4 (Q8_ODD: scale i % 8 of rows i / 8 and 8 + i / 8)
    const uint16_t* sodd[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) sodd[n] = a.sc + (int64_t)min(task * 16 + 8 * n + (lane >> 3), a.V - 1) * nblk;
    const char* ssrc = (const char*)(a.sc + (int64_t)min(task * 16 + (lane >> 2), a.V - 1) * nblk) + (ANY_C ? 0 : (lane & 3) * 4);
    auto copy_s = [&](int c) {
        if constexpr (ROWS == Q8_ODD) {
#pragma unroll
            for (int n = 0; n < 2; ++n)
                __builtin_amdgcn_global_load_lds((gptr_t)(sodd[n] + min(c * 8 + (lane & 7), nblk - 1)), (lptr_t)(sl_ + (c % 2) * SB + n * 256), 2, 0, 0);
            return;
        }
        __builtin_amdgcn_global_load_lds((gptr_t)(ssrc + (ANY_C ? min(c * 16 + (lane & 3) * 4, nblk * 2 - 4) : c * 16)), (lptr_t)(sl_ + (c % 2) * SB), 4, 0, 0);
    };
    const uint32_t xrow = (uint32_t)r * XPITCH, xsw = (uint32_t)r;
    const uint32_t wsw = (uint32_t)((r >> 1) & 7);
    const uint32_t w0 = (uint32_t)r * 128 + (((uint32_t)(2 * g) ^ wsw) << 4), w1 = (uint32_t)r * 128 + (((uint32_t)(2 * g + 1) ^ wsw) << 4);

    float4v acc[NBLK];
#pragma unroll
    for (int nb = 0; nb < NBLK; ++nb) acc[nb] = float4v{0.f, 0.f, 0.f, 0.f};

    // Issue order per wave (X = this wave's x copy of a chunk, S = scales of a chunk, W = the 2 copies of a step):
    // S(c) goes right before W(2c); step s starts (even s: after the wait and the barrier, then X(s/2 + 1)) with the
    // refill of step s + 2.  Waits count the operations that may stay in flight:
    //   even s (needs X, S, W of its chunk):  W(s+1) -> 2
    //   odd s (needs W(s)):  X S W(s+1) W(s+2) -> 4 + SC + x   (x: this wave's XI copies)
    // and fall back to "everything" near the end of the row, where refills stop.
    auto refill = [&](int f) {
        if (f < nsteps) {
            if (!(f & 1)) copy_s(f >> 1);
            copy_w(f);
        }
    };
    copy_x(0);
#pragma unroll
    for (int t = 0; t < Q8_RING - 1; ++t) refill(t);
    if constexpr (CVT) put_x(0, int_c<4 + SC>());
    // CVT: x of the next chunk, before the barrier that opens it.  Behind its load: the refills of the chunk's steps
    auto next_x = [&](int s) __attribute__((always_inline)) {
        if constexpr (CVT) {
            const int cx = s / XS, f = s + Q8_RING - 1;               // (f: the step that this one's refill was for)
            if ((XS == 2 && !(s & 1)) || cx + 1 >= nchunks) return;
            if (f >= nsteps) put_x(cx + 1, int_c<0>());
            else if (XS == 2) put_x(cx + 1, int_c<4 + SC>());
            else if (f & 1) put_x(cx + 1, int_c<2>());
            else put_x(cx + 1, int_c<2 + SC>());
        }
    };
    // (the wait before a barrier, also for this wave's writes to LDS where there are any)
    auto ready = [&](auto newer) __attribute__((always_inline)) {
        if constexpr (CVT) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_waitcnt(q8_vmcnt(decltype(newer)::value));
    };
    auto step = [&](int s, auto odd) __attribute__((always_inline)) {
        const int c = s >> 1, cx = s / XS;         // chunk of scales, step in it, chunk of x
        if (XS == 1) {
            // every step opens an x chunk: X(s) was issued one step ago, before [S] W(s + 1)
            if (s + 1 < nsteps) { if (odd) ready(int_c<2 + SC>()); else ready(int_c<2>()); }
            else ready(int_c<0>());
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            if (cx + 1 < nchunks) copy_x(cx + 1);
            refill(s + Q8_RING - 1);
        } else if (!odd) {
            if (s + 1 < nsteps) ready(int_c<2>());
            else ready(int_c<0>());
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_sched_barrier(0);
            if (cx + 1 < nchunks) copy_x(cx + 1);
            refill(s + Q8_RING - 1);
        } else {
            refill(s + Q8_RING - 1);
            if (s + Q8_RING - 1 < nsteps) {
                if (xo) __builtin_amdgcn_s_waitcnt(q8_vmcnt(4 + SC + XI));
                else __builtin_amdgcn_s_waitcnt(q8_vmcnt(4 + SC));
            } else {
                __builtin_amdgcn_s_waitcnt(q8_vmcnt(0));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char* st = wl + (s % Q8_RING) * 2048;
        if constexpr (ANY_C) {
            typedef std::conditional_t<ROWS == Q8_ODD, u32x4, u32x2> scales_t;
            scales_t sb[4];                                     // the four blocks' scales of this lane's four output rows
#pragma unroll
            for (int v = 0; v < 4; ++v) sb[v] = *reinterpret_cast<const scales_t*>(sl_ + (c % 2) * SB + ((4 * g + v) * 2 + odd) * (SB / 32));
            const unsigned char* xc = xs + (cx & 1) * XBUF + xrow;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                if (s * 4 + b >= nblk) break;                   // (uniform: behind the row's end)
                const u32x2 wq = *reinterpret_cast<const u32x2*>(st + r * 128 + (((uint32_t)(2 * b + (g >> 1)) ^ wsw) << 4) + (g & 1) * 8);
                half2v p[4];
                i8x4_to_h2(wq[0], p[0], p[1]);
                i8x4_to_h2(wq[1], p[2], p[3]);
                half8v w;
                float sf[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    w[2 * k] = p[k][0]; w[2 * k + 1] = p[k][1];
                    sf[k] = h2f((uint16_t)(ROWS == Q8_ODD ? sb[k][b] : sb[k][b >> 1] >> ((b & 1) * 16)));
                }
                const uint32_t px = (uint32_t)((s % XS) * 16 + b * 4 + g);
#pragma unroll
                for (int nb = 0; nb < NBLK; ++nb) {
                    const half8v xv = *reinterpret_cast<const half8v*>(xc + nb * (16 * XPITCH) + ((px ^ xsw) << 4));
                    const float4v d = __builtin_amdgcn_mfma_f32_16x16x32_f16(w, xv, float4v{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[nb][v] += sf[v] * d[v];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            next_x(s);
            return;
        }
        const u32x4 wq[2] = {*reinterpret_cast<const u32x4*>(st + w0), *reinterpret_cast<const u32x4*>(st + w1)};
        const half_t sh = __builtin_bit_cast(half_t, *reinterpret_cast<const uint16_t*>(sl_ + (c % 2) * SB + r * 16 + odd * 8 + g * 2));
        const half2v s2 = {sh, sh};
        const unsigned char* xc = xs + (cx & 1) * XBUF + xrow;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            half2v p[8];
#pragma unroll
            for (int k = 0; k < 4; ++k) i8x4_to_h2(wq[j][k], p[2 * k], p[2 * k + 1]);
#pragma unroll
            for (int k = 0; k < 8; ++k) p[k] = p[k] * s2;
            half8v a0, a1;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                a0[2 * k] = p[k][0]; a0[2 * k + 1] = p[k][1];
                a1[2 * k] = p[4 + k][0]; a1[2 * k + 1] = p[4 + k][1];
            }
            const uint32_t p0 = (uint32_t)((s % XS) * 16 + (2 * g + j) * 2);   // x pieces (8 halves each) of these 16 columns
#pragma unroll
            for (int nb = 0; nb < NBLK; ++nb) {
                const unsigned char* xt = xc + nb * (16 * XPITCH);
                const half8v x0 = *reinterpret_cast<const half8v*>(xt + ((p0 ^ xsw) << 4));
                const half8v x1 = *reinterpret_cast<const half8v*>(xt + (((p0 + 1) ^ xsw) << 4));
                acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, x0, acc[nb], 0, 0, 0);
                acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, x1, acc[nb], 0, 0, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        next_x(s);
    };
    // Pairs of steps, each compiled for its place: us, step by step / so, 24 rows of 20,000 x 3,584 27.0 / 24.5, 64 of 8,000 x 3,584 23.3 / 21.4, 16 of
    // 152,064 x 3,584 112.5 / 111.2; but 24 and 32 rows of fp16 of the last 117.5 and 120.4 / 119.2 and 122.7
    if constexpr (!CVT && NBLK == 2 && WAVES == 8 && !ANY_C) {
        for (int s = 0; s < nsteps; ++s) step(s, s & 1);
    } else {
        for (int s = 0; s < nsteps; s += 2) {
            step(s, int_c<0>());
            step(s + 1, int_c<1>());
        }
    }
    if (!active) return;
    const int orow = task * 16 + g * 4;
#pragma unroll
    for (int nb = 0; nb < NBLK; ++nb) {
        if (nb * 16 + r >= nrows) continue;
        const int tok = tgroup * (NBLK * 16) + nb * 16 + r;
        if (a.vec_y && a.y_dtype != SQ_F32 && orow + 4 <= a.V) {
            uint16_t o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = a.y_dtype == SQ_BF16 ? f2bf(acc[nb][e]) : f2h(acc[nb][e]);
            *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(a.y) + (int64_t)tok * a.ldy + orow) =
                u32x2{(uint32_t)o[0] | ((uint32_t)o[1] << 16), (uint32_t)o[2] | ((uint32_t)o[3] << 16)};
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (orow + e < a.V) store_y(a.y, a.y_dtype, (int64_t)tok * a.ldy + orow + e, acc[nb][e]);
        }
    }
}

// N consecutive outputs of type T from fp32 values: 16-byte stores when the destination allows it.
template <int DT, int N>
__device__ __forceinline__ void store_run(typename store_as<DT>::type* dst, const float (&v)[N], bool vec) {
    typedef typename store_as<DT>::type T;
    if (vec) {
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int k = 0; k < N; k += 4)
                *reinterpret_cast<float4v*>(dst + k) = float4v{v[k], v[k + 1], v[k + 2], v[k + 3]};
        } else {
#pragma unroll
            for (int k = 0; k < N; k += 8) {
                u32x4 p;
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    p[e] = (uint32_t)store_as<DT>::cvt(v[k + 2 * e]) | ((uint32_t)store_as<DT>::cvt(v[k + 2 * e + 1]) << 16);
                *reinterpret_cast<u32x4*>(dst + k) = p;
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < N; ++k) dst[k] = store_as<DT>::cvt(v[k]);
    }
}

// Rows [r0, r1) as dense values, one 16-byte load (16 weights, half a block) per thread.
template <int DT>
__global__ __launch_bounds__(256) void q8_dequant_kernel(const int8_t* __restrict__ q, const uint16_t* __restrict__ sc,
                                                         int C, typename store_as<DT>::type* __restrict__ out,
                                                         int64_t ld_out, int r0, int64_t n16, int vec) {
    const int per_row = C >> 4;
    for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < n16; t += (int64_t)gridDim.x * 256) {
        const int rr = (int)(t / per_row), c = (int)(t - (int64_t)rr * per_row) * 16;
        const int64_t row = r0 + rr;
        const u32x4 v = *reinterpret_cast<const u32x4*>(q + row * C + c);
        const float s = h2f(sc[row * (C >> 5) + (c >> 5)]);
        float o[16];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t w = v[k];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[4 * k + e] = (float)(int8_t)(w >> (8 * e)) * s;
        }
        store_run<DT, 16>(out + (int64_t)rr * ld_out + c, o, vec != 0);
    }
}

// Embedding rows: 8 weights and one 16-byte store per thread, so a wave stores whole lines one after another (a block of 32 weights per thread left 64
// bytes between the lanes' stores and a quarter of the waves: 2,048 rows of 3,584 columns, 14.7 MB of results, 9.0 us, 6.9 so; with a head of
// 16 rows of 152,064 x 3,584 120.3 / 118.2 us).  Numbers of pieces are 32-bit where they fit: a division for each.  Ids outside [0, V) give a row of zeros.
template <int DT, class I>
__global__ __launch_bounds__(256) void q4_embed_kernel(const uint8_t* __restrict__ q, const uint16_t* __restrict__ sc,
                                                       int V, int C, const int64_t* __restrict__ ids, I total,
                                                       typename store_as<DT>::type* __restrict__ out, int64_t ld_out, int vec) {
    const int nblk = C >> 5, pieces = C >> 3;
    for (I t = (I)blockIdx.x * 256 + threadIdx.x; t < total; t += (I)gridDim.x * 256) {
        const I i = t / pieces;
        const int p = (int)(t - i * pieces);
        const int64_t id = ids[i];
        float o[8] = {};
        if (id >= 0 && id < V) {
            const uint32_t w = *reinterpret_cast<const uint32_t*>(q + id * (C >> 1) + p * 4);
            const float s = h2f(sc[id * nblk + (p >> 2)]);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (float)((int)((w >> (4 * e)) & 15u) - 8) * s;
        }
        store_run<DT, 8>(out + (int64_t)i * ld_out + p * 8, o, vec != 0);
    }
}

static int q8_pass_rows(int B, int C) {
    int nb = B > 2 ? 4 : B > 1 ? 2 : 1;
    while (nb > 1 && nb * C > Q8_LDS_HALVES) nb >>= 1;
    return nb;
}

// The MFMA passes need 64 activation rows of C halves within 32-bit offsets.
static bool q8_mfma_ok(int C) { return C % 32 == 0 && (int64_t)C * 64 < ((int64_t)1 << 31); }

// from 3 rows the MFMA passes win over the 4-row kernel (152,064 x 3,584: 106 against 148 us; 248,320 x 5,120: 246
// against 255 us); 2 rows stay on the exact-product kernel (106-115 / 228 us)
// Rows that are not whole 256-column chunks, us, exact-product kernel or (above 32 rows) decode + tile GEMM / these passes: 25 rows of
// 141,347 x 1,408 348 / 47, of 9,823 x 3,456 102 / 29, 8 of 70,061 x 1,216 63 / 24.5.  A small grid is bound by the length of a wave's
// chain, 0.8 us per 128 columns: 3 rows of 9,823 x 3,456 15.9 / 24, of 16,000 x 1,216 8.3 / 10.7, of 32,000 x 640 8.9 / 7.9, of 30,000 x 1,216
// 15.1 / 12.1; 5 of 9,823 x 3,456 25.2 / 22.6, of 8,192 x 1,408 10.4 / 11.7; 16 of 1,024 x 1,408 23.3 / 12.4; 64 of 9,823 x 3,456 45.5 / 39,
// of 16,000 x 3,456 59.5 / 38, of 8,211 x 576 33 / 18.  A second pass: 100 rows of
// 30,000 x 1,216 41.3 / 41.9, of 32,000 x 640 33.6 / 27.6, of 50,000 x 3,520 203 / 106, 200 of 70,061 x 1,216 164 / 170.
// Rows of an odd number of blocks: 8 / 16 / 32 / 64 rows of 150,000 x 3,488 246 / 490 / 974 / 877 (127 / 131 / 144 / 189 here), of 8,400 x 2,528 24 / 45 / 88 /
// 95 (24 / 19 / 24 / 32), 4 of 60,000 x 2,080 39 / 30; of 30,000 x 608 both are done before an eager call is issued, 4 / 5 / 8 rows 14 / 17 / 20 there and 17.5
// here, when its calls still launched a copy of x.
// 3 rows of 105,038 x 3,392, which the 256 MB last-level cache does not hold from call to call: 86.5 / 90.5; 5 take two passes there.
bool q8_mid(int V, int C, int B) {
    if (B <= 2 || !q8_mfma_ok(C)) return false;
    if (C % 256 == 0) return B <= Q8_MFMA_MAX_ROWS;
    if (C % 64 && B <= 5 && (int64_t)V * C < (int64_t)48 << 20) return false;
    if (B <= 4) return V >= 30000 && (int64_t)V * C <= (int64_t)240 << 20;
    if (B > 64) return V >= 30000 && B <= 128;
    if (B <= 8) return V >= 9000;
    return V >= 1024 && (B <= 32 || V >= 8000 || C <= 2048);
}
size_t q8_mid_workspace(int V, int C, int B) { return q8_mid(V, C, B) ? (((size_t)B * C * 2) + 255) & ~(size_t)255 : 0; }

int launch_q8_mid(const int8_t* q, const uint16_t* sc, int V, int C, const void* x, int x_dtype, int64_t ldx, void* y,
                  int y_dtype, int64_t ldy, int B, void* ws, size_t ws_bytes, hipStream_t s) {
    if (ws_bytes < q8_mid_workspace(V, C, B)) return fail(SQ_EWORKSPACE, "sq_q8_linear: workspace %zu < %zu", ws_bytes, q8_mid_workspace(V, C, B));
    const size_t ys = y_dtype == SQ_F32 ? 4 : 2;
    // Activations with 16-byte aligned rows go to LDS from where they are, anything else goes through an fp16 copy in the workspace first; bf16 too
    // where many rows (> 32) make the conversion in the kernel, 0.17 us per step of 128 columns and round of workgroups, longer than the launch.
    // us per eager call, copy / converted in the kernel: 4 rows of 8,000 x 1,024 16.7 / 14.5, of 32,000 x 3,584 24.2 / 22.1, 16 of 64,000 x 2,048 27.1 /
    // 25.0, of 152,064 x 3,584 111.9 / 109.7; 64 of 32,000 x 1,024 16.8 / 14.6, of 8,000 x 3,584 20.4 / 23.3, of 152,064 x 3,584 151 / 160.
    const uint16_t* xh = (const uint16_t*)x;
    int64_t ldxh = ldx;
    const int cus = device_cus(), tasks = (V + 15) / 16, n4 = (tasks + 3) / 4, n8 = (tasks + 7) / 8, n16 = (tasks + 15) / 16;
    bool cvt = x_dtype == SQ_BF16 && (B <= 32 || (n8 <= cus && C <= 1920));
    int rc;
    if ((x_dtype != SQ_F16 && !cvt) || ((uintptr_t)x & 15) || ldx % 8 || ldx * 64 >= ((int64_t)1 << 31)) {
        const int64_t n = (int64_t)B * C;
        const int64_t want = (n + 255) / 256;
        hipLaunchKernelGGL(q8_x_kernel, dim3((unsigned)(want < 4096 ? want : 4096)), dim3(256), 0, s, (const uint16_t*)x, ldx, B,
                           C, x_dtype, (uint16_t*)ws);
        rc = check_launch("q8_x_kernel");
        if (rc) return rc;
        xh = (const uint16_t*)ws;
        ldxh = C;
        cvt = false;
    }
    for (int b0 = 0; b0 < B;) {
        const int pass = B - b0 > 32 ? 64 : 32;                  // activation rows of this pass at most
        Q8MfmaArgs a{};
        a.q = q; a.sc = sc;
        a.xh = xh + (int64_t)b0 * ldxh;
        a.ldxh = (int)ldxh;
        a.y = (char*)y + (size_t)b0 * ldy * ys;
        a.ldy = ldy; a.V = V; a.C = C; a.B = B - b0 < pass ? B - b0 : pass; a.y_dtype = y_dtype; a.tasks = tasks;
        a.vec_y = ((uintptr_t)a.y & 7) == 0 && ldy % 4 == 0;
        // 17-32 rows: one workgroup of 16 waves per CU sharing 256-column x chunks, unless its workgroups fill the last
        // round of the chip badly; then 8 waves with 128-column chunks (a barrier per step, two workgroups per CU).
        // Measured: 152,064 x 3,584 (594 workgroups of 16 waves, 2.3 rounds) 126 against 116 us; 248,320 x 5,120
        // (970, 3.8 rounds) 265 against 278 us.
        const bool x128 = (double)n16 / ((double)((n16 + cus - 1) / cus) * cus) < 0.85;
        const int rows = C % 256 == 0 ? Q8_CHUNKS : C % 64 == 0 ? Q8_PAIRS : Q8_ODD;
        a.groups = 1;
        auto go = [&](auto chunks, auto pairs, auto odd, int nblk, int waves, int xs) {
            const int wgs = (tasks + waves - 1) / waves;
            hipLaunchKernelGGL(rows == Q8_CHUNKS ? chunks : rows == Q8_PAIRS ? pairs : odd, dim3((unsigned)(a.groups > 1 ? (wgs + 7) / 8 * 8 * a.groups : wgs)),
                               dim3((unsigned)waves * 64), q8l_lds_bytes(nblk, waves, xs, rows), s, a);
        };
        static bool raised = false;
        if (!raised) {
            auto raise = [](auto... k) { ((void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024), ...); };
#define SQ_Q8C(CV, N, W, X, ...) q8_mfma_kernel<N, W, X, Q8_CHUNKS, CV, ##__VA_ARGS__>, q8_mfma_kernel<N, W, X, Q8_PAIRS, CV, ##__VA_ARGS__>, q8_mfma_kernel<N, W, X, Q8_ODD, CV, ##__VA_ARGS__>
#define SQ_Q8(...) SQ_Q8C(false, __VA_ARGS__), SQ_Q8C(true, __VA_ARGS__)
            raise(SQ_Q8(1, 8, 2), SQ_Q8(2, 16, 2), SQ_Q8(2, 8, 1), SQ_Q8(4, 16, 1), SQ_Q8(4, 8, 1), SQ_Q8(4, 8, 1, 4));
#undef SQ_Q8
            (void)hipGetLastError();
            raised = true;
        }
#define SQ_GO(N, W, X, WAVES, ...) do { if (cvt) go(SQ_Q8C(true, N, W, X, ##__VA_ARGS__), N, WAVES, X); else go(SQ_Q8C(false, N, W, X, ##__VA_ARGS__), N, WAVES, X); } while (0)
        // Small heads: half the waves per workgroup, each making twice the copies of x, spread the same waves over twice the CUs (LDS reads,
        // conversions and matrix instructions are what they take).  us, before / so: 16 rows of 9,728 x 3,584 19.7 /
        // 17.8, of 10,000 x 2,048 12.7 / 12.1, of 30,000 x 2,048 14.3 / 14.8; 64 rows of 9,728 x 3,584 44.7 / 30.5, of 32,000 x 3,584 45.9 / 31.9,
        // of 60,000 x 2,048 31.0 / 37.4.  Where the weights' tiles still leave half of the CUs idle, groups of tokens take workgroups of their
        // own: 64 rows of 8,000 x 3,584 29.4 / 18.5, of 16,000 x 3,456 37.5 / 25.8 (of 20,000 x 3,584, more than half, 29.3 / 31.4), 24 of 8,000 x 3,584
        // 20.0 / 17.9, of 16,000 x 3,456 27.9 / 23.5.
        // 33-64 rows of larger heads: two workgroups of 7 waves to a CU where those of 16 fill the last round badly (64 rows of 152,064 x 896 52.7 / 44.7,
        // of 152,064 x 3,584 151.8 / 150.4, of 100,000 x 2,048 55.7 / 50.8, of 40,000 x 3,584 45.7 / 39.9; of 64,000 x 2,048, one round, 33.9 / 41.6); with
        // the scales of an odd number of blocks two do not fit (152,064 x 1,056 69 / 79).
        const bool small = a.B > 32 ? n8 <= cus : n8 <= cus / 2;
        if (small && a.B > 32 && 2 * n4 <= cus) {
            a.groups = 2;
            SQ_GO(2, 4, 1, 4);
        } else if (small && a.B > 32 && 2 * n8 <= cus) {
            a.groups = 2;
            SQ_GO(2, 8, 1, 8);
        } else if (small && a.B > 32) {
            SQ_GO(4, 8, 1, 8);
        } else if (small) {
            a.groups = a.B > 16 ? 2 : 1;
            SQ_GO(1, 4, 2, 4);
        } else if (a.B > 32 && x128 && rows != Q8_ODD) {
            SQ_GO(4, 8, 1, 7, 4);
        } else if (a.B > 32) {                                       // 33-64 rows: 16 waves share 128-column chunks of 64 tokens
            SQ_GO(4, 16, 1, 16);
        } else if (a.B > 16 && x128) {
            SQ_GO(2, 8, 1, 8);
        } else if (a.B > 16) {
            SQ_GO(2, 16, 2, 16);
        } else {
            SQ_GO(1, 8, 2, 8);
        }
#undef SQ_GO
#undef SQ_Q8C
        rc = check_launch("q8_mfma_kernel");
        if (rc) return rc;
        b0 += a.B;
    }
    return SQ_OK;
}

int launch_q8_small(const int8_t* q, const uint16_t* sc, int V, int C, const void* x, int x_dtype, int64_t ldx, void* y,
                    int y_dtype, int64_t ldy, int B, hipStream_t s) {
    if (C > Q8_LDS_HALVES) return fail(SQ_EUNSUPPORTED, "sq_q8_linear: C %d > %d", C, Q8_LDS_HALVES);
    const size_t ys = y_dtype == SQ_F32 ? 4 : 2;
    const int tasks = (V + Q8_TASK_ROWS - 1) / Q8_TASK_ROWS;
    const int max_wgs = 2 * device_cus();
    const int per = (tasks + max_wgs - 1) / max_wgs;
    const unsigned grid = (unsigned)((tasks + per - 1) / per);
    for (int b0 = 0; b0 < B;) {
        const int nb = q8_pass_rows(B - b0, C);
        Q8Args a{};
        a.q = q; a.sc = sc;
        a.x = (const uint16_t*)x + (int64_t)b0 * ldx;
        a.y = (char*)y + (size_t)b0 * ldy * ys;
        a.ldx = ldx; a.ldy = ldy; a.V = V; a.C = C;
        a.B = B - b0 < nb ? B - b0 : nb;
        a.x_dtype = x_dtype; a.y_dtype = y_dtype; a.tasks = tasks;
        a.x_vec = ((uintptr_t)a.x & 15) == 0 && (a.B == 1 || ldx % 8 == 0) && C % 8 == 0;
        const size_t lds = (size_t)nb * C * 2;
        if (nb == 4) hipLaunchKernelGGL(q8_gemv_kernel<4>, dim3(grid), dim3(256), lds, s, a);
        else if (nb == 2) hipLaunchKernelGGL(q8_gemv_kernel<2>, dim3(grid), dim3(256), lds, s, a);
        else hipLaunchKernelGGL(q8_gemv_kernel<1>, dim3(grid), dim3(256), lds, s, a);
        int rc = check_launch("q8_gemv_kernel");
        if (rc) return rc;
        b0 += a.B;
    }
    return SQ_OK;
}

int launch_q8_dequant(const int8_t* q, const uint16_t* sc, int C, void* out, int out_dtype, int64_t ld_out, int r0, int r1,
                      hipStream_t s) {
    const int64_t n16 = (int64_t)(r1 - r0) * (C >> 4);
    if (n16 == 0) return SQ_OK;
    const int64_t want = (n16 + 255) / 256;
    const unsigned grid = (unsigned)(want < 65536 ? want : 65536);
    const int64_t per16 = out_dtype == SQ_F32 ? 4 : 8;          // elements per 16 bytes
    const int vec = ((uintptr_t)out & 15) == 0 && ld_out % per16 == 0;
    if (out_dtype == SQ_F32)
        hipLaunchKernelGGL(q8_dequant_kernel<SQ_F32>, dim3(grid), dim3(256), 0, s, q, sc, C, (float*)out, ld_out, r0, n16, vec);
    else if (out_dtype == SQ_F16)
        hipLaunchKernelGGL(q8_dequant_kernel<SQ_F16>, dim3(grid), dim3(256), 0, s, q, sc, C, (uint16_t*)out, ld_out, r0, n16, vec);
    else
        hipLaunchKernelGGL(q8_dequant_kernel<SQ_BF16>, dim3(grid), dim3(256), 0, s, q, sc, C, (uint16_t*)out, ld_out, r0, n16, vec);
    return check_launch("q8_dequant_kernel");
}

int launch_q4_embed(const uint8_t* q, const uint16_t* sc, int V, int C, const int64_t* ids, int64_t n_ids, void* out,
                    int out_dtype, int64_t ld_out, hipStream_t s) {
    const int64_t total = n_ids * (C >> 3);
    if (total == 0) return SQ_OK;
    const int64_t want = (total + 255) / 256;
    const unsigned grid = (unsigned)(want < 65536 ? want : 65536);
    const int64_t per16 = out_dtype == SQ_F32 ? 4 : 8;
    const int vec = ((uintptr_t)out & 15) == 0 && ld_out % per16 == 0;
#define SQ_GO(DT) do { \
        if (total < ((int64_t)1 << 31)) hipLaunchKernelGGL((q4_embed_kernel<DT, uint32_t>), dim3(grid), dim3(256), 0, s, q, sc, V, C, ids, (uint32_t)total, (store_as<DT>::type*)out, ld_out, vec); \
        else hipLaunchKernelGGL((q4_embed_kernel<DT, int64_t>), dim3(grid), dim3(256), 0, s, q, sc, V, C, ids, total, (store_as<DT>::type*)out, ld_out, vec); \
    } while (0)
    if (out_dtype == SQ_F32) SQ_GO(SQ_F32);
    else if (out_dtype == SQ_F16) SQ_GO(SQ_F16);
    else SQ_GO(SQ_BF16);
#undef SQ_GO
    return check_launch("q4_embed_kernel");
}

}  // namespace sq
