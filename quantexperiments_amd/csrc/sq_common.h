// Shared device helpers for the gfx950 codebook-linear kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/sqhip.h"

namespace sq {

typedef _Float16 half_t;
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4v __attribute__((ext_vector_type(4)));
typedef _Float16 half8v __attribute__((ext_vector_type(8)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int WAVE = 64;

__device__ __forceinline__ float h2f(uint16_t b) { return (float)__builtin_bit_cast(half_t, b); }
__device__ __forceinline__ float bf2f(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }

// fp32 -> bf16 bits, round to nearest even, NaN stays NaN: one v_cvt_pk_bf16_f32, which takes two values (the rounding
// written out in integers cost 30 us of a 520 us product with a 2048 x 37888 bf16 output).
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ uint32_t f2bf_x2(float lo, float hi) {
    typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v){lo, hi}, bf2v));
}
// fp32 -> fp16 bits, round to nearest even.  The empty asm hides where f came from: a multiply feeding this conversion
// is otherwise folded into v_fma_mixlo_f16, which rounds the exact product to fp16 once, while the same expression
// elsewhere in a kernel stays v_mul_f32 + v_cvt_f16_f32 (two roundings, the reference's arithmetic) and differs in
// the last bit of about one value in 2000.
__device__ __forceinline__ uint16_t f2h(float f) {
    asm("" : "+v"(f));
    return __builtin_bit_cast(uint16_t, (half_t)f);
}

__device__ __forceinline__ uint32_t f2h_x2(float lo, float hi) {
    asm("" : "+v"(lo), "+v"(hi));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((float2v){lo, hi}, half2v));
}

// bf16 bits -> fp16 value (through fp32; exact whenever the value is an fp16 normal,
// rounds to nearest even in the fp16 subnormal range, +-inf beyond 65504).
__device__ __forceinline__ half_t bf2h(uint16_t b) { return (half_t)bf2f(b); }

// two packed bf16 (one dword) -> two packed fp16
__device__ __forceinline__ uint32_t bf2h_x2(uint32_t v) {
    half2v h;
    h.x = (half_t)__builtin_bit_cast(float, v << 16);
    h.y = (half_t)__builtin_bit_cast(float, v & 0xFFFF0000u);
    return __builtin_bit_cast(uint32_t, h);
}

// 16-bit activations of a run-time dtype (SQ_F16 / SQ_BF16)
__device__ __forceinline__ float load16(const void* p, int dtype, int64_t i) {
    const uint16_t b = reinterpret_cast<const uint16_t*>(p)[i];
    return dtype == SQ_BF16 ? bf2f(b) : h2f(b);
}
__device__ __forceinline__ uint16_t round16(float v, int dtype) { return dtype == SQ_BF16 ? f2bf(v) : f2h(v); }

// silu(g) * u with the reference's rounding points (shapequant/kernels/decode_e2e.py:125-136): SiLU in fp32 rounded
// to the model dtype, then the product rounded to the model dtype.  One definition, because the stand-alone kernel
// and the products that compute their own input must agree bit for bit.
__device__ __forceinline__ uint16_t silu_mul_one(uint16_t g, uint16_t u, int dtype) {
    if (dtype == SQ_BF16) {
        const float a = bf2f(g);
        return f2bf(bf2f(f2bf(a / (1.f + __expf(-a)))) * bf2f(u));
    }
    const float a = h2f(g);
    const half_t s = (half_t)(a / (1.f + __expf(-a)));
    return __builtin_bit_cast(uint16_t, (half_t)(s * __builtin_bit_cast(half_t, u)));
}

template <int DT> struct store_as;
template <> struct store_as<SQ_F32> { typedef float type; static __device__ __forceinline__ float cvt(float f) { return f; } };
template <> struct store_as<SQ_F16> { typedef uint16_t type; static __device__ __forceinline__ uint16_t cvt(float f) { return f2h(f); } };
template <> struct store_as<SQ_BF16> { typedef uint16_t type; static __device__ __forceinline__ uint16_t cvt(float f) { return f2bf(f); } };

// Two 16-bit results of one token, of neighbouring weight rows; over: the first one's row less the number of rows (-2 and less: both are there)
__device__ __forceinline__ void store_pair(uint16_t* at, uint32_t v, int over, bool whole) {
    if (whole && over <= -2) { *reinterpret_cast<uint32_t*>(at) = v; return; }
    if (over < 0) at[0] = (uint16_t)v;
    if (over < -1) at[1] = (uint16_t)(v >> 16);
}

__device__ __forceinline__ void store_y(void* y, int y_dtype, int64_t o, float v) {
    if (y_dtype == SQ_BF16) reinterpret_cast<uint16_t*>(y)[o] = f2bf(v);
    else if (y_dtype == SQ_F16) reinterpret_cast<uint16_t*>(y)[o] = f2h(v);
    else reinterpret_cast<float*>(y)[o] = v;
}

// Tag j of a row's little-endian bit stream (any width 1..16).  `W` bounds the second word.
__device__ __forceinline__ uint32_t tag_at(const uint32_t* __restrict__ row, int W, int bits, int j) {
    const int p = j * bits, w = p >> 5, s = p & 31;
    const uint32_t lo = row[w];
    const uint32_t hi = (s + bits > 32 && w + 1 < W) ? row[w + 1] : 0u;
    const uint64_t v = ((uint64_t)hi << 32) | lo;
    return (uint32_t)(v >> s) & ((1u << bits) - 1u);
}

// Sum over the wave, the same in every lane: v += v of lane ^ 32, then ^ 16, 8, 4, 2, 1.  In registers: swaps of half waves and of
// rows of 16 lanes, and rotations of a row, whose values repeat every 8, 4, 2 lanes by the time they are rotated by 4, 2, 1 (through
// __shfl_xor, six LDS round trips one behind the other, an add + norm of 8 x 3584 took 0.3 us more).
template <int N> __device__ __forceinline__ uint32_t row_rotated_bits(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x120 + N, 0xF, 0xF, false);
}
template <int N> __device__ __forceinline__ float row_rotated(float v) {
    return __builtin_bit_cast(float, row_rotated_bits<N>(__builtin_bit_cast(uint32_t, v)));
}
__device__ __forceinline__ float lane_groups_sum(float v) {        // over lanes 16 apart
    const uint32_t a = __builtin_bit_cast(uint32_t, v);
    const auto h = __builtin_amdgcn_permlane32_swap(a, a, false, false);
    v = __builtin_bit_cast(float, (uint32_t)h[0]) + __builtin_bit_cast(float, (uint32_t)h[1]);
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    return __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
}
__device__ __forceinline__ float wave_sum(float v) {
    v = lane_groups_sum(v);
    v += row_rotated<8>(v); v += row_rotated<4>(v); v += row_rotated<2>(v);
    return v + row_rotated<1>(v);
}

// A caller's workspace starts with SQ_WS_HEADER bytes that only the tag-stream kernel touches: the partial sums its
// workgroups exchange.  Every word of them is zero whenever no call is running (a partial sum doubles as its own arrival
// flag and whoever adds it up puts zero back), so they must be zero when the workspace is first handed over and nothing
// else may ever be written there; the other launchers get the part behind the header.
constexpr size_t SQ_WS_HEADER = (size_t)32 << 20;
// The partial sums fill at most the first SQ_WS_SUMS bytes of the header; its last page holds the error word of the
// exchange (at SQ_WS_ERR_OFF): set by a workgroup that gave up waiting for a partial sum, read by every later launch
// (which then writes NaN everywhere: partial sums that arrive late leave the header dirty, and a dirty header must
// never yield finite numbers), cleared by sq_workspace_reset.
constexpr size_t SQ_WS_SUMS = SQ_WS_HEADER - 4096;
constexpr size_t SQ_WS_ERR_OFF = SQ_WS_HEADER - 256;

// error plumbing shared by the launchers (defined in sq_api.hip)
int fail(int code, const char* fmt, ...);
int check_launch(const char* what);
int device_cus();       // compute units of the current device (cached)

// launchers implemented in the kernel translation units
int launch_dequant(const sq_matrix& m, void* out, int out_dtype, int64_t ld_out, int r0, int r1, hipStream_t s,
                   bool raw = false);
int launch_small(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype,
                 int64_t ldy, int B, void* ws, size_t ws_bytes, void* sums, hipStream_t s,
                 const sq_producer* from = nullptr);
// one activation row of these pieces is a single launch of the tag-stream kernel, which can produce its own x
int sieve_group(const sq_matrix* mats, int n, int T);
size_t sieve_workspace(const sq_matrix* mats, int n, int T);
// What sq_linear_small_noalloc has behind its header.  Kernels that keep sums for up to SQ_SMALL_BMAX rows take the same cuts, and so the same sums, with this much
// as with more: in parts of the rows, or because they plan with no more than this.  The _least sizes are what they can do with, in more launches: this, or less
// where there is less to keep
constexpr size_t SMALL_ROOM = (size_t)16 << 20;
size_t sieve_workspace_least(const sq_matrix* mats, int n, int T);
int launch_sieve(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws, size_t ws_bytes, hipStream_t s);
bool small_fuses_producer(const sq_matrix* mats, int n, int B);
// the two pieces are a gate and an up projection whose launch can write SiLU(gate) * up itself
bool small_fuses_silu(const sq_matrix* mats, int n, int B);
int launch_small_silu(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* act, int64_t ld_act, int B,
                      void* sums, hipStream_t s, const sq_producer* from = nullptr);
size_t small_workspace(const sq_matrix* mats, int n, int B);
size_t small_workspace_least(const sq_matrix* mats, int n, int B);     // what launch_small can do with
// some piece runs the tag-stream kernel, whose partial sums live in the workspace header (`sums` above)
bool small_uses_sums(const sq_matrix* mats, int n);
int launch_gemm(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype,
                int64_t ldy, int T, void* ws, size_t ws_bytes, void* sums, hipStream_t s);
// stacks with column orders and more than a few activation rows: sq_linear_small runs the decode + tile GEMM route
bool small_takes_gemm_route(const sq_matrix* mats, int n, int B, const void* x, int64_t ldx);
size_t small_gemm_route_workspace(const sq_matrix* mats, int n, int B);
bool has_orders(const sq_matrix* mats, int n);
constexpr int MID_PIECES = 8;          // (kernel arguments of 1 KB)
// the piece would run on the vector kernels at B rows; how many such pieces sq_linear_small decodes and multiplies from there; their call
bool small_vector(const sq_matrix& m, int B);
int vector_decoded(const sq_matrix* mats, int n, int B);
size_t decoded_workspace(const sq_matrix* mats, int n, int T);
// (wide: bf16 activations keep their range and bits, up to 48 rows)
int launch_decoded(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws, hipStream_t s,
                   bool wide = false);
// products in one pass over the tags (sq_mid.h): whether it is the way of these pieces in any case, its cut with the estimated time (with `room` bytes for sums; nt = 0
// and a very long time: not for these), and its call, with the cut that mid_plan gave for a workspace of any size or without it
struct MidPlan { int nt, tw, nw, st, ks; float us; };
MidPlan mid_plan(const sq_matrix* mats, int n, int T, size_t room = SIZE_MAX);
bool mma_shape(const sq_matrix& m);
bool mid_ok(const sq_matrix* mats, int n, int T);
inline bool mid_x_ok(int64_t ldx, int T) { return (int64_t)T * ldx * 2 < (int64_t)1 << 32; }     // 32-bit offsets
size_t mid_workspace(const sq_matrix* mats, int n, int T, const MidPlan* planned = nullptr);
size_t mid_least(const sq_matrix* mats, int n, int T);                   // (where mid_ok)
int launch_mid(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws,
               size_t ws_bytes, hipStream_t s, const MidPlan* planned = nullptr);
// the same for weights already decoded to fp16, w[i] = [R, C] of piece i without row scales (1 .. 256 activation rows)
bool mid_dense_ok(const sq_matrix* mats, int n, int T);
size_t mid_dense_workspace(const sq_matrix* mats, int n, int T);
int launch_mid_decoded(const sq_matrix* mats, int n, const void* const* w, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T,
                       void* ws, hipStream_t s, bool wide);
// more rows in tiles whose weights are gathered on their way into LDS (sq_fused.h)
struct FusedPlan { int nw, tw, ks, tbs, t; };      // (t: activation rows)
FusedPlan fused_plan(const sq_matrix* mats, int n, int T);               // nw = 0: not for these
bool fused_two_blocks(const FusedPlan& p, const sq_matrix* mats, int n);      // of tokens, in one round of workgroups
float fused_us(const FusedPlan& p, const sq_matrix* mats, int n);        // (d = 8: of those)
size_t fused_workspace(const FusedPlan& p, const sq_matrix* mats, int n, int T);
int launch_fused(const FusedPlan& p, const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws, hipStream_t s);
// most activation rows for which passes of SQ_SMALL_BMAX rows through the decode-time kernel beat decode + GEMM
// for these pieces (0: never), where they cannot share a pass
int small_pass_limit(const sq_matrix* mats, int n);
size_t gemm_workspace(const sq_matrix* mats, int n, int T);
constexpr int PLANE_PRODUCT_MIN_T = 17;
struct PlanePlan { int tw, nt, pl, parts[MID_PIECES]; double us; };
// The kernel that sq_linear_gemm runs n pieces on at more than SQ_SMALL_BMAX rows of aligned activations, given the workspace: sq_fused.h,
// sq_plane_product.hip, sq_mid.h, passes of the decode-time kernel, decoded rows on sq_mid.h, the tile GEMM behind a decode (in 128 x 128 tiles: none)
enum GemmKernel { GEMM_FUSED = 1, GEMM_COLUMNS, GEMM_MID, GEMM_PASSES, GEMM_DECODED, GEMM_TILES };
struct GemmRoute { GemmKernel kernel; FusedPlan fused; MidPlan mid; PlanePlan columns; };      // and the cuts that were planned on the way (nw = 0, nt = 0: none)
GemmRoute gemm_route(const sq_matrix* mats, int n, int T, int x_dtype);
// what launch_gemm can do with less: the same product without the kernel of sq_mid.h
size_t gemm_workspace_without_mid(const sq_matrix* mats, int n, int T);
// Row scales of a product whose R rows are n stacked pieces: rows end[i - 1] .. end[i] - 1 are scaled by p[i]; n = 0: no scales.
// (Eight: kernel arguments of 1 KB in the stacked decode; longer stacks take a product per eight pieces.  Four had sent stacks of five
// pieces through five products.)
constexpr int GEMM256_PIECES = 8;
struct Gemm256Scales { const uint16_t* p[GEMM256_PIECES]; int end[GEMM256_PIECES]; int n; };
int launch_bf16_to_f16(const uint16_t* x, int64_t ldx, int T, int C, uint16_t* out, hipStream_t s);
// 16-bit tags of width 8 decoded a column of the codebook at a time, results and activations in plane order (sq_planes.hip)
bool planes_ok(const sq_matrix* mats, int n);
bool planes_route(const sq_matrix* mats, int n, int T, int x_dtype);      // the tile GEMM's decode goes that way
size_t planes_bytes(int n);
int launch_planes(const sq_matrix* mats, int n, uint16_t* out, uint16_t* planes, const void* x, int x_dtype, int64_t ldx, int T, uint16_t* xout, hipStream_t s);
// 17 to 128 activation rows of 16-bit tags of width 8, a column of the codebook at a time (sq_plane_product.hip): how many of the n pieces, the first
// one on, it takes in one launch; 0 where the other kernels are the faster way
int plane_product_group(const sq_matrix* mats, int n, int T, PlanePlan& planned, const MidPlan* mid = nullptr);      // (mid: mid_plan of all n, where it is known)
size_t plane_product_workspace(const sq_matrix* mats, int n, int T, const PlanePlan* planned = nullptr);
size_t plane_product_workspace_least(const sq_matrix* mats, int n, int T, const PlanePlan* planned);     // (up to SQ_SMALL_BMAX rows)
int launch_plane_product(const sq_matrix* mats, int n, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype, int64_t ldy, int T, void* ws, size_t ws_bytes,
                         hipStream_t s, const PlanePlan* planned = nullptr);
int launch_dequant_stack(const sq_matrix* mats, int n, void* out, int raw, const uint16_t* x, int64_t ldx, int T, int C, uint16_t* xout, hipStream_t s);
int launch_gemm_dense(const void* w, int w_dtype, int64_t ldw, int R, int C, const void* x, int x_dtype, int64_t ldx,
                      void* y, int y_dtype, int64_t ldy, int T, hipStream_t s, void* ws = nullptr, size_t ws_bytes = 0);
size_t gemm_dense_workspace(int R, int C, int T);

// d = 4 / 12-bit pieces at 1 or 2 activation rows, from the file's row-major tags (sq_segs.hip)
bool segs_shape(const sq_matrix& m);
bool segs_fits(const sq_matrix* mats, int cnt, int B, int cus);
int launch_segs_group(const sq_matrix* mats, int cnt, const void* x, int x_dtype, int64_t ldx, void* y, int y_dtype,
                      int64_t ldy, int B, int cus, hipStream_t s);

// tile-major copy of the tags for the matrix-core decode kernel (host routines, sq_gemv.hip)
bool tiled_format_ok(int R, int W, int C, int d, int bits);
int unit_dwords(int bits);
int row_units(int C, int d, int bits);             // lane units of a row, the last one perhaps not whole
bool whole_units(const sq_matrix& m);              // its rows are whole lane units, without pad bits
size_t tiled_bytes(int R, int C, int bits);
void tiled_build(const uint32_t* tags, int R, int W, int C, int bits, uint32_t* out);

// the block-32 side formats (8-bit output head, 4-bit embedding)
int launch_q8_small(const int8_t* q, const uint16_t* sc, int V, int C, const void* x, int x_dtype, int64_t ldx, void* y,
                    int y_dtype, int64_t ldy, int B, hipStream_t s);
bool q8_mid(int V, int C, int B);             // 3 .. 320 activation rows on MFMA passes of up to 64
size_t q8_mid_workspace(int V, int C, int B);
int launch_q8_mid(const int8_t* q, const uint16_t* sc, int V, int C, const void* x, int x_dtype, int64_t ldx, void* y,
                  int y_dtype, int64_t ldy, int B, void* ws, size_t ws_bytes, hipStream_t s);
size_t q8_workspace(int V, int C, int T);
int launch_q8_large(const int8_t* q, const uint16_t* sc, int V, int C, const void* x, int x_dtype, int64_t ldx, void* y,
                    int y_dtype, int64_t ldy, int T, void* ws, size_t ws_bytes, hipStream_t s);
int launch_q8_dequant(const int8_t* q, const uint16_t* sc, int C, void* out, int out_dtype, int64_t ld_out, int r0, int r1,
                      hipStream_t s);
int launch_q4_embed(const uint8_t* q, const uint16_t* sc, int V, int C, const int64_t* ids, int64_t n_ids, void* out,
                    int out_dtype, int64_t ld_out, hipStream_t s);

// elementwise neighbours of the decode-time products (sq_neighbours.hip)
int launch_addnorm(const float* h_in, float* h_out, int64_t ld_h, const void* add, int add_dtype, int64_t ld_add, const void* w,
                   int w_dtype, const int32_t* perms, int M, int B, int C, float eps, void* out, int out_dtype, hipStream_t s);
int launch_silu_mul(const void* gate, const void* up, int dtype, int64_t ld, const int32_t* perms, int M, int B, int C, void* out,
                    hipStream_t s);

}  // namespace sq
