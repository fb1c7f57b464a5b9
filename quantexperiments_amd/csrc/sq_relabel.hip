// Codewords relabelled on the GPU so that every slice of 4096 of a codebook carries the same share of a matrix' tags: counts,
// the dealing of sq_stream_build.hip's deal_codewords with the same result, and the tags and table rewritten through it.
#include <algorithm>
#include "sq_stream.h"

namespace sq {

constexpr int DEAL_NT = 1024, DEAL_WAVES = DEAL_NT / 64;
constexpr int DEAL_SLICE = 1 << STREAM_SLICE_BITS;
constexpr int DEAL_RUNS = 6144;              // run starts that LDS holds; codewords behind them are dealt one by one
constexpr int DEAL_LDS = 65536 * 2 + DEAL_WAVES * 256 * 4 + DEAL_RUNS * 2;

constexpr int RELABEL_RANGE = 32768;         // codewords a workgroup counts at a time

struct RelabelPiece {
    const uint32_t* tags;
    uint32_t* tags_out;
    const u32x4* table;                      // rows of eight fp16
    u32x4* table_out;
    const uint8_t* row_book;
    uint32_t* partial;                       // [parts, G << bits]
    uint32_t* count;                         // [G << bits]
    uint16_t* remap;                         // [G << bits]: new label within the book
    int R, W, U, bits, G;
    int parts;                               // of the rows, counted side by side
    int wg_rows, wg_book, wg_out;            // first workgroup of this piece: tags counted; codebooks dealt; tags and table rewritten
};
struct RelabelArgs {
    RelabelPiece p[RELABEL_PIECES];
    int n;
};

__device__ __forceinline__ uint32_t relabel_book(const RelabelPiece& P, int r) {
    return P.row_book ? ((uint32_t)P.row_book[r] & (uint32_t)(P.G - 1)) << P.bits : 0u;
}

// How often every codeword is named: counters in LDS, a workgroup per range of RELABEL_RANGE codewords and part of the rows, which
// writes its counts out; the sums over the parts are a second kernel.  An atomic in memory per tag (each has to pass the caches,
// and popular codewords queue at one address) took 61 us for 3584 x 448 evenly spread tags and 3.2 ms for 5120 x 640 of a power
// law; now 19 and 30 with the sums.  A thread takes 32 tags, which are whole words.
__global__ __launch_bounds__(1024) void relabel_count_kernel(RelabelArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char relabel_lds[];
    uint32_t* c = reinterpret_cast<uint32_t*>(relabel_lds);
    int pi = 0;
    while (pi + 1 < a.n && (int)blockIdx.x >= a.p[pi + 1].wg_rows) ++pi;
    const RelabelPiece& P = a.p[pi];
    const int wg = (int)blockIdx.x - P.wg_rows, part = wg % P.parts, tid = threadIdx.x;
    const uint32_t all = (uint32_t)P.G << P.bits, r0 = (uint32_t)(wg / P.parts) * RELABEL_RANGE, range = min(all - r0, (uint32_t)RELABEL_RANGE);
    for (uint32_t k = tid; k < range; k += 1024) c[k] = 0u;
    __syncthreads();
    const int units = (P.U + 31) / 32;
    const int64_t n = (int64_t)P.R * units, i1 = n * (part + 1) / P.parts;
    for (int64_t i = n * part / P.parts + tid; i < i1; i += 1024) {
        const int r = (int)(i / units), u = (int)(i - (int64_t)r * units), m = min(32, P.U - u * 32);
        const uint32_t* w = P.tags + (int64_t)r * P.W + u * P.bits;
        const uint32_t book = relabel_book(P, r);
        if (P.bits == 16 && m == 32) {
            uint32_t v[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) v[k] = w[k];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const uint32_t lo = (book | (v[k] & 0xFFFFu)) - r0, hi = (book | v[k] >> 16) - r0;
                if (lo < range) atomicAdd(&c[lo], 1u);
                if (hi < range) atomicAdd(&c[hi], 1u);
            }
        } else {
            for (int k = 0; k < m; ++k) {
                const uint32_t t = (book | tag_at(w, P.W - u * P.bits, P.bits, k)) - r0;
                if (t < range) atomicAdd(&c[t], 1u);
            }
        }
    }
    __syncthreads();
    for (uint32_t k = tid; k < range; k += 1024) P.partial[(size_t)part * all + r0 + k] = c[k];
}

__global__ __launch_bounds__(256) void relabel_sum_kernel(RelabelArgs a) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    for (int k = 0; k < a.n; ++k) {
        const size_t all = (size_t)a.p[k].G << a.p[k].bits;
        if (i >= all) continue;
        uint32_t v = 0;
        for (int p = 0; p < a.p[k].parts; ++p) v += a.p[k].partial[p * all + i];
        a.p[k].count[i] = v;
    }
}

// over the 16 lanes of a DPP row; 64 bits where a matrix has 2^28 tags or more
template <int N, typename T> __device__ __forceinline__ T ror16(T v) {
    const int lo = __builtin_amdgcn_update_dpp((int)(uint32_t)v, (int)(uint32_t)v, 0x120 + N, 0xF, 0xF, false);
    if constexpr (sizeof(T) == 4) return (T)(uint32_t)lo;
    else {
        const int hi = __builtin_amdgcn_update_dpp((int)(v >> 32), (int)(v >> 32), 0x120 + N, 0xF, 0xF, false);
        return (T)(uint32_t)hi << 32 | (uint32_t)lo;
    }
}
template <typename T> __device__ __forceinline__ T deal_min16(T v) {
    v = min(v, ror16<8>(v)); v = min(v, ror16<4>(v)); v = min(v, ror16<2>(v)); v = min(v, ror16<1>(v));
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    if constexpr (sizeof(T) == 4) return lo;
    else return (T)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 | lo;
}
// how many of the 16 values are smaller (they differ, but for ~0)
template <int N, typename T> __device__ __forceinline__ int deal_below(T v) {
    if constexpr (N == 16) return 0;
    else return (int)(ror16<N>(v) < v) + deal_below<N + 1>(v);
}

// A step of the dealing: of sorted codewords k .. k + n - 1, number j goes to the slice of rank j % nf, whose next free label is base[j % nf]
// before the step, as its j / nf-th.
struct DealStep {
    uint32_t k, n, nf, inverse;              // inverse: j / nf for j <= 65536 is the high half of j * inverse (nf > 1)
    uint16_t base[16];
};
constexpr int DEAL_STEPS = 256, DEAL_LONG = 4096;
static_assert(DEAL_STEPS * sizeof(DealStep) <= DEAL_WAVES * 256 * 4, "the steps lie where the digits were counted");

// One workgroup per codebook.  Codewords go, most used first (equal counts by id), to the slice with the fewest tags so far that
// has room (ties: the lowest).  What bounds it is that this is a chain of 65,536 choices, 4 ms at 150 clocks each.  But of
// codewords of equal count c the slices whose loads lie less than c above the least take one each, in order of load, before any
// gets a second one or a slice that is further behind gets one; so a step deals a round to those slices, or as many rounds as
// leave that so.  One wave works the steps out, up to DEAL_STEPS ahead (its chain is instructions: with all sixteen doing the same beside
// it a step took twice as long), then all write the codewords' labels.  The codewords are sorted by count with a stable radix sort, 8 bits
// a pass, ids in LDS and between two passes in registers (a wave owns a 16th of them); counts below 256, the usual ones, are one pass of
// as many bits as they have, read from the counts in order, and its digits' places are where the runs of equal counts start.
// 65,536 codewords: 3584 x 448 evenly spread tags 95 to 102 us (sorting 40, 73 steps 42, labels 19), 190 with the sort in general passes, the runs' starts
// searched in the sorted counts and every wave at the steps; 1057 x 64 58, 130; 5120 x 640 of a power law 0.89 ms (a load of that matrix 2.62 ms, 3.23).
// On the host, with the copies and the synchronisation around it, 480 us of a load for every matrix of a stack.
template <int PER, typename T>               // ids per lane: K / DEAL_NT (0: codebooks of one slice); a slice's tags (less than 2^(bits - 4))
__global__ __launch_bounds__(DEAL_NT) void deal_kernel(RelabelArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char deal_lds[];
    int pi = 0;
    while (pi + 1 < a.n && (int)blockIdx.x >= a.p[pi + 1].wg_book) ++pi;
    const RelabelPiece& P = a.p[pi];
    const int K = 1 << P.bits, NS = K >> STREAM_SLICE_BITS, tid = threadIdx.x, lane = tid & 63, sl = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t* count = P.count + ((size_t)((int)blockIdx.x - P.wg_book) << P.bits);
    uint16_t* remap = P.remap + ((size_t)((int)blockIdx.x - P.wg_book) << P.bits);
    if constexpr (PER == 0) {                // a codebook of one slice keeps its labels
        for (int k = tid; k < K; k += DEAL_NT) remap[k] = (uint16_t)k;
    } else {
    uint16_t* ids = reinterpret_cast<uint16_t*>(deal_lds);                  // [65536]
    uint32_t* ctr = reinterpret_cast<uint32_t*>(deal_lds + 65536 * 2);      // [wave][digit]
    uint16_t* starts = reinterpret_cast<uint16_t*>(ctr + DEAL_WAVES * 256);
    __shared__ uint32_t shared_most, wave_sum4[4], wave_starts[DEAL_WAVES];
    __shared__ int shared_steps, shared_long;

    const int w0 = wave * (K / DEAL_WAVES);                                 // the wave's first id
    uint32_t most = 0;
#pragma unroll 8
    for (int i = 0; i < PER; ++i) most = max(most, count[w0 + i * 64 + lane]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, o, 64));
    if (tid == 0) shared_most = 0u;
    __syncthreads();
    if (lane == 0) atomicMax(&shared_most, most);
    __syncthreads();
    most = (uint32_t)__builtin_amdgcn_readfirstlane((int)shared_most);
    const bool single = most < 256;
    const int nb = single ? max(1, 32 - __builtin_clz(most | 1u)) : 8;       // bits of a digit; the largest comes first
    const uint32_t top = (1u << nb) - 1u;
    int runs = 0;
    auto clear = [&]() {
        for (int k = tid; k < DEAL_WAVES * 256; k += DEAL_NT) ctr[k] = 0u;
        __syncthreads();
    };
    auto tally = [&](uint32_t dg) {          // (a wave all of whose digits are the same, as the high ones mostly are, would queue at one counter)
        if (__all((int)dg == __builtin_amdgcn_readfirstlane((int)dg))) { if (lane == 0) atomicAdd(&ctr[wave * 256 + dg], 64u); }
        else atomicAdd(&ctr[wave * 256 + dg], 1u);
    };
    // exclusive sums over (digit, wave): thread d < 256 takes the 16 waves of digit d.  The digits in use are the runs of a single pass.
    auto sums = [&]() {
        __syncthreads();
        uint32_t mine = 0, before = 0;
        uint64_t used = 0;
        if (tid < 256) {
            for (int w = 0; w < DEAL_WAVES; ++w) mine += ctr[w * 256 + tid];
            before = mine;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t v = __shfl_up(before, o, 64);
                if (lane >= o) before += v;
            }
            used = __ballot(mine > 0);
            if (lane == 63) {
                wave_sum4[wave] = before;
                wave_starts[wave] = (uint32_t)__popcll(used);
            }
        }
        __syncthreads();
        runs = (int)(wave_starts[0] + wave_starts[1] + wave_starts[2] + wave_starts[3]);
        if (tid < 256) {
            uint32_t at = before - mine, run = (uint32_t)__popcll(used & (((uint64_t)1 << lane) - 1));
            for (int w = 0; w < wave; ++w) {
                at += wave_sum4[w];
                run += wave_starts[w];
            }
            if (mine > 0) starts[run] = (uint16_t)at;
            for (int w = 0; w < DEAL_WAVES; ++w) {
                const uint32_t n = ctr[w * 256 + tid];
                ctr[w * 256 + tid] = at;
                at += n;
            }
        }
        __syncthreads();
    };
    auto place = [&](uint32_t dg, uint32_t id, int bits) {
        uint32_t lo = ~0u, hi = ~0u;                                        // the lanes whose digit is the same
#pragma unroll
        for (int b = 0; b < bits; ++b) {
            const uint32_t mask = (uint32_t)-(int)((dg >> b) & 1);
            const uint64_t set = __ballot(mask != 0);
            lo &= ~((uint32_t)set ^ mask);
            hi &= ~((uint32_t)(set >> 32) ^ mask);
        }
        const uint64_t same = (uint64_t)hi << 32 | lo;
        const int rank = __popcll(same & (((uint64_t)1 << lane) - 1));
        volatile uint32_t* c = &ctr[wave * 256 + dg];                // (this wave's counter: its LDS accesses stay in order)
        const uint32_t at = *c;
        ids[at + rank] = (uint16_t)id;
        if (rank == 0) *c = at + (uint32_t)__popcll(same);
        __threadfence_block();
    };
    if (single) {
        clear();
        // (few digits: 2^copies counters of each, its lanes dealt among them, or they would queue: 4 bits 24 us, now 7)
        const int copies = nb <= 6 ? 8 - nb : 0;
        uint32_t* mine = ctr + wave * 256;
#pragma unroll 8
        for (int i = 0; i < PER; ++i) atomicAdd(&mine[(top - count[w0 + i * 64 + lane]) << copies | (uint32_t)(lane & ((1 << copies) - 1))], 1u);
        if (copies) {
            const u32x4 four = *reinterpret_cast<const u32x4*>(mine + lane * 4);
            uint32_t of = four.x + four.y + four.z + four.w;
            for (int o = 1; o < 1 << (copies - 2); o <<= 1) of += (uint32_t)__shfl_xor((int)of, o, 64);
            __threadfence_block();           // (a wave's own counters: its LDS accesses stay in order)
            *reinterpret_cast<u32x4*>(mine + lane * 4) = u32x4{0u, 0u, 0u, 0u};
            __threadfence_block();
            if ((lane & ((1 << (copies - 2)) - 1)) == 0) mine[lane >> (copies - 2)] = of;
        }
        sums();
        for (int i0 = 0; i0 < PER; i0 += 8) {
            uint32_t c8[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) c8[i] = count[w0 + (i0 + i) * 64 + lane];
#pragma unroll
            for (int i = 0; i < 8; ++i) place(top - c8[i], (uint32_t)(w0 + (i0 + i) * 64 + lane), nb);
        }
        __syncthreads();
    } else {
#pragma unroll 8
        for (int i = 0; i < PER; ++i) ids[w0 + i * 64 + lane] = (uint16_t)(w0 + i * 64 + lane);
    }
    for (int shift = 0; !single && shift < 32 && (most >> shift) != 0; shift += 8) {
        clear();
        uint32_t held[PER / 2];                                             // ids in pairs
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if (i % 8 == 0) __builtin_amdgcn_sched_barrier(0);              // (as many loads at a time as there are registers for)
            const uint32_t id = ids[w0 + i * 64 + lane];
            held[i / 2] = i % 2 ? held[i / 2] | id << 16 : id;
            tally(top - ((count[id] >> shift) & 255u));
        }
#pragma unroll
        for (int i = 0; i < PER / 2; ++i) asm volatile("" : "+v"(held[i]));  // (kept packed: unpacked ahead of their use they spill)
        sums();
#pragma unroll
        for (int i = 0; i < PER; i += 8) {
            __builtin_amdgcn_sched_barrier(0);
            uint32_t c8[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) c8[j] = count[(held[(i + j) / 2] >> (16 * (j % 2))) & 0xFFFFu];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                __builtin_amdgcn_sched_barrier(0);
                place(top - ((c8[j] >> shift) & 255u), held[(i + j) / 2] >> (16 * (j % 2)), 8);
            }
        }
        __syncthreads();
    }

    if (!single) {                           // where runs of equal counts start, in order
        int found = 0;
        uint64_t firsts = 0;                                                // bit i: this lane's id i starts one
#pragma unroll 8
        for (int i = 0; i < PER; ++i) {
            const int k = w0 + i * 64 + lane;
            const bool first = k == 0 || count[ids[k]] != count[ids[k - 1]];
            firsts |= (uint64_t)first << i;
            found += __popcll(__ballot(first));
        }
        if (lane == 0) wave_starts[wave] = (uint32_t)found;
        __syncthreads();
        int at = 0;
        runs = 0;
        for (int w = 0; w < DEAL_WAVES; ++w) {
            if (w < wave) at += (int)wave_starts[w];
            runs += (int)wave_starts[w];
        }
#pragma unroll 8
        for (int i = 0; i < PER; ++i) {
            const bool first = firsts >> i & 1;
            const uint64_t all = __ballot(first);
            const int o = at + __popcll(all & (((uint64_t)1 << lane) - 1));
            if (first && o < DEAL_RUNS) starts[o] = (uint16_t)(w0 + i * 64 + lane);
            at += __popcll(all);
        }
        __syncthreads();
    }

    DealStep* steps = reinterpret_cast<DealStep*>(ctr);
    // wave 0: tags and codewords of slice sl; 64 runs at a time, one a lane (behind DEAL_RUNS of them 64 codewords), and what is left of the run it deals
    const int listed = min(runs, DEAL_RUNS);
    T load = 0, c = 0;
    int fill = 0, next_run = 0, next_lone = listed < runs ? starts[listed - 1] + 1 : K, have = 0, at = 0, lane_k = 0, lane_m = 0, k = 0, m = 0;
    uint32_t lane_c = 0, lane_r = 0, recip = 0;
    const uint32_t lane_inverse = lane > 1 ? 0xFFFFFFFFu / (uint32_t)lane + 1u : 0u;       // (of nf = 2 .. 16, divisions out of the chain)
    bool more = true;
    while (more) {
        if (wave == 0) {
            int ns = 0, first_long = DEAL_STEPS;
            while (ns < DEAL_STEPS) {
                if (m == 0) {
                    if (at == have) {
                        if (next_run < listed) {
                            const int r = min(next_run + lane, listed - 1);
                            lane_k = starts[r];
                            lane_m = (r + 1 < listed ? starts[r + 1] : listed == runs ? K : lane_k + 1) - lane_k;
                            have = min(64, listed - next_run);
                            next_run += have;
                        } else if (next_lone < K) {
                            lane_k = min(next_lone + lane, K - 1);
                            lane_m = 1;
                            have = min(64, K - next_lone);
                            next_lone += have;
                        } else {
                            break;
                        }
                        lane_c = count[ids[lane_k]];
                        lane_r = lane_c ? 0xFFFFFFFFu / lane_c : 0u;
                        at = 0;
                    }
                    k = __builtin_amdgcn_readlane(lane_k, at);
                    m = __builtin_amdgcn_readlane(lane_m, at);
                    c = (T)(uint32_t)__builtin_amdgcn_readlane((int)lane_c, at);
                    recip = (uint32_t)__builtin_amdgcn_readlane((int)lane_r, at);
                    ++at;
                }
                const bool open = sl < NS && fill < DEAL_SLICE;
                const T none = ~(T)0, key = open ? load << 4 | (T)sl : none, least = deal_min16(key), lo = least >> 4;
                // the slices that are next (c = 0: the least loaded one until it is full) and their order
                const bool next = open && (c ? load - lo < c : key == least);
                const int nf = __popcll(__ballot(next) & 0xFFFF), rank = deal_below<1>(key);
                const int room = (int)deal_min16((uint32_t)(next ? DEAL_SLICE - fill : DEAL_SLICE));
                const uint32_t inverse = (uint32_t)__builtin_amdgcn_readlane((int)lane_inverse, nf);
                const int rounds = nf == 1 ? m : (int)__umulhi((uint32_t)m, inverse);
                // whole rounds: until the codewords or the room end, or the least loaded of them passes one that was behind
                int q = min(rounds, room), last = room;
                const T above = deal_min16(open && !next ? load : none);
                if (c && above != none && above - lo < (uint64_t)c * (uint64_t)(q + 1)) {
                    uint32_t of;                                             // (above - lo) / c
                    if constexpr (sizeof(T) == 4) {                          // (the product is one too small at most, or none)
                        of = __umulhi((uint32_t)(above - lo), recip);
                        of += (above - lo) - of * (uint32_t)c >= (uint32_t)c;
                    } else {
                        of = (uint32_t)((above - lo) / c);
                    }
                    last = min(room, (int)of);
                }
                q = min(q, last);
                const int rem = q == rounds && q < last ? m - q * nf : 0, n = q * nf + rem;
                if (n > DEAL_LONG) first_long = min(first_long, ns);
                DealStep& st = steps[ns++];
                if (lane == 0) { st.k = (uint32_t)k; st.n = (uint32_t)n; st.nf = (uint32_t)nf; st.inverse = inverse; }
                if (lane < 16 && next) st.base[rank] = (uint16_t)(sl * DEAL_SLICE + fill);
                const int got = next ? q + (rank < rem) : 0;
                load += c * (T)got;
                fill += got;
                k += n;
                m -= n;
            }
            if (lane == 0) { shared_steps = ns; shared_long = first_long; }
        }
        __syncthreads();
        const int ns = shared_steps;
        more = ns == DEAL_STEPS;
        auto write = [&](int i, int j0, int stride) {
            const int n = (int)steps[i].n, nf = (int)steps[i].nf, first = (int)steps[i].k;
            const uint32_t inverse = steps[i].inverse;
            const int base = steps[i].base[sl];
#pragma unroll 4
            for (; j0 < n; j0 += stride) {
                const int j = min(j0 + lane, n - 1), round = nf == 1 ? j : (int)__umulhi((uint32_t)j, inverse), label = __shfl(base, j - round * nf, 64) + round;
                remap[ids[first + j]] = (uint16_t)label;
            }
        };
        for (int i = wave; i < ns; i += DEAL_WAVES)                          // a wave a step, but of long ones every wave each 16th group of 64 codewords
            if (steps[i].n <= DEAL_LONG) write(i, 0, 64);
        for (int i = shared_long; i < ns; ++i)
            if (steps[i].n > DEAL_LONG) write(i, wave * 64, DEAL_NT);
        __syncthreads();
    }
    }
}

// tags_out = tags through remap, a thread per 32 tags (which are whole words), the table's rows moved to their new labels.  What
// lies behind a row's last tag stays: the rest of its word as zeros, whole words as they are.
__global__ __launch_bounds__(256) void relabel_write_kernel(RelabelArgs a) {
    int pi = 0;
    while (pi + 1 < a.n && (int)blockIdx.x >= a.p[pi + 1].wg_out) ++pi;
    const RelabelPiece& P = a.p[pi];
    const int64_t i = (int64_t)((int)blockIdx.x - P.wg_out) * 256 + threadIdx.x;
    const int bits = P.bits, units = (P.U + 31) / 32;
    if (i < (int64_t)P.G << bits) P.table_out[(i >> bits << bits) + P.remap[i]] = P.table[i];
    if (i >= (int64_t)P.R * units) return;
    const int r = (int)(i / units), u = (int)(i - (int64_t)r * units);
    const uint32_t* w = P.tags + (int64_t)r * P.W + u * bits;
    uint32_t* o = P.tags_out + (int64_t)r * P.W + u * bits;
    const int nw = u + 1 < units ? bits : P.W - u * bits, n = min(32, P.U - u * 32);
    const uint16_t* map = P.remap + relabel_book(P, r);
    const uint32_t mask = (1u << bits) - 1u;
    uint64_t in = 0, out = 0;
    int have = 0, held = 0, rd = 0, wr = 0;
    for (int k = 0; k < n; ++k) {
        if (have < bits) { in |= (uint64_t)(rd < nw ? w[rd] : 0u) << have; ++rd; have += 32; }
        out |= (uint64_t)map[(uint32_t)in & mask] << held;
        in >>= bits; have -= bits; held += bits;
        if (held >= 32) { o[wr++] = (uint32_t)out; out >>= 32; held -= 32; }
    }
    if (held > 0) o[wr++] = (uint32_t)out;
    for (; wr < nw; ++wr) o[wr] = w[wr];
}

static int relabel_parts(const sq_matrix& m) {
    return (int)std::max<int64_t>(1, std::min<int64_t>(64, (int64_t)m.R * (m.C / m.d) >> 16));
}
static size_t relabel_bytes(const sq_matrix& m) { return ((((size_t)m.G << m.bits) * (4 * (size_t)relabel_parts(m) + 6)) + 255) & ~(size_t)255; }

size_t relabel_scratch_bytes(const sq_matrix* mats, int n) {
    size_t b = 0;
    for (int i = 0; i < n; ++i) b += relabel_bytes(mats[i]);
    return b;
}

static void raise_lds_limits() {
    static bool raised = false;
    if (!raised) {
        for (const void* f : {(const void*)deal_kernel<8, uint32_t>, (const void*)deal_kernel<8, uint64_t>, (const void*)deal_kernel<16, uint32_t>, (const void*)deal_kernel<16, uint64_t>, (const void*)deal_kernel<32, uint32_t>, (const void*)deal_kernel<32, uint64_t>, (const void*)deal_kernel<64, uint32_t>, (const void*)deal_kernel<64, uint64_t>})
            (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, DEAL_LDS);
        (void)hipFuncSetAttribute((const void*)relabel_count_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, RELABEL_RANGE * 4);
        (void)hipGetLastError();
        raised = true;
    }
}

template <typename T>
static void launch_deal(const RelabelArgs& a, int bits, int books, hipStream_t s) {
    const dim3 grid((unsigned)books), block(DEAL_NT);
    switch (bits) {
        case 16: hipLaunchKernelGGL((deal_kernel<64, T>), grid, block, DEAL_LDS, s, a); break;
        case 15: hipLaunchKernelGGL((deal_kernel<32, T>), grid, block, DEAL_LDS, s, a); break;
        case 14: hipLaunchKernelGGL((deal_kernel<16, T>), grid, block, DEAL_LDS, s, a); break;
        case 13: hipLaunchKernelGGL((deal_kernel<8, T>), grid, block, DEAL_LDS, s, a); break;
        default: hipLaunchKernelGGL((deal_kernel<0, T>), grid, block, 0, s, a);
    }
}

// d = 8 matrices that stream_format_ok takes; tags_out / table_out: buffers of the same size as tags / table.  Neighbours with
// tags of one width share a launch.
int launch_relabel(const sq_matrix* mats, int n, void* const* tags_out, void* const* table_out, void* scratch, hipStream_t s) {
    raise_lds_limits();
    char* next = (char*)scratch;
    for (int i0 = 0; i0 < n;) {
        RelabelArgs a{};
        int64_t counted = 0, books = 0, out = 0, most = 0, tags = 0;
        for (; a.n < RELABEL_PIECES && i0 + a.n < n && mats[i0 + a.n].bits == mats[i0].bits; ++a.n) {
            const sq_matrix& m = mats[i0 + a.n];
            RelabelPiece& P = a.p[a.n];
            const int64_t codewords = (int64_t)m.G << m.bits;
            P.tags = (const uint32_t*)m.tags; P.tags_out = (uint32_t*)tags_out[i0 + a.n];
            P.table = (const u32x4*)m.table; P.table_out = (u32x4*)table_out[i0 + a.n];
            P.row_book = m.G > 1 ? m.row_book : nullptr;
            P.parts = relabel_parts(m);
            P.partial = (uint32_t*)next; P.count = P.partial + codewords * P.parts; P.remap = (uint16_t*)(P.count + codewords);
            next += relabel_bytes(m);
            P.R = m.R; P.W = m.W; P.U = m.C / m.d; P.bits = m.bits; P.G = m.G;
            P.wg_rows = (int)counted; P.wg_book = (int)books; P.wg_out = (int)out;
            counted += (codewords + RELABEL_RANGE - 1) / RELABEL_RANGE * P.parts;
            books += m.G;
            tags = std::max(tags, (int64_t)m.R * P.U);
            out += (std::max((int64_t)m.R * ((P.U + 31) / 32), codewords) + 255) / 256;
            most = std::max(most, codewords);
        }
        if (out >= ((int64_t)1 << 31)) return fail(SQ_EUNSUPPORTED, "sq_codebook_rebalance_device: matrix too large");
        const size_t lds = (size_t)std::min<int64_t>(most, RELABEL_RANGE) * 4;
        hipLaunchKernelGGL(relabel_count_kernel, dim3((unsigned)counted), dim3(1024), lds, s, a);
        hipLaunchKernelGGL(relabel_sum_kernel, dim3((unsigned)((most + 255) / 256)), dim3(256), 0, s, a);
        if (tags < (int64_t)1 << 28) launch_deal<uint32_t>(a, mats[i0].bits, (int)books, s);
        else launch_deal<uint64_t>(a, mats[i0].bits, (int)books, s);
        hipLaunchKernelGGL(relabel_write_kernel, dim3((unsigned)out), dim3(256), 0, s, a);
        if (const int rc = check_launch("sq_codebook_rebalance_device")) return rc;
        i0 += a.n;
    }
    return SQ_OK;
}

}  // namespace sq
