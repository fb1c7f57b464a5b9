// Load-time builder of the bucketed tag stream (layout: sq_stream.hip and sq_stream.h), on the host and on the GPU.
#include <algorithm>
#include <atomic>
#include <memory>
#include <new>
#include <string.h>
#include <thread>
#include <vector>
#include "sq_stream.h"

constexpr int STREAM_CLIMB = 1;      // hill-climbing passes of the entry ordering (load time against LDS collisions)

namespace sq {

// A run: groups g0 .. g0 + ng - 1 of every bucket.  Its rows belong to `norders` column orders (one without row orders);
// the groups of order[i] begin at group bound[i] of the run (bound[0] = 0), and the kernel keeps copy i of x, gathered
// through that order, in LDS for them.
// u0: the index of the run's first unit (units are counted run after run).
struct StreamRun { int32_t g0, ng, norders, u0; uint8_t bound[STREAM_RUN_ORDERS]; uint8_t order[STREAM_RUN_ORDERS]; };
static_assert(sizeof(StreamRun) == 32, "run records are read as 8 dwords");

StreamGeom stream_geom(int C, int d, int bits, int groups, int runs, bool balanced, int fs) {
    StreamGeom g;
    g.U = C / d;
    g.NS = 1 << (bits - STREAM_SLICE_BITS);
    g.KP = (g.U + STREAM_PART_MAX - 1) / STREAM_PART_MAX;
    g.PC = (g.U + g.KP - 1) / g.KP;
    g.NV = g.NS * g.KP;
    g.NG = groups;
    g.runs = runs;
    g.fmt = stream_fmt(g.PC);
    g.fs = fs < 1 ? g.fmt.pf : fs < g.fmt.pf ? fs : g.fmt.pf;
    g.off_slots = ((size_t)g.NV * g.NG * 16 + 255) & ~(size_t)255;          // four words per (bucket, group)
    g.off_runs = (g.off_slots + (size_t)g.NV * g.NG * 64 * 2 + 255) & ~(size_t)255;
    g.off_rows = (g.off_runs + (size_t)runs * sizeof(StreamRun) + 255) & ~(size_t)255;
    size_t end = (g.off_rows + (size_t)g.NG * 64 * 4 + 255) & ~(size_t)255;
    g.off_table = g.off_unmap = 0;
    if (balanced) {
        g.off_table = end;
        g.off_unmap = end + ((size_t)d * 2 << bits);
        end = (g.off_unmap + ((size_t)2 << bits) + 255) & ~(size_t)255;
    }
    g.off_steps = end;
    g.total_steps = 0;
    return g;
}

// (R + 64 * 256 bounds the places: every column order can leave one group short)
bool stream_format_ok(int R, int C, int d, int bits, int G) {
    if (G < 1 || (G & (G - 1)) != 0 || bits < 1 || bits > 16) return false;
    const int lb = stream_label_bits(bits, G);
    return d == 8 && lb > STREAM_SLICE_BITS && (1 << (lb - STREAM_SLICE_BITS)) <= (G > 1 ? STREAM_SLICES_MAX : 16) && C % d == 0 &&
           R > 0 && R + 64 * 256 < (int)STREAM_NO_ROW;
}

static inline uint32_t host_tag(const uint32_t* row, int W, int bits, int j) {
    const int64_t p = (int64_t)j * bits;
    const int w = (int)(p >> 5), s = (int)(p & 31);
    uint64_t v = row[w];
    if (s + bits > 32 && w + 1 < W) v |= (uint64_t)row[w + 1] << 32;
    return (uint32_t)(v >> s) & ((1u << bits) - 1u);
}

// fn(a, b) over blocks of `grain` of the indices 0 .. n - 1, on up to 16 threads that take the next block as they get to
// it.  `grain` is what makes a block worth a thread: one group's entry ordering takes milliseconds (with a fixed minimum of
// 64 indices per thread the 896 groups of a 3584-row matrix ran on one).
static void parallel_blocks(int n, int grain, const std::function<void(int, int)>& fn) {
    const int blocks = (n + grain - 1) / grain;
    const int nt = std::min({(int)std::max(1u, std::thread::hardware_concurrency()), 16, blocks});
    if (nt <= 1) { if (n > 0) fn(0, n); return; }
    std::atomic<int> next{0};
    auto work = [&]() {
        for (int k; (k = next.fetch_add(1, std::memory_order_relaxed)) < blocks;) fn(k * grain, std::min(n, (k + 1) * grain));
    };
    std::vector<std::thread> th;
    for (int t = 1; t < nt; ++t) th.emplace_back(work);
    work();
    for (auto& t : th) t.join();
}

struct StreamPlan {
    StreamGeom g;
    int GR;                          // groups in the longest run
    int orders_max;                  // most column orders in one run
    std::vector<StreamRun> runs;
    std::vector<uint32_t> base;      // [NG * 64]: rows ordered by column order, STREAM_NO_ROW where a group is short
    std::vector<uint16_t> cnt;       // [NV][R]
    std::vector<uint32_t> pos;       // [NV][R]: lane position (group * 64 + lane) of row r in bucket v
    std::vector<uint32_t> goff;      // [NV * NG + 1]: the groups' steps counted bucket after bucket, group after group (how the
                                     // builder lays them out before they move to their places)
    uint64_t logical_steps;          // goff[NV * NG]
    int NU;                          // units of one bucket
    std::vector<uint32_t> slot32;    // [NV * NG * 64]: place | count << STREAM_ROW_BITS per lane (STREAM_NO_ROW: no row), the
                                     // builder's own form of the slots
    std::vector<uint32_t> run_of;    // [NG]: the run of a group
    std::vector<uint32_t> head4;     // [NV * NG][4]: {rest, nst, unit0, split}, what the buffer holds per (bucket, group)
    std::vector<uint16_t> remap;     // balanced streams: file id -> new id (empty: identity)
};

// Relabelling of the codewords for a stream with a codebook of its own: the codewords are dealt, most used first, to
// whichever slice of 4096 carries the fewest tags so far and still has room, so every slice ends up with the same
// share of the tags (a slice is one workgroup's work) whatever the distribution of the tags is, and a slice's popular
// codewords get consecutive places, i.e. different LDS bank groups.
// With several codebooks (row_book names a row's) every codebook is relabelled by itself, over its own slices:
// remap[book << bits | label] is the new label within the book; a codebook of at most one slice keeps its labels.
// count[book << bits | label]: how many tags name each codeword.
static void deal_codewords(const uint32_t* count, int bits, std::vector<uint16_t>& remap, int G) {
    const int K = 1 << bits, NS = K >> STREAM_SLICE_BITS, SL = 1 << STREAM_SLICE_BITS;
    remap.assign((size_t)G * K, 0);
    if (NS < 2) {
        for (size_t k = 0; k < remap.size(); ++k) remap[k] = (uint16_t)(k & (size_t)(K - 1));
        return;
    }
    std::vector<uint32_t> ids(K), first;
    std::vector<uint64_t> load(NS);
    std::vector<int> fill(NS);
    for (int b = 0; b < G; ++b) {
        const uint32_t* cb = count + (size_t)b * K;
        // ids by count, most used first, equal counts by id: a counting sort (counts are small when the tags spread)
        const uint32_t most = *std::max_element(cb, cb + K);
        if (most < (1u << 20)) {
            first.assign((size_t)most + 2, 0);
            for (int k = 0; k < K; ++k) ++first[most - cb[k] + 1];
            for (size_t c = 1; c < first.size(); ++c) first[c] += first[c - 1];
            for (int k = 0; k < K; ++k) ids[first[most - cb[k]]++] = (uint32_t)k;
        } else {
            for (int k = 0; k < K; ++k) ids[k] = (uint32_t)k;
            std::stable_sort(ids.begin(), ids.end(), [cb](uint32_t x, uint32_t y) { return cb[x] > cb[y]; });
        }
        std::fill(load.begin(), load.end(), 0);
        std::fill(fill.begin(), fill.end(), 0);
        for (int k = 0; k < K; ++k) {
            int best = -1;
            for (int sl = 0; sl < NS; ++sl)
                if (fill[sl] < SL && (best < 0 || load[sl] < load[best])) best = sl;
            remap[(size_t)b * K + ids[k]] = (uint16_t)(best * SL + fill[best]);
            ++fill[best];
            load[best] += cb[ids[k]];
        }
    }
}

static void balance_codewords(const uint32_t* tags, int R, int W, int U, int bits, std::vector<uint16_t>& remap, int G = 1,
                              const uint8_t* row_book = nullptr) {
    std::vector<uint32_t> count((size_t)G << bits, 0);
    if ((1 << bits) >> STREAM_SLICE_BITS >= 2)
        for (int r = 0; r < R; ++r) {
            const uint32_t* row = tags + (size_t)r * W;
            uint32_t* cb = count.data() + ((size_t)(row_book ? row_book[r] & (G - 1) : 0) << bits);
            for (int j = 0; j < U; ++j) ++cb[host_tag(row, W, bits, j)];
        }
    deal_codewords(count.data(), bits, remap, G);
}

// Three steps: the rows' order, groups and runs; how many entries every row has in every bucket; and from those counts the
// lanes' places, the groups' lengths and where their steps go.  The counts come from the host's or the device's tags.
static void plan_rows(int R, int C, int d, int lbits, const uint8_t* row_mask, int runs, StreamPlan& P, bool balanced) {
    // rows by column order, groups and runs
    std::vector<uint32_t> order(R);
    for (int r = 0; r < R; ++r) order[r] = (uint32_t)r;
    if (row_mask)
        std::stable_sort(order.begin(), order.end(), [row_mask](uint32_t a, uint32_t b) { return row_mask[a] < row_mask[b]; });
    StreamGeom g0 = stream_geom(C, d, lbits, 0, 0);
    if (runs <= 0) runs = (STREAM_DEFAULT_WGS + g0.NV / 2) / g0.NV;
    if (runs < 1) runs = 1;
    // Groups per column order.  A run takes the groups of one order, GR at a time, or, when orders are small, the whole
    // groups of up to `cap` orders that follow each other (a masked k projection has 64 rows per order: one run per order
    // would be 16 workgroups of one group each per bucket).  cap: as many gathered copies of x as fit LDS beside the slice
    // and the run's partial sums, and as the staging loop covers with four chunks per thread.
    std::vector<int> first, ngm;
    for (int a = 0; a < R;) {
        int b = a;
        const int m = row_mask ? row_mask[order[a]] : 0;
        while (b < R && (row_mask ? row_mask[order[b]] : 0) == m) ++b;
        first.push_back(a);
        ngm.push_back((b - a + 63) / 64);
        a = b;
    }
    first.push_back(R);
    int total_groups = 0;
    for (int q : ngm) total_groups += q;
    const int xs_bytes = g0.fmt.narrow ? 8192 : (g0.PC + 16) * 16;     // (stream_xs)
    int cap = (160 * 1024 - 65536 - STREAM_RUN_MAX * 256 - 1024) / xs_bytes;
    cap = std::min(cap, std::min(4, 4096 / g0.PC));            // (4: two activation rows per pass still fit LDS at C = 5120)
    if (cap < 1 || !row_mask) cap = 1;
    // the runs for a run length GR (into `out` if given): returns their number
    auto pack = [&](int GR, std::vector<StreamRun>* out, int* longest) {
        int64_t n = 0;
        StreamRun cur{0, 0, 0, 0, {0}, {0}};
        int gbase = 0, lg = 1;
        auto flush = [&]() {
            if (cur.ng > 0) { ++n; lg = std::max(lg, cur.ng); if (out) out->push_back(cur); }
            cur = StreamRun{0, 0, 0, 0, {0}, {0}};
        };
        for (size_t i = 0; i < ngm.size(); ++i) {
            const int q = ngm[i], m = row_mask ? row_mask[order[first[i]]] : 0;
            if (q > GR) {                                        // an order longer than a run: runs of its own
                flush();
                for (int p0 = 0; p0 < q; p0 += GR) {
                    cur = StreamRun{gbase + p0, std::min(GR, q - p0), 1, 0, {0}, {(uint8_t)m}};
                    flush();
                }
            } else if (cur.ng > 0 && cur.ng + q <= GR && cur.norders < cap) {
                cur.bound[cur.norders] = (uint8_t)cur.ng;
                cur.order[cur.norders] = (uint8_t)m;
                ++cur.norders;
                cur.ng += q;
            } else {
                flush();
                cur = StreamRun{gbase, q, 1, 0, {0}, {(uint8_t)m}};
            }
            gbase += q;
        }
        flush();
        if (longest) *longest = lg;
        return n;
    };
    // GR = the fewest groups per run that keep the run count within the request.  A run's partial sums are staged in
    // LDS: no run longer than STREAM_RUN_MAX groups (more runs than asked for then).
    int GR = 1;
    while (GR < STREAM_RUN_MAX && GR < total_groups && pack(GR, nullptr, nullptr) > runs) ++GR;
    // With one column order the kernel derives the cut from the run count alone, as ceil(groups / runs) per run: settle
    // on a run length that this formula gives back.
    if (ngm.size() == 1)
        for (;;) {
            const int n = (ngm[0] + GR - 1) / GR, g2 = (ngm[0] + n - 1) / n;
            if (g2 == GR) break;
            GR = g2;
        }
    P.runs.clear();
    P.base.clear();
    pack(GR, &P.runs, &P.GR);
    P.orders_max = 1;
    for (const StreamRun& run : P.runs) P.orders_max = std::max(P.orders_max, (int)run.norders);
    for (size_t i = 0; i < ngm.size(); ++i) {
        const int a = first[i], b = first[i + 1];
        for (int k = 0; k < ngm[i] * 64; ++k) P.base.push_back(a + k < b ? order[a + k] : STREAM_NO_ROW);
    }
    P.g = stream_geom(C, d, lbits, (int)(P.base.size() / 64), (int)P.runs.size(), balanced);
}

static void plan_counts(const uint32_t* tags, int R, int W, int bits, const uint16_t* remap, int G, const uint8_t* row_book, StreamPlan& P) {
    const StreamGeom& g = P.g;
    P.cnt.assign((size_t)g.NV * R, 0);
    parallel_blocks(R, 64, [&](int a, int b) {
        for (int r = a; r < b; ++r) {
            const uint32_t* row = tags + (size_t)r * W;
            const uint32_t book = row_book ? (uint32_t)(row_book[r] & (G - 1)) << bits : 0u;
            for (int j = 0; j < g.U; ++j) {
                uint32_t t = host_tag(row, W, bits, j);
                if (remap) t = remap[t];
                t |= book;
                const int v = (j / g.PC) * g.NS + (int)(t >> STREAM_SLICE_BITS);
                ++P.cnt[(size_t)v * R + r];
            }
        }
    });
}

// From the groups' step counts ([NV * NG]): their offsets, units and places.
static void plan_layout(const uint32_t* steps, StreamPlan& P) {
    const StreamGeom& g = P.g;
    const size_t nvg = (size_t)g.NV * g.NG;
    P.goff.assign(nvg + 1, 0);
    uint64_t tot = 0;
    for (size_t k = 0; k < nvg; ++k) { P.goff[k] = (uint32_t)tot; tot += steps[k]; }
    P.goff[nvg] = (uint32_t)tot;
    P.logical_steps = tot;
    // Units and places: the first-steps region (NU units x NV buckets x FS steps) comes first, the groups'
    // remaining steps follow bucket after bucket, group after group.
    P.NU = 0;
    P.run_of.assign(g.NG, 0);
    for (size_t ri = 0; ri < P.runs.size(); ++ri) {
        StreamRun& run = P.runs[ri];
        run.u0 = P.NU;
        P.NU += run.ng * stream_split_of(run.ng);
        for (int k = 0; k < run.ng; ++k) P.run_of[run.g0 + k] = (uint32_t)ri;
    }
    // FS: the longest unit's step count, at most the prefetch depth
    const uint32_t PF = (uint32_t)g.fmt.pf;
    uint32_t fs = 1;
    for (int v = 0; v < g.NV; ++v)
        for (int gi = 0; gi < g.NG; ++gi) {
            const uint32_t split = (uint32_t)stream_split_of(P.runs[P.run_of[gi]].ng), nst = steps[(size_t)v * g.NG + gi];
            fs = std::max(fs, std::min(PF, (nst + split - 1) / split));
        }
    P.g.fs = (int)fs;
    P.head4.assign((size_t)g.NV * g.NG * 4, 0);
    uint64_t at = (uint64_t)P.NU * g.NV * fs;
    for (int v = 0; v < g.NV; ++v)
        for (int gi = 0; gi < g.NG; ++gi) {
            const StreamRun& run = P.runs[P.run_of[gi]];
            const uint32_t split = (uint32_t)stream_split_of(run.ng), nst = steps[(size_t)v * g.NG + gi];
            uint32_t* h = &P.head4[((size_t)v * g.NG + gi) * 4];
            h[0] = (uint32_t)at;
            h[1] = nst;
            h[2] = (uint32_t)run.u0 + (uint32_t)(gi - run.g0) * split;
            h[3] = split | ((uint32_t)run.g0 << 8);
            if (nst / split >= PF) at += nst - split * PF;
        }
    P.g.total_steps = at;
}

static void plan_places(int R, StreamPlan& P) {
    const StreamGeom& g = P.g;
    P.pos.assign((size_t)g.NV * R, 0);
    std::vector<uint32_t> steps((size_t)g.NV * g.NG, 0);
    parallel_blocks(g.NV, 1, [&](int a, int b) {
        std::vector<uint32_t> rows;
        for (int v = a; v < b; ++v) {
            const uint16_t* c = &P.cnt[(size_t)v * R];
            for (const StreamRun& run : P.runs) {
                // rows move between the groups of one column order only: a group reads one copy of x
                for (int oi = 0; oi < run.norders; ++oi) {
                    const int ga = run.g0 + run.bound[oi], gb = run.g0 + (oi + 1 < run.norders ? run.bound[oi + 1] : run.ng);
                    rows.clear();
                    for (int k = ga * 64; k < gb * 64; ++k)
                        if (P.base[k] != STREAM_NO_ROW) rows.push_back(P.base[k]);
                    std::stable_sort(rows.begin(), rows.end(), [c](uint32_t x, uint32_t y) { return c[x] > c[y]; });
                    for (size_t k = 0; k < rows.size(); ++k) P.pos[(size_t)v * R + rows[k]] = (uint32_t)(ga * 64 + k);
                    for (size_t k = 0; k < rows.size(); k += 64)
                        steps[(size_t)v * g.NG + ga + k / 64] = (c[rows[k]] + (uint32_t)g.fmt.eps - 1u) / (uint32_t)g.fmt.eps;
                }
            }
        }
    });
    plan_layout(steps.data(), P);
}

static int runs_word(const StreamPlan& P) { return P.g.runs | (P.GR << 16) | ((P.orders_max - 1) << 24) | ((P.g.fs - 1) << 27); }

// every lane's place and entry count (slot32), and the slots in the buffer's 16-bit form (place counted from the run's
// first place, entries or none)
static void plan_slots(int R, StreamPlan& P) {
    const StreamGeom& g = P.g;
    std::vector<uint32_t> place(R);
    for (size_t k = 0; k < P.base.size(); ++k)
        if (P.base[k] != STREAM_NO_ROW) place[P.base[k]] = (uint32_t)k;
    P.slot32.assign((size_t)g.NV * g.NG * 64, STREAM_NO_ROW);
    parallel_blocks(g.NV, 1, [&](int a, int b) {
        for (int v = a; v < b; ++v)
            for (int r = 0; r < R; ++r)
                P.slot32[(size_t)v * g.NG * 64 + P.pos[(size_t)v * R + r]] = place[r] | ((uint32_t)P.cnt[(size_t)v * R + r] << STREAM_ROW_BITS);
    });
}

static void encode_slots(const StreamPlan& P, uint16_t* slot16) {
    parallel_blocks(P.g.NV * P.g.NG, 256, [&](int a, int b) {
        for (int vg = a; vg < b; ++vg) {
            const uint32_t p0 = (P.head4[(size_t)vg * 4 + 3] >> 8) * 64u;
            for (int lane = 0; lane < 64; ++lane) {
                const uint32_t s32 = P.slot32[(size_t)vg * 64 + lane];
                slot16[(size_t)vg * 64 + lane] = (s32 & STREAM_NO_ROW) == STREAM_NO_ROW
                    ? (uint16_t)STREAM_SLOT_NONE
                    : (uint16_t)(((s32 & STREAM_NO_ROW) - p0) | ((s32 >> STREAM_ROW_BITS) ? STREAM_SLOT_HAS : 0u));
            }
        }
    });
}

// (G > 1: the labels a row's tags become are book << bits | tag, see sq_stream.h; `balanced` is for one codebook only)
static void plan_stream(const uint32_t* tags, int R, int W, int C, int d, int bits, const uint8_t* row_mask, int runs,
                        StreamPlan& P, bool balanced, int G, const uint8_t* row_book) {
    P.remap.clear();
    if (balanced) balance_codewords(tags, R, W, C / d, bits, P.remap);
    plan_rows(R, C, d, stream_label_bits(bits, G), row_mask, runs, P, balanced);
    plan_counts(tags, R, W, bits, balanced ? P.remap.data() : nullptr, G, row_book, P);
    plan_places(R, P);
}

void stream_balance_host(const uint32_t* tags, int R, int W, int C, int d, int bits, uint16_t* remap_out, int G,
                         const uint8_t* row_book) {
    std::vector<uint16_t> remap;
    balance_codewords(tags, R, W, C / d, bits, remap, G, row_book);
    memcpy(remap_out, remap.data(), remap.size() * sizeof(uint16_t));
}

size_t stream_bytes_host(const uint32_t* tags, int R, int W, int C, int d, int bits, const uint8_t* row_mask, int runs,
                         const uint16_t* table, int G, const uint8_t* row_book) {
    StreamPlan P;
    plan_stream(tags, R, W, C, d, bits, row_mask, runs, P, table != nullptr, G, row_book);
    return P.g.off_steps + (size_t)P.g.total_steps * P.g.fmt.step_bytes;
}

// The lanes of a wave that one clock of a 16-byte LDS read serves.  A ds_read_b128 takes four clocks; measured on
// gfx950 (two lanes reading different rows of one bank group while every other lane reads a third address: one extra
// clock exactly for the pairs listed together here; 256 random address patterns then fit "sum over the four sets of
// the most distinct addresses in one group of four banks" to within 1 percent), the sets are not 16 consecutive lanes:
#define SQ_LDS_CLOCK_LANES { \
    {0, 1, 2, 3, 12, 13, 14, 15, 20, 21, 22, 23, 24, 25, 26, 27}, \
    {4, 5, 6, 7, 8, 9, 10, 11, 16, 17, 18, 19, 28, 29, 30, 31}, \
    {32, 33, 34, 35, 44, 45, 46, 47, 52, 53, 54, 55, 56, 57, 58, 59}, \
    {36, 37, 38, 39, 40, 41, 42, 43, 48, 49, 50, 51, 60, 61, 62, 63}}
static const int LDS_CLOCK_LANES[4][16] = SQ_LDS_CLOCK_LANES;
__constant__ uint8_t STREAM_CLOCK_LANES_DEV[4][16] = SQ_LDS_CLOCK_LANES;

// Orders the entries of the 16 lanes of one LDS clock (see the second pass of stream_build_host): every entry slot
// should hold, over the 16 lanes, 16 different codeword bank groups (tag mod 16) and 16 different bank groups of x
// (chunk mod 16).  A greedy fill (each lane takes the entry that collides least with the lanes before it) followed by
// hill climbing over the whole group: a lane that collides in a slot swaps that entry with one of its other slots when
// the two slots together get cheaper.
struct BankMatch {
    static constexpr uint32_t NONE = 0xFFFFFFFFu;
    std::vector<uint32_t> ent[16];           // [lane][slot]: the lane's real entries in slot order
    std::vector<uint8_t> ha, hb;             // [slot][16]: lanes per codeword / x bank group
    std::vector<uint8_t> mx;                 // [slot][4]: fullest codeword group, groups that full; the same for x
    uint32_t cnt[16];
    uint32_t eps = 4;                        // entries per lane and step (StreamFmt.eps)

    // entry n of a lane in a group whose steps begin at base: entries are kept one per word, [step][lane][eps], until
    // they are moved to their places
    uint32_t* rec_of(uint32_t* base, int lane, uint32_t n) const { return base + ((size_t)(n / eps) * 64 + lane) * eps + n % eps; }
    static int ga(uint32_t e) { return (int)(e & 15u); }
    static int gb(uint32_t e) { return (int)((e >> STREAM_SLICE_BITS) & 15u); }
    void add(uint32_t n, uint32_t e, int d) { ha[n * 16 + ga(e)] += d; hb[n * 16 + gb(e)] += d; }

    // zero_chunk: the first of the 16 chunks of x that the kernel keeps at zero
    void order_lanes(uint32_t* base, const uint32_t* sl, const int* lanes, uint32_t ns, uint32_t zero_chunk) {
        uint32_t most = 0;
        for (int l = 0; l < 16; ++l) {
            const uint32_t s0 = sl[lanes[l]];
            cnt[l] = (s0 & STREAM_NO_ROW) == STREAM_NO_ROW ? 0u : s0 >> STREAM_ROW_BITS;
            ent[l].resize(cnt[l]);
            for (uint32_t n = 0; n < cnt[l]; ++n) ent[l][n] = *rec_of(base, lanes[l], n);
            most = std::max(most, cnt[l]);
        }
        if (most == 0) return;
        ha.assign((size_t)ns * 16, 0);
        hb.assign((size_t)ns * 16, 0);
        // greedy fill, slot by slot; the lanes with the fewest entries left choose first
        int order[16];
        for (int l = 0; l < 16; ++l) order[l] = l;
        std::sort(order, order + 16, [this](int x, int y) { return cnt[x] != cnt[y] ? cnt[x] < cnt[y] : x < y; });
        for (uint32_t n = 0; n < most; ++n)
            for (int d = 0; d < 16; ++d) {
                const int l = order[d];
                if (cnt[l] <= n) continue;
                uint32_t bi = n;
                int bc = 1 << 30;
                for (uint32_t i = n; i < cnt[l]; ++i) {
                    const int c = ha[n * 16 + ga(ent[l][i])] + hb[n * 16 + gb(ent[l][i])];
                    if (c < bc) { bc = c; bi = i; if (c == 0) break; }
                }
                std::swap(ent[l][n], ent[l][bi]);
                add(n, ent[l][n], 1);
            }
        // Hill climbing.  What a slot costs is the fullest bank group of its codeword reads plus that of its x reads
        // (clocks); with 16 lanes on 16 bank groups some collisions are forced, and they are cheapest when they share
        // slots.  A lane in a fullest group swaps that entry with one of its other slots when the clocks of the two
        // slots together go down (ties: when the sum of squared group counts does).  The fullest group's count after
        // moving one lane from group p to group q follows from the count, the current maximum and how many groups hold
        // it, so a candidate costs a few operations.
        mx.assign((size_t)most * 4, 0);
        auto rescan = [&](uint32_t n) {
            uint8_t* m4 = &mx[n * 4];
            m4[0] = m4[1] = m4[2] = m4[3] = 0;
            for (int k = 0; k < 16; ++k) {
                const uint8_t a = ha[n * 16 + k], b = hb[n * 16 + k];
                if (a > m4[0]) { m4[0] = a; m4[1] = 1; } else if (a == m4[0]) ++m4[1];
                if (b > m4[2]) { m4[2] = b; m4[3] = 1; } else if (b == m4[2]) ++m4[3];
            }
        };
        // fullest count of histogram h (maximum M held by `at` groups) once a lane leaves group p and joins group q
        auto moved = [](const uint8_t* h, int M, int at, int p, int q) {
            if (p == q) return M;
            if (h[q] + 1 > M) return h[q] + 1;
            return (h[p] == M && at == 1 && h[q] + 1 < M) ? M - 1 : M;
        };
        for (uint32_t n = 0; n < most; ++n) rescan(n);
        for (int pass = 0; pass < STREAM_CLIMB; ++pass) {
            bool improved = false;
            for (uint32_t n = 0; n < most; ++n) {
                const uint8_t* an = &ha[n * 16];
                const uint8_t* bn = &hb[n * 16];
                const uint8_t* xn = &mx[n * 4];
                if (xn[0] + xn[2] <= 2) continue;
                for (int l = 0; l < 16; ++l) {
                    if (cnt[l] <= n) continue;
                    const uint32_t e = ent[l][n];
                    const int ae = ga(e), be = gb(e);
                    if (!((an[ae] == xn[0] && xn[0] > 1) || (bn[be] == xn[2] && xn[2] > 1))) continue;
                    int best = 0;
                    uint32_t bm = n;
                    for (uint32_t m = 0; m < cnt[l]; ++m) {
                        if (m == n) continue;
                        const uint32_t f = ent[l][m];
                        const int af = ga(f), bf = gb(f);
                        const uint8_t* am = &ha[m * 16];
                        const uint8_t* bq = &hb[m * 16];
                        const uint8_t* xm = &mx[m * 4];
                        const int clocks = moved(an, xn[0], xn[1], ae, af) + moved(bn, xn[2], xn[3], be, bf) +
                                           moved(am, xm[0], xm[1], af, ae) + moved(bq, xm[2], xm[3], bf, be) -
                                           (xn[0] + xn[2] + xm[0] + xm[2]);
                        if (clocks > 0) continue;
                        int sq = 0;
                        if (af != ae) sq += 4 + 2 * ((int)an[af] - an[ae] + am[ae] - am[af]);
                        if (bf != be) sq += 4 + 2 * ((int)bn[bf] - bn[be] + bq[be] - bq[bf]);
                        const int delta = clocks * 1024 + sq;
                        if (delta < best) { best = delta; bm = m; }
                    }
                    if (bm != n) {
                        const uint32_t f = ent[l][bm];
                        add(n, e, -1); add(bm, f, -1); add(n, f, 1); add(bm, e, 1);
                        std::swap(ent[l][n], ent[l][bm]);
                        rescan(n);
                        rescan(bm);
                        improved = true;
                        if (xn[0] + xn[2] <= 2) break;
                    }
                }
            }
            if (!improved) break;
        }
        // Write the slots back.  A lane that has run out repeats one of its own codewords (from the least used bank
        // group) against one of the 16 chunks of x that are kept at zero (one per bank group).  A lane without a row,
        // or whose row has no entry here, reads what a neighbour reads (the same addresses are one broadcast read); the
        // kernel drops its sum.
        for (uint32_t n = 0; n < ns; ++n) {
            uint32_t chosen[16];
            int donor = -1;
            for (int l = 0; l < 16; ++l)
                if (cnt[l] > n) { chosen[l] = ent[l][n]; if (donor < 0) donor = l; }
            for (int l = 0; l < 16; ++l) {
                if (cnt[l] > n || cnt[l] == 0) continue;
                uint32_t bi = 0;
                for (uint32_t i = 1; i < cnt[l]; ++i)
                    if (ha[n * 16 + ga(ent[l][i])] < ha[n * 16 + ga(ent[l][bi])]) bi = i;
                int kb = 0;
                for (int k = 1; k < 16; ++k)
                    if (hb[n * 16 + k] < hb[n * 16 + kb]) kb = k;
                chosen[l] = (ent[l][bi] & ((1u << STREAM_SLICE_BITS) - 1u)) | ((uint32_t)(zero_chunk + kb) << STREAM_SLICE_BITS);
                add(n, chosen[l], 1);
                if (donor < 0) donor = l;
            }
            for (int l = 0; l < 16; ++l) {
                if (cnt[l] == 0) chosen[l] = donor >= 0 ? chosen[donor] : 0u;
                *rec_of(base, lanes[l], n) = chosen[l];
            }
        }
    }
};

// One step of 64 lanes x eps entries (one per word) into its bytes: 3 bytes per entry (wide), or the three 21-bit
// entries of a lane in one 64-bit word (narrow).
static void encode_step(const uint32_t* e, const StreamFmt& f, unsigned char* out) {
    for (int lane = 0; lane < 64; ++lane) {
        const uint32_t* r = e + (size_t)lane * f.eps;
        unsigned char* o = out + (size_t)lane * f.lane_bytes;
        if (f.narrow) {
            const uint64_t w = (uint64_t)r[0] | (uint64_t)r[1] << 21 | (uint64_t)r[2] << 42;
            for (int b = 0; b < 8; ++b) o[b] = (unsigned char)(w >> (8 * b));
        } else {
            for (int k = 0; k < 4; ++k) { o[3 * k] = (unsigned char)r[k]; o[3 * k + 1] = (unsigned char)(r[k] >> 8); o[3 * k + 2] = (unsigned char)(r[k] >> 16); }
        }
    }
}

int stream_build_host(const uint32_t* tags, int R, int W, int C, int d, int bits, const uint8_t* row_mask, int runs,
                      unsigned char* out, size_t bytes, int* runs_out, int* groups_out, const uint16_t* table, int G,
                      const uint8_t* row_book) {
    StreamPlan P;
    plan_stream(tags, R, W, C, d, bits, row_mask, runs, P, table != nullptr, G, row_book);
    const uint16_t* remap = table ? P.remap.data() : nullptr;
    const StreamGeom& g = P.g;
    const StreamFmt f = g.fmt;
    const uint32_t EPS = (uint32_t)f.eps, PF = (uint32_t)f.pf, FS = (uint32_t)g.fs;
    const size_t need = g.off_steps + (size_t)g.total_steps * f.step_bytes;
    if (g.total_steps >= ((uint64_t)1 << 32) || g.runs >= (1 << 16)) return fail(SQ_EUNSUPPORTED, "sq_stream_build: matrix too large");
    if (bytes < need) return fail(SQ_EINVAL, "sq_stream_build: buffer %zu < %zu", bytes, need);
    memset(out, 0, need);
    memcpy(out, P.head4.data(), P.head4.size() * 4);
    memcpy(out + g.off_runs, P.runs.data(), P.runs.size() * sizeof(StreamRun));
    memcpy(out + g.off_rows, P.base.data(), P.base.size() * 4);
    if (table) {
        uint16_t* tab = (uint16_t*)(out + g.off_table);
        uint16_t* unmap = (uint16_t*)(out + g.off_unmap);
        for (int k = 0; k < (1 << bits); ++k) {
            memcpy(tab + (size_t)remap[k] * d, table + (size_t)k * d, (size_t)d * 2);
            unmap[remap[k]] = (uint16_t)k;
        }
    }
    plan_slots(R, P);
    uint32_t* slots = P.slot32.data();
    // the steps are made group after group (P.goff), one entry per word, and moved to their places at the end
    std::vector<uint32_t> laid((size_t)P.logical_steps * 64 * EPS, 0);
    uint32_t* steps = laid.data();
    auto rec = [&](size_t step0, uint32_t lane, uint32_t n) { return steps + ((step0 + n / EPS) * 64 + lane) * EPS + n % EPS; };
    parallel_blocks(R, 64, [&](int a, int b) {
        std::vector<uint32_t> q(g.NV), last(g.NV);
        for (int r = a; r < b; ++r) {
            const uint32_t* row = tags + (size_t)r * W;
            const uint32_t book = row_book ? (uint32_t)(row_book[r] & (G - 1)) << bits : 0u;
            std::fill(q.begin(), q.end(), 0u);
            std::fill(last.begin(), last.end(), 0u);
            for (int j = 0; j < g.U; ++j) {
                uint32_t t = host_tag(row, W, bits, j);
                if (remap) t = remap[t];
                t |= book;
                const int kp = j / g.PC, v = kp * g.NS + (int)(t >> STREAM_SLICE_BITS);
                const uint32_t k = P.pos[(size_t)v * R + r], n = q[v]++;
                const uint32_t e = (t & ((1u << STREAM_SLICE_BITS) - 1u)) | ((uint32_t)(j - kp * g.PC) << STREAM_SLICE_BITS);
                *rec(P.goff[(size_t)v * g.NG + (k >> 6)], k & 63, n) = e;
                last[v] = e & ((1u << STREAM_SLICE_BITS) - 1u);
            }
            // Padding up to the group's longest row: the row's last codeword of the bucket again, at the chunk of x
            // that the kernel keeps at zero, so padding adds exactly nothing and needs no test in the inner loop
            // (a codeword that is not finite is already part of the row's sum; a row without entries in the
            // bucket is dropped by its slot).
            for (int v = 0; v < g.NV; ++v) {
                const uint32_t k = P.pos[(size_t)v * R + r];
                const size_t gi = (size_t)v * g.NG + (k >> 6);
                const uint32_t cap = (P.goff[gi + 1] - P.goff[gi]) * EPS;
                const uint32_t e = last[v] | ((uint32_t)g.PC << STREAM_SLICE_BITS);
                for (uint32_t n = q[v]; n < cap; ++n) *rec(P.goff[gi], k & 63, n) = e;
            }
        }
    });
    // Second pass, group by group: the order of a lane's entries is free (padding stays behind them), so it is
    // chosen to keep the LDS gathers apart.  A 16-byte LDS read of a wave takes four clocks of 16 lanes each
    // (LDS_CLOCK_LANES), and two lanes of a clock collide when their addresses differ but fall into the same group
    // of four banks (address / 16 mod 16): BankMatch arranges the entries of each clock's lanes.
    parallel_blocks(g.NV * g.NG, 4, [&](int a, int b) {
        BankMatch bm;
        bm.eps = EPS;
        for (int vg = a; vg < b; ++vg) {
            const uint32_t st0 = P.goff[vg], ns = (P.goff[vg + 1] - st0) * EPS;
            if (ns == 0) continue;
            const uint32_t* sl = slots + (size_t)vg * 64;
            uint32_t* base = steps + (size_t)st0 * 64 * EPS;
            for (int q = 0; q < 4; ++q) bm.order_lanes(base, sl, LDS_CLOCK_LANES[q], ns, (uint32_t)g.PC);
        }
    });
    // to their places: the first FS steps of every unit into the first-steps region, the rest behind each other
    encode_slots(P, (uint16_t*)(out + g.off_slots));
    parallel_blocks(g.NV * g.NG, 64, [&](int a, int b) {
        for (int vg = a; vg < b; ++vg) {
            const uint32_t* h = &P.head4[(size_t)vg * 4];
            const int v = vg / g.NG, nst = (int)h[1], split = (int)(h[3] & 0xFFu);
            const uint32_t* src = steps + (size_t)P.goff[vg] * 64 * EPS;
            for (int j = 0; j < split; ++j) {
                const int s0 = nst * j / split, s1 = nst * (j + 1) / split;
                for (int t = s0; t < s1; ++t) {
                    const uint64_t to = (uint32_t)(t - s0) < PF ? ((uint64_t)(h[2] + j) * g.NV + v) * FS + (t - s0)
                                                                 : (uint64_t)h[0] + t - (uint64_t)PF * (j + 1);
                    encode_step(src + (size_t)t * 64 * EPS, f, out + g.off_steps + to * f.step_bytes);
                }
            }
        }
    });
    if (runs_out) *runs_out = runs_word(P) | (table ? STREAM_BALANCED : 0);
    if (groups_out) *groups_out = g.NG;
    return SQ_OK;
}


// ------------------------------------------------------------------------------------------ on the GPU
//
// The same buffer, byte for byte, from tags that are already in device memory.  What is serial and small stays on the host
// (the rows' order and runs, the groups' places from their step counts); what walks tags or rows runs here: counting, the sort of
// the rows of a run by entry count, collecting every lane's entries, ordering them for the LDS banks, encoding.  The ordering is what the host
// spends its time on (16 cores: 150 ms for 18944 x 3584, 2.5 s for 3584 x 18944 on one).  Whole load of a matrix, tags on
// the GPU to stream on the GPU, the host builder / this one: 3584 x 3584 363 / 0.83 ms, 18944 x 3584 155 / 1.8, 3584 x 18944 2525 / 4.4.

// A row's codebook as these kernels index with it: below G (a power of two) whatever row_book holds, as in the host builder.
// The callers have refused a row_book that names another one, except where it may have been written since.
__device__ __forceinline__ uint32_t stream_book(const uint8_t* row_book, int r, int G, int bits) {
    return row_book ? ((uint32_t)row_book[r] & (uint32_t)(G - 1)) << bits : 0u;
}

// count[book << bits | label] += 1 for every tag (one wave per row)
__global__ __launch_bounds__(256) void stream_codeword_count_kernel(const uint32_t* __restrict__ tags, int R, int W, int U, int bits, int G,
                                                                    const uint8_t* __restrict__ row_book, uint32_t* __restrict__ count) {
    const int r = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (r >= R) return;
    const uint32_t* row = tags + (int64_t)r * W;
    const uint32_t book = stream_book(row_book, r, G, bits);
    for (int j = lane; j < U; j += 64) atomicAdd(count + (book | tag_at(row, W, bits, j)), 1u);
}

__global__ __launch_bounds__(256) void stream_clear_kernel(uint32_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// rewrites the tags of a matrix through remap[book << bits | label] in place; a thread owns 32 tags, which are whole words
__global__ __launch_bounds__(256) void stream_relabel_kernel(uint32_t* __restrict__ tags, int R, int W, int U, int bits, int G,
                                                             const uint8_t* __restrict__ row_book, const uint16_t* __restrict__ remap) {
    const int units = (U + 31) / 32;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)R * units) return;
    const int r = (int)(i / units), u = (int)(i - (int64_t)r * units);
    uint32_t* w = tags + (int64_t)r * W + u * bits;
    const int nw = min(bits, W - u * bits), n = min(32, U - u * 32);
    const uint16_t* map = remap + stream_book(row_book, r, G, bits);
    const uint32_t mask = (1u << bits) - 1u;
    uint64_t in = 0, out = 0;
    int have = 0, held = 0, rd = 0, wr = 0;
    for (int k = 0; k < n; ++k) {
        if (have < bits) { in |= (uint64_t)(rd < nw ? w[rd] : 0u) << have; ++rd; have += 32; }
        out |= (uint64_t)map[(uint32_t)in & mask] << held;
        in >>= bits; have -= bits; held += bits;
        if (held >= 32) { w[wr++] = (uint32_t)out; out >>= 32; held -= 32; }
    }
    // the bits behind a row's last tag are zero, as pack_bits leaves them
    if (held > 0) w[wr++] = (uint32_t)out;
}

// cnt[v * R + r]: entries of row r in bucket v (one wave per row; its counters in LDS)
__global__ __launch_bounds__(64) void stream_count_kernel(const uint32_t* __restrict__ tags, int R, int W, int U, int bits, int G, int PC, int NS, int NV,
                                                          const uint8_t* __restrict__ row_book, uint16_t* __restrict__ cnt) {
    extern __shared__ uint32_t stream_count_lds[];
    const int r = (int)blockIdx.x, lane = (int)threadIdx.x;
    for (int v = lane; v < NV; v += 64) stream_count_lds[v] = 0u;
    __syncthreads();
    const uint32_t* row = tags + (int64_t)r * W;
    const uint32_t book = stream_book(row_book, r, G, bits);
    for (int j = lane; j < U; j += 64)
        atomicAdd(&stream_count_lds[(j / PC) * NS + (int)((book | tag_at(row, W, bits, j)) >> STREAM_SLICE_BITS)], 1u);
    __syncthreads();
    for (int v = lane; v < NV; v += 64) cnt[(int64_t)v * R + r] = (uint16_t)stream_count_lds[v];
}

struct StreamFillArgs {
    const uint32_t* tags;
    const uint8_t* row_book;
    const uint32_t* heads;      // [NV * NG][4], in the stream buffer
    const uint32_t* rows;       // [NV * NG * 64]: the row of every lane (STREAM_NO_ROW: none)
    const uint32_t* goff;       // [NV * NG + 1]: the groups' steps counted one behind the other
    unsigned char* steps;       // the stream buffer's steps
    unsigned char* work;        // groups that LDS does not hold: STREAM_FILL_BYTES per entry slot of every group
    int W, U, bits, G, PC, NS, NV, NG, fs;
    int wg0;                    // the first workgroup of this matrix
};
constexpr int STREAM_FILL_PIECES = 8;
struct StreamFillStack {
    StreamFillArgs p[STREAM_FILL_PIECES];
    int n;
};

// Bytes one entry slot (64 lanes) of a group takes: 65 words of entries (the odd pitch spreads one lane's entries over the
// banks), 16 + 16 bank-group counts for each of the four clocks, and their maxima.
constexpr int STREAM_FILL_BYTES = 65 * 4 + 4 * 32 + 4 * 4;
constexpr int STREAM_FILL_LDS = 156 * 1024;

// over the 16 threads of a DPP row: four rotations of a few cycles each; and over the wave, the four rows' results as scalars
template <int N> __device__ __forceinline__ int row_ror(int v) { return __builtin_amdgcn_update_dpp(v, v, 0x120 + N, 0xF, 0xF, false); }
__device__ __forceinline__ int min16(int v) {
    v = min(v, row_ror<8>(v)); v = min(v, row_ror<4>(v)); v = min(v, row_ror<2>(v));
    return min(v, row_ror<1>(v));
}
__device__ __forceinline__ int max16(int v) {
    v = max(v, row_ror<8>(v)); v = max(v, row_ror<4>(v)); v = max(v, row_ror<2>(v));
    return max(v, row_ror<1>(v));
}
__device__ __forceinline__ int add16(int v) {
    v += row_ror<8>(v); v += row_ror<4>(v); v += row_ror<2>(v);
    return v + row_ror<1>(v);
}
__device__ __forceinline__ int min64(int v) {
    v = min16(v);
    return min(min(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               min(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}
__device__ __forceinline__ int stream_ga(uint32_t e) { return (int)(e & 15u); }
__device__ __forceinline__ int stream_gb(uint32_t e) { return (int)((e >> STREAM_SLICE_BITS) & 15u); }
// thread K of each four
template <int K> __device__ __forceinline__ int quad_lane(int v) { return __builtin_amdgcn_update_dpp(v, v, K * 0x55, 0xF, 0xF, false); }
// The dwords that hold tags j .. j + 7 of a row (j a multiple of 8 behind the start of a part; past the row's end: its last dword),
// and the tags in them.
typedef uint32_t u32x4_by4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void stream_fetch8(const uint32_t* row, int W, int bits, int j, uint32_t (&d)[5]) {
    const int w = (int)((int64_t)j * bits >> 5);
    d[4] = 0u;
    if (w + 5 <= W) {
        const u32x4_by4 x = *reinterpret_cast<const u32x4_by4*>(row + w);
        d[0] = x[0]; d[1] = x[1]; d[2] = x[2]; d[3] = x[3];
        if (bits != 16 || (j & 1)) d[4] = row[w + 4];
    } else {
#pragma unroll
        for (int i = 0; i < 5; ++i) d[i] = row[min(w + i, W - 1)];
    }
}
__device__ __forceinline__ void stream_split8(const uint32_t (&d)[5], int bits, int j, uint32_t (&g)[8]) {
    if (bits == 16 && (j & 1) == 0) {
#pragma unroll
        for (int k = 0; k < 8; ++k) g[k] = d[k / 2] >> (k % 2 * 16) & 0xFFFFu;
        return;
    }
    const uint32_t s = (uint32_t)((int64_t)j * bits & 31), mask = (1u << bits) - 1u;
    uint32_t x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], s);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        g[k] = x[0] & mask;
#pragma unroll
        for (int i = 0; i < 3; ++i) x[i] = __builtin_amdgcn_alignbit(x[i + 1], x[i], bits);
        x[3] >>= bits;
    }
}

// One workgroup per (bucket, group), one wave per clock of the group: it collects its 16 rows' entries (four threads per
// row), orders them (the steps of BankMatch::order_lanes with ties resolved the same way; the 64 threads search a lane's
// candidates together), and the four waves write the encoded steps to their places.  Each wave is one serial chain, four or five of
// them share a SIMD, and the older go first, so what counts is the instructions and the LDS round trips of a link (one clock per
// wave: with four on one wave their branches took turns, 3584 x 18944 49 ms against 10).  3584, 512 and 512 rows of 448 chunks in one
// launch take 0.44 ms, 1.02 with tags collected one by one (470 us of it; now 16 us a group: eight tags a thread and load), the
// greedy fill through LDS counters (200 us; registers and ballots about half) and a search for every lane of every slot (350 us; now
// only for the lanes that a ballot finds in a fullest group, with half the arithmetic).  Matrices of a stack are filled side by
// side: each takes the length of its chains however small it is (one launch each: 1.9 times as long).
template <bool LDS>
__global__ __launch_bounds__(256) void stream_fill_kernel(StreamFillStack stack) {
    extern __shared__ __attribute__((aligned(16))) unsigned char stream_fill_lds[];
    int pi = 0;
    while (pi + 1 < stack.n && (int)blockIdx.x >= stack.p[pi + 1].wg0) ++pi;
    const StreamFillArgs& a = stack.p[pi];
    const int vg = (int)blockIdx.x - a.wg0, v = vg / a.NG, q = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), t = (int)threadIdx.x & 63, sub = t & 15;
    const StreamFmt f = stream_fmt(a.PC);
    const int nst = (int)a.heads[(size_t)vg * 4 + 1], ns = nst * f.eps;
    if (ns == 0) return;
    unsigned char* mem = LDS ? stream_fill_lds : a.work + (size_t)a.goff[vg] * f.eps * STREAM_FILL_BYTES;
    uint32_t* ent = reinterpret_cast<uint32_t*>(mem);                        // [slot][65]
    uint8_t* h = mem + (size_t)ns * (260 + 32 * q);                          // this clock's [slot][32]: codeword groups, x groups
    uint8_t* mx = mem + (size_t)ns * (260 + 128 + 4 * q);                    // and [slot][4]: their maxima

    // entries of the clock's rows in this bucket, in chunk order: the four threads of a row take 32 of its tags at a time, eight each
    const int crow = STREAM_CLOCK_LANES_DEV[q][t >> 2];
    const uint32_t row_id = a.rows[(size_t)vg * 64 + crow];
    int total = 0;
    if (row_id != STREAM_NO_ROW) {
        const uint32_t* row = a.tags + (int64_t)row_id * a.W;
        const uint32_t book = stream_book(a.row_book, (int)row_id, a.G, a.bits);
        const int kp = v / a.NS, sl = v - kp * a.NS, p0 = kp * a.PC, len = min(a.PC, a.U - p0);
        uint32_t d[5], ahead[5];
        stream_fetch8(row, a.W, a.bits, p0 + (t & 3) * 8, d);
        for (int i0 = 0; i0 < len; i0 += 32) {
            const int i = i0 + (t & 3) * 8;
            stream_fetch8(row, a.W, a.bits, p0 + i + 32, ahead);
            uint32_t g[8];
            stream_split8(d, a.bits, p0 + i, g);
            int n = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                g[k] |= book;
                n += (int)(g[k] >> STREAM_SLICE_BITS) == sl && i + k < len;
            }
            const int n0 = quad_lane<0>(n), n1 = quad_lane<1>(n), n2 = quad_lane<2>(n), n3 = quad_lane<3>(n);
            int slot = total + ((t & 3) > 0 ? n0 : 0) + ((t & 3) > 1 ? n1 : 0) + ((t & 3) > 2 ? n2 : 0);
            total += n0 + n1 + n2 + n3;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if ((int)(g[k] >> STREAM_SLICE_BITS) == sl && i + k < len) {
                    if (slot < ns) ent[slot * 65 + crow] = (g[k] & ((1u << STREAM_SLICE_BITS) - 1u)) | ((uint32_t)(i + k) << STREAM_SLICE_BITS);
                    ++slot;
                }
#pragma unroll
            for (int k = 0; k < 5; ++k) d[k] = ahead[k];
        }
    }
    for (int i = t; i < ns * 8; i += 64) reinterpret_cast<uint32_t*>(h)[i] = 0u;
    __syncthreads();

    const int cnt = __shfl(total, sub * 4, 64), my_lane = STREAM_CLOCK_LANES_DEV[q][sub];   // thread `sub`: its lane of this clock
    const bool has_row = __shfl((int)(row_id != STREAM_NO_ROW), sub * 4, 64) != 0;
    const int packed = cnt << 6 | my_lane;
    auto packed_of = [&](int l) { return __builtin_amdgcn_readlane(packed, l); };
    const int most = __builtin_amdgcn_readfirstlane(max16(cnt));
    // greedy fill: the lanes with the fewest entries choose first
    int rank = 0;
    for (int l = 0; l < 16; ++l) {
        const int c = packed_of(l) >> 6;
        rank += c < cnt || (c == cnt && l < sub);
    }
    int at_rank = 0;                                                         // thread d: the lane of rank d
    for (int l = 0; l < 16; ++l)
        if (__builtin_amdgcn_readlane(rank, l) == sub) at_rank = l;
    const int ranked = __shfl(packed, at_rank, 64);
    if (most <= 64) {
        // thread t holds entry t of every lane; the slot's counts are nibbles of two scalars (the newest, which may be the 16th of its
        // group, is held back), and the first cheapest entry is the first set bit of a ballot: no LDS in the chain, a dozen vector
        // instructions a link, which is what counts with four waves and more on a SIMD
        uint32_t E[16];
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            const int pk = __builtin_amdgcn_readlane(ranked, d);
            E[d] = t < pk >> 6 ? ent[t * 65 + (pk & 63)] : 0u;
        }
        for (int n = 0; n < most; ++n) {
            uint64_t A = 0, B = 0, newA = 0, newB = 0;
#pragma unroll
            for (int d = 0; d < 16; ++d) {
                const int cl = __builtin_amdgcn_readlane(ranked, d) >> 6;
                if (cl <= n) continue;
                A += newA;
                B += newB;
                const uint64_t open = (~0ull >> (64 - cl)) & (~0ull << n);   // entries n .. cl - 1
                const int cost = ((int)(A >> 4 * stream_ga(E[d])) & 15) + ((int)(B >> 4 * stream_gb(E[d])) & 15);
                uint64_t best = 0;
                for (int c = 0; best == 0; ++c) best = __ballot(cost == c) & open;      // (entry n is open: its cost ends the loop)
                const int bi = __builtin_ctzll(best);
                const int en = __builtin_amdgcn_readlane((int)E[d], n), eb = __builtin_amdgcn_readlane((int)E[d], bi);
                E[d] = (uint32_t)(t == n ? eb : t == bi ? en : (int)E[d]);
                newA = 1ull << 4 * stream_ga((uint32_t)eb);
                newB = 1ull << 4 * stream_gb((uint32_t)eb);
            }
            const uint64_t C = t < 16 ? A : B, newC = t < 16 ? newA : newB;
            if (t < 32) h[n * 32 + t] = (uint8_t)(((C >> 4 * sub) & 15) + ((newC >> 4 * sub) & 15));
        }
#pragma unroll
        for (int d = 0; d < 16; ++d) {
            const int pk = __builtin_amdgcn_readlane(ranked, d);
            if (t < pk >> 6) ent[t * 65 + (pk & 63)] = E[d];
        }
        __threadfence_block();
    } else {
        for (int n = 0; n < most; ++n)
            for (int d = 0; d < 16; ++d) {
                const int pk = __builtin_amdgcn_readlane(ranked, d), cl = pk >> 6, ln = pk & 63;
                if (cl <= n) continue;
                int key = 0x7FFFFFFF;                                        // cost << 16 | slot: the first cheapest
                for (int i = n + t; i < cl; i += 64) {
                    const uint32_t e = ent[i * 65 + ln];
                    key = min(key, ((int)h[n * 32 + stream_ga(e)] + (int)h[n * 32 + 16 + stream_gb(e)]) << 16 | i);
                }
                const int bi = min64(key) & 0xFFFF;
                const uint32_t en = ent[n * 65 + ln], eb = ent[bi * 65 + ln];
                if (t == 0) {
                    ent[n * 65 + ln] = eb;
                    ent[bi * 65 + ln] = en;
                    ++h[n * 32 + stream_ga(eb)];
                    ++h[n * 32 + 16 + stream_gb(eb)];
                }
                __threadfence_block();
            }
    }
    // the maxima of four slots at a time, 16 threads each
    auto rescan = [&](int n) {
        const int ca = h[n * 32 + sub], cb = h[n * 32 + 16 + sub];
        const int ma = max16(ca), mb = max16(cb);
        const int na = add16(ma > 0 && ca == ma), nb = add16(mb > 0 && cb == mb);
        if (sub == 0) *reinterpret_cast<uint32_t*>(mx + n * 4) = (uint32_t)ma | (uint32_t)na << 8 | (uint32_t)mb << 16 | (uint32_t)nb << 24;
    };
    for (int n = 0; n < most; n += 4) rescan(min(n + (t >> 4), most - 1));
    __threadfence_block();
    for (int pass = 0; pass < STREAM_CLIMB; ++pass)
        for (int n = 0; n < most; ++n) {
            const uint8_t* an = h + n * 32;
            const uint8_t* bn = an + 16;
            int x0, x1, x2, x3, ane16 = 0, bne16 = 0;                        // maximum and how many groups hold it, twice; thread `sub`:
            uint32_t e16 = 0;                                                // its lane's entry and the counts of its groups
            auto look = [&]() {                                              // the lanes that are in a fullest group, one bit each
                const int xw = __builtin_amdgcn_readfirstlane((int)*reinterpret_cast<const uint32_t*>(mx + n * 4));
                x0 = xw & 0xFF; x1 = xw >> 8 & 0xFF; x2 = xw >> 16 & 0xFF; x3 = xw >> 24 & 0xFF;
                if (x0 + x2 <= 2) return 0u;
                if (cnt > n) {
                    e16 = ent[n * 65 + my_lane];
                    ane16 = an[stream_ga(e16)];
                    bne16 = bn[stream_gb(e16)];
                }
                return (uint32_t)__ballot(cnt > n && ((ane16 == x0 && x0 > 1) || (bne16 == x2 && x2 > 1))) & 0xFFFFu;
            };
            uint32_t todo = look();
            while (todo) {
                const int l = __builtin_ctz(todo), pk = packed_of(l), cl = pk >> 6, ln = pk & 63;
                todo &= todo - 1;
                const uint32_t e = (uint32_t)__builtin_amdgcn_readlane((int)e16, l);
                const int ae = stream_ga(e), be = stream_gb(e), ane = __builtin_amdgcn_readlane(ane16, l), bne = __builtin_amdgcn_readlane(bne16, l);
                // What a swap with slot m changes: the fullest group's count of slot n once e left for f's group, of slot m the other way
                // round (a group that alone is fullest lets the maximum sink by one, the joined one may raise it), and for ties the
                // squares, which weigh less than one clock.  Nothing where f's group is e's (the slot itself).
                const int an0 = x0 - (ane == x0 && x1 == 1), bn0 = x2 - (bne == x2 && x3 == 1);
                int key = 0;                                                 // delta << 13 | slot; only gains are below 0
                for (int m = t; m < cl; m += 64) {
                    const uint32_t fm = ent[m * 65 + ln];
                    const int af = stream_ga(fm), bf = stream_gb(fm);
                    const uint8_t* am = h + m * 32;
                    const uint8_t* bq = am + 16;
                    const int xm = *reinterpret_cast<const int*>(mx + m * 4), y0 = xm & 0xFF, y2 = xm >> 16 & 0xFF;
                    const int anf = an[af], bnf = bn[bf], ame = am[ae], amf = am[af], bqe = bq[be], bqf = bq[bf];
                    const int am0 = (xm & 0xFFFF) == (amf | 1 << 8) ? y0 - 1 : y0, bm0 = xm >> 16 == (bqf | 1 << 8) ? y2 - 1 : y2;
                    const int da = (max(anf + 1, an0) + max(ame + 1, am0) - x0 - y0) * 1024 + 4 + 2 * (anf - ane + ame - amf);
                    const int db = (max(bnf + 1, bn0) + max(bqe + 1, bm0) - x2 - y2) * 1024 + 4 + 2 * (bnf - bne + bqe - bqf);
                    const int delta = (af != ae ? da : 0) + (bf != be ? db : 0);
                    if (delta < 0) key = min(key, delta * 8192 + m);
                }
                if (!__any(key < 0)) continue;                               // (nothing changed: the other bits stand)
                key = min64(key);
                const int bm = key & 0x1FFF;                                 // (the least key: the largest gain, its first slot)
                const uint32_t fm = ent[bm * 65 + ln];
                if (t == 0) {
                    const int af = stream_ga(fm), bf = stream_gb(fm);
                    --h[n * 32 + ae]; --h[n * 32 + 16 + be]; --h[bm * 32 + af]; --h[bm * 32 + 16 + bf];
                    ++h[n * 32 + af]; ++h[n * 32 + 16 + bf]; ++h[bm * 32 + ae]; ++h[bm * 32 + 16 + be];
                    ent[n * 65 + ln] = fm;
                    ent[bm * 65 + ln] = e;
                }
                __threadfence_block();
                rescan(t & 16 ? bm : n);
                __threadfence_block();
                todo = look() & (0xFFFEu << l);
            }
        }
    // padding: a lane that has run out repeats one of its codewords (least used bank group) against a zero chunk of x; a
    // lane without entries reads what a neighbour reads (in a clock without any entry: codeword 0 against a zero chunk)
    for (int n = 0; n < ns; ++n) {
        const uint32_t full = (uint32_t)__ballot(cnt > n) & 0xFFFFu;
        uint32_t todo = (uint32_t)__ballot(cnt <= n && cnt > 0) & 0xFFFFu;
        const int donor = full ? __builtin_ctz(full) : todo ? __builtin_ctz(todo) : 16;
        int ca = h[n * 32 + sub], cb = h[n * 32 + 16 + sub];                 // thread `sub`: the counts of group sub
        while (todo) {
            const int l = __builtin_ctz(todo), pk = packed_of(l), cl = pk >> 6, ln = pk & 63;
            todo &= todo - 1;
            int key = 0x7FFFFFFF;
            for (int i0 = 0; i0 < cl; i0 += 64) {                            // (all threads: a count comes from the thread that has it)
                const int i = min(i0 + t, cl - 1);
                key = min(key, __shfl(ca, stream_ga(ent[i * 65 + ln]), 64) << 16 | i);
            }
            const int bi = min64(key) & 0xFFFF;
            const int kb = min16(cb << 4 | sub) & 15;
            const uint32_t c = (ent[bi * 65 + ln] & ((1u << STREAM_SLICE_BITS) - 1u)) | ((uint32_t)(a.PC + kb) << STREAM_SLICE_BITS);
            if (t == 0) ent[n * 65 + ln] = c;
            ca += sub == stream_ga(c);
            cb += sub == stream_gb(c);
        }
        __threadfence_block();
        const int dl = packed_of(donor & 15) & 63;
        if (cnt == 0 && t < 16) ent[n * 65 + my_lane] = donor < 16 ? ent[n * 65 + dl] : has_row ? (uint32_t)a.PC << STREAM_SLICE_BITS : 0u;
    }
    __syncthreads();

    const uint32_t* hd = a.heads + (size_t)vg * 4;
    const int split = (int)(hd[3] & 0xFFu);
    for (int j = 0; j < split; ++j) {
        const int s0 = nst * j / split, s1 = nst * (j + 1) / split;
        for (int st = s0 + q; st < s1; st += 4) {
            const uint64_t to = st - s0 < f.pf ? ((uint64_t)(hd[2] + j) * a.NV + v) * a.fs + (st - s0) : (uint64_t)hd[0] + st - (uint64_t)f.pf * (j + 1);
            unsigned char* o = a.steps + to * f.step_bytes + t * f.lane_bytes;
            const uint32_t* e = ent + st * f.eps * 65 + t;
            if (f.narrow) {
                const uint64_t w = (uint64_t)e[0] | (uint64_t)e[65] << 21 | (uint64_t)e[130] << 42;
                *reinterpret_cast<u32x2*>(o) = u32x2{(uint32_t)w, (uint32_t)(w >> 32)};
            } else {
                const uint32_t e0 = e[0] & 0xFFFFFFu, e1 = e[65] & 0xFFFFFFu, e2 = e[130] & 0xFFFFFFu, e3 = e[195] & 0xFFFFFFu;
                uint32_t* o4 = reinterpret_cast<uint32_t*>(o);
                o4[0] = e0 | e1 << 24;
                o4[1] = e1 >> 8 | e2 << 16;
                o4[2] = e2 >> 16 | e3 << 8;
            }
        }
    }
}

// the tile-major copy of the tags (tiled_build) from tags in device memory: a thread moves one unit of a row
__global__ __launch_bounds__(256) void tiled_build_kernel(const uint32_t* __restrict__ tags, int R, int W, int U, int ud, uint32_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;          // (tile, unit, row of the tile)
    if (i >= (int64_t)((R + 15) / 16) * 16 * U) return;
    const int k = (int)(i & 15);
    const int64_t tu = i >> 4;
    const int u = (int)(tu % U), r = (int)(tu / U) * 16 + k;
    uint32_t* dst = out + i * ud;
    const uint32_t* src = tags + (int64_t)r * W + u * ud;
    for (int w = 0; w < ud; ++w) dst[w] = r < R && u * ud + w < W ? src[w] : 0u;
}

int stream_balance_device(const uint32_t* tags, int R, int W, int C, int d, int bits, uint32_t* counts, uint16_t* remap_out, int G,
                          const uint8_t* row_book, hipStream_t s) {
    const int64_t n = (int64_t)G << bits;
    hipLaunchKernelGGL(stream_clear_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, counts, n);
    hipLaunchKernelGGL(stream_codeword_count_kernel, dim3((unsigned)((R + 3) / 4)), dim3(256), 0, s, tags, R, W, C / d, bits, G, row_book, counts);
    int rc = check_launch("sq_codebook_balance_device");
    if (rc) return rc;
    std::vector<uint32_t> host((size_t)n);
    hipError_t e = hipMemcpyAsync(host.data(), counts, (size_t)n * 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return fail(SQ_ELAUNCH, "sq_codebook_balance_device: %s", hipGetErrorString(e));
    std::vector<uint16_t> remap;
    deal_codewords(host.data(), bits, remap, G);
    memcpy(remap_out, remap.data(), remap.size() * sizeof(uint16_t));
    return SQ_OK;
}

int stream_relabel_device(uint32_t* tags, int R, int W, int C, int d, int bits, int G, const uint8_t* row_book, const uint16_t* remap, hipStream_t s) {
    const int64_t n = (int64_t)R * ((C / d + 31) / 32);
    if (n == 0) return SQ_OK;
    hipLaunchKernelGGL(stream_relabel_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, tags, R, W, C / d, bits, G, row_book, remap);
    return check_launch("sq_codebook_relabel_device");
}

// One column order's rows of one run: groups ga .. ga + ng - 1, places from ga * 64; p0: the run's first place.
struct StreamSegment { int32_t ga, ng, p0, pad; };

struct StreamSortArgs {
    const uint16_t* cnt;        // [NV][R]
    const uint32_t* base;       // [NG * 64]: the row of every place
    const StreamSegment* seg;
    uint32_t* steps;            // [NV * NG], or NULL
    uint32_t* rows;             // [NV * NG * 64]: the row of every lane, or NULL
    uint16_t* slots;            // the buffer's slots, with rows
    int R, NG, eps;
};

// The rows of a segment in one bucket by entry count, most first, equal counts in the order of their places: a bitonic sort of
// (count, place) in LDS.  Runs of 256 rows (3584 rows in 14, 16 buckets) take 11 us; on the host, with the counts' way there and the
// places' way back, it was 600 us of every matrix' load, however small.
__global__ __launch_bounds__(1024) void stream_sort_kernel(StreamSortArgs a) {
    extern __shared__ uint32_t stream_sort_lds[];
    const StreamSegment sg = a.seg[blockIdx.x];
    const int v = (int)blockIdx.y, n = sg.ng * 64, tid = (int)threadIdx.x, nt = (int)blockDim.x;
    int size = 64;
    while (size < n) size *= 2;
    for (int i = tid; i < size; i += nt) {
        const uint32_t row = i < n ? a.base[sg.ga * 64 + i] : STREAM_NO_ROW;
        stream_sort_lds[i] = row == STREAM_NO_ROW ? 0xFFFFFFFFu : (8191u - a.cnt[(size_t)v * a.R + row]) << 13 | (uint32_t)i;
    }
    for (int k = 2; k <= size; k *= 2)
        for (int j = k / 2; j > 0; j /= 2) {
            __syncthreads();
            for (int t = tid; t < size / 2; t += nt) {
                const int i = (t & ~(j - 1)) * 2 | (t & (j - 1));
                const uint32_t x = stream_sort_lds[i], y = stream_sort_lds[i + j];
                if ((x > y) == ((i & k) == 0)) {
                    stream_sort_lds[i] = y;
                    stream_sort_lds[i + j] = x;
                }
            }
        }
    __syncthreads();
    for (int i = tid; i < n; i += nt) {
        const uint32_t key = stream_sort_lds[i], c = key == 0xFFFFFFFFu ? 0u : 8191u - (key >> 13);
        const size_t at = ((size_t)v * a.NG + sg.ga) * 64 + i;
        if (a.steps && i % 64 == 0) a.steps[at / 64] = (c + (uint32_t)a.eps - 1u) / (uint32_t)a.eps;
        if (a.rows) {
            const uint32_t place = (uint32_t)sg.ga * 64u + (key & 8191u);
            a.rows[at] = key == 0xFFFFFFFFu ? STREAM_NO_ROW : a.base[place];
            a.slots[at] = key == 0xFFFFFFFFu ? (uint16_t)STREAM_SLOT_NONE : (uint16_t)((place - (uint32_t)sg.p0) | (c ? STREAM_SLOT_HAS : 0u));
        }
    }
}

// The stream buffer in front of its steps from what the host has planned (heads, runs and rows lie in `plan` one behind the
// other), and zeros everywhere else.
__global__ __launch_bounds__(256) void stream_front_kernel(const uint32_t* __restrict__ plan, int64_t heads, int64_t runs0, int64_t runs, int64_t rows0,
                                                           int64_t rows, uint32_t* __restrict__ out, int64_t words) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= words) return;
    uint32_t v = 0u;
    if (i < heads) v = plan[i];
    else if (i >= runs0 && i < runs0 + runs) v = plan[heads + i - runs0];
    else if (i >= rows0 && i < rows0 + rows) v = plan[heads + runs + i - rows0];
    out[i] = v;
}

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

static void launch_count_and_sort(const StreamPlan& P, const uint32_t* tags, int R, int W, int bits, int G, const uint8_t* row_book, uint16_t* cnt,
                                  const StreamSortArgs& a, int segments, hipStream_t s) {
    const StreamGeom& g = P.g;
    int size = 64;
    while (size < P.GR * 64) size *= 2;
    hipLaunchKernelGGL(stream_count_kernel, dim3((unsigned)R), dim3(64), (size_t)g.NV * 4, s, tags, R, W, g.U, bits, G, g.PC, g.NS, g.NV, row_book, cnt);
    hipLaunchKernelGGL(stream_sort_kernel, dim3((unsigned)segments, (unsigned)g.NV), dim3((unsigned)std::min(1024, std::max(64, size / 2))), (size_t)size * 4, s, a);
}

static std::vector<StreamSegment> plan_segments(const StreamPlan& P) {
    std::vector<StreamSegment> seg;
    for (const StreamRun& run : P.runs)
        for (int i = 0; i < run.norders; ++i)
            seg.push_back({run.g0 + run.bound[i], (i + 1 < run.norders ? run.bound[i + 1] : run.ng) - run.bound[i], run.g0 * 64, 0});
    return seg;
}

// the counts, the groups' step counts, the segments and the places' rows; every column order can leave one group short
size_t stream_counts_bytes(int R, int C, int d, int bits, int G) {
    const size_t NV = (size_t)stream_geom(C, d, stream_label_bits(bits, G), 0, 0).NV, groups = (size_t)R / 64 + 256;
    return align256(NV * R * 2) + align256(NV * groups * 4) + groups * sizeof(StreamSegment) + groups * 64 * 4;
}

// A plan on its way from stream_plan_device to stream_fill_device.
struct StreamDevicePlan {
    StreamPlan P;
    std::vector<StreamSegment> seg;
    std::vector<uint32_t> upload;    // heads, runs, rows; then the groups' offsets and the segments
    int R, W, C, d, bits, G;
    bool tiled, in_lds;
    size_t bytes, scratch, at_goff, at_seg, at_rows, at_cnt, at_work;   // places in the scratch
};

int stream_plan_device(const uint32_t* tags, int R, int W, int C, int d, int bits, int G, const uint8_t* row_book, const uint8_t* row_mask_host,
                       int runs, void* counts, StreamDevicePlan** out, size_t* bytes, size_t* scratch, int* runs_out, int* groups_out, hipStream_t s) {
    std::unique_ptr<StreamDevicePlan> D(new StreamDevicePlan);
    D->R = R; D->W = W; D->C = C; D->d = d; D->bits = bits; D->G = G;
    D->tiled = !stream_format_ok(R, C, d, bits, G);
    D->in_lds = false;
    if (D->tiled) {
        D->bytes = tiled_bytes(R, C, bits);
        D->scratch = 0;
        *runs_out = *groups_out = 0;
    } else {
        StreamPlan& P = D->P;
        plan_rows(R, C, d, stream_label_bits(bits, G), row_mask_host, runs, P, false);
        const StreamGeom& g = P.g;
        const size_t nvg = (size_t)g.NV * g.NG;
        D->seg = plan_segments(P);
        char* at = (char*)counts;
        StreamSortArgs a{};
        a.cnt = (uint16_t*)at; at += align256((size_t)g.NV * R * 2);
        a.steps = (uint32_t*)at; at += align256((size_t)g.NV * ((size_t)R / 64 + 256) * 4);
        a.seg = (StreamSegment*)at;
        a.base = (uint32_t*)(at + D->seg.size() * sizeof(StreamSegment));
        a.R = R; a.NG = g.NG; a.eps = g.fmt.eps;
        std::vector<uint32_t> up(D->seg.size() * (sizeof(StreamSegment) / 4) + P.base.size()), steps(nvg);
        memcpy(up.data(), D->seg.data(), D->seg.size() * sizeof(StreamSegment));
        memcpy(up.data() + up.size() - P.base.size(), P.base.data(), P.base.size() * 4);
        hipError_t e = hipMemcpyAsync(at, up.data(), up.size() * 4, hipMemcpyHostToDevice, s);
        if (e != hipSuccess) return fail(SQ_ELAUNCH, "sq_stream_plan_device: %s", hipGetErrorString(e));
        launch_count_and_sort(P, tags, R, W, bits, G, row_book, (uint16_t*)counts, a, (int)D->seg.size(), s);
        int rc = check_launch("sq_stream_plan_device");
        e = hipMemcpyAsync(steps.data(), a.steps, nvg * 4, hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipStreamSynchronize(s);        // (also where the launch failed: the copy out of `up` has ended)
        if (rc) return rc;
        if (e != hipSuccess) return fail(SQ_ELAUNCH, "sq_stream_plan_device: %s", hipGetErrorString(e));
        plan_layout(steps.data(), P);
        if (g.total_steps >= ((uint64_t)1 << 32) || g.runs >= (1 << 16)) return fail(SQ_EUNSUPPORTED, "sq_stream_plan_device: matrix too large");
        D->bytes = g.off_steps + (size_t)g.total_steps * g.fmt.step_bytes;
        const uint32_t longest = nvg ? *std::max_element(steps.begin(), steps.end()) : 0u;
        D->in_lds = (size_t)longest * g.fmt.eps * STREAM_FILL_BYTES <= STREAM_FILL_LDS;
        // what the host uploads in one piece
        auto put = [&](const void* p, size_t n) {
            const uint32_t* w = (const uint32_t*)p;
            D->upload.insert(D->upload.end(), w, w + n / 4);
        };
        put(P.head4.data(), P.head4.size() * 4);
        put(P.runs.data(), P.runs.size() * sizeof(StreamRun));
        put(P.base.data(), P.base.size() * 4);
        D->at_goff = D->upload.size() * 4;
        put(P.goff.data(), P.goff.size() * 4);
        D->at_seg = D->upload.size() * 4;
        put(D->seg.data(), D->seg.size() * sizeof(StreamSegment));
        // scratch: that, the rows of the lanes, the counts, and the groups themselves when one is too long for LDS
        D->at_rows = align256(D->upload.size() * 4);
        D->at_cnt = align256(D->at_rows + nvg * 64 * 4);
        D->at_work = align256(D->at_cnt + (size_t)g.NV * R * 2);
        D->scratch = D->at_work + (D->in_lds ? 0 : (size_t)P.logical_steps * g.fmt.eps * STREAM_FILL_BYTES);
        *runs_out = runs_word(P);
        *groups_out = g.NG;
    }
    *bytes = D->bytes;
    *scratch = D->scratch;
    *out = D.release();
    return SQ_OK;
}

// Enqueues what writes the buffers.
static int launch_stream_fill(const StreamFill* fills, int n, hipStream_t s) {
    for (int i = 0; i < n; ++i) {
        const StreamDevicePlan& D = *fills[i].plan;
        if (D.tiled) continue;
        const hipError_t e = hipMemcpyAsync(fills[i].scratch, D.upload.data(), D.upload.size() * 4, hipMemcpyHostToDevice, s);
        if (e != hipSuccess) return fail(SQ_ELAUNCH, "sq_stream_fill_device: %s", hipGetErrorString(e));
    }
    StreamFillStack stack{};
    int wgs = 0;
    size_t lds = 0;
    auto fill = [&]() {
        if (stack.n == 0) return;
        if (lds) hipLaunchKernelGGL((stream_fill_kernel<true>), dim3((unsigned)wgs), dim3(256), lds, s, stack);
        else hipLaunchKernelGGL((stream_fill_kernel<false>), dim3((unsigned)wgs), dim3(256), 0, s, stack);
        stack.n = wgs = 0;
        lds = 0;
    };
    (void)hipFuncSetAttribute((const void*)stream_fill_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, STREAM_FILL_LDS);
    (void)hipGetLastError();
    for (int i = 0; i < n; ++i) {
        const StreamDevicePlan& D = *fills[i].plan;
        unsigned char *out = fills[i].out, *scratch = fills[i].scratch;
        if (D.tiled) {
            const int ud = unit_dwords(D.bits), U = row_units(D.C, D.d, D.bits);
            const int64_t units = (int64_t)((D.R + 15) / 16) * 16 * U;
            if (units > 0)
                hipLaunchKernelGGL(tiled_build_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0, s, fills[i].tags, D.R, D.W, U, ud, (uint32_t*)out);
            continue;
        }
        const StreamPlan& P = D.P;
        const StreamGeom& g = P.g;
        const size_t nvg = (size_t)g.NV * g.NG;
        const int64_t words = (int64_t)(D.bytes / 4);
        hipLaunchKernelGGL(stream_front_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s, (const uint32_t*)scratch, (int64_t)P.head4.size(),
                           (int64_t)(g.off_runs / 4), (int64_t)(P.runs.size() * sizeof(StreamRun) / 4), (int64_t)(g.off_rows / 4), (int64_t)P.base.size(),
                           (uint32_t*)out, words);
        StreamSortArgs b{};
        b.cnt = (uint16_t*)(scratch + D.at_cnt);
        b.base = (const uint32_t*)(out + g.off_rows);
        b.seg = (const StreamSegment*)(scratch + D.at_seg);
        b.rows = (uint32_t*)(scratch + D.at_rows);
        b.slots = (uint16_t*)(out + g.off_slots);
        b.R = D.R; b.NG = g.NG; b.eps = g.fmt.eps;
        launch_count_and_sort(P, fills[i].tags, D.R, D.W, D.bits, D.G, fills[i].row_book, (uint16_t*)(scratch + D.at_cnt), b, (int)D.seg.size(), s);
        uint32_t longest = 0;
        for (size_t k = 0; k < nvg; ++k) longest = std::max(longest, P.goff[k + 1] - P.goff[k]);
        // neighbours whose groups fit LDS, or neighbours whose do not, up to STREAM_FILL_PIECES
        if (stack.n == STREAM_FILL_PIECES || (stack.n && (lds != 0) != D.in_lds) || (int64_t)wgs + (int64_t)nvg >= ((int64_t)1 << 31)) fill();
        StreamFillArgs& a = stack.p[stack.n++];
        a.tags = fills[i].tags; a.row_book = fills[i].row_book;
        a.heads = (const uint32_t*)out;
        a.rows = b.rows;
        a.goff = (const uint32_t*)(scratch + D.at_goff);
        a.steps = out + g.off_steps;
        a.work = scratch + D.at_work;
        a.W = D.W; a.U = g.U; a.bits = D.bits; a.G = D.G; a.PC = g.PC; a.NS = g.NS; a.NV = g.NV; a.NG = g.NG; a.fs = g.fs;
        a.wg0 = wgs;
        wgs += (int)nvg;
        if (D.in_lds) lds = std::max({lds, (size_t)longest * g.fmt.eps * STREAM_FILL_BYTES, (size_t)16});
    }
    fill();
    return check_launch("sq_stream_fill_device");
}

// Slice streams are whole when this returns: the caller may free the plans, the scratch and the tags and may multiply on any stream.
// (Also where a launch failed: what was enqueued before it still reads the plans and writes the buffers.)  Tile-major copies by
// themselves are only enqueued: they have neither plan data nor scratch on their way, and a wait per matrix makes the start of a layer of them
// a fifth longer (14 matrices: 3.35 ms, with waits 4.0).
int stream_fill_device(const StreamFill* fills, int n, hipStream_t s) {
    const int rc = launch_stream_fill(fills, n, s);
    if (std::all_of(fills, fills + n, [](const StreamFill& f) { return f.plan->tiled; })) return rc;
    const hipError_t e = hipStreamSynchronize(s);
    if (rc || e == hipSuccess) return rc;
    return fail(SQ_ELAUNCH, "sq_stream_fill_device: %s", hipGetErrorString(e));
}

void stream_plan_free(StreamDevicePlan* D) { delete D; }

}  // namespace sq
