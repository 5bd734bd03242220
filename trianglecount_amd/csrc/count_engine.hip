// count_engine.hip -- persistent triangle-counting engine (gfx950, wave64).
//
// Count of a graph = sum over owned rows u of sum_{w in N+(u)} |N+(u) n N+(w)|
// (src/WithoutPartition/ShareKernelTCV62_update_v1.cu:43-191 summed as at
// :271-277; owned rows only as in src/WithPartition/without_sorting_tc.cu:400).
//
// Every arc (u, w) contributes |N+(u) n N+(w)|, found by hashing one list into
// LDS and streaming the other through it.  A work item hashes one row r:
//   kind A (source side): N+(r) hashed; the lists N+(w), w in N+(r), streamed.
//   kind B (target side): N+(r) hashed; the lists N+(u) of in-neighbours u
//            (from the graph's in-lists) streamed.
// With in-lists present ("split" counting) kind A keeps only arcs with
// d+(w) < d+(r) and kind B covers the rest (the in-lists hold exactly the arcs
// u -> w with d+(u) <= d+(w)), so each arc streams its shorter list.  Without
// in-lists every arc is a kind A arc.
//
// Plan (k_plan_rows): every planned row with d+ >= 2 emits its kind A item
// (source side; owned rows only) and kind B items (one kInChunk-source chunk of
// its in-list each), binned by the hashed row's d+ into one queue, largest bin
// first; rows with d+ <= tiny_max go to the tiny region
// instead.  Items of rows above small_max form "big" tickets (kBigGroup items each);
// smaller ones form "small" tickets of small_group items (by default chosen by
// the planner from the small items per workgroup).  k_count reads it from ctl.
// Launches of at most kSmallPlan rows are planned by one workgroup (k_plan_small).
//
// One graph large enough for it is counted from 16-bit hub codes instead
// (hubcode.h, hubplan.h, hubwalk.h; k_count_hub): its plan kernels write that
// walk's queue.  Batches, and graphs whose hubs the device finds to cover too
// few of their columns, are counted by k_count.
//
// Count (k_count, one persistent launch): each workgroup of WAVES waves (2, 4 or
// 8: the workgroup size is a tuning knob) starts with the ticket of its own number
// and takes the next from the atomic heads (see kHeads).
//   big item  : the whole workgroup builds one LDS hash table (up to 1024 slots
//               per wave: 4096 with 4 waves; load <= 1/2, longer rows are tiled)
//               and the waves split the 64-segment windows round-robin;
//   small item: one wave, a private 1024-slot slice of the same LDS.
// Walk of one window: one segment per lane (id, start, length), inclusive scan
// of lengths, empty segments compacted out; then the flat sequence of entries
// is consumed in rounds of UNROLL chunks of 64, whose segment ends the wave walks
// with uniform lane reads (a chunk inside one segment takes its base from a
// scalar; segwalk.h).  Rounds are software-pipelined: round r+1 is addressed and
// loaded (global loads, never FLAT) before round r is probed, lockstep over its
// UNROLL chunks.  Hits are counted per lane and reduced across the wave per
// item; the workgroup issues one uint64 atomic per graph it counted.
#include <mutex>
#include <unordered_map>

#include "count_engine.h"
#include "hubplan.h"
#include "hubwalk.h"
#include "segwalk.h"
#include "wave.h"

namespace lstc {

static constexpr uint32_t kEmpty = 0xFFFFFFFFu;
static constexpr uint32_t kNoId = 0xFFFFFFFEu;  // never a vertex id (ids < 2^32 - 2), never kEmpty
static constexpr uint32_t kSliceLog2 = 10;
static constexpr uint32_t kSlice = 1u << kSliceLog2;  // wave-private slice (small items)
// LDS table of a workgroup: one slice per wave; a big item uses all of it as one
// table (2^big_log2 slots), filled with at most half as many keys per tile.
template <int WAVES>
constexpr uint32_t big_log2() { return kSliceLog2 + (WAVES >= 8 ? 3 : WAVES >= 4 ? 2 : 1); }
template <int WAVES>
constexpr uint32_t tab_slots() { return 1u << big_log2<WAVES>(); }
static constexpr int kBins = 6;                       // hash-path bins
static constexpr int kTinyBin = kBins;                // the lane-per-arc rows
static constexpr int kSlots = kBins + 1;              // queue regions
static constexpr uint32_t kBigGroup = 2;              // big items per ticket

// Tickets are dealt in classes: ticket t belongs to class t % classes, and each
// class has its own head, on a 128-byte line of its own.  Workgroup b starts with
// ticket b (no atomic) and goes on with its class, then with the others' leftovers.
// A launch of a few hundred tickets then costs few atomics where every one of the
// resident workgroups used to ask the one head (1009-vertex uniform graph: k_count
// 39.5 -> 20 us), and launches of short items do not queue on one address.  Long items are
// balanced better by fewer classes (ms with 1, 4 and 8):
//   mixed batch of 66 graphs 3.02, -, 2.84; 64 RMAT s14 1.30, 1.02, 0.98; RMAT s16 0.21, 0.17, 0.17
//   8 Chung-Lu graphs of 100 thousand vertices 2.09, 2.11, 2.60; 8 RMAT s17 1.84, 1.88, 2.12;
//   4 RMAT s18 1.55, 1.54, 1.64; 16 RMAT s17 3.21, 2.89, 3.12; 2 RMAT s21 6.65, 6.19, 6.27
// so launches of graphs of kLongArcs arcs in the mean have kFewHeads.  Without in-lists the items
// are longer still (RMAT s21 5.38 with one class, 5.50 with 8; 8 RMAT s17 1.70, 1.96), and
// only launches below kShortArcs arcs have more than one class (20 thousand uniform vertices, 0.2M
// arcs, 0.076, 0.047; RMAT s15, 0.4M, 0.089, 0.073; s16, 0.9M, 0.155, 0.158).
static constexpr uint32_t kHeads = 8, kFewHeads = 4;
static constexpr uint64_t kLongArcs = 3ull << 19, kShortArcs = 1ull << 19;
static constexpr uint64_t kFineArcs = 400;  // arcs per ticket of single items on one head (plan_tickets)
static constexpr uint32_t kHeadStride = 32;  // words between heads

// ctl (uint32) layout
enum { C_CNT = 0, C_NBIG = 13, C_NSMALL = 14, C_NTICK = 15, C_NTINY = 16, C_TINY0 = 17, C_NSMALLT = 18,
       C_SGROUP = 19, C_CLASSES = 20, C_HEADS = 32, C_WORDS = C_HEADS + kHeads * kHeadStride };

// work item: row (bits 0-31) | chunk (32-51) | kind (52) | graph (53-63).
// A row's in-degree is below 2^32 (m < 2^32), so its chunk index fits 20 bits.
__device__ __forceinline__ unsigned long long make_item(uint32_t g, uint32_t kind, uint32_t chunk, uint32_t r) {
    return ((unsigned long long)g << 53) | ((unsigned long long)kind << 52) | ((unsigned long long)chunk << 32) | r;
}
struct Item {
    uint32_t row, chunk, kind, g;
};
__device__ __forceinline__ Item decode(unsigned long long it) {
    return Item{(uint32_t)it, (uint32_t)(it >> 32) & 0xFFFFFu, (uint32_t)(it >> 52) & 1u, (uint32_t)(it >> 53)};
}

TuneR resolve_tune(const lstc_tune *t) {
    // defaults: the fastest point of a (table_scale, small_max, grid_per_cu, unroll)
    // sweep at RMAT scales 16, 21 and 23 on MI355X (table_scale 6: rows of up to
    // 170 keys keep a wave-private table)
    TuneR r{6, 256, 0, 0, 4, kTinyMax, 4};  // small_group 0: chosen by the planner
    if (t) {
        if (t->tiny_max) r.tiny_max = t->tiny_max == 1 ? 0u : t->tiny_max;  // 1 = off
        if (t->table_scale) r.table_scale = t->table_scale;
        if (t->small_max) r.small_max = t->small_max;
        if (t->small_group) r.small_group = t->small_group;
        if (t->grid_per_cu) r.grid_per_cu = t->grid_per_cu;
        if (t->unroll) r.unroll = t->unroll;
        if (t->waves) r.waves = t->waves;
    }
    r.table_scale = hmax(2u, hmin(16u, r.table_scale));
    // a small row must fit its slice at the chosen load factor
    r.small_max = hmax(64u, hmin(kSlice / r.table_scale, r.small_max));
    if (r.small_group) r.small_group = hmax(4u, hmin(256u, r.small_group));
    r.unroll = r.unroll >= 8 ? 8 : 4;
    r.waves = r.waves >= 8 ? 8 : r.waves >= 4 ? 4 : 2;
    // default: 32 waves per CU (k_count fits them in LDS and VGPRs), 8 workgroups of 4 waves
    if (r.grid_per_cu == 0) r.grid_per_cu = 32 / r.waves;
    r.grid_per_cu = hmax(1u, hmin(32u, r.grid_per_cu));
    r.tiny_max = hmin(kTinyMax, r.tiny_max);
    if (r.tiny_max < 2) r.tiny_max = 0;
    return r;
}

// A launch of few arcs has few items per wave: rows above 128 keys then
// share a workgroup table, so their lists spread over four waves (RMAT s16,
// 0.9M arcs: 20% faster; no change from 2^23 arcs up, where the default keeps
// rows of up to 1024 / table_scale keys wave-private).  Only a default
// small_max is capped; an explicit one is kept.
TuneR effective_tune(const lstc_tune *t, uint64_t total_m) {
    TuneR r = resolve_tune(t);
    if ((!t || !t->small_max) && total_m < (1ull << 23) && r.small_max > 128) r.small_max = 128;
    return r;
}

lstc_status validate_graph(const HostGraph &h, const char *who) {
    if (h.n_owned > h.n_rows) return fail(LSTC_ERR_INVALID, "%s: n_owned %u > n_rows %u", who, h.n_owned, h.n_rows);
    if (h.n_rows == 0xFFFFFFFFu) return fail(LSTC_ERR_INVALID, "%s: n_rows must be < 2^32-1", who);
    if (h.m >= 0xFFFFF000ull)
        return fail(LSTC_ERR_INVALID, "%s: m = %llu arcs exceeds 2^32-4096", who, (unsigned long long)h.m);
    if (h.n_owned && (!h.off || (h.m && !h.col))) return fail(LSTC_ERR_INVALID, "%s: NULL CSR arrays", who);
    if ((h.in_off == nullptr) != (h.in_col == nullptr))
        return fail(LSTC_ERR_INVALID, "%s: give both in-list arrays or neither", who);
    if ((h.col_seg == nullptr) != (h.in_seg == nullptr))
        return fail(LSTC_ERR_INVALID, "%s: give both segment-word arrays or neither", who);
    if (h.col_seg && !h.in_off) return fail(LSTC_ERR_INVALID, "%s: segment words without in-lists", who);
    if (h.scol && (!h.col_seg || h.scol_len >= 0xFFFFF000ull))
        return fail(LSTC_ERR_INVALID, "%s: a streaming copy needs segment words and < 2^32-4096 entries", who);
    return LSTC_OK;
}

struct Bounds {
    uint32_t hi[kBins];  // bin b holds d+ in (hi[b-1], hi[b]], bin 0 starts at 2
    uint32_t tiny_max;   // rows of graphs with in-lists and 2 <= d+ <= tiny_max go to the tiny region
};

// UNIFORM: g is the same in every lane, so the entry is read through the
// scalar cache into scalar registers.
template <bool UNIFORM = false>
__device__ __forceinline__ GraphDev graph_at(const GraphSet &gs, uint32_t g) {
    if (!gs.table) return gs.one;
    if (UNIFORM) {
        const LSTC_CONST_AS GraphDev *q = (const LSTC_CONST_AS GraphDev *)(gs.table + g);
        GraphDev d;
        d.off = q->off;
        d.col = q->col;
        d.per_row = q->per_row;
        d.in_off = q->in_off;
        d.in_col = q->in_col;
        d.n_rows = q->n_rows;
        d.n_owned = q->n_owned;
        d.col_seg = q->col_seg;
        d.in_seg = q->in_seg;
        d.scol = q->scol;
        return d;
    }
    const LSTC_GLOBAL_AS GraphDev *q = (const LSTC_GLOBAL_AS GraphDev *)(gs.table + g);
    GraphDev d;
    d.off = q->off;
    d.col = q->col;
    d.per_row = q->per_row;
    d.in_off = q->in_off;
    d.in_col = q->in_col;
    d.n_rows = q->n_rows;
    d.n_owned = q->n_owned;
    d.scol = q->scol;
    return d;
}

__device__ __forceinline__ uint32_t table_log2_for(uint32_t keys, uint32_t scale, uint32_t max_log2) {
    uint32_t l = 6;
    while (l < max_log2 && (1u << l) < scale * keys) ++l;
    return l;
}

__device__ __forceinline__ uint64_t umin64(uint64_t a, uint64_t b) { return a < b ? a : b; }

// ------------------------------------------------------------------ planning
// The ticket counts of a plan whose regions hold n_big, n_small and n_tiny items
// (in this order in the queue), and what the count starts from: the heads behind
// the first `grid` tickets (the workgroups' own) and zero counts.  Run by one
// workgroup.
// small_group 0: the planner picks the small items per ticket, the largest
// power of two up to (small items per workgroup) / 32, within [16, 64]: about
// 32-64 small tickets per workgroup (measured on RMAT s21 and s23: fewer,
// larger tickets leave a ragged tail, more of them queue on the ticket heads).
// A launch with less than 16 small items per workgroup takes one per wave, so
// that its items spread over the chip (a 1009-vertex uniform graph has 2000), if that makes
// at most `fine` tickets: with one head, more of them queue on it unless the items are
// long (uniform graphs without in-lists, 16 / 1 item per wave: 30 thousand vertices of mean degree 40
// 0.054 / 0.108 ms, 15 thousand of 100 0.071 / 0.078, 20 thousand of 200 0.175 / 0.153).
__device__ __forceinline__ void plan_tickets(uint32_t *ctl, uint32_t n_big, uint32_t n_small, uint32_t n_tiny,
                                             uint32_t small_group, uint32_t grid, uint32_t waves, uint32_t classes,
                                             uint32_t fine, uint32_t tid) {
    if (tid < classes) ctl[C_HEADS + tid * kHeadStride] = (grid + classes - 1 - tid) / classes;
    if (tid != 0) return;
    ctl[C_CLASSES] = classes;
    uint32_t sg = small_group;
    if (sg == 0) {
        const uint32_t per_wg = n_small / (grid ? grid : 1u);
        sg = 16;
        while (sg < 64 && 2 * sg <= per_wg / 32) sg *= 2;
        if (per_wg < 16 && n_small <= (uint64_t)fine * waves) sg = waves;
    }
    ctl[C_SGROUP] = sg;
    const uint32_t small_t = (n_small + sg - 1) / sg;
    const uint32_t tiny_t = (n_tiny + waves * 64 - 1) / (waves * 64);  // 64 rows per wave
    ctl[C_NBIG] = n_big;
    ctl[C_NSMALL] = n_small;
    ctl[C_NSMALLT] = small_t;
    ctl[C_NTINY] = n_tiny;
    ctl[C_TINY0] = n_big + n_small;
    ctl[C_NTICK] = (n_big + kBigGroup - 1) / kBigGroup + small_t + tiny_t;
}

// The plan splits the owned rows of the launch (graph after graph) into
// kPlanWaves contiguous ranges, one per wave of the plan grid.  Pass 0 counts
// each range's items per bin into wcnt[slot][wave]; k_plan_scan turns that into
// exclusive queue positions (slot-major: bins 5,4,3 = big, largest first, then
// 2,1,0 = small); pass 1 writes the items, in row order within a bin and range.
// No atomics: the queue is the same on every run.
static constexpr uint32_t kPlanBlocks = 1012;
static constexpr uint32_t kPlanWaves = kPlanBlocks * 4;
static constexpr uint32_t kPlanEntries = kSlots * kPlanWaves;

// queue region of a bin: hash bins 5..0 in slots 0..5, the tiny rows in slot 6
__device__ __forceinline__ int slot_of(int b) { return b < kBins ? kBins - 1 - b : kTinyBin; }

// What one planned row puts into the queue.
struct RowPlan {
    int bin = -1;  // -1: nothing
    uint32_t g = 0, u = 0, n_a = 0, n_b = 0, tiny_kind = 0;
    __device__ __forceinline__ uint32_t items() const { return bin < 0 ? 0u : bin == kTinyBin ? 1u : n_a + n_b; }
    __device__ __forceinline__ void write(unsigned long long *q) const {
        if (bin == kTinyBin) {
            q[0] = make_item(g, tiny_kind, 0, u);
        } else {
            if (n_a) *q++ = make_item(g, 0, 0, u);
            for (uint32_t j = 0; j < n_b; ++j) q[j] = make_item(g, 1, j, u);
        }
    }
};

// Planned row r of the launch (r < total_rows); its graph is g0 or a later one.
__device__ __forceinline__ RowPlan plan_row(const GraphSet &gs, const Bounds &bd, uint64_t r, uint32_t g0 = 0) {
    RowPlan p;
    if (gs.table) {  // last g with row_base[g] <= r
        uint32_t lo = g0, hi = gs.G;
        if (r < gload(gs.row_base + lo + 1)) hi = lo + 1;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (gload(gs.row_base + mid) <= r) lo = mid; else hi = mid;
        }
        p.g = lo;
        p.u = (uint32_t)(r - gload(gs.row_base + lo));
    } else {
        p.u = (uint32_t)r;
    }
    const GraphDev G = graph_at(gs, p.g);
    const bool owned = p.u < G.n_owned;  // rows past n_owned are visited only for split counting
    const uint64_t k = gload(G.off + p.u + 1) - gload(G.off + p.u);
    const uint64_t kb = G.in_off ? gload(G.in_off + p.u + 1) - gload(G.in_off + p.u) : 0;
    if (k >= 2 && G.in_off && k <= bd.tiny_max) {
        // one entry; kind 1 = in side only (a halo row owns no out side)
        if (owned || kb) {
            p.bin = kTinyBin;
            p.tiny_kind = owned ? 0u : 1u;
        }
    } else if (k >= 2) {
        const uint32_t sb = in_chunk(kb);
        p.n_a = owned ? 1u : 0u;
        p.n_b = (uint32_t)((kb + sb - 1) / sb);
        if (p.n_a + p.n_b) {
            p.bin = kBins - 1;
            for (int i = kBins - 2; i >= 0; --i)
                if (k <= bd.hi[i]) p.bin = i;
        }
    }
    return p;
}

template <int PASS>
__global__ __launch_bounds__(256) void k_plan_rows(GraphSet gs, Bounds bd, uint32_t *__restrict__ wcnt,
                                                   unsigned long long *__restrict__ queue, HubSet hs) {
    if (hs.hctl && sload(hs.hctl + HC_ON)) return hub_plan_rows<PASS>(gs.one, hs);
    const uint32_t lane = lane_id();
    const uint32_t wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint64_t total = gs.total_rows;
    const uint64_t chunk = (total + kPlanWaves - 1) / kPlanWaves;
    const uint64_t r_begin = umin64(total, (uint64_t)wave * chunk), r_end = umin64(total, r_begin + chunk);
    uint32_t run[kSlots];
#pragma unroll
    for (int i = 0; i < kSlots; ++i) run[i] = PASS == 1 ? wcnt[slot_of(i) * kPlanWaves + wave] : 0u;
    uint32_t g0 = 0;  // graph of the range's last row so far
    for (uint64_t r0 = r_begin; r0 < r_end; r0 += 64) {
        const uint64_t r = r0 + lane;
        RowPlan p;
        if (r < r_end) p = plan_row(gs, bd, r, g0);
        g0 = read_lane(p.g, 63);  // (0 behind the range's end, where no row follows)
        const int b = p.bin;
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
            if (ballot(b == i) == 0) continue;
            const uint32_t c = (b == i) ? p.items() : 0u;
            if (PASS == 0) {
                run[i] += c;
            } else {
                const uint32_t incl = wave_incl_scan(c, lane);
                if (b == i) p.write(queue + run[i] + (incl - c));
                run[i] += read_lane(incl, 63);
            }
        }
    }
    if (PASS == 0) {
#pragma unroll
        for (int i = 0; i < kSlots; ++i) {
            const uint32_t sum = wave_sum32(run[i]);
            if (lane == 0) wcnt[slot_of(i) * kPlanWaves + wave] = sum;
        }
    }
}

// One workgroup of 1024: exclusive scan of wcnt in place (kPlanEntries values,
// 28 per thread), then the ticket counts.  Item totals stay below 2^32
// (checked on the host against the queue capacity).
__global__ __launch_bounds__(1024) void k_plan_scan(uint32_t *__restrict__ wcnt, uint32_t *__restrict__ ctl,
                                                    unsigned long long *__restrict__ counts, uint32_t G,
                                                    uint32_t small_group, uint32_t grid, uint32_t waves, uint32_t classes,
                                                    uint32_t fine, HubSet hs, uint32_t hub_grid) {
    if (hs.hctl && sload(hs.hctl + HC_ON)) return hub_plan_scan(hs, counts, hub_grid);
    constexpr uint32_t kPer = (kPlanEntries + 4095) / 4096 * 4;  // 16-byte loads and stores
    static_assert(kPlanEntries % 4 == 0, "plan entries come in whole 16-byte words");
    __shared__ uint32_t s_wave[16];
    __shared__ uint32_t s_slot[kSlots + 1];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    uint32_t v[kPer];
#pragma unroll
    for (uint32_t i = 0; i < kPer; i += 4) {
        const uint32_t e = tid * kPer + i;
        const uint4 q = e < kPlanEntries ? *(const uint4 *)(wcnt + e) : uint4{0, 0, 0, 0};
        v[i] = q.x, v[i + 1] = q.y, v[i + 2] = q.z, v[i + 3] = q.w;
    }
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        sum += v[i];
    }
    const uint32_t incl = wave_incl_scan(sum, lane);
    if (lane == 63) s_wave[wv] = incl;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < wv; ++w) before += s_wave[w];
    uint32_t run = before + incl - sum;
#pragma unroll
    for (uint32_t i = 0; i < kPer; ++i) {
        const uint32_t e = tid * kPer + i;
        if (e < kPlanEntries && e % kPlanWaves == 0) s_slot[e / kPlanWaves] = run;
        const uint32_t x = v[i];
        v[i] = run;
        run += x;
    }
#pragma unroll
    for (uint32_t i = 0; i < kPer; i += 4) {
        const uint32_t e = tid * kPer + i;
        if (e < kPlanEntries) *(uint4 *)(wcnt + e) = uint4{v[i], v[i + 1], v[i + 2], v[i + 3]};
    }
    if (tid == 1023) s_slot[kSlots] = run;
    __syncthreads();
    for (uint32_t i = tid; i < G; i += 1024) counts[i] = 0;
    // slots 0..2 hold bins 5,4,3 (big), slots 3..5 bins 2,1,0 (small), slot 6 the tiny rows
    plan_tickets(ctl, s_slot[3], s_slot[6] - s_slot[3], s_slot[7] - s_slot[6], small_group, grid, waves, classes, fine, tid);
}

// The whole plan of a launch of at most kSmallPlan rows in one workgroup: the
// same queue regions (rows in another order within a bin), one launch instead of
// three, each of which would cost more than the work of this one.
static constexpr uint32_t kSmallPlanPer = 4;
static constexpr uint32_t kSmallPlan = 1024 * kSmallPlanPer;

__global__ __launch_bounds__(1024) void k_plan_small(GraphSet gs, Bounds bd, uint32_t *__restrict__ ctl,
                                                     unsigned long long *__restrict__ queue,
                                                     unsigned long long *__restrict__ counts, uint32_t small_group,
                                                     uint32_t grid, uint32_t waves, uint32_t classes, uint32_t fine) {
    __shared__ uint32_t s_wave[kSlots][16];
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    RowPlan p[kSmallPlanPer];
#pragma unroll
    for (uint32_t i = 0; i < kSmallPlanPer; ++i) {
        const uint64_t r = (uint64_t)i * 1024 + tid;
        if (r < gs.total_rows) p[i] = plan_row(gs, bd, r);
    }
    uint32_t mine[kSlots], excl[kSlots];  // this thread's items per slot, and its place within the wave
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        uint32_t c = 0;
#pragma unroll
        for (uint32_t i = 0; i < kSmallPlanPer; ++i) c += p[i].bin >= 0 && slot_of(p[i].bin) == s ? p[i].items() : 0u;
        const uint32_t incl = wave_incl_scan(c, lane);
        mine[s] = c;
        excl[s] = incl - c;
        if (lane == 63) s_wave[s][wv] = incl;
    }
    __syncthreads();
    uint32_t base = 0, n_big = 0, n_small = 0;  // first queue position of the slot
#pragma unroll
    for (int s = 0; s < kSlots; ++s) {
        uint32_t before = 0, total = 0;
        for (uint32_t w = 0; w < 16; ++w) {
            const uint32_t v = s_wave[s][w];
            before += w < wv ? v : 0u;
            total += v;
        }
        uint32_t pos = base + before + excl[s];
        if (mine[s]) {
#pragma unroll
            for (uint32_t i = 0; i < kSmallPlanPer; ++i) {
                if (p[i].bin < 0 || slot_of(p[i].bin) != s) continue;
                p[i].write(queue + pos);
                pos += p[i].items();
            }
        }
        base += total;
        if (s == 2) n_big = base;
        if (s == 5) n_small = base - n_big;
    }
    for (uint32_t i = tid; i < gs.G; i += 1024) counts[i] = 0;
    plan_tickets(ctl, n_big, n_small, base - n_big - n_small, small_group, grid, waves, classes, fine, tid);
}

// ------------------------------------------------------------------ table build
// A key whose home bucket is full moves on; its home is then marked in the
// overflow bitmap `ovf` (one bit per bucket).  table_mark afterwards records
// the mark in the bucket itself by the order of its first two slots (an
// overflowed bucket is full: slot 0 > slot 1; any other: slot 0 < slot 1, or
// an empty slot 1), so a probe learns from its one bucket read whether a key
// of that home can lie further on.
__device__ __forceinline__ void table_insert(uint32_t *tab, uint32_t *ovf, uint32_t tlog2,
                                             const uint32_t *__restrict__ col, uint64_t b0, uint32_t nk, uint32_t tid,
                                             uint32_t nthreads) {
    const uint32_t qmask = (1u << (tlog2 - 2)) - 1, qshift = 34 - tlog2;
    for (uint32_t j = tid; j < nk; j += nthreads) {
        const uint32_t key = gload(col + b0 + j);
        const uint32_t home = hquad(key, qshift);
        uint32_t h = home;
        // A slot is tried only once the ones before it in the bucket are taken.
        // At most 1/2 of the slots are filled, so a free slot lies within one
        // lap of the buckets; the lap bound makes the loop finite by
        // construction as well.
        for (uint32_t step = 0; step <= qmask; ++step) {
            uint32_t *b = tab + 4 * h;
            if (atomicCAS(b, kEmpty, key) == kEmpty || atomicCAS(b + 1, kEmpty, key) == kEmpty ||
                atomicCAS(b + 2, kEmpty, key) == kEmpty || atomicCAS(b + 3, kEmpty, key) == kEmpty)
                break;
            h = (h + 1) & qmask;
        }
        if (h != home) atomicOr(ovf + (home >> 5), 1u << (home & 31u));
    }
}

// Orders the first two slots of every bucket by its overflow mark (the keys
// stay in the bucket, so every chain and membership is unchanged).
__device__ __forceinline__ void table_mark(uint32_t *tab, const uint32_t *ovf, uint32_t tlog2, uint32_t tid,
                                           uint32_t nthreads) {
    for (uint32_t b = tid; b < (1u << (tlog2 - 2)); b += nthreads) {
        const uint2 v = *(const uint2 *)(tab + 4 * b);
        const bool over = (ovf[b >> 5] >> (b & 31u)) & 1u;
        if (over ? v.x < v.y : v.x > v.y) *(uint2 *)(tab + 4 * b) = uint2{v.y, v.x};
    }
}

// ------------------------------------------------------------------ walk
// Probes one round through tab: linear probing over 4-slot buckets, the
// first bucket of all UNROLL chunks in lockstep, one 16-byte LDS read per
// chunk.  A lane is done once it hits or reads a bucket whose last slot is
// empty (no chain continues past such a bucket; tables are at most half full,
// so every chain has one).  Positions past the window's end carry an id that
// no table holds (kNoId: ids are below 2^32 - 2).
// Each compare is balloted on its own (a ballot of one compare is the
// compare's lane mask; a ballot of a combined condition would go through a
// VGPR), the masks are combined in scalar registers, and the hit mask is added
// to the per-lane counter as the carry-in of one vector add.  The few lanes
// whose chain goes on (about one lane in a hundred at the default table scale)
// are queued (their ids) in the window's segment table, which the rounds no
// longer read (bases and ends are in registers), and probed 64 at a time when
// the queue fills and at the window's end.
__device__ __forceinline__ uint64_t bucket_hits(const uint4 &v, uint32_t x) {
    return ballot(v.x == x) | ballot(v.y == x) | ballot(v.z == x) | ballot(v.w == x);
}

// Probes the queued lanes of a window (ids qx[i], i < qn, whose home bucket
// was full without a hit) as one chunk, from the bucket after their home to
// the end of their chains.
__device__ __forceinline__ void drain_queue(const uint4 *buckets, uint32_t qmask, uint32_t qshift, uint32_t lane,
                                            uint32_t &lane_hits, const uint32_t *qx, uint32_t qn) {
    const bool act = lane < qn;
    const uint32_t xv = act ? qx[lane] : kNoId;
    uint32_t q = (hquad(xv, qshift) + 1u) & qmask;
    uint64_t live = ballot(act);
    // Every chain ends at a hit or at a bucket whose last slot is empty: slots
    // fill in order, so a bucket with its last slot taken is full, and with at
    // most 1/2 of the slots filled at least half of the buckets end chains.
    // A chain therefore ends within one lap; the lap bound keeps the loop
    // finite by construction as well.
    for (uint32_t step = 0; live != 0 && step < qmask; ++step) {
        const uint4 w = buckets[q];
        const uint64_t H = bucket_hits(w, xv) & live;
        add_lane_bit(lane_hits, H);
        live &= ~(H | ballot(w.w == kEmpty));
        q = (q + 1) & qmask;
    }
}

template <int UNROLL, bool FULL>
__device__ __forceinline__ void probe_round(const uint32_t (&xin)[UNROLL], uint32_t B, uint32_t total, const uint32_t *tab,
                                            uint32_t qmask, uint32_t qshift, uint32_t lane, uint32_t &lane_hits,
                                            uint32_t *qx, uint32_t &qn) {
    const uint4 *buckets = (const uint4 *)tab;
    const uint64_t active = ballot(true);
    uint32_t x[UNROLL], p[UNROLL];
#pragma unroll
    for (int k = 0; k < UNROLL; ++k) {
        x[k] = FULL || B + 64u * k + lane < total ? xin[k] : kNoId;
        p[k] = hquad(x[k], qshift);
    }
    uint4 v[UNROLL];
#pragma unroll
    for (int k = 0; k < UNROLL; ++k) v[k] = buckets[p[k]];
    // lanes whose chain goes on (bits of inactive lanes may be set here; they
    // are masked off below)
    uint64_t going[UNROLL], any = 0;
#pragma unroll
    for (int k = 0; k < UNROLL; ++k) {
        const uint64_t H = bucket_hits(v[k], x[k]);
        add_lane_bit(lane_hits, H);
        going[k] = ~(H | ballot(v[k].x <= v[k].y));  // no hit and the home bucket overflowed
        any |= going[k];
    }
    if ((any & active) == 0) return;
    // queue them (id, next bucket); a full queue is probed first
#pragma unroll
    for (int k = 0; k < UNROLL; ++k) {
        const uint64_t g = going[k] & active;
        if (g != 0) {
            const uint32_t c = (uint32_t)__popcll(g);
            if (qn + c > 64u) {
                drain_queue(buckets, qmask, qshift, lane, lane_hits, qx, qn);
                qn = 0;
            }
            if (lane_in(g)) qx[qn + mask_rank(g)] = x[k];
            qn += c;
        }
    }
}

// Streams the lists N+(s) of the segment ids s = seg[j], j in [w0, nseg) step
// wstep (windows of 64), through tab.  A segment whose list is not shorter than
// `below` is skipped (below = 0: none skipped); ids >= n_rows have no list.
// With segment words (segw[j] = start | length << 32 of N+(seg[j])) a window
// reads one coalesced word per segment instead of two row offsets at a random
// place, and the next window's words are loaded while this one streams.
// Rounds are software-pipelined over two buffers: the loads of round r+1 are
// issued before round r is probed, so a wave keeps up to 2*UNROLL chunk loads
// in flight.
template <int UNROLL, bool NARROW>
__device__ __forceinline__ uint32_t walk(const uint64_t *__restrict__ off, const uint32_t *__restrict__ col,
                                                   uint32_t n_rows, const uint32_t *__restrict__ seg,
                                                   const uint64_t *__restrict__ segw, uint32_t nseg_all,
                                                   uint32_t below, uint32_t w0, uint32_t wstep, const uint32_t *tab,
                                                   uint32_t tlog2, uint32_t *s_base, uint32_t *s_end,
                                                   uint32_t lane) {
    constexpr uint32_t RB = 64u * UNROLL;
    const uint32_t qmask = (1u << (tlog2 - 2)) - 1, qshift = 34 - tlog2;
    uint32_t lane_hits = 0;
    // the next window's segment words are loaded while this window streams
    uint64_t sw_next = segw && w0 + lane < nseg_all ? gload(segw + w0 + lane) : 0;
    for (uint32_t j0 = w0; j0 < nseg_all; j0 += wstep) {
        const uint32_t j = j0 + lane;
        uint32_t s = 0, len = 0;
        if (segw) {
            const uint64_t sw = sw_next;  // one coalesced word: start | length << 32 (0 past the end)
            s = (uint32_t)sw;
            len = (uint32_t)(sw >> 32);
            if (below && len >= below) len = 0;  // that arc is counted from the other side
            sw_next = j + wstep < nseg_all ? gload(segw + j + wstep) : 0;
        } else if (j < nseg_all) {
            const uint32_t w = gload(seg + j);
            if (w < n_rows) {
                const uint64_t s0 = gload(off + w);
                s = (uint32_t)s0;
                len = (uint32_t)(gload(off + w + 1) - s0);
            }
            if (below && len >= below) len = 0;
        }
        const uint32_t incl = wave_incl_scan(len, lane);
        const uint32_t total = uniform(gather(incl, 63));
        if (total == 0) continue;
        const uint64_t nzm = ballot(len != 0);
        const uint32_t nseg = (uint32_t)__popcll(nzm);
        if (len != 0) {
            const uint32_t slot = mask_rank(nzm);
            s_base[slot] = s - (incl - len);
            s_end[slot] = incl;
        }
        const uint32_t mybase = s_base[lane];
        const uint32_t myend = lane < nseg ? s_end[lane] : kEmpty;
        uint32_t xa[UNROLL], xb[UNROLL];
        uint32_t qn = 0;  // queued lanes (in s_base from here on)
        // Each round's indices come from one of three cases (inside one
        // segment, crossed by segment ends, the window's partial last round);
        // the loads and the probe follow in one common path, so the two
        // buffers keep their registers and the wait for the probed buffer
        // never covers the loads just issued.
        uint32_t idx[UNROLL];
        {
            const uint32_t sg = first_segment(0, myend);
            if (RB > total)
                index_walk<UNROLL, false, col_shift<NARROW>()>(0, total, mybase, myend, sg, lane, idx);
            else if (one_segment<UNROLL>(0, myend))
                index_single<UNROLL, col_shift<NARROW>()>((uint32_t)__builtin_amdgcn_readlane((int)mybase, (int)sg), lane, idx);
            else
                index_walk<UNROLL, true, col_shift<NARROW>()>(0, total, mybase, myend, sg, lane, idx);
        }
        load_round<UNROLL, NARROW>(col, idx, xa);
        uint32_t B = 0;
        for (; B + 3 * RB <= total; B += 2 * RB) {
            // rounds B + RB and B + 2 * RB are full
            uint32_t sg = first_segment(B + RB, myend);
            if (one_segment<UNROLL>(B + RB, myend))
                index_single<UNROLL, col_shift<NARROW>()>((uint32_t)__builtin_amdgcn_readlane((int)mybase, (int)sg) + B + RB, lane, idx);
            else
                index_walk<UNROLL, true, col_shift<NARROW>()>(B + RB, total, mybase, myend, sg, lane, idx);
            load_round<UNROLL, NARROW>(col, idx, xb);
            probe_round<UNROLL, true>(xa, B, total, tab, qmask, qshift, lane, lane_hits, s_base, qn);
            sg = first_segment(B + 2 * RB, myend);
            if (one_segment<UNROLL>(B + 2 * RB, myend))
                index_single<UNROLL, col_shift<NARROW>()>((uint32_t)__builtin_amdgcn_readlane((int)mybase, (int)sg) + B + 2 * RB, lane,
                                     idx);
            else
                index_walk<UNROLL, true, col_shift<NARROW>()>(B + 2 * RB, total, mybase, myend, sg, lane, idx);
            load_round<UNROLL, NARROW>(col, idx, xa);
            probe_round<UNROLL, true>(xb, B + RB, total, tab, qmask, qshift, lane, lane_hits, s_base, qn);
        }
        // Tail: round B is in xa; rounds B + RB and B + 2 * RB may follow
        // (B + 3 * RB > total, so the last one is partial).
        if (B + RB >= total) {
            probe_round<UNROLL, false>(xa, B, total, tab, qmask, qshift, lane, lane_hits, s_base, qn);
        } else {
            index_walk<UNROLL, false, col_shift<NARROW>()>(B + RB, total, mybase, myend, first_segment(B + RB, myend), lane, idx);
            load_round<UNROLL, NARROW>(col, idx, xb);
            probe_round<UNROLL, true>(xa, B, total, tab, qmask, qshift, lane, lane_hits, s_base, qn);
            if (B + 2 * RB < total) {
                index_walk<UNROLL, false, col_shift<NARROW>()>(B + 2 * RB, total, mybase, myend, first_segment(B + 2 * RB, myend), lane,
                                          idx);
                load_round<UNROLL, NARROW>(col, idx, xa);
                probe_round<UNROLL, true>(xb, B + RB, total, tab, qmask, qshift, lane, lane_hits, s_base, qn);
                probe_round<UNROLL, false>(xa, B + 2 * RB, total, tab, qmask, qshift, lane, lane_hits, s_base, qn);
            } else {
                probe_round<UNROLL, false>(xb, B + RB, total, tab, qmask, qshift, lane, lane_hits, s_base, qn);
            }
        }
        // the next window rewrites the segment tables
        if (qn != 0) drain_queue((const uint4 *)tab, qmask, qshift, lane, lane_hits, s_base, qn);
    }
    // an item streams at most m < 2^32 entries, so its hits fit 32 bits
    return wave_sum32(lane_hits);
}

// The segment source of a work item: kind A walks N+(r) with the split filter,
// kind B walks one chunk of r's in-list unfiltered.
struct Segs {
    const uint32_t *ids;
    const uint64_t *seg;  // the ids' segment words, or null
    uint32_t n;
    uint32_t below;
};

__device__ __forceinline__ Segs item_segs(const GraphDev &G, uint32_t kind, uint32_t chunk, uint32_t r, uint64_t rb,
                                          uint32_t K) {
    if (kind == 0) return Segs{G.col + rb, G.col_seg ? G.col_seg + rb : nullptr, K, G.in_off ? K : 0u};
    const uint64_t ib = sload(G.in_off + r), ie = sload(G.in_off + r + 1);
    const uint32_t sb = in_chunk(ie - ib);
    const uint64_t c0 = ib + (uint64_t)chunk * sb;
    const uint64_t c1 = (c0 + sb < ie) ? c0 + sb : ie;
    return Segs{G.in_col + c0, G.in_seg ? G.in_seg + c0 : nullptr, (uint32_t)(c1 - c0), 0u};
}

// ------------------------------------------------------------------ tiny rows
// Rows with 2 <= d+ <= tiny_max of a graph with in-lists.  Under the split rule
// every arc such a row r owns joins two lists of at most d+(r) entries:
//   out side: arcs (r, x) with d+(x) < d+(r), from N+(r);
//   in side : arcs (u, r) from r's in-list (d+(u) <= d+(r)).
// So each arc is one lane's job: compare the two lists, at most kTinyMax^2
// equality tests, no hash table and no probing.  The wave's lanes hold up to 64
// rows of graph G (mine); their lists are staged once in the wave's LDS slice
// (row of lane i at tab[i*kTinyMax ...]), then their out-sides and in-sides are
// walked flat, 64 arcs per step, with the same end-marking as the hash walk.
// Each lane loads the other list of its arc into registers.
__device__ __forceinline__ uint32_t tiny_walk(const GraphDev &G, bool mine, bool out_side, uint32_t r, uint32_t *tab,
                                              uint32_t *s_base, uint32_t *s_end, uint8_t *s_src, uint8_t *flag,
                                              uint32_t lane) {
    uint32_t ro = 0, rd = 0;  // this lane's row: start and length of N+(r)
    if (mine) {
        const uint64_t o0 = gload(G.off + r);
        ro = (uint32_t)o0;
        rd = (uint32_t)(gload(G.off + r + 1) - o0);
#pragma unroll
        for (uint32_t j = 0; j < kTinyMax; ++j)
            if (j < rd) tab[lane * kTinyMax + j] = gload(G.col + ro + j);
    }
    uint32_t lane_hits = 0;
#pragma unroll 1
    for (int side = 0; side < 2; ++side) {
        uint32_t s = 0, len = 0;
        if (mine) {
            if (side == 0) {
                s = ro;
                len = out_side ? rd : 0u;
            } else {
                const uint64_t i0 = gload(G.in_off + r);
                s = (uint32_t)i0;
                len = (uint32_t)(gload(G.in_off + r + 1) - i0);
            }
        }
        const uint32_t *list = side == 0 ? G.col : G.in_col;
        const uint32_t incl = wave_incl_scan(len, lane);
        const uint32_t total = uniform(gather(incl, 63));
        if (total == 0) continue;
        const uint64_t nzm = ballot(len != 0);
        const uint32_t nseg = (uint32_t)__popcll(nzm);
        if (len != 0) {
            const uint32_t slot = mask_rank(nzm);
            s_base[slot] = s - (incl - len);
            s_end[slot] = incl;
            s_src[slot] = (uint8_t)lane;
        }
        const uint32_t mybase = s_base[lane];
        const uint32_t myend = lane < nseg ? s_end[lane] : kEmpty;
        const uint32_t mysrc = s_src[lane];
        for (uint32_t B = 0; B < total; B += 64) {
            uint32_t sg = (uint32_t)__popcll(ballot(myend <= B));
            const bool mk = myend > B && myend < B + 64;
            if (mk) flag[myend - B] = 1;
            const uint64_t M = ballot(flag[lane] != 0);
            if (mk) flag[myend - B] = 0;
            if (M != 0) sg += (uint32_t)__popcll(M & ((2ull << lane) - 1ull));
            sg &= 63u;  // lanes past the end take some owner; their arc is not counted
            const uint32_t base = gather(mybase, sg), src = gather(mysrc, sg);
            const uint32_t t = B + lane;
            const uint32_t x = gload(t < total ? list + (uint32_t)(base + t) : list);
            const uint32_t ard = gather(rd, src);
            // x's list: with segment words, the arc's own word (coalesced) gives its start in the
            // streamed array (the row-aligned copy, or col) and d+(x); else two row offsets
            const uint64_t *words = side == 0 ? G.col_seg : G.in_seg;
            const uint32_t *xl = words ? G.scol : G.col;
            uint32_t xo, xd;
            if (words) {
                const uint64_t w = gload(t < total ? words + (uint32_t)(base + t) : words);
                xo = (uint32_t)w;
                xd = t < total ? (uint32_t)(w >> 32) : 0u;  // 0 for ids that are no row
            } else {
                const uint32_t xi = t < total ? x : 0u;
                const uint64_t xo0 = gload(G.off + xi);
                xo = (uint32_t)xo0;
                xd = (uint32_t)(gload(G.off + xi + 1) - xo0);
            }
            // the out side keeps d+(x) < d+(r); the in side holds only d+(x) <= d+(r)
            const bool live = t < total && xd != 0 && (side == 1 || xd < ard);
            uint32_t b[kTinyMax];
#pragma unroll
            for (uint32_t j = 0; j < kTinyMax; ++j)  // unconditional, in bounds (xl[0] when unused)
                b[j] = gload(live && j < xd ? xl + xo + j : xl);
            if (live) {
                const uint32_t *a = tab + src * kTinyMax;
                uint32_t c = 0;
#pragma unroll
                for (uint32_t i = 0; i < kTinyMax; ++i) {
                    if (i < ard) {
                        const uint32_t ai = a[i];
#pragma unroll
                        for (uint32_t j = 0; j < kTinyMax; ++j) c += (j < xd && ai == b[j]) ? 1u : 0u;
                    }
                }
                lane_hits += c;
            }
        }
    }
    return wave_sum32(lane_hits);
}

// ------------------------------------------------------------------ tickets
// One thread's view of the ticket heads: its class's next ticket, and when that
// class has run out, the other classes' leftovers, each class left for good once
// it is empty (kEmpty when none is left).  Asking before the current ticket's work
// rather than after it was slower (s23 17.06 against 16.90 ms): the loads of the
// asking wave wait behind the atomic.
struct Tickets {
    uint32_t *heads;
    uint32_t n, classes, cls;
    __device__ __forceinline__ Tickets(uint32_t *ctl, uint32_t n_tickets)
        : heads(ctl + C_HEADS), n(n_tickets), classes(sload(ctl + C_CLASSES)), cls(blockIdx.x % classes) {}
    // A head never passes its class's ticket count by more than the workgroups
    // asking, so a ticket number stays below 2^32.
    __device__ __forceinline__ uint32_t next() {
        if (n <= gridDim.x) return kEmpty;  // every ticket was some workgroup's first
        uint64_t t = (uint64_t)atomicAdd(heads + cls * kHeadStride, 1u) * classes + cls;
        for (uint32_t left = classes - 1; t >= n && left; --left) {
            cls = cls + 1 == classes ? 0 : cls + 1;
            uint32_t *head = heads + cls * kHeadStride;
            const uint32_t h = __hip_atomic_load(head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((uint64_t)h * classes + cls < n) t = (uint64_t)atomicAdd(head, 1u) * classes + cls;
        }
        return t < n ? (uint32_t)t : kEmpty;
    }
};

// One atomic per graph per workgroup for what its waves still hold.
template <int WAVES>
__device__ __forceinline__ void flush_counts(unsigned long long *counts, unsigned long long *s_acc, uint32_t *s_g,
                                             unsigned long long acc, uint32_t cur_g, uint32_t tid, uint32_t wv,
                                             uint32_t lane) {
    if (lane == 0) { s_acc[wv] = acc; s_g[wv] = cur_g; }
    __syncthreads();
    if (tid == 0) {
        for (int i = 0; i < WAVES; ++i) {
            if (s_g[i] == kEmpty) continue;
            unsigned long long sum = s_acc[i];
            for (int j = i + 1; j < WAVES; ++j)
                if (s_g[j] == s_g[i]) { sum += s_acc[j]; s_g[j] = kEmpty; }
            if (sum) atomicAdd(counts + s_g[i], sum);
        }
    }
}

// ------------------------------------------------------------------ persistent count kernel
// NARROW: every graph of the launch has m <= 2^30 arcs (and a streaming copy of at
// most 2^30 entries).
// Occupancy target (the second launch bound is waves per SIMD): 8 with UNROLL 4,
// 6 with UNROLL 8, whatever the workgroup size.
template <int UNROLL, bool NARROW, int WAVES>
__global__ __launch_bounds__(WAVES * 64, UNROLL == 4 ? 8 : 6) void k_count(GraphSet gs, const unsigned long long *__restrict__ queue,
                                                       uint32_t *__restrict__ ctl,
                                                       unsigned long long *__restrict__ counts, uint32_t scale,
                                                       const uint32_t *__restrict__ skip) {
    constexpr uint32_t kTab = tab_slots<WAVES>();
    __shared__ __align__(16) uint32_t s_tab[kTab];
    __shared__ uint32_t s_ovf[kTab / 128];  // overflow bits, one per 4-slot bucket
    __shared__ uint32_t s_base[WAVES][64];
    __shared__ uint32_t s_end[WAVES][64];
    __shared__ __align__(16) uint32_t s_flag[WAVES][16];  // 64 position flags per wave (tiny rows)
    __shared__ uint8_t s_src[WAVES][64];
    __shared__ uint32_t s_ticket[2];
    __shared__ unsigned long long s_acc[WAVES];
    __shared__ uint32_t s_g[WAVES];

    // item and graph fields are wave-uniform: they live in scalar registers
    const uint32_t tid = threadIdx.x, wv = uniform(tid >> 6), lane = tid & 63;
    if (skip && sload(skip)) return;  // the launch is counted by k_count_hub
    if (lane < 16) s_flag[wv][lane] = 0;
    const uint32_t n_big = sload(ctl + C_NBIG), n_small = sload(ctl + C_NSMALL), n_tickets = sload(ctl + C_NTICK);
    const uint32_t n_bigt = (n_big + kBigGroup - 1) / kBigGroup;  // big tickets
    const uint32_t small_end = n_bigt + sload(ctl + C_NSMALLT);  // first tiny ticket
    const uint32_t small_group = sload(ctl + C_SGROUP);
    const uint32_t tiny0 = sload(ctl + C_TINY0), tiny_end = tiny0 + sload(ctl + C_NTINY);
    uint32_t cur_g = kEmpty;
    unsigned long long acc = 0;

    Tickets tk(ctl, n_tickets);
    uint32_t turn = 0;
    for (uint32_t t = blockIdx.x; t < n_tickets;) {
        if (t < n_bigt) {
          // big items (kBigGroup per ticket): the whole workgroup shares one table
          for (uint32_t bi = t * kBigGroup, be = min(bi + kBigGroup, n_big); bi < be; ++bi) {
            const Item itm = decode(sload(queue + bi));
            const uint32_t u = itm.row, chunk = itm.chunk, kind = itm.kind, g = itm.g;
            const GraphDev G = graph_at<true>(gs, g);
            const uint64_t rb = sload(G.off + u);
            const uint32_t K = (uint32_t)(sload(G.off + u + 1) - rb);
            const Segs sg = item_segs(G, kind, chunk, u, rb, K);
            unsigned long long hits = 0;
            constexpr uint32_t kBigTile = kTab / 2;  // keys per table fill of a big row
            for (uint32_t t0 = 0; t0 < K; t0 += kBigTile) {
                const uint32_t tk = min(K - t0, kBigTile);
                const uint32_t tl = table_log2_for(tk, scale, big_log2<WAVES>());
                for (uint32_t i = tid; i < (1u << tl); i += WAVES * 64) s_tab[i] = kEmpty;
                if (tid < kTab / 128) s_ovf[tid] = 0;
                __syncthreads();
                table_insert(s_tab, s_ovf, tl, G.col, rb + t0, tk, tid, WAVES * 64);
                __syncthreads();
                table_mark(s_tab, s_ovf, tl, tid, WAVES * 64);
                __syncthreads();
                hits += walk<UNROLL, NARROW>(G.off, sg.seg ? G.scol : G.col, G.n_rows, sg.ids, sg.seg, sg.n, sg.below, wv * 64, WAVES * 64, s_tab, tl,
                                     s_base[wv], s_end[wv], lane);
                __syncthreads();
            }
            if (g != cur_g) {
                if (cur_g != kEmpty && acc != 0 && lane == 0) atomicAdd(counts + cur_g, acc);
                cur_g = g;
                acc = 0;
            }
            acc += hits;
            if (G.per_row && lane == 0 && hits) atomicAdd(G.per_row + u, hits);
          }
        } else if (t >= small_end) {
            // tiny rows: 64 per wave, lane-per-arc; the lanes are split by graph
            const uint32_t e0 = tiny0 + (t - small_end) * (WAVES * 64) + wv * 64;
            const uint32_t e = e0 + lane;
            const bool valid = e < tiny_end;
            Item itm{0, 0, 0, 0};
            if (valid) itm = decode(gload(queue + e));
            uint64_t rem = ballot(valid);
            while (rem) {
                const uint32_t g = read_lane(itm.g, (uint32_t)__builtin_ctzll(rem));
                const bool mine = valid && itm.g == g;
                rem &= ~ballot(mine);
                const GraphDev G = graph_at<true>(gs, g);
                const uint32_t hits = tiny_walk(G, mine, mine && itm.kind == 0, itm.row, s_tab + wv * kSlice,
                                                s_base[wv], s_end[wv], s_src[wv], (uint8_t *)s_flag[wv], lane);
                if (g != cur_g) {
                    if (cur_g != kEmpty && acc != 0 && lane == 0) atomicAdd(counts + cur_g, acc);
                    cur_g = g;
                    acc = 0;
                }
                acc += hits;
            }
        } else {
            // small items: each wave takes every WAVES-th item of the group
            const uint32_t first = n_big + (t - n_bigt) * small_group;
            const uint32_t last = min(first + small_group, n_big + n_small);
            uint32_t *tab = s_tab + wv * kSlice;
            for (uint32_t q = first + wv; q < last; q += WAVES) {
                const Item itm = decode(sload(queue + q));
                const uint32_t u = itm.row, chunk = itm.chunk, kind = itm.kind, g = itm.g;
                const GraphDev G = graph_at<true>(gs, g);
                const uint64_t rb = sload(G.off + u);
                const uint32_t K = (uint32_t)(sload(G.off + u + 1) - rb);
                const Segs sg = item_segs(G, kind, chunk, u, rb, K);
                const uint32_t tl = table_log2_for(K, scale, kSliceLog2);
                uint32_t *ovf = s_ovf + wv * (kSlice / 128);
                for (uint32_t i = lane; i < (1u << tl); i += 64) tab[i] = kEmpty;
                if (lane < kSlice / 128) ovf[lane] = 0;
                table_insert(tab, ovf, tl, G.col, rb, K, lane, 64);
                table_mark(tab, ovf, tl, lane, 64);
                const unsigned long long hits =
                    walk<UNROLL, NARROW>(G.off, sg.seg ? G.scol : G.col, G.n_rows, sg.ids, sg.seg, sg.n, sg.below, 0, 64, tab, tl,
                                 s_base[wv], s_end[wv], lane);
                if (g != cur_g) {
                    if (cur_g != kEmpty && acc != 0 && lane == 0) atomicAdd(counts + cur_g, acc);
                    cur_g = g;
                    acc = 0;
                }
                acc += hits;
                if (G.per_row && lane == 0) G.per_row[u] = hits;
            }
        }
        // two slots in turn: a slot is written again only after the barrier that
        // every wave passes with its last reading of it behind
        if (tid == 0) s_ticket[turn] = tk.next();
        __syncthreads();
        t = uniform(s_ticket[turn]);
        turn ^= 1u;
    }
    flush_counts<WAVES>(counts, s_acc, s_g, acc, cur_g, tid, wv, lane);
}

// ------------------------------------------------------------------ hub count kernel
// The count over hub codes (hubcode.h), with in-lists (SPLIT) or without: every item is
// one wave's, one wave per workgroup (9.1 KB of LDS: 16 waves per CU).
//
// What bounds it (RMAT s23, 8.8 ms; k_count took 16.9): the loads behind the L2, 6.7 TB/s of
// them (k_count 7.2); the texture data unit is busy 99% of the time, 58% of it stalled on the
// cache; so bytes and L2
// hits are what counts.  k_count fetched 121 GB a launch.  16-bit codes and bitmaps
// of the top hubs: 75 GB.  Parts of heavy rows per XCD and step (hubcode.h), so that
// lists are met again while they are in L2: 62 GB; the same share of a row's own arcs
// and in-list in each part, lists from 128-byte boundaries, words and ids read
// non-temporally: 56 GB (10.3, 9.8, 8.8 ms).  48 steps' parts instead of 32, 8 parts
// from 256 lists or 32 from 1024 on: no faster.  A round of 4 chunks of codes: 2 or 3
// chunks 11.0 / 10.7 against 10.7 ms a call.
// The headers of a ticket's items (queue entry, row offsets, record: three
// dependent loads) are loaded by the lanes together, and what an item starts from
// (its row's block, its first 64 lists) while the item before it is walked.
template <int U, bool SPLIT>
__global__ __launch_bounds__(64, 4) void k_count_hub(GraphDev G, HubSet hs, unsigned long long *__restrict__ counts) {
    __shared__ __align__(16) HubLds s;
    __shared__ __align__(16) uint32_t s_flag[16];
    __shared__ uint8_t s_src[64];

    if (!sload(hs.hctl + HC_ON)) return;  // counted by k_count
    const uint32_t lane = threadIdx.x;
    if (lane < 16) s_flag[lane] = 0;
    const uint32_t tiny_end = sload(hs.hctl + HC_TINY0) + sload(hs.hctl + HC_TINY);
    const uint64_t *units = hs.units;
    unsigned long long acc = 0;

    HubTickets tk(hs.hctl);
    for (HubTicket t = tk.first(); uniform(t.n); t = tk.next(lane)) {
        t = HubTicket{uniform(t.at), uniform(t.n), uniform(t.tiny) != 0};
        if (SPLIT && t.tiny) {
            const uint32_t e = t.at + lane;
            const uint64_t q = e < tiny_end ? gload(hs.queue + e) : 0;
            acc += tiny_walk(G, e < tiny_end, e < tiny_end && !(q >> 32), (uint32_t)q, s.bits, s.base, s.end, s_src,
                             (uint8_t *)s_flag, lane);
            continue;
        }
        // lane i: item i's header
        uint32_t len = 0, own = 0, n_own = 0, in = 0, n_l = 0;
        uint64_t rec = 0;
        if (lane < t.n) {
            const uint64_t q = gload(hs.queue + t.at + lane);
            const uint32_t row = (uint32_t)q, chunk = (uint32_t)(q >> 32);
            rec = gload(hs.rec + row);
            const uint64_t r0 = gload(G.off + row), i0 = SPLIT ? gload(G.in_off + row) : 0;
            len = (uint32_t)(gload(G.off + row + 1) - r0);
            const uint32_t k = row < G.n_owned ? len : 0u;
            const uint32_t kb = SPLIT ? (uint32_t)(gload(G.in_off + row + 1) - i0) : 0u;
            const uint32_t chunks = hub_split(k + kb).chunks();
            // the chunk's share of both, so that equal parts of rows cover much the same ids
            const uint32_t a0 = (uint32_t)((uint64_t)k * chunk / chunks), b0 = (uint32_t)((uint64_t)kb * chunk / chunks);
            own = (uint32_t)r0 + a0;
            in = (uint32_t)i0 + b0;
            n_own = (uint32_t)((uint64_t)k * (chunk + 1) / chunks) - a0;
            n_l = n_own + (uint32_t)((uint64_t)kb * (chunk + 1) / chunks) - b0;
        }
        auto item = [&](uint32_t i) {
            return HubItem{read_lane(len, i), read_lane(own, i), read_lane(n_own, i), read_lane(in, i), read_lane(n_l, i),
                           split_rec(read_lane64(rec, i))};
        };
        HubItem it = item(0);
        HubAhead ahead = hub_ahead<SPLIT>(G, it, units, lane);
        for (uint32_t i = 0; i < t.n; ++i) {
            const HubItem cur = it;
            HubAhead a = ahead;
            const bool kept = list_kept<SPLIT>(G, cur, lane, a.word, a.id);
            const uint64_t lrec = gload(hs.rec + (kept ? a.id : 0u));
            hub_insert(cur, a, units, s, lane);
            if (i + 1 < t.n) {
                it = item(i + 1);
                ahead = hub_ahead<SPLIT>(G, it, units, lane);
            }
            acc += hub_walk<U, SPLIT>(G, hs.rec, cur, a, lrec, kept, units, s, lane);
        }
    }
    if (acc != 0 && lane == 0) atomicAdd(counts, acc);
}

// ------------------------------------------------------------------ host side
// Workgroups of `kern` that fit on one CU at once (registers, LDS), cached per
// kernel; 0 when the runtime cannot tell.
static uint32_t resident_blocks(const void *kern, int threads) {
    static std::mutex mu;
    static std::unordered_map<const void *, uint32_t> cache;
    std::lock_guard<std::mutex> lk(mu);
    auto it = cache.find(kern);
    if (it != cache.end()) return it->second;
    int blocks = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kern, threads, 0) != hipSuccess || blocks < 0) blocks = 0;
    (void)hipGetLastError();
    cache[kern] = (uint32_t)blocks;
    return (uint32_t)blocks;
}

static constexpr int kHubU = 4;

// queue entries: per row one kind A item and at most 1 + in-degree / kInChunk kind B items
static uint64_t queue_cap(uint64_t total_rows, uint64_t total_m) { return 2 * total_rows + total_m / kInChunk + 1; }

// The engine's own arrays, first in its workspace.
struct PlanArrays {
    uint32_t *ctl, *wcnt;
    unsigned long long *queue;
};
static PlanArrays plan_arrays(Carver &c, uint64_t total_rows, uint64_t total_m) {
    PlanArrays a;
    a.ctl = c.take<uint32_t>(C_WORDS);
    a.wcnt = c.take<uint32_t>(kPlanEntries);
    a.queue = c.take<unsigned long long>(queue_cap(total_rows, total_m));
    return a;
}

// The code arrays of a launch over one graph, behind them (hctl null: it counts from ids).
static HubSet code_arrays(Carver &c, uint32_t rows, uint32_t owned, uint64_t m, bool split) {
    if (!hub_fits(rows, m, split) || !hub_worth(rows, owned, m, split)) return HubSet{};
    const HubSet h = hub_layout(c, rows, m);
    return c.ok() ? h : HubSet{};
}

size_t count_ws_base(uint64_t total_rows, uint64_t total_m) {
    Carver c(nullptr, 0);
    (void)plan_arrays(c, total_rows, total_m);
    return c.need();
}

size_t count_ws_bytes(uint64_t rows, uint64_t m) {
    Carver c(nullptr, 0);
    c.take<char>(count_ws_base(rows, m));
    if (hub_fits(rows, m)) (void)hub_layout(c, rows, m);
    return c.need();
}

lstc_status count_path(uint32_t n_rows, uint32_t n_owned, uint64_t m, bool split, void *ws, size_t ws_bytes,
                       hipStream_t st, uint32_t *path) {
    *path = 0;
    const uint64_t planned = split ? n_rows : n_owned;
    Carver c(ws, ws_bytes);
    (void)plan_arrays(c, planned, m);
    const HubSet hs = planned ? code_arrays(c, n_rows, n_owned, m, split) : HubSet{};
    if (!hs.hctl) return LSTC_OK;
    uint32_t words[HC_CHOSEN + 1];
    LSTC_HIP(hipMemcpyAsync(words, hs.hctl, sizeof(words), hipMemcpyDeviceToHost, st));
    LSTC_HIP(hipStreamSynchronize(st));
    *path = LSTC_PATH_DECIDED | (words[HC_CHOSEN] ? LSTC_PATH_BUILT : 0u) | (words[HC_ON] ? LSTC_PATH_CODES : 0u);
    return LSTC_OK;
}

lstc_status count_launch(const HostGraph *hosts, uint32_t G, const GraphDev *d_table, const uint64_t *d_row_base,
                         unsigned long long *d_counts, const lstc_tune *tune, void *ws, size_t ws_bytes,
                         hipStream_t st, bool timed) {
    if (G == 0) return LSTC_OK;
    if (G > kMaxGraphs) return fail(LSTC_ERR_INVALID, "count: at most %u graphs per launch", kMaxGraphs);
    if (!d_counts) return fail(LSTC_ERR_INVALID, "count: NULL counts");
    if (G > 1 && (!d_table || !d_row_base)) return fail(LSTC_ERR_INVALID, "count: batch needs device descriptors");
    uint64_t total = 0, total_m = 0;
    for (uint32_t g = 0; g < G; ++g) {
        total += plan_rows(hosts[g]);
        total_m += hosts[g].m;
    }
    const TuneR tr = effective_tune(tune, total_m);
    if (total >= 0xFFFFFFFFull) return fail(LSTC_ERR_INVALID, "count: more than 2^32-1 owned rows in one launch");
    Carver c(ws, ws_bytes);
    if (queue_cap(total, total_m) >= 0xFFFFFFFFull)
        return fail(LSTC_ERR_INVALID, "count: more than 2^32-1 work items in one launch");
    const PlanArrays arrays = plan_arrays(c, total, total_m);
    uint32_t *ctl = arrays.ctl, *wcnt = arrays.wcnt;
    unsigned long long *queue = arrays.queue;
    if (!ws || !c.ok()) return fail(LSTC_ERR_WORKSPACE, "count: workspace %zu < %zu bytes", ws_bytes, c.need());

    GraphSet gs{};
    gs.G = G;
    gs.total_rows = total;
    if (G == 1) {
        gs.one = to_dev(hosts[0]);
    } else {
        gs.table = d_table;
        gs.row_base = d_row_base;
    }
    for (uint32_t g = 0; g < G; ++g)
        if (hosts[g].per_row) LSTC_TRY(fill_u64(hosts[g].per_row, 0, hosts[g].n_owned, st));
    if (total == 0) return fill_u64((uint64_t *)d_counts, 0, G, st);
    const int cus = device_cus();
    Bounds bd{{16, 64, tr.small_max, 1024, 2048, 0xFFFFFFFFu}, tr.tiny_max};
    bool narrow = true;
    for (uint32_t g = 0; g < G; ++g)
        narrow = narrow && hosts[g].m <= (1ull << 30) && hosts[g].scol_len <= (1ull << 30);
    using Kern = void (*)(GraphSet, const unsigned long long *, uint32_t *, unsigned long long *, uint32_t, const uint32_t *);
    // [unroll 4/8][narrow][waves 2/4/8]
    static const Kern kerns[2][2][3] = {
        {{k_count<4, false, 2>, k_count<4, false, 4>, k_count<4, false, 8>},
         {k_count<4, true, 2>, k_count<4, true, 4>, k_count<4, true, 8>}},
        {{k_count<8, false, 2>, k_count<8, false, 4>, k_count<8, false, 8>},
         {k_count<8, true, 2>, k_count<8, true, 4>, k_count<8, true, 8>}}};
    const Kern kern = kerns[tr.unroll == 8][narrow][tr.waves == 2 ? 0 : tr.waves == 4 ? 1 : 2];
    // a persistent grid beyond what fits at once would only wait for the queue to drain
    uint32_t grid = (uint32_t)cus * tr.grid_per_cu;
    const uint32_t fit = resident_blocks((const void *)kern, tr.waves * 64);
    if (fit && grid > (uint32_t)cus * fit) grid = (uint32_t)cus * fit;
    bool split = false;
    for (uint32_t g = 0; g < G; ++g) split = split || split_ok(hosts[g]);
    const uint32_t classes = split ? (total_m < kLongArcs * G ? kHeads : kFewHeads) : total_m < kShortArcs ? kHeads : 1u;
    const uint32_t fine = classes > 1 ? 0xFFFFFFFFu : hmax(grid, (uint32_t)(total_m / kFineArcs));
    // Codes: one graph with in-lists and segment words, or counted without in-lists
    // and without per-row output, and a workspace that holds their arrays (count_ws_base is
    // still enough for k_count).  Whether its hubs cover its columns well enough is
    // decided on the device: both count kernels are launched and one leaves at once.
    HubSet hs{};
    uint32_t hub_grid = 0;
    using HubKern = void (*)(GraphDev, HubSet, unsigned long long *);
    const HubKern hub_kern = split ? (HubKern)k_count_hub<kHubU, true> : (HubKern)k_count_hub<kHubU, false>;
    if (G == 1 && (split ? seg_ok(hosts[0]) : !hosts[0].per_row))
        hs = code_arrays(c, hosts[0].n_rows, hosts[0].n_owned, total_m, split);
    if (hs.hctl) {
        const uint32_t hfit = resident_blocks((const void *)hub_kern, 64);
        hub_grid = (uint32_t)cus * (hfit ? hfit : 1u);
        LSTC_TRY(hub_build(gs.one, total_m, hs, st));
    }
    const uint32_t *hub_on = hub_grid ? hs.hctl + HC_ON : nullptr;
    if (total <= kSmallPlan && !hub_grid) {
        hipLaunchKernelGGL(k_plan_small, dim3(1), dim3(1024), 0, st, gs, bd, ctl, queue, d_counts, tr.small_group, grid,
                           tr.waves, classes, fine);
        LSTC_LAUNCHED("k_plan_small");
    } else {
        hipLaunchKernelGGL(k_plan_rows<0>, dim3(kPlanBlocks), dim3(256), 0, st, gs, bd, wcnt, queue, hs);
        LSTC_LAUNCHED("k_plan_rows<0>");
        hipLaunchKernelGGL(k_plan_scan, dim3(1), dim3(1024), 0, st, wcnt, ctl, d_counts, G, tr.small_group, grid,
                           tr.waves, classes, fine, hs, hub_grid);
        LSTC_LAUNCHED("k_plan_scan");
        hipLaunchKernelGGL(k_plan_rows<1>, dim3(kPlanBlocks), dim3(256), 0, st, gs, bd, wcnt, queue, hs);
        LSTC_LAUNCHED("k_plan_rows<1>");
    }
    {
        const TimingMark tm = timed ? timing_begin(st) : TimingMark{nullptr, nullptr};
        if (hub_grid) {
            hipLaunchKernelGGL(hub_kern, dim3(hub_grid), dim3(64), 0, st, gs.one, hs, d_counts);
            LSTC_LAUNCHED("k_count_hub");
        }
        hipLaunchKernelGGL(kern, dim3(grid), dim3(tr.waves * 64), 0, st, gs, queue, ctl, d_counts, tr.table_scale,
                           hub_on);
        LSTC_LAUNCHED("k_count");
        timing_end(tm, st);
    }
    return LSTC_OK;
}

}  // namespace lstc
