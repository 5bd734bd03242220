// hubwalk.h -- the count kernel's walk over hub codes, hub bitmaps and tails
// (hubcode.h).  One wave works on one item: a planned row r and up to kHubChunk of
// the lists it meets.  Row r's hubs are a bitmap of 2^16 bits in the wave's LDS
// (8 KB); code c is bit c % 32 of word c / 32, so a probe is one bit-field extract
// at the code (which takes the low five bits).  A
// window holds up to 64 lists, one per lane:
//   bitmaps: lane i holds two words of r's top-hub bits; one 8-byte load, two ANDs and
//            bit counts per list that has a bitmap;
//   codes  : the lists' codes as one flat sequence of 8-byte units (four codes), 64
//            units per chunk, U chunks per round, two rounds in flight;
//   tails  : the lists' ids (two per unit) through a 2048-bit filter of r's tail, a
//            passing id compared with every id of r's tail.
#pragma once
#include "hubcode.h"
#include "segwalk.h"

namespace lstc {

static constexpr uint32_t kHubWords = kCodes / 32;
static constexpr uint32_t kFilterWords = 64;

// The wave's LDS.
struct HubLds {
    uint32_t bits[kHubWords];
    uint32_t filter[kFilterWords];
    uint32_t base[64], end[64];
    uint32_t queue[64];  // ids that passed the filter
};

__device__ __forceinline__ uint32_t tail_hash(uint32_t x) { return (x * 0x9E3779B1u) >> 21; }  // 11 bits

// One item: n_own of the row's own arcs (from entry `own` of the columns) and
// then n - n_own entries of its in-list (from entry `in`).  Everything is uniform
// across the wave.
struct HubItem {
    uint32_t len, own, n_own, in, n;  // len: d+ of the row
    RowRec row;
};

// What the wave loads of an item before it starts on it.
struct HubAhead {
    uint64_t word;   // lane's list: its segment word
    uint32_t id;     // and its id
    uint64_t codes;  // lane's unit of the row's codes
    uint64_t top;    // lane's words of the row's bitmap (0 without one)
    uint32_t tail;   // lane's id of the row's tail (kEmptyId past its end)
};
static constexpr uint32_t kEmptyId = 0xFFFFFFFFu;

// SPLIT: the graph has in-lists and segment words (`word` is list j's); without
// them every own arc is counted here, and only rows have lists.
template <bool SPLIT>
__device__ __forceinline__ void list_load(const GraphDev &G, const HubItem &it, uint32_t j, uint64_t &word, uint32_t &id) {
    word = 0;
    id = 0xFFFFFFFFu;
    if (!SPLIT) {
        if (j < it.n) id = __builtin_nontemporal_load((const LSTC_GLOBAL_AS uint32_t *)(G.col + it.own + j));
        return;
    }
    const bool own = j < it.n_own, in = j < it.n;
    const uint32_t at = own ? it.own + j : it.in + (j - it.n_own);
    const uint64_t *w = own ? G.col_seg : G.in_seg;
    const uint32_t *c = own ? G.col : G.in_col;
    if (in) {
        // read once per count: kept out of the way of the lists in L2
        word = __builtin_nontemporal_load((const LSTC_GLOBAL_AS uint64_t *)(w + at));
        id = __builtin_nontemporal_load((const LSTC_GLOBAL_AS uint32_t *)(c + at));
    }
}
// Whether list j of the item is streamed: it has entries, and one of the row's own
// arcs is counted here only if its list is shorter than the row.
template <bool SPLIT>
__device__ __forceinline__ bool list_kept(const GraphDev &G, const HubItem &it, uint32_t j, uint64_t word, uint32_t id) {
    if (!SPLIT) return id < G.n_rows;
    const uint32_t d = (uint32_t)(word >> 32);
    return d != 0 && (j >= it.n_own || d < it.len);
}

template <bool SPLIT>
__device__ __forceinline__ HubAhead hub_ahead(const GraphDev &G, const HubItem &it, const uint64_t *__restrict__ units, uint32_t lane) {
    HubAhead a;
    list_load<SPLIT>(G, it, lane, a.word, a.id);
    a.codes = ~0ull;
    a.top = 0;
    a.tail = kEmptyId;
    if (lane < it.row.units) a.codes = gload(units + it.row.start + lane);
    if (it.row.bitmap) a.top = gload(units + it.row.start - kTopUnits + lane);
    if (lane < 2 * it.row.tail) a.tail = gload((const uint32_t *)(units + it.row.start + it.row.units) + lane);
    return a;
}

__device__ __forceinline__ void set_codes(uint32_t *bits, uint64_t x) {
    const uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
    const uint32_t c[4] = {lo & 0xFFFFu, lo >> 16, hi & 0xFFFFu, hi >> 16};
#pragma unroll
    for (int s = 0; s < 4; ++s)
        if (c[s] != kNoCode) atomicOr(bits + (c[s] >> 5), 1u << (c[s] & 31u));
}

// Writes the item's row into the wave's LDS.  A padding id becomes kEmptyId in
// a.tail, which no streamed id equals.
__device__ __forceinline__ void hub_insert(const HubItem &it, HubAhead &a, const uint64_t *__restrict__ units, HubLds &s,
                                           uint32_t lane) {
#pragma unroll
    for (uint32_t i = 0; i < kHubWords / 256; ++i) ((uint4 *)s.bits)[64 * i + lane] = uint4{0, 0, 0, 0};
    if (it.row.bitmap) {  // (the row's codes are all behind the top hubs then)
        s.bits[2 * lane] = (uint32_t)a.top;
        s.bits[2 * lane + 1] = (uint32_t)(a.top >> 32);
    }
    set_codes(s.bits, a.codes);
    for (uint32_t u = 64 + lane; u < it.row.units; u += 64) set_codes(s.bits, gload(units + it.row.start + u));
    if (it.row.tail == 0) return;
    s.filter[lane] = 0;
    if (a.tail == kTailPad) a.tail = kEmptyId;
    if (a.tail != kEmptyId) atomicOr(s.filter + (tail_hash(a.tail) >> 5), 0x80000000u >> (tail_hash(a.tail) & 31u));
    const uint32_t *ids = (const uint32_t *)(units + it.row.start + it.row.units);
    for (uint32_t i = 64 + lane; i < 2 * it.row.tail; i += 64) {
        const uint32_t x = gload(ids + i);
        if (x != kTailPad) atomicOr(s.filter + (tail_hash(x) >> 5), 0x80000000u >> (tail_hash(x) & 31u));
    }
}

// Counts the queued ids that the row's tail holds.
__device__ __forceinline__ void tail_drain(const HubItem &it, const HubAhead &a, const uint64_t *__restrict__ units,
                                           const HubLds &s, uint32_t n, uint32_t lane, uint32_t &hits) {
    const uint32_t x = lane < n ? s.queue[lane] : kTailPad;
    const uint32_t total = 2 * it.row.tail;
    const uint32_t *ids = (const uint32_t *)(units + it.row.start + it.row.units);
    uint64_t found = 0;
    uint32_t t = a.tail;
    for (uint32_t i0 = 0; i0 < total; i0 += 64) {
        if (i0) {
            t = i0 + lane < total ? gload(ids + i0 + lane) : kEmptyId;
            if (t == kTailPad) t = kEmptyId;
        }
        const uint32_t m = total - i0 < 64 ? total - i0 : 64u;
        for (uint32_t k = 0; k < m; ++k) found |= ballot(read_lane(t, k) == x);
    }
    if (lane_in(found)) ++hits;
}

template <int U>
__device__ __forceinline__ void load_units(const uint64_t *__restrict__ units, const uint32_t (&idx)[U], uint64_t (&x)[U]) {
#pragma unroll
    for (int k = 0; k < U; ++k) x[k] = gload_off32(units, idx[k]);
}

// Probes a round of codes (units [B, B + 64 U) of the window's sequence).
template <int U, bool FULL>
__device__ __forceinline__ void probe_codes(const uint64_t (&x)[U], uint32_t B, uint32_t total, const uint32_t *bits,
                                            uint32_t lane, uint32_t &hits) {
    uint32_t c[U][4], w[U][4];
#pragma unroll
    for (int k = 0; k < U; ++k) {
        const bool in = FULL || B + 64u * k + lane < total;
        const uint32_t lo = in ? (uint32_t)x[k] : 0xFFFFFFFFu, hi = in ? (uint32_t)(x[k] >> 32) : 0xFFFFFFFFu;
        c[k][0] = lo;
        c[k][1] = lo >> 16;
        c[k][2] = hi;
        c[k][3] = hi >> 16;
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
        if (!FULL && B + 64u * k >= total) continue;  // (uniform)
#pragma unroll
        for (int s = 0; s < 4; ++s)
            w[k][s] = *(const uint32_t *)((const char *)bits + ((c[k][s] >> 3) & 0x1FFCu));
    }
#pragma unroll
    for (int k = 0; k < U; ++k) {
        if (!FULL && B + 64u * k >= total) continue;
#pragma unroll
        for (int s = 0; s < 4; ++s) hits += __builtin_amdgcn_ubfe(w[k][s], c[k][s], 1);
    }
}

// Probes 64 units of tails: ids that pass the filter are queued.
__device__ __forceinline__ void probe_tail(uint64_t x, uint32_t B, uint32_t total, const HubItem &it, const HubAhead &a,
                                           const uint64_t *__restrict__ units, HubLds &s, uint32_t &qn, uint32_t lane,
                                           uint32_t &hits) {
    const bool in = B + lane < total;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t id = k ? (uint32_t)(x >> 32) : (uint32_t)x, h = tail_hash(id);
        const uint64_t H = ballot(in && (int32_t)(s.filter[h >> 5] << (h & 31u)) < 0);
        if (H == 0) continue;
        const uint32_t c = (uint32_t)__popcll(H);
        if (qn + c > 64u) {
            tail_drain(it, a, units, s, qn, lane, hits);
            qn = 0;
        }
        if (lane_in(H)) s.queue[qn + mask_rank(H)] = id;
        qn += c;
    }
}

// ------------------------------------------------------------------ tickets
// Ticket h of XCD x: first its own region's, then every eighth of the light, the
// small and the tiny rows'.  A wave whose XCD has run out takes what the others have left.
struct HubTicket {
    uint32_t at, n;  // first item, items (0: nothing left; of a tiny ticket 64 at most, not counted)
    bool tiny;
};
struct HubTickets {
    uint32_t *hctl;
    uint32_t x, left;
    __device__ __forceinline__ HubTickets(uint32_t *h) : hctl(h), x(blockIdx.x % kXcds), left(kXcds - 1) {}
    __device__ __forceinline__ HubTicket look(uint32_t h) const {
        const uint32_t own = sload(hctl + HC_OWN_T + x);
        if (h < own) {
            const uint32_t at = sload(hctl + HC_OWN0 + x) + h * kOwnGroup;
            return HubTicket{at, min(kOwnGroup, sload(hctl + HC_OWN_END + x) - at), false};
        }
        uint64_t t = (uint64_t)(h - own) * kXcds + x;
        const uint32_t light = sload(hctl + HC_LIGHT_T);
        if (t < light) {
            const uint32_t i = (uint32_t)t * kLightGroup;
            return HubTicket{sload(hctl + HC_LIGHT0) + i, min(kLightGroup, sload(hctl + HC_LIGHT) - i), false};
        }
        t -= light;
        const uint32_t small = sload(hctl + HC_SMALL_T);
        if (t < small) {
            const uint32_t i = (uint32_t)t * kSmallGroup;
            return HubTicket{sload(hctl + HC_SMALL0) + i, min(kSmallGroup, sload(hctl + HC_SMALL) - i), false};
        }
        t -= small;
        if (t < sload(hctl + HC_TINY_T)) return HubTicket{sload(hctl + HC_TINY0) + (uint32_t)t * 64, 64, true};
        return HubTicket{0, 0, false};
    }
    // wave-uniform; the first ticket costs no atomic
    __device__ __forceinline__ HubTicket first() { return find(uniform(blockIdx.x / kXcds)); }
    __device__ __forceinline__ HubTicket next(uint32_t lane) { return find(take(lane)); }
    __device__ __forceinline__ uint32_t take(uint32_t lane) {
        uint32_t h = 0;
        if (lane == 0) h = atomicAdd(hctl + HC_HEADS + 32 * x, 1u);
        return uniform(h);
    }
    __device__ __forceinline__ HubTicket find(uint32_t h) {
        HubTicket t = look(h);
        while (t.n == 0 && left) {
            --left;
            x = x + 1 == kXcds ? 0 : x + 1;
            // (a head only grows: an old value can only cost one atomic)
            h = uniform(__hip_atomic_load(hctl + HC_HEADS + 32 * x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            if (look(h).n == 0) continue;
            t = look(take(lane_id()));
        }
        return t;
    }
};

// Places the lanes' lists of `len` units starting at `start` behind one another:
// the lanes' bases and ends as index_walk takes them; returns the sequence's length.
__device__ __forceinline__ uint32_t lay_out(uint32_t start, uint32_t len, HubLds &s, uint32_t lane, uint32_t &base,
                                            uint32_t &end) {
    const uint32_t incl = wave_incl_scan(len, lane);
    const uint64_t nz = ballot(len != 0);
    if (len != 0) {
        const uint32_t slot = mask_rank(nz);
        s.base[slot] = start - (incl - len);
        s.end[slot] = incl;
    }
    base = s.base[lane];
    end = lane < (uint32_t)__popcll(nz) ? s.end[lane] : 0xFFFFFFFFu;
    return read_lane(incl, 63);
}

// The matches of the item's lists, summed over the wave.
template <int U, bool SPLIT>
__device__ __forceinline__ uint32_t hub_walk(const GraphDev &G, const uint64_t *__restrict__ recs, const HubItem &it,
                                             const HubAhead &a, uint64_t rec, bool kept,
                                             const uint64_t *__restrict__ units, HubLds &s, uint32_t lane) {
    constexpr uint32_t RB = 64u * U;
    uint32_t hits = 0, qn = 0;
    const uint32_t top0 = s.bits[2 * lane], top1 = s.bits[2 * lane + 1];  // this lane's words of the row's top hubs
    for (uint32_t j0 = 0; j0 < it.n; j0 += 64) {
        const RowRec R = split_rec(kept ? rec : 0);
        uint64_t word;
        uint32_t id;
        list_load<SPLIT>(G, it, j0 + 64 + lane, word, id);  // the next window's
        // the first round of tails and of codes
        uint32_t tbase = 0, tend = 0, ttotal = 0, ti[1] = {0};
        uint64_t tx[1] = {0};
        if (it.row.tail) {
            ttotal = lay_out(R.start + R.units, R.tail, s, lane, tbase, tend);
            if (ttotal) index_walk<1, false, 3>(0, ttotal, tbase, tend, 0, lane, ti);
            load_units<1>(units, ti, tx);
        }
        uint32_t mybase, myend;
        const uint32_t total = lay_out(R.start, R.units, s, lane, mybase, myend);
        uint32_t ia[U];
        uint64_t xa[U], xb[U];
        if (RB > total)
            index_walk<U, false, 3>(0, total, mybase, myend, 0, lane, ia);
        else
            index_walk<U, true, 3>(0, total, mybase, myend, 0, lane, ia);
        load_units<U>(units, ia, xa);
        for (uint64_t bm = ballot(R.bitmap != 0); bm;) {
            uint64_t v[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                v[k] = 0;
                if (bm) {
                    const uint32_t b = read_lane(R.start, (uint32_t)__builtin_ctzll(bm)) - kTopUnits;
                    bm &= bm - 1;
                    v[k] = gload(units + b + lane);
                }
            }
#pragma unroll
            for (int k = 0; k < 8; ++k)
                hits += (uint32_t)__popc((uint32_t)v[k] & top0) + (uint32_t)__popc((uint32_t)(v[k] >> 32) & top1);
        }
        kept = list_kept<SPLIT>(G, it, j0 + 64 + lane, word, id);
        rec = gload(recs + (kept ? id : 0u));
        uint32_t B = 0;
        if (total) {
            for (; B + 3 * RB <= total; B += 2 * RB) {
                // rounds B + RB and B + 2 * RB are full
                index_walk<U, true, 3>(B + RB, total, mybase, myend, first_segment(B + RB, myend), lane, ia);
                load_units<U>(units, ia, xb);
                probe_codes<U, true>(xa, B, total, s.bits, lane, hits);
                index_walk<U, true, 3>(B + 2 * RB, total, mybase, myend, first_segment(B + 2 * RB, myend), lane, ia);
                load_units<U>(units, ia, xa);
                probe_codes<U, true>(xb, B + RB, total, s.bits, lane, hits);
            }
            if (B + RB >= total) {
                probe_codes<U, false>(xa, B, total, s.bits, lane, hits);
            } else {
                index_walk<U, false, 3>(B + RB, total, mybase, myend, first_segment(B + RB, myend), lane, ia);
                load_units<U>(units, ia, xb);
                probe_codes<U, true>(xa, B, total, s.bits, lane, hits);
                if (B + 2 * RB < total) {
                    index_walk<U, false, 3>(B + 2 * RB, total, mybase, myend, first_segment(B + 2 * RB, myend), lane, ia);
                    load_units<U>(units, ia, xa);
                    probe_codes<U, true>(xb, B + RB, total, s.bits, lane, hits);
                    probe_codes<U, false>(xa, B + 2 * RB, total, s.bits, lane, hits);
                } else {
                    probe_codes<U, false>(xb, B + RB, total, s.bits, lane, hits);
                }
            }
        }
        for (uint32_t T = 0; T < ttotal; T += 64) {
            if (T) {
                index_walk<1, false, 3>(T, ttotal, tbase, tend, first_segment(T, tend), lane, ti);
                load_units<1>(units, ti, tx);
            }
            probe_tail(tx[0], T, ttotal, it, a, units, s, qn, lane, hits);
        }
    }
    if (qn) tail_drain(it, a, units, s, qn, lane, hits);
    // an item streams fewer than 2^32 entries, so its hits fit 32 bits
    return wave_sum32(hits);
}

}  // namespace lstc
