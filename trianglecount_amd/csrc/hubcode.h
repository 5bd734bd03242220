// hubcode.h -- a graph's rows as 16-bit hub codes, hub bitmaps and tails
// (hubcode.hip), read by the count kernel's hub walk (hubwalk.h).
//
// The kHubs vertices that occur most often in the columns (by a sample of them;
// exactness does not depend on which) have a 16-bit code, the most frequent ones
// the smallest.  On power-law graphs nearly every entry the count streams is a
// hub's (RMAT s23: 93%), so a list takes half the bytes and is tested against a
// bitmap of 2^16 bits instead of a hash table of ids.  A row with many of the kTop
// most frequent hubs keeps those as a bitmap of kTop bits (one 8-byte word per
// lane) and only the others as codes: two such rows meet in one AND and one bit
// count per lane.  The other vertices of a row, its tail, stay 32-bit ids.
//
// A row's block lies in 8-byte units: its bitmap if it has one (kTopUnits, from a
// 128-byte boundary), its codes (four to a unit), its tail (two ids to a unit).
// Row r starts at unit off[r] / 2 + 2 * r, or from there at the next 16-unit
// boundary if it has a bitmap or room for that: a row of d entries takes at most
// (d + 1) / 2 + 1 units (a bitmap replaces at least kTopMin = 192 entries, 96 units
// of ids, and takes 15 + 64), so blocks never meet and no scan is needed.
#pragma once
#include "count_engine.h"

namespace lstc {

static constexpr uint32_t kCodes = 1u << 16;
static constexpr uint32_t kNoCode = kCodes - 1;  // padding, and "no hub" in the code table
static constexpr uint32_t kHubs = kNoCode;       // codes 0 .. kNoCode - 1
static constexpr uint32_t kTop = 4096;           // hubs of the bitmaps: two 32-bit words per lane
static constexpr uint32_t kTopWords = kTop / 32;
static constexpr uint32_t kTopUnits = kTopWords / 2;  // 64: one unit per lane
static constexpr uint32_t kTopMin = 192;         // a row with this many of them gets a bitmap
static constexpr uint32_t kLongRow = 96;         // entries from which a row has a wave of its own in the build
static constexpr uint32_t kTailPad = 0xFFFFFFFEu;  // fills a tail's last unit; never an id
static constexpr uint32_t kMaxHubRow = 1u << 17;   // longest row whose lengths fit a record
// Longest tail.  A streamed id that passes the 2048-bit filter is compared with every
// id of the row's tail, so the cost per id grows with the tail twice.  Power-law graphs stay
// far below (RMAT s23 has tails of at most 89, Chung-Lu graphs of 1M to 3M vertices 46); uniform
// graphs are still faster from codes with tails of 350 (100 thousand vertices, mean degree
// 1000: 8.1 ms against 9.3 from ids) and 546 (90 thousand, 2000: 28.6 / 31.0); with
// tails of 65 thousand one list alone takes 0.2 s.
static constexpr uint32_t kMaxTail = 512;

// Work items.  A row's lists (its own arcs, then its in-list) are one sequence of n;
// an item is a chunk of it.  A row of kHeavy lists or more is cut into 8 parts, one
// per XCD, or into 8 * kSteps: part p holds the lists from the p-th fraction of the
// row's ascending ids, so the same part of different rows meets much the same
// lists.  Every XCD works through its own parts, step by step, all its waves on one
// step at a time, so that the lists of a step stay in its L2 (measured at RMAT s23,
// where 44 thousand rows of 512 lists or more stream 88% of the bytes: see k_count_hub).
static constexpr uint32_t kXcds = 8;
static constexpr uint32_t kSteps = 4;
static constexpr uint32_t kHeavy = 512;         // lists from which a row is cut into 8 parts
static constexpr uint32_t kHeavier = 2048;      // and into 8 * kSteps
static constexpr uint32_t kHubChunk = 1024;     // most lists per item
struct HubSplit {
    uint32_t parts, per_part;  // items = parts * per_part
    __host__ __device__ __forceinline__ uint32_t chunks() const { return parts * per_part; }
};
__host__ __device__ __forceinline__ HubSplit hub_split(uint32_t n) {
    const uint32_t parts = n < kHeavy ? 1u : n < kHeavier ? kXcds : kXcds * kSteps;
    return HubSplit{parts, (uint32_t)((n + (uint64_t)parts * kHubChunk - 1) / ((uint64_t)parts * kHubChunk))};
}
// Queue regions, in this order: per XCD its steps and then the 8-part rows' part;
// rows below kHeavy lists, from 64 and below; the tiny rows.
static constexpr uint32_t kXcdSlots = kSteps + 1;
static constexpr uint32_t kSlotLight = kXcds * kXcdSlots, kSlotSmall = kSlotLight + 1, kSlotTiny = kSlotLight + 2;
static constexpr uint32_t kHubSlots = kSlotLight + 3;
static_assert(kHubSlots <= 64, "the planner keeps one counter per lane");
static constexpr uint32_t kLight = 64;

// Per row: first unit of its codes (29 bits; a bitmap lies before them), units of
// codes (16), units of tail (18), bitmap or not (1).
__host__ __device__ __forceinline__ uint64_t make_rec(uint32_t start, uint32_t units, uint32_t tail, uint32_t bitmap) {
    return (uint64_t)start | ((uint64_t)units << 29) | ((uint64_t)tail << 45) | ((uint64_t)bitmap << 63);
}
struct RowRec {
    uint32_t start, units, tail, bitmap;
};
__device__ __forceinline__ RowRec split_rec(uint64_t r) {
    return RowRec{(uint32_t)r & 0x1FFFFFFFu, (uint32_t)(r >> 29) & 0xFFFFu, (uint32_t)(r >> 45) & 0x3FFFFu,
                  (uint32_t)(r >> 63)};
}

// words of the selection (uint32)
enum { HC_ON = 0, HC_LONG_ROWS = 1, HC_DONE = 2, HC_CUT = 3, HC_REST = 4,
       HC_CHOSEN = 5,  // HC_ON as it was chosen, before rows that codes cannot hold took it back
       HC_LEN = 8, HC_LENS = 10, HC_SQ = 12,  // 64-bit sums
       HC_HIST = 64, HC_SUM = HC_HIST + 256,
       HC_BASE = HC_SUM + 256, HC_USED = HC_BASE + 256,
       // the plan: first item and tickets of each XCD's own region; the light and the tiny rows
       HC_OWN0 = HC_USED + 256, HC_OWN_T = HC_OWN0 + 8, HC_OWN_END = HC_OWN_T + 8, HC_LIGHT0 = HC_OWN_END + 8,
       HC_LIGHT, HC_LIGHT_T, HC_SMALL0, HC_SMALL, HC_SMALL_T, HC_TINY0, HC_TINY, HC_TINY_T,
       HC_HEADS = HC_OWN0 + 64,  // ticket heads, on lines of their own
       HC_WORDS = HC_HEADS + 8 * 32 };

struct HubSet {
    uint32_t *hctl;       // selection words; hctl[HC_ON]: whether this launch is counted from codes
    uint32_t *cnt;        // per row: occurrences in the sample
    uint16_t *code;       // per row: its vertex's code
    uint64_t *rec;        // per row
    uint32_t *long_rows;  // rows of at least kLongRow entries
    uint64_t *units;
    uint32_t *plan_cnt;   // [kHubSlots][plan_waves]
    uint32_t plan_waves;
    uint64_t *queue;      // row | chunk << 32; tiny rows: 1 << 32 if only their in-list counts
};
// Waves of the plan: one per 512 rows, up to this many (the scan of their counters is
// one workgroup's, 18 us for 2048 waves).
static constexpr uint32_t kHubPlanWaves = 2048;
// Items per ticket (at most 64), by region: a ticket of the small rows is worth one
// item of the others, and the last tickets decide how long the chip waits for its
// last wave.
static constexpr uint32_t kOwnGroup = 4, kLightGroup = 4, kSmallGroup = 16;

// Whether a graph of this size may use codes: enough arcs, and enough per row, that
// building them pays (see count_launch), and positions that fit 32-bit byte offsets.
bool hub_fits(uint64_t rows, uint64_t m, bool split = true);
// Whether enough of it is owned that a count may look for codes.
bool hub_worth(uint64_t rows, uint64_t owned, uint64_t m, bool split);
// Takes the arrays from the carver (also to size a workspace).
HubSet hub_layout(Carver &c, uint64_t rows, uint64_t m);
// Selects the hubs of the graph and builds its rows' blocks (kernels only).  m: its arcs, or more.
lstc_status hub_build(const GraphDev &g, uint64_t m, const HubSet &hs, hipStream_t st);

}  // namespace lstc
