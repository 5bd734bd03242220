// hubcode.hip -- selects a graph's hub vertices and writes its rows as 16-bit
// codes, hub bitmaps and tails (hubcode.h).  No counterpart in the reference,
// whose count reads 32-bit columns (ShareKernelTCV62_update_v1.cu:43-191).
//
//   k_hub_init   : clears the selection words and the occurrences
//   k_hub_sample : occurrences of each vertex in every stride-th 64-entry chunk of the columns
//   k_hub_pick   : vertices and occurrences per occurrence bin (8 bins per octave); the bins
//                  whose vertices become hubs, their first codes, and whether codes pay
//   k_hub_assign : every vertex's code
//   k_hub_short  : the blocks of rows below kLongRow entries, 16 lanes per row
//   k_hub_long   : the others, a wave per row
#include "hubcode.h"
#include "wave.h"

namespace lstc {

// Sampled entries (RMAT s23, ms a count: 11.1 with 2^20, 10.7 with 2^21, 10.8 with
// 2^22), and at most one in 16: the hubs' counters are hot addresses.
static constexpr uint64_t kSamples = 2u << 20, kMinStride = 16;
// When codes pay.  What they save is in proportion to what is streamed: per arc of the
// owned rows, with in-lists at most the smaller of the mean d+ of its two ends' rows
// (`from` and `to`, each a mean over arcs), without in-lists its target's row.  What they
// cost, the build, is in proportion to all arcs; so these means count times the owned
// rows' share of the arcs.  Three decisions:
//   hub_worth       on the host, by the sizes;
//   worth_sampling  before the sample, by the row lengths (a graph that it refuses has
//                   cost 0.02 to 0.04 ms; refused after the sample, 0.1 to 0.3 ms);
//   k_hub_pick      after it, with `to`, the share c of the columns that hubs cover, and
//                   the share of tails in what would be streamed.
// The figures are ms a call from ids / from codes (CL: Chung-Lu graphs of the gamma, mean
// degree and number of vertices; ER: uniform graphs of the vertices and mean degree).
//
// worth_sampling with in-lists, `from`:
//   RMAT s18 109 0.428 / 0.403, s21 189 3.14 / 2.15, s23 270 16.9 / 10.3
//   CL 2.1, 50: 300K 65 0.594 / 0.638, 1M 84 1.70 / 1.85, 2M 96 3.57 / 3.59, 3M 103 5.59 / 5.39
//   CL 2.3, 150, 300K 104 1.57 / 1.45; CL 2.5, 150, 300K 84 1.47 / 1.54
// The line rises with the vertices, of which the hubs are a smaller part.  Below kSmall
// arcs ids wait for the items of the largest hubs, which codes cut into parts:
//   RMAT s17 90 0.338 / 0.273; CL 2.1, 50: 80K 47 0.40 / 0.32, 110K 51 0.32 / 0.34,
//   150K 55 0.41 / 0.39, 230K 61 0.52 / 0.52, 260K (5.9M arcs) 63 0.53 / 0.56
static constexpr double kMinFrom = 86, kMinFromMore = 14, kMinFromRows = 1 << 21;  // 86 to 100
static constexpr double kMinFromSmall = 44;
static constexpr uint64_t kSmall = 11ull << 19;
// Without in-lists; from kBigPlain arcs on ids no longer stream from the caches:
//   CL 2.1, 50: 300K 65 0.568 / 0.605, 500K 73 1.03 / 0.94; CL 2.5, 150, 300K 84 1.58 / 1.39
//   CL 2.3, 50: 1M (25M arcs) 43 1.61 / 1.79, 2M 45 3.67 / 3.43, 3M 47 6.01 / 5.29
static constexpr double kMinFromPlain = 70, kMinFromPlainBig = 45;
static constexpr uint64_t kBigPlain = 1ull << 25;
// Parts, `from` times the share with in-lists: RMAT s21 in two 95 1.77 / 1.47, in eight 25
// 0.65 / 0.78, s23 in eight 35 2.72 / 2.80, in 32 10 1.23 / 1.69.  Without them:
// s23 in eight 35 4.79 / 3.03, in 32 10 1.54 / 1.64.
static constexpr double kMinFromOwnedPlain = 12;
// Below this many arcs of owned rows (by the rows' share) a part's count is over before
// a build pays, or before the launches that would find it out: s21 in eight, 6.3M,
// 0.65 / 0.78 with in-lists; in 32, 2.6M, 0.31 / 0.51, and 0.36 / 0.56 without; the first
// row of s23 alone 0.01 / 1.42.
static constexpr double kMinOwned = 12 << 20, kMinOwnedPlain = 3 << 20;
// Uniform graphs.  Where neither degree nor id means anything, d+ runs evenly from 0 to
// twice its mean, and its mean over arcs is 4/3 of that (ER with mean degrees of 40 to 1800
// 1.25 to 1.32; power laws of gamma 2.5 1.14 to 1.22, 2.3 from 1.4 on, RMAT from 2.8 on).
// Ids are fast there, and without hubs the codes cover what their number covers:
//   ER 100K, 400 1.70 / 1.53; 115K, 400 1.93 / 2.14; 130K, 600 4.4 / 7.7; 160K, 400, without in-lists 3.0 / 5.5
// With fewer vertices, by the sum of the squares of the row lengths:
//   with in-lists: 20K, 200 2e8 0.170 / 0.212; 10K, 400 (2M arcs) 5e8 0.230 / 0.281;
//     40K, 200 (4M arcs) 5e8 0.306 / 0.293; 8K, 500 6e8 0.268 / 0.319; 60K, 200 8e8 0.439 / 0.379;
//     4K, 1000 1e9 0.456 / 0.367
//   without: 80K, 200 1e9 0.450 / 0.467; 100K, 200 1.3e9 0.603 / 0.619; 60K, 400 3e9 1.00 / 0.78
static constexpr double kUniformLow = 1.23, kUniformHigh = 1.4;
static constexpr uint32_t kMaxUniformRows = 105000;
static constexpr double kMinUniform = 7e8, kMinUniformMore = 4.5e8, kMinUniformPlain = 2e9;
static constexpr uint64_t kUniformMore = 7ull << 19;  // arcs from which kMinUniformMore holds
// k_hub_pick with in-lists, min(from, to) (2 c - 1) times the share: CL 2.1, 50, 3M 52 5.59 /
// 5.39; CL 2.5, 150, 1M 23 4.73 / 5.72; kMinWorthFlat where arcs point at the shorter rows: ER
// 100K, 200 56 0.672 / 0.639.
static constexpr double kMinWorth = 40, kMinWorthFlat = 50;
// Without, `to`: CL 2.3, 50: 1M 111 1.61 / 1.79, 2M 128 3.67 / 3.43; times the share: s21 in
// eight 47 0.88 / 0.75, s23 in eight 73 4.79 / 3.03, in 32 20 1.54 / 1.64.
static constexpr double kMinPlainLen = 120, kMinPlainLenOwned = 40;
// Either way hubs cover half of the sample at least.
static constexpr uint32_t kCoverPct = 50;
// Tails are walked at a quarter of the codes' speed.  They are measured (in 10 us) where arcs
// point at the shorter rows: ER 100K 3.3% of the entries, 115K 6.6%, 130K 10%.  Graphs
// whose arcs point at the longer rows hardly stream any (CL 2.1 and RMAT below 1%; CL
// 2.5, 150, 1M 6%, without in-lists 6.80 / 5.19).
static constexpr double kMaxTailShare = 0.08;
// Smaller graphs and shorter rows keep ids: the build is worth 0.1 ms (RMAT s14, 0.7M arcs,
// 0.147 / 0.229).  Without in-lists ids have less to lose to (CL 2.1, 50, 150K, 3.3M arcs,
// 0.261 / 0.377; RMAT s19, 7.7M arcs, 0.88 / 0.63).
static constexpr uint64_t kMinArcs = 3ull << 19, kMinArcsPlain = 6ull << 20, kMinPerRow = 16;
static constexpr uint64_t kArcSeed = 0x68756263;  // of the arcs that stand for all when the tails are measured
static constexpr uint32_t kAbsent = 0xFFFFFFFFu;  // past the end of a row (ids are below 2^32 - 2)

__device__ __forceinline__ uint32_t occ_bin(uint32_t c) {
    if (c < 16) return c;
    const uint32_t lg = 31 - __clz(c);
    return 8 * (lg - 2) + ((c >> (lg - 3)) & 7u);
}

// The code of id x in a graph of n rows whose codes start at `code`; an id
// without a row (halo ids outside the part) has none.
__device__ __forceinline__ uint32_t code_of(const uint16_t *code, uint32_t n, uint32_t x) {
    return x < n ? gload(code + x) : kNoCode;
}

// The arcs there are: the launch knows a bound (the server's arrays are sized before
// their graph is cleaned), and what lies behind them in the columns is anything.
__device__ __forceinline__ uint64_t arcs_of(const GraphDev &G) { return sload(G.off + G.n_rows); }
// The share of them that the owned rows have.
__device__ __forceinline__ double owned_share(const GraphDev &G) {
    return (double)sload(G.off + G.n_owned) / (double)arcs_of(G);
}

// Whether the graph may be worth codes, from the sum of the squares of its row lengths.
__device__ __forceinline__ bool worth_sampling(const GraphDev &G, double squares, bool split) {
    const double arcs = (double)arcs_of(G), from = squares / arcs, share = owned_share(G), mean = arcs / G.n_rows;
    if (from >= kUniformLow * mean && from <= kUniformHigh * mean) {
        const double line = !split ? kMinUniformPlain : arcs < (double)kUniformMore ? kMinUniform : kMinUniformMore;
        return G.n_rows <= kMaxUniformRows && squares * share >= line;
    }
    if (split) {
        const double large = kMinFrom + kMinFromMore * fmin(1., G.n_rows / kMinFromRows);
        return from * share >= (arcs < (double)kSmall ? kMinFromSmall : large);
    }
    return from >= (arcs >= (double)kBigPlain ? kMinFromPlainBig : kMinFromPlain) && from * share >= kMinFromOwnedPlain;
}

// First unit of the block of row r, whose columns start at o.
__device__ __forceinline__ uint32_t block_of(uint64_t r, uint64_t o) { return (uint32_t)((o >> 1) + 2 * r); }

// Also the sum of the squares of the rows' lengths, one share per workgroup (at most
// kInitBlocks of them, in the plan's counters, which are free until the plan).
static constexpr uint32_t kInitBlocks = 1024;
static_assert(kInitBlocks * 2 <= kHubSlots * kHubPlanWaves, "the shares' place");
__global__ __launch_bounds__(256) void k_hub_init(HubSet hs, const uint64_t *__restrict__ off, uint32_t n) {
    __shared__ unsigned long long s_sq;
    if (threadIdx.x == 0) s_sq = 0;
    __syncthreads();
    if (blockIdx.x == 0)
        for (uint32_t i = threadIdx.x; i < HC_WORDS; i += 256) hs.hctl[i] = 0;
    unsigned long long sq = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * 256 + threadIdx.x; v < n; v += (uint64_t)gridDim.x * 256) {
        hs.cnt[v] = 0;
        const uint64_t d = gload(off + v + 1) - gload(off + v);
        sq += d * d;
    }
    if (sq) atomicAdd(&s_sq, sq);
    __syncthreads();
    if (threadIdx.x == 0) ((unsigned long long *)hs.plan_cnt)[blockIdx.x] = s_sq;
}

// A wave takes four chunks at a time; every fourth wave measures the rows of one of
// them (in turn the first to the fourth, which lie a quarter of the columns apart in a graph of
// up to 2^25 arcs): HC_LEN, the sum of their lengths, HC_LENS: how many.  It leaves
// at once if the row lengths speak against codes.
__global__ __launch_bounds__(256) void k_hub_sample(GraphDev G, uint32_t stride, HubSet hs, uint32_t shares,
                                                    bool split) {
    constexpr uint32_t kPer = 4;
    uint32_t *cnt = hs.cnt, *hctl = hs.hctl;
    const uint64_t m = arcs_of(G);
    {
        __shared__ unsigned long long s_sq;
        if (threadIdx.x == 0) s_sq = 0;
        __syncthreads();
        unsigned long long sq = 0;
        for (uint32_t i = threadIdx.x; i < shares; i += 256) sq += ((const unsigned long long *)hs.plan_cnt)[i];
        if (sq) atomicAdd(&s_sq, sq);
        __syncthreads();
        const unsigned long long all = s_sq;
        if (blockIdx.x == 0 && threadIdx.x == 0) *(unsigned long long *)(hctl + HC_SQ) = all;
        if (!worth_sampling(G, (double)all, split)) return;
    }
    uint32_t len = 0, lens = 0;
    const uint32_t lane = threadIdx.x & 63;
    const uint64_t waves = (uint64_t)gridDim.x * 4, wave = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint64_t chunks = (m + 64ull * stride - 1) / (64ull * stride);
    for (uint64_t c0 = wave; c0 < chunks; c0 += waves * kPer) {
        const uint32_t here = (uint32_t)min((uint64_t)kPer, (chunks - c0 + waves - 1) / waves);
        const uint32_t measured = (uint32_t)(c0 / 4) % here;
        uint32_t x[kPer], of = kAbsent;
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) {
            const uint64_t j = (c0 + q * waves) * 64 * stride + lane;
            x[q] = kAbsent;
            if (j < m) x[q] = gload(G.col + j);
        }
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) {
            if (x[q] < G.n_rows) atomicAdd(cnt + x[q], 1u);
            of = q == measured ? x[q] : of;
        }
        if (c0 % 4 == 0 && of < G.n_rows) {
            len += (uint32_t)min(gload(G.off + of + 1) - gload(G.off + of), (uint64_t)kMaxHubRow);
            ++lens;
        }
    }
    if (ballot(lens != 0) == 0) return;
    // (a wave has at most a few dozen chunks of 64 lengths of at most 2^17: 32 bits hold the sum)
    len = wave_sum32(len);
    lens = wave_sum32(lens);
    if (lane == 0) {
        atomicAdd((unsigned long long *)(hctl + HC_LEN), (unsigned long long)len);
        atomicAdd((unsigned long long *)(hctl + HC_LENS), (unsigned long long)lens);
    }
}

// The tails' share of the entries that arcs stream, by a workgroup of 256: kArcs arcs per
// thread, kEntries entries of each one's target's row.  Vertices of bins below `cut` and cut_tail of
// that bin's are no hubs.
__device__ __forceinline__ double tail_share(const GraphDev &G, const uint32_t *__restrict__ cnt, uint32_t cut,
                                             double cut_tail) {
    constexpr uint32_t kArcs = 2, kEntries = 4;
    __shared__ uint64_t s_entries[4], s_tails[4];
    const uint32_t tid = threadIdx.x, n = G.n_rows, some = (uint32_t)(16 * cut_tail);  // in sixteenths
    uint32_t x[kArcs], y[kArcs][kEntries];
    uint64_t o[kArcs], d[kArcs], entries = 0, tails = 0;
#pragma unroll
    for (uint32_t q = 0; q < kArcs; ++q) x[q] = gload(G.col + rng64(kArcSeed, q * 256 + tid) % arcs_of(G));
#pragma unroll
    for (uint32_t q = 0; q < kArcs; ++q) {
        o[q] = gload(G.off + (x[q] < n ? x[q] : 0u));
        d[q] = gload(G.off + (x[q] < n ? x[q] + 1 : 0u)) - o[q];  // (an id without a row: no entries)
    }
#pragma unroll
    for (uint32_t q = 0; q < kArcs; ++q)
#pragma unroll
        for (uint32_t k = 0; k < kEntries; ++k)
            y[q][k] = d[q] ? gload(G.col + o[q] + (2 * k + 1) * d[q] / (2 * kEntries)) : kAbsent;
#pragma unroll
    for (uint32_t q = 0; q < kArcs; ++q) {
        uint32_t t = 0;
#pragma unroll
        for (uint32_t k = 0; k < kEntries; ++k) {
            const uint32_t c = y[q][k] < n ? cnt[y[q][k]] : 0u, bin = occ_bin(c);
            t += c == 0 || bin < cut ? 16u : bin == cut ? some : 0u;
        }
        entries += d[q] * kEntries * 16;
        tails += d[q] * t;
    }
    entries = wave_sum64(entries);
    tails = wave_sum64(tails);
    if ((tid & 63) == 0) s_entries[tid >> 6] = entries, s_tails[tid >> 6] = tails;
    __syncthreads();
    return (double)(s_tails[0] + s_tails[1] + s_tails[2] + s_tails[3]) /
           (double)(s_entries[0] + s_entries[1] + s_entries[2] + s_entries[3] + 1);
}

// Every workgroup adds its share to the bins; the last one to do so picks.  Bins
// above HC_CUT are hubs; of bin HC_CUT the first HC_REST vertices that ask.
__global__ __launch_bounds__(256) void k_hub_pick(GraphDev G, const uint32_t *__restrict__ cnt, bool split,
                                                  uint32_t *__restrict__ hctl) {
    if (!sload(hctl + HC_LENS)) return;  // nothing was sampled
    const uint32_t n = G.n_rows;
    __shared__ uint32_t s_n[257], s_add[256];
    __shared__ unsigned long long s_sum[257];
    __shared__ uint32_t s_last;
    const uint32_t b = threadIdx.x;
    s_n[b] = 0;
    s_add[b] = 0;
    __syncthreads();
    constexpr uint32_t kPer = 8;
    const uint64_t step = (uint64_t)gridDim.x * 256;
    for (uint64_t v = (uint64_t)blockIdx.x * 256 + b; v < n; v += step * kPer) {
        uint32_t c[kPer];
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) c[q] = v + q * step < n ? cnt[v + q * step] : 0u;
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) {
            if (c[q] == 0) continue;
            atomicAdd(&s_n[occ_bin(c[q])], 1u);
            atomicAdd(&s_add[occ_bin(c[q])], c[q]);
        }
    }
    __syncthreads();
    if (s_n[b]) {
        atomicAdd(hctl + HC_HIST + b, s_n[b]);
        atomicAdd(hctl + HC_SUM + b, s_add[b]);
    }
    __threadfence();
    __syncthreads();
    if (b == 0) s_last = atomicAdd(hctl + HC_DONE, 1u) == gridDim.x - 1 ? 1u : 0u;
    __syncthreads();
    if (!s_last) return;
    auto read = [](uint32_t *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    const uint32_t own_n = read(hctl + HC_HIST + b);
    const unsigned long long own_sum = read(hctl + HC_SUM + b);
    uint32_t sn = own_n;  // over bins b, b + 1, ...
    unsigned long long ssum = own_sum;
    if (b == 0) s_n[256] = 0, s_sum[256] = 0;
    for (uint32_t d = 1; d < 256; d <<= 1) {
        s_n[b] = sn;
        s_sum[b] = ssum;
        __syncthreads();
        if (b + d < 256) sn += s_n[b + d], ssum += s_sum[b + d];
        __syncthreads();
    }
    s_n[b] = sn;
    s_sum[b] = ssum;
    __syncthreads();
    hctl[HC_BASE + b] = s_n[b + 1];
    const unsigned long long all = s_sum[0];
    __shared__ uint32_t s_cut, s_rest;
    __shared__ unsigned long long s_cov;
    if (b == 0) s_cut = s_rest = 0, s_cov = all;
    __syncthreads();
    if (s_n[0] > kHubs && sn > kHubs && s_n[b + 1] <= kHubs) {
        s_cut = b;
        s_rest = kHubs - s_n[b + 1];
        s_cov = s_sum[b + 1] + own_sum * s_rest / own_n;
    }
    __syncthreads();
    const uint32_t cut = s_cut, rest = s_rest, cut_n = s_n[cut] - s_n[cut + 1];
    const unsigned long long covered = s_cov;
    if (all == 0 || covered * 100 < all * kCoverPct) return;  // (off)
    auto read64 = [&](uint32_t w) {
        return (double)__hip_atomic_load((unsigned long long *)(hctl + w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    const double to = read64(HC_LEN) / read64(HC_LENS), from = read64(HC_SQ) / (double)arcs_of(G);
    const double cover = (double)covered / (double)all, share = owned_share(G);
    bool on = split ? fmin(from, to) * share * (2 * cover - 1) >= (to < from ? kMinWorthFlat : kMinWorth)
                    : to >= kMinPlainLen && to * share >= kMinPlainLenOwned;
    if (on && to < from && n > kHubs)
        on = tail_share(G, cnt, cut, cut_n ? (double)(cut_n - rest) / cut_n : 1.) <= kMaxTailShare;
    if (b != 0) return;
    hctl[HC_CUT] = cut;
    hctl[HC_REST] = rest;
    hctl[HC_ON] = hctl[HC_CHOSEN] = on ? 1u : 0u;
}

// A workgroup takes 4096 vertices at a time and one place per bin among all of them.
__global__ __launch_bounds__(256) void k_hub_assign(const uint32_t *__restrict__ cnt, uint32_t n,
                                                    uint32_t *__restrict__ hctl, uint16_t *__restrict__ code) {
    __shared__ uint32_t s_n[256], s_at[256];
    if (!sload(hctl + HC_ON)) return;
    const uint32_t cut = sload(hctl + HC_CUT), rest = sload(hctl + HC_REST), tid = threadIdx.x;
    for (uint64_t v0 = (uint64_t)blockIdx.x * 4096; v0 < n; v0 += (uint64_t)gridDim.x * 4096) {
        s_n[tid] = 0;
        __syncthreads();
        uint32_t c[16], at[16];
#pragma unroll
        for (uint32_t i = 0; i < 16; ++i) {
            const uint64_t v = v0 + i * 256 + tid;
            c[i] = v < n ? cnt[v] : 0u;
        }
#pragma unroll
        for (uint32_t i = 0; i < 16; ++i) {
            const uint32_t b = occ_bin(c[i]);
            at[i] = c[i] != 0 && b >= cut ? atomicAdd(&s_n[b], 1u) : 0u;
        }
        __syncthreads();
        s_at[tid] = s_n[tid] ? atomicAdd(hctl + HC_USED + tid, s_n[tid]) : 0u;
        __syncthreads();
#pragma unroll
        for (uint32_t i = 0; i < 16; ++i) {
            const uint64_t v = v0 + i * 256 + tid;
            const uint32_t b = occ_bin(c[i]), p = s_at[b] + at[i];
            const bool hub = c[i] != 0 && (b > cut || (b == cut && p < rest));
            if (v < n) code[v] = (uint16_t)(hub ? hctl[HC_BASE + b] + p : kNoCode);
        }
        __syncthreads();
    }
}

// One wave per 64 rows: four short rows at a time, 16 lanes each, their entries in
// registers (at most six per lane).  Long rows are listed for k_hub_long; a row
// longer than a record can say takes the launch back to k_count.
__global__ __launch_bounds__(256) void k_hub_short(GraphDev G, HubSet hs) {
    constexpr uint32_t kPer = kLongRow / 16;
    static_assert(kLongRow % 16 == 0, "a short row's entries per lane");
    __shared__ uint32_t s_n, s_at, s_on;
    // one read per workgroup: its waves must agree while another one clears the flag (a
    // scalar load: as an atomic one from every workgroup 1.10 ms for 0.43 at RMAT s23)
    const uint32_t on = sload(hs.hctl + HC_ON);
    if (threadIdx.x == 0) {
        s_n = 0;
        s_on = on;
    }
    __syncthreads();
    if (!s_on) return;
    const uint32_t lane = threadIdx.x & 63, sub = lane & 15, grp = lane >> 4;
    const uint64_t r0 = ((uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * 64, r = r0 + lane;
    const bool valid = r < G.n_rows;
    const uint64_t o = valid ? gload(G.off + r) : 0, e = valid ? gload(G.off + r + 1) : 0;
    if (e - o >= kMaxHubRow) hs.hctl[HC_ON] = 0;
    const uint32_t d = (uint32_t)min(e - o, (uint64_t)kMaxHubRow);
    const uint32_t start = block_of(r, o);
    const bool lng = d >= kLongRow;
    uint32_t place = 0;
    if (lng) place = atomicAdd(&s_n, 1u);
    __syncthreads();
    if (threadIdx.x == 0 && s_n) s_at = atomicAdd(hs.hctl + HC_LONG_ROWS, s_n);
    __syncthreads();
    if (lng) hs.long_rows[s_at + place] = (uint32_t)r;
    uint16_t *codes = (uint16_t *)hs.units;
    uint32_t *tails = (uint32_t *)hs.units;
    uint64_t mine = 0;  // this lane's row's record
    const uint64_t some = ballot(!lng && d != 0);
    for (uint32_t k = 0; k < 16; ++k) {
        if ((some >> (4 * k) & 15u) == 0) continue;
        const uint32_t src = 4 * k + grp;
        const uint32_t rd = gather(lng ? 0u : d, src);
        const uint32_t rs = gather(start, src);
        const uint32_t *pc = G.col + gather64(o, src);
        uint32_t x[kPer], c[kPer];
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) {
            const uint32_t i = 16 * q + sub;
            x[q] = kAbsent;
            if (i < rd) x[q] = gload(pc + i);
        }
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) {
            c[q] = kNoCode;
            if (x[q] != kAbsent) c[q] = code_of(hs.code, G.n_rows, x[q]);
        }
        const uint32_t sh = 16 * grp;
        uint32_t nh = 0;
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) nh += (uint32_t)__popc((uint32_t)(ballot(c[q] != kNoCode) >> sh) & 0xFFFFu);
        const uint32_t units = (nh + 3) / 4, nt = rd - nh;
        uint32_t ph = rs * 4, pt = (rs + units) * 2;
        const uint32_t below = (1u << sub) - 1u;
#pragma unroll
        for (uint32_t q = 0; q < kPer; ++q) {
            const bool h = c[q] != kNoCode, t = !h && x[q] != kAbsent;
            const uint32_t hm = (uint32_t)(ballot(h) >> sh) & 0xFFFFu, tm = (uint32_t)(ballot(t) >> sh) & 0xFFFFu;
            if (h) codes[ph + __popc(hm & below)] = (uint16_t)c[q];
            if (t) tails[pt + __popc(tm & below)] = x[q];
            ph += __popc(hm);
            pt += __popc(tm);
        }
        if (sub < ((0u - nh) & 3u)) codes[ph + sub] = (uint16_t)kNoCode;
        if (sub == 0 && (nt & 1u)) tails[pt] = kTailPad;
        // lane src of the wave takes the record of its row (held by lanes of group src & 3)
        const uint64_t rec = make_rec(rs, units, (nt + 1) / 2, 0);
        const uint64_t got = gather64(rec, 16 * (lane & 3));
        if (lane >> 2 == k) mine = got;
    }
    if (valid && !lng) hs.rec[r] = mine;
}

// A wave per long row, 512 entries in registers at a time (read twice if there are more).  A tail of more than
// kMaxTail ids takes the launch back to k_count.  A wave takes kBatch rows together: their headers (four
// dependent loads) come in by lane at once.
__global__ __launch_bounds__(256) void k_hub_long(GraphDev G, HubSet hs) {
    constexpr uint32_t kRegs = 8, kStep = 64 * kRegs, kBatch = 8;
    __shared__ uint32_t s_word[4][kTopWords];
    if (!sload(hs.hctl + HC_ON)) return;
    const uint32_t lane = threadIdx.x & 63, wv = uniform(threadIdx.x >> 6);
    uint32_t *word = s_word[wv];
    const uint32_t n_long = sload(hs.hctl + HC_LONG_ROWS);
    uint16_t *codes = (uint16_t *)hs.units;
    uint32_t *tails = (uint32_t *)hs.units;
    for (uint32_t i0 = (blockIdx.x * 4 + wv) * kBatch; i0 < n_long; i0 += gridDim.x * 4 * kBatch) {
        const uint32_t nb = min(kBatch, n_long - i0);
        uint32_t l_row = 0, l_d = 0, l_start = 0;
        uint64_t l_off = 0;
        if (lane < nb) {
            l_row = gload(hs.long_rows + i0 + lane);
            l_off = gload(G.off + l_row);
            l_d = (uint32_t)(gload(G.off + l_row + 1) - l_off);
            l_start = block_of(l_row, l_off);
        }
        for (uint32_t ib = 0; ib < nb; ++ib) {
            const uint32_t r = read_lane(l_row, ib), d = read_lane(l_d, ib), start = read_lane(l_start, ib);
            const uint32_t *colr = G.col + read_lane64(l_off, ib);
            uint32_t x[kRegs], c[kRegs];
            auto fetch = [&](uint32_t p0) {
#pragma unroll
                for (uint32_t q = 0; q < kRegs; ++q) {
                    const uint32_t p = p0 + 64 * q + lane;
                    x[q] = kAbsent;
                    if (p < d) x[q] = gload(colr + p);
                }
#pragma unroll
                for (uint32_t q = 0; q < kRegs; ++q) {
                    c[q] = kNoCode;
                    if (x[q] != kAbsent) c[q] = code_of(hs.code, G.n_rows, x[q]);
                }
            };
            uint32_t top = 0, hub = 0;
            for (uint32_t p0 = 0; p0 < d; p0 += kStep) {
                fetch(p0);
#pragma unroll
                for (uint32_t q = 0; q < kRegs; ++q) {
                    top += (uint32_t)__popcll(ballot(c[q] < kTop));
                    hub += (uint32_t)__popcll(ballot(c[q] != kNoCode));
                }
            }
            const bool bm = top >= kTopMin;
            const uint32_t floor = bm ? kTop : 0u;  // codes below go to the bitmap
            const uint32_t nh = bm ? hub - top : hub, units = (nh + 3) / 4, nt = d - hub;
            if (nt > kMaxTail && lane == 0) hs.hctl[HC_ON] = 0;  // (this launch's waves read it before their rows)
            // from a 128-byte boundary: with a bitmap there is always room for that, else if there is
            const uint32_t aligned = (start + 15u) & ~15u;
            const bool fits = aligned - start + units + (nt + 1) / 2 <= (d + 1) / 2 + 1;
            const uint32_t first = bm ? aligned + kTopUnits : fits ? aligned : start;
            word[lane] = word[64 + lane] = 0;
            uint32_t ph = first * 4, pt = (first + units) * 2;
            for (uint32_t p0 = 0; p0 < d; p0 += kStep) {
                if (d > kStep) fetch(p0);
#pragma unroll
                for (uint32_t q = 0; q < kRegs; ++q) {
                    const bool in = x[q] != kAbsent, h = c[q] != kNoCode && c[q] >= floor, t = in && c[q] == kNoCode;
                    const uint64_t hm = ballot(h), tm = ballot(t);
                    if (h) codes[ph + mask_rank(hm)] = (uint16_t)c[q];
                    else if (t) tails[pt + mask_rank(tm)] = x[q];
                    else if (in) atomicOr(&word[c[q] >> 5], 1u << (c[q] & 31u));
                    ph += (uint32_t)__popcll(hm);
                    pt += (uint32_t)__popcll(tm);
                }
            }
            if (lane < ((0u - nh) & 3u)) codes[ph + lane] = (uint16_t)kNoCode;
            if (lane == 0 && (nt & 1u)) tails[pt] = kTailPad;
            if (bm) hs.units[first - kTopUnits + lane] = (uint64_t)word[2 * lane + 1] << 32 | word[2 * lane];
            if (lane == 0) hs.rec[r] = make_rec(first, units, (nt + 1) / 2, bm ? 1u : 0u);
        }
    }
}

static uint64_t hub_units(uint64_t rows, uint64_t m) { return m / 2 + 2 * rows + 64; }

bool hub_fits(uint64_t rows, uint64_t m, bool split) {
    return m >= (split ? kMinArcs : kMinArcsPlain) && m >= kMinPerRow * rows && rows < (1ull << 32) &&
           hub_units(rows, m) < (1ull << 29);
}

bool hub_worth(uint64_t rows, uint64_t owned, uint64_t m, bool split) {
    return owned == rows || (double)m * (double)owned >= (split ? kMinOwned : kMinOwnedPlain) * (double)rows;
}

HubSet hub_layout(Carver &c, uint64_t rows, uint64_t m) {
    HubSet h{};
    h.hctl = c.take<uint32_t>(HC_WORDS);
    h.cnt = c.take<uint32_t>(rows + 1);
    h.code = c.take<uint16_t>(rows + 1);
    h.rec = c.take<uint64_t>(rows + 1);
    h.long_rows = c.take<uint32_t>(m / kLongRow + 1);
    h.units = c.take<uint64_t>(hub_units(rows, m));
    h.plan_cnt = c.take<uint32_t>((size_t)kHubSlots * kHubPlanWaves);
    h.plan_waves = (uint32_t)hmin<uint64_t>(kHubPlanWaves, (rows + 2047) / 2048 * 4);  // a multiple of four
    // a row of n >= kHeavy lists has at most n / 64 items, any other one; all rows have at most 2 m lists
    h.queue = c.take<uint64_t>(rows + m / 32 + 1);
    return h;
}

lstc_status hub_build(const GraphDev &g, uint64_t m, const HubSet &hs, hipStream_t st) {
    const uint32_t n = g.n_rows, cus = (uint32_t)device_cus();
    const uint32_t stride = (uint32_t)hmax<uint64_t>(kMinStride, m / kSamples);
    const uint32_t blocks = ceil_div_u32(n, 256);  // a wave per 64 rows
    const uint32_t flat = hmin(hmin(blocks, cus * 4), kInitBlocks);
    hipLaunchKernelGGL(k_hub_init, dim3(flat), dim3(256), 0, st, hs, g.off, n);
    LSTC_LAUNCHED("k_hub_init");
    hipLaunchKernelGGL(k_hub_sample, dim3(cus * 8), dim3(256), 0, st, g, stride, hs, flat,
                       g.in_off != nullptr);
    LSTC_LAUNCHED("k_hub_sample");
    hipLaunchKernelGGL(k_hub_pick, dim3(hmin(blocks, cus)), dim3(256), 0, st, g, (const uint32_t *)hs.cnt,
                       g.in_off != nullptr, hs.hctl);
    LSTC_LAUNCHED("k_hub_pick");
    hipLaunchKernelGGL(k_hub_assign, dim3(hmin(ceil_div_u32(n, 4096), cus * 8)), dim3(256), 0, st,
                       (const uint32_t *)hs.cnt, n, hs.hctl, hs.code);
    LSTC_LAUNCHED("k_hub_assign");
    hipLaunchKernelGGL(k_hub_short, dim3(blocks), dim3(256), 0, st, g, hs);
    LSTC_LAUNCHED("k_hub_short");
    hipLaunchKernelGGL(k_hub_long, dim3(cus * 8), dim3(256), 0, st, g, hs);
    LSTC_LAUNCHED("k_hub_long");
    return LSTC_OK;
}

}  // namespace lstc
