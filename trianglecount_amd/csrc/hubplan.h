// hubplan.h -- the work queue of a count over hub codes (hubcode.h), written by the
// engine's plan kernels in place of their own queue when the launch uses codes.
#pragma once
#include "hubcode.h"
#include "wave.h"

namespace lstc {

// As the engine's plan, but each wave has every plan_waves-th group of 64 rows
// (heavy rows often lie together: 325 -> 64 us at RMAT s23 for the writing pass
// against contiguous ranges): pass 0 counts its items per queue region,
// hub_plan_scan turns that into positions, pass 1 writes the items.  Lane s keeps
// the counter of region s.  Tiny rows are those of up to kTinyMax entries whatever the
// tune says (limits of 8, 4 and none, ms a call: RMAT s21 2.15, 2.25, 2.36, s23 10.26, 10.54, 11.05, where ids
// are fastest with 4).
template <int PASS>
__device__ __forceinline__ void hub_plan_rows(const GraphDev &G, const HubSet &hs) {
    if (blockIdx.x * 4 >= hs.plan_waves) return;
    const uint32_t lane = threadIdx.x & 63, wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const uint64_t end = G.n_rows;
    uint32_t run = 0;
    if (PASS == 1 && lane < kHubSlots) run = hs.plan_cnt[lane * hs.plan_waves + wave];
    const uint32_t xcd = lane / kXcdSlots, step = lane % kXcdSlots;  // of lanes below kSlotLight
    for (uint64_t r0 = wave * 64ull; r0 < end; r0 += hs.plan_waves * 64ull) {
        const uint64_t r = r0 + lane;
        uint32_t n = 0, in_only = 0;
        bool tiny = false;
        if (r < end) {
            const uint32_t k = (uint32_t)(gload(G.off + r + 1) - gload(G.off + r));
            const uint32_t kb = G.in_off ? (uint32_t)(gload(G.in_off + r + 1) - gload(G.in_off + r)) : 0u;
            in_only = r >= G.n_owned;
            tiny = G.in_off && k >= 2 && k <= kTinyMax;
            n = k < 2 ? 0u : (in_only ? 0u : k) + kb;
        }
        for (uint64_t heavy = ballot(n >= kHeavy); heavy; heavy &= heavy - 1) {
            const uint32_t j = (uint32_t)__builtin_ctzll(heavy);
            const HubSplit sp = hub_split(read_lane(n, j));
            // this lane's part of the row, if it has one
            const bool mine = lane < kSlotLight && (sp.parts == kXcds ? step == kSteps : step < kSteps);
            const uint32_t part = sp.parts == kXcds ? xcd : xcd * kSteps + step;
            if (mine) {
                if (PASS == 1) {
                    for (uint32_t i = 0; i < sp.per_part; ++i)
                        hs.queue[run + i] = (r0 + j) | ((uint64_t)(part * sp.per_part + i) << 32);
                }
                run += sp.per_part;
            }
        }
#pragma unroll
        for (uint32_t slot = kSlotLight; slot <= kSlotTiny; ++slot) {
            const bool in = n != 0 && n < kHeavy &&
                            (slot == kSlotTiny ? tiny : !tiny && (slot == kSlotLight ? n >= kLight : n < kLight));
            const uint64_t m = ballot(in);
            if (PASS == 1 && in)
                hs.queue[read_lane(run, slot) + mask_rank(m)] = r | (slot == kSlotTiny ? (uint64_t)in_only << 32 : 0);
            if (lane == slot) run += (uint32_t)__popcll(m);
        }
    }
    if (PASS == 0 && lane < kHubSlots) hs.plan_cnt[lane * hs.plan_waves + wave] = run;
}

// One workgroup: exclusive scan of the counters in place, then the tickets.
__device__ __forceinline__ void hub_plan_scan(const HubSet &hs, unsigned long long *counts, uint32_t grid) {
    constexpr uint32_t kRound = 4096;
    const uint32_t all = kHubSlots * hs.plan_waves;  // (a slot starts on a 16-byte word)
    __shared__ uint32_t s_wave[16], s_slot[kHubSlots + 1];
    uint32_t *hctl = hs.hctl;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    uint32_t before = 0;
    for (uint32_t e0 = 0; e0 < all; e0 += kRound) {
        const uint32_t e = e0 + 4 * tid;
        uint4 *p = (uint4 *)(hs.plan_cnt + e);
        uint4 v = e < all ? *p : uint4{0, 0, 0, 0};
        const uint32_t sum = v.x + v.y + v.z + v.w;
        const uint32_t incl = wave_incl_scan(sum, lane);
        __syncthreads();
        if (lane == 63) s_wave[wv] = incl;
        __syncthreads();
        uint32_t run = before + incl - sum;
        for (uint32_t w = 0; w < 16; ++w) {
            run += w < wv ? s_wave[w] : 0u;
            before += s_wave[w];
        }
        if (e < all) {
            if (e % hs.plan_waves == 0) s_slot[e / hs.plan_waves] = run;
            const uint4 q{run, run + v.x, run + v.x + v.y, run + v.x + v.y + v.z};
            *p = q;
        }
    }
    if (tid == 0) s_slot[kHubSlots] = before;
    __syncthreads();
    if (tid < kXcds) {
        const uint32_t a = s_slot[tid * kXcdSlots], b = s_slot[(tid + 1) * kXcdSlots];
        hctl[HC_OWN0 + tid] = a;
        hctl[HC_OWN_END + tid] = b;
        hctl[HC_OWN_T + tid] = (b - a + kOwnGroup - 1) / kOwnGroup;
        hctl[HC_HEADS + 32 * tid] = (grid + kXcds - 1 - tid) / kXcds;  // behind the waves' first tickets
    }
    if (tid == 0) {
        counts[0] = 0;
        const uint32_t light = s_slot[kSlotSmall] - s_slot[kSlotLight], small = s_slot[kSlotTiny] - s_slot[kSlotSmall];
        const uint32_t tiny = s_slot[kHubSlots] - s_slot[kSlotTiny];
        hctl[HC_LIGHT0] = s_slot[kSlotLight];
        hctl[HC_LIGHT] = light;
        hctl[HC_LIGHT_T] = (light + kLightGroup - 1) / kLightGroup;
        hctl[HC_SMALL0] = s_slot[kSlotSmall];
        hctl[HC_SMALL] = small;
        hctl[HC_SMALL_T] = (small + kSmallGroup - 1) / kSmallGroup;
        hctl[HC_TINY0] = s_slot[kSlotTiny];
        hctl[HC_TINY] = tiny;
        hctl[HC_TINY_T] = (tiny + 63) / 64;
    }
}

}  // namespace lstc
