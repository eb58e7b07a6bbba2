// The workers' LDS sorts of their shares of a wide nucleus, and the group records they leave for the tail.
#pragma once

#include "lds_sort.h"
#include "radix_sort.h"
#include "sorted_tail.h"
#include "unsorted_shares.h"

namespace mako {

// The worker's share as the second pass left it (cnt <= kSegCap entries, bits(q) in ks and token ids in is, any
// order): asked for with fetch_staged_share() (the loads stay in flight while the caller goes on), sorted into
// kout / iout by lds_sort_staged().
struct StagedShare {
    uint32_t k[kSortPer], id[kSortPer];
};
__device__ __forceinline__ void fetch_staged_share(const uint32_t* ks, const uint32_t* is, uint32_t cnt, StagedShare& s)
{
    const GlobalKeys gk{ks}, gi{is};
#pragma unroll
    for (uint32_t t = 0; t < kSortPer; ++t) { // (all loads first, from clamped positions; cnt > 0)
        const uint32_t e = min(t * kThreads + threadIdx.x, cnt - 1u);
        s.k[t] = gk[e];
        s.id[t] = gi[e];
    }
}
__device__ __forceinline__ bool lds_sort_staged(StagedShare& s, uint32_t key_lo, uint32_t key_hi, uint32_t cnt,
                                                uint32_t* kout, uint32_t* iout, unsigned long long* dyn, FinishShared& sm,
                                                uint32_t* sorted_lds = nullptr)
{
    uint32_t* hist = reinterpret_cast<uint32_t*>(dyn + kSegCap + 4u); // (lds_bucket_sort()'s)
    const uint32_t tid = threadIdx.x;
    for (uint32_t b = tid; b <= kFine; b += kThreads)
        hist[b] = 0;
    if (tid == 0)
        sm.flag = 0;
    lds_barrier();
#pragma unroll
    for (uint32_t t = 0; t < kSortPer; ++t) {
        uint32_t k = s.k[t];
        asm volatile("" : "+v"(k)); // (used here and not before: the loads are to be waited for no earlier)
        s.k[t] = min(max(k, key_lo), key_hi - 1u); // (clamped: a bucket index is always valid)
    }
    MAKO_STAMP(13);
    return lds_bucket_sort(s.k, s.id, cnt, key_lo, key_hi, kout, iout, dyn, sm, sorted_lds);
}

// A share too large for one LDS sort is cut by value into runs that fit: one counting sweep over the share (the
// same kFine buckets as the sort uses) finds run boundaries at bucket edges (plan_runs()), then each run is collected from
// the share and sorted on its own.  Returns the runs, 0 (the caller falls back to the radix sort through global memory)
// when a single bucket holds more than fits.  Run r covers buckets [sm.hist[r], sm.hist[64 + r]) = entries
// [sm.run[r], sm.run[r] + sm.run[64 + r]) of the sorted share.
__device__ uint32_t plan_runs(const uint32_t* ks, uint32_t key_lo, uint32_t key_hi, uint32_t cnt, unsigned long long* dyn, FinishShared& sm)
{
    uint32_t* hist = reinterpret_cast<uint32_t*>(dyn + kSegCap + 4u); // [kFine + 1] (lds_bucket_sort()'s)
    const uint32_t tid = threadIdx.x;
    const uint32_t range = key_hi - key_lo;
    const uint32_t shift = range > kFine ? 32u - (uint32_t)__clz((range - 1u) >> 11) : 0u;
    for (uint32_t b = tid; b <= kFine; b += kThreads)
        hist[b] = 0;
    __syncthreads();
    constexpr uint32_t kTrip = 8; // loads in flight per thread: the sweep is bound by memory latency
    for (uint32_t base = 0; base < cnt; base += kTrip * kThreads) {
        uint32_t k[kTrip];
#pragma unroll
        for (uint32_t u = 0; u < kTrip; ++u)
            k[u] = ks[min(base + u * kThreads + tid, cnt - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < kTrip; ++u)
            if (base + u * kThreads + tid < cnt)
                atomicAdd(&hist[(key_hi - 1u - min(max(k[u], key_lo), key_hi - 1u)) >> shift], 1u);
    }
    __syncthreads();
    // bucket starts (exclusive scan), kept in sm.hist / sm.run as run boundaries below
    uint32_t total;
    uint32_t c[kFinePer], mine = 0;
#pragma unroll
    for (uint32_t j = 0; j < kFinePer; ++j) {
        c[j] = hist[kFinePer * tid + j];
        mine += c[j];
    }
    uint32_t ex = block_excl_scan_u32(mine, total, sm.bs);
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kFinePer; ++j) {
        hist[kFinePer * tid + j] = ex;
        ex += c[j];
    }
    if (tid == 0)
        hist[kFine] = total;
    __syncthreads();
    // runs: greedily as many whole buckets as fit (thread 0; a handful of runs)
    if (tid == 0) {
        uint32_t runs = 0, b0 = 0;
        while (b0 < kFine && runs < 64u) {
            uint32_t b1 = b0 + 1u;
            if (hist[b1] - hist[b0] > kRunMost) { // one bucket alone is too much
                runs = 0;
                b0 = kFine;
                break;
            }
            { // the last bucket edge within reach: the bucket starts never decrease, so bisect
                uint32_t lo = b1, hi = kFine;
                while (lo < hi) {
                    const uint32_t mid = (lo + hi + 1u) / 2u;
                    if (hist[mid] - hist[b0] <= kRunMost)
                        lo = mid;
                    else
                        hi = mid - 1u;
                }
                b1 = lo;
            }
            if (hist[b1] != hist[b0]) {
                sm.hist[runs] = b0;
                sm.hist[64u + runs] = b1;
                sm.run[runs] = hist[b0];
                sm.run[64u + runs] = hist[b1] - hist[b0];
                ++runs;
            }
            b0 = b1;
        }
        sm.ticket = b0 < kFine ? 0u : runs;
    }
    __syncthreads();
    const uint32_t runs = sm.ticket;
    __syncthreads();
    return runs;
}

// Run r's n entries, those of the share with lo_r <= bits(q) < hi_r, as fetch_staged_share() leaves a whole share.
__device__ bool collect_run(const uint32_t* ks, const uint32_t* is, uint32_t key_lo, uint32_t key_hi, uint32_t cnt, uint32_t lo_r, uint32_t hi_r,
                            uint32_t n, unsigned long long* dyn, FinishShared& sm, StagedShare& s)
{
    uint2* A = reinterpret_cast<uint2*>(dyn);
    const uint32_t tid = threadIdx.x, lane = lane_id();
    __syncthreads();
    if (tid == 0)
        sm.ticket = 0;
    __syncthreads();
    constexpr uint32_t kTrip = 6;
    const unsigned long long lower = (1ull << lane) - 1ull;
    for (uint32_t base = 0; base < cnt; base += kTrip * kThreads) {
        uint32_t k[kTrip], id[kTrip];
#pragma unroll
        for (uint32_t u = 0; u < kTrip; ++u) {
            const uint32_t e = min(base + u * kThreads + tid, cnt - 1u);
            k[u] = ks[e];
            id[u] = is[e];
        }
        // slots for the whole trip from one LDS atomic per wave
        bool mine[kTrip];
        uint32_t before = 0, wave_total = 0;
#pragma unroll
        for (uint32_t u = 0; u < kTrip; ++u) {
            k[u] = min(max(k[u], key_lo), key_hi - 1u);
            mine[u] = base + u * kThreads + tid < cnt && k[u] >= lo_r && k[u] < hi_r;
            const unsigned long long bal = __ballot(mine[u]);
            before += (uint32_t)__popcll(bal & lower);
            wave_total += (uint32_t)__popcll(bal);
        }
        if (wave_total) { // uniform
            uint32_t slot = 0;
            if (lane == 0)
                slot = atomicAdd(&sm.ticket, wave_total);
            slot = uniform_u32(slot) + before;
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u)
                if (mine[u]) {
                    if (slot < kSegCap)
                        A[slot] = make_uint2(k[u], id[u]);
                    ++slot;
                }
        }
    }
    __syncthreads();
    if (sm.ticket != n) // (cannot happen: the same keys were counted by plan_runs())
        return false;
#pragma unroll
    for (uint32_t t = 0; t < kSortPer; ++t) {
        const uint2 x = A[min(t * kThreads + tid, n - 1u)];
        s.k[t] = x.x;
        s.id[t] = x.y;
    }
    __syncthreads(); // (the sort puts the entries there again, in the order of their buckets)
    return true;
}

// ---- shares that need no sorting (unsorted_shares.h) ---------------------------------------------------------------
//
// The record of an unsorted share, by ONE wave (a collector workgroup's waves take a share each: no barrier,
// nothing shared).  ks: the share's cnt weights as bits(q), in device memory, any order.  `lds`: kOpaqueLdsWords words
// of LDS of the wave's own.  The share is streamed once (sixteen loads per lane in flight): its fp64 sum, its largest
// weight, the sums of the increments of the weights that are no exact ties, and the ties themselves (kept apart, up
// to kOpaqueTies of either kind); only a share with ties is streamed again, for the sums between neighbouring ties.
constexpr uint32_t kOpaqueLdsWords = 4u * kOpaqueTies;
__device__ void opaque_share(const uint32_t* ks, uint32_t cnt, uint32_t off, int e_tot, int e_walk, GroupRec* rec, uint32_t* lds)
{
    using namespace seqfp;
    constexpr uint32_t kTrip = 16;
    uint32_t* tie_key = lds;                       // [2][kOpaqueTies] as found
    uint32_t* tie_sorted = lds + 2u * kOpaqueTies; // [2][kOpaqueTies] heaviest first
    const GlobalKeys gk{ks};
    const uint32_t lane = (uint32_t)lane_id();
    const unsigned long long lower = (1ull << lane) - 1ull;
    // (weights and epochs of such a share: the weights lie binades below; e_walk 0: no map for the walk)
    const float base_t = binade_base(e_tot), half_t = half_ulp(e_tot);
    const float base_w = binade_base(e_walk), half_w = half_ulp(e_walk);
    double sum = 0.0;
    uint32_t n_t = 0u, n_w = 0u; // (uniform)
    float acc_t = 0.0f, acc_w = 0.0f; // a lane's multiples of the epochs' last places: exact up to 2^24 of them, beyond after that
    for (uint32_t base = 0; base < cnt; base += kTrip * kWave) {
        uint32_t k[kTrip];
#pragma unroll
        for (uint32_t u = 0; u < kTrip; ++u)
            k[u] = gk[min(base + u * kWave + lane, cnt - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < kTrip; ++u) {
            const uint32_t kv = base + u * kWave + lane < cnt ? k[u] : 0u;
            const float q = __uint_as_float(kv);
            sum += (double)q;
            const float t = increment(q, base_t);
            const bool tie_t = is_tie(q, t, half_t);
            acc_t += tie_t ? 0.0f : t;
            const unsigned long long bal_t = __ballot(tie_t);
            if (bal_t) { // (uniform, rare)
                const uint32_t slot = n_t + (uint32_t)__popcll(bal_t & lower);
                if (tie_t && slot < kOpaqueTies)
                    tie_key[slot] = kv;
                n_t += (uint32_t)__popcll(bal_t);
            }
            if (e_walk > 0) { // uniform
                const float w = increment(q, base_w);
                const bool tie_w = is_tie(q, w, half_w);
                acc_w += tie_w ? 0.0f : w;
                const unsigned long long bal_w = __ballot(tie_w);
                if (bal_w) {
                    const uint32_t slot = n_w + (uint32_t)__popcll(bal_w & lower);
                    if (tie_w && slot < kOpaqueTies)
                        tie_key[kOpaqueTies + slot] = kv;
                    n_w += (uint32_t)__popcll(bal_w);
                }
            }
        }
    }
    const double sum64 = __ockl_wfred_add_f64(sum);
    // One kind of increments: the sum of the multiples between neighbouring ties (heaviest first), with each tie's own
    // two-valued step composed in at its place.
    auto share_incs = [&](uint32_t which, uint32_t n, int e, float from, float half, float acc) {
        if (e <= 0 || n > kOpaqueTies) // uniform
            return make_float2(INFINITY, INFINITY);
        const float all = readlane_f32(wave_scan_add_f32(acc), kWave - 1);
        const uint32_t units = all < binade_top(e) ? (uint32_t)__builtin_ldexpf(all, 150 - e) : kSat; // (below 2^24, and whole)
        if (n == 0u)
            return make_float2(all, all);
        // the ties by weight, heaviest first (equal ones in any order: they are the same step)
        __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0): the wave's own writes of the ties
        const uint32_t mine = lane < n ? tie_key[which * kOpaqueTies + lane] : 0u;
        uint32_t rank = 0;
        for (uint32_t j = 0; j < n; ++j) {
            const uint32_t other = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)j);
            rank += (other > mine || (other == mine && j < lane)) ? 1u : 0u;
        }
        if (lane < n)
            tie_sorted[which * kOpaqueTies + rank] = mine;
        __builtin_amdgcn_s_waitcnt(0xc07f);
        // the share again, once per tie: the multiples of the weights above it (and no tie themselves)
        Step32 v = identity32();
        uint32_t taken = 0u;
        for (uint32_t i = 0; i < n && units != kSat; ++i) {
            const uint32_t tk = uniform_u32(tie_sorted[which * kOpaqueTies + i]);
            float part = 0.0f;
            for (uint32_t base = 0; base < cnt; base += kTrip * kWave) {
                uint32_t k[kTrip];
#pragma unroll
                for (uint32_t u = 0; u < kTrip; ++u)
                    k[u] = gk[min(base + u * kWave + lane, cnt - 1u)];
#pragma unroll
                for (uint32_t u = 0; u < kTrip; ++u) {
                    const float q = __uint_as_float(k[u]);
                    const float t = increment(q, from);
                    part += (base + u * kWave + lane < cnt && k[u] > tk && !is_tie(q, t, half)) ? t : 0.0f;
                }
            }
            const uint32_t above = (uint32_t)__builtin_ldexpf(readlane_f32(wave_scan_add_f32(part), kWave - 1), 150 - e);
            v = compose32(v, Step32{above - taken, above - taken});
            v = compose32(v, step32_flat(__uint_as_float(tk), e));
            taken = above;
        }
        const uint32_t rest = units == kSat ? kSat : units - taken;
        v = compose32(v, Step32{rest, rest});
        auto as_float = [e](uint32_t d) { return d < (1u << 24) ? __builtin_ldexpf((float)d, e - 150) : INFINITY; };
        return make_float2(as_float(v.d0), as_float(v.d1));
    };
    const float2 m0 = share_incs(0u, n_t, e_tot, base_t, half_t, acc_t);
    const float2 m1 = share_incs(1u, n_w, e_walk, base_w, half_w, acc_w);
    if (lane == 0u)
        store_group_rec(rec, sum64, m0, m1, off, kOpaque | ((uint32_t)e_tot << kSumExpShift) | ((uint32_t)max(e_walk, 0) << kWalkExpShift));
}

// The record of one group (q: its entries, four per lane; `before` / `after`: the mass in front of it and behind it; r0:
// the estimate of where the walk starts): increments only where the binade is not expected to change inside the group,
// which is replayed there.  (A walk that starts at 0 passes the groups in front of the first weight.  Left without increments
// for that, 64 rows drawn at u = 0 behind a masked half of 129 280 logits took 372 us, with them 84.)  One wave.
__device__ __forceinline__ void group_record(const float (&q)[4], uint32_t start, uint32_t len, double sum, double before, double after, double r0,
                                             GroupRec* rec)
{
    const uint32_t es = uniform_u32((uint32_t)exponent_of((float)before)), es_end = uniform_u32((uint32_t)exponent_of((float)after));
    float2 inc = make_float2(INFINITY, INFINITY), walk = inc;
    if (es == es_end)
        inc = span_incs(q, (int)es);
    const double r_here = r0 - before, r_after = r0 - after;
    uint32_t ew = 0;
    if (uniform_u32(r_here >= 0.0 && r_after >= 0.0 ? 1u : 0u)) {
        ew = uniform_u32((uint32_t)exponent_of((float)r_here));
        if (ew == es && es == es_end && ew == uniform_u32((uint32_t)exponent_of((float)r_after)))
            walk = inc; // (one binade for both)
        else if (ew == uniform_u32((uint32_t)exponent_of((float)r_after)))
            walk = span_incs(q, (int)ew);
        else
            ew = 0;
    }
    if (lane_id() == 0)
        store_group_rec(rec, sum, inc, walk, start, len | (es << kSumExpShift) | (ew << kWalkExpShift));
}

// Group records of a worker's sorted range (cnt entries from position off of the list kf).
// kf_lds (optional): the worker's cnt sorted weights in LDS (outside L.sortk's first 16 KB), read instead of kf + off.
// mass: the estimate of the sum above the range; r0: of where the walk starts, u * top_p * (the row's total).
__device__ void worker_groups(const uint32_t* kf, uint32_t off, uint32_t cnt, GroupRec* rec, double mass, const FinishLds L,
                              const uint32_t* kf_lds = nullptr, double r0 = 0.0)
{
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x;
    const uint32_t* src = kf_lds ? kf_lds : kf + off; // uniform
    double* gs = reinterpret_cast<double*>(L.sortk); // [groups] their sums
    double* gb = gs + kMaxGroups;                    // [groups] the estimate of the sum before each
    const uint32_t groups = (cnt + kGroup - 1u) / kGroup;
    if (kf_lds) // uniform: the copy is in place (its writers' barrier), nothing in device memory is waited for
        lds_barrier();
    else
        __syncthreads();
    for (uint32_t g = wave_id(); g < groups; g += kWaves) {
        float q[4];
        load_span(src, g * kGroup, min(kGroup, cnt - g * kGroup), q);
        const double s = __ockl_wfred_add_f64((((double)q[0] + (double)q[1]) + (double)q[2]) + (double)q[3]);
        if (lane_id() == 0)
            gs[g] = s;
    }
    MAKO_STAMP(16);
    // the sums before each group.  Up to a wave's worth of groups, every wave scans them for itself (the values are those
    // of the workgroup's scan, whose first wave adds them up the same way) and goes on at once.
    const bool few = groups <= (uint32_t)kWave; // uniform
    double before_l = 0; // (few: lane g holds group g's)
    if (few) {
        if (kf_lds)
            lds_barrier();
        else
            __syncthreads();
        const double v = (uint32_t)lane_id() < groups ? gs[lane_id()] : 0.0;
        before_l = mass + (__ockl_wfscan_add_f64(v, true) - v);
    } else {
        __syncthreads();
        for (uint32_t g0 = 0; g0 < groups; g0 += kThreads) {
            const uint32_t g = g0 + tid;
            const double v = g < groups ? gs[g] : 0.0;
            double all;
            const double incl = block_incl_scan_f64(v, all, sm.bs);
            if (g < groups)
                gb[g] = mass + (incl - v);
            mass += all;
        }
        __syncthreads();
    }
    MAKO_STAMP(19);
    for (uint32_t g = wave_id(); g < groups; g += kWaves) {
        const uint32_t len = min(kGroup, cnt - g * kGroup);
        float q[4];
        load_span(src, g * kGroup, len, q);
        const double before = few ? readlane_f64(before_l, g) : gb[g], sum = gs[g];
        group_record(q, off + g * kGroup, len, sum, before, before + sum, r0, rec + g);
    }
}

} // namespace mako
