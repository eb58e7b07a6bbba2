// The whole-row path: exact for every parameter combination, one workgroup per row.
#pragma once

#include "lds_sort.h"
#include "nth_steps.h"
#include "radix_sort.h"
#include "slice_load.h"
#include "sorted_tail.h"

namespace mako {

__device__ void sort_survivors(uint32_t* k0, uint32_t* i0, uint32_t* k1, uint32_t* i1, uint32_t n, const FinishLds& L);
__device__ MAKO_RARE_CALL bool sort_picked(uint32_t* k0, uint32_t* i0, uint32_t n, uint32_t key_lo, const FinishLds& L);

// libstdc++'s __heap_select(first, nth + 1, last) followed by iter_swap(first, nth) (bits/stl_algo.h:1956-1960,
// stl_heap.h): where introselect ends up when its depth limit is spent.  The arrangement it leaves is the library's,
// entry for entry, but the time is bounded:
//  * __make_heap sifts the parents from the last one down to the root.  A sift only touches the subtree of its
//    node and the subtrees of one level are disjoint, so a level's sifts run side by side, one thread each, level
//    after level from the bottom: the heap's depth in rounds instead of its size in dependent steps.
//  * the sweep `for (i = middle; i < last; ++i) if (comp(i, first)) __pop_heap(...)` is done by one wave, 64 entries
//    per ballot against the current root: entries that do not beat the root cost nothing, the first that does is
//    popped in (a sequential sift from the root), the lanes behind it are asked again (the root only ever moves
//    towards the heavy end, so whoever failed before fails again).
//  * the heap's first `cache_cap` entries (its upper levels, or all of it) live in LDS while this runs.
// get / put: the range in device memory.  cache: room for cache_cap values in LDS.  All threads call.
template <typename Get, typename Put>
__device__ void heap_select_rest(Get get, Put put, uint32_t first, uint32_t last, uint32_t nth, lds_ptr<unsigned long long> cache,
                                 uint32_t cache_cap)
{
    typedef unsigned long long u64;
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const uint32_t middle = nth + 1u - first, len = last - first;
    const uint32_t cached = min(middle, cache_cap);
    for (uint32_t i = tid; i < cached; i += kThreads)
        cache[i] = get(first + i);
    __syncthreads();
    auto hget = [&](uint32_t j) -> u64 { return j < cached ? cache[j] : get(first + j); };
    auto hput = [&](uint32_t j, u64 v) {
        if (j < cached)
            cache[j] = v;
        else
            put(first + j, v);
    };
    auto sift = [&](uint32_t hole, u64 v) { // __adjust_heap: the hole sinks to a leaf, v rises from there
        const uint32_t top = hole;
        uint32_t child = hole;
        while (child < (middle - 1u) / 2u) {
            child = 2u * (child + 1u);
            if (hget(child) < hget(child - 1u))
                --child;
            hput(hole, hget(child));
            hole = child;
        }
        if ((middle & 1u) == 0 && middle >= 2u && child == (middle - 2u) / 2u) {
            child = 2u * (child + 1u);
            hput(hole, hget(child - 1u));
            hole = child - 1u;
        }
        while (hole > top) {
            const uint32_t parent = (hole - 1u) / 2u;
            if (!(hget(parent) < v))
                break;
            hput(hole, hget(parent));
            hole = parent;
        }
        hput(hole, v);
    };
    if (middle >= 2u) {
        const uint32_t last_parent = (middle - 2u) / 2u;
        // (node p sits on level floor(log2(p + 1)), which holds the nodes 2^level - 1 .. 2^(level + 1) - 2)
        for (int level = 31 - __clz((int)(last_parent + 1u)); level >= 0; --level) {
            const uint32_t lo = (1u << level) - 1u, hi = min(last_parent, (2u << level) - 2u);
            for (uint32_t p = lo + tid; p <= hi; p += kThreads)
                sift(p, hget(p));
            __syncthreads();
        }
    }
    if (wave_id() == 0 && middle < len) {
        constexpr uint32_t kTrip = 4;
        u64 root = hget(0u); // (the same in every lane)
        for (uint32_t base = middle; base < len; base += kWave * kTrip) {
            u64 v[kTrip];
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u)
                v[u] = get(first + min(base + u * kWave + lane, len - 1u));
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u) {
                const bool in = base + u * kWave + lane < len;
                u64 bal = __ballot(in && v[u] < root);
                while (bal) { // uniform
                    const int l = __ffsll((long long)bal) - 1;
                    const u64 hit = ((u64)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v[u] >> 32), l) << 32) |
                                    (u64)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v[u], l);
                    // __pop_heap(first, middle, i): the root goes to the entry's place, the entry sinks in from the root
                    // (every lane does the same stores and loads: each then reads back what it wrote itself)
                    put(first + base + u * kWave + (uint32_t)l, root);
                    sift(0u, hit);
                    root = hget(0u);
                    bal = __ballot(in && v[u] < root) & ~((2ull << l) - 1ull);
                }
            }
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < cached; i += kThreads)
        put(first + i, cache[i]);
    __syncthreads();
    if (tid == 0) {
        const u64 a = get(first), b = get(nth);
        put(first, b);
        put(nth, a);
    }
    __syncthreads();
}

// std::ranges::nth_element(cand, cand + nth, desc) of src/gen/sampler.cpp:41 as libstdc++ 11 runs it (introselect,
// bits/stl_algo.h:1964), leaving the first nth candidates in exactly the arrangement that library leaves: the
// reference keeps those (sampler.cpp:42) and sums and walks them in that order when no top-p follows.  What lies behind
// a cut that the rounds leave behind them is not kept up.  key/idx hold n candidates (~bits(q), token id); `desc` is
// the order of the 64-bit values key << 32 | idx, all distinct.
// One round = median of three to the front, then the unguarded Hoare partition of the rest around it.  That
// partition swaps the t-th entry from the left that belongs right ("hole") with the t-th entry from the right that belongs
// left ("filler") for as long as the former lies before the latter, and cuts behind the entries that belong left.
// Three ways to make a round, as the range shrinks (nth_element_row()), behind those that several workgroups have made of a long
// row (nth_steps.h):
//   in device memory   nth_rounds_memory(): one pass over the keys, sixteen bytes per lane and load, leaves a bit per
//                      entry in LDS; what changes places goes through LDS block by block;
//   in registers       nth_rounds_registers(): up to kNthRegs entries, sixteen per thread; what changes places goes through LDS;
//   by one wave        nth_rounds_wave(): up to kNthWave entries, four per lane, without a barrier.
// The depth limit's heap select is heap_select_rest() above.
// (A batch of 32 rows of 12 000 candidates, 40 kept: 81 us with every round in device memory or LDS, two passes over the keys
// each and through pointers that the compiler could not tell from each other; 60 us now.  64 rows of 129 280, bound by the
// rounds in device memory of the row with the unluckiest pivots: 225 to 235 us, 150 to 162 with the first rounds made by several
// workgroups; one such row 144, 72 so.)
constexpr uint32_t kNthChunks = 4;                                     // of four entries in a row per thread:
constexpr uint32_t kNthRegs = kNthChunks * 4u * (uint32_t)kThreads; // what a workgroup takes into registers
constexpr uint32_t kNthWave = 256;                                     // and one wave
static_assert(kNthUntil == kNthRegs - 4u, "wherever the range begins, from a multiple of four on");

// Rounds on entries [first, last) in device memory until no more than `until` are left or the depth limit is reached.
// far: room for n / 32 words of device memory behind which nobody looks (the bits of ranges that LDS has no room for).
// ready: the first round's pivot is at `first` already, and these are its bits (nth_steps.h); nullptr: they are not.
// lds: kTailLds bytes.  All threads call.
// (A workgroup's four SIMDs look at 256 entries a cycle, one instruction each, and a CU fetches 40 GB/s from the memory
// behind its L2: a row of 129 280 keys takes it 13 us to read, 0.2 us to give one instruction to.  So the keys are read
// once a round, a bit per entry is kept in LDS, and the entries that change places are read and written where they lie, block
// by block, through LDS.  The first round of such a row takes 49 us: the keys 14, what moves 33.)
__device__ __forceinline__ void nth_rounds_memory(global_ptr<uint32_t> key, global_ptr<uint32_t> idx, uint32_t& first, uint32_t& last, uint32_t nth,
                                                  uint32_t& depth, uint32_t until, global_ptr<uint32_t> far, const uint32_t* ready,
                                                  lds_ptr<unsigned long long> lds, FinishShared& sm)
{
    typedef unsigned long long u64;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    static_assert(kGroup == 4u * (uint32_t)kWave, "a block of entries: entry 64 j + l is lane l's j-th");
    constexpr uint32_t kBlocksMax = (kMaxSlices * kSliceMax) / kGroup + 1u, kBlocksInLds = 2048;
    static_assert(kBlocksMax <= 4u * (uint32_t)kThreads + 1u && kTailLds >= kBlocksInLds * 36u + 8192u && kTailLds >= (kBlocksMax + 1u) * 4u + 8192u, "");
    while (last - first > until && depth > 0u) {
        --depth;
        const uint32_t lo = uniform_u32(first + 1u), end = uniform_u32(last);
        if (wave == 0 && !ready) { // (one trip to memory)
            const uint32_t ix = lo, iy = first + (end - first) / 2u, iz = end - 1u;
            const uint32_t p = lane == 0 ? ix : (lane == 1 ? iy : (lane == 2 ? iz : first));
            const uint32_t k = key[p], i = idx[p];
            auto at = [&](int l) { return ((u64)(uint32_t)__builtin_amdgcn_readlane((int)k, l) << 32) | (u64)(uint32_t)__builtin_amdgcn_readlane((int)i, l); };
            u64 med;
            uint32_t im;
            median_of_three(at(0), at(1), at(2), ix, iy, iz, med, im);
            if (lane == 3) {
                key[im] = k;
                idx[im] = i;
                key[first] = (uint32_t)(med >> 32);
                idx[first] = (uint32_t)med;
                sm.bs.f64[0] = __longlong_as_double((long long)med); // (the pivot, for everyone)
            }
        }
        __syncthreads();
        const u64 pivot = (u64)__double_as_longlong(sm.bs.f64[0]); // (of no use where the bits are there)
        const uint32_t pivot_key = uniform_u32((uint32_t)(pivot >> 32)), pivot_id = uniform_u32((uint32_t)pivot);
        // blocks of 256 positions, to the waves in turn
        const uint32_t b0 = lo / kGroup, n_blocks = (end - 1u) / kGroup + 1u - b0;
        const bool bits_in_lds = n_blocks <= kBlocksInLds; // uniform
        // LDS: smalls before each block, the blocks' bits (four words, word j: the entries at 64 j + l), entries on the move
        const lds_ptr<uint32_t> pre = (lds_ptr<uint32_t>)lds;
        const lds_ptr<u64> bits = lds + (n_blocks + 2u) / 2u;
        const global_ptr<u64> bits_far = (global_ptr<u64>)far;
        const lds_ptr<u64> moving = bits + (bits_in_lds ? n_blocks * 4u : 0u);
        const uint32_t room = kTailLds / 8u - (n_blocks + 2u) / 2u - (bits_in_lds ? n_blocks * 4u : 0u);
        constexpr uint32_t kTrip = 8, kFills = 4;
        if (ready) { // uniform
            const global_ptr<const u64> done = (global_ptr<const u64>)as_global(ready);
            for (uint32_t b = tid; b < n_blocks; b += (uint32_t)kThreads) {
                uint32_t n = 0;
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    const u64 m = done[(b0 + b) * 4u + j];
                    n += (uint32_t)__popcll(m);
                    if (bits_in_lds) // uniform
                        bits[b * 4u + j] = m;
                    else
                        bits_far[b * 4u + j] = m;
                }
                pre[b] = n;
            }
        }
        for (uint32_t b = wave; !ready && b < n_blocks; b += kTrip * (uint32_t)kWaves) {
            uint32_t k[kTrip][4];
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u)
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    k[u][j] = key[(size_t)(b0 + min(b + u * (uint32_t)kWaves, n_blocks - 1u)) * kGroup + (uint32_t)kWave * j + lane];
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u) {
                const uint32_t bb = b + u * (uint32_t)kWaves;
                if (bb >= n_blocks) // uniform
                    break;
                const uint32_t p0 = (b0 + bb) * kGroup;
                u64 m[4], ties = 0;
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    m[j] = __builtin_amdgcn_ballot_w64(k[u][j] < pivot_key);
                    ties |= __builtin_amdgcn_ballot_w64(k[u][j] == pivot_key);
                }
                if (p0 < lo || p0 + kGroup > end) { // uniform: the range's first and last block
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j)
                        m[j] &= __builtin_amdgcn_ballot_w64(p0 + (uint32_t)kWave * j + lane >= lo && p0 + (uint32_t)kWave * j + lane < end);
                }
                if (ties) { // (rare: entries of the pivot's weight)
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t p = p0 + (uint32_t)kWave * j + lane;
                        bool l = false;
                        if (k[u][j] == pivot_key && p >= lo && p < end)
                            l = idx[p] < pivot_id;
                        m[j] |= __builtin_amdgcn_ballot_w64(l);
                    }
                }
                const u64 w = lane == 0 ? m[0] : (lane == 1 ? m[1] : (lane == 2 ? m[2] : m[3]));
                if (lane < 4) {
                    if (bits_in_lds) // uniform
                        bits[bb * 4u + lane] = w;
                    else
                        bits_far[bb * 4u + lane] = w;
                }
                if (lane == 0)
                    pre[bb] = (uint32_t)(__popcll(m[0]) + __popcll(m[1]) + __popcll(m[2]) + __popcll(m[3]));
            }
        }
        __syncthreads();
        ready = nullptr;
        // the counts' prefix sums, up to four blocks a thread
        uint32_t smalls;
        {
            uint32_t c[4], mine = 0;
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                c[j] = 4u * tid + j < n_blocks ? pre[4u * tid + j] : 0u;
                mine += c[j];
            }
            uint32_t at = block_excl_scan_u32(mine, smalls, sm.bs);
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if (4u * tid + j < n_blocks) {
                    pre[4u * tid + j] = at;
                    at += c[j];
                }
            if (tid == 0)
                pre[n_blocks] = smalls;
        }
        __syncthreads();
        smalls = uniform_u32(smalls);
        const uint32_t cut = lo + smalls, cut_block = cut / kGroup - b0;
        // When the rounds go on in the left part (cut > nth), what lies behind the cut is never read again (nth_element's
        // caller keeps the first nth entries only): the holes' entries need not be moved there.
        const bool right_kept = cut <= nth;
        auto block_bits = [&](uint32_t b, u64 (&m)[4]) {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                m[j] = bits_in_lds ? bits[b * 4u + j] : bits_far[b * 4u + j];
        };
        // smalls in front of the cut, of all; so many pairs change places
        uint32_t before_cut = smalls;
        if (cut_block < n_blocks) {
            u64 m[4];
            block_bits(cut_block, m);
            before_cut = pre[cut_block];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                before_cut += (uint32_t)__popcll(m[j] & __builtin_amdgcn_ballot_w64((b0 + cut_block) * kGroup + (uint32_t)kWave * j + lane < cut));
        }
        const uint32_t pairs = uniform_u32(smalls - before_cut);
        // The fillers (small s of all is the filler of pair smalls - 1 - s) go to LDS, from there to the holes (the entry at p
        // is the hole of pair (p - lo) - smalls before it): from the range's end on as many blocks at a time as there is
        // room for the smalls of, up to four a wave, whose loads are in flight together.
        for (uint32_t t0 = 0, b_hi = n_blocks; t0 < pairs;) {
            uint32_t b_lo = b_hi - min(b_hi - cut_block, kFills * (uint32_t)kWaves);
            const uint32_t s_hi = uniform_u32(pre[b_hi]);
            while (s_hi - uniform_u32(pre[b_lo]) > room)
                b_lo = b_hi - (b_hi - b_lo) / 2u;
            const uint32_t s_lo = max(uniform_u32(pre[b_lo]), before_cut), t1 = t0 + (s_hi - s_lo);
            uint32_t k[kFills][4], i[kFills][4];
#pragma unroll
            for (uint32_t u = 0; u < kFills; ++u) {
                const size_t at = (size_t)(b0 + min(b_lo + wave + u * (uint32_t)kWaves, b_hi - 1u)) * kGroup + lane;
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    k[u][j] = key[at + (uint32_t)kWave * j];
                    i[u][j] = idx[at + (uint32_t)kWave * j];
                }
            }
            // (turn 1, where the right part is kept: the holes' entries, left in LDS in the fillers' stead, to the fillers)
            auto fills = [&](bool to_fillers) {
#pragma unroll
                for (uint32_t u = 0; u < kFills; ++u) {
                    const uint32_t b = b_lo + wave + u * (uint32_t)kWaves;
                    if (b >= b_hi) // uniform
                        break;
                    u64 m[4];
                    block_bits(b, m);
                    uint32_t s0 = uniform_u32(pre[b]);
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t s = s0 + mask_rank(m[j]);
                        if (((m[j] >> lane) & 1ull) && s >= s_lo) { // (all but those in front of the cut in its block)
                            if (!to_fillers) {
                                moving[s_hi - 1u - s] = ((u64)k[u][j] << 32) | (u64)i[u][j];
                            } else {
                                const u64 v = moving[s_hi - 1u - s];
                                const uint32_t p = (b0 + b) * kGroup + (uint32_t)kWave * j + lane;
                                key[p] = (uint32_t)(v >> 32);
                                idx[p] = (uint32_t)v;
                            }
                        }
                        s0 += (uint32_t)__popcll(m[j]);
                    }
                }
            };
            fills(false);
            lds_barrier();
            for (uint32_t b = wave; b <= min(cut_block, n_blocks - 1u); b += (uint32_t)kWaves) {
                const uint32_t p0 = (b0 + b) * kGroup, s0 = uniform_u32(pre[b]);
                // holes before the block, and before the next
                const uint32_t h0 = max(p0, lo) - lo - s0, h1 = p0 + kGroup - lo - uniform_u32(pre[b + 1u]);
                if (h1 <= t0 || h0 >= t1) // uniform
                    continue;
                u64 m[4];
                block_bits(b, m);
                uint32_t s = s0;
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    const uint32_t p = p0 + (uint32_t)kWave * j + lane, t = p - lo - (s + mask_rank(m[j]));
                    if (!((m[j] >> lane) & 1ull) && p >= lo && p < cut && t >= t0 && t < t1) {
                        const u64 v = moving[t - t0];
                        if (right_kept)
                            moving[t - t0] = ((u64)key[p] << 32) | (u64)idx[p];
                        key[p] = (uint32_t)(v >> 32);
                        idx[p] = (uint32_t)v;
                    }
                    s += (uint32_t)__popcll(m[j]);
                }
            }
            lds_barrier();
            if (right_kept) { // uniform
                fills(true);
                lds_barrier();
            }
            t0 = t1;
            b_hi = b_lo;
        }
        __syncthreads();
        if (right_kept)
            first = cut;
        else
            last = cut;
    }
}

// Rounds on at most kNthRegs entries in registers: position origin + 4096 c + 4 tid + j is x[c][j] (first, last, nth and the
// positions here: less origin).  buf: kNthRegs / 2 values in LDS.  All threads call.
__device__ __forceinline__ void nth_rounds_registers(unsigned long long (&x)[kNthChunks][4], uint32_t& first, uint32_t& last, uint32_t nth, uint32_t& depth,
                                                     uint32_t until, lds_ptr<unsigned long long> buf, FinishShared& sm)
{
    typedef unsigned long long u64;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    constexpr uint32_t kChunk = 4u * (uint32_t)kThreads;
    const lds_ptr<u64> piv = as_lds(sm.bs.u64);   // [4]
    const lds_ptr<uint32_t> cnt = as_lds(sm.hist); // [kNthChunks][kWaves]
    // (has the wave entries in [first, to)?  If not, the round is over for it but for the barriers, and the four SIMDs are the others':
    // 64 rows of 16 000, top-k alone, 70.2 us with every wave at work in every chunk that the range is in, 67.4 so)
    auto touches = [&](uint32_t c, uint32_t to) {
        const uint32_t at = uniform_u32(c * kChunk + wave * kGroup);
        return at < to && at + kGroup > first;
    };
    while (last - first > until && depth > 0u) {
        --depth;
        first = uniform_u32(first);
        last = uniform_u32(last);
        const uint32_t ps[4] = {first + 1u, first + (last - first) / 2u, last - 1u, first};
        // (the owners of the three, and of the first entry, say what they are)
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (((ps[i] >> 8) & ((uint32_t)kWaves - 1u)) == wave && ((ps[i] >> 2) & 63u) == lane) {
                const uint32_t j = ps[i] & 3u;
#pragma unroll
                for (uint32_t c = 0; c < kNthChunks; ++c)
                    if (ps[i] / kChunk == c) // uniform
                        piv[i] = j == 0u ? x[c][0] : (j == 1u ? x[c][1] : (j == 2u ? x[c][2] : x[c][3]));
            }
        lds_barrier();
        const u64 vr = piv[3];
        u64 med;
        uint32_t im;
        median_of_three((u64)piv[0], (u64)piv[1], (u64)piv[2], ps[0], ps[1], ps[2], med, im);
        const uint32_t lo = first + 1u;
        uint32_t own = 0; // bit 4 c + j: the entry belongs left
#pragma unroll
        for (uint32_t c = 0; c < kNthChunks; ++c) {
            uint32_t mine = 0;
            if (touches(c, last)) { // uniform
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    const uint32_t p = c * kChunk + 4u * tid + j;
                    x[c][j] = p == im ? vr : (p == first ? med : x[c][j]);
                    const bool left = p >= lo && p < last && x[c][j] < med;
                    own |= (left ? 1u : 0u) << (4u * c + j);
                    mine += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(left));
                }
            }
            if (lane == 0)
                cnt[c * (uint32_t)kWaves + wave] = mine;
        }
        lds_barrier();
        static_assert(kNthChunks * (uint32_t)kWaves == (uint32_t)kWave, "a count per lane");
        const uint32_t c_l = cnt[lane], upto = __ockl_wfscan_add_u32(c_l, true);
        const uint32_t smalls = (uint32_t)__builtin_amdgcn_readlane((int)upto, kWave - 1), cut = lo + smalls;
        const bool right_kept = cut <= nth;
        uint32_t place[kNthChunks][4]; // in buf, of what changes places
#pragma unroll
        for (uint32_t c = 0; c < kNthChunks; ++c) {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                place[c][j] = kNone;
            if (!touches(c, last)) // uniform
                continue;
            uint32_t rank = (uint32_t)__builtin_amdgcn_readlane((int)(upto - c_l), (int)(c * (uint32_t)kWaves + wave));
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                rank += mask_rank(__builtin_amdgcn_ballot_w64((own >> (4u * c + j)) & 1u));
            }
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) { // (rank: entries before the position that belong left)
                const uint32_t p = c * kChunk + 4u * tid + j;
                const bool left = (own >> (4u * c + j)) & 1u;
                if (left && p >= cut) { // the t-th from the right
                    place[c][j] = smalls - 1u - rank;
                    buf[place[c][j]] = x[c][j];
                } else if (!left && p >= lo && p < cut) { // the t-th from the left
                    place[c][j] = p - lo - rank;
                }
                rank += left ? 1u : 0u;
            }
        }
        lds_barrier();
#pragma unroll
        for (uint32_t c = 0; c < kNthChunks; ++c)
            if (touches(c, cut)) { // uniform
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    if (place[c][j] != kNone && c * kChunk + 4u * tid + j < cut) {
                        const u64 v = buf[place[c][j]];
                        if (right_kept)
                            buf[place[c][j]] = x[c][j];
                        x[c][j] = v;
                    }
            }
        if (right_kept) { // uniform
            lds_barrier();
#pragma unroll
            for (uint32_t c = 0; c < kNthChunks; ++c)
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    if (place[c][j] != kNone && c * kChunk + 4u * tid + j >= cut)
                        x[c][j] = buf[place[c][j]];
            first = cut;
        } else {
            last = cut;
        }
    }
    first = uniform_u32(first);
    last = uniform_u32(last);
}

// The last rounds by one wave: entries [f, l) of the len <= kNthWave at `range`, four in a lane's registers (entry
// 64 j + lane), of which only those of the range are looked at.  tmp: kNthWave values.  Leaves `range` as introselect arranges
// it; returns false when the depth limit is reached first.  One wave calls.
// (A round of the whole workgroup takes 2 us on a range this short, most of it barriers and trips through LDS; one of a
// wave 0.6 us.  From 512 or 1 024 entries on the wave is the slower one, with 50 instructions per 64 entries.)
__device__ __forceinline__ bool nth_rounds_wave(lds_ptr<unsigned long long> range, uint32_t len, uint32_t& f, uint32_t& l, uint32_t nth,
                                                uint32_t& depth, lds_ptr<unsigned long long> tmp)
{
    typedef unsigned long long u64;
    constexpr uint32_t kItems = kNthWave / (uint32_t)kWave;
    const uint32_t lane = lane_id();
    const lds_ptr<u64> tmp_a = tmp;
    const lds_ptr<u64> tmp_b = tmp + kNthWave / 2u; // (at most half of the entries change places with the other half)
    auto lds_turn = []() { // (a wave's LDS operations complete in order: only the compiler has to be told)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    u64 x[kItems];
#pragma unroll
    for (uint32_t j = 0; j < kItems; ++j)
        x[j] = range[min(j * kWave + lane, len - 1u)];
    f = uniform_u32(f);
    l = uniform_u32(l);
    while (l - f > 3u && depth > 0u) {
        --depth;
        const uint32_t ix = f + 1u, iy = f + (l - f) / 2u, iz = l - 1u;
        // (the three and the first entry through LDS: picked out of the registers they would take a chain of moves)
        const u64 vx = range[ix], vy = range[iy], vz = range[iz], vr = range[f];
        u64 med;
        uint32_t im;
        median_of_three(vx, vy, vz, ix, iy, iz, med, im);
        im = uniform_u32(im);
        const uint32_t lo = f + 1u;
        u64 left[kItems];
        uint32_t smalls = 0;
#pragma unroll
        for (uint32_t j = 0; j < kItems; ++j) {
            left[j] = 0ull;
            if (j * kWave < l && (j + 1u) * kWave > f) { // uniform
                const uint32_t p = j * kWave + lane;
                x[j] = p == f ? med : (p == im ? vr : x[j]);
                left[j] = __builtin_amdgcn_ballot_w64(p >= lo && p < l && x[j] < med);
                smalls += (uint32_t)__popcll(left[j]);
            }
        }
        const uint32_t cut = lo + smalls;
        uint32_t before = 0; // smalls in front of the register's entries
#pragma unroll
        for (uint32_t j = 0; j < kItems; ++j)
            if (j * kWave < l && (j + 1u) * kWave > f) { // uniform
                const uint32_t p = j * kWave + lane, s = before + mask_rank(left[j]);
                const bool is_left = (left[j] >> lane) & 1ull;
                if (is_left && p >= cut)
                    tmp_b[smalls - 1u - s] = x[j];
                if (!is_left && p >= lo && p < cut)
                    tmp_a[p - lo - s] = x[j];
                before += (uint32_t)__popcll(left[j]);
            }
        lds_turn();
        before = 0;
#pragma unroll
        for (uint32_t j = 0; j < kItems; ++j)
            if (j * kWave < l && (j + 1u) * kWave > f) { // uniform
                const uint32_t p = j * kWave + lane, s = before + mask_rank(left[j]);
                const bool is_left = (left[j] >> lane) & 1ull;
                if (is_left && p >= cut)
                    x[j] = tmp_a[smalls - 1u - s];
                if (!is_left && p >= lo && p < cut)
                    x[j] = tmp_b[p - lo - s];
                if (p < l)
                    range[p] = x[j];
                before += (uint32_t)__popcll(left[j]);
            }
        lds_turn();
        if (cut <= nth)
            f = cut;
        else
            l = cut;
    }
    const bool done = l - f <= 3u;
    if (done && l > f) { // __insertion_sort: the entries are distinct
        u64 a = range[f], b = f + 1u < l ? range[f + 1u] : ~0ull, c = f + 2u < l ? range[f + 2u] : ~0ull;
        auto order = [](u64& lo, u64& hi) {
            const u64 t = lo < hi ? lo : hi;
            hi = lo < hi ? hi : lo;
            lo = t;
        };
        order(a, b);
        order(b, c);
        order(a, b);
        lds_turn();
        range[f] = a; // (every lane the same)
        if (f + 1u < l)
            range[f + 1u] = b;
        if (f + 2u < l)
            range[f + 2u] = c;
    }
    return done;
}

// What other workgroups have done of it (nth_steps.h): `used` rounds, which left `len` entries; `ready` as for
// nth_rounds_memory().  picked: the list is what a wide row keeps, and more, none with less bits(q) than `used`.
struct NthDone {
    uint32_t used, len;
    const uint32_t* ready;
    bool picked;
};
constexpr NthDone kNthNothing = {0u, kNone, nullptr, false};
// The row's candidates in device memory (key[i], idx[i]; far: n / 32 words of it that are free), n of them to begin with.  All threads call.
__device__ MAKO_RARE_CALL void nth_element_row(uint32_t* key_p, uint32_t* idx_p, uint32_t n, uint32_t nth, uint32_t* far, const FinishLds& L,
                                               NthDone done = kNthNothing)
{
    assume_lds(L);
    typedef unsigned long long u64;
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x;
    if (n == 0 || nth >= n)
        return;
    uint32_t first = 0, last = min(n, done.len);
    uint32_t depth = 2u * (31u - (uint32_t)__clz((int)n)) - done.used;
    const global_ptr<uint32_t> key = as_global(key_p), idx = as_global(idx_p);
    const lds_ptr<u64> lds = as_lds(L.sortk);
    auto get = [=](uint32_t i) { return ((u64)key[i] << 32) | (u64)idx[i]; };
    auto put = [=](uint32_t i, u64 v) {
        key[i] = (uint32_t)(v >> 32);
        idx[i] = (uint32_t)v;
    };
    __syncthreads();
    MAKO_STAMP(20);
    nth_rounds_memory(key, idx, first, last, nth, depth, kNthUntil, as_global(far), done.ready, lds, sm);
    MAKO_STAMP(21);
    first = uniform_u32(first);
    last = uniform_u32(last);
    if (last - first <= kNthUntil) { // uniform
        const uint32_t origin = first & ~3u, from = first;
        u64 x[kNthChunks][4];
#pragma unroll
        for (uint32_t c = 0; c < kNthChunks; ++c) {
            // (rows' arrays are a multiple of 1 024 long)
            const uint32_t p = min(origin + c * 4u * (uint32_t)kThreads + 4u * tid, (last - 1u) & ~3u);
            const u32x4 k = *(global_ptr<const u32x4>)(key + p), i = *(global_ptr<const u32x4>)(idx + p);
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                x[c][j] = ((u64)k[j] << 32) | (u64)i[j];
        }
        first -= origin;
        last -= origin;
        nth_rounds_registers(x, first, last, nth - origin, depth, kNthWave, lds, sm);
        MAKO_STAMP(22);
        // what is settled goes back, the rest to one wave's list in LDS, or back too if the depth limit has been reached
        const uint32_t len = last - first;
        const bool by_wave = len <= kNthWave; // uniform
        const lds_ptr<u64> range = lds;       // [kNthWave], and twice as much for the wave's own use
        lds_barrier(); // (the exchange buffer has been read)
#pragma unroll
        for (uint32_t c = 0; c < kNthChunks; ++c)
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t p = c * 4u * (uint32_t)kThreads + 4u * tid + j;
                if (p + origin >= from && p < (by_wave ? first : last))
                    put(origin + p, x[c][j]);
                else if (by_wave && p >= first && p < last)
                    range[p - first] = x[c][j];
            }
        lds_barrier();
        bool arranged = false;
        if (by_wave) { // uniform
            if (wave_id() == 0) {
                uint32_t f = 0, l = len, dep = depth;
                const bool ok = nth_rounds_wave(range, len, f, l, nth - origin - first, dep, range + kNthWave);
                if (lane_id() == 0) {
                    sm.bs.u64[0] = ok ? 1u : 0u;
                    sm.bs.u64[1] = ((u64)f << 32) | (u64)l;
                }
            }
            lds_barrier();
            arranged = sm.bs.u64[0] != 0u;
            if (tid < len)
                put(origin + first + tid, range[tid]);
            last = first + (uint32_t)sm.bs.u64[1];
            first += (uint32_t)(sm.bs.u64[1] >> 32);
        }
        first += origin;
        last += origin;
        __syncthreads();
        MAKO_STAMP(23);
        if (arranged)
            return;
    }
    // the depth limit
    heap_select_rest(get, put, first, last, nth, lds, kDynLds / 8u);
}

// key0 / idx0 <- the row's candidates in index order (~bits(q), token id), from its bits(q) array qb[0 .. V) (bits(q)
// of every candidate at its index, 0 elsewhere), as general_row() first leaves them.  All threads call.  (Only for
// the rare second look at a row: one entry per lane and round.)
__device__ MAKO_RARE_CALL void compact_candidates(const uint32_t* qb, uint32_t V, uint32_t* key0, uint32_t* idx0, FinishShared& sm)
{
    const uint32_t lane = lane_id(), wave = wave_id();
    const uint32_t chunk = (V + kWaves - 1u) / kWaves;
    const uint32_t beg = min(V, wave * chunk), end = min(V, beg + chunk);
    uint32_t mine = 0;
    for (uint32_t i = beg + lane; i < end; i += kWave)
        mine += qb[i] ? 1u : 0u;
    mine = __ockl_wfred_add_u32(mine);
    __syncthreads();
    if (lane == 0)
        sm.bs.u64[wave] = mine;
    __syncthreads();
    uint32_t at = 0;
    for (uint32_t w = 0; w < wave; ++w)
        at += (uint32_t)sm.bs.u64[w];
    for (uint32_t base = beg; base < end; base += kWave) {
        const uint32_t i = base + lane;
        const uint32_t k = i < end ? qb[i] : 0u;
        const unsigned long long bal = __ballot(k != 0u);
        if (k) {
            const uint32_t pos = at + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
            key0[pos] = ~k;
            idx0[pos] = i;
        }
        at += (uint32_t)__popcll(bal);
    }
    __syncthreads();
}

// Common tail of the whole-row paths.  key[0]/idx[0] of the row hold n0 candidates (~bits(q), token id) in index
// order.  Sorts them by (q desc, idx asc) when top-k or top-p is active, truncates (src/gen/sampler.cpp:39-61)
// and draws.  `total64` (when have_total) is the fp64 sum of q over all candidates of the row, of which the list
// may be only the heaviest part; otherwise it is summed from the list.  key0 / idx0: the list, key1 / idx1: a second buffer.
// done: what is behind a row's nth_element already (then the list is what the rounds left of it; n0 as it was).
// qk: the row's bits(q) array (bits(q) of every candidate at its index, 0 elsewhere), wanted for a second look at a cut too
// close to call; without one (nullptr) such a row is left undone and false is returned.
// (TOPK_ALONE = false leaves the top-k-without-top-p branch out of the instance inside plan_kernel: that kernel is
// only launched for batches whose host copy of the parameters shows a top-p on every sampled row, and the branch's
// registers would be spilled around the top-k rows' fast path, +3.5 us on a 256-row batch.)
template <bool TOPK_ALONE>
__device__ bool sort_truncate_draw(const mako_sample_desc& d, uint32_t row, const mako_sampling_params& P, uint32_t* key0, uint32_t* idx0,
                                   uint32_t* key1, uint32_t* idx1, const uint32_t* qk, uint32_t n0, bool have_total, double total64,
                                   uint32_t path, const FinishLds& L, NthDone done = kNthNothing)
{
    assume_lds(L);
    FinishShared& sm = *L.sm;

    // order by (q desc, idx asc): stable LSD radix sort of ~bits(q), ascending
    const bool topk_active = P.top_k > 0 && P.top_k < n0;
    const bool topp_active = P.top_p < 1.0f;
    // top-k alone: the survivors stay in the order nth_element leaves them (sampler.cpp:39-43, then :79-83)
    const bool nth_order = TOPK_ALONE && topk_active && !topp_active;
    if (nth_order)
        nth_element_row(key0, idx0, n0, P.top_k, key1, L, done);
    else if (topk_active && done.picked) {
        const uint32_t n = min(done.len, kNthPickedMax);
        if (!sort_picked(key0, idx0, n, done.used, L)) { // (a crowded bucket: what was picked is cut to what is kept first)
            nth_element_row(key0, idx0, n, P.top_k, key1, L);
            sort_survivors(key0, idx0, key1, idx1, P.top_k, L);
        }
    } else if (topk_active) {
        // a top-p follows: the survivors are sorted, so only which candidates they are matters, and `desc` is a total
        // order: nth_element's first top_k entries are the top_k first of the sorted list, in some order.  The
        // partitions and a sort of top_k entries cost a quarter of the sort of all candidates.
        nth_element_row(key0, idx0, n0, P.top_k, key1, L, done);
        sort_survivors(key0, idx0, key1, idx1, P.top_k, L);
    } else if (topp_active)
        sort_segment(key0, idx0, key1, idx1, n0, L);
    const uint32_t *ks = key0, *is = idx0;
    MAKO_STAMP(12);
    const uint32_t n1 = topk_active ? P.top_k : n0; // sampler.cpp:40-43
    // (sorted_tail's one-wave path for lists of up to kGroup entries adds and walks them in the order given, whatever
    // it is, and without a top-p it cuts nothing: nth_element's survivors take it too)
    if (nth_order ? n1 <= kGroup : (topk_active || topp_active)) {
        // (A call: with the tail in line this function and its callers are a call more, each of which stores the registers of sixteen
        // waves: three rows of 2 048 logits, top-k alone, 20 of them allowed, 83 us, 68 so; 251 rows of 1 865 59.9 and 54.4; 85 of
        // 43 705, top_k 200 to 1 000, 63.2 and 61.5.)
        bool drawn;
        MAKO_CALL drawn = sorted_tail(d, row, P, ks, is, n1, have_total, total64, path, L);
        if (drawn)
            return true;
        // Too close to call (top-p rows only): the reference's total decides, summed in the order its candidates have
        // at that point (sampler.cpp:40-48).
        if (!qk)
            return false;
        if (topk_active) {
            // the order nth_element leaves the survivors in: from the candidates in index order again
            compact_candidates(qk, d.n_vocab, key0, idx0, sm);
            nth_element_row(key0, idx0, n0, P.top_k, key1, L);
            total64 = reference_total([=](uint32_t i) { return __uint_as_float(~key0[i]); }, n1, sm);
            sort_survivors(key0, idx0, key1, idx1, n1, L); // (equal weights by token id, as in the list of all candidates)
        } else {
            // index order: the row's bits(q) array (the zeros of the logits that are no candidates add nothing)
            total64 = reference_total([=](uint32_t i) { return __uint_as_float(qk[i]); }, d.n_vocab, sm);
        }
        sorted_tail_exact(d, row, P, ks, is, n1, total64, path, L);
        return true;
    }
    // nth_element's order (long lists), or neither top-k nor top-p: the candidates stay in index order
    // (qk: general_row(), whose long lists gain from addresses in scalar registers; general_row_from_weights(), whose registers
    // those are short of, loses by them: 64 rows, top_k 200 to 1 000, 71.4 us and 72.3)
    auto draw = [&](auto kf, auto jf) {
        draw_from_list(
            d, row, [=](uint32_t i) { return __uint_as_float(~kf[i]); }, [=](uint32_t i) { return jf[i]; }, n1, path, sm);
    };
    if (qk) // uniform
        draw(uniform_ptr(as_global(ks)), uniform_ptr(as_global(is)));
    else
        draw(GlobalKeys{ks}, GlobalKeys{is});
    return true;
}

// Bitonic sort, descending, of 1024 * ITEMS keys held ITEMS per thread: key[t] is element t * 1024 + tid.
// Partners 1024 or more apart are other registers of the same thread, partners less than 64 apart are lanes
// of the same wave (shuffles); only the strides in between go through LDS (two barriers each).
template <int ITEMS>
__device__ void bitonic_sort_regs(unsigned long long (&key)[ITEMS], lds_ptr<unsigned long long> lds)
{
    const uint32_t tid = threadIdx.x;
    for (uint32_t k = 2; k <= 1024u * ITEMS; k <<= 1)
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            if (j >= 1024u) {
                // register-to-register stage; every index below is a compile-time constant so that key[]
                // stays in registers
#pragma unroll
                for (uint32_t dj = 1; dj < (uint32_t)ITEMS; dj <<= 1)
                    if (j == dj * 1024u) {
#pragma unroll
                        for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t)
                            if ((t & dj) == 0) {
                                const bool desc = ((t * 1024u + tid) & k) == 0;
                                const unsigned long long a = key[t], b = key[t | dj];
                                const bool swap = (a < b) == desc;
                                key[t] = swap ? b : a;
                                key[t | dj] = swap ? a : b;
                            }
                    }
            } else if (j >= (uint32_t)kWave) {
#pragma unroll
                for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t)
                    lds[t * 1024u + tid] = key[t];
                __syncthreads();
#pragma unroll
                for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t) {
                    const unsigned long long other = lds[t * 1024u + (tid ^ j)];
                    const bool keep_max = ((tid & j) == 0) == (((t * 1024u + tid) & k) == 0);
                    key[t] = keep_max ? (key[t] > other ? key[t] : other) : (key[t] < other ? key[t] : other);
                }
                __syncthreads();
            } else {
#pragma unroll
                for (uint32_t t = 0; t < (uint32_t)ITEMS; ++t) {
                    const unsigned long long other = __shfl_xor(key[t], (int)j);
                    const bool keep_max = ((tid & j) == 0) == (((t * 1024u + tid) & k) == 0);
                    key[t] = keep_max ? (key[t] > other ? key[t] : other) : (key[t] < other ? key[t] : other);
                }
            }
        }
}

// Sorts n (key, id) pairs in any order at (k0, i0) by key, then id, both ascending; (k1, i1): a second buffer.
// (Up to 4096 of them in registers, by one bitonic sort of both: 1000 pairs took the radix sorts' eight passes through
// device memory 60 us.)
__device__ void sort_survivors(uint32_t* k0, uint32_t* i0, uint32_t* k1, uint32_t* i1, uint32_t n, const FinishLds& L)
{
    assume_lds(L);
    typedef unsigned long long u64;
    const uint32_t tid = threadIdx.x;
    if (n > 4096u) { // (stable sorts: ids first, then the keys)
        sort_segment(i0, k0, i1, k1, n, L);
        sort_segment(k0, i0, k1, i1, n, L);
        return;
    }
    const global_ptr<uint32_t> k = as_global(k0), i = as_global(i0);
    __syncthreads();
    auto sort = [&](auto items) {
        constexpr int kItems = decltype(items)::value;
        u64 key[kItems]; // (complements: the sort is a descending one)
#pragma unroll
        for (uint32_t t = 0; t < (uint32_t)kItems; ++t) {
            const uint32_t e = t * kThreads + tid, at = min(e, n - 1u);
            key[t] = e < n ? ~(((u64)k[at] << 32) | (u64)i[at]) : 0ull;
        }
        bitonic_sort_regs<kItems>(key, as_lds(L.sortk));
#pragma unroll
        for (uint32_t t = 0; t < (uint32_t)kItems; ++t)
            if (t * kThreads + tid < n) {
                k[t * kThreads + tid] = ~(uint32_t)(key[t] >> 32);
                i[t * kThreads + tid] = ~(uint32_t)key[t];
            }
    };
    if (n <= 1024u)
        sort(std::integral_constant<int, 1>());
    else
        sort(std::integral_constant<int, 4>());
    __syncthreads();
}

// The n <= kNthPickedMax entries that nth_pick() has left at (k0, i0), none with less bits(q) than key_lo, by key, then id, both
// ascending.  Returns false, and has moved nothing, where they crowd few of the sort's buckets.
__device__ MAKO_RARE_CALL bool sort_picked(uint32_t* k0, uint32_t* i0, uint32_t n, uint32_t key_lo, const FinishLds& L)
{
    assume_lds(L);
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x;
    const uint32_t key_hi = 0x3f800001u; // (just above 1.0)
    static_assert((kSegCap + 4u) * 8u + (kFine + 4u) * 4u <= kTailLds, "the sort's buckets");
    uint32_t* hist = reinterpret_cast<uint32_t*>(L.sortk + kSegCap + 4u); // (lds_bucket_sort()'s)
    const global_ptr<const uint32_t> k = as_global(k0), i = as_global(i0);
    uint32_t key[kSortPer], id[kSortPer];
    __syncthreads();
#pragma unroll
    for (uint32_t t = 0; t < kSortPer; ++t) {
        const uint32_t e = min(t * kThreads + tid, n - 1u);
        key[t] = min(max(~k[e], key_lo), key_hi - 1u);
        id[t] = i[e];
    }
    for (uint32_t b = tid; b <= kFine; b += kThreads)
        hist[b] = 0;
    if (tid == 0)
        sm.flag = 0;
    __syncthreads(); // (everything has been read)
    const bool sorted = lds_bucket_sort(key, id, n, key_lo, key_hi, k0, i0, L.sortk, sm);
    __syncthreads();
    return sorted;
}

// The row's logits, -inf where the mask says so, to wbuf.  All threads call.
// (Sixteen logits a thread and trip, all asked for before anything is waited for: they may be in host memory, a trip over the bus
// away.  One row of 129 280 equal logits through the host call: 339 us with one logit a thread and trip from device memory, 433
// from host memory, 333 from there so; 64 such rows 360 us, 339 so.)
__device__ MAKO_RARE_CALL void copy_masked_row(const mako_sample_desc& d, uint32_t row, const mako_sampling_params& P, float* wbuf)
{
    const uint32_t tid = threadIdx.x;
    for (uint32_t lo = 0; lo < d.n_vocab; lo += kSliceMax) {
        const uint32_t hi = min(d.n_vocab, lo + kSliceMax);
        RawSlice raw;
        load_raw<false>(d, row, lo, hi, raw);
        settle_slice<false>(raw, lo, hi);
        float w[16];
        finish_slice<false>(raw, lo, hi, P, false, nullptr, w, d.mask != nullptr);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t i = elem_index(lo, tid, 4u * k);
            if (i + 3u < hi) {
                *reinterpret_cast<float4*>(wbuf + i) = make_float4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
            } else {
#pragma unroll
                for (uint32_t c = 0; c < 4; ++c)
                    if (i + c < hi)
                        wbuf[i + c] = w[4 * k + c];
            }
        }
    }
}

// Whole-row path: exact for every parameter combination.  One workgroup rebuilds the penalised
// row in scratch, keeps the candidates, sorts them by (q desc, idx asc) when top-k or top-p is
// active, truncates, and draws.  src/gen/sampler.cpp:20-62.
// (SITE: sort_kernel, its usual place, has an instance to itself, so that the compiler treats that kernel the same
// whether or not the instances inside plan_kernel exist.)
template <int SITE>
__device__ MAKO_RARE_CALL void general_row(const mako_sample_desc& d, const Scratch& sc, uint32_t row, const mako_sampling_params& P,
                            float m, uint32_t argidx, const FinishLds& L)
{
    assume_lds(L);
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x;
    const uint32_t V = d.n_vocab;
    float* wbuf = sc.wbuf + (size_t)row * sc.vpad;
    uint32_t* cnt = sc.cnt + (size_t)row * sc.vpad;
    uint32_t* key0 = sc.key[0] + (size_t)row * sc.vpad;
    uint32_t* idx0 = sc.idx[0] + (size_t)row * sc.vpad;

    // 1. masked copy, then the penalties once per distinct history token
    copy_masked_row(d, row, P, wbuf);
    __syncthreads();
    const uint32_t hl = d.hist_tokens ? d.hist_len[row] : 0u;
    if (hl > 0 && !penalties_neutral(P)) {
        const int32_t* ht = d.hist_tokens + (int64_t)row * d.hist_stride;
        const uint32_t* hc = d.hist_counts ? d.hist_counts + (int64_t)row * d.hist_stride : nullptr;
        for (uint32_t h = tid; h < hl; h += kThreads) {
            const uint32_t t = (uint32_t)ht[h];
            if (t < V)
                atomicAdd(&cnt[t], hc ? hc[h] : 1u);
        }
        __syncthreads();
        for (uint32_t h = tid; h < hl; h += kThreads) {
            const uint32_t t = (uint32_t)ht[h];
            if (t < V) {
                const uint32_t c = atomicExch(&cnt[t], 0u); // claims the token and restores the zero
                if (c)
                    wbuf[t] = penalize(wbuf[t], c, P.repetition_penalty, P.presence_penalty, P.frequency_penalty);
            }
        }
        __syncthreads();
    }

    // 2. weights and the min_p / q > 0 filter, compacted in index order (sampler.cpp:29-36).  Wave w owns the w-th
    // sixteenth of the row (a multiple of 256 logits, lane l entries 4l..4l+3 of each 256): a sweep that leaves bits(q)
    // of every candidate (0 otherwise) in place of the logit and counts them, one exchange of the waves' totals, and
    // a sweep in which every lane reads back what it wrote and a wave scan ranks it.  No barrier inside the sweeps.
    const float inv_t = 1.0f / P.temperature;
    const float floor_q = (1.0f < P.min_p) ? 1.0f : P.min_p; // std::min(min_p, 1.0f)
    uint32_t* qb = reinterpret_cast<uint32_t*>(wbuf);
    // (The arrays by typed addresses in scalar registers, for the draw too: in vector registers they are spilled, and fetched from
    // scratch memory again for every 256 logits.  Rows in token order with gaps whose candidates are written out: three of 136 640
    // logits 500 us, 430 so; 39 of 34 688 325 and 282.  One row of 300 000 1 016 and 925.)
    const global_ptr<float> wg = uniform_ptr(as_global(wbuf));
    const global_ptr<uint32_t> qg = (global_ptr<uint32_t>)wg, kg = uniform_ptr(as_global(key0)), ig = uniform_ptr(as_global(idx0));
    const uint32_t lane = lane_id(), wave = wave_id();
    const uint32_t chunk = ((V + kThreads * 4u - 1u) / (kThreads * 4u)) * kGroup;
    const uint32_t beg = min(V, wave * chunk), end = min(V, beg + chunk);
    uint32_t mine = 0;
    for (uint32_t base = beg; base < end; base += kGroup) {
        const uint32_t i = base + lane * 4u;
        float w[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        const bool whole = i + 3u < end;
        if (whole) {
            const f32x4 x = *(global_ptr<const f32x4>)(wg + i);
            w[0] = x.x, w[1] = x.y, w[2] = x.z, w[3] = x.w;
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if (i + j < end)
                    w[j] = wg[i + j];
        }
        uint32_t k[4];
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const float q = weight_of(w[j], m, inv_t, sm.tab);
            k[j] = (i + j < end && q >= floor_q && q > 0.0f) ? __float_as_uint(q) : 0u;
            mine += k[j] ? 1u : 0u;
        }
        if (whole) {
            *(global_ptr<u32x4>)(qg + i) = u32x4{k[0], k[1], k[2], k[3]};
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if (i + j < end)
                    qg[i + j] = k[j];
        }
    }
    mine = __ockl_wfred_add_u32(mine);
    if (lane == 0)
        sm.bs.u64[wave] = mine;
    __syncthreads();
    uint32_t n0 = 0, at = 0;
    for (int w = 0; w < kWaves; ++w) {
        const uint32_t x = (uint32_t)sm.bs.u64[w];
        if (w < (int)wave)
            at += x;
        n0 += x;
    }
    for (uint32_t base = beg; base < end; base += kGroup) {
        const uint32_t i = base + lane * 4u;
        uint32_t k[4] = {0u, 0u, 0u, 0u};
        if (i + 3u < end) {
            const u32x4 x = *(global_ptr<const u32x4>)(qg + i);
            k[0] = x.x, k[1] = x.y, k[2] = x.z, k[3] = x.w;
        } else {
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                if (i + j < end)
                    k[j] = qg[i + j];
        }
        const uint32_t c = (k[0] ? 1u : 0u) + (k[1] ? 1u : 0u) + (k[2] ? 1u : 0u) + (k[3] ? 1u : 0u);
        const uint32_t incl = __ockl_wfscan_add_u32(c, true);
        uint32_t pos = at + incl - c;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
            if (k[j]) {
                MAKO_CHECK(sc, kCheckCompact, pos < n0 && (uint64_t)pos < sc.vpad);
                kg[pos] = ~k[j];
                ig[pos] = i + j;
                ++pos;
            }
        at += (uint32_t)__builtin_amdgcn_readlane((int)incl, kWave - 1);
    }
    __syncthreads();

    if (n0 == 0) {
        fallback_row(d, row, argidx);
        return;
    }
    sort_truncate_draw<SITE == 0>(d, row, P, key0, idx0, sc.key[1] + (size_t)row * sc.vpad, sc.idx[1] + (size_t)row * sc.vpad, qb, n0, false,
                                  0.0, MAKO_PATH_GENERAL, L);
}

// The whole-row path for a row whose weights are already in place: key[0] of the row holds ~bits(q) of every candidate at
// its index and ~0 elsewhere (index_weights_kernel, with a workgroup per 16 384 logits instead of one for the row).  Counts
// and compacts the candidates in index order into the row's second buffers and goes on like general_row().  All threads
// call; m, argidx: the row's maximum and where it is first; n_all: its candidates.
// When that kernel found every logit a candidate (no mask, no floor, no underflow: the usual row) it has left the token ids as
// well, i at i in idx[0] of the row: the list is there, nothing to compact.  Rows long enough for nth_steps.h have their list
// where the last step has left it.
// Returns false where a cut is too close to call: general_row() has to look at the row again, from the logits on.
template <int SITE>
__device__ MAKO_RARE_CALL bool general_row_from_weights(const mako_sample_desc& d, const Scratch& sc, uint32_t row,
                                                        const mako_sampling_params& P, float m, uint32_t argidx, uint32_t n_all,
                                                        const FinishLds& L)
{
    assume_lds(L);
    FinishShared& sm = *L.sm;
    const uint32_t V = d.n_vocab;
    uint32_t* k_from = sc.key[0] + (size_t)row * sc.vpad;
    uint32_t* i_from = sc.idx[0] + (size_t)row * sc.vpad;
    uint32_t* k_to = sc.key[1] + (size_t)row * sc.vpad;
    uint32_t* i_to = sc.idx[1] + (size_t)row * sc.vpad;
    uint32_t n0 = n_all;
    bool listed = n_all == V; // in the first buffers
    NthDone done = kNthNothing;
    if (!nth_steps_for(V) && wide_row(P) && nth_picks_for(V)) { // uniform
        uint32_t from = 0;
        const uint32_t picked = nth_pick(d, sc, row, 0u, 1u, n0, P.top_k, from, L.sortk, sm.bs);
        if (picked != kNone)
            done = NthDone{from, picked, nullptr, true};
        __syncthreads();
    }
    if (done.picked) {
        listed = false; // (in the second buffers)
    } else if (nth_steps_for(V)) { // uniform
        const NthState s0 = *nth_state(sc.plan + row, 0u), s1 = *nth_state(sc.plan + row, 1u);
        const bool odd = (sc.plan[row].cap[kNthMade] & 1u) != 0u;
        const uint32_t buf = odd ? s1.buf : s0.buf;
        const uint32_t pre = odd ? s1.pre : s0.pre;
        done = NthDone{odd ? s1.used : s0.used, odd ? s1.len : s0.len, pre == kNthBits ? nth_bits(sc, row, buf) : nullptr, pre == kNthPicked};
        listed = buf == 0u;
    } else if (!listed) {
        const global_ptr<const uint32_t> from = as_global(k_from);
        const global_ptr<uint32_t> kd = as_global(k_to), id = as_global(i_to);
        const uint32_t lane = lane_id(), wave = wave_id();
        // (wave w owns the w-th sixteenth of the row, a multiple of 256 logits; of each 256, lane l takes l, l + 64, ...;
        // eight such blocks' loads are in flight per trip, from clamped addresses and masked afterwards: one round trip to
        // memory per 2 048 entries of the wave instead of one per 256)
        const uint32_t chunk = ((V + kThreads * 4u - 1u) / (kThreads * 4u)) * kGroup;
        const uint32_t beg = uniform_u32(min(V, wave * chunk)), end = uniform_u32(min(V, beg + chunk));
        constexpr uint32_t kTrip = 8;
        auto load_trip = [&](uint32_t base, uint32_t (&k)[kTrip][4]) {
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u)
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    k[u][j] = from[min(base + u * kGroup + j * (uint32_t)kWave + lane, V - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u)
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    k[u][j] = base + u * kGroup + j * (uint32_t)kWave + lane < end ? k[u][j] : ~0u;
        };
        uint32_t mine = 0;
        for (uint32_t base = beg; base < end; base += kGroup * kTrip) {
            uint32_t k[kTrip][4];
            load_trip(base, k);
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u)
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    mine += (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(k[u][j] != ~0u));
        }
        __syncthreads();
        if (lane == 0)
            sm.bs.u64[wave] = mine;
        __syncthreads();
        uint32_t at = 0;
        n0 = 0;
        for (int w = 0; w < kWaves; ++w) {
            const uint32_t x = (uint32_t)sm.bs.u64[w];
            if (w < (int)wave)
                at += x;
            n0 += x;
        }
        at = uniform_u32(at);
        n0 = uniform_u32(n0);
        for (uint32_t base = beg; base < end; base += kGroup * kTrip) {
            uint32_t k[kTrip][4];
            load_trip(base, k);
#pragma unroll
            for (uint32_t u = 0; u < kTrip; ++u)
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    const unsigned long long is = __builtin_amdgcn_ballot_w64(k[u][j] != ~0u);
                    if (k[u][j] != ~0u) {
                        const uint32_t pos = at + mask_rank(is);
                        MAKO_CHECK(sc, kCheckCompact, pos < n0 && (uint64_t)pos < sc.vpad);
                        kd[pos] = k[u][j];
                        id[pos] = base + u * kGroup + j * (uint32_t)kWave + lane;
                    }
                    at += (uint32_t)__popcll(is);
                }
        }
        __syncthreads();
    }
    if (n0 == 0) {
        fallback_row(d, row, argidx);
        return true;
    }
    return sort_truncate_draw<SITE == 0>(d, row, P, listed ? k_from : k_to, listed ? i_from : i_to, listed ? k_to : k_from, listed ? i_to : i_from,
                                       nullptr, n0, false, 0.0, MAKO_PATH_GENERAL, L, done);
}

} // namespace mako
