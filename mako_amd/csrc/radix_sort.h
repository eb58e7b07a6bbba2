// Stable radix sorts of pairs in device memory, by one workgroup.
#pragma once

#include "workgroup_state.h"

namespace mako {

// Lanes of this wave whose `digit` equals mine, restricted to `valid` lanes.
__device__ __forceinline__ unsigned long long match_digit(uint32_t digit, bool valid)
{
    unsigned long long m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const bool bit = (digit >> b) & 1u;
        const unsigned long long bal = __ballot(bit);
        m &= bit ? bal : ~bal;
    }
    return m;
}

// One stable counting-sort pass on bits [shift, shift + 8) of the keys, ascending, by one workgroup.
// Wave w owns the contiguous chunk [w * C, (w + 1) * C) of the input and walks it 64 pairs at a time: lanes
// with equal digits find each other with ballots (match_digit), so ranks inside a group need no atomics, and
// the wave's running output offsets per digit live in its private row of LDS.  Three barriers per pass.
// Returns false (and moves nothing) when every key has the same digit.
__device__ bool radix_pass(const uint32_t* ksrc, const uint32_t* isrc, uint32_t* kdst, uint32_t* idst, uint32_t n,
                           uint32_t shift, const FinishLds& L)
{
    assume_lds(L);
    FinishShared& sm = *L.sm;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    const uint32_t chunk = ((n + kThreads - 1u) / kThreads) * kWave; // per wave, a multiple of 64
    const uint32_t beg = min(n, wave * chunk), end = min(n, beg + chunk);
    uint32_t* woff = L.wcount + wave * 256u;
    for (uint32_t j = lane; j < 256u; j += kWave)
        woff[j] = 0;
    if (tid == 0)
        sm.flag = 0;
    const unsigned long long lower = (1ull << lane) - 1ull;
    // per-wave digit counts (the row is private to the wave: in-order LDS, no barrier needed).  Four groups
    // are fetched per trip, from clamped positions, so that their latencies overlap.
    for (uint32_t base = beg; base < end; base += 4u * kWave) {
        uint32_t key[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u)
            key[u] = ksrc[min(base + u * kWave + lane, end - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const bool valid = base + u * kWave + lane < end;
            const uint32_t dg = valid ? ((key[u] >> shift) & 255u) : 0u;
            const unsigned long long mm = match_digit(dg, valid);
            if (valid && (mm & lower) == 0)
                woff[dg] += (uint32_t)__popcll(mm);
        }
    }
    __syncthreads();
    // digit totals -> global offsets; wave rows become each wave's first output position per digit
    uint32_t mine = 0;
    if (tid < 256)
        for (int w = 0; w < kWaves; ++w)
            mine += L.wcount[w * 256 + tid];
    if (tid < 256 && mine == n)
        sm.flag = 1;
    uint32_t tot;
    uint32_t acc = block_excl_scan_u32(mine, tot, sm.bs); // its barriers publish sm.flag
    if (sm.flag)
        return false;
    if (tid < 256)
        for (int w = 0; w < kWaves; ++w) {
            const uint32_t t = L.wcount[w * 256 + tid];
            L.wcount[w * 256 + tid] = acc;
            acc += t;
        }
    __syncthreads();
    for (uint32_t base = beg; base < end; base += 4u * kWave) {
        uint32_t key[4], id[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t i = min(base + u * kWave + lane, end - 1u);
            key[u] = ksrc[i];
            id[u] = isrc[i];
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const bool valid = base + u * kWave + lane < end;
            const uint32_t dg = valid ? ((key[u] >> shift) & 255u) : 0u;
            const unsigned long long mm = match_digit(dg, valid);
            const uint32_t off = woff[dg];
            if (valid) {
                const uint32_t pos = off + (uint32_t)__popcll(mm & lower);
                kdst[pos] = key[u];
                idst[pos] = id[u];
                if ((mm & lower) == 0)
                    woff[dg] = off + (uint32_t)__popcll(mm);
            }
        }
    }
    __syncthreads();
    return true;
}

// Sorts n (key, id) pairs at (k0, i0) by key ascending, stably, with (k1, i1) as the second buffer; the result
// ends in (k0, i0).
__device__ void sort_segment(uint32_t* k0, uint32_t* i0, uint32_t* k1, uint32_t* i1, uint32_t n, const FinishLds& L)
{
    assume_lds(L);
    if (n < 2)
        return;
    uint32_t *ks = k0, *is = i0, *kd = k1, *id = i1;
    for (uint32_t shift = 0; shift < 32; shift += 8) {
        if (radix_pass(ks, is, kd, id, n, shift, L)) {
            uint32_t* t = ks;
            ks = kd;
            kd = t;
            t = is;
            is = id;
            id = t;
        }
        __syncthreads();
    }
    if (ks != k0) {
        for (uint32_t i = threadIdx.x; i < n; i += kThreads) {
            k0[i] = ks[i];
            i0[i] = is[i];
        }
        __syncthreads();
    }
}

} // namespace mako
