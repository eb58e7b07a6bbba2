// The first rounds of the whole-row class's nth_element (whole_row.h), with several workgroups per row.
//
// libstdc++'s introselect halves its range round by round, and one workgroup is bound by what its CU can read and move: a row
// of 129 280 candidates kept it 88 us before what is left fits its registers (186 for the row with the unluckiest pivots of
// 64), while three quarters of the chip had nothing to do.  A round needs its pivot, the number of entries that belong left of
// it, and for every entry that moves its place, all of which follow from one bit per entry ("belongs left").  So a launch in
// which several workgroups share a row (a "step") makes a round out of the bits that the launch before left, and leaves the
// next round's:
//   index_weights_kernel   weights a workgroup per 16 384 logits; a row whose every logit is a candidate is its own list, so
//                          the first pivot is the median of three logits known beforehand: leaves the first round's bits
//                          (and the bits of who is a candidate);
//   step 1                 such a row: the first round.  Any other: the candidates moved together.
//   step 2, 3, ...         a round each, until what is left fits a workgroup's registers (kNthUntil), where the row's one
//                          workgroup goes on in the last launch.
// A top-k before a top-p (wide_row()) needs no rounds: its survivors end up sorted, so only which candidates they are matters.
// index_weights_kernel counts the weights by value, and step 1 picks those from the bin that holds the k-th on, which the last
// launch sorts.  (64 rows of 129 280, top_k 200 to 1 000: 183 us with the rounds, 75 so.)  Where the bin is too crowded, as on a
// grid of few weights, the rounds are made.
// Beside rows of other kinds, where a launch that no row needs would be paid for all the same, the sort's launch makes all steps:
// a row's workgroups, as many as there are CUs for, meet after each (nth_steps_at_once()).  (Of 24 rows of 151 553 of all
// kinds 205 us with the first step alone there, 140 so; top-k alone, 8 rows of 129 280: 157 and 121, 100 rows: 294 and 276.  A
// batch of such rows alone keeps its launches: two workgroups share a CU there, and 64 rows take 162 us instead of 172.)
// A step writes the list it makes beside the old one, with the next round's pivot already swapped to the front; its workgroups
// take 4 096 entries of the new list at a time.  An entry that belongs left and lies in front of the cut stays where it is; a
// hole's filler comes through LDS: the holes of 4 096 places in a row are filled from one stretch of the old list, from its
// end backwards.
#pragma once

#include "sampler_common.h"
#include "workgroup_state.h"

namespace mako {

constexpr uint32_t kNthUntil = 16380;       // entries that a workgroup takes into registers wherever they begin
constexpr uint32_t kNthChunk = 4096;        // of the new list, per workgroup and turn: four per thread
constexpr uint32_t kNthMaxVocab = kMaxGroups * kGroup;
constexpr uint32_t kNthWords = kNthMaxVocab / 64u; // of a row's bits
constexpr uint32_t kNthLds = kNthChunk * 8u + kNthWords * 12u + 64u;

// Where a row stands: two records in turn in the row's plan (a step reads one and writes the other), in the words its workers
// would use.  len entries of key[buf] / idx[buf] are what is left of the list, `used` rounds
// behind them.  pre: kNthBits: the next round's pivot is at the front and its bits are in place; kNthPicked: the list is what a
// wide row keeps, and more, in any order, and `used` the least bits(q) it may hold.
struct alignas(4) NthState {
    uint32_t len, pre, used, buf;
};
constexpr uint32_t kNthBits = 1, kNthPicked = 2;
// (words of the plan's `cap`: what step 1 has picked; the row's workgroups that have made a step, all steps together (nth_meet());
// the steps that all of them have made)
constexpr uint32_t kNthCursor = 16, kNthMet = 17, kNthMade = 18;
static_assert(2u * sizeof(NthState) <= kNthCursor * 4u && sizeof(BigPlan::cap) > kNthMade * 4u, "");
// The first pivot of a row that is its own list, where it came from, and the key of its first entry.
struct NthFirst {
    uint32_t pivot_key, pivot_id, from, first_key;
};
__device__ __forceinline__ NthState* nth_state(BigPlan* plan, uint32_t slot)
{
    return reinterpret_cast<NthState*>(plan->cap) + slot;
}
__device__ __forceinline__ NthFirst* nth_first(BigPlan* plan)
{
    return reinterpret_cast<NthFirst*>(plan->stage_off);
}
// A row's bits, entry i at bit i & 31 of word i >> 5, in the memory of its penalised logits: of the list in key[buf], and of
// the row's candidates (buf = 2).  (Written in blocks of 256 entries.)
__device__ __forceinline__ uint32_t* nth_bits(const Scratch& sc, uint32_t row, uint32_t buf)
{
    return reinterpret_cast<uint32_t*>(sc.wbuf + (size_t)row * sc.vpad) + buf * (uint32_t)(sc.vpad / 32u + 256u);
}
// Is the row one of these?  (The others of its class stay in token order: index_rows.h.)
__host__ __device__ __forceinline__ bool nth_row(const mako_sampling_params& P)
{
    return classify(P) == kGeneral && P.top_k != 0u;
}
// Are there steps for rows of this many logits?  (Below, a round in device memory takes a workgroup 12 us at most, and a step's
// launch 8, and all of its rows may be masked down to a few candidates: 64 rows of 19 392, half of them masked, 82 us without
// steps, 91 with two.)
__host__ __device__ __forceinline__ bool nth_steps_for(uint32_t n_vocab)
{
    return n_vocab > 32768u && n_vocab <= kNthMaxVocab;
}

// How many launches of their own, of rows the least of whose top_k is this?  Each costs 8 to 10 us and leaves 0.44 of the list: as
// many as bring the 64 rows' unluckiest near what a workgroup takes into its registers (64 rows of 129 280, top_k 40: 185 us with
// two, 172, 164, 162, 168 with six; of 40 000: 104 with two, 105, 110), but none for a list that is expected to be less than twice
// top_k long, since a row is done with steps once its cut lies in front of its top_k.  (64 rows of 129 280, one to four launches:
// top_k 1 293 260 us, 239, 230, 234; 6 464 315, 318, 330, 341; 25 856 468, 484, 496, 507; 64 640 637, 653, 659, 664; 129 280 580,
// 582, 585, 589; one row, top_k 6 464: 188, 184, 184, 186.)
inline uint32_t nth_launches(uint32_t n_vocab, uint32_t least_top_k)
{
    const uint32_t most = n_vocab <= 65536u ? 2u : 4u;
    uint32_t n = 1;
    for (float left = 0.44f * (float)n_vocab; n < most && left > 2.0f * (float)least_top_k; left *= 0.44f)
        ++n;
    return n;
}

// ... and of those, a top-k before a top-p?
__host__ __device__ __forceinline__ bool wide_row(const mako_sampling_params& P)
{
    return nth_row(P) && P.top_p < 1.0f;
}
// Are a wide row's picked, of so many logits?  Where there are steps, by the first of them, else by the row's one workgroup in the
// last launch.  (16 000 of them: 89 us with the rounds in that workgroup's registers, 45 so; 48 with a step.)
__host__ __device__ __forceinline__ bool nth_picks_for(uint32_t n_vocab)
{
    return n_vocab > 2048u && n_vocab <= kNthMaxVocab;
}
// A wide row's weights counted by value, a table per 16 384 logits, behind the bits: 64 bins a binade for the four heaviest
// binades, where a flat row has all of its weights, four a binade below.
constexpr uint32_t kNthBins = 768, kNthFine = 256;
constexpr uint32_t kNthPickedMax = kSegCap; // entries that step 1 may pick: what one sort in LDS holds
static_assert(kNthPickedMax * 8u + 64u <= kNthLds, "");
__device__ __forceinline__ uint32_t nth_bin(uint32_t q_bits) // (heaviest first)
{
    static_assert(kNthFine + ((0x3f800000u - (kNthFine << 17)) >> 21) < kNthBins, "weights are at most 1");
    const uint32_t d = 0x3f800000u - q_bits;
    return d < kNthFine << 17 ? d >> 17 : kNthFine + ((d - (kNthFine << 17)) >> 21);
}
__device__ __forceinline__ uint32_t nth_bin_edge(uint32_t bin) // the bits of the lightest weight in it
{
    const uint32_t d = (bin < kNthFine ? (bin + 1u) << 17 : (kNthFine << 17) + ((bin + 1u - kNthFine) << 21)) - 1u;
    return d < 0x3f800000u ? 0x3f800000u - d : 1u;
}
__device__ __forceinline__ uint32_t* nth_hist(const Scratch& sc, uint32_t row, uint32_t piece)
{
    static_assert(3u * (kNthUntil / 32u + 256u) + kNthMaxVocab / kSliceMax * kNthBins <= kNthUntil, "a row's bits and tables in the place of its logits");
    return nth_bits(sc, row, 3u) + piece * kNthBins;
}

__device__ __forceinline__ uint32_t mask_rank(unsigned long long m)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// The median of three and its position (__move_median_to_first(first, first + 1, mid, last - 1)).
template <typename T>
__device__ __forceinline__ void median_of_three(T vx, T vy, T vz, uint32_t ix, uint32_t iy, uint32_t iz, T& med, uint32_t& im)
{
    const bool xy = vx < vy, yz = vy < vz, xz = vx < vz;
    im = xy == yz ? iy : (xy == xz ? iz : ix);
    med = xy == yz ? vy : (xy == xz ? vz : vx);
}

// Four bits per lane (of entries 4 l .. 4 l + 3) as words of 32: the first lane of every eight holds theirs.
__device__ __forceinline__ uint32_t eight_nibbles(uint32_t nibble)
{
    uint32_t v = nibble << (4u * ((uint32_t)lane_id() & 7u));
    v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, false);  // quad_perm: lane ^ 1
    v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, false);  // quad_perm: lane ^ 2
    v |= (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, false); // row_half_mirror: the other four
    return v;
}

// What a wide row keeps, by workgroup w of W (step 1): the entries from the bin that holds the nth-heaviest on, in any
// order, to key[1] / idx[1].  Returns how many that is in all, kNone if it is too many (or nothing is cut off): then nothing has been written.  All threads call.
__device__ __forceinline__ uint32_t nth_pick(const mako_sample_desc& d, const Scratch& sc, uint32_t row, uint32_t w, uint32_t W, uint32_t n0, uint32_t nth,
                                             uint32_t& from, unsigned long long* lds_dyn, BlockScratch& bs)
{
    typedef unsigned long long u64;
    const uint32_t tid = threadIdx.x;
    if (nth >= n0) // uniform
        return kNone;
    const lds_ptr<u64> kept = as_lds(lds_dyn);                                        // [kNthPickedMax]
    const lds_ptr<uint32_t> found = (lds_ptr<uint32_t>)(kept + kNthPickedMax);        // the bin, the entries from it on, this workgroup's, their place
    // (thread t: bin t)
    const uint32_t pieces = (d.n_vocab + kSliceMax - 1u) / kSliceMax;
    uint32_t c = 0;
    if (tid < kNthBins)
        for (uint32_t p = 0; p < pieces; ++p)
            c += as_global(nth_hist(sc, row, p))[tid];
    uint32_t all;
    const uint32_t above = block_excl_scan_u32(c, all, bs);
    if (above < nth && above + c >= nth) {
        found[0] = tid;
        found[1] = above + c;
        found[2] = 0u;
    }
    __syncthreads();
    from = nth_bin_edge(uniform_u32(found[0]));
    const uint32_t n = uniform_u32(found[1]);
    if (n > kNthPickedMax) // uniform
        return kNone;
    const global_ptr<const uint32_t> key = as_global(sc.key[0]) + (size_t)row * sc.vpad;
    constexpr uint32_t kTrip = 4;
    for (uint32_t c0 = w; c0 * kNthChunk < d.n_vocab; c0 += W * kTrip) { // uniform
        u32x4 k[kTrip];
#pragma unroll
        for (uint32_t u = 0; u < kTrip; ++u) // (rows' arrays are a multiple of 1 024 long)
            k[u] = *(global_ptr<const u32x4>)(key + min((c0 + u * W) * kNthChunk + 4u * tid, (d.n_vocab - 1u) & ~3u));
#pragma unroll
        for (uint32_t u = 0; u < kTrip; ++u)
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t i = (c0 + u * W) * kNthChunk + 4u * tid + j;
                if (i < d.n_vocab && ~k[u][j] >= from && k[u][j] != ~0u) { // (few)
                    const uint32_t at = __hip_atomic_fetch_add(found + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    if (at < kNthPickedMax)
                        kept[at] = ((u64)k[u][j] << 32) | (u64)i;
                }
            }
    }
    __syncthreads();
    const uint32_t mine = min(uniform_u32(found[2]), kNthPickedMax);
    if (tid == 0)
        found[3] = mine ? __hip_atomic_fetch_add(as_global(&sc.plan[row].cap[kNthCursor]), mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
    __syncthreads();
    const uint32_t base = uniform_u32(found[3]);
    const global_ptr<uint32_t> kout = as_global(sc.key[1]) + (size_t)row * sc.vpad, iout = as_global(sc.idx[1]) + (size_t)row * sc.vpad;
    for (uint32_t e = tid; e < mine && base + e < kNthPickedMax; e += (uint32_t)kThreads) {
        MAKO_CHECK(sc, kCheckCompact, base + e < n);
        kout[base + e] = (uint32_t)(kept[e] >> 32);
        iout[base + e] = (uint32_t)kept[e];
    }
    return n;
}

// One step of row `row`, by workgroup w of W.  lds: kNthLds bytes, or what the row's bits, and the first step's picks, take of it.  All threads call.
// Returns (the same to all of the row's workgroups) kNthNone if the row is none of these, kNthLast, or kNthMore if there is a next step.
enum NthMadeOf : uint32_t { kNthNone, kNthLast, kNthMore };
__device__ __forceinline__ NthMadeOf nth_step(const mako_sample_desc& d, const Scratch& sc, uint32_t row, uint32_t w, uint32_t W, uint32_t step,
                                         unsigned long long* lds_dyn, BlockScratch& bs)
{
    typedef unsigned long long u64;
    const uint32_t tid = threadIdx.x, lane = lane_id(), wave = wave_id();
    BigPlan* plan = sc.plan + row;
    const uint32_t pieces = (d.n_vocab + kSliceMax - 1u) / kSliceMax;
    // (one trip to memory)
    const uint32_t flag = plan->flag, counted = plan->cursor[min(lane, kWorkers - 1u)];
    const mako_sampling_params P = d.params[row];
    NthState now = *nth_state(plan, (step - 1u) & 1u);
    const NthFirst first = *nth_first(plan);
    static_assert(kNthWords <= 4u * (uint32_t)kThreads, "four words of bits a thread");
    const uint32_t usual = (step - 1u) & 1u, words_max = (d.n_vocab + 63u) / 64u; // (where the bits of a row that goes on are)
    u64 x[4];
    auto load_bits = [&](uint32_t buf, uint32_t words) {
        const global_ptr<const u64> from = (global_ptr<const u64>)as_global(nth_bits(sc, row, buf));
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            x[i] = from[min(4u * tid + i, words - 1u)];
    };
    load_bits(usual, words_max);
    const uint32_t nth = P.top_k;
    if (!nth_row(P) || flag != kIndexClaimed) // uniform (a row of another kind; one whose token is forced)
        return kNthNone;
    auto leave = [&](uint32_t n, uint32_t pre, uint32_t rounds, uint32_t in) {
        if (w == 0u && tid == 0u) {
            NthState* s = nth_state(plan, step & 1u);
            s->len = n;
            s->pre = pre;
            s->used = rounds;
            s->buf = in;
        }
    };
    bool compact = false;
    if (step == 1u) {
        const uint32_t n0 = uniform_u32(__ockl_wfred_add_u32(lane < pieces ? counted : 0u));
        compact = n0 != d.n_vocab;
        // (a whole list that nothing is cut off stays as it is)
        now = NthState{d.n_vocab, compact || nth < n0 ? kNthBits : 0u, 0u, 0u};
        if (wide_row(P)) { // uniform
            uint32_t from = 0;
            const uint32_t picked = nth_pick(d, sc, row, w, W, n0, nth, from, lds_dyn, bs);
            if (picked != kNone) {
                leave(picked, kNthPicked, from, 1u);
                return kNthLast;
            }
            __syncthreads();
        }
    }
    const uint32_t len = uniform_u32(now.len), from_buf = uniform_u32(now.buf), used = now.used;
    const lds_ptr<u64> buf = as_lds(lds_dyn);                // [kNthChunk] fillers
    const lds_ptr<u64> bits = buf + kNthChunk;               // [words]
    const uint32_t words = (len + 63u) / 64u;
    const lds_ptr<uint32_t> pre = (lds_ptr<uint32_t>)(bits + words); // [words + 1] set bits in front of each
    const uint32_t to_buf = from_buf ^ 1u;
    const global_ptr<const uint32_t> kin = as_global(sc.key[from_buf]) + (size_t)row * sc.vpad, iin = as_global(sc.idx[from_buf]) + (size_t)row * sc.vpad;
    const global_ptr<uint32_t> kout = as_global(sc.key[to_buf]) + (size_t)row * sc.vpad, iout = as_global(sc.idx[to_buf]) + (size_t)row * sc.vpad;
    bool go = uniform_u32(now.pre) == kNthBits;
    uint32_t smalls = 0;
    if (go) { // uniform
        if (compact || from_buf != usual) // uniform
            load_bits(compact ? 2u : from_buf, words);
        uint32_t mine = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            mine += 4u * tid + i < words ? (uint32_t)__popcll(x[i]) : 0u;
        uint32_t at = block_excl_scan_u32(mine, smalls, bs);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i)
            if (4u * tid + i < words) {
                bits[4u * tid + i] = x[i];
                pre[4u * tid + i] = at;
                at += (uint32_t)__popcll(x[i]);
            }
        smalls = uniform_u32(smalls);
        if (tid == 0)
            pre[words] = smalls;
        __syncthreads();
    }
    const uint32_t out_len = compact ? smalls : smalls + 1u; // (the cut: behind the pivot and what belongs left)
    if (go && !compact && out_len <= nth)                    // uniform: the rounds go on in the right part, by one workgroup
        go = false;
    if (!go) { // uniform
        if (step == 1u) {
            // (a list that stays where it is has no token ids yet)
            const global_ptr<uint32_t> ids = as_global(sc.idx[0]) + (size_t)row * sc.vpad;
            for (uint32_t i = w * (uint32_t)kThreads + tid; i < len; i += W * (uint32_t)kThreads)
                ids[i] = i;
        }
        leave(len, step == 1u ? 0u : now.pre, used, from_buf);
        return kNthLast;
    }
    const bool goes_on = out_len > kNthUntil && nth < out_len; // uniform
    // the entry at i of the old list; a row that is its own list has no token ids, and its first entry has yet to change places
    // with the pivot
    NthFirst own = {0u, 0u, kNone, 0u};
    if (step == 1u && !compact)
        own = first;
    const bool ids_implied = step == 1u;
    auto entry = [&](uint32_t i) {
        i = min(i, len - 1u);
        const uint32_t k = kin[i], id = ids_implied ? i : iin[i];
        return i == own.from ? ((u64)own.first_key << 32) : (((u64)k << 32) | (u64)id);
    };
    auto ones_before = [&](uint32_t p) { return pre[p >> 6] + (uint32_t)__popcll(bits[p >> 6] & ((1ull << (p & 63u)) - 1ull)); };
    // the place of the s-th set bit, by one wave
    auto word_of = [&](uint32_t s) {
        const uint32_t c = (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(lane * 64u <= words && pre[min(lane * 64u, words)] <= s)) - 1u;
        const uint32_t i = c * 64u + lane;
        return c * 64u + (uint32_t)__popcll(__builtin_amdgcn_ballot_w64(i < words && pre[min(i, words)] <= s)) - 1u;
    };
    auto place_of = [&](uint32_t s) {
        const uint32_t j = word_of(s);
        const u64 x = bits[j];
        const u64 hit = __builtin_amdgcn_ballot_w64(((x >> lane) & 1ull) && mask_rank(x) == s - pre[j]);
        return j * 64u + (uint32_t)__ffsll((long long)hit) - 1u;
    };
    // what the new list has at p (> 0 unless the list is only moved together)
    auto source = [&](uint32_t p) {
        if (compact)
            return place_of(p);
        if ((bits[p >> 6] >> (p & 63u)) & 1ull) // uniform
            return p;
        return place_of(smalls - 1u - (p - 1u - ones_before(p)));
    };
    // Which entries the next pivot is chosen from, and what is at the front until then (the waves ask for one each, and go on)
    u64 mine = 0, pivot = 0, front = 0;
    uint32_t pivot_at = kNone;
    if (wave < 4u && out_len != 0u && (goes_on || wave == 3u)) {
        const uint32_t p = wave == 0u ? 1u : (wave == 1u ? out_len / 2u : (wave == 2u ? out_len - 1u : 0u));
        if (wave == 3u && !compact)
            mine = step == 1u ? ((u64)own.pivot_key << 32) | (u64)own.pivot_id : entry(0u);
        else
            mine = entry(uniform_u32(source(p)));
    }
    uint32_t* bits_out = nth_bits(sc, row, to_buf);
    // (equal shares for the workgroups, in as few turns as hold them.  Where few entries are left their fillers come from far
    // apart, and in pieces of 4 096 one workgroup of eight went through half of the old list for them, 22 us)
    const uint32_t shares = W * ((out_len + W * kNthChunk - 1u) / (W * kNthChunk));
    const uint32_t chunk = out_len ? (((out_len + shares - 1u) / shares) + kGroup - 1u) & ~(kGroup - 1u) : kNthChunk;
    for (uint32_t c = w; c * chunk < out_len; c += W) { // uniform
        const uint32_t p0 = c * chunk, p1 = min(p0 + chunk, out_len);
        const uint32_t p = p0 + 4u * tid, pc = min(p, (out_len - 1u) & ~3u); // (rows' arrays are a multiple of 1 024 long)
        u32x4 k = {0u, 0u, 0u, 0u}, id = {0u, 0u, 0u, 0u};
        // set bits [s_lo, s_hi) are wanted here: those of the holes' fillers, of which the hole in front takes the last, or
        // the entries themselves
        uint32_t s_lo = p0, s_hi = p1, holes_before = 0;
        if (!compact) { // uniform
            k = *(global_ptr<const u32x4>)(kin + pc);
            if (ids_implied)
                id = u32x4{pc, pc + 1u, pc + 2u, pc + 3u};
            else
                id = *(global_ptr<const u32x4>)(iin + pc);
            holes_before = p0 ? p0 - 1u - uniform_u32(ones_before(p0)) : 0u;
            const uint32_t holes_to = p1 - 1u - uniform_u32(p1 < len ? ones_before(p1) : smalls);
            s_lo = smalls - holes_to;
            s_hi = smalls - holes_before;
        }
        if (s_lo < s_hi) { // uniform
            const uint32_t b_lo = uniform_u32(word_of(s_lo)) / 4u, b_hi = uniform_u32(word_of(s_hi - 1u)) / 4u;
            constexpr uint32_t kTrip = 2;
            for (uint32_t b = b_lo + wave; b <= b_hi; b += kTrip * (uint32_t)kWaves) { // uniform per wave
                u32x4 fk[kTrip], fi[kTrip];
#pragma unroll
                for (uint32_t u = 0; u < kTrip; ++u) {
                    const uint32_t at = min((b + u * (uint32_t)kWaves) * kGroup + 4u * lane, (len - 1u) & ~3u);
                    fk[u] = *(global_ptr<const u32x4>)(kin + at);
                    if (ids_implied)
                        fi[u] = u32x4{at, at + 1u, at + 2u, at + 3u};
                    else
                        fi[u] = *(global_ptr<const u32x4>)(iin + at);
                }
#pragma unroll
                for (uint32_t u = 0; u < kTrip; ++u) {
                    const uint32_t at = (b + u * (uint32_t)kWaves) * kGroup + 4u * lane;
                    if (b + u * (uint32_t)kWaves > b_hi || at >= len)
                        continue;
                    const u64 x = bits[at >> 6];
                    uint32_t s = pre[at >> 6] + (uint32_t)__popcll(x & ((1ull << (at & 63u)) - 1ull));
                    const uint32_t nibble = (uint32_t)(x >> (at & 63u)) & 15u;
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j)
                        if ((nibble >> j) & 1u) {
                            const u64 v = at + j == own.from ? ((u64)own.first_key << 32) : (((u64)fk[u][j] << 32) | (u64)fi[u][j]);
                            if (s >= s_lo && s < s_hi)
                                buf[compact ? s - s_lo : s_hi - 1u - s] = v;
                            ++s;
                        }
                }
            }
        }
        if (c == w && wave < 4u && lane == 0u)
            bs.u64[wave] = mine;
        __syncthreads();
        if (c == w) { // uniform
            front = bs.u64[3];
            if (goes_on)
                median_of_three<u64>(bs.u64[0], bs.u64[1], bs.u64[2], 1u, out_len / 2u, out_len - 1u, pivot, pivot_at);
        }
        u64 v[4];
        uint32_t hole = 0, nibble = 0;
        if (!compact) { // uniform
            const u64 x = bits[pc >> 6];
            nibble = (uint32_t)(x >> (pc & 63u)) & 15u;
            hole = (pc ? pc - 1u : 0u) - (pre[pc >> 6] + (uint32_t)__popcll(x & ((1ull << (pc & 63u)) - 1ull))) - holes_before;
        }
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) {
            const uint32_t pj = p + j;
            if (compact) {
                v[j] = buf[min(pj - p0, kNthChunk - 1u)];
            } else if (pj == 0u) {
                v[j] = front;
            } else if ((nibble >> j) & 1u) {
                v[j] = pj == own.from ? ((u64)own.first_key << 32) : (((u64)k[j] << 32) | (u64)id[j]);
            } else {
                v[j] = buf[min(hole, kNthChunk - 1u)];
                ++hole;
            }
        }
        uint32_t left = 0;
        if (goes_on) { // uniform: the next pivot to the front, and who belongs left of it
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t pj = p + j;
                v[j] = pj == pivot_at ? front : v[j];
                left |= (pj != 0u && pj < out_len && v[j] < pivot ? 1u : 0u) << j;
                v[j] = pj == 0u ? pivot : v[j];
            }
        }
        if (p < p1) {
            MAKO_CHECK(sc, kCheckCompact, (uint64_t)p + 3u < sc.vpad);
            *(global_ptr<u32x4>)(kout + p) = u32x4{(uint32_t)(v[0] >> 32), (uint32_t)(v[1] >> 32), (uint32_t)(v[2] >> 32), (uint32_t)(v[3] >> 32)};
            *(global_ptr<u32x4>)(iout + p) = u32x4{(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
        }
        if (goes_on) { // uniform
            const uint32_t word = eight_nibbles(left);
            if ((lane & 7u) == 0u && (p & ~(kGroup - 1u)) < p1)
                as_global(bits_out)[p >> 5] = word;
        }
        __syncthreads(); // (the fillers' buffer)
    }
    leave(out_len, goes_on ? kNthBits : 0u, used + (compact ? 0u : 1u), to_buf);
    return goes_on ? kNthMore : kNthLast;
}

// The row's workgroups meet behind step `step` (without `wait` they only count).  Returns whether they go on with the next.  They
// don't where one has waited `polls` times: the others may have to wait for a CU themselves, behind another stream's work, and
// nothing may depend on that.  Whoever gives up says so and the rest follow, each at its next meeting at the latest; the row's
// one workgroup in the last launch goes on from the last step that all W have made, whose list no later step has touched (two
// lists, two records and two rows of bits, in turn).  All threads of all of the row's W workgroups call.
__device__ __forceinline__ bool nth_meet(BigPlan* plan, uint32_t step, uint32_t W, bool wait, uint32_t polls, BlockScratch& bs)
{
    constexpr uint32_t kGivenUp = 0x80000000u;
    const global_ptr<uint32_t> met = as_global(plan->cap + kNthMet);
    if (wait) // uniform: the wave's stores have arrived where the fence finds them
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) {
        if (wait)
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const uint32_t upto = W * step;
        bool all = ((__hip_atomic_fetch_add(met, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u) & ~kGivenUp) == upto;
        if (all) // (the last of them; of different steps' last, the later step counts)
            __hip_atomic_fetch_max(as_global(plan->cap + kNthMade), step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (uint32_t i = 0; wait && !all; ++i) {
            const uint32_t v = __hip_atomic_load(met, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            all = (v & ~kGivenUp) >= upto;
            if (all || (v & kGivenUp))
                break;
            if (i >= polls) {
                __hip_atomic_fetch_or(met, kGivenUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
            __builtin_amdgcn_s_sleep(2);
        }
        if (wait)
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        bs.bcast = all ? 1u : 0u;
    }
    if (!wait) // uniform
        return false;
    __syncthreads();
    const bool go = bs.bcast != 0u;
    __syncthreads();
    return go;
}

// All of a row's steps by the same workgroups, in one launch that has other work besides (sort_beside_kernel).  All threads call.
__device__ __forceinline__ void nth_steps_at_once(const mako_sample_desc& d, const Scratch& sc, uint32_t row, uint32_t w, uint32_t W,
                                                  unsigned long long* lds_dyn, BlockScratch& bs)
{
    constexpr uint32_t kStepsMax = 12; // (of the 30 rounds and more before the depth limit)
    // (140 us: twice what all steps of 24 rows of 151 553 take.  A checked build's even rows don't wait at all.)
#ifdef MAKO_CHECKED
    const uint32_t polls = (row & 1u) ? 400u : 0u;
#else
    constexpr uint32_t polls = 400u;
#endif
    // (the first step apart, which has no token ids to read: one workgroup takes 97 us for it, 117 otherwise)
    NthMadeOf made = nth_step(d, sc, row, w, W, 1u, lds_dyn, bs);
    if (made == kNthNone)
        return;
    if (made == kNthLast || W == 1u) { // uniform; all of them make the first
        if (w == 0u && threadIdx.x == 0u)
            sc.plan[row].cap[kNthMade] = 1u;
        return;
    }
    for (uint32_t step = 1; nth_meet(sc.plan + row, step, W, made == kNthMore && step < kStepsMax, polls, bs);) {
        // (one step's addresses are not kept for the next: the scalar registers do not suffice)
        uint32_t r = uniform_u32(row), wr = uniform_u32(w), Wr = uniform_u32(W);
        asm volatile("" : "+s"(r), "+s"(wr), "+s"(Wr));
        made = nth_step(d, sc, r, wr, Wr, ++step, lds_dyn, bs);
    }
}

} // namespace mako
