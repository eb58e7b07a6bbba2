// A thread's sixteen logits of a slice: loaded, masked and penalised (src/gen/sampler.cpp:22-28).
#pragma once

#include "sampler_common.h"

namespace mako {

// Thread t of a slice owns 16 logits: for k = 0..3 the four consecutive ones at lo + k * kBlock + 4 * t.  A wavefront's
// loads are contiguous and each logit is read once.
constexpr uint32_t kBlock = 4u * (uint32_t)kThreads;
__device__ __forceinline__ uint32_t elem_index(uint32_t lo, uint32_t tid, uint32_t j)
{
    return lo + (j >> 2) * kBlock + tid * 4u + (j & 3u);
}
// The t that a thread is there.  MIXED: a wave has sixteen logits of every 256, in place of 256 of every 4 096.
template <bool MIXED>
__device__ __forceinline__ uint32_t slice_thread()
{
    const uint32_t tid = threadIdx.x;
    return MIXED ? (tid & 3u) | ((tid >> 6) << 2) | ((tid & 0x3cu) << 4) : tid;
}

// A slice that scan_kernel takes MIXED: too long for a candidate list of all of it, and so short that the waves have 256 logits in
// a row each, or none.  The smallest of the waves' thresholds is the slice's, so that a single wave whose logits are not like the
// others' makes the list overflow: one without logits, whose threshold is -inf, or the first tokens', which a long history
// penalises most.  The row is then left to the whole-row path.  (Flat rows with penalties over histories of 5 000 tokens, mixed and
// not: six of 2 067 33 us and 74, 17 of 4 101 17.9 and 86; a top-k row of 1 003 12.1 and 39.  From 5 120 on the waves that
// hold the first tokens have others besides: 17 of 5 125 17.6 either way.)
__host__ __device__ inline bool short_slice(uint32_t len) // (len: as slice_len, rounded up to a multiple of four)
{
    // (128 groups of four at least, eight a wave, as many as a top_k of kTopKFast asks each for)
    static_assert(kTopKFast <= (kCap / 4u / (kSliceThreads / 64u)) * (kSliceThreads / 64u), "no wave is asked for more logits than it has");
    return len < 5u * kSliceThreads && len > kCap;
}

// accept() history -> per-token counts for [lo, hi) in LDS (src/gen/sampler.cpp:15-18); generic form used
// when a row's history is too long for the register-resident scheme of load_penalised().
__device__ __forceinline__ void build_counts(const mako_sample_desc& d, uint32_t row, uint32_t hl, uint32_t lo,
                                             uint32_t hi, uint32_t slice_len, uint32_t* s_cnt)
{
    const uint32_t tid = threadIdx.x;
    uint4* z = reinterpret_cast<uint4*>(s_cnt); // slice_len is a multiple of 4
    for (uint32_t i = tid; i < slice_len / 4; i += kThreads)
        z[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    const global_ptr<const int32_t> ht = as_global(d.hist_tokens) + (int64_t)row * d.hist_stride;
    const global_ptr<const uint32_t> hc = d.hist_counts ? as_global(d.hist_counts) + (int64_t)row * d.hist_stride : nullptr;
    for (uint32_t h = tid; h < hl; h += kThreads) {
        const uint32_t t = (uint32_t)ht[h];
        if (t >= lo && t < hi)
            atomicAdd(&s_cnt[t - lo], hc ? hc[h] : 1u);
    }
    __syncthreads();
}

// The thread's 16 logits, raw, plus the mask bits of each group of four.
// Issued before anything else so that the HBM latency overlaps the LDS work that follows.
// ALIGNED: the rows are 16-byte aligned and a multiple of four long.  Of any other row a group of four is loaded the same way,
// from a multiple of four bytes, and the row's last group from four logits in front of its end (settle_slice()).  (One logit
// at a time, 1 024 apart, the loads take four times the instructions and twice the registers, and no two workgroups of
// scan_kernel and index_weights_kernel shared a CU: 64 rows of 129 281 logits, temperature only, 84 us and 79 so; a decode
// batch of 64 such rows 71 and 63; 256 top-k rows under masks 105 and 42, and 40 where the rows are aligned.)
struct RawSlice {
    float4 v[4];
    uint32_t bits[4]; // bit c of bits[k] = logit 4k+c allowed
};
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

template <bool ALIGNED, bool MIXED = false>
__device__ __forceinline__ void load_raw(const mako_sample_desc& d, uint32_t row, uint32_t lo, uint32_t hi, RawSlice& r)
{
    const uint32_t tid = slice_thread<MIXED>();
    const global_ptr<const float> lrow = as_global(d.logits) + (int64_t)row * d.logits_stride;
    const global_ptr<const uint32_t> mrow = d.mask ? as_global(d.mask) + (int64_t)row * d.mask_stride : nullptr;
    // all four loads go out back to back, from clamped addresses and without a branch between them (a branch
    // would make the compiler wait for each load before the next); what lies past the slice is dropped after
    uint32_t at[4];
    if (!ALIGNED && d.n_vocab < 4u) { // uniform
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            at[k] = 0u;
            float* v = reinterpret_cast<float*>(&r.v[k]);
#pragma unroll
            for (uint32_t c = 0; c < 4; ++c) // (where settle_slice() expects them)
                v[c] = lrow[c + d.n_vocab > 4u ? c + d.n_vocab - 4u : 0u];
        }
    } else {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t i = lo + k * kBlock + tid * 4u;
            at[k] = i < hi ? i : (hi - 1u) & ~3u;
            f32x4 x;
            if (ALIGNED)
                x = *(global_ptr<const f32x4>)(lrow + at[k]);
            else
                x = *(global_ptr<const f32x4_any>)(lrow + min(at[k], d.n_vocab - 4u));
            r.v[k] = make_float4(x.x, x.y, x.z, x.w);
        }
    }
    if (mrow) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            r.bits[k] = mrow[at[k] >> 5] >> (at[k] & 31u);
    }
    if (!mrow) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            r.bits[k] = 0xfu;
    }
    // (finish_slice() replaces what was read past the slice: nothing here touches the loaded values, so the
    // loads stay in flight while the caller goes on)
}

// The row's last group, of one to three logits, moved to the front of its four, behind it NaN.  (A slice ends behind a whole
// group everywhere else.)
template <bool ALIGNED, bool MIXED = false>
__device__ __forceinline__ void settle_slice(RawSlice& r, uint32_t lo, uint32_t hi)
{
    if (ALIGNED || (hi & 3u) == 0u) // uniform
        return;
    const float nan = __uint_as_float(0x7fc00000u);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (lo + k * kBlock + slice_thread<MIXED>() * 4u == (hi & ~3u)) {
            const uint32_t n = hi & 3u;
            const float4 x = r.v[k];
            r.v[k].x = n == 3u ? x.y : (n == 2u ? x.z : x.w);
            r.v[k].y = n == 3u ? x.z : (n == 2u ? x.w : nan);
            r.v[k].z = n == 3u ? x.w : nan;
            r.v[k].w = nan;
        }
    }
}

// How many of the thread's logits (as the sampler is given them: a token the mask clears is -inf) are strictly
// greater than v: the count of ReasoningBudget::forced, src/server/openai.cpp:599-602.
template <bool MIXED>
__device__ __forceinline__ uint32_t count_above(const RawSlice& r, uint32_t lo, uint32_t hi, float v)
{
    const uint32_t tid = slice_thread<MIXED>();
    uint32_t c = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        if (lo + k * kBlock + tid * 4u < hi) { // (what lies behind the row's last logit in its group is NaN)
            c += ((r.bits[k] & 1u) && r.v[k].x > v) ? 1u : 0u;
            c += ((r.bits[k] & 2u) && r.v[k].y > v) ? 1u : 0u;
            c += ((r.bits[k] & 4u) && r.v[k].z > v) ? 1u : 0u;
            c += ((r.bits[k] & 8u) && r.v[k].w > v) ? 1u : 0u;
        }
    }
    return c;
}

// Mask and penalties (src/gen/sampler.cpp:22-28) applied to the raw logits; slots past the end of the
// slice hold NaN, which never wins a comparison and never becomes a candidate.
template <bool ALIGNED, bool MIXED = false>
__device__ __forceinline__ void finish_slice(const RawSlice& r, uint32_t lo, uint32_t hi, const mako_sampling_params& P,
                                             bool pen, const uint32_t* s_cnt, float (&wv)[16], bool masked)
{
    const uint32_t tid = slice_thread<MIXED>();
    const float nan = __uint_as_float(0x7fc00000u);
    if (!masked) { // uniform: no mask, nothing to clear
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const bool inside = lo + k * kBlock + tid * 4u < hi;
            wv[4 * k + 0] = !inside ? nan : r.v[k].x;
            wv[4 * k + 1] = !inside ? nan : r.v[k].y;
            wv[4 * k + 2] = !inside ? nan : r.v[k].z;
            wv[4 * k + 3] = !inside ? nan : r.v[k].w;
        }
    } else {
        // (a mask bit spread over a word, then one bit-field insert: the logit where the bit is set, -inf elsewhere)
        auto pick = [](uint32_t bits, uint32_t c, float v) {
            const uint32_t m = (uint32_t)((int32_t)(bits << (31u - c)) >> 31); // all ones if bit c is set
            return __uint_as_float((__float_as_uint(v) & m) | (0xff800000u & ~m));
        };
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t i = lo + k * kBlock + tid * 4u;
            // (a bit behind the row's last logit may be anything)
            auto inside = [&](uint32_t c) { return ALIGNED ? i < hi : i + c < hi; };
            wv[4 * k + 0] = !inside(0u) ? nan : pick(r.bits[k], 0, r.v[k].x);
            wv[4 * k + 1] = !inside(1u) ? nan : pick(r.bits[k], 1, r.v[k].y);
            wv[4 * k + 2] = !inside(2u) ? nan : pick(r.bits[k], 2, r.v[k].z);
            wv[4 * k + 3] = !inside(3u) ? nan : pick(r.bits[k], 3, r.v[k].w);
        }
    }
    if (pen) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) {
            const uint32_t i = lo + k * kBlock + tid * 4u;
            if (i < hi) {
                const uint4 n = *reinterpret_cast<const uint4*>(s_cnt + (i - lo));
                if (n.x | n.y | n.z | n.w) {
                    if (n.x)
                        wv[4 * k + 0] = penalize(wv[4 * k + 0], n.x, P.repetition_penalty, P.presence_penalty, P.frequency_penalty);
                    if (n.y)
                        wv[4 * k + 1] = penalize(wv[4 * k + 1], n.y, P.repetition_penalty, P.presence_penalty, P.frequency_penalty);
                    if (n.z)
                        wv[4 * k + 2] = penalize(wv[4 * k + 2], n.z, P.repetition_penalty, P.presence_penalty, P.frequency_penalty);
                    if (n.w)
                        wv[4 * k + 3] = penalize(wv[4 * k + 3], n.w, P.repetition_penalty, P.presence_penalty, P.frequency_penalty);
                }
            }
        }
    }
}

// The thread's logits after the mask and the penalties (src/gen/sampler.cpp:22-28): wv[16] in the slice layout.
//
// KH > 0 (histories of at most KH * kThreads entries): thread t handles history entries t, t + kThreads, ...  The
// per-token counts are accumulated in LDS; for every distinct token of the slice the thread holding its first
// entry (an election, so that each token is handled once) computes the penalised logit: one IEEE division per
// history entry instead of one per logit slot.  The logit travels through the token's slot of the LDS table:
// its owner puts the masked raw value there, the elected thread replaces it by the penalised one, the owner
// takes it back.  (A gather from device memory instead would return behind every streaming load in flight, and
// costs the slices that hold most of a Zipf history a microsecond more.)
// KH == 0: any history length; counts in LDS, every owner penalises its own logits.
struct NoOverlap {
    __device__ __forceinline__ void operator()() const {}
};

// A slice's loads on their way: the thread's logits and history entries (KH > 0).
template <int KH>
struct SliceLoads {
    RawSlice raw;
    uint32_t tok[KH > 0 ? KH : 1], cnt[KH > 0 ? KH : 1];
};
template <bool ALIGNED, int KH, bool MIXED = false>
__device__ __forceinline__ void issue_slice(const mako_sample_desc& d, uint32_t row, uint32_t lo, uint32_t hi, SliceLoads<KH>& s)
{
    const uint32_t tid = threadIdx.x;
    // My history entries go first: loads return in the order they were issued, so whatever waits for these does not
    // wait for the logits behind them, and the counting in LDS below runs while the logits are still on their way.
    // (Loads from clamped positions, issued without branches between them; what was not wanted is dropped
    // afterwards: a branch around each load would make every load wait for the one before.)
    // Whether they are asked for depends on the kernel's arguments alone, not on the row's parameters or its history
    // length: a caller may still be waiting for those when these loads and the logits' go out.
    if (KH > 0 && d.hist_tokens != nullptr && d.hist_stride > 0) { // uniform
        const global_ptr<const int32_t> ht = as_global(d.hist_tokens) + (int64_t)row * d.hist_stride;
        const uint32_t last = (uint32_t)d.hist_stride - 1u; // (entries past the row's length are read and dropped)
#pragma unroll
        for (int k = 0; k < KH; ++k)
            s.tok[k] = (uint32_t)ht[min(tid + (uint32_t)k * kThreads, last)];
        if (d.hist_counts) {
            const global_ptr<const uint32_t> hc = as_global(d.hist_counts) + (int64_t)row * d.hist_stride;
#pragma unroll
            for (int k = 0; k < KH; ++k)
                s.cnt[k] = hc[min(tid + (uint32_t)k * kThreads, last)];
        }
    }
    load_raw<ALIGNED, MIXED>(d, row, lo, hi, s.raw);
}
// (the table of counts is cleared while the loads are on their way, also for a row that may turn out to have no history;
// `penalised`: it has penalties, and a use for them)
template <int KH>
__device__ __forceinline__ void clear_counts(const mako_sample_desc& d, bool penalised, uint32_t slice_len, uint32_t* s_cnt)
{
    if (KH > 0 && penalised && d.hist_tokens != nullptr && d.hist_stride > 0) { // uniform
        uint4* z = reinterpret_cast<uint4*>(s_cnt); // slice_len is a multiple of 4
        for (uint32_t i = threadIdx.x; i < slice_len / 4; i += kThreads)
            z[i] = make_uint4(0, 0, 0, 0);
    }
}

// The rest, on what issue_slice() has asked for; the table is clear.
template <bool ALIGNED, int KH, bool MIXED = false>
__device__ __forceinline__ void finish_penalised(const mako_sample_desc& d, uint32_t row, uint32_t lo, uint32_t hi, uint32_t slice_len,
                                                 const mako_sampling_params& P, uint32_t hl, bool pen, uint32_t* s_cnt, SliceLoads<KH>& s,
                                                 float (&wv)[16], bool want_above = false, float close_v = 0.0f, uint32_t* above = nullptr)
{
    const uint32_t tid = threadIdx.x, mine = slice_thread<MIXED>();
    RawSlice& raw = s.raw;
    uint32_t (&tok)[KH > 0 ? KH : 1] = s.tok;
    uint32_t (&cnt)[KH > 0 ? KH : 1] = s.cnt;
    const bool hc = d.hist_counts != nullptr;
    bool have[KH > 0 ? KH : 1];
    if (want_above) { // uniform
        settle_slice<ALIGNED, MIXED>(raw, lo, hi);
        *above = count_above<MIXED>(raw, lo, hi, close_v);
    }
    auto settle = [&]() {
        if (!want_above)
            settle_slice<ALIGNED, MIXED>(raw, lo, hi);
    };
    if (!pen) {
        settle();
        finish_slice<ALIGNED, MIXED>(raw, lo, hi, P, false, s_cnt, wv, d.mask != nullptr);
        return;
    }
    if (KH == 0) {
        build_counts(d, row, hl, lo, hi, slice_len, s_cnt);
        settle();
        finish_slice<ALIGNED, MIXED>(raw, lo, hi, P, true, s_cnt, wv, d.mask != nullptr);
        return;
    }
#pragma unroll
    for (int k = 0; k < KH; ++k) {
        if (!hc)
            cnt[k] = 1;
        // (an entry that counts no occurrence is no entry: the reference's table holds what accept() has seen)
        have[k] = tid + (uint32_t)k * kThreads < hl;
        if (!(have[k] && tok[k] >= lo && tok[k] < hi && cnt[k] != 0u)) {
            tok[k] = kNone;
            cnt[k] = 0;
        }
    }
    // (barriers that order LDS traffic only: the logits stay in flight)
    MAKO_STAMP(20);
    lds_barrier();
    MAKO_STAMP(21);
    // every entry adds its occurrences to its token's slot; the entry that finds the slot empty speaks for the
    // token from here on (which of a token's entries that is does not matter: it only carries the logit through
    // penalize() once)
    bool elected[KH > 0 ? KH : 1];
#pragma unroll
    for (int k = 0; k < KH; ++k) {
        elected[k] = false;
        if (tok[k] != kNone)
            elected[k] = atomicAdd(&s_cnt[tok[k] - lo], cnt[k]) == 0u;
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < KH; ++k)
        if (elected[k])
            cnt[k] = s_cnt[tok[k] - lo]; // occurrences of the token in the whole history
    lds_barrier(); // (the slots are about to be overwritten)
    MAKO_STAMP(22);
    settle();
    finish_slice<ALIGNED, MIXED>(raw, lo, hi, P, false, s_cnt, wv, d.mask != nullptr);
    MAKO_STAMP(23);
    // owners: a logit whose slot is taken goes into the slot (its bits); `moved` remembers which of the sixteen
    uint32_t moved = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t i = lo + k * kBlock + mine * 4u;
        if (i < hi) {
            uint4* slot = reinterpret_cast<uint4*>(s_cnt + (i - lo));
            const uint4 n = *slot;
            if (n.x | n.y | n.z | n.w) {
                *slot = make_uint4(n.x ? __float_as_uint(wv[4 * k + 0]) : 0u, n.y ? __float_as_uint(wv[4 * k + 1]) : 0u,
                                   n.z ? __float_as_uint(wv[4 * k + 2]) : 0u, n.w ? __float_as_uint(wv[4 * k + 3]) : 0u);
                moved |= ((n.x ? 1u : 0u) | (n.y ? 2u : 0u) | (n.z ? 4u : 0u) | (n.w ? 8u : 0u)) << (4u * k);
            }
        }
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < KH; ++k)
        if (elected[k]) {
            const float rv = __uint_as_float(s_cnt[tok[k] - lo]); // (already -inf where the mask clears the token)
            s_cnt[tok[k] - lo] =
                __float_as_uint(penalize(rv, cnt[k], P.repetition_penalty, P.presence_penalty, P.frequency_penalty));
        }
    lds_barrier();
    if (moved) {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if ((moved >> (4u * k)) & 0xfu) {
                const uint4 v = *reinterpret_cast<const uint4*>(s_cnt + (k * kBlock + mine * 4u));
                wv[4 * k + 0] = (moved >> (4u * k)) & 1u ? __uint_as_float(v.x) : wv[4 * k + 0];
                wv[4 * k + 1] = (moved >> (4u * k)) & 2u ? __uint_as_float(v.y) : wv[4 * k + 1];
                wv[4 * k + 2] = (moved >> (4u * k)) & 4u ? __uint_as_float(v.z) : wv[4 * k + 2];
                wv[4 * k + 3] = (moved >> (4u * k)) & 8u ? __uint_as_float(v.w) : wv[4 * k + 3];
            }
    }
}

// `overlap` runs right after the slice's loads have been issued: work that does not depend on them hides
// behind their latency.  It must be reached by the whole workgroup or by none of it.
template <bool ALIGNED, int KH, bool MIXED = false, typename Overlap = NoOverlap>
__device__ __forceinline__ void load_penalised(const mako_sample_desc& d, uint32_t row, uint32_t lo, uint32_t hi,
                                               uint32_t slice_len, const mako_sampling_params& P, bool penalised, uint32_t hl, bool pen,
                                               uint32_t* s_cnt, float (&wv)[16], Overlap overlap = Overlap(),
                                               bool want_above = false, float close_v = 0.0f, uint32_t* above = nullptr)
{
    SliceLoads<KH> s;
    issue_slice<ALIGNED, KH, MIXED>(d, row, lo, hi, s);
    clear_counts<KH>(d, penalised, slice_len, s_cnt);
    overlap();
    finish_penalised<ALIGNED, KH, MIXED>(d, row, lo, hi, slice_len, P, hl, pen, s_cnt, s, wv, want_above, close_v, above);
}

} // namespace mako
