// A sorted (or token-ordered) list of weights in groups of 256: what a group adds to the running fp32 sum and takes off
// the walk's r as one number, and the exact replay of a group in which the binade changes.
#pragma once

#include "workgroup_state.h"
#include "unsorted_shares.h"

namespace mako {

// A double from a lane whose number is the same for the whole wave.
__device__ __forceinline__ double readlane_f64(double v, uint32_t lane)
{
    const long long b = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, (int)lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), (int)lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

__device__ __forceinline__ float readlane_f32(float v, uint32_t lane)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), (int)lane));
}
__device__ __forceinline__ float uniform_f32(float v)
{
    return __uint_as_float((uint32_t)__builtin_amdgcn_readfirstlane((int)__float_as_uint(v)));
}

// Cross-lane moves on the VALU data path (DPP) instead of through the LDS crossbar: a dependent chain of six
// of them costs tens of cycles, not hundreds.  Lanes without a source lane receive 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_or_zero(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xf, false);
}

// Inclusive scan, in lane order, of the 64 lanes' maps under composition.
__device__ __forceinline__ void wave_scan_maps(uint32_t& d0, uint32_t& d1)
{
    using seqfp::Step32;
#define MAKO_SCAN_STEP(CTRL, ROW_MASK)                                                                               \
    {                                                                                                                \
        const Step32 t = Step32{dpp_or_zero<CTRL, ROW_MASK>(d0), dpp_or_zero<CTRL, ROW_MASK>(d1)};                   \
        const Step32 r = seqfp::compose32(t, Step32{d0, d1}); /* earlier lanes first; {0, 0} is the identity */      \
        d0 = r.d0;                                                                                                   \
        d1 = r.d1;                                                                                                   \
    }
    MAKO_SCAN_STEP(0x111, 0xf) // row_shr:1
    MAKO_SCAN_STEP(0x112, 0xf) // row_shr:2
    MAKO_SCAN_STEP(0x114, 0xf) // row_shr:4
    MAKO_SCAN_STEP(0x118, 0xf) // row_shr:8
    MAKO_SCAN_STEP(0x142, 0xa) // row_bcast:15 into rows 1 and 3
    MAKO_SCAN_STEP(0x143, 0xc) // row_bcast:31 into rows 2 and 3
#undef MAKO_SCAN_STEP
}

__device__ __forceinline__ int exponent_of(float x)
{
    uint32_t M;
    int e;
    seqfp::split(x, M, e);
    return e;
}

// A sorted list's keys, wherever they are (LDS or device memory: loads through a generic pointer, which the
// hardware completes in no particular order, so that the code has to wait for all of them at once) ...
struct AnyKeys {
    const uint32_t* p;
    __device__ __forceinline__ uint32_t operator[](uint32_t i) const { return p[i]; }
    __device__ __forceinline__ uint4 vec(uint32_t i) const { return *reinterpret_cast<const uint4*>(p + i); }
};
// ... or known to be in device memory: plain global loads, which can be left in flight and waited for one by one.
struct GlobalKeys {
    const uint32_t* p;
    __device__ __forceinline__ uint32_t operator[](uint32_t i) const
    {
        return ((const __attribute__((address_space(1))) uint32_t*)p)[i];
    }
    __device__ __forceinline__ uint4 vec(uint32_t i) const
    {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        const u32x4 v = *((const __attribute__((address_space(1))) u32x4*)(p + i));
        return make_uint4(v.x, v.y, v.z, v.w);
    }
};

// The four weights a lane owns in the span of `len` (<= kGroup) entries that starts at kf[start]: entries
// 4 * lane .. 4 * lane + 3, 0.0f past the end.  kf itself is 16-byte aligned.
template <typename Keys>
__device__ __forceinline__ void load_span(Keys kf, uint32_t start, uint32_t len, float (&q)[4])
{
    const uint32_t i = lane_id() * 4u;
    uint32_t k[4] = {0u, 0u, 0u, 0u}; // bits(0.0f)
    if ((start & 3u) == 0 && i + 3 < len) {
        const uint4 x = kf.vec(start + i);
        k[0] = ~x.x;
        k[1] = ~x.y;
        k[2] = ~x.z;
        k[3] = ~x.w;
    } else if (len) {
        // (every load from a position inside the span, and what lies past the end masked with an AND: a select
        // would be turned into a branch around each load, and each would wait for the one before)
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
            k[j] = ~kf[start + min(i + j, len - 1u)] & (i + j < len ? 0xffffffffu : 0u);
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
        q[j] = __uint_as_float(k[j]);
}
__device__ __forceinline__ void load_span(const uint32_t* kf, uint32_t start, uint32_t len, float (&q)[4])
{
    load_span(AnyKeys{kf}, start, len, q);
}

// The entries of one span (at most 256), one per lane and register: x[j] of lane l is entry 64 * j + l, 0.0f past
// the end.
template <typename Keys>
__device__ __forceinline__ void load_span_lanes(Keys kf, uint32_t start, uint32_t len, float (&x)[4])
{
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t i = j * kWave + lane_id();
        // (every lane loads, from inside the span; masked with an AND, as in load_span)
        x[j] = __uint_as_float(~kf[start + min(i, len - 1u)] & (i < len ? 0xffffffffu : 0u));
    }
}
// A sequential chain over 64 entries, one per lane: behind it lane t holds what `for (...) v += x` (or `v -= x`) holds
// behind entry t.  Every step is the same instruction: a lane takes the value of the lane below it and adds its own
// entry, lane 0, which has none below, keeps v0 + x.  Step k makes lane k's value right, and as the lane below it stays
// right, it stays so: after `steps` of them the lanes up to `steps` are done (whatever the others hold).  One dependent
// instruction per entry, 5 ns, and every intermediate value at hand at the end.  (s_nop: a DPP operand is read two cycles
// after it was written at the earliest.)
template <bool SUB>
__device__ __forceinline__ float lane_chain(float v0, float x, uint32_t steps)
{
    float v = SUB ? v0 - x : v0 + x; // (right in lane 0)
#define MAKO_CHAIN4(OP) \
    asm volatile("s_nop 1\n\t" OP "\n\ts_nop 1\n\t" OP "\n\ts_nop 1\n\t" OP "\n\ts_nop 1\n\t" OP : "+v"(v) : "v"(x));
    for (uint32_t k = 0; k < steps; k += 16u) { // uniform
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            if (SUB)
                MAKO_CHAIN4("v_sub_f32_dpp %0, %0, %1 wave_shr:1 row_mask:0xf bank_mask:0xf")
            else
                MAKO_CHAIN4("v_add_f32_dpp %0, %0, %1 wave_shr:1 row_mask:0xf bank_mask:0xf")
        }
    }
#undef MAKO_CHAIN4
    return v;
}

// S plus the entries of one span (n in 1..256, in registers as load_span_lanes() leaves them), added one by one in fp32
// (src/gen/sampler.cpp:80-82).  One wave.
__device__ __forceinline__ float lanes_sum(const float (&x)[4], uint32_t n, float S)
{
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
        if (j * kWave < n) { // uniform
            const uint32_t m = min(n - j * kWave, (uint32_t)kWave);
            S = readlane_f32(lane_chain<false>(S, x[j], m), m - 1u);
        }
    return S;
}

// The entries of one span (likewise; the span starts at entry `beg` of the list) subtracted from r one by one
// (src/gen/sampler.cpp:67-71).  Returns true and the entry's position in the list when the walk stops inside the span,
// else false and the new r.  One wave.
// The walk stops at the first entry with r < x, which is the first entry whose subtraction turns r negative (x != r
// gives a nonzero difference, denormals kept), and a negative r stays negative under every later subtraction of a
// weight.
__device__ __forceinline__ bool walk_lanes(const float (&x)[4], uint32_t n, uint32_t beg, float& r, uint32_t& pos)
{
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
        if (j * kWave < n) { // uniform
            const uint32_t m = min(n - j * kWave, (uint32_t)kWave);
            const float v = lane_chain<true>(r, x[j], m);
            const unsigned long long neg = __ballot((uint32_t)lane_id() < m && v < 0.0f);
            if (neg) {
                pos = beg + j * kWave + (uint32_t)__ffsll((long long)neg) - 1u;
                return true;
            }
            r = readlane_f32(v, m - 1u);
        }
    return false;
}

// ---- increments ----------------------------------------------------------------------------------------------------
//
// Inside one binade of the running value an addend that is no exact tie adds a multiple of the binade's last place U
// (seqfp.h's increment()); sums of such multiples are exact in fp32 up to 2^24 U, in any order, and anything beyond stays
// beyond.  So a span without ties is ONE float, its sum of multiples, the value behind it is S + that sum, and it is the
// sequential loop's value if (and only if) it still lies in the binade: additions never fall, so that nothing inside the
// span can have left a binade that its end lies in; and going down, a value that ends above R0 never was at or below R0
// on the way, nor was it below the next weight (it would have turned negative), so the walk cannot have stopped there.

// Inclusive sum over the lanes, for values whose sums are exact.
__device__ __forceinline__ float wave_scan_add_f32(float v)
{
#define MAKO_SCAN_ADD(CTRL, ROW_MASK) v += __uint_as_float(dpp_or_zero<CTRL, ROW_MASK>(__float_as_uint(v)));
    MAKO_SCAN_ADD(0x111, 0xf) // row_shr:1
    MAKO_SCAN_ADD(0x112, 0xf) // row_shr:2
    MAKO_SCAN_ADD(0x114, 0xf) // row_shr:4
    MAKO_SCAN_ADD(0x118, 0xf) // row_shr:8
    MAKO_SCAN_ADD(0x142, 0xa) // row_bcast:15 into rows 1 and 3
    MAKO_SCAN_ADD(0x143, 0xc) // row_bcast:31 into rows 2 and 3
#undef MAKO_SCAN_ADD
    return v;
}
// What one span (q: four consecutive entries per lane, 0.0f past its end) adds in the binade with exponent e, to a value
// whose last bit is even (x) and odd (y); the same for subtractions.  Different only where the span holds exact ties;
// INFINITY: no usable guess of the binade.  One wave.
__device__ __forceinline__ float2 span_incs(const float (&q)[4], int e)
{
    using namespace seqfp;
    if (e <= 0 || e > 200) // uniform (weights are at most 1: no sum of them gets near the upper bound)
        return make_float2(INFINITY, INFINITY);
    const float base = binade_base(e), half = half_ulp(e);
    float t[4];
    bool tie = false;
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        t[j] = increment(q[j], base);
        tie |= is_tie(q[j], t[j], half);
    }
    if (__ballot(tie) == 0ull) {
        const float all = readlane_f32(wave_scan_add_f32(((t[0] + t[1]) + t[2]) + t[3]), kWave - 1);
        return make_float2(all, all);
    }
    Step32 st = identity32(); // (ties: not the lowest binade)
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
        st = compose32(st, step32_fp(q[j], e));
    wave_scan_maps(st.d0, st.d1);
    const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)st.d0, kWave - 1);
    const uint32_t d1 = (uint32_t)__builtin_amdgcn_readlane((int)st.d1, kWave - 1);
    auto as_float = [e](uint32_t d) { return d < (1u << 24) ? __builtin_ldexpf((float)d, e - 150) : INFINITY; };
    return make_float2(as_float(d0), as_float(d1));
}

// A group's record into device memory (two 128-bit stores).
__device__ __forceinline__ void store_group_rec(GroupRec* rec, double sum, float2 inc, float2 walk, uint32_t start, uint32_t pack)
{
    static_assert(sizeof(GroupRec) == 32 && offsetof(GroupRec, inc) == 8 && offsetof(GroupRec, walk) == 16 && offsetof(GroupRec, pack) == 28, "");
    const unsigned long long b = (unsigned long long)__double_as_longlong(sum);
    const global_ptr<u32x4> p = (global_ptr<u32x4>)as_global(rec);
    p[0] = u32x4{(uint32_t)b, (uint32_t)(b >> 32), __float_as_uint(inc.x), __float_as_uint(inc.y)};
    p[1] = u32x4{__float_as_uint(walk.x), __float_as_uint(walk.y), start, pack};
}

// ---- replays -------------------------------------------------------------------------------------------------------

// Where a replay stands: all of the span applied, stopped in it (the walk), or to be gone on with entry by entry.
enum SpanEnd { kSpanDone = 0, kSpanStopped = 1, kSpanRest = 2 };

// The span's entries (q: four consecutive ones per lane, 0.0f past its end) added to S one by one, or, SUB, taken off it
// until S < entry (src/gen/sampler.cpp:80-82, :67-71).  One wave; S is the same in every lane.
// A round applies everything up to the first entry that leaves the binade or is an exact tie, and that entry with a real
// fp32 operation: a scan of the lanes' sums says where that is and what S is in front of it.  Sixty instructions a
// round, where going entry by entry takes 256 dependent ones; a span rarely takes more than two rounds.  After
// kSpanRounds the rest is left (kSpanRest, from entry `at` on).
constexpr uint32_t kSpanRounds = 4;
template <bool SUB>
__device__ __forceinline__ SpanEnd span_steps(float (&q_io)[4], float& S_io, uint32_t& at_io)
{
    const uint32_t i0 = (uint32_t)lane_id() * 4u;
    float q0 = q_io[0], q1 = q_io[1], q2 = q_io[2], q3 = q_io[3]; // (by name: an array picked from by an index would go to LDS)
    float S = S_io;
    uint32_t at = 0;
    SpanEnd end = kSpanDone;
    for (uint32_t round = 0;; ++round) {
        const uint32_t ex = uniform_u32((__float_as_uint(S) >> 23) & 0xffu);
        const int e = ex ? (int)ex : 1;
        const float base = seqfp::binade_base(e), top = seqfp::binade_top(e), low = seqfp::binade_low(e), half = seqfp::half_ulp(e);
        const float t0 = seqfp::increment(q0, base), t1 = seqfp::increment(q1, base), t2 = seqfp::increment(q2, base), t3 = seqfp::increment(q3, base);
        const float p1 = t0 + t1, p2 = p1 + t2, p3 = p2 + t3;
        const float incl = wave_scan_add_f32(p3);
        const float excl = __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(incl), 0x138 /* wave_shr:1 */, 0xf, 0xf, false));
        // S in front of the lane's entries and behind each of them (exact as far as the binade goes)
        const float before = SUB ? S - excl : S + excl;
        const float a0 = SUB ? before - t0 : before + t0, a1 = SUB ? before - p1 : before + p1;
        const float a2 = SUB ? before - p2 : before + p2, a3 = SUB ? before - p3 : before + p3;
        auto event = [&](float a, float q, float t) { return !(SUB ? a > low : a < top) || seqfp::is_tie(q, t, half); };
        const bool v0 = event(a0, q0, t0), v1 = event(a1, q1, t1), v2 = event(a2, q2, t2), v3 = event(a3, q3, t3);
        const unsigned long long bal = __ballot(v0 || v1 || v2 || v3);
        if (bal == 0ull) {
            S = readlane_f32(a3, kWave - 1);
            break;
        }
        if (round == kSpanRounds) {
            end = kSpanRest;
            break;
        }
        const uint32_t f = (uint32_t)__ffsll((long long)bal) - 1u;
        const uint32_t i_l = v0 ? i0 : (v1 ? i0 + 1u : (v2 ? i0 + 2u : i0 + 3u));
        const float b_l = v0 ? before : (v1 ? a0 : (v2 ? a1 : a2));
        const float q_l = v0 ? q0 : (v1 ? q1 : (v2 ? q2 : q3));
        const float b = readlane_f32(b_l, f), x = readlane_f32(q_l, f);
        at = (uint32_t)__builtin_amdgcn_readlane((int)i_l, (int)f);
        if (SUB && __ballot(b < x) != 0ull) {
            S = b;
            end = kSpanStopped;
            break;
        }
        S = SUB ? b - x : b + x;
        ++at;
        // (what has been applied is taken out)
        q0 = i0 < at ? 0.0f : q0;
        q1 = i0 + 1u < at ? 0.0f : q1;
        q2 = i0 + 2u < at ? 0.0f : q2;
        q3 = i0 + 3u < at ? 0.0f : q3;
    }
    q_io[0] = q0, q_io[1] = q1, q_io[2] = q2, q_io[3] = q3;
    S_io = S;
    at_io = at;
    return end;
}

// The walk over the first `n` entries of the list, staged in LDS as floats (16-byte aligned): every lane of the
// wave reads the same four entries with one broadcast load and subtracts them in turn, two nanoseconds an entry
// (lane_chain() takes five).  Blocks of 64 blind; the one it stops in, and what is left, by lane_chain().
// Returns true and the position when the walk stops, else false and the new r.
// (The list is read as LDS, not through the generic pointer: generic loads wait for one another in full, and the
// first subtraction of a block would wait for the block's last entry.)
typedef __attribute__((address_space(3))) const float LdsFloat;
typedef float LdsFloat4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ bool walk_lds(const float* sx_any, uint32_t n, float& r, uint32_t& pos)
{
    LdsFloat* sx = (LdsFloat*)sx_any;
    typedef const __attribute__((address_space(3))) LdsFloat4* Vec4Ptr;
    float v = r;
    uint32_t base = 0;
    // Blocks of 64 in two halves, each half's loads issued while the other half is subtracted (the scheduling
    // barriers keep the loads where they are written: the compiler would otherwise issue each only just before its
    // use, to save registers, and every fourth subtraction would wait for LDS).  The loads run up to 32 entries past
    // the block; the staged list has a wave's worth of room behind it.
    LdsFloat4 xa[8], xb[8];
    if (kWave <= n) {
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i)
            xa[i] = ((Vec4Ptr)sx)[i];
    }
    for (; base + kWave <= n; base += kWave) {
        Vec4Ptr p = (Vec4Ptr)(sx + base);
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i)
            xb[i] = p[8u + i];
        __builtin_amdgcn_sched_barrier(0);
        float t = v;
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            t -= xa[i].x;
            t -= xa[i].y;
            t -= xa[i].z;
            t -= xa[i].w;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i)
            xa[i] = p[16u + i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            t -= xb[i].x;
            t -= xb[i].y;
            t -= xb[i].z;
            t -= xb[i].w;
        }
        __builtin_amdgcn_sched_barrier(0);
        if (__ballot(t < 0.0f) != 0ull)
            break; // the walk stops in this block: found below
        v = t;
    }
    if (base < n) { // the block the walk stops in, or what is left
        const uint32_t m = min(n - base, (uint32_t)kWave);
        const float x = sx[base + (uint32_t)lane_id()];
        const float t = lane_chain<true>(v, (uint32_t)lane_id() < m ? x : 0.0f, m);
        const unsigned long long neg = __ballot((uint32_t)lane_id() < m && t < 0.0f);
        if (neg) {
            pos = base + (uint32_t)__ffsll((long long)neg) - 1u;
            return true;
        }
        v = readlane_f32(t, m - 1u);
    }
    r = v;
    return false;
}

// S plus the first `n` entries of a list staged in LDS as for walk_lds(), added one by one in fp32.
__device__ __forceinline__ float sum_lds(const float* sx_any, uint32_t n, float S)
{
    LdsFloat* sx = (LdsFloat*)sx_any;
    typedef const __attribute__((address_space(3))) LdsFloat4* Vec4Ptr;
    uint32_t base = 0;
    // (blocks of 64 in two halves, loads and additions interleaved as in walk_lds())
    LdsFloat4 xa[8], xb[8];
    if (kWave <= n) {
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i)
            xa[i] = ((Vec4Ptr)sx)[i];
    }
    for (; base + kWave <= n; base += kWave) {
        Vec4Ptr p = (Vec4Ptr)(sx + base);
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i)
            xb[i] = p[8u + i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            S += xa[i].x;
            S += xa[i].y;
            S += xa[i].z;
            S += xa[i].w;
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i)
            xa[i] = p[16u + i];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i) {
            S += xb[i].x;
            S += xb[i].y;
            S += xb[i].z;
            S += xb[i].w;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if (base < n) {
        const uint32_t m = min(n - base, (uint32_t)kWave);
        const float x = sx[base + (uint32_t)lane_id()];
        S = readlane_f32(lane_chain<false>(S, (uint32_t)lane_id() < m ? x : 0.0f, m), m - 1u);
    }
    return S;
}

// A group's entries in LDS (x: 256 floats, 16-byte aligned, 0.0f past the group's end, 64 more readable behind them)
// replayed: span_steps(), and what that leaves entry by entry.  SUB: returns true and the entry's number in the group
// where the walk stops (and may leave the entries changed).  One wave.
template <bool SUB>
__device__ __forceinline__ bool replay_group(float* x_any, uint32_t len, float& S, uint32_t& at)
{
    typedef __attribute__((address_space(3))) f32x4 LdsVec;
    const uint32_t lane = (uint32_t)lane_id();
    LdsVec* x = (LdsVec*)x_any;
    const f32x4 v = x[lane];
    float q[4] = {v.x, v.y, v.z, v.w};
    const SpanEnd end = span_steps<SUB>(q, S, at);
    if (end != kSpanRest) // uniform
        return end == kSpanStopped;
    const uint32_t from = at & ~3u;
    x[lane] = f32x4{q[0], q[1], q[2], q[3]}; // (zeros in front of entry `at`)
    __builtin_amdgcn_s_waitcnt(0xc07f);     // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    const uint32_t n = len - from;
    if (SUB) {
        uint32_t pos = 0;
        if (!walk_lds(x_any + from, n, S, pos))
            return false;
        at = from + pos;
        return true;
    }
    S = sum_lds(x_any + from, n, S);
    x[lane] = v; // (the walk may want the group again)
    return false;
}

// ---- the groups of a list, in LDS -----------------------------------------------------------------------------------

constexpr uint32_t kHeadStaged = 12;                     // groups at the head of a list that are kept in LDS
constexpr uint32_t kHeadLen = kHeadStaged * kGroup;
struct GroupLds { // carved from the dynamic LDS block once sorting is over
    unsigned char* base;
    // [kMaxGroups + 2] fp64 sum of the entries before each group
    __device__ __forceinline__ double* pg() const { return reinterpret_cast<double*>(base); }
    // [kMaxGroups] what the group adds in the binade guessed for it, and what it takes off r in the one guessed for that
    __device__ __forceinline__ float2* inc() const { return reinterpret_cast<float2*>(pg() + kMaxGroups + 2); }
    __device__ __forceinline__ float2* winc() const { return inc() + kMaxGroups; }
    __device__ __forceinline__ uint32_t* start() const { return reinterpret_cast<uint32_t*>(winc() + kMaxGroups); } // first entry
    __device__ __forceinline__ uint32_t* pack() const { return start() + kMaxGroups; } // as GroupRec::pack, and the slot + 1
    __device__ __forceinline__ uint32_t* misc() const { return pack() + kMaxGroups; }  // [16]
    __device__ __forceinline__ uint32_t* staged() const { return misc() + 16; }        // [64] the groups in the slots
    // [kMaxGroups] groups whose increment for the running sum is to be made, then [kMaxGroups] those for the walk
    __device__ __forceinline__ uint16_t* todo() const { return reinterpret_cast<uint16_t*>(staged() + 64); }
    // [kHeadLen + kWave] the first entries of the list
    __device__ __forceinline__ float* head() const { return reinterpret_cast<float*>(todo() + 2u * kMaxGroups); }
    // [kSlots][kGroup] entries of the groups that are expected to be replayed; the last slot is for any other
    __device__ __forceinline__ float* slot(uint32_t s) const { return head() + kHeadLen + kWave + s * kGroup; }
};
constexpr uint32_t kSlots = 39;
constexpr uint32_t kSlotShift = 26; // (of GroupLds::pack())
constexpr uint32_t kGroupLdsHead = (kMaxGroups + 2u) * 8u + kMaxGroups * (8u + 8u + 4u + 4u + 4u) + (16u + 64u) * 4u;
static_assert(kGroupLdsHead % 16u == 0 && kGroupLdsHead + (kHeadLen + kWave + kSlots * kGroup + kWave) * 4u <= kTailLds && kSlots < 64u,
              "the groups' records, the slots and what walk_lds() may read behind them fit the dynamic LDS block");

__device__ __forceinline__ GroupLds group_lds(const FinishLds& L)
{
    assume_lds(L);
    return GroupLds{reinterpret_cast<unsigned char*>(L.sortk)};
}

// The group of a rejected draft during its redraw, and the draft's number in it: that entry counts as 0.0f.
struct LeftOut {
    uint32_t group = kNone, entry = 0;
};

// One group's entries into a slot, by one wave.
template <typename Keys>
__device__ __forceinline__ void stage_group(Keys kf, const GroupLds G, uint32_t g, uint32_t s, const LeftOut out)
{
    float q[4];
    load_span(kf, uniform_u32(G.start()[g]), uniform_u32(G.pack()[g]) & kLenMask, q);
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j)
        q[j] = (g == out.group && (uint32_t)lane_id() * 4u + j == out.entry) ? 0.0f : q[j];
    *(reinterpret_cast<float4*>(G.slot(s)) + lane_id()) = make_float4(q[0], q[1], q[2], q[3]);
}

// Is group g expected to be replayed: by the running sum (its binade changes in it), or by the walk from r0 (likewise, or
// it ends there)?
__device__ __forceinline__ bool sum_changes_binade(const GroupLds G, uint32_t g)
{
    return g == 0u || exponent_of((float)G.pg()[g]) != exponent_of((float)G.pg()[g + 1u]);
}
__device__ __forceinline__ bool walk_changes_binade(const GroupLds G, uint32_t g, double r0)
{
    const double b = r0 - G.pg()[g], a = r0 - G.pg()[g + 1u];
    return b > 0.0 && (!(a > 0.0) || exponent_of((float)b) != exponent_of((float)a));
}

// Which groups are expected to be replayed (their entries go to the slots), and which others lack an increment for the
// binade expected now: thread g decides for group g, of those from `from` on; `sum`, `walk`: for which of the two, the
// latter from r0 (the sum's first `lead` groups need neither).  (All threads call, the caller's barriers around it.)  A group
// that is expected to be replayed anyway, and one the walk is not expected to reach, gets no increment.  G.misc()[3] counts the
// slots, G.misc()[7] and [8] the increments to be made, the sum's and the walk's.
template <bool UNSORTED>
__device__ __forceinline__ void plan_groups(const GroupLds G, uint32_t lead, uint32_t from, uint32_t groups, bool sum, bool walk, double r0, const LeftOut out)
{
    const uint32_t g = threadIdx.x;
    const uint32_t pk = G.pack()[min(g, groups - 1u)];
    if (g < from || g >= groups || (UNSORTED && (pk & kOpaque)))
        return;
    const bool replay_s = sum && g >= lead && sum_changes_binade(G, g), replay_w = walk && walk_changes_binade(G, g, r0);
    if (replay_s || replay_w) {
        const uint32_t s = atomicAdd(&G.misc()[3], 1u);
        if (s < kSlots - 1u) {
            G.staged()[s] = g;
            G.pack()[g] = pk | ((s + 1u) << kSlotShift);
        }
    }
    const double b = G.pg()[g];
    if (sum && g >= lead && !replay_s && ((pk >> kSumExpShift) & 0xffu) != (uint32_t)exponent_of((float)b))
        G.todo()[atomicAdd(&G.misc()[7], 1u)] = (uint16_t)g;
    // (at r = 0 too: the walk passes what weighs nothing there, in a row whose first candidates are behind a masked stretch)
    if (walk && !replay_w && r0 - b >= 0.0 && g != out.group && ((pk >> kWalkExpShift) & 0xffu) != (uint32_t)exponent_of((float)(r0 - b)))
        G.todo()[kMaxGroups + atomicAdd(&G.misc()[8], 1u)] = (uint16_t)g;
}
template <typename Keys>
__device__ __forceinline__ void fill_staged(Keys kf, const GroupLds G, const LeftOut out = LeftOut{})
{
    const uint32_t n = min(uniform_u32(G.misc()[3]), kSlots - 1u);
    for (uint32_t s = (uint32_t)wave_id(); s < n; s += (uint32_t)kWaves)
        stage_group(kf, G, uniform_u32(G.staged()[s]), s, out);
}

// The increments to be made: the running sum's, the walk's.  The calling wave is number `part` of `parts` that share the work; up
// to four groups per trip to memory.
// Never beside the chain that uses them: an increment and the binade it is for (in pack()) are two words, and a chain beside the
// writer could find the old binade with the new increment.  That binade may be the running value's own, where the fp64 sums
// that the guesses come from lie on the other side of a power of two.
template <typename Keys>
__device__ __forceinline__ void build_incs(Keys kf, double r0, const GroupLds G, bool sum, bool walk, uint32_t part, uint32_t parts)
{
    const uint32_t n_sum = sum ? uniform_u32(G.misc()[7]) : 0u, n = n_sum + (walk ? uniform_u32(G.misc()[8]) : 0u);
    for (uint32_t i0 = part; i0 < n; i0 += parts * 4u) {
        float q[4][4];
        uint32_t item[4];
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            const uint32_t i = min(i0 + u * parts, n - 1u);
            item[u] = uniform_u32(G.todo()[i < n_sum ? i : kMaxGroups + (i - n_sum)]);
            load_span(kf, uniform_u32(G.start()[item[u]]), i0 + u * parts < n ? uniform_u32(G.pack()[item[u]]) & kLenMask : 0u, q[u]);
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) {
            if (i0 + u * parts >= n) // uniform
                break;
            const uint32_t g = item[u];
            const bool for_sum = i0 + u * parts < n_sum;
            const double b = G.pg()[g];
            const uint32_t e = uniform_u32((uint32_t)exponent_of((float)(for_sum ? b : r0 - b)));
            const float2 inc = span_incs(q[u], (int)e);
            if (lane_id() == 0) {
                const uint32_t shift = for_sum ? kSumExpShift : kWalkExpShift;
                (for_sum ? G.inc() : G.winc())[g] = inc;
                atomicAnd(&G.pack()[g], ~(0xffu << shift)); // (another wave may be at work on the other one)
                atomicOr(&G.pack()[g], e << shift);
            }
        }
    }
}

// Entries of group g for a replay: from its slot, or fetched into the last one.  Wave 0's chains call it.
template <typename Keys>
__device__ __forceinline__ float* replay_entries(Keys kf, const GroupLds G, uint32_t g, uint32_t pk, const LeftOut out)
{
    const uint32_t s = pk >> kSlotShift;
    if (s)
        return G.slot(s - 1u);
    stage_group(kf, G, g, kSlots - 1u, out);
    __builtin_amdgcn_s_waitcnt(0xc07f); // lgkmcnt(0)
    __builtin_amdgcn_wave_barrier();
    return G.slot(kSlots - 1u);
}

// The running fp32 sum over all groups, from 0.0f (src/gen/sampler.cpp:80-82).  One wave.  The first `lead` groups (their
// lead_n entries), where the sum changes binade every few entries, from the staged head one by one; then 64 groups at a time, one per
// lane: a scan of the increments says how far the sum stays in its binade; the first group that leaves it (or whose
// increments are for another binade) is replayed, and the scan goes on behind it.  A group with exact ties has two
// increments and is taken on its own.  Returns false (UNSORTED) when a share that was left unsorted would have to be
// replayed.
template <bool UNSORTED, typename Keys>
__device__ __forceinline__ bool chain_sum(Keys kf, const GroupLds G, uint32_t groups, uint32_t lead, uint32_t lead_n, float& S_out)
{
    const uint32_t lane = (uint32_t)lane_id();
    float S = sum_lds(G.head(), lead_n, 0.0f);
    for (uint32_t base = 0; base < groups; base += (uint32_t)kWave) {
        const uint32_t gl = min(base + lane, groups - 1u);
        const uint32_t pk_l = G.pack()[gl];
        const float2 inc_l = G.inc()[gl];
        const uint32_t cnt = min((uint32_t)kWave, groups - base);
        uint32_t done = base == 0u ? lead : 0u;
        while (done < cnt) {
            const uint32_t ex = uniform_u32((__float_as_uint(S) >> 23) & 0xffu), e = ex ? ex : 1u;
            const float top = seqfp::binade_top((int)e);
            const bool plain = ((pk_l >> kSumExpShift) & 0xffu) == e && inc_l.x == inc_l.y;
            const float after = S + wave_scan_add_f32(lane < done ? 0.0f : (plain ? inc_l.x : INFINITY));
            const unsigned long long bad = __ballot(lane >= done && lane < cnt && !(after < top));
            const uint32_t f = bad ? (uint32_t)__ffsll((long long)bad) - 1u : cnt;
            if (f > done)
                S = readlane_f32(after, f - 1u);
            if (f >= cnt)
                break;
            done = f + 1u;
            const uint32_t pk = (uint32_t)__builtin_amdgcn_readlane((int)pk_l, (int)f);
            if (((pk >> kSumExpShift) & 0xffu) == e) { // (exact ties in it, or the binade ends)
                const float behind = S + ((__float_as_uint(S) & 1u) ? readlane_f32(inc_l.y, f) : readlane_f32(inc_l.x, f));
                if (__ballot(behind < top) != 0ull) {
                    S = behind;
                    continue;
                }
            }
            if (UNSORTED && (pk & kOpaque))
                return false;
            uint32_t at = 0;
            replay_group<false>(replay_entries(kf, G, base + f, pk, LeftOut{}), pk & kLenMask, S, at);
            S = uniform_f32(S);
        }
    }
    S_out = S;
    return true;
}

// The walk over the groups from `first` on, from r (src/gen/sampler.cpp:67-71).  One wave; the same way.  Returns
// kWalkEnd when the list ends first, kWalkStopped (and the position in the list), kWalkGaveUp (UNSORTED) as above, or
// kWalkRebuild when the increments ahead are for other binades than r turns out to be in (`first` and r are then where it
// stands): r close to the walk's end is a small difference of large numbers, and what was guessed for it worth little.
enum WalkEnd { kWalkEnd = 0, kWalkStopped = 1, kWalkGaveUp = 2, kWalkRebuild = 3 };
constexpr uint32_t kWalkStray = 4; // groups replayed for a wrong guess before the increments ahead are made again
template <bool UNSORTED, typename Keys>
__device__ __forceinline__ WalkEnd chain_walk(Keys kf, const GroupLds G, uint32_t groups, uint32_t& first, float& r, uint32_t& pos,
                                              const LeftOut out)
{
    const uint32_t lane = (uint32_t)lane_id();
    uint32_t stray = 0;
    while (first < groups) {
        const uint32_t base = first;
        const uint32_t gl = min(base + lane, groups - 1u);
        const uint32_t pk_l = G.pack()[gl];
        const float2 inc_l = G.winc()[gl];
        const uint32_t cnt = min((uint32_t)kWave, groups - base);
        uint32_t done = 0;
        while (done < cnt) {
            const uint32_t ex = uniform_u32((__float_as_uint(r) >> 23) & 0xffu), e = ex ? ex : 1u;
            const float low = seqfp::binade_low((int)e);
            const bool plain = ((pk_l >> kWalkExpShift) & 0xffu) == e && inc_l.x == inc_l.y;
            const float after = r - wave_scan_add_f32(lane < done ? 0.0f : (plain ? inc_l.x : INFINITY));
            const unsigned long long bad = __ballot(lane >= done && lane < cnt && !(after > low));
            const uint32_t f = bad ? (uint32_t)__ffsll((long long)bad) - 1u : cnt;
            if (f > done)
                r = readlane_f32(after, f - 1u);
            if (f >= cnt)
                break;
            done = f + 1u;
            const uint32_t pk = (uint32_t)__builtin_amdgcn_readlane((int)pk_l, (int)f);
            const bool for_here = ((pk >> kWalkExpShift) & 0xffu) == e;
            if (for_here) {
                const float behind = r - ((__float_as_uint(r) & 1u) ? readlane_f32(inc_l.y, f) : readlane_f32(inc_l.x, f));
                if (__ballot(behind > low) != 0ull) {
                    r = behind;
                    continue;
                }
            }
            if (UNSORTED && (pk & kOpaque))
                return kWalkGaveUp;
            const uint32_t g = base + f;
            if (!for_here && (pk >> kSlotShift) == 0u && ++stray > kWalkStray) {
                first = g;
                return kWalkRebuild;
            }
            uint32_t at = 0;
            if (replay_group<true>(replay_entries(kf, G, g, pk, out), pk & kLenMask, r, at)) {
                pos = (uint32_t)__builtin_amdgcn_readlane((int)G.start()[gl], (int)f) + at;
                return kWalkStopped;
            }
            r = uniform_f32(r);
        }
        first = base + cnt;
    }
    return kWalkEnd;
}

} // namespace mako
