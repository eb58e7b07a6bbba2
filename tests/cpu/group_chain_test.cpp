// Host restatement of the kernels' chains over groups of 256 weights (mako_amd/csrc/group_chain.h), lane by lane, on the
// arithmetic the two share (seqfp.h): what a span adds in a binade as one number (span_incs), the replay of a span that leaves
// its binade (span_steps), the running sum and the walk over 64 groups at a time (chain_sum, chain_walk).  Compared with what
// the reference does (src/gen/sampler.cpp:80-82, :67-71), real fp32 operations one by one: sums and r bit for bit, the
// walk's stop, over every binade the lowest included, ties, duplicates, zeros, and binades guessed right and wrong.
//
//   g++ -O2 -std=c++17 -ffp-contract=off -I ../../mako_amd/csrc group_chain_test.cpp -o group_chain_test
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "seqfp.h"

using namespace seqfp;

constexpr uint32_t kWave = 64, kGroup = 256, kSpanRounds = 4;

struct Lanes {
    float v[kWave];
};
// wave_scan_add_f32(): the steps of the wave's scan in their order
static Lanes scan_add(Lanes a)
{
    for (uint32_t s : {1u, 2u, 4u, 8u}) {
        const Lanes b = a;
        for (uint32_t l = 0; l < kWave; ++l)
            a.v[l] = b.v[l] + ((l & 15u) >= s ? b.v[l - s] : 0.0f);
    }
    for (uint32_t l = 0; l < kWave; ++l)
        if ((l >> 4) & 1u)
            a.v[l] += a.v[(l & ~15u) - 1u];
    for (uint32_t l = 32; l < kWave; ++l)
        a.v[l] += a.v[31];
    return a;
}
static int exponent_of(float x)
{
    uint32_t M;
    int e;
    split(x, M, e);
    return e;
}

struct Incs {
    float x, y;
};
// span_incs(): q holds 256 entries, 0.0f past the span's end
static Incs span_incs(const float* q, int e)
{
    if (e <= 0 || e > 200)
        return {INFINITY, INFINITY};
    const float base = binade_base(e), half = half_ulp(e);
    bool tie = false;
    Lanes sum;
    for (uint32_t l = 0; l < kWave; ++l) {
        float t[4];
        for (uint32_t j = 0; j < 4; ++j) {
            t[j] = increment(q[4 * l + j], base);
            tie |= is_tie(q[4 * l + j], t[j], half);
        }
        sum.v[l] = ((t[0] + t[1]) + t[2]) + t[3];
    }
    if (!tie) {
        const float all = scan_add(sum).v[kWave - 1];
        return {all, all};
    }
    Step32 st = identity32();
    for (uint32_t i = 0; i < kGroup; ++i)
        st = compose32(st, step32_fp(q[i], e));
    auto as_float = [e](uint32_t d) { return d < (1u << 24) ? ldexpf((float)d, e - 150) : INFINITY; };
    return {as_float(st.d0), as_float(st.d1)};
}

// span_steps() and what it leaves, entry by entry; returns true and the entry where the walk stops
template <bool SUB>
static bool replay(const float* q_in, uint32_t len, float& S, uint32_t& at, long& rounds_taken)
{
    float q[kGroup];
    std::copy(q_in, q_in + kGroup, q);
    for (uint32_t round = 0;; ++round) {
        const int e = exponent_of(S);
        const float base = binade_base(e), top = binade_top(e), low = binade_low(e), half = half_ulp(e);
        float t[kGroup];
        Lanes p3;
        for (uint32_t l = 0; l < kWave; ++l) {
            for (uint32_t j = 0; j < 4; ++j)
                t[4 * l + j] = increment(q[4 * l + j], base);
            p3.v[l] = ((t[4 * l] + t[4 * l + 1]) + t[4 * l + 2]) + t[4 * l + 3];
        }
        const Lanes incl = scan_add(p3);
        uint32_t first = kGroup;
        float b = 0.0f, last = 0.0f;
        for (uint32_t l = 0; l < kWave && first == kGroup; ++l) {
            const float excl = l ? incl.v[l - 1] : 0.0f, before = SUB ? S - excl : S + excl;
            float p = 0.0f, prev = before;
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t i = 4 * l + j;
                p = j ? p + t[i] : t[i];
                const float a = SUB ? before - p : before + p;
                if (!(SUB ? a > low : a < top) || is_tie(q[i], t[i], half)) {
                    first = i;
                    b = prev;
                    break;
                }
                prev = last = a;
            }
        }
        if (first == kGroup) {
            S = last;
            return false;
        }
        if (round == kSpanRounds)
            break;
        ++rounds_taken;
        if (SUB && b < q[first]) {
            S = b;
            at = first;
            return true;
        }
        S = SUB ? b - q[first] : b + q[first];
        std::fill(q, q + first + 1, 0.0f);
    }
    for (uint32_t i = 0; i < len; ++i) {
        if (SUB && S < q[i]) {
            at = i;
            return true;
        }
        S = SUB ? S - q[i] : S + q[i];
    }
    return false;
}

struct Group {
    float q[kGroup];
    uint32_t start, len;
    int e_sum, e_walk; // the guesses
    Incs inc, walk;
};

struct Count {
    long groups = 0, replays = 0, rounds = 0, lowest = 0;
};

static float chain_sum(const std::vector<Group>& g, float S, Count& n)
{
    for (size_t base = 0; base < g.size(); base += kWave) {
        const uint32_t cnt = (uint32_t)std::min<size_t>(kWave, g.size() - base);
        uint32_t done = 0;
        while (done < cnt) {
            const int e = exponent_of(S);
            const float top = binade_top(e);
            Lanes x;
            for (uint32_t l = 0; l < kWave; ++l) {
                const Group& m = g[std::min(base + l, g.size() - 1)];
                x.v[l] = l < done ? 0.0f : (m.e_sum == e && m.inc.x == m.inc.y ? m.inc.x : INFINITY);
            }
            const Lanes sc = scan_add(x);
            uint32_t f = done;
            while (f < cnt && S + sc.v[f] < top)
                ++f;
            n.groups += f - done;
            n.lowest += e == 1 ? f - done : 0;
            if (f > done)
                S = S + sc.v[f - 1];
            if (f >= cnt)
                break;
            done = f + 1;
            const Group& m = g[base + f];
            if (m.e_sum == e) {
                const float behind = S + ((f2u(S) & 1u) ? m.inc.y : m.inc.x);
                if (behind < top) {
                    S = behind;
                    ++n.groups;
                    continue;
                }
            }
            uint32_t at = 0;
            ++n.replays;
            replay<false>(m.q, m.len, S, at, n.rounds);
        }
    }
    return S;
}

static bool chain_walk(const std::vector<Group>& g, float& r, size_t& pos, Count& n)
{
    for (size_t base = 0; base < g.size(); base += kWave) {
        const uint32_t cnt = (uint32_t)std::min<size_t>(kWave, g.size() - base);
        uint32_t done = 0;
        while (done < cnt) {
            const int e = exponent_of(r);
            const float low = binade_low(e);
            Lanes x;
            for (uint32_t l = 0; l < kWave; ++l) {
                const Group& m = g[std::min(base + l, g.size() - 1)];
                x.v[l] = l < done ? 0.0f : (m.e_walk == e && m.walk.x == m.walk.y ? m.walk.x : INFINITY);
            }
            const Lanes sc = scan_add(x);
            uint32_t f = done;
            while (f < cnt && r - sc.v[f] > low)
                ++f;
            n.groups += f - done;
            n.lowest += e == 1 ? f - done : 0;
            if (f > done)
                r = r - sc.v[f - 1];
            if (f >= cnt)
                break;
            done = f + 1;
            const Group& m = g[base + f];
            if (m.e_walk == e) {
                const float behind = r - ((f2u(r) & 1u) ? m.walk.y : m.walk.x);
                if (behind > low) {
                    r = behind;
                    ++n.groups;
                    continue;
                }
            }
            uint32_t at = 0;
            ++n.replays;
            if (replay<true>(m.q, m.len, r, at, n.rounds)) {
                pos = m.start + at;
                return true;
            }
        }
    }
    return false;
}

static std::vector<Group> cut(const std::vector<float>& q, float S0, float r0, std::mt19937_64& rng, int wrong)
{
    std::vector<Group> out((q.size() + kGroup - 1) / kGroup);
    double before = 0.0;
    for (size_t k = 0; k < out.size(); ++k) {
        Group& g = out[k];
        g.start = (uint32_t)(k * kGroup);
        g.len = (uint32_t)std::min<size_t>(kGroup, q.size() - g.start);
        std::fill(g.q, g.q + kGroup, 0.0f);
        std::copy(q.begin() + g.start, q.begin() + g.start + g.len, g.q);
        g.e_sum = exponent_of((float)(S0 + before));
        const double rb = (double)r0 - before;
        g.e_walk = rb >= 0.0 ? exponent_of((float)rb) : 0;
        if (wrong && rng() % 8 == 0) { // (a guess a binade off, or none: costs a replay, never the result)
            g.e_sum = std::max(0, g.e_sum + (int)(rng() % 3) - 1);
            g.e_walk = std::max(0, g.e_walk + (int)(rng() % 3) - 1);
        }
        g.inc = span_incs(g.q, g.e_sum);
        g.walk = span_incs(g.q, g.e_walk);
        for (uint32_t i = 0; i < g.len; ++i)
            before += (double)g.q[i];
    }
    return out;
}

static long check(const std::vector<float>& q, float S0, float r0, std::mt19937_64& rng, int wrong, const char* what, Count& n)
{
    const std::vector<Group> g = cut(q, S0, r0, rng, wrong);
    long bad = 0;
    float S = S0;
    for (float x : q)
        S += x;
    const float got = chain_sum(g, S0, n);
    if (f2u(S) != f2u(got)) {
        ++bad;
        std::printf("FAIL sum (%s): n %zu S0 %a want %a got %a\n", what, q.size(), S0, S, got);
    }
    float r = r0, rg = r0;
    size_t stop = 0, pos = 0;
    bool stopped = false;
    for (; stop < q.size(); ++stop) {
        if (r < q[stop]) {
            stopped = true;
            break;
        }
        r -= q[stop];
    }
    const bool got_stop = chain_walk(g, rg, pos, n);
    if (got_stop != stopped || (stopped ? pos != stop : f2u(r) != f2u(rg))) {
        ++bad;
        std::printf("FAIL walk (%s): n %zu r0 %a want %d %zu %a got %d %zu %a\n", what, q.size(), r0, stopped, stop, r, got_stop, pos, rg);
    }
    return bad;
}

int main()
{
    std::mt19937_64 rng(20261202);
    long cases = 0, failures = 0;
    Count n;
    { // a weight of the lowest binade's upper half in front of a heavy last one, and an r one last place below it
        std::vector<float> q(129280, 0.0f);
        q[5000] = 0x1.01b1bap-126f;
        q.back() = 1.0f;
        for (float r0 : {0x1.01b1b8p-126f, 0x1.01b1bap-126f, 0x1.01b1bcp-126f, 0x1.fffffep-126f, 0x1p-126f, 0x1p-149f, 0.0f}) {
            ++cases;
            failures += check(q, 0.0f, r0, rng, 0, "lowest binade", n);
        }
    }
    for (int rep = 0; rep < 24000; ++rep) {
        // the binade the running value starts near: the lowest ones often, or any
        const int e = rep % 2 ? 1 + (int)(rng() % 6) : 1 + (int)(rng() % 150);
        const int keep_bits = rep % 3 == 0 ? 24 : 1 + (int)(rng() % 24); // (few significant bits: ties and duplicates)
        const int below = (int)(rng() % (rep % 4 == 1 ? 3 : 27)), width = 1 + (int)(rng() % 4);
        const size_t len = 1 + rng() % (rep % 40 == 0 ? 40000 : 1500);
        std::vector<float> q(len);
        for (auto& x : q) {
            const int ex = e + 1 - below - (int)(rng() % (uint32_t)width);
            uint32_t m = (uint32_t)(rng() & 0x7fffffu) & ~((1u << (24 - keep_bits)) - 1u);
            if (ex < 1)
                x = u2f((0x800000u | m) >> std::min(1 - ex, 24));
            else
                x = u2f(((uint32_t)std::min(ex, 190) << 23) | m);
            if (rng() % 16 == 0)
                x = 0.0f;
        }
        if (rep % 5 == 0)
            std::fill(q.begin(), q.begin() + (long)(rng() % len), 0.0f);
        if (rep % 7 == 0)
            std::sort(q.begin(), q.end(), std::greater<float>());
        double mass = 0.0;
        for (float x : q)
            mass += (double)x;
        float S0 = u2f(((uint32_t)e << 23) | (uint32_t)(rng() & 0x7fffffu));
        if (rep % 4 == 1)
            S0 = 0.0f;
        if (rep % 4 == 2)
            S0 = u2f((uint32_t)(rng() & 0xffffffu)); // the lowest binade
        float r0 = rep % 4 == 3 ? S0 : (float)(mass * ((double)(rng() % 1001) / 1000.0));
        if (rep % 11 == 0)
            r0 = u2f((uint32_t)(rng() & 0xffffffu));
        if (rep % 13 == 0)
            r0 = 0.0f;
        ++cases;
        failures += check(q, S0, r0, rng, rep % 2, "random", n);
    }
    std::printf("%ld lists: %ld groups by their increments (%ld of them in the lowest binade), %ld replayed (%ld rounds): %ld failures\n", cases,
                n.groups, n.lowest, n.replays, n.rounds, failures);
    // (worth nothing if the increments hardly ever apply)
    if (n.groups < n.replays || n.lowest < 1000) {
        std::printf("too few groups by their increments for the test to mean anything\n");
        return 1;
    }
    return failures ? 1 : 0;
}
