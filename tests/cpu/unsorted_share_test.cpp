// Host restatement of opaque_share() (mako_amd/csrc/worker_sort.h), the record that stands for a share of a sorted
// list that was never sorted: inside one binade of the running fp32 sum the addends that are no exact ties add constant
// multiples of its last place and commute, so the multiples' SUM, a float, is what they add whatever their order; the exact
// ties are kept apart, ordered by weight, and each one's own step is composed in between the sums of the weights on either
// side of it.  The arithmetic is the kernels' (seqfp.h), lane by lane.
//
// Checked against what the reference does (src/gen/sampler.cpp:80-82, :67-71): the weights sorted descending, added to
// (subtracted from) a running float one by one with real fp32 operations.  Whenever the record passes the test under
// which the chains of group_chain.h apply it (the binade is the one it is for, and the value behind it is still inside), that
// value must be the sequential loop's, bit for bit, and the walk must not have stopped inside the share; every binade, shares
// with up to a dozen exact ties, duplicated weights, multiples of zero and weights from higher binades are among the cases.
//
//   g++ -O2 -std=c++17 -ffp-contract=off -I ../../mako_amd/csrc unsorted_share_test.cpp -o unsorted_share_test
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "seqfp.h"

using namespace seqfp;

constexpr uint32_t kWave = 64, kOpaqueTies = 16;

struct Incs {
    float x, y;
};

// The lanes' sums over the wave.  (Below the binade's top any order of addition is exact; whatever the order, what is not
// below it stays so.)
static float over_lanes(const float (&acc)[kWave])
{
    float all = 0.0f;
    for (float v : acc)
        all += v;
    return all;
}

// share_incs(): what the share adds to a value of the binade with exponent e whose last bit is even and odd.
static Incs share_incs(const std::vector<float>& q, int e, uint32_t& n_ties)
{
    const float base = binade_base(e), half = half_ulp(e);
    std::vector<uint32_t> ties;
    float acc[kWave] = {};
    for (size_t i = 0; i < q.size(); ++i) {
        const float t = increment(q[i], base);
        if (is_tie(q[i], t, half))
            ties.push_back(f2u(q[i]));
        else
            acc[i % kWave] += t;
    }
    n_ties = (uint32_t)ties.size();
    if (n_ties > kOpaqueTies)
        return {INFINITY, INFINITY};
    const float all = over_lanes(acc);
    const uint32_t units = all < binade_top(e) ? (uint32_t)ldexpf(all, 150 - e) : kSat;
    if (n_ties == 0)
        return {all, all};
    std::sort(ties.begin(), ties.end(), std::greater<uint32_t>());
    Step32 v = identity32();
    uint32_t taken = 0;
    for (size_t k = 0; k < ties.size() && units != kSat; ++k) {
        float part[kWave] = {};
        for (size_t i = 0; i < q.size(); ++i) {
            const float t = increment(q[i], base);
            if (f2u(q[i]) > ties[k] && !is_tie(q[i], t, half))
                part[i % kWave] += t;
        }
        const uint32_t above = (uint32_t)ldexpf(over_lanes(part), 150 - e);
        v = compose32(v, Step32{above - taken, above - taken});
        v = compose32(v, step32_flat(u2f(ties[k]), e));
        taken = above;
    }
    const uint32_t rest = units == kSat ? kSat : units - taken;
    v = compose32(v, Step32{rest, rest});
    auto as_float = [e](uint32_t d) { return d < (1u << 24) ? ldexpf((float)d, e - 150) : INFINITY; };
    return {as_float(v.d0), as_float(v.d1)};
}

int main()
{
    std::mt19937_64 rng(20261125);
    long cases = 0, applied_add = 0, applied_sub = 0, with_ties = 0, applied_ties = 0, failures = 0;
    for (int rep = 0; rep < 60000; ++rep) {
        // the running value: a float in a random binade (the lowest ones often), and a share of weights some binades below it
        const int e = rep % 5 == 0 ? 1 + (int)(rng() % 30) : 40 + (int)(rng() % 150);
        const uint32_t M = e == 1 && rng() % 2 ? (uint32_t)(rng() & 0x7fffffu) : (1u << 23) | (uint32_t)(rng() & 0x7fffffu);
        const int shift_lo = (int)(rng() % 14), shift_hi = shift_lo + 1 + (int)(rng() % 6);
        const size_t n = 1 + rng() % (rep % 7 == 0 ? 3000 : 200);
        // (few mantissa bits: exact ties and duplicates become common)
        const int keep_bits = rep % 3 == 0 ? 24 : 1 + (int)(rng() % 12);
        std::vector<float> q(n);
        for (auto& x : q) {
            const int ex = e - shift_lo - (int)(rng() % (uint32_t)(shift_hi - shift_lo + 1));
            uint32_t m = (uint32_t)(rng() & 0x7fffffu);
            m &= ~((1u << (24 - keep_bits)) - 1u) & 0x7fffffu;
            x = ex >= 1 ? u2f(((uint32_t)ex << 23) | m) : u2f((0x800000u | m) >> std::min(1 - ex, 24));
        }
        if (rep % 50 == 0)
            q[rng() % n] = u2f(((uint32_t)(e + 1) << 23) | 5u); // a weight from a higher binade
        std::vector<float> sorted = q;
        std::sort(sorted.begin(), sorted.end(), std::greater<float>());
        std::shuffle(q.begin(), q.end(), rng);
        ++cases;

        uint32_t n_ties = 0;
        const Incs inc = share_incs(q, e, n_ties);
        with_ties += n_ties != 0;
        const float start = join(M, e), by = (f2u(start) & 1u) ? inc.y : inc.x;
        // the running sum
        if (start + by < binade_top(e)) {
            float S = start;
            for (float x : sorted)
                S += x;
            if (f2u(S) != f2u(start + by)) {
                ++failures;
                printf("FAIL add: rep %d n %zu e %d M %u ties %u: %a vs %a\n", rep, n, e, M, n_ties, S, start + by);
            }
            ++applied_add;
            applied_ties += n_ties != 0;
        }
        // the walk
        if (start - by > binade_low(e)) {
            float r = start;
            bool stopped = false;
            for (float x : sorted) {
                if (r < x) {
                    stopped = true;
                    break;
                }
                r -= x;
            }
            if (stopped || f2u(r) != f2u(start - by)) {
                ++failures;
                printf("FAIL sub: rep %d n %zu e %d M %u ties %u stopped %d: %a vs %a\n", rep, n, e, M, n_ties, (int)stopped, r, start - by);
            }
            ++applied_sub;
        }
    }
    printf("%ld shares (%ld with exact ties): record applied to %ld running sums (%ld of them with ties) and %ld walks: %ld failures\n",
           cases, with_ties, applied_add, applied_ties, applied_sub, failures);
    // (the test is worth nothing if the records hardly ever pass the tests)
    if (applied_add < cases / 4 || applied_sub < cases / 8 || applied_ties < cases / 50) {
        printf("too few applications for the test to mean anything\n");
        return 1;
    }
    return failures ? 1 : 0;
}
