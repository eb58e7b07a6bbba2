// The kernels' expf (mako_amd/csrc/exp_form.h) against the oracle's, all 2^32 arguments.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <thread>
#include <vector>

#include "../../mako_amd/csrc/exp_form.h"

extern "C" float or_expf(float);

static uint64_t tab[32]; // as the kernels' source has it, one entry per argument of the program

static uint64_t differing(uint64_t lo, uint64_t hi)
{
    uint64_t n = 0;
    for (uint64_t u = lo; u < hi; ++u) {
        const uint32_t bits = (uint32_t)u;
        float x;
        std::memcpy(&x, &bits, 4);
        if (x != x)
            continue;
        const float a = mako::exp_form(x < mako::kExpLow ? mako::kExpLow : (x > mako::kExpHigh ? mako::kExpHigh : x), tab), b = or_expf(x);
        n += std::memcmp(&a, &b, 4) != 0;
    }
    return n;
}

int main(int argc, char** argv)
{
    if (argc != 33)
        return 2;
    for (int i = 0; i < 32; ++i) {
        unsigned long v;
        if (std::sscanf(argv[1 + i], "%lx", &v) != 1)
            return 2;
        tab[i] = v;
    }
    constexpr uint64_t kThreads = 8, kPer = (1ull << 32) / kThreads;
    std::vector<uint64_t> n(kThreads);
    std::vector<std::thread> pool;
    for (uint64_t t = 0; t < kThreads; ++t)
        pool.emplace_back([&n, t] { n[t] = differing(t * kPer, (t + 1) * kPer); });
    uint64_t all = 0;
    for (uint64_t t = 0; t < kThreads; ++t) {
        pool[t].join();
        all += n[t];
    }
    std::printf("differ %llu\n", (unsigned long long)all);
    return all != 0;
}
