// mako_amd/csrc/host_stage.h over a link whose copies read the staging memory as late as they may: only when they are waited
// for.  Whatever is put must be in the block then, rows apart from each other and staging memory used many times over
// included; and behind a copy that fails none may be left that would read what the next call writes.
//
//   g++ -O2 -std=c++17 -I ../../mako_amd/csrc host_stage_test.cpp -o host_stage_test
#include <cstdio>
#include <random>
#include <vector>

#include "host_stage.h"

struct Wire {
    struct Copy {
        size_t to, bytes;
        const void* from;
    };
    std::vector<unsigned char> block;
    std::vector<Copy> pending;
    int copies = 0, fail_at = -1;
};
struct LateLink {
    Wire* w;
    int copy(size_t to, const void* from, size_t bytes)
    {
        if (w->copies++ == w->fail_at)
            return 2;
        w->pending.push_back({to, bytes, from});
        return 0;
    }
    int wait()
    {
        for (const Wire::Copy& c : w->pending)
            memcpy(w->block.data() + c.to, c.from, c.bytes);
        w->pending.clear();
        return 0;
    }
};

int main()
{
    std::mt19937_64 rng(20261203);
    long calls = 0, failed = 0, failures = 0;
    for (int rep = 0; rep < 300; ++rep) {
        const size_t staging = rep % 3 == 0 ? 777 : (rep % 3 == 1 ? 4096 + rng() % 100000 : mako::kStageCopy + rng() % (3 * mako::kStageCopy));
        std::vector<unsigned char> mem(staging);
        Wire w;
        w.block.resize((size_t)8 << 20);
        // several calls over the same staging memory, some of them with a copy that fails
        for (int call = 0; call < 4; ++call) {
            w.copies = 0;
            w.fail_at = rng() % 3 == 0 ? (int)(rng() % 6) : -1;
            mako::HostStage<LateLink> stage(LateLink{&w}, mem.data(), mem.size(), w.block.size());
            std::vector<std::vector<unsigned char>> src;
            std::vector<size_t> place, stride, bytes, src_stride;
            for (int a = 0; a < 5; ++a) {
                const uint32_t rows = 1 + (uint32_t)(rng() % 5);
                const size_t b = 1 + rng() % (rng() % 4 ? 3000 : 300000), s = b + rng() % 40, ss = b + (rng() % 2 ? rng() % 50 : 0);
                src.emplace_back(rows * ss);
                for (auto& x : src.back())
                    x = (unsigned char)rng();
                place.push_back(stage.put_rows(src.back().data(), ss, b, s, rows));
                stride.push_back(s);
                bytes.push_back(b);
                src_stride.push_back(ss);
            }
            const bool meant_to_fail = w.fail_at >= 0;
            const int e = stage.send();
            ++calls;
            if (e != 0) {
                ++failed;
                if (!meant_to_fail || !w.pending.empty()) {
                    ++failures;
                    printf("FAIL: rep %d call %d: error %d, %zu copies under way\n", rep, call, e, w.pending.size());
                }
                w.pending.clear();
                continue;
            }
            (void)LateLink{&w}.wait();
            for (size_t a = 0; a < src.size(); ++a)
                for (size_t r = 0; r * src_stride[a] < src[a].size(); ++r)
                    if (place[a] % mako::kStageAlign || memcmp(w.block.data() + place[a] + r * stride[a], src[a].data() + r * src_stride[a], bytes[a]) != 0) {
                        ++failures;
                        printf("FAIL: rep %d call %d array %zu row %zu differs\n", rep, call, a, r);
                    }
        }
    }
    { // a block that is too small
        Wire w;
        w.block.resize(1024);
        std::vector<unsigned char> mem(4096), x(2000);
        mako::HostStage<LateLink> stage(LateLink{&w}, mem.data(), mem.size(), w.block.size());
        stage.put(x.data(), 100);
        stage.put(x.data(), 2000);
        if (stage.send() == 0 || !w.pending.empty()) {
            ++failures;
            printf("FAIL: a call larger than the block was accepted\n");
        }
    }
    printf("%ld calls, %ld of them failed on purpose: %ld failures\n", calls, failed, failures);
    return failures || failed < calls / 20 ? 1 : 0;
}
