// Copies of results that arrive in pieces (regf_pack.cpp), built and run by
// tests/test_copy_cpu.py: every piece is copied once and only after it has
// arrived, and the pool takes another caller's job while a copy waits.
//   copy_check pieces | pool | few
// few: the process may start a few threads only; a job runs on those.
#include <stdio.h>
#include <string.h>
#include <sys/resource.h>

#include <algorithm>
#include <functional>
#include <thread>
#include <vector>

#include "../../abyss_amd/csrc/regf_pack.h"

static int fails = 0;
#define CHECK(c)                                                       \
    do {                                                               \
        if (!(c)) {                                                    \
            fprintf(stderr, "check failed: %s (line %d)\n", #c, __LINE__); \
            ++fails;                                                   \
        }                                                              \
    } while (0)

static void pieces()
{
    for (int steps : {1, 2, 5, 17})
        for (int parts : {1, 3, abyss::host_parts()})
            for (int early : {0, 1, 3})   // pieces that arrive with the one waited for
                for (int bad : {-1, 0, steps - 1}) {
                    constexpr int kLen = 1003;
                    std::vector<int> src(steps * kLen, 0), dst(steps * kLen, 0);
                    int arrived = 0;
                    const auto bring = [&](int upto) {
                        for (; arrived < std::min(upto, steps); ++arrived)
                            for (int e = 0; e < kLen; ++e) src[arrived * kLen + e] = arrived + 1;
                    };
                    const bool ok = abyss::copy_arriving(
                        steps, parts,
                        [&](int k) {
                            if (k == bad) return false;
                            bring(k + 1 + early);
                            return true;
                        },
                        [&](int k) { return k < arrived && k != bad; },
                        [&](int k0, int k1, int p, int n) {
                            const long a = (long)k0 * kLen, len = (long)(k1 - k0) * kLen;
                            for (long e = a + len * p / n; e < a + len * (p + 1) / n; ++e)
                                dst[e] += src[e];
                        });
                    CHECK(ok == (bad < 0));
                    const int done = bad < 0 ? steps : bad;
                    bool same = true;
                    for (int k = 0; k < steps; ++k)
                        for (int e = 0; e < kLen; ++e)
                            same = same && dst[k * kLen + e] == (k < done ? k + 1 : 0);
                    CHECK(same);
                }
}

static void pool()
{
    if (abyss::host_parts() < 2) return;
    int taken = 0;
    const auto other = [](int) {};
    abyss::copy_arriving(
        4, abyss::host_parts(),
        [&](int) {
            // a caller of another context, while this one waits for the GPU
            std::thread t([&] { taken += abyss::host_run(2, other); });
            t.join();
            return true;
        },
        [](int) { return false; }, [](int, int, int, int) {});
    CHECK(taken == 4);
}

static void few()
{
    // address space for the stacks of a few threads
    struct rlimit lim;
    CHECK(getrlimit(RLIMIT_AS, &lim) == 0);
    lim.rlim_cur = 40u << 20;
    CHECK(setrlimit(RLIMIT_AS, &lim) == 0);
    const int parts = abyss::host_parts();
    CHECK(parts >= 1 && parts <= 8);
    std::vector<int> ran(8, 0);
    CHECK(abyss::host_run(parts, [&](int p) { ran[p] += 1; }));
    for (int p = 0; p < 8; ++p) CHECK(ran[p] == (p < parts ? 1 : 0));
}

int main(int argc, char **argv)
{
    const char *what = argc > 1 ? argv[1] : "";
    if (!strcmp(what, "pieces")) pieces();
    else if (!strcmp(what, "pool")) pool();
    else if (!strcmp(what, "few")) few();
    else return 2;
    printf("OK: %d failure(s)\n", fails);
    return fails ? 1 : 0;
}
