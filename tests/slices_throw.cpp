// parallel_slices when its slices throw: all slices have ended before the caller goes on, the first exception reaches the
// caller, and nothing ends the process.
#include <cstdio>
#include <new>

#include "../mms_amd/csrc/mmsim_host.h"

int main() {
    const int64_t n = 4096;
    for (int bad = -1; bad < 3; ++bad) {  // none, the first one, a later one, all
        std::vector<std::atomic<int>> seen(n);
        std::atomic<int> ended{0};
        std::atomic<bool> threw{false};
        bool thrown = false;
        try {
            mmsim::parallel_slices(n, 1, [&](int64_t lo, int64_t hi) {
                for (int64_t i = lo; i < hi; ++i) seen[(size_t)i] += 1;
                ++ended;
                if (bad == 2 || (bad == 0 && lo == 0) || (bad == 1 && lo > n / 2)) {
                    threw = true;
                    throw std::bad_alloc();
                }
            });
        } catch (const std::bad_alloc &) {
            thrown = true;
        }
        for (auto &s : seen)
            if (s != 1) return 1;
        if (thrown != threw) return 2;
        if (ended < 1) return 3;
    }
    std::puts("ok");
    return 0;
}
