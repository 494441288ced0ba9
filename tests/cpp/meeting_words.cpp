// The words a step's grids meet at, left between two meetings by a wait that gave up: the step's
// first launch sets them to zero, and a sort in several workgroups after it is right.
#include <algorithm>
#include <cstdio>
#include <numeric>
#include <random>
#include <vector>

#include "k_step.hpp"

using namespace axm;

#define OK(e)                                   \
    do {                                        \
        if ((e) != hipSuccess) {                \
            std::printf("failed: %s\n", #e);    \
            return 1;                           \
        }                                       \
    } while (0)

int main() {
    const uint32_t sizes[] = {12289, 50001, 131072};
    const uint32_t cap = 131072;
    Counters* cnt;
    GridBar* bar;
    uint32_t *meet, *tmp, *buf[4];
    OK(hipMalloc((void**)&cnt, sizeof(Counters)));
    OK(hipMalloc((void**)&bar, sizeof(GridBar)));
    OK(hipMalloc((void**)&meet, 4 * radix_meet_words()));
    OK(hipMalloc((void**)&tmp, 4 * radix_tmp_words(cap)));
    for (uint32_t*& b : buf) OK(hipMalloc((void**)&b, 4 * cap));
    OK(hipMemset(cnt, 0, sizeof(Counters)));
    OK(hipMemset(tmp, 0, 4 * radix_tmp_words(cap)));
    if (!radix_setup()) return 1;
    std::mt19937 rng(1);
    for (uint32_t n : sizes) {
        std::vector<uint32_t> key(n), val(n), want(n), out(n), outv(n);
        for (uint32_t& k : key) k = rng() & 0x3FFFFFFFu;
        std::iota(val.begin(), val.end(), 0u);
        want = val;
        std::stable_sort(want.begin(), want.end(), [&](uint32_t a, uint32_t b) { return key[a] < key[b]; });
        // part of an arrival count, some generation, a stale count of the colouring
        OK(hipMemset(meet, 0x03, 4 * radix_meet_words()));
        OK(hipMemset(bar, 0x05, sizeof(GridBar)));
        OK(hipMemcpy(buf[0], key.data(), 4 * n, hipMemcpyHostToDevice));
        OK(hipMemcpy(buf[1], val.data(), 4 * n, hipMemcpyHostToDevice));
        launch_counters_begin(cnt, nullptr, Meeting{bar, meet}, 0);
        uint32_t words[SORT_MEET_WORDS + 4];
        OK(hipMemcpy(words, meet, 4 * SORT_MEET_WORDS, hipMemcpyDeviceToHost));
        OK(hipMemcpy(words + SORT_MEET_WORDS, bar, sizeof(GridBar), hipMemcpyDeviceToHost));
        for (uint32_t w : words)
            if (w != 0u) {
                std::printf("a meeting word is not zero\n");
                return 1;
            }
        const int alt = radix_sort_u32(buf[0], buf[1], buf[2], buf[3], n, 30, tmp, meet, 256, 0, &cnt->sticky);
        OK(hipDeviceSynchronize());
        OK(hipMemcpy(out.data(), buf[alt ? 2 : 0], 4 * n, hipMemcpyDeviceToHost));
        OK(hipMemcpy(outv.data(), buf[alt ? 3 : 1], 4 * n, hipMemcpyDeviceToHost));
        uint32_t sticky = 0;
        OK(hipMemcpy(&sticky, &cnt->sticky, 4, hipMemcpyDeviceToHost));
        if (sticky != 0u || outv != want) {
            std::printf("%u keys: sticky %u, order %s\n", n, sticky, outv == want ? "right" : "wrong");
            return 1;
        }
        for (uint32_t i = 0; i < n; ++i)
            if (out[i] != key[want[i]]) return 1;
    }
    std::printf("OK\n");
    return 0;
}
