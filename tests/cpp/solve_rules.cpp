// The rule by which the register sweep takes the islands of 257 to 4096 manifolds, on the host.
#include <cstdio>

#include "k_step.hpp"

using namespace axm;

static int failed = 0;
#define CHECK(x)                                                   \
    do {                                                           \
        if (!(x)) {                                                \
            std::printf("line %d: %s\n", __LINE__, #x);            \
            failed = 1;                                            \
        }                                                          \
    } while (0)

int main() {
    const uint32_t G = 256;
    Counters c{};
    c.max_colour = 12;
    c.m_glob = 0;
    c.isl_wide = 10;  // one island of 300
    c.isl_most = 300;
    c.m_eff = 300;
    CHECK(wide_pieces(&c, G) == 10);
    // the last slot's inbox ends within the buffer, or the sweep does not take them
    const uint32_t most = (uint32_t)(FLOW_INBOX_BYTES / (INBOX_WORDS * 8u));
    c.m_eff = most;
    CHECK(((uint64_t)(most - 1u) + 1u) * INBOX_WORDS * 8u <= FLOW_INBOX_BYTES);
    CHECK(wide_pieces(&c, G) == 10);
    for (uint32_t m : {most + 1u, 1u << 25, 1u << 26, 1u << 27, 0xFFFFFFFFu}) {
        c.m_eff = m;
        CHECK(wide_pieces(&c, G) == 0);
    }
    // more colours than a mask holds; more pieces than waves, one long island against many
    c.m_eff = 300;
    c.max_colour = 65;
    CHECK(wide_pieces(&c, G) == 0);
    c.max_colour = 64;
    c.isl_wide = G * FLOW_WAVES;
    CHECK(wide_pieces(&c, G) == G * FLOW_WAVES);
    c.isl_wide = G * FLOW_WAVES + 1u;
    CHECK(wide_pieces(&c, G) == 0);
    c.isl_most = 4096;
    CHECK(wide_pieces(&c, G) == G * FLOW_WAVES + 1u);
    if (!failed) std::printf("OK\n");
    return failed;
}
