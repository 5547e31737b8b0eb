// Runs the PCG host loop (csrc/k_groups.hpp) against a simulated stream and
// checks every solve of `k` working iterations under every budget: see
// tests/test_pcg_groups.py.
#include <cstdio>
#include <cstdlib>

#include "k_groups.hpp"

#define REQUIRE(c)                                                                                    \
    do {                                                                                              \
        if (!(c)) {                                                                                   \
            std::printf("line %d: %s (k %d, limit %d, launched %d)\n", __LINE__, #c, k, limit, next); \
            std::exit(1);                                                                             \
        }                                                                                             \
    } while (0)

// Times in us. The solve is over after iteration k - 1 (or the budget's last);
// an iteration costs the host `launch` and the device `work`, or `empty` once
// the solve is over.
struct Stream {
    int k = 0, limit = 0;
    double launch_us = 0, work = 0, empty = 0;
    double copy_us = 8, event_wait = 20, all_wait = 10, host = 0, device = 0;
    int next = 0, fail_at = -1;
    struct Mirror {
        double landed = 0;
        bool before = true, after = true;  // slot 0: the end of an earlier solve
    } m[2];
    bool ended() const { return next >= k || next >= limit; }
    int launch(int it) {
        if (it == fail_at) return -7;
        REQUIRE(it == next && it < limit);
        host += launch_us;
        device = std::max(device, host) + (ended() ? empty : work);
        next++;
        return 0;
    }
    int post(int s) {
        REQUIRE(m[s].landed <= host);  // no copy of this slot is still on its way
        host += 3;
        device = std::max(device, host) + copy_us;
        m[s].before = m[s].after;
        m[s].after = ended();
        m[s].landed = device;
        return 0;
    }
    int wait(int s, bool all) {
        host = std::max(host, all ? device : m[s].landed) + (all ? all_wait : event_wait);
        return 0;
    }
    bool over(int s) {
        REQUIRE(m[s].landed <= host);
        return m[s].after;
    }
    bool seen_over(int s) { return m[s].landed <= host ? m[s].after : m[s].before; }
    double finish() { return std::max(host, device); }
};

static Stream stream(int k, int limit, double launch, double work, double empty) {
    Stream s;
    s.k = k;
    s.limit = limit;
    s.launch_us = launch;
    s.work = work;
    s.empty = empty;
    s.m[1].before = s.m[1].after = false;  // the state at the entry
    return s;
}

// groups of 4, 8, ... 64, each waited for
static double doubling(int k, int limit, double launch, double work, double empty) {
    Stream s = stream(k, limit, launch, work, empty);
    for (int batch = 4; !s.m[1].after; batch = std::min(2 * batch, 64)) {
        for (int i = 0; i < batch && s.next < limit; i++) s.launch(s.next);
        s.post(1);
        s.wait(1, true);
    }
    return s.finish();
}

int main() {
    const double devices[][3] = {{25, 30, 8}, {25, 15, 5}, {20, 160, 10}, {15, 750, 12}, {60, 10, 8}};
    for (const auto& d : devices)
        for (int short_its = 0; short_its < 2; short_its++)
            for (int limit = 1; limit <= 140; limit++)
                for (int k = 1; k <= limit + 1; k++) {
                    Stream s = stream(k, limit, d[0], d[1], d[2]);
                    int last = -1, next = 0;
                    const int rc = ifl::run_groups(s, limit, short_its != 0, &last);
                    next = s.next;
                    REQUIRE(rc == 0 && (last == 0 || last == 1));
                    REQUIRE(s.over(last));
                    const int worked = std::min(k, limit);
                    REQUIRE(next >= worked && next <= limit);
                    // the rest of its group and one group more
                    REQUIRE(next - worked <= (short_its || worked <= 12 ? 7 : 15));
                }
    // a failed launch ends the loop with its error
    for (int at = 0; at < 40; at++) {
        Stream s = stream(1000, 1000, 25, 30, 8);
        s.fail_at = at;
        int last, k = 1000, limit = 1000, next = at;
        REQUIRE(ifl::run_groups(s, limit, at % 2 != 0, &last) == -7 && s.next == at);
    }
    // A small grid of one strip: no solve takes longer than with doubling
    // groups by more than two iterations' launches (what the host may have
    // sent before the copy that it looks at has landed).
    for (int k = 1; k <= 90; k++) {
        Stream s = stream(k, 600, 25, 30, 8);
        int last, limit = 600, next = 0;
        ifl::run_groups(s, limit, ifl::short_iterations(16, 1), &last);
        REQUIRE(s.finish() <= doubling(k, limit, 25, 30, 8) + 2 * 25);
    }
    std::printf("ok\n");
    return 0;
}
