// Blocks as threads through grid_meet and grid_part (grid_form.hpp), one of them
// held back at a chosen place until the search has ended or, if it has not, for a
// while.  Prints how many blocks gave up at the barrier, read a plan other than
// the search's, or ended a search, over three searches one after the other.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "../mcac_amd/csrc/grid_form.hpp"

using Clock = std::chrono::steady_clock;

struct Counters {
    std::atomic<unsigned> bar{0}, done{0}, ended{0}, gave_up{0}, other_plan{0};
    std::atomic<int> plan{0};
};

struct Grid {
    Counters &c;
    unsigned search;
    bool held_at_barrier;
    Clock::time_point since{};
    void hold() const {  // until the search has ended: 200 ms at most
        const auto t0 = Clock::now();
        while (c.ended.load() == search && Clock::now() - t0 < std::chrono::milliseconds(200)) std::this_thread::yield();
    }
    void publish() const {}
    void arrive() { c.bar.fetch_add(1), since = Clock::now(); }
    unsigned arrived() {
        if (held_at_barrier) hold();
        held_at_barrier = false;
        return c.bar.load();
    }
    bool out_of_time() const { return Clock::now() - since > std::chrono::seconds(2); }
    void pause() const { std::this_thread::yield(); }
    void give_up() const { c.gave_up.fetch_add(1); }
    unsigned ticket() const { return c.done.fetch_add(1); }
};

int main(int argc, char **argv) {
    const unsigned blocks = static_cast<unsigned>(std::atoi(argv[1])), working = static_cast<unsigned>(std::atoi(argv[2]));
    const bool at_barrier = argc > 3 && std::atoi(argv[3]) != 0;
    Counters c;
    for (unsigned search = 0; search < 3; ++search) {
        const int plan = 100 + static_cast<int>(search);
        c.plan = plan;
        std::vector<std::thread> all;
        for (unsigned me = 0; me < blocks; ++me)
            all.emplace_back([&, me] {
                const bool held = me == blocks - 1;
                Grid g{c, search, held && at_barrier};
                if (!mcac_dev::grid_meet(g, blocks)) return;
                if (held && !at_barrier) g.hold();
                if (c.plan.load() != plan) c.other_plan.fetch_add(1);
                if (!mcac_dev::grid_part(g, blocks, me < working)) return;
                c.plan = -1;  // the box as the step leaves it
                c.bar = 0;
                c.done = 0;
                c.ended.fetch_add(1);
            });
        for (auto &t : all) t.join();
    }
    std::printf("%u %u %u\n", c.gave_up.load(), c.other_plan.load(), c.ended.load());
    return 0;
}
