// Driver for the seating of resident workgroups (csrc/seating.h), built by
// tests/test_seating.py with g++ and run on the CPU: whatever arrives between
// a workgroup's look at the count and its calling off, all workgroups decide
// alike. Prints "done, N failures".
#include "seating.h"

#include <atomic>
#include <cstdio>
#include <random>
#include <thread>
#include <vector>

using namespace dimgpu;

namespace {

int g_fail = 0;

// a count to which `between` workgroups add themselves right after a load
struct Scripted {
    unsigned value, between;
    unsigned load() {
        const unsigned c = value;
        value += between;
        between = 0;
        return c;
    }
    bool replace(unsigned from, unsigned to) {
        if (value != from)
            return false;
        value = to;
        return true;
    }
};

void scripted() {
    for (unsigned need = 1; need <= 6; ++need)
        for (unsigned before = 1; before <= need; ++before)
            for (unsigned between = 0; before + between <= need; ++between) {
                Scripted c{before, between};
                // one that has waited long enough, until it decides
                Seats first;
                do
                    first = look_at_seats(c, need, true);
                while (first == Seats::kWaiting);
                c.value += need - before - between; // the rest arrive
                const Seats other = look_at_seats(c, need, false);
                if (other != first) {
                    std::printf("need %u, %u there, %u between: %d and %d\n", need, before, between,
                                static_cast<int>(first), static_cast<int>(other));
                    ++g_fail;
                }
            }
}

struct Shared {
    std::atomic<unsigned>& v;
    unsigned load() { return v.load(); }
    bool replace(unsigned from, unsigned to) { return v.compare_exchange_strong(from, to); }
};

void threads() {
    std::mt19937 g(1);
    int complete = 0, off = 0;
    for (int run = 0; run < 300; ++run) {
        constexpr unsigned kNeed = 6;
        std::atomic<unsigned> count{0};
        std::vector<Seats> got(kNeed);
        std::vector<unsigned> patience(kNeed);
        const unsigned least = 64u << run % 14; // looks; some runs complete, some do not
        for (unsigned& p : patience)
            p = least + g() % least;
        std::vector<std::thread> all;
        for (unsigned i = 0; i < kNeed; ++i)
            all.emplace_back([&, i] {
                count.fetch_add(1);
                Shared s{count};
                Seats d = Seats::kWaiting;
                for (unsigned look = 0; d == Seats::kWaiting; ++look)
                    d = look_at_seats(s, kNeed, look > patience[i]);
                got[i] = d;
            });
        for (std::thread& t : all)
            t.join();
        for (const Seats d : got)
            if (d != got[0]) {
                std::printf("run %d: workgroups decided differently\n", run);
                ++g_fail;
                break;
            }
        ++(got[0] == Seats::kComplete ? complete : off);
    }
    std::printf("%d complete, %d called off\n", complete, off);
}

} // namespace

int main() {
    scripted();
    threads();
    std::printf("done, %d failures\n", g_fail);
    return g_fail != 0;
}
