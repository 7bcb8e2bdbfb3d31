// The election of scirs_amd/csrc/elect.hpp with a thread per workgroup: random dies, random
// starts, and a first participant that reports a failure as soon as all the places are
// taken, while other workgroups have yet to start.  Prints "ok" or what went wrong.
#include "elect.hpp"
#include <atomic>
#include <cstdio>
#include <random>
#include <thread>
#include <vector>

struct Launch {
    std::atomic<int> count[8] = {}, won{0}, info{0}, timeouts{0}, taken{0};
};
struct Workgroup {
    Launch *l;
    int die;
    bool stopped() const { return l->info != 0; }
    int add() { return l->count[die]++; }
    void claim()
    {
        int none = 0;
        l->won.compare_exchange_strong(none, die + 1);
    }
    int winner() const
    {
        std::this_thread::yield();
        return l->won;
    }
    int mine() const { return die + 1; }
    void timed_out() { ++l->timeouts; }
};

int main()
{
    std::mt19937 rng(7);
    for (int trial = 0; trial < 400; ++trial) {
        const int places = 1 + trial % 5, n = 8 * (places - 1) + 1;
        const bool fails = trial % 2, before = trial % 7 == 0;
        Launch l;
        l.info = before;
        std::vector<int> place(n, -2), die(n), wait(n);
        for (int w = 0; w < n; ++w) {
            die[w] = (int)(rng() % 8);
            wait[w] = (int)(rng() % 40);
        }
        std::vector<std::thread> ts;
        for (int w = 0; w < n; ++w)
            ts.emplace_back([&, w] {
                for (int i = 0; i < wait[w]; ++i) std::this_thread::yield();
                Workgroup m{&l, die[w]};
                place[w] = elect::place(m, places, 1u << 30);
                if (place[w] < 0) return;
                ++l.taken;   // its first candidate
                while (l.taken < places) std::this_thread::yield();
                if (place[w] == 0 && fails) l.info = 1;
            });
        for (auto &t : ts) t.join();
        std::vector<int> who(places, -1);
        int in = 0;
        for (int w = 0; w < n; ++w) {
            if (place[w] < 0) continue;
            ++in;
            if (place[w] >= places || who[place[w]] >= 0 || die[w] + 1 != l.won) {
                std::printf("trial %d: place %d of die %d\n", trial, place[w], die[w]);
                return 1;
            }
            who[place[w]] = w;
        }
        if (in != (before ? 0 : places) || l.timeouts) {
            std::printf("trial %d: %d of %d places, %d timeouts\n", trial, in, places, (int)l.timeouts);
            return 1;
        }
    }
    std::printf("ok\n");
    return 0;
}
