// The arrival count of scirs_amd/csrc/arrive.hpp over every order in which the
// workgroups of one launch can start, register and, workgroup 0, report a failure.
// Prints "ok" or the first order that leaves the count above zero.
#include "arrive.hpp"
#include <cstdio>
#include <vector>

struct Launch { int count = 0, info = 0, last = 0; };
struct Workgroup {
    Launch *l;
    int info;
    int add() { return l->count++; }
    void clear() { l->count = 0; }
    bool stopped() const { return info != 0; }
};

static bool orders(Launch l, std::vector<int> state, std::vector<int> seen, bool fails, std::vector<int> &path, long &n)
{
    const int g = (int)state.size();
    bool moved = false;
    for (int w = 0; w < g; ++w) {
        // 0: not started, 1: info read, 2: registered, 3: done (workgroup 0 has reported)
        if (state[w] == 3 || (state[w] == 2 && w != 0)) continue;
        moved = true;
        Launch m = l;
        auto st = state, sn = seen;
        if (st[w] == 0) {
            sn[w] = m.info;
        } else if (st[w] == 1) {
            Workgroup me{&m, sn[w]};
            const arrive::Entry e = arrive::enter(me, g);
            m.last += e.last;
            if (w == 0 && (e.stop || !fails)) st[w] = 2;   // nothing to report
        } else if (fails) {
            m.info = 1;
        }
        ++st[w];
        path.push_back(w);
        if (!orders(m, st, sn, fails, path, n)) return false;
        path.pop_back();
    }
    if (!moved) {
        ++n;
        if (l.count != 0 || l.last != 1) {
            std::printf("count %d, %d last ones after", l.count, l.last);
            for (int w : path) std::printf(" %d", w);
            std::printf("\n");
            return false;
        }
    }
    return true;
}

int main()
{
    long n = 0;
    for (int g = 1; g <= 5; ++g)
        for (int before = 0; before < 2; ++before)
            for (int fails = 0; fails < 2; ++fails) {
                Launch l;
                l.info = before;
                std::vector<int> path;
                if (!orders(l, std::vector<int>(g, 0), std::vector<int>(g, 0), fails != 0, path, n)) return 1;
            }
    std::printf("ok %ld\n", n);
    return 0;
}
