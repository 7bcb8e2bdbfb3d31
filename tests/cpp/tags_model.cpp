// The candidate words of scirs_amd/csrc/tags.hpp through several restarts of their tags:
// panels of changing numbers of waves write their slots column by column, and a reader may
// see either word of any slot as it was left by an earlier column.  No such pair may pass
// for the current one.  Prints "ok" or the pair that does.
#include "tags.hpp"
#include <cstdio>
#include <cstdlib>
#include <vector>

int main()
{
    constexpr int W = 32, G = 128;
    static tags::u64 key[2][G][2] = {};
    unsigned next = 1, rng = 12345;
    long clears = 0, columns = 0;
    for (int panel = 0; panel < 3 * 65536 / W; ++panel) {
        const tags::Range r = tags::draw(next, W, tags::CANDIDATE_TOP);
        if (r.clear) {
            ++clears;
            for (auto &b : key)
                for (auto &g : b) g[0] = g[1] = 0;
        }
        next = r.next;
        rng = rng * 1664525u + 1013904223u;
        // the others keep what they held: half of them over 2048 panels, 65536 tags, from a
        // panel of one column
        const bool all = panel % 2048 == 0;
        const int waves = all ? G : 1 + (int)((rng >> 16) % (G / 2)), width = all ? 1 : 1 + (int)((rng >> 8) % W);
        for (int j = 0; j < width; ++j, ++columns) {
            const unsigned tag = r.base + (unsigned)j;
            auto &slots = key[j & 1];
            for (int g = 0; g < G; ++g)
                // the old pair, and the pair half overwritten by this column's first word
                if (tags::current(slots[g][0], slots[g][1], tag) ||
                    tags::current(tags::value_word(tag, 7u), slots[g][1], tag) ||
                    tags::current(slots[g][0], tags::position_word(tag, 3u, 9u), tag)) {
                    std::printf("tag %u: slot %d passes with the words of an earlier column\n", tag, g);
                    return 1;
                }
            for (int g = 0; g < waves; ++g) {
                const unsigned pos = (unsigned)(g * 255 + j), hi = 0x7ff00000u - (unsigned)g, lo = 0xffffffffu - (unsigned)j;
                slots[g][0] = tags::value_word(tag, hi);
                slots[g][1] = tags::position_word(tag, pos, lo);
                if (!tags::current(slots[g][0], slots[g][1], tag) || (unsigned)slots[g][0] != hi ||
                    (unsigned)slots[g][1] != lo || tags::position(slots[g][1]) != pos) {
                    std::printf("tag %u: a current pair does not read back\n", tag);
                    return 1;
                }
            }
        }
    }
    if (clears < 2) {
        std::printf("no restart seen\n");
        return 1;
    }
    std::printf("ok %ld columns, %ld restarts\n", columns, clears);
    return 0;
}
