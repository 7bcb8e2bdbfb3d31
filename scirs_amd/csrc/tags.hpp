// Tags of the words that workgroups exchange: a reader takes a word as current when it
// carries its launch's tag, so no tag may return while an older word with it can still lie
// in the buffer.
#pragma once

namespace tags {

typedef unsigned long long u64;

// A launch's tags base .. base + span - 1, never 0 (a cleared word) and never above top.
struct Range {
    unsigned base, next;
    bool clear;   // the count restarted: clear the buffers ahead of the launch
};
constexpr Range draw(unsigned next, unsigned span, unsigned top)
{
    const bool restart = next == 0u || span == 0u || next > top - span;
    const unsigned base = restart ? 1u : next;
    return Range{base, base + (span ? span : 1u), restart};
}

// A candidate pivot in two words, each with its whole tag: |v|'s top word beside 32 bits of
// tag, the low word and the 16-bit position beside 16 bits.  Its tags are therefore drawn
// from 1 .. CANDIDATE_TOP.
constexpr unsigned CANDIDATE_TOP = 0xffffu;
constexpr u64 value_word(unsigned tag, unsigned hi) { return ((u64)tag << 32) | hi; }
constexpr u64 position_word(unsigned tag, unsigned pos, unsigned lo)
{
    return ((u64)((tag << 16) | (pos & 0xffffu)) << 32) | lo;
}
constexpr unsigned position(u64 w) { return (unsigned)(w >> 32) & 0xffffu; }
constexpr bool current(u64 value, u64 pos, unsigned tag)
{
    return (unsigned)(value >> 32) == tag && (unsigned)(pos >> 48) == tag;
}

} // namespace tags
