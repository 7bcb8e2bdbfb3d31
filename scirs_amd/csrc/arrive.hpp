// The arrival count of a launch: every workgroup registers once, the last one knows
// that all the others have read what it is about to overwrite, and clears the count for
// the next launch.  Nobody waits.
#pragma once

namespace arrive {

struct Entry {
    bool last;   // all the other workgroups of the launch have registered
    bool stop;   // an earlier failure: nothing to do
};

// Registers ahead of the decision to stop: a workgroup that left unregistered, because
// another one of the same launch had already reported a failure, would leave the count
// above zero for every later launch.  M: add() (adds one, the old count), clear(),
// stopped().
template <typename M> constexpr Entry enter(M &m, int workgroups)
{
    const bool last = m.add() == workgroups - 1;
    if (last) m.clear();
    return Entry{last, m.stopped()};
}

} // namespace arrive
