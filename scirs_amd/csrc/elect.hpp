// Which of a launch's workgroups take part in a panel that runs on one die.
#pragma once

namespace elect {

// The place 0 .. places - 1 of a workgroup among those of the elected die, or -1: it takes
// no part.  The first die on which `places` workgroups have registered is elected; with
// 8 (places - 1) + 1 workgroups on 8 dies one of them gets there.  One thread asks for the
// whole workgroup: M's stopped() may turn true while the launch is running (the panel's
// first wave reports a singular column), and waves that looked for themselves could
// disagree.  All that take part have looked before the first column can end.
// M: stopped(); add(), the workgroup's number on its die; claim(), its die's bid;
// winner(), the elected die + 1 or 0; mine(), this die + 1; timed_out(), waited in vain.
template <typename M> constexpr int place(M &m, int places, unsigned limit)
{
    const bool stop = m.stopped();
    const int number = m.add();
    if (stop) return -1;
    if (number == places - 1) m.claim();
    int won = 0;
    for (unsigned q = 0; q < limit && won == 0; ++q) won = m.winner();
    if (won == 0) m.timed_out();
    return won == m.mine() && number < places ? number : -1;
}

} // namespace elect
