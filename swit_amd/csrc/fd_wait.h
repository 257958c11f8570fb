// When a wave of a resident time loop stops waiting for a neighbour's message.
#pragma once

namespace swit {
namespace rk {

// A group's windows start one by one, and one whose turn comes while other launches hold the
// chip starts when one of these ends, after minutes if that is a survey of long records: a wave that waits for such a
// window waits for room, not for a neighbour that is stuck.  So the limit counts from the time
// at which the whole group is known to run; up to there a wave waits kRoomWaits limits, so
// that every wave ends in any case.
constexpr unsigned long long kRoomWaits = 20;

struct Wait {
    unsigned long long from = 0;    // start of the wait, or when its group was seen to run
    bool runs = false;
};

// Whether a wait ends unfinished at the clock's `now` (never 0).  group_runs(): every window of the
// group has started; asked only past the limit.
template <class F>
constexpr bool wait_over(unsigned long long now, unsigned long long limit, Wait &w, F group_runs) {
    if (w.from == 0) w.from = now;
    if (now - w.from < limit) return false;
    if (w.runs) return true;
    if (!group_runs()) return now - w.from >= kRoomWaits * limit;
    w.runs = true;
    w.from = now;
    return limit == 0;
}

}  // namespace rk
}  // namespace swit
