// When a wave of a resident time loop stops waiting.
#pragma once

namespace swit {
namespace rk {

// A neighbour's message may take one limit.  But a group's windows start one by one, and one whose
// turn comes while other launches hold the chip starts when one of these ends, after minutes if
// that is a survey of long records: where the group does not run as a whole at the end of the limit,
// the wait may take kRoomWaits of it.  Every wave ends in any case.
constexpr unsigned kRoomWaits = 20;

// Limits count in units of 2^kWaitShift ticks of the 100 MHz clock (0.66 ms), so that kRoomWaits of
// the longest (kMaxWaitMs) are a number of 32 bits.
constexpr int kWaitShift = 16, kMaxWaitMs = 100000000;
constexpr unsigned wait_limit(int ms) { return (unsigned)((unsigned long long)ms * 100000u >> kWaitShift); }

// Whether a wait that began at clock `from` (0: begins now; the clock is never 0) has lasted the limit.
constexpr bool wait_over(unsigned long long now, unsigned long long &from, unsigned limit) {
    if (from == 0) from = now;
    return (now - from) >> kWaitShift >= limit;
}

}  // namespace rk
}  // namespace swit
