// Whether the workgroups of a resident launch run (resident.hip).
#pragma once

namespace dimgpu {

constexpr unsigned kCalledOff = 0x10000; // in the count: the launch does not take place

enum class Seats { kWaiting, kComplete, kCalledOff };

// One look at the count of running workgroups by one of them. A workgroup that
// has waited long enough calls the launch off, but only from the incomplete
// count that it saw: a count that has become complete in between stays so, and
// a complete one is never called off, so all of them decide alike.
//
// count.load() reads it; count.replace(from, to) changes it in one step if it
// still is `from` and says whether it did. (constexpr: for the device and, in
// tests, for the host.)
template<typename Count>
constexpr Seats look_at_seats(Count& count, unsigned need, bool waited_enough) {
    const unsigned c = count.load();
    if (c == need)
        return Seats::kComplete;
    if (c >= kCalledOff)
        return Seats::kCalledOff;
    if (waited_enough && count.replace(c, c + kCalledOff))
        return Seats::kCalledOff;
    return Seats::kWaiting;
}

} // namespace dimgpu
