// The host's wait for what a kernel leaves in pinned memory.
#pragma once
#include <chrono>

// Asks `ready` again and again; false: it has not come true within `most`.  (The clock is read between two questions: how often one can ask in that time differs several-fold
// between processors.)
template <class Clock = std::chrono::steady_clock, class Ready>
inline bool n2_poll(Ready ready, typename Clock::duration most) {
	const auto until = Clock::now() + most;
	do {
		if (ready()) return true;
	} while (Clock::now() < until);
	return false;
}
