// slots.h -- the host's side of a copy-out: staging slots that are filled in
// stream order, and the threads that take their contents.  No device code, so
// that it runs against a made-up device as well.
#pragma once

#include <emmintrin.h>

#include <atomic>
#include <cstdint>
#include <system_error>
#include <thread>

namespace gphi {

constexpr uint32_t kSlots = 24;        // slots of a ring
constexpr uint32_t kParts = 8;         // pieces of a slot the host threads take
constexpr uint32_t kMaxHelpers = 11;   // host threads beside the caller's
constexpr int kSlotsStalled = 1;       // run_slots: nothing is under way that would fill the next slot

// Takes nslots slots through a ring of R <= kSlots, with nh <= kMaxHelpers
// threads beside the calling one.  issue(i) enqueues what fills slot i (0, or
// an error, which ends the run); filled(i) says whether it has; look(&idle)
// says whether the stream has anything left to do (0, or its error); take(i,
// part), on any thread, turns part 0..kParts-1 of a filled slot into output.
// Returns 0 when every part has been taken, an error of issue or look, or
// kSlotsStalled for a stream that went idle without filling a slot; after an
// error, slots may still be filled by what was issued.
template <class Issue, class Filled, class Look, class Take>
int run_slots(uint64_t nslots, uint32_t R, uint32_t nh, Issue issue, Filled filled, Look look, Take take)
{
	std::atomic<uint64_t> next{0}, ready{0};
	std::atomic<uint32_t> taken[kSlots];
	for (auto &x : taken) x.store(0);
	std::atomic<bool> stop{false};
	const uint64_t all = nslots * kParts;
	// takes the next part; waits (or not) until its slot is filled
	auto take_parts = [&](bool wait) {
		for (;;) {
			uint64_t p = next.load(std::memory_order_relaxed);
			if (p >= all || stop.load(std::memory_order_relaxed)) return;
			if (ready.load(std::memory_order_acquire) <= p / kParts) {
				if (!wait) return;
				_mm_pause();
				continue;
			}
			if (!next.compare_exchange_weak(p, p + 1, std::memory_order_relaxed)) continue;
			take(p / kParts, (uint32_t)(p % kParts));
			taken[p / kParts % R].fetch_add(1, std::memory_order_release);
		}
	};
	std::thread helpers[kMaxHelpers];
	uint32_t started = 0, spin = 0, idle_looks = 0;
	uint64_t issued = 0;
	int rc = 0;
	auto issue_free = [&] {
		// a slot is filled again once its last contents were taken
		while (rc == 0 && issued < nslots &&
		       (issued < R || taken[issued % R].load(std::memory_order_acquire) == issued / R * kParts))
			if ((rc = issue(issued)) == 0) ++issued;
	};
	issue_free();
	try {
		for (; rc == 0 && started < nh; ++started) helpers[started] = std::thread(take_parts, true);
	} catch (const std::system_error &) {
		// fewer helpers: the calling thread takes every part that is left
	}
	while (rc == 0 && ready.load(std::memory_order_relaxed) < nslots) {
		const uint64_t r = ready.load(std::memory_order_relaxed);
		if (r < issued && filled(r)) {
			ready.store(r + 1, std::memory_order_release);
			spin = idle_looks = 0;
		} else if (r < issued && ++spin % 4096 == 0) {
			bool idle = false;
			rc = look(&idle);
			// an idle stream has filled every slot it was given
			if (rc == 0 && idle && ++idle_looks > 2) rc = kSlotsStalled;
		}
		if (rc == 0) issue_free();
		if (started == 0) take_parts(false);
		_mm_pause();
	}
	if (rc) stop.store(true);
	take_parts(true);
	for (uint32_t i = 0; i < started; ++i) helpers[i].join();
	return rc;
}

}  // namespace gphi
