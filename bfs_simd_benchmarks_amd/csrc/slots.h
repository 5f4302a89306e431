// slots.h -- the host's side of a copy-out: staging slots that are filled in
// stream order, and the threads that take their contents.  No device code, so
// that it runs against a made-up device as well.
#pragma once

#include <emmintrin.h>
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <system_error>
#include <thread>

namespace gphi {

constexpr uint32_t kSlots = 24;        // slots of a ring
constexpr uint32_t kParts = 8;         // pieces of a slot the host threads take
constexpr uint32_t kMaxHelpers = 11;   // host threads beside the caller's
constexpr uint32_t kAllHelpers = 22;   // threads that help the copy-outs of a process at one time, at most
constexpr int kSlotsStalled = 1;       // run_slots: nothing is under way that would fill the next slot

// One turn of a wait for memory that a kernel or another thread writes: the
// first ones, some tens of microseconds, keep the core; later ones give it to
// whoever wants it, above all to the threads this one waits for.
struct Turn {
	uint32_t n = 0;
	void wait()
	{
		if (++n < 2048)
			_mm_pause();
		else
			(void)sched_yield();
	}
	void reset() { n = 0; }
};

// Helpers of the copy-outs under way, over the process: several calls at once
// (the lanes of a server, contexts of several threads) share the cores that one
// call may use, instead of each taking as many.  Batches of 64 sources with rows
// of 2^20 levels on 16 cores, a round of one batch per context: 6 contexts 20 ->
// 6.8 ms, 12 contexts 54 -> 13.7, one or two as before.
inline std::atomic<uint32_t> g_helpers{0};
inline uint32_t lease_helpers(uint32_t want, uint32_t limit)
{
	uint32_t cur = g_helpers.load(std::memory_order_relaxed), n;
	do {
		n = std::min(want, limit > cur ? limit - cur : 0u);
	} while (n && !g_helpers.compare_exchange_weak(cur, cur + n, std::memory_order_relaxed));
	return n;
}
inline void return_helpers(uint32_t n) { g_helpers.fetch_sub(n, std::memory_order_relaxed); }

// Takes nslots slots through a ring of R <= kSlots, with up to `want` <=
// kMaxHelpers threads beside the calling one, as far as they keep the process's
// helpers within `limit`.  issue(i) enqueues what fills slot i (0, or
// an error, which ends the run); filled(i) says whether it has; look(&idle)
// says whether the stream has anything left to do (0, or its error); take(i,
// part), on any thread, turns part 0..kParts-1 of a filled slot into output.
// Returns 0 when every part has been taken, an error of issue or look, or
// kSlotsStalled for a stream that went idle without filling a slot; after an
// error, slots may still be filled by what was issued.
template <class Issue, class Filled, class Look, class Take>
int run_slots(uint64_t nslots, uint32_t R, uint32_t want, uint32_t limit, Issue issue, Filled filled, Look look, Take take)
{
	std::atomic<uint64_t> next{0}, ready{0};
	std::atomic<uint32_t> taken[kSlots];
	for (auto &x : taken) x.store(0);
	std::atomic<bool> stop{false};
	const uint64_t all = nslots * kParts;
	// takes the next part; waits (or not) until its slot is filled
	auto take_parts = [&](bool wait) {
		for (Turn turn;;) {
			uint64_t p = next.load(std::memory_order_relaxed);
			if (p >= all || stop.load(std::memory_order_relaxed)) return;
			if (ready.load(std::memory_order_acquire) <= p / kParts) {
				if (!wait) return;
				turn.wait();
				continue;
			}
			turn.reset();
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
	const uint32_t leased = rc == 0 ? lease_helpers(want, limit) : 0;
	try {
		for (; started < leased; ++started) helpers[started] = std::thread(take_parts, true);
	} catch (const std::system_error &) {
		// fewer helpers: the calling thread takes every part that is left
	}
	for (Turn turn; rc == 0 && ready.load(std::memory_order_relaxed) < nslots; turn.wait()) {
		const uint64_t r = ready.load(std::memory_order_relaxed);
		if (r < issued && filled(r)) {
			ready.store(r + 1, std::memory_order_release);
			spin = idle_looks = 0;
			turn.reset();
		} else if (r < issued && ++spin % 4096 == 0) {
			bool idle = false;
			rc = look(&idle);
			// an idle stream has filled every slot it was given
			if (rc == 0 && idle && ++idle_looks > 2) rc = kSlotsStalled;
		}
		if (rc == 0) issue_free();
		if (started == 0) take_parts(false);
	}
	if (rc) stop.store(true);
	take_parts(true);
	for (uint32_t i = 0; i < started; ++i) helpers[i].join();
	return_helpers(leased);
	return rc;
}

}  // namespace gphi
