"""Host-side logic of the library's headers, compiled with g++ and run on the
CPU: what a GPU run reaches only with graphs too large to test, or with a
device that fails."""
import subprocess

import pytest

from bfs_simd_benchmarks_amd import build as B


def run_cpp(tmp_path, body, *, timeout=60):
    """Compile `body` (main() included) against csrc/ and run it; its output."""
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(body)
    subprocess.run(["g++", *B.HOST_FLAGS, f"-I{B.CSRC}", str(src), "-o", str(exe), "-pthread"], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=timeout)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


def test_path_sums_do_not_wrap(tmp_path):
    run_cpp(tmp_path, r"""
#include "internal.h"
#include <algorithm>
int main()
{
	const uint32_t ds[] = {0, 1, 255, 1000000000u, 0x7FFFFFFEu, 0x7FFFFFFFu};
	const uint32_t ws[] = {0, 1, 255, 0x7FFFFFFFu, 0x80000000u, 0xFFFFFFFEu, 0xFFFFFFFFu};
	for (uint32_t d : ds)
		for (uint32_t w : ws) {
			const uint64_t want = std::min<uint64_t>((uint64_t)d + w, UINT32_MAX);
			if (gphi::path_sum(d, w) != want) return printf("%u + %u: %u\n", d, w, gphi::path_sum(d, w)), 1;
		}
	if (gphi::level_limit(UINT32_MAX) != 0x100000001ull) return 1;
	return 0;
}
""")


def test_a_dropped_queue_means_a_dense_step(tmp_path):
    """M may be anything below 2^32, and |F| + sum deg(F) more than that."""
    run_cpp(tmp_path, r"""
#include "internal.h"
int main()
{
	const uint32_t m = UINT32_MAX;
	const uint32_t fs[] = {1, 2, 1000, 1u << 25, UINT32_MAX};
	const uint32_t ds[] = {0, 1, m / 20 - 1, m / 20, m / 20 + 1, m / 2, m / 2 + 1, m - (1u << 25), m - 1, m};
	for (uint32_t threshold : {0u, 1u, m / 20, m / 2, m})
		for (uint32_t f : fs)
			for (uint32_t d : ds) {
				if (gphi::queue_dropped(d, threshold) && !gphi::dense_step(f, d, threshold))
					return printf("|F| %u, degrees %u, threshold %u: no queue for a sparse step\n", f, d, threshold), 1;
				// without a wrap it is the rule in 32 bits
				if (f + d >= f && gphi::dense_step(f, d, threshold) != (f + d > threshold)) return 1;
			}
	return 0;
}
""")


SLOTS_MAIN = r"""
#include "slots.h"
#include <cstdio>
#include <cstdlib>
using namespace gphi;
static void need(bool ok, const char *what)
{
	if (!ok) printf("%s\n", what), exit(1);
}
"""


def test_slots_in_turn(tmp_path):
    """Every part of every slot is taken once, from what its own fill left."""
    run_cpp(tmp_path, SLOTS_MAIN + r"""
int main()
{
	for (uint32_t R : {1u, 3u, kSlots})
		for (uint32_t nh : {0u, 1u, 5u, kMaxHelpers})
			for (uint64_t n : {1ull, 2ull, 3ull, 25ull, 200ull}) {
				// the device: what was issued, in order, a while later
				uint64_t slot[kSlots] = {}, issued = 0, done = 0, delay = 0;
				std::atomic<uint32_t> got[200 * kParts] = {};
				const int rc = run_slots(
				    n, R, nh, kAllHelpers, [&](uint64_t i) { return need(i == issued++, "issued in order"), 0; },
				    [&](uint64_t i) {
					    if (done < issued && ++delay % 7 == 0) slot[done % R] = done + 1, ++done;
					    return i < done;
				    },
				    [&](bool *idle) { return *idle = done == issued, 0; },
				    [&](uint64_t i, uint32_t part) {
					    need(slot[i % R] == i + 1, "a part of another fill");
					    got[i * kParts + part].fetch_add(1);
				    });
				need(rc == 0, "ends well");
				for (uint64_t k = 0; k < n * kParts; ++k) need(got[k] == 1, "each part once");
			}
	return 0;
}
""")


@pytest.mark.parametrize("what", ["refused", "never filled", "stream error"])
def test_slots_end_when_the_device_does_not_fill_them(tmp_path, what):
    """A launch that is refused, a stream that goes idle with a slot not filled,
    a stream in error: the run ends with that, every thread with it."""
    run_cpp(tmp_path, SLOTS_MAIN + f"""
int main()
{{
	const bool refused = {int(what == "refused")}, error = {int(what == "stream error")};
""" + r"""
	for (uint64_t bad : {0ull, 5ull, 30ull})
		for (uint32_t nh : {0u, 3u}) {
			uint64_t issued = 0;
			const int rc = run_slots(
			    40, 8, nh, kAllHelpers, [&](uint64_t i) { return refused && i == bad ? -5 : (++issued, 0); },
			    [&](uint64_t i) { return i < bad && i < issued; },
			    [&](bool *idle) { return *idle = !error, error ? -6 : 0; }, [](uint64_t, uint32_t) {});
			need(rc == (refused ? -5 : error ? -6 : kSlotsStalled), "ends with the error");
		}
	return 0;
}
""", timeout=20)


def test_pinned_memory_is_coherent(tmp_path):
    """The host polls words that kernels write: every pinned allocation asks for
    coherent memory, whatever HIP_HOST_COHERENT says."""
    run_cpp(tmp_path, r"""
#include "internal.h"
static unsigned seen;
extern "C" hipError_t hipHostMalloc(void **p, size_t, unsigned flags) { return seen = flags, *p = nullptr, hipSuccess; }
int main()
{
	void *p;
	if (gphi::pinned_alloc(&p, 64) != hipSuccess || !(seen & hipHostMallocCoherent)) return 1;
	return 0;
}
""")
    calls = [(f.name, line) for f in sorted(B.CSRC.iterdir()) for line in f.read_text().splitlines()
             if "hipHostMalloc(" in line]
    assert len(calls) == 1 and calls[0][0] == "internal.h", calls


def test_copy_outs_at_once_share_their_helpers(tmp_path):
    """Eight calls that would each start 11 threads have 5 between them."""
    run_cpp(tmp_path, SLOTS_MAIN + r"""
#include <cstring>
static int threads()
{
	char line[128];
	int n = 0;
	FILE *f = fopen("/proc/self/status", "r");
	while (f && fgets(line, sizeof line, f))
		if (!strncmp(line, "Threads:", 8)) n = atoi(line + 8);
	if (f) fclose(f);
	return n;
}
int main()
{
	constexpr int kCalls = 8;
	std::atomic<int> most{0}, running{0};
	std::thread calls[kCalls];
	for (auto &c : calls)
		c = std::thread([&] {
			for (++running; running < kCalls;) sched_yield();
			std::atomic<uint32_t> parts{0};
			const int rc = run_slots(
			    100, kSlots, kMaxHelpers, 5, [](uint64_t) { return 0; }, [](uint64_t) { return true; },
			    [](bool *idle) { return *idle = false, 0; },
			    [&](uint64_t, uint32_t part) {
				    ++parts;
				    if (part) return;
				    const int n = threads();
				    for (int m = most; m < n && !most.compare_exchange_weak(m, n);) {}
			    });
			need(rc == 0 && parts == 100 * kParts, "each part once");
		});
	for (auto &c : calls) c.join();
	need(most > 1 && most <= 1 + kCalls + 5, "helpers within the limit");
	need(lease_helpers(11, 5) == 5 && lease_helpers(1, 5) == 0, "all were given back");
	return 0;
}
""")


def test_waits_give_the_core_away(tmp_path):
    """A slot that is filled only once the waiting threads have yielded."""
    run_cpp(tmp_path, SLOTS_MAIN + r"""
static std::atomic<int> yields{0};
extern "C" int sched_yield() noexcept { return ++yields, 0; }
int main()
{
	for (uint32_t nh : {0u, 2u}) {
		yields = 0;
		const int rc = run_slots(
		    3, 1, nh, kAllHelpers, [](uint64_t) { return 0; }, [](uint64_t i) { return yields > 10 * (int)(i + 1); },
		    [](bool *idle) { return *idle = false, 0; }, [](uint64_t, uint32_t) {});
		need(rc == 0, "ends well");
	}
	Turn t;
	for (int i = yields = 0; i < 4096; ++i) t.wait();
	need(yields > 0, "a long wait yields");
	return 0;
}
""", timeout=20)


def test_lane_estimate_covers_its_allocations(tmp_path):
    """The server admits a graph by an estimate of its lanes' memory: it is no
    less than what the lanes allocate, for few edges and for many per vertex."""
    run_cpp(tmp_path, r"""
#include "internal.h"
#include <algorithm>
using namespace gphi;
int main()
{
	for (uint32_t n : {1000u, 8000u, 50000u, 3000000u, 33554432u})
		for (uint64_t ef : {1ull, 16ull, 100ull, 1000ull, 4000ull})
			for (uint32_t W : {16u, 512u, 4096u})
				for (uint32_t k : {1u, 64u, 256u}) {
					DevGraph G;
					G.n = n, G.m = n * ef, G.W = W;
					if (G.m >= 1ull << 32 || ef >= n) continue;
					G.n_pad = n / kPadVerts * kPadVerts + kPadVerts;
					G.nchunks = (G.m + kChunk - 1) / kChunk;
					G.side = (n + W - 1) / W;
					const uint64_t np = G.n_pad, nblk = np / kPadVerts, nw = k <= 64 ? 1 : k <= 128 ? 2 : 4;
					// levels, parents, distances, state bytes, two bitmaps, row stamps and column counts
					uint64_t sum = 3 * 4 * np + np + 2 * np / 8 + 2 * 4 * ((uint64_t)G.side + 1);
					// queue and degree prefix, tile partition, live lists, counters, trace, scan blocks
					sum += 2 * 2 * 4 * (uint64_t)queue_stride(G.n_pad, G.m) + 2 * 4 * (uint64_t)tile_lo_stride(G.m) +
					       4 * kNumXcd * (uint64_t)live_list_capacity(G.nchunks) + 4 + kLiveCntBytes +
					       sizeof(StepCtrl) + 16 * (GPHI_MAX_STEPS + 1) + nblk * (16 + 8 + 4 * 8);
					if (k > 1) {
						// masks, levels, touched bitmap and counts, live slots, start levels
						sum += (3 * 8 + 64) * nw * np + np / 8 + 64 * 256 * 4 + 65 * 128 + 257 * 4 + 16;
						// in-edges, their offsets; pieces of up to kPullPiece of vertices above kPullLight
						sum += 4 * G.m + 4 * ((uint64_t)n + 1);
						sum += 8 * (1 + G.m / kPullPiece + std::min<uint64_t>(n, G.m / kPullLight));
					}
					if (lane_state_bytes(G, k) < sum)
						return printf("n %u, m %llu, W %u, %u sources: %llu of %llu bytes\n", n, (unsigned long long)G.m, W,
						              k, (unsigned long long)lane_state_bytes(G, k), (unsigned long long)sum), 1;
				}
	return 0;
}
""")
