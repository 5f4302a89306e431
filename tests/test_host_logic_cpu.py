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
