// copyout.hip -- results from HBM to the caller's host arrays.
//
// A hipMemcpy into pageable memory goes through the runtime's own staging
// buffer and one host thread: 134 MB of levels took 13 ms (10 GB/s) and 1 MB
// 0.4 ms, where the link carries 56 GB/s.  Here a kernel writes each piece of
// the results into a slot of pinned memory, as narrow as the values allow,
// and host threads turn finished slots into the caller's arrays while the
// next ones cross the link:
//
//   levels  : 4 bits per level below 15 (every level of a shallow traversal),
//             else 8, as level + 1 with 0 for unreached; widened by the host.
//             The host's first touch of the array then sets the pace (about
//             100 GB/s over 8 threads; up to 12 take part), not the link.
//   distances: 4, 8 or 16 bits when the largest one fits, found by a pass over
//             them first (from kNarrowBytes of output on), as distance + 1 with
//             0 for unreached
//   others  : 4-byte words as they are
//
// A slot is finished when the flag beside it holds its sequence number: a
// one-thread kernel stores it behind the kernel that filled the slot, and the
// host sees it 5 us sooner than an event or a stream synchronization.
//
// Reference: the results stay in host memory there (apps/bfs_simd/bfs.cpp:
// 753-963); this is the copy that takes their place.
#include <hip/hip_runtime.h>

#include <emmintrin.h>
#include <sched.h>

#include <algorithm>
#include <cstring>
#include <mutex>

#include "internal.h"
#include "slots.h"

namespace gphi {

namespace {

constexpr size_t kSlotBytes = 2u << 20;
constexpr uint64_t kHelperBytes = 2u << 20;  // a helper per this much output (starting one takes about 20 us)
constexpr uint64_t kNarrowBytes = 1u << 20;  // distances: output from which a pass for the largest pays (10 us)
constexpr unsigned kFillGrid = 256;    // blocks that fill a slot: enough to keep the link busy

__global__ void slot_done_kernel(unsigned long long *flag, unsigned long long seq)
{
	__hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// four levels as bytes, each + 1 modulo 256 (255, unreached, becomes 0)
__device__ __forceinline__ uint32_t inc_bytes(uint32_t x)
{
	return ((x & 0x7F7F7F7Fu) + 0x01010101u) ^ (x & 0x80808080u);
}

// the low nibbles of four bytes, in 16 bits
__device__ __forceinline__ uint32_t squeeze(uint32_t x)
{
	x &= 0x0F0F0F0Fu;
	x = (x | (x >> 4)) & 0x00FF00FFu;
	return (x | (x >> 8)) & 0xFFFFu;
}

// 32 values of one row from element v (a multiple of 32) as level + 1 bytes
struct WordLevels {  // int32 levels, valid where state is not 0
	const int32_t *level;
	const uint8_t *state;
	__device__ __forceinline__ void load(uint32_t, uint32_t v, uint32_t (&x)[8]) const
	{
		const uint4 *l = reinterpret_cast<const uint4 *>(level + v);
		const uint4 *s = reinterpret_cast<const uint4 *>(state + v);
		const uint4 sa = s[0], sb = s[1];
		const uint32_t st[8] = {sa.x, sa.y, sa.z, sa.w, sb.x, sb.y, sb.z, sb.w};
#pragma unroll
		for (int i = 0; i < 8; ++i) {
			const uint4 q = l[i];
			const uint32_t b[4] = {q.x, q.y, q.z, q.w};
			x[i] = 0;
#pragma unroll
			for (int k = 0; k < 4; ++k)
				x[i] |= ((st[i] >> (8 * k)) & 0xFFu ? (b[k] + 1u) & 0xFFu : 0u) << (8 * k);
		}
	}
};
struct ByteLevels {  // uint8 levels, 255 unreached; row r is row slot[r] of the array
	const uint8_t *level;
	uint32_t pitch;
	uint8_t slot[kBatchMaxSources];
	__device__ __forceinline__ void load(uint32_t row, uint32_t v, uint32_t (&x)[8]) const
	{
		const uint4 *p = reinterpret_cast<const uint4 *>(level + (uint64_t)slot[row] * pitch + v);
		const uint4 a = p[0], b = p[1];
		x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
#pragma unroll
		for (int i = 0; i < 8; ++i) x[i] = inc_bytes(x[i]);
	}
};

// elements [first, first + count) of the rows laid end to end (rowlen each, a
// multiple of 32), 32 per lane; kBits per element
template <int kBits, class Src>
__global__ __launch_bounds__(kBlock) void fill_levels_kernel(Src src, uint64_t first, uint64_t count, uint32_t rowlen,
                                                             uint4 *__restrict__ out)
{
	for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < count / 32; i += (uint64_t)gridDim.x * kBlock) {
		const uint64_t e = first + i * 32;
		const uint32_t row = (uint32_t)(e / rowlen), v = (uint32_t)(e % rowlen);
		uint32_t x[8];
		src.load(row, v, x);
		if (kBits == 4) {
			out[i] = make_uint4(squeeze(x[0]) | squeeze(x[1]) << 16, squeeze(x[2]) | squeeze(x[3]) << 16,
			                    squeeze(x[4]) | squeeze(x[5]) << 16, squeeze(x[6]) | squeeze(x[7]) << 16);
		} else {
			out[2 * i] = make_uint4(x[0], x[1], x[2], x[3]);
			out[2 * i + 1] = make_uint4(x[4], x[5], x[6], x[7]);
		}
	}
}

// 4-byte words, 4 per lane; with a state array, -1 where it is 0
__global__ __launch_bounds__(kBlock) void fill_words_kernel(const uint4 *__restrict__ src,
                                                            const uint32_t *__restrict__ state, uint64_t first,
                                                            uint64_t count, uint4 *__restrict__ out)
{
	for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < (count + 3) / 4;
	     i += (uint64_t)gridDim.x * kBlock) {
		uint4 x = src[first / 4 + i];
		if (state) {
			const uint32_t s = state[first / 4 + i];
			if (!(s & 0xFFu)) x.x = ~0u;
			if (!(s & 0xFF00u)) x.y = ~0u;
			if (!(s & 0xFF0000u)) x.z = ~0u;
			if (!(s & 0xFF000000u)) x.w = ~0u;
		}
		out[i] = x;
	}
}

// the largest of n distances that is not `none`, into *word (0 before)
__global__ __launch_bounds__(kBlock) void max_dist_kernel(const uint4 *__restrict__ dist, uint64_t n, uint32_t none,
                                                          uint32_t *word)
{
	uint32_t m = 0;
	for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < n / 4; i += (uint64_t)gridDim.x * kBlock) {
		const uint4 x = dist[i];
		m = max(max(m, x.x == none ? 0u : x.x), x.y == none ? 0u : x.y);
		m = max(max(m, x.z == none ? 0u : x.z), x.w == none ? 0u : x.w);
	}
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 64));
	if (threadIdx.x % 64 == 0 && m) atomicMax(word, m);
}
// *word into the slot, and cleared for the next pass
__global__ void report_word_kernel(uint32_t *word, uint32_t *out)
{
	*out = *word;
	*word = 0;
}

__device__ __forceinline__ uint32_t dist_code(uint32_t d, uint32_t none) { return d == none ? 0u : d + 1; }

// n distances from `first` (a multiple of 32), 32 per lane (the array is padded)
template <int kBits>
__global__ __launch_bounds__(kBlock) void fill_dist_kernel(const uint32_t *__restrict__ dist, uint32_t none,
                                                           uint64_t first, uint64_t count, uint4 *__restrict__ out)
{
	for (uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x; i < (count + 31) / 32;
	     i += (uint64_t)gridDim.x * kBlock) {
		const uint4 *p = reinterpret_cast<const uint4 *>(dist + first + i * 32);
		constexpr int kPer = 32 / kBits;  // codes per word
		uint32_t w[kBits];
#pragma unroll
		for (int j = 0; j < kBits; ++j) w[j] = 0;
#pragma unroll
		for (int q = 0; q < 8; ++q) {
			const uint4 x = p[q];
			const uint32_t d[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
			for (int j = 0; j < 4; ++j) w[(4 * q + j) / kPer] |= dist_code(d[j], none) << (kBits * ((4 * q + j) % kPer));
		}
#pragma unroll
		for (int j = 0; j < kBits / 4; ++j)
			out[i * (kBits / 4) + j] = make_uint4(w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]);
	}
}

// rows of a vertex-major array (kSsspBatchMax words per vertex): a slot holds
// the rows' values of `count` vertices from `first`, row by row; a lane per
// vertex, so its reads share cache lines and a wavefront's writes of a row are
// consecutive.  (In 16-bit codes the rows take as long: the host's first touch
// of them sets the pace.)
__global__ __launch_bounds__(kBlock) void fill_vertex_rows_kernel(const uint32_t *__restrict__ src, uint32_t k,
                                                                  uint32_t first, uint32_t count,
                                                                  uint32_t *__restrict__ out)
{
	for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < count; i += gridDim.x * kBlock) {
		const uint4 *p = reinterpret_cast<const uint4 *>(src + (uint64_t)(first + i) * kSsspBatchMax);
#pragma unroll
		for (uint32_t q = 0; q < kSsspBatchMax / 4; ++q) {
			if (4 * q >= k) break;
			const uint4 x = p[q];
			const uint32_t b[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
			for (uint32_t j = 0; j < 4; ++j)
				if (4 * q + j < k) out[(4 * q + j) * count + i] = b[j];
		}
	}
}

// The host's widening of packed levels: element i of p (kBits each, level + 1)
// to dst, for count elements from an even element.
template <int kBits>
void widen(const uint8_t *p, uint64_t i, uint64_t count, uint8_t *dst)
{
	const __m128i one = _mm_set1_epi8(1), low = _mm_set1_epi8(15);
	uint64_t k = 0;
	if (kBits == 4) {
		const uint8_t *q = p + i / 2;
		for (; k + 32 <= count; k += 32) {
			const __m128i x = _mm_loadu_si128(reinterpret_cast<const __m128i *>(q + k / 2));
			const __m128i a = _mm_and_si128(x, low), b = _mm_and_si128(_mm_srli_epi16(x, 4), low);
			_mm_storeu_si128(reinterpret_cast<__m128i *>(dst + k), _mm_sub_epi8(_mm_unpacklo_epi8(a, b), one));
			_mm_storeu_si128(reinterpret_cast<__m128i *>(dst + k + 16), _mm_sub_epi8(_mm_unpackhi_epi8(a, b), one));
		}
		for (; k < count; ++k) dst[k] = (uint8_t)(((q[k / 2] >> (4 * (k & 1))) & 15) - 1);
	} else {
		const uint8_t *q = p + i;
		for (; k + 16 <= count; k += 16)
			_mm_storeu_si128(reinterpret_cast<__m128i *>(dst + k),
			                 _mm_sub_epi8(_mm_loadu_si128(reinterpret_cast<const __m128i *>(q + k)), one));
		for (; k < count; ++k) dst[k] = (uint8_t)(q[k] - 1);
	}
}

inline void widen16(__m128i x, int32_t *dst)  // 16 bytes to 16 words, each - 1
{
	const __m128i zero = _mm_setzero_si128(), one = _mm_set1_epi32(1);
	const __m128i a = _mm_unpacklo_epi8(x, zero), b = _mm_unpackhi_epi8(x, zero);
	__m128i *o = reinterpret_cast<__m128i *>(dst);
	_mm_storeu_si128(o, _mm_sub_epi32(_mm_unpacklo_epi16(a, zero), one));
	_mm_storeu_si128(o + 1, _mm_sub_epi32(_mm_unpackhi_epi16(a, zero), one));
	_mm_storeu_si128(o + 2, _mm_sub_epi32(_mm_unpacklo_epi16(b, zero), one));
	_mm_storeu_si128(o + 3, _mm_sub_epi32(_mm_unpackhi_epi16(b, zero), one));
}

template <int kBits>
void widen(const uint8_t *p, uint64_t i, uint64_t count, int32_t *dst)
{
	const __m128i low = _mm_set1_epi8(15);
	uint64_t k = 0;
	if (kBits == 4) {
		const uint8_t *q = p + i / 2;
		for (; k + 32 <= count; k += 32) {
			const __m128i x = _mm_loadu_si128(reinterpret_cast<const __m128i *>(q + k / 2));
			const __m128i a = _mm_and_si128(x, low), b = _mm_and_si128(_mm_srli_epi16(x, 4), low);
			widen16(_mm_unpacklo_epi8(a, b), dst + k);
			widen16(_mm_unpackhi_epi8(a, b), dst + k + 16);
		}
		for (; k < count; ++k) dst[k] = (int32_t)((q[k / 2] >> (4 * (k & 1))) & 15) - 1;
	} else {
		const uint8_t *q = p + i;
		for (; k + 16 <= count; k += 16) widen16(_mm_loadu_si128(reinterpret_cast<const __m128i *>(q + k)), dst + k);
		for (; k < count; ++k) dst[k] = (int32_t)q[k] - 1;
	}
}

// codes (distance + 1, 0 unreached) to distances: 4 words at a time
inline __m128i decode4(__m128i x, __m128i none)
{
	const __m128i zero = _mm_cmpeq_epi32(x, _mm_setzero_si128());
	return _mm_or_si128(_mm_and_si128(zero, none), _mm_andnot_si128(zero, _mm_sub_epi32(x, _mm_set1_epi32(1))));
}
inline void decode16(__m128i x, __m128i none, uint32_t *dst)  // 16 bytes
{
	const __m128i zero = _mm_setzero_si128();
	const __m128i a = _mm_unpacklo_epi8(x, zero), b = _mm_unpackhi_epi8(x, zero);
	__m128i *o = reinterpret_cast<__m128i *>(dst);
	_mm_storeu_si128(o, decode4(_mm_unpacklo_epi16(a, zero), none));
	_mm_storeu_si128(o + 1, decode4(_mm_unpackhi_epi16(a, zero), none));
	_mm_storeu_si128(o + 2, decode4(_mm_unpacklo_epi16(b, zero), none));
	_mm_storeu_si128(o + 3, decode4(_mm_unpackhi_epi16(b, zero), none));
}

// element i of p (kBits each) to dst, for count elements from an even element
template <int kBits>
void decode(const uint8_t *p, uint64_t i, uint64_t count, uint32_t none, uint32_t *dst)
{
	const __m128i nn = _mm_set1_epi32((int)none), low = _mm_set1_epi8(15), zero = _mm_setzero_si128();
	const uint8_t *q = p + i * kBits / 8;
	auto at = [&](uint64_t k) -> uint32_t {
		if (kBits == 4) return (q[k / 2] >> (4 * (k & 1))) & 15u;
		if (kBits == 8) return q[k];
		return (uint32_t)q[2 * k] | (uint32_t)q[2 * k + 1] << 8;
	};
	uint64_t k = 0;
	for (; k + 32 <= count; k += 32) {
		if (kBits == 4) {
			const __m128i x = _mm_loadu_si128(reinterpret_cast<const __m128i *>(q + k / 2));
			const __m128i a = _mm_and_si128(x, low), b = _mm_and_si128(_mm_srli_epi16(x, 4), low);
			decode16(_mm_unpacklo_epi8(a, b), nn, dst + k);
			decode16(_mm_unpackhi_epi8(a, b), nn, dst + k + 16);
		} else if (kBits == 8) {
			decode16(_mm_loadu_si128(reinterpret_cast<const __m128i *>(q + k)), nn, dst + k);
			decode16(_mm_loadu_si128(reinterpret_cast<const __m128i *>(q + k + 16)), nn, dst + k + 16);
		} else {
			for (int j = 0; j < 4; ++j) {
				const __m128i x = _mm_loadu_si128(reinterpret_cast<const __m128i *>(q + 2 * k + 16 * j));
				__m128i *o = reinterpret_cast<__m128i *>(dst + k + 8 * j);
				_mm_storeu_si128(o, decode4(_mm_unpacklo_epi16(x, zero), nn));
				_mm_storeu_si128(o + 1, decode4(_mm_unpackhi_epi16(x, zero), nn));
			}
		}
	}
	for (; k < count; ++k) dst[k] = at(k) ? at(k) - 1 : none;
}

// Pinned slots, leased for one copy-out.  Making a ring takes 0.3 ms (one
// slot) to 1 ms (kSlots), which would be paid on every context's first call,
// so finished copy-outs leave theirs for the next: up to kIdleRings of each
// size stay with the process while it has a context, and none after that.
// Single slots are what the lanes of a server lease at the same time: with two
// kept, 59 queries on graphs of 16384 vertices took 2.0 ms, with sixteen 1.35.
struct Ring {
	uint8_t *mem = nullptr;      // the slots, then their flags, a line apart
	uint32_t slots = 0;
	unsigned long long seq = 0;  // sequence number of the slot filled last
};
constexpr uint32_t kIdleRings[2] = {2, 16};  // of kSlots slots, of one: 128 MiB in all
std::mutex g_ring_mu;  // guards the three below
Ring g_idle[2][16];
uint32_t g_idle_count[2] = {0, 0};
uint32_t g_contexts = 0;

int lease_ring(gphi_ctx *ctx, bool one, Ring *out)
{
	{
		std::lock_guard<std::mutex> lk(g_ring_mu);
		uint32_t &c = g_idle_count[one];
		if (c) {
			*out = g_idle[one][--c];
			return GPHI_OK;
		}
	}
	const uint32_t slots = one ? 1 : kSlots;
	const hipError_t e = pinned_alloc((void **)&out->mem, slots * (kSlotBytes + 128));
	if (e != hipSuccess) {
		out->mem = nullptr;
		return set_error(ctx, GPHI_E_OOM, "pinned staging of %u slots: %s", slots, hipGetErrorString(e));
	}
	memset(out->mem + slots * kSlotBytes, 0, slots * 128);
	out->slots = slots;
	return GPHI_OK;
}

void return_ring(bool one, const Ring &r)
{
	{
		std::lock_guard<std::mutex> lk(g_ring_mu);
		if (g_idle_count[one] < kIdleRings[one]) {
			g_idle[one][g_idle_count[one]++] = r;
			return;
		}
	}
	(void)hipHostFree(r.mem);
}

// helpers a copy-out is worth, and those the process may have at one time
uint32_t helper_count(uint64_t nslots, uint64_t out_bytes)
{
	if (nslots <= 1 && out_bytes < 4 * kHelperBytes) return 0;
	return (uint32_t)std::min<uint64_t>(kMaxHelpers, out_bytes / kHelperBytes);
}
uint32_t helper_limit()
{
	cpu_set_t set;
	const int cpus = sched_getaffinity(0, sizeof set, &set) == 0 ? CPU_COUNT(&set) : 1;
	return (uint32_t)std::min<int>(kAllHelpers, std::max(cpus - 1, 0));
}

// fill(slot number, slot) enqueues the kernel that fills a slot; take(slot
// number, part, slot) turns part 0..kParts-1 of a filled slot into output, on
// any thread.  Returns when every part has been taken.
template <class Fill, class Take>
int stream_out(gphi_ctx *ctx, uint64_t nslots, uint64_t out_bytes, Fill fill, Take take)
{
	if (nslots == 0) return GPHI_OK;
	const bool one = nslots == 1;
	Ring ring;
	int rc = lease_ring(ctx, one, &ring);
	if (rc) return rc;
	const uint32_t R = ring.slots;
	hipStream_t s = ctx->stream;
	uint8_t *mem = ring.mem;
	auto flag = [&](uint64_t i) {
		return reinterpret_cast<unsigned long long *>(mem + R * kSlotBytes + (i % R) * 128);
	};
	auto slot = [&](uint64_t i) { return mem + (i % R) * kSlotBytes; };
	const unsigned long long seq0 = ring.seq + 1;  // slot i is filled when its flag is seq0 + i
	ring.seq += nslots;
	const uint32_t want = helper_count(nslots, out_bytes);
	rc = run_slots(
	    nslots, R, want, want ? helper_limit() : 0,
	    [&](uint64_t i) -> int {
		    fill(i, slot(i));
		    slot_done_kernel<<<1, 1, 0, s>>>(flag(i), seq0 + i);
		    GPHI_HIP(ctx, hipGetLastError());
		    return GPHI_OK;
	    },
	    [&](uint64_t i) { return __atomic_load_n(flag(i), __ATOMIC_ACQUIRE) >= seq0 + i; },
	    [&](bool *idle) -> int {
		    const hipError_t e = hipStreamQuery(s);
		    if (e != hipSuccess && e != hipErrorNotReady) return hip_fail(ctx, e, "copy-out", __FILE__, __LINE__);
		    *idle = e == hipSuccess;
		    return GPHI_OK;
	    },
	    [&](uint64_t i, uint32_t part) { take(i, part, (const uint8_t *)slot(i)); });
	if (rc == kSlotsStalled) rc = set_error(ctx, GPHI_E_STATE, "copy-out made no progress");
	if (rc) {
		// fills may be under way: the ring goes back if they end, and is not used again otherwise
		if (hipStreamSynchronize(s) == hipSuccess) return_ring(one, ring);
		return rc;
	}
	return_ring(one, ring);
	return GPHI_OK;
}

// part `part` of kParts of `count` elements, cut at multiples of 64
inline void part_range(uint64_t count, uint32_t part, uint64_t *lo, uint64_t *hi)
{
	const uint64_t per = (count / kParts + 63) / 64 * 64 + 64;
	*lo = std::min(count, part * per);
	*hi = std::min(count, *lo + per);
	if (part == kParts - 1) *hi = count;
}

unsigned fill_grid(uint64_t lanes) { return (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(kFillGrid, (lanes + kBlock - 1) / kBlock)); }

// nrows rows of n levels each into rows[i]; every level is below 2^kBits - 1
template <int kBits, class Src, class T>
int out_level_rows(gphi_ctx *ctx, Src src, uint32_t n, uint32_t nrows, T *const *rows)
{
	const uint32_t rowlen = (n + 31) / 32 * 32;
	const uint64_t total = (uint64_t)rowlen * nrows, per = kSlotBytes * 8 / kBits;
	const uint64_t nslots = (total + per - 1) / per;
	hipStream_t s = ctx->stream;
	return stream_out(
	    ctx, nslots, (uint64_t)n * nrows * sizeof(T),
	    [&](uint64_t i, uint8_t *slot) {
		    const uint64_t count = std::min(per, total - i * per);
		    fill_levels_kernel<kBits><<<fill_grid(count / 32), kBlock, 0, s>>>(src, i * per, count, rowlen,
		                                                                       reinterpret_cast<uint4 *>(slot));
	    },
	    [&](uint64_t i, uint32_t part, const uint8_t *slot) {
		    uint64_t lo, hi;
		    part_range(std::min(per, total - i * per), part, &lo, &hi);
		    while (lo < hi) {  // the stretch of one row at a time
			    const uint64_t e = i * per + lo;
			    const uint32_t row = (uint32_t)(e / rowlen), v = (uint32_t)(e % rowlen);
			    const uint64_t len = std::min<uint64_t>(hi - lo, rowlen - v);
			    if (v < n) widen<kBits>(slot, lo, std::min<uint64_t>(len, n - v), rows[row] + v);
			    lo += len;
		    }
	    });
}

template <int kBits>
int out_codes(gphi_ctx *ctx, const uint32_t *dev, uint32_t none, uint32_t n, uint32_t *dst)
{
	const uint64_t per = kSlotBytes * 8 / kBits, nslots = (n + per - 1) / per;
	hipStream_t s = ctx->stream;
	return stream_out(
	    ctx, nslots, (uint64_t)n * 4,
	    [&](uint64_t i, uint8_t *slot) {
		    const uint64_t count = std::min<uint64_t>(per, n - i * per);
		    fill_dist_kernel<kBits><<<fill_grid(count / 32 + 1), kBlock, 0, s>>>(dev, none, i * per, count,
		                                                                        reinterpret_cast<uint4 *>(slot));
	    },
	    [&](uint64_t i, uint32_t part, const uint8_t *slot) {
		    uint64_t lo, hi;
		    part_range(std::min<uint64_t>(per, n - i * per), part, &lo, &hi);
		    if (lo < hi) decode<kBits>(slot, lo, hi - lo, none, dst + i * per + lo);
	    });
}

// the largest of n (a multiple of 4) distances that is not `none`
int largest_dist(gphi_ctx *ctx, const uint32_t *dev, uint64_t n, uint32_t none, uint32_t *out)
{
	hipStream_t s = ctx->stream;
	if (!ctx->d_word) {
		int rc = dmalloc(ctx, (void **)&ctx->d_word, 4, nullptr);
		if (rc) return rc;
		fill_words(ctx, ctx->d_word, 1, 0);
	}
	return stream_out(
	    ctx, 1, 4,
	    [&](uint64_t, uint8_t *slot) {
		    max_dist_kernel<<<(unsigned)std::min<uint64_t>(512, n / 4 / kBlock + 1), kBlock, 0, s>>>(
		        reinterpret_cast<const uint4 *>(dev), n, none, ctx->d_word);
		    report_word_kernel<<<1, 1, 0, s>>>(ctx->d_word, reinterpret_cast<uint32_t *>(slot));
	    },
	    [&](uint64_t, uint32_t part, const uint8_t *slot) {
		    if (part == 0) memcpy(out, slot, 4);
	    });
}

}  // namespace

int out_words(gphi_ctx *ctx, const void *dev, const uint8_t *state, uint32_t n, void *dst)
{
	const uint64_t per = kSlotBytes / 4, nslots = ((uint64_t)n + per - 1) / per;
	hipStream_t s = ctx->stream;
	return stream_out(
	    ctx, nslots, (uint64_t)n * 4,
	    [&](uint64_t i, uint8_t *slot) {
		    const uint64_t count = std::min<uint64_t>(per, n - i * per);
		    fill_words_kernel<<<fill_grid(count / 4 + 1), kBlock, 0, s>>>(
		        static_cast<const uint4 *>(dev), reinterpret_cast<const uint32_t *>(state), i * per, count,
		        reinterpret_cast<uint4 *>(slot));
	    },
	    [&](uint64_t i, uint32_t part, const uint8_t *slot) {
		    uint64_t lo, hi;
		    part_range(std::min<uint64_t>(per, n - i * per), part, &lo, &hi);
		    if (lo < hi) memcpy(static_cast<uint8_t *>(dst) + (i * per + lo) * 4, slot + lo * 4, (hi - lo) * 4);
	    });
}

int out_bfs_levels(gphi_graph *gr, uint32_t deepest, int32_t *levels)
{
	const WordLevels src{gr->level, gr->flag};
	if (deepest <= 14) return out_level_rows<4>(gr->ctx, src, gr->g.n, 1, &levels);
	if (deepest <= 254) return out_level_rows<8>(gr->ctx, src, gr->g.n, 1, &levels);
	return out_words(gr->ctx, gr->level, gr->flag, gr->g.n, levels);
}

template <class T>
int out_batch_rows(gphi_graph *gr, const uint32_t *slots, uint32_t deepest, uint32_t nrows, T *const *rows)
{
	ByteLevels src{gr->b_level, gr->g.n_pad, {}};
	for (uint32_t i = 0; i < nrows; ++i) src.slot[i] = (uint8_t)slots[i];
	if (deepest <= 14) return out_level_rows<4>(gr->ctx, src, gr->g.n, nrows, rows);
	return out_level_rows<8>(gr->ctx, src, gr->g.n, nrows, rows);
}
template int out_batch_rows(gphi_graph *, const uint32_t *, uint32_t, uint32_t, uint8_t *const *);
template int out_batch_rows(gphi_graph *, const uint32_t *, uint32_t, uint32_t, int32_t *const *);

int out_dist(gphi_ctx *ctx, const uint32_t *dev, uint32_t none, uint32_t n, uint32_t n_pad, uint32_t *dst)
{
	if ((uint64_t)n * 4 < kNarrowBytes) return out_words(ctx, dev, nullptr, n, dst);
	uint32_t top = 0;
	int rc = largest_dist(ctx, dev, n_pad, none, &top);
	if (rc) return rc;
	if (top < 15) return out_codes<4>(ctx, dev, none, n, dst);
	if (top < 255) return out_codes<8>(ctx, dev, none, n, dst);
	if (top < 65535) return out_codes<16>(ctx, dev, none, n, dst);
	return out_words(ctx, dev, nullptr, n, dst);
}

int out_sssp_rows(gphi_graph *gr, uint32_t k, uint32_t *const *rows)
{
	gphi_ctx *ctx = gr->ctx;
	const uint32_t n = gr->g.n;
	const uint32_t per = (uint32_t)(kSlotBytes / 4 / k) / 64 * 64;  // vertices per slot
	const uint64_t nslots = ((uint64_t)n + per - 1) / per;
	hipStream_t s = ctx->stream;
	return stream_out(
	    ctx, nslots, (uint64_t)n * k * 4,
	    [&](uint64_t i, uint8_t *slot) {
		    const uint32_t first = (uint32_t)(i * per), count = std::min(per, n - first);
		    fill_vertex_rows_kernel<<<fill_grid(count), kBlock, 0, s>>>(gr->sb_dist, k, first, count,
		                                                                reinterpret_cast<uint32_t *>(slot));
	    },
	    [&](uint64_t i, uint32_t part, const uint8_t *slot) {
		    const uint32_t first = (uint32_t)(i * per), count = std::min(per, n - first);
		    for (uint32_t r = part; r < k; r += kParts)
			    if (rows[r]) memcpy(rows[r] + first, slot + (size_t)r * count * 4, (size_t)count * 4);
	    });
}

void out_context_opened()
{
	std::lock_guard<std::mutex> lk(g_ring_mu);
	++g_contexts;
}

void out_context_closed()
{
	std::lock_guard<std::mutex> lk(g_ring_mu);
	if (--g_contexts) return;
	for (int k = 0; k < 2; ++k)
		while (g_idle_count[k]) (void)hipHostFree(g_idle[k][--g_idle_count[k]].mem);
}

}  // namespace gphi
