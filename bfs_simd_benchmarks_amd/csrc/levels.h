// levels.h -- the level loop with a device-driven frontier: the totals of each
// level, the frontier's advance, and the host that follows the device.
//
// A level's totals are the accumulators the advance of the level before it
// added to (LevelRec, a ring over the levels); every block of the next
// expansion reads them and applies the direction rule itself, so no kernel
// decides for the others.  The first block of an expansion writes the level it
// starts, and at the end the totals, to pinned host memory (LevelBoard).  The
// host keeps kAhead levels enqueued past the one it sees there, so the device
// never waits for it, and stops when it sees the end: nothing is read back,
// and at most kAhead levels are launched for nothing.
#pragma once

#include <algorithm>

#include "slots.h"
#include "sweep.h"

namespace gphi {

constexpr uint32_t kAhead = 2;  // levels enqueued past the one the device has started

// What a level's expansion reads of its totals, and the direction (dense_step)
struct Step {
	uint32_t fsize, fdeg, qsize;
	bool dense;
};

// The frontier of a traversal and what builds the next one.
struct Frontier {
	uint32_t n_pad, W, threshold;
	const uint32_t *deg;
	uint8_t *flag;
	int32_t *level;                         // BFS
	uint32_t *visited, *col_unvis;          // BFS
	uint32_t *cur, *row_stamp;
	QueueBufs qb;
	LevelRec *rec;
	LevelBoard *board;
	const uint32_t *err;                    // multi-source: stops the traversal when set
	const unsigned long long *sums;         // multi-source: totals over the sources
};

__device__ __forceinline__ LevelRec *rec_of(const Frontier &t, uint32_t level) { return t.rec + level % kLevelRing; }

__device__ __forceinline__ Step step_of(const Frontier &t, uint32_t level)
{
	const LevelRec *r = rec_of(t, level);
	const unsigned long long qp = r->qpack;
	const uint32_t f = r->fsize, d = (uint32_t)qp;
	return Step{f, d, (uint32_t)(qp >> 32), dense_step(f, d, t.threshold)};
}

// The start of a level, one thread: the previous step's chunk count and this
// step's trace entry, the totals, the ring entry of a later level, and the
// progress word.  The end is stored with a system-scope release, after which
// the host may read the whole board.
__device__ __forceinline__ void publish_level(const Frontier &t, uint32_t level, uint32_t fsize, uint32_t fdeg, uint32_t dir)
{
	LevelRec *r = rec_of(t, level);
	LevelBoard *b = t.board;
	unsigned long long reached = 0, traversed = 0;
	bool ended = false;
	if (level) {
		const LevelRec *p = rec_of(t, level - 1);
		reached = p->reached;
		traversed = p->traversed;
		ended = p->fsize == 0;
		if (!ended && level <= GPHI_MAX_STEPS) b->trace[level - 1].w = p->chunks;
	}
	if (!ended) {
		r->reached = reached + fsize;
		r->traversed = traversed + fdeg;
		*rec_of(t, level + kLevelRing / 2) = LevelRec{};
		if (fsize) {
			if (level < GPHI_MAX_STEPS) {
				b->trace[level].x = dir;
				b->trace[level].y = fsize;
				b->trace[level].z = fdeg;
				b->trace[level].w = 0u;
			}
			__hip_atomic_store(&b->progress, (unsigned long long)(level + 1) << 1, __ATOMIC_RELAXED,
			                   __HIP_MEMORY_SCOPE_SYSTEM);
		} else {
			// a multi-source traversal keeps its own totals, over its sources
			b->reached = t.sums ? t.sums[0] : reached;
			b->traversed = t.sums ? t.sums[1] : traversed;
			b->err = t.err ? *t.err : 0u;
			b->levels = level;
			b->t_end = wall_clock64();
			__hip_atomic_store(&b->progress, ((unsigned long long)(level + 1) << 1) | 1ull, __ATOMIC_RELEASE,
			                   __HIP_MEMORY_SCOPE_SYSTEM);
		}
	}
}

// The next frontier from the state bytes and its queue, in one pass.  A lane
// owns kLaneVerts consecutive vertices: a frontier of a few thousand vertices
// then spreads over enough wavefronts that none has more than one round of
// degree loads, one prefix sum and kLaneVerts queue entries per lane to do
// (a lane per 32-vertex word, as in frontier_mark_kernel, took 16 us on the
// 9 blocks of a 65536-vertex graph).  A block adds its totals to the next
// level's accumulators, which gives it its queue position and degree prefix;
// the blocks' shares of the queue come in any order.  Once the degrees added
// so far pass the direction rule's threshold the next step is dense and needs
// no queue.
// Blocks are 256 threads up to kAdvanceNarrow vertices and 1024 above: a block
// makes two atomics, all on one line (on 1.6M vertices 256-thread blocks took
// 19 us for a dense level, 15 of them the atomics, and 1024-thread ones 11;
// on 65536 vertices, with nothing to queue for, they took 5.4 and 6.0).
constexpr uint32_t kLaneVerts = 8;
constexpr uint32_t kAdvanceNarrow = 1u << 18;
static_assert(kPadVerts % (1024 * kLaneVerts) == 0, "whole blocks over the padded vertices");

template <bool kBfs, uint32_t kThreads>
__device__ __forceinline__ void advance_block(const Frontier &t, uint32_t level)
{
	if (rec_of(t, level)->fsize == 0 || (t.err && *t.err)) return;
	LevelRec *nr = rec_of(t, level + 1);
	const uint32_t next_level = level + 1;
	const uint32_t i = blockIdx.x * kThreads + threadIdx.x, v0 = i * kLaneVerts;
	const uint32_t lane = lane_id(), wid = threadIdx.x >> 6;
	uint2 *fp = reinterpret_cast<uint2 *>(t.flag) + i;
	const uint2 f8 = *fp;
	uint32_t bits = 0;
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		bits |= ((f8.x >> (8 * k)) & 1u) << k;
		bits |= ((f8.y >> (8 * k)) & 1u) << (4 + k);
	}
	// byte i of the bitmaps: bits of the lane's vertices
	reinterpret_cast<uint8_t *>(t.cur)[i] = (uint8_t)bits;
	uint32_t d[kLaneVerts], q = 0, dsum = 0;
#pragma unroll
	for (uint32_t k = 0; k < kLaneVerts; ++k) d[k] = 0;
	if (bits) {
		const uint4 da = reinterpret_cast<const uint4 *>(t.deg + v0)[0], db = reinterpret_cast<const uint4 *>(t.deg + v0)[1];
		if (kBfs) {
			constexpr uint32_t kLow = 0x01010101u;  // state 1 -> kVisited
			*fp = make_uint2(f8.x + (f8.x & kLow), f8.y + (f8.y & kLow));
			reinterpret_cast<uint8_t *>(t.visited)[i] |= (uint8_t)bits;
#pragma unroll
			for (uint32_t k = 0; k < kLaneVerts; ++k)
				if ((bits >> k) & 1u) t.level[v0 + k] = (int32_t)next_level;
		} else {
			*fp = make_uint2(0, 0);
		}
		const uint32_t dd[kLaneVerts] = {da.x, da.y, da.z, da.w, db.x, db.y, db.z, db.w};
#pragma unroll
		for (uint32_t k = 0; k < kLaneVerts; ++k) {
			d[k] = (bits >> k) & 1u ? dd[k] : 0u;
			q += d[k] > 0;
			dsum += d[k];
		}
		if (t.W % kLaneVerts == 0) {  // one row for the lane's vertices
			if (q) t.row_stamp[v0 / t.W] = next_level;
		} else {
#pragma unroll
			for (uint32_t k = 0; k < kLaneVerts; ++k)
				if (d[k]) t.row_stamp[(v0 + k) / t.W] = next_level;
		}
	}
	const uint32_t nf = (uint32_t)__popc(bits);
	__shared__ uint32_t s_red[3][kThreads / 64];
	__shared__ unsigned long long s_base;
	uint32_t ftot, qtot, dtot;
	const uint32_t qx = wave_excl_scan(q, &qtot), dx = wave_excl_scan(dsum, &dtot);
	ftot = wave_sum(nf);
	if (lane == 0) {
		s_red[0][wid] = ftot;
		s_red[1][wid] = qtot;
		s_red[2][wid] = dtot;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		uint32_t f = 0, qb = 0, db = 0;
		for (uint32_t k = 0; k < kThreads / 64; ++k) {
			f += s_red[0][k];
			qb += s_red[1][k];
			db += s_red[2][k];
		}
		unsigned long long base = ~0ull;
		if (f) atomicAdd(&nr->fsize, f);
		if (qb) {
			base = atomicAdd(&nr->qpack, ((unsigned long long)qb << 32) | db);
			if (queue_dropped((uint32_t)base + db, t.threshold)) base = ~0ull;  // the next step is dense
		}
		s_base = base;
	}
	if (kBfs && ftot) {
		// column counts of unvisited vertices: one atomic per wavefront when
		// its vertices share a column, else one per lane (or vertex)
		const uint32_t wv0 = v0 - lane * kLaneVerts;
		if (wv0 / t.W == (wv0 + 64 * kLaneVerts - 1) / t.W) {
			if (lane == 0) atomicSub(t.col_unvis + wv0 / t.W, ftot);
		} else if (t.W % kLaneVerts == 0) {
			if (nf) atomicSub(t.col_unvis + v0 / t.W, nf);
		} else {
			for (uint32_t b = bits; b; b &= b - 1) atomicSub(t.col_unvis + (v0 + __ffs(b) - 1) / t.W, 1u);
		}
	}
	__syncthreads();
	if (s_base == ~0ull || q == 0) return;
	uint32_t pos = (uint32_t)(s_base >> 32) + qx, off = (uint32_t)s_base + dx;
	for (uint32_t k = 0; k < wid; ++k) {
		pos += s_red[1][k];
		off += s_red[2][k];
	}
	const uint32_t par = next_level & 1u;
	uint32_t *__restrict__ queue = t.qb.queue + par * t.qb.qstride;
	uint32_t *__restrict__ qoff = t.qb.qoff + par * t.qb.qstride;
	uint32_t *__restrict__ tile_lo = t.qb.tile_lo + par * t.qb.tstride;
#pragma unroll
	for (uint32_t k = 0; k < kLaneVerts; ++k) {
		if (!d[k]) continue;
		queue[pos] = v0 + k;
		qoff[pos] = off;
		// tiles of the next push whose first edge falls in [off, off + d)
		for (uint32_t x = (off + kSparseTile - 1) / kSparseTile; (uint64_t)x * kSparseTile < (uint64_t)off + d[k]; ++x)
			tile_lo[x] = pos;
		pos += 1;
		off += d[k];
	}
}

// threads per block and blocks of an advance
inline unsigned advance_threads(uint32_t n_pad) { return n_pad <= kAdvanceNarrow ? 256 : 1024; }
inline unsigned advance_blocks(uint32_t n_pad) { return n_pad / (advance_threads(n_pad) * kLaneVerts); }

inline Frontier make_frontier(gphi_graph *gr, uint32_t threshold)
{
	const DevGraph &G = gr->g;
	Frontier f = {};
	f.n_pad = G.n_pad, f.W = G.W, f.threshold = threshold;
	f.deg = G.deg;
	f.flag = gr->flag, f.cur = gr->cur, f.row_stamp = gr->row_stamp;
	f.level = gr->level, f.visited = gr->visited, f.col_unvis = gr->col_unvis;
	f.qb = gr->queue_bufs();
	f.rec = gr->rec();
	f.board = gr->ctx->h_board;
	return f;
}

// Waits until the count in the upper 63 bits of a progress word passes `seen`
// (for LevelBoard::progress, levels started, the end counting as one more);
// the word in *out.  The stream is looked at now
// and then, so that an error on the device ends the wait.
inline int wait_progress(gphi_ctx *ctx, const unsigned long long *word, unsigned long long seen,
                         unsigned long long *out)
{
	uint32_t idle = 0;
	Turn turn;
	for (uint32_t spin = 1;; ++spin) {
		const unsigned long long p = __atomic_load_n(word, __ATOMIC_ACQUIRE);
		if ((p >> 1) > seen) {
			*out = p;
			return GPHI_OK;
		}
		if (spin % 4096 == 0) {
			const hipError_t e = hipStreamQuery(ctx->stream);
			if (e != hipSuccess && e != hipErrorNotReady) return hip_fail(ctx, e, "level loop", __FILE__, __LINE__);
			// an idle stream has published every enqueued level
			if (e == hipSuccess && ++idle > 2) return set_error(ctx, GPHI_E_STATE, "level loop made no progress");
		}
		turn.wait();
	}
}

// Before the kernel that opens a traversal is launched.  One that returned an
// error before its end may have kernels in flight that still write the board
// (after an end is reported none does): those are waited for.
inline int reset_board(gphi_ctx *ctx)
{
	if (ctx->board_busy) GPHI_HIP(ctx, hipStreamSynchronize(ctx->stream));
	ctx->board_busy = true;
	__atomic_store_n(&ctx->h_board->progress, 0ull, __ATOMIC_RELEASE);
	return GPHI_OK;
}

// enqueue(level) launches a level; until the device reports the end
template <class F>
int follow_levels(gphi_ctx *ctx, F enqueue)
{
	uint32_t enq = 0, started = 0;
	for (;;) {
		for (; enq < std::max(started, 1u) + kAhead; ++enq) {
			const int rc = enqueue(enq);
			if (rc) return rc;
		}
		GPHI_HIP(ctx, hipGetLastError());
		unsigned long long p;
		const int rc = wait_progress(ctx, &ctx->h_board->progress, started, &p);
		if (rc) return rc;
		if (p & 1ull) {
			ctx->board_busy = false;
			return GPHI_OK;
		}
		started = (uint32_t)(p >> 1);
	}
}

inline float board_ms(const gphi_ctx *ctx)
{
	return (float)((double)(ctx->h_board->t_end - ctx->h_board->t_begin) / ctx->wall_clock_khz);
}

}  // namespace gphi
