// small.hip -- the BFS and SSSP level loop of graphs whose levels take less
// time than their launches.
//
// The level loop of device.hip runs five kernels per level (push or chunk
// selection, sweep, mark, scan, emit), eight levels per read-back.  On a
// graph of a few million vertices a level's work takes a few microseconds,
// and the launches, about 2.6 us each, set the pace: the 43 launches of a
// 1024-vertex BFS took 215 us.  Here a level is two launches:
//
//   expand  : the CSR push of a sparse step, or the tile sweep of a dense
//             step, whose blocks each test a fixed share of the chunks for
//             liveness instead of walking a list a kernel before made
//   advance : the next frontier from the state bytes -- bitmap, levels, row
//             stamps, column counts -- and its queue, at positions reserved
//             with one atomic per block, so that no scan comes between
//
// A level's totals are the accumulators the advance of the level before it
// added to (LevelRec, a ring over the levels); every block of the next
// expansion reads them and applies the direction rule itself.
//
// The first block of an expansion writes the level it starts, and at the end
// the totals, to pinned host memory (LevelBoard).  The host keeps kAhead
// levels enqueued past the one it sees there, so the device never waits for
// it, and stops when it sees the end: nothing is read back, and at most
// kAhead levels are launched for nothing.
//
// Reference: the level loop of apps/bfs_simd/bfs.cpp:795-910 and
// apps/sssp_simd/sssp.cpp:1000-1100.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstring>

#include "sweep.h"

namespace gphi {

namespace {

constexpr uint32_t kAhead = 2;  // levels enqueued past the one the device has started

// What the kernels of one traversal share.
struct Trav {
	uint32_t n, n_pad, n_words, W, side, threshold, win_rows;
	uint32_t nchunks, run, slots;  // chunks per run, chunks tested per block
	const uint32_t *row_off, *cols, *csr_w, *deg;
	const uint32_t *heads, *tails, *coo_w;
	const uint16_t *heads16, *tails16;
	const uint8_t *coo_w8;
	const ChunkMeta *meta;
	const ChunkPack *pack;
	int32_t *level, *parent;
	uint32_t *dist;
	uint8_t *flag;
	uint32_t *visited, *cur, *row_stamp, *col_unvis;
	QueueBufs qb;
	LevelRec *rec;
	LevelBoard *board;
};

__device__ __forceinline__ LevelRec *rec_of(const Trav &t, uint32_t level) { return t.rec + level % kLevelRing; }

// All state of a traversal set up for its source, in one launch: every word
// is written once, with the source's part in it.
template <bool kBfs>
__global__ __launch_bounds__(kBlock) void small_init_kernel(Trav t, uint32_t src)
{
	const uint32_t d = t.deg[src];
	const uint32_t nf = t.n_pad / 16, ntile = (d + kSparseTile - 1) / kSparseTile;
	const uint32_t stride = gridDim.x * kBlock, i0 = blockIdx.x * kBlock + threadIdx.x;
	if (!kBfs)
		for (uint32_t i = i0; i < t.n_pad; i += stride) t.dist[i] = i == src ? 0u : (uint32_t)INT_MAX;
	for (uint32_t i = i0; i < max(max(nf, t.n_words), max(t.side, ntile + 1)); i += stride) {
		if (i < nf) {
			uint4 f = make_uint4(0, 0, 0, 0);
			if (kBfs && src / 16 == i) {
				const uint32_t b = (uint32_t)kVisited << (8 * (src % 4)), k = src % 16 / 4;
				f.x = k == 0 ? b : 0u, f.y = k == 1 ? b : 0u, f.z = k == 2 ? b : 0u, f.w = k == 3 ? b : 0u;
			}
			reinterpret_cast<uint4 *>(t.flag)[i] = f;
		}
		if (i < t.n_words) {
			const uint32_t b = src / 32 == i ? 1u << (src % 32) : 0u;
			t.cur[i] = b;
			if (kBfs) t.visited[i] = b;
		}
		if (i < t.side) {
			t.row_stamp[i] = i == src / t.W ? 0u : UINT32_MAX;
			if (kBfs) t.col_unvis[i] = ((i + 1 == t.side) ? t.n - i * t.W : t.W) - (i == src / t.W);
		}
		if (i < ntile + 1) t.qb.tile_lo[i] = 0;
		if (i < kLevelRing) {
			LevelRec r = {};
			if (i == 0) {
				r.fsize = 1;
				r.qpack = ((unsigned long long)(d ? 1 : 0) << 32) | d;
			}
			t.rec[i] = r;
		}
	}
	if (i0 == 0) {
		if (kBfs) {
			t.level[src] = 0;
			t.parent[src] = (int32_t)src;
		}
		t.qb.queue[0] = src;
		t.qb.qoff[0] = 0;
		t.board->t_begin = wall_clock64();
	}
}

// The start of a level, one thread: the previous step's chunk count and this
// step's trace entry, the totals, the ring entry of a later level, and the
// progress word.  The end is stored with a system-scope release, after which
// the host may read the whole board.
__device__ void publish_level(const Trav &t, uint32_t level, uint32_t fsize, uint32_t fdeg, uint32_t dir)
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
			b->reached = reached;
			b->traversed = traversed;
			b->levels = level;
			b->t_end = wall_clock64();
			__hip_atomic_store(&b->progress, ((unsigned long long)(level + 1) << 1) | 1ull, __ATOMIC_RELEASE,
			                   __HIP_MEMORY_SCOPE_SYSTEM);
		}
	}
}

// CSR push of a sparse step: a block per tile of kSparseTile frontier edges
// (its first queue entry in tile_lo), 4 edges per lane whose loads go out
// together.  Tails are marked in their state byte; the advance does the rest.
constexpr uint32_t kPushEntry = kSparseTile + 2;  // LDS: degree prefix, vertex and CSR base of the tile's entries
template <bool kBfs>
__device__ __forceinline__ void small_push(uint32_t *s_mem, const Trav &t, uint32_t level, uint32_t qsize,
                                           uint32_t qdeg)
{
	uint32_t *s_off = s_mem, *s_u = s_mem + kPushEntry, *s_base = s_mem + 2 * kPushEntry;
	const uint32_t par = level & 1u;
	const uint32_t *__restrict__ queue = t.qb.queue + par * t.qb.qstride;
	const uint32_t *__restrict__ qoff = t.qb.qoff + par * t.qb.qstride;
	const uint32_t *__restrict__ tile_lo = t.qb.tile_lo + par * t.qb.tstride;
	const uint32_t ntile = (qdeg + kSparseTile - 1) / kSparseTile;
	constexpr int kPer = kSparseTile / kBlock;
	for (uint32_t k = blockIdx.x; k < ntile; k += gridDim.x) {
		const uint32_t lo = tile_lo[k];
		uint32_t hi = (k + 1 < ntile) ? tile_lo[k + 1] : qsize - 1;
		if (hi > qsize - 1) hi = qsize - 1;
		const uint32_t cnt = hi - lo + 1;
		for (uint32_t j = threadIdx.x; j < cnt; j += kBlock) {
			const uint32_t u = queue[lo + j];
			s_off[j] = qoff[lo + j];
			s_u[j] = u;
			s_base[j] = t.row_off[u];
		}
		__syncthreads();
		const uint32_t e0 = k * kSparseTile, e1 = min(e0 + kSparseTile, qdeg);
		uint32_t uu[kPer], vv[kPer], ix[kPer];
		bool on[kPer];
#pragma unroll
		for (int r = 0; r < kPer; ++r) {
			const uint32_t e = e0 + threadIdx.x + r * kBlock;
			on[r] = e < e1;
			uint32_t a = 0, b = cnt;  // largest j with s_off[j] <= e
			while (b - a > 1) {
				const uint32_t mid = (a + b) >> 1;
				if (s_off[mid] <= e)
					a = mid;
				else
					b = mid;
			}
			uu[r] = s_u[a];
			ix[r] = on[r] ? s_base[a] + (e - s_off[a]) : 0u;
			vv[r] = on[r] ? t.cols[ix[r]] : 0u;
		}
		if (kBfs) {
			uint32_t sv[kPer];
#pragma unroll
			for (int r = 0; r < kPer; ++r) sv[r] = on[r] ? t.flag[vv[r]] : 1u;
#pragma unroll
			for (int r = 0; r < kPer; ++r)
				if (sv[r] == 0) {
					t.parent[vv[r]] = (int32_t)uu[r];
					t.flag[vv[r]] = 1;
				}
		} else {
			// as in the dense sweep: an edge that beats the dist[v] it read
			// lowers it and marks v, which then improved in this step
			uint32_t nd[kPer], dv[kPer];
#pragma unroll
			for (int r = 0; r < kPer; ++r) {
				nd[r] = on[r] ? t.dist[uu[r]] + t.csr_w[ix[r]] : UINT32_MAX;
				dv[r] = t.dist[vv[r]];
			}
#pragma unroll
			for (int r = 0; r < kPer; ++r)
				if (nd[r] < dv[r]) {
					atomicMin(t.dist + vv[r], nd[r]);
					t.flag[vv[r]] = 1;
				}
		}
		__syncthreads();
	}
}

// A chunk is live when a head row of it holds a frontier vertex with
// out-edges and, for BFS, a tail column of it has an unvisited vertex
// (apps/bfs_simd/bfs.cpp:275); ranges of more than 16 rows or columns count
// as holding one.
template <bool kBfs>
__device__ __forceinline__ bool chunk_live(const Trav &t, uint32_t c, uint32_t level)
{
	const ChunkMeta md = t.meta[c];
	if (md.row_lo > md.row_hi) return false;
	const uint32_t nr = md.row_hi - md.row_lo + 1, nc = md.col_hi - md.col_lo + 1;
	bool rows = nr > 16, colm = !kBfs || nc > 16;
#pragma unroll
	for (uint32_t k = 0; k < 16; ++k) {
		rows |= nr <= 16 && k < nr && t.row_stamp[md.row_lo + k] == level;
		if (kBfs) colm |= nc <= 16 && k < nc && t.col_unvis[md.col_lo + k] != 0;
	}
	return rows && colm;
}

// kWeights: 0 BFS, 1 SSSP with 1-byte weights, 4 SSSP with 32-bit weights
template <int kWeights>
__global__ __launch_bounds__(kBlock, kWeights ? 5 : 7) void small_expand_kernel(Trav t, uint32_t level)
{
	constexpr bool kBfs = kWeights == 0;
	// the push's entries, or the sweep's windows
	constexpr uint32_t kMem = std::max<uint32_t>(3 * kPushEntry, (kBfs ? 2 : 1) * kWinWords);
	__shared__ uint4 s_mem[(kMem + 3) / 4];
	LevelRec *r = rec_of(t, level);
	const uint32_t fsize = r->fsize;
	const unsigned long long qp = r->qpack;
	const uint32_t fdeg = (uint32_t)qp;
	// the first step is sparse (apps/bfs_simd/bfs.cpp:807), then the rule of :829-834
	const bool dense = level > 0 && fsize + fdeg > t.threshold;
	if (blockIdx.x == 0 && threadIdx.x == 0) publish_level(t, level, fsize, fdeg, dense);
	if (fsize == 0) return;
	if (!dense) {
		small_push<kBfs>(reinterpret_cast<uint32_t *>(s_mem), t, level, (uint32_t)(qp >> 32), fdeg);
		return;
	}
	// this block's share of the chunks: runs of t.run consecutive chunks (they
	// share LDS windows), run j of block b at run j * gridDim + b
	__shared__ uint32_t s_list[kBlock];
	__shared__ uint32_t s_cnt[kBlock / 64];
	const uint32_t tid = threadIdx.x, wid = tid >> 6;
	const uint32_t c = (tid / t.run * gridDim.x + blockIdx.x) * t.run + tid % t.run;
	const bool live = tid < t.slots && c < t.nchunks && chunk_live<kBfs>(t, c, level);
	const unsigned long long m = __ballot(live);
	if (lane_id() == 0) s_cnt[wid] = (uint32_t)__popcll(m);
	__syncthreads();
	uint32_t at = 0, total = 0;
	for (uint32_t k = 0; k < kBlock / 64; ++k) {
		if (k < wid) at += s_cnt[k];
		total += s_cnt[k];
	}
	if (live) s_list[at + __popcll(m & ((1ull << lane_id()) - 1ull))] = c;
	if (tid == 0 && total) atomicAdd(&r->chunks, total);
	__syncthreads();
	total = (uint32_t)__builtin_amdgcn_readfirstlane((int)total);
	if constexpr (kBfs)
		bfs_dense_walk(s_mem, s_mem + kWinWords / 4, LdsChunkList{s_list}, 0, total, 0, t.heads, t.tails, t.heads16, t.tails16, t.meta, t.pack, t.cur,
		               t.visited, t.n_words, t.W, t.win_rows, t.flag, t.parent);
	else
		sssp_dense_walk<kWeights == 1>(s_mem, LdsChunkList{s_list}, 0, total, 0, t.heads, t.tails, t.heads16, t.tails16,
		                               t.coo_w, t.coo_w8, t.meta, t.pack, t.cur, t.n_words, t.W, t.win_rows, t.dist,
		                               t.flag);
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
__global__ __launch_bounds__(kThreads) void small_advance_kernel(Trav t, uint32_t level)
{
	if (rec_of(t, level)->fsize == 0) return;
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
			if ((uint32_t)base + db > t.threshold) base = ~0ull;  // the next step is dense
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

}  // namespace

// whether the loop is the faster one (kSmallVerts)
bool small_graph(const DevGraph &G, bool bfs)
{
	return G.n <= kSmallVerts && G.nchunks <= (bfs ? kSmallChunksBfs : kSmallChunksSssp);
}

template <bool kBfs>
int small_level_loop(gphi_graph *gr, uint32_t src, gphi_stats *st, uint32_t *steps)
{
	gphi_ctx *ctx = gr->ctx;
	const DevGraph &G = gr->g;
	hipStream_t s = ctx->stream;
	LevelBoard *board = ctx->h_board;
	Trav t;
	t.n = G.n, t.n_pad = G.n_pad, t.n_words = G.n_words, t.W = G.W, t.side = G.side;
	t.threshold = (uint32_t)G.m / ctx->t_ratio;
	t.win_rows = dense_window_rows(G.W);
	t.nchunks = (uint32_t)G.nchunks;
	t.row_off = G.row_off, t.cols = G.cols, t.csr_w = G.csr_w, t.deg = G.deg;
	t.heads = G.heads, t.tails = G.tails, t.coo_w = G.coo_w;
	t.heads16 = G.heads16, t.tails16 = G.tails16, t.coo_w8 = G.coo_w8;
	t.meta = G.meta, t.pack = G.pack;
	t.level = gr->level, t.parent = gr->parent, t.dist = gr->dist;
	t.flag = gr->flag, t.visited = gr->visited, t.cur = gr->cur;
	t.row_stamp = gr->row_stamp, t.col_unvis = gr->col_unvis;
	t.qb = gr->queue_bufs();
	t.rec = gr->rec;
	t.board = board;
	// Every block is resident at once.  A block takes runs of chunks, as long
	// as they leave no block with more than a tenth over its share.
	static const unsigned resident[3] = {resident_grid(reinterpret_cast<const void *>(small_expand_kernel<0>)),
	                                     resident_grid(reinterpret_cast<const void *>(small_expand_kernel<1>)),
	                                     resident_grid(reinterpret_cast<const void *>(small_expand_kernel<4>))};
	const unsigned grid = (unsigned)std::min<uint64_t>(resident[kBfs ? 0 : G.coo_w8 ? 1 : 2],
	                                                   std::max<uint64_t>(G.nchunks, 1));
	for (t.run = kDenseRun;; t.run /= 2) {
		const uint32_t nruns = (t.nchunks + t.run - 1) / t.run;
		t.slots = (nruns + grid - 1) / grid * t.run;
		if (t.run == 1 || (uint64_t)t.slots * grid <= t.nchunks + t.nchunks / 10) break;
	}
	if (t.slots > kBlock) return set_error(ctx, GPHI_E_STATE, "%u chunks exceed the small level loop", t.nchunks);
	const unsigned adv = G.n_pad <= kAdvanceNarrow ? 256 : 1024, nblk = G.n_pad / (adv * kLaneVerts);
	*(volatile unsigned long long *)&board->progress = 0;
	const uint64_t items = std::max<uint64_t>({G.n_pad / (kBfs ? 16 : 1), G.n_words, G.side});
	small_init_kernel<kBfs><<<(unsigned)std::min<uint64_t>((items + kBlock - 1) / kBlock, 2048), kBlock, 0, s>>>(t, src);
	uint32_t enq = 0, seen = 0, idle = 0;
	for (;;) {
		for (; enq <= seen + kAhead; ++enq) {
			if (kBfs)
				small_expand_kernel<0><<<grid, kBlock, 0, s>>>(t, enq);
			else if (G.coo_w8)
				small_expand_kernel<1><<<grid, kBlock, 0, s>>>(t, enq);
			else
				small_expand_kernel<4><<<grid, kBlock, 0, s>>>(t, enq);
			if (adv == 256)
				small_advance_kernel<kBfs, 256><<<nblk, 256, 0, s>>>(t, enq);
			else
				small_advance_kernel<kBfs, 1024><<<nblk, 1024, 0, s>>>(t, enq);
		}
		GPHI_HIP(ctx, hipGetLastError());
		// the level the device has started last; the stream is looked at now
		// and then, so that an error on the device ends the wait
		unsigned long long p;
		for (uint32_t spin = 0;; ++spin) {
			p = __atomic_load_n(&board->progress, __ATOMIC_ACQUIRE);
			if ((p & 1ull) || (p >> 1) > seen + 1) break;
			if (spin % 4096 == 4095) {
				const hipError_t e = hipStreamQuery(s);
				if (e != hipSuccess && e != hipErrorNotReady)
					return hip_fail(ctx, e, "level loop", __FILE__, __LINE__);
				// an idle stream has published every enqueued level
				if (e == hipSuccess && ++idle > 2) return set_error(ctx, GPHI_E_STATE, "level loop made no progress");
			}
			__builtin_ia32_pause();
		}
		idle = 0;
		if (p & 1ull) break;
		seen = (uint32_t)(p >> 1) - 1;
	}
	if (steps) *steps = board->levels;
	if (st) {
		const uint32_t ns = std::min<uint32_t>(board->levels, GPHI_MAX_STEPS);
		st->steps = ns;
		for (uint32_t k = 0; k < ns; ++k) {
			const uint4 r = board->trace[k];
			st->dir[k] = r.x;
			st->fsize[k] = r.y;
			st->fdeg[k] = r.z;
			st->chunks[k] = r.w;
		}
		st->reached = board->reached;
		st->edges_traversed = board->traversed;
		st->total_ms = (float)((double)(board->t_end - board->t_begin) / ctx->wall_clock_khz);
	}
	return GPHI_OK;
}
template int small_level_loop<true>(gphi_graph *, uint32_t, gphi_stats *, uint32_t *);
template int small_level_loop<false>(gphi_graph *, uint32_t, gphi_stats *, uint32_t *);

}  // namespace gphi
