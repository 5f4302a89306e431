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
// How the direction is decided and the host follows: levels.h.
//
// Reference: the level loop of apps/bfs_simd/bfs.cpp:795-910 and
// apps/sssp_simd/sssp.cpp:1000-1100.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstring>

#include "levels.h"

namespace gphi {

namespace {

// What the kernels of one traversal share.
struct Trav : Frontier {
	uint32_t n, n_words, side, win_rows;
	uint32_t nchunks, run, slots;  // chunks per run, chunks tested per block
	const uint32_t *row_off, *cols, *csr_w;
	const uint32_t *heads, *tails, *coo_w;
	const uint16_t *heads16, *tails16;
	const uint8_t *coo_w8;
	const ChunkMeta *meta;
	const ChunkPack *pack;
	int32_t *parent;
	uint32_t *dist;
};

// All state of a traversal set up for its source, in one launch: every word
// is written once, with the source's part in it.
template <bool kBfs>
__global__ __launch_bounds__(kBlock) void small_init_kernel(Trav t, uint32_t src)
{
	const uint32_t d = t.deg[src];
	const uint32_t nf = t.n_pad / 16, ntile = (d + kSparseTile - 1) / kSparseTile;
	const uint32_t stride = gridDim.x * kBlock, i0 = blockIdx.x * kBlock + threadIdx.x;
	if (i0 == 0) t.board->t_begin = wall_clock64();
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
				nd[r] = on[r] ? path_sum(t.dist[uu[r]], t.csr_w[ix[r]]) : UINT32_MAX;
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
	const Step st = step_of(t, level);
	const bool dense = level > 0 && st.dense;  // the first step is sparse (apps/bfs_simd/bfs.cpp:807)
	if (blockIdx.x == 0 && threadIdx.x == 0) publish_level(t, level, st.fsize, st.fdeg, dense);
	if (st.fsize == 0) return;
	if (!dense) {
		small_push<kBfs>(reinterpret_cast<uint32_t *>(s_mem), t, level, st.qsize, st.fdeg);
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

template <bool kBfs, uint32_t kThreads>
__global__ __launch_bounds__(kThreads) void small_advance_kernel(Frontier t, uint32_t level)
{
	advance_block<kBfs, kThreads>(t, level);
}

// ---------------------------------------------------------------------------
// tiny graphs: the whole traversal in one block
// ---------------------------------------------------------------------------
// With up to kTinyVerts vertices and kTinyChunks chunks of edges, a level's
// work is smaller than the two launches it takes.  Here one block of 1024
// threads runs all levels: frontier, visited set, queue and (SSSP) distances
// live in LDS, a thread keeps the degrees and CSR offsets of its 8 vertices in
// registers, and only edges, parents and levels cross to memory.  The steps,
// the direction rule and the chunks a dense step takes are those of the
// two-launch loop.  Whole calls, against that loop: BFS 89 -> 45 us at 1024
// vertices (6 chunks), 106 -> 78 at 8000 (29), SSSP 175 -> 77 and 187 -> 155; past
// 32 chunks the edges are more than one CU should read.
struct TinyShared {
	uint32_t cur[kTinyVerts / 32], hot[kTinyVerts / 32];  // frontier; its vertices with out-edges
	uint32_t next[kTinyVerts / 32];                       // frontier of the next step
	uint32_t visited[kTinyVerts / 32];                    // BFS
	uint32_t off[kTinyVerts], base[kTinyVerts];           // queue: degree prefix, CSR offset
	uint16_t queue[kTinyVerts];
	uint16_t chunks[kTinyChunks];
	uint32_t red[3][kTinyThreads / 64];
	uint32_t nchunks;
};

// some vertex of [a, b) has its bit set in `bits` (cleared, with flip ~0), by one wavefront
__device__ __forceinline__ bool any_bit(const uint32_t *bits, uint32_t flip, uint32_t a, uint32_t b, uint32_t lane)
{
	bool any = false;
	for (uint32_t w = a / 32 + lane; w <= (b - 1) / 32; w += 64) {
		uint32_t x = bits[w] ^ flip;
		if (w == a / 32) x &= ~0u << (a % 32);
		if (w == (b - 1) / 32) x &= ~0u >> (31 - (b - 1) % 32);
		any |= x != 0;
	}
	return __ballot(any) != 0;
}

template <int kWeights>
__global__ __launch_bounds__(kTinyThreads) void tiny_kernel(Trav t, uint32_t src)
{
	constexpr bool kBfs = kWeights == 0;
	constexpr uint32_t kOwn = kTinyVerts / kTinyThreads;
	static_assert(kOwn == 8, "a thread's vertices are a byte of the bitmaps");
	__shared__ TinyShared s;
	__shared__ uint32_t s_dist[kBfs ? 1 : kTinyVerts];
	const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, v0 = tid * kOwn;
	LevelBoard *board = t.board;
	if (tid == 0) board->t_begin = wall_clock64();
	uint32_t d[kOwn], base[kOwn];
#pragma unroll
	for (uint32_t k = 0; k < kOwn; ++k) {
		const bool in = v0 + k < t.n;
		d[k] = in ? t.deg[v0 + k] : 0u;
		base[k] = in ? t.row_off[v0 + k] : 0u;
		if (!kBfs) s_dist[v0 + k] = v0 + k == src ? 0u : (uint32_t)INT_MAX;
	}
	uint8_t *cur8 = reinterpret_cast<uint8_t *>(s.cur), *hot8 = reinterpret_cast<uint8_t *>(s.hot);
	uint8_t *next8 = reinterpret_cast<uint8_t *>(s.next), *vis8 = reinterpret_cast<uint8_t *>(s.visited);
	next8[tid] = vis8[tid] = src / kOwn == tid ? (uint8_t)(1u << (src % kOwn)) : 0;
	if (kBfs && tid == 0) {
		t.level[src] = 0;
		t.parent[src] = (int32_t)src;
	}
	unsigned long long reached = 0, traversed = 0;
	uint32_t level = 0;
	bool over = false;
	for (;; ++level) {
		__syncthreads();
		// the next frontier becomes the current one; its queue
		const uint32_t bits = next8[tid];
		uint32_t q = 0, dsum = 0, hot = 0;
#pragma unroll
		for (uint32_t k = 0; k < kOwn; ++k)
			if (((bits >> k) & 1u) && d[k]) {
				++q;
				dsum += d[k];
				hot |= 1u << k;
			}
		cur8[tid] = (uint8_t)bits;
		hot8[tid] = (uint8_t)hot;
		next8[tid] = 0;
		uint32_t qtot, dtot;
		uint32_t pos = wave_excl_scan(q, &qtot), off = wave_excl_scan(dsum, &dtot);
		const uint32_t ftot = wave_sum((uint32_t)__popc(bits));
		if (lane == 0) {
			s.red[0][wid] = ftot;
			s.red[1][wid] = qtot;
			s.red[2][wid] = dtot;
		}
		if (tid == 0) s.nchunks = 0;
		__syncthreads();
		uint32_t fsize = 0, qsize = 0, fdeg = 0;
		for (uint32_t k = 0; k < kTinyThreads / 64; ++k) {
			if (k < wid) {
				pos += s.red[1][k];
				off += s.red[2][k];
			}
			fsize += s.red[0][k];
			qsize += s.red[1][k];
			fdeg += s.red[2][k];
		}
		over = fsize != 0 && level > level_limit(t.n);
		if (fsize == 0 || over) break;  // uniform
		reached += fsize;
		traversed += fdeg;
#pragma unroll
		for (uint32_t k = 0; k < kOwn; ++k)
			if ((hot >> k) & 1u) {
				s.queue[pos] = (uint16_t)(v0 + k);
				s.off[pos] = off;
				s.base[pos] = base[k];
				++pos;
				off += d[k];
			}
		const bool dense = level > 0 && dense_step(fsize, fdeg, t.threshold);  // the first step is sparse
		uint32_t nlive = 0;
		// edge u -> v, its weight from w
		auto relax = [&](uint32_t u, uint32_t v, uint32_t w) {
			const uint32_t bit = 1u << (v & 31);
			if (kBfs) {
				if ((s.visited[v >> 5] & bit) || (atomicOr(&s.visited[v >> 5], bit) & bit)) return;
				t.parent[v] = (int32_t)u;
				t.level[v] = (int32_t)level + 1;
				atomicOr(&s.next[v >> 5], bit);
			} else {
				const uint32_t nd = path_sum(s_dist[u], w);
				if (nd < s_dist[v] && nd < atomicMin(&s_dist[v], nd)) atomicOr(&s.next[v >> 5], bit);
			}
		};
		if (!dense) {
			__syncthreads();
			// the frontier's edges, one per thread and round
			for (uint32_t e = tid; e < fdeg; e += kTinyThreads) {
				uint32_t a = 0, b = qsize;  // last entry with off <= e
				while (b - a > 1) {
					const uint32_t mid = (a + b) >> 1;
					if (s.off[mid] <= e)
						a = mid;
					else
						b = mid;
				}
				const uint32_t x = s.base[a] + (e - s.off[a]);
				relax(s.queue[a], t.cols[x], kBfs ? 0u : t.csr_w[x]);
			}
		} else {
			// the live chunks, a wavefront per chunk
			for (uint32_t c = wid; c < t.nchunks; c += kTinyThreads / 64) {
				const ChunkMeta md = t.meta[c];
				if (md.row_lo > md.row_hi) continue;
				bool live = md.row_hi - md.row_lo >= 16 ||
				            any_bit(s.hot, 0u, md.row_lo * t.W, (uint32_t)min((uint64_t)(md.row_hi + 1) * t.W, (uint64_t)t.n), lane);
				if (kBfs && live)
					live = md.col_hi - md.col_lo >= 16 ||
					       any_bit(s.visited, ~0u, md.col_lo * t.W, (uint32_t)min((uint64_t)(md.col_hi + 1) * t.W, (uint64_t)t.n), lane);
				if (live && lane == 0) s.chunks[atomicAdd(&s.nchunks, 1u)] = (uint16_t)c;
			}
			__syncthreads();
			nlive = s.nchunks;
			// 4 edges per thread and round; padding edges have head n
			constexpr uint32_t kQuads = kChunk / 4;
			for (uint32_t x = tid; x < nlive * kQuads; x += kTinyThreads) {
				const uint32_t at = s.chunks[x / kQuads] * kQuads + x % kQuads;
				const uint4 h4 = reinterpret_cast<const uint4 *>(t.heads)[at];
				const uint4 t4 = reinterpret_cast<const uint4 *>(t.tails)[at];
				const uint32_t h[4] = {h4.x, h4.y, h4.z, h4.w}, v[4] = {t4.x, t4.y, t4.z, t4.w};
				uint32_t w[4] = {0u, 0u, 0u, 0u};
				if (kWeights == 1) {
					const uint32_t w4 = reinterpret_cast<const uint32_t *>(t.coo_w8)[at];
					w[0] = w4 & 0xFFu, w[1] = (w4 >> 8) & 0xFFu, w[2] = (w4 >> 16) & 0xFFu, w[3] = w4 >> 24;
				} else if (kWeights == 4) {
					const uint4 w4 = reinterpret_cast<const uint4 *>(t.coo_w)[at];
					w[0] = w4.x, w[1] = w4.y, w[2] = w4.z, w[3] = w4.w;
				}
#pragma unroll
				for (int j = 0; j < 4; ++j)
					if (h[j] < t.n && ((s.cur[h[j] >> 5] >> (h[j] & 31)) & 1u)) relax(h[j], v[j], w[j]);
			}
		}
		if (tid == 0 && level < GPHI_MAX_STEPS) {
			uint4 *tr = board->trace + level;
			tr->x = dense;
			tr->y = fsize;
			tr->z = fdeg;
			tr->w = nlive;
		}
	}
	// what the two-launch loop leaves in memory: state bytes, or distances
	if (kBfs) {
		const uint32_t b = vis8[tid];
		uint2 f = make_uint2(0, 0);
#pragma unroll
		for (int k = 0; k < 4; ++k) {
			f.x |= (((b >> k) & 1u) ? (uint32_t)kVisited : 0u) << (8 * k);
			f.y |= (((b >> (4 + k)) & 1u) ? (uint32_t)kVisited : 0u) << (8 * k);
		}
		if (v0 < t.n_pad) reinterpret_cast<uint2 *>(t.flag)[tid] = f;
	} else {
#pragma unroll
		for (uint32_t k = 0; k < kOwn; ++k)
			if (v0 + k < t.n_pad) t.dist[v0 + k] = s_dist[v0 + k];
	}
	if (tid == 0) {
		board->reached = reached;
		board->traversed = traversed;
		board->levels = level;
		board->err = over;
		board->t_end = wall_clock64();
		__hip_atomic_store(&board->progress, 3ull, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
	}
}

}  // namespace

// blocks of small_expand_kernel that are resident at once (bfs, 1-byte and 32-bit weights)
static unsigned expand_resident(const DevGraph &G, bool bfs)
{
	static const unsigned resident[3] = {resident_grid(reinterpret_cast<const void *>(small_expand_kernel<0>)),
	                                     resident_grid(reinterpret_cast<const void *>(small_expand_kernel<1>)),
	                                     resident_grid(reinterpret_cast<const void *>(small_expand_kernel<4>))};
	return resident[bfs ? 0 : G.coo_w8 ? 1 : 2];
}

// whether the loop is the faster one (kSmallVerts) and a block's list holds its
// share of the chunks (on a card cut into partitions it may not)
bool small_graph(const DevGraph &G, bool bfs)
{
	return G.n <= kSmallVerts && G.nchunks <= (bfs ? kSmallChunksBfs : kSmallChunksSssp) &&
	       G.nchunks <= (uint64_t)expand_resident(G, bfs) * kBlock;
}

static void small_stats(const gphi_ctx *ctx, gphi_stats *st, uint32_t *steps)
{
	const LevelBoard *board = ctx->h_board;
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
		st->total_ms = board_ms(ctx);
	}
}

template <bool kBfs>
int small_level_loop(gphi_graph *gr, uint32_t src, gphi_stats *st, uint32_t *steps)
{
	gphi_ctx *ctx = gr->ctx;
	const DevGraph &G = gr->g;
	hipStream_t s = ctx->stream;
	LevelBoard *board = ctx->h_board;
	Trav t = {};
	static_cast<Frontier &>(t) = make_frontier(gr, (uint32_t)G.m / ctx->t_ratio);
	t.n = G.n, t.n_words = G.n_words, t.side = G.side;
	t.win_rows = dense_window_rows(G.W);
	t.nchunks = (uint32_t)G.nchunks;
	t.row_off = G.row_off, t.cols = G.cols, t.csr_w = G.csr_w;
	t.heads = G.heads, t.tails = G.tails, t.coo_w = G.coo_w;
	t.heads16 = G.heads16, t.tails16 = G.tails16, t.coo_w8 = G.coo_w8;
	t.meta = G.meta, t.pack = G.pack;
	t.parent = gr->parent, t.dist = gr->dist;
	int rc = reset_board(ctx);
	if (rc) return rc;
	if (G.n <= kTinyVerts && G.nchunks <= kTinyChunks) {
		if (kBfs)
			tiny_kernel<0><<<1, kTinyThreads, 0, s>>>(t, src);
		else if (G.coo_w8)
			tiny_kernel<1><<<1, kTinyThreads, 0, s>>>(t, src);
		else
			tiny_kernel<4><<<1, kTinyThreads, 0, s>>>(t, src);
		GPHI_HIP(ctx, hipGetLastError());
		unsigned long long p;
		if ((rc = wait_progress(ctx, &board->progress, 0, &p))) return rc;
		ctx->board_busy = false;
		if (board->err) return set_error(ctx, GPHI_E_STATE, "frontier loop did not terminate");
		small_stats(ctx, st, steps);
		return GPHI_OK;
	}
	// Every block is resident at once.  A block takes runs of chunks, as long
	// as they leave no block with more than a tenth over its share.
	const unsigned grid = (unsigned)std::min<uint64_t>(expand_resident(G, kBfs), std::max<uint64_t>(G.nchunks, 1));
	for (t.run = kDenseRun;; t.run /= 2) {
		const uint32_t nruns = (t.nchunks + t.run - 1) / t.run;
		t.slots = (nruns + grid - 1) / grid * t.run;
		if (t.run == 1 || (t.slots <= kBlock && (uint64_t)t.slots * grid <= t.nchunks + t.nchunks / 10)) break;
	}
	const unsigned adv = advance_threads(G.n_pad), nblk = advance_blocks(G.n_pad);
	const uint64_t items = std::max<uint64_t>({G.n_pad / (kBfs ? 16 : 1), G.n_words, G.side});
	small_init_kernel<kBfs><<<(unsigned)std::min<uint64_t>((items + kBlock - 1) / kBlock, 2048), kBlock, 0, s>>>(t, src);
	rc = follow_levels(ctx, [&](uint32_t level) -> int {
		if (level > level_limit(G.n) + kAhead) return set_error(ctx, GPHI_E_STATE, "frontier loop did not terminate");
		if (kBfs)
			small_expand_kernel<0><<<grid, kBlock, 0, s>>>(t, level);
		else if (G.coo_w8)
			small_expand_kernel<1><<<grid, kBlock, 0, s>>>(t, level);
		else
			small_expand_kernel<4><<<grid, kBlock, 0, s>>>(t, level);
		if (adv == 256)
			small_advance_kernel<kBfs, 256><<<nblk, 256, 0, s>>>(t, level);
		else
			small_advance_kernel<kBfs, 1024><<<nblk, 1024, 0, s>>>(t, level);
		return GPHI_OK;
	});
	if (rc) return rc;
	small_stats(ctx, st, steps);
	return GPHI_OK;
}
template int small_level_loop<true>(gphi_graph *, uint32_t, gphi_stats *, uint32_t *);
template int small_level_loop<false>(gphi_graph *, uint32_t, gphi_stats *, uint32_t *);

}  // namespace gphi
