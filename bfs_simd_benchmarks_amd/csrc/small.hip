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
	const unsigned adv = advance_threads(G.n_pad), nblk = advance_blocks(G.n_pad);
	reset_board(board);
	const uint64_t items = std::max<uint64_t>({G.n_pad / (kBfs ? 16 : 1), G.n_words, G.side});
	small_init_kernel<kBfs><<<(unsigned)std::min<uint64_t>((items + kBlock - 1) / kBlock, 2048), kBlock, 0, s>>>(t, src);
	const int rc = follow_levels(ctx, [&](uint32_t level) {
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
	return GPHI_OK;
}
template int small_level_loop<true>(gphi_graph *, uint32_t, gphi_stats *, uint32_t *);
template int small_level_loop<false>(gphi_graph *, uint32_t, gphi_stats *, uint32_t *);

}  // namespace gphi
