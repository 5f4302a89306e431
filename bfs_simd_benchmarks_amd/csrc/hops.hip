// hops.hip -- hop relaxation over the tile arrays.
//
// apps/bellman-ford_simd/bellman-ford.cpp:129-191,291-392: sweeps of dist[t] =
// min(dist[t], dist[h] + 1) over every edge; a sweep that lowers nothing is the
// fixpoint, where further sweeps would change nothing.
//
// A sweep over every edge is bound by its distance lookups, two per edge, at
// random in an array that does not fit an XCD's L2 (65M edges: 223 us, where
// their bytes take 55).  An edge can lower its tail only if its head was
// lowered since the edge was looked at last, that is in the sweep before or,
// by a block ahead of this one, in this sweep; so a vertex carries the low
// byte of the sweep it was lowered in, and a tile row the sweep:
//   - a chunk none of whose head rows was lowered is skipped;
//   - the distances of a chunk's head rows come from LDS, loaded once for the
//     run of chunks that share them, with the heads that were not lowered
//     marked there, so that an edge costs one LDS read, and a lookup of its
//     tail only behind a lowered head.
// On rmat22 (65M edges, 7 sweeps) the sweeps take 9, 44, 315, 155, 12, 7 and 4
// us, all of them 1.79 ms before; the two large ones are bound by the tails'
// lookups, atomics and stamps.
// The order within a sweep is free, as it was: a block sees what other blocks
// lowered before it loads its rows, and the rest in the next sweep.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>

#include "levels.h"

namespace gphi {

namespace {

constexpr uint32_t kHopInf = INT_MAX - 2;   // unreached, as bellman-ford.cpp's init
constexpr uint32_t kHopSkip = UINT32_MAX;   // LDS: head not lowered lately
constexpr uint32_t kHopWin = 4096;          // vertices of an LDS row window (16 KiB)
constexpr uint32_t kHopRun = 2;             // consecutive chunks a block takes at a time (they share rows)
static_assert(kBlock % kHopRun == 0, "whole runs per round");

struct Hops {
	uint32_t n, n_pad, W, nchunks;
	const uint32_t *heads, *tails;
	const uint16_t *heads16, *tails16;
	const ChunkMeta *meta;
	const ChunkPack *pack;      // null without the 16-bit forms
	uint32_t *dist;
	uint32_t *row_sweep;        // sweep + 1 a row's vertex was lowered in last, 0 never
	uint8_t *stamp;             // its low byte, per vertex
	LevelRec *rec;              // ring over the sweeps; fsize: the sweep lowered something
	LevelBoard *board;
};

__global__ __launch_bounds__(kBlock) void hop_init_kernel(Hops t, uint32_t side, uint32_t src)
{
	const uint32_t stride = gridDim.x * kBlock, i0 = blockIdx.x * kBlock + threadIdx.x;
	if (i0 == 0) t.board->t_begin = wall_clock64();
	for (uint32_t i = i0; i < t.n_pad; i += stride) t.dist[i] = i == src ? 0u : kHopInf;
	// sweep 0 lowered the source.  (A byte left from 256 sweeps ago, or from
	// here, may match a later sweep's: its edges are then looked at again.)
	for (uint32_t i = i0; i < t.n_pad / 4; i += stride)
		reinterpret_cast<uint32_t *>(t.stamp)[i] = i == src / 4 ? 1u << (8 * (src % 4)) : 0u;
	for (uint32_t i = i0; i < side; i += stride) t.row_sweep[i] = i == src / t.W ? 1u : 0u;
	if (i0 < kLevelRing) {
		LevelRec r = {};
		r.fsize = i0 == 0;
		t.rec[i0] = r;
	}
}

// a head row of the chunk was lowered in sweep k - 1 or, as far as this block
// sees, k; more than 16 rows count as lowered
__device__ __forceinline__ bool rows_lowered(const Hops &t, const ChunkMeta &md, uint32_t k)
{
	if (md.row_lo > md.row_hi) return false;
	const uint32_t nr = md.row_hi - md.row_lo + 1;
	bool any = nr > 16;
#pragma unroll
	for (uint32_t i = 0; i < 16; ++i)
		any |= nr <= 16 && i < nr &&
		       __hip_atomic_load(t.row_sweep + md.row_lo + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= k;
	return any;
}

// Sweep k = 1, 2, ...; the one after the last of max, or after one that
// lowered nothing, only reports the end.
__global__ __launch_bounds__(kBlock) void hop_sweep_kernel(Hops t, uint32_t k, uint32_t max)
{
	__shared__ uint4 s_head4[kHopWin / 4];
	__shared__ uint32_t s_list[kBlock];
	__shared__ uint32_t s_cnt[kBlock / 64];
	LevelRec *mine = t.rec + k % kLevelRing;
	if (k - 1 > max) return;
	const bool fix = t.rec[(k - 1) % kLevelRing].fsize == 0;  // the sweep before lowered nothing
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		LevelBoard *b = t.board;
		if (!fix && k <= max) {
			*(t.rec + (k + kLevelRing / 2) % kLevelRing) = LevelRec{};
			__hip_atomic_store(&b->progress, (unsigned long long)k << 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
		} else if (k < 2 || t.rec[(k - 2) % kLevelRing].fsize) {  // the first to see it
			b->levels = k - 1;
			b->t_end = wall_clock64();
			__hip_atomic_store(&b->progress, (unsigned long long)k << 1 | 1ull, __ATOMIC_RELEASE,
			                   __HIP_MEMORY_SCOPE_SYSTEM);
		}
	}
	if (fix || k > max) return;
	const uint32_t *s_head = reinterpret_cast<const uint32_t *>(s_head4);
	const uint32_t tid = threadIdx.x, wid = tid >> 6;
	const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)wid);
	const uint8_t before = (uint8_t)k, now = (uint8_t)(k + 1);  // stamps of sweeps k - 1 and k
	bool lowered = false;
	// rounds of kBlock chunks: this block's runs of kHopRun consecutive ones,
	// run j of the round at run (round + j) * gridDim + block
	const uint32_t nruns = (t.nchunks + kHopRun - 1) / kHopRun;
	for (uint32_t j0 = 0; (uint64_t)j0 * gridDim.x + blockIdx.x < nruns; j0 += kBlock / kHopRun) {
		const uint64_t run = (uint64_t)(j0 + tid / kHopRun) * gridDim.x + blockIdx.x;
		const uint32_t cand = (uint32_t)run * kHopRun + tid % kHopRun;
		const bool live = run < nruns && cand < t.nchunks && rows_lowered(t, t.meta[cand], k);
		const unsigned long long m = __ballot(live);
		__syncthreads();  // the list of the round before was read
		if (lane_id() == 0) s_cnt[wid] = (uint32_t)__popcll(m);
		__syncthreads();
		uint32_t at = 0, total = 0;
		for (uint32_t w = 0; w < kBlock / 64; ++w) {
			if (w < wid) at += s_cnt[w];
			total += s_cnt[w];
		}
		if (live) s_list[at + __popcll(m & ((1ull << lane_id()) - 1ull))] = cand;
		__syncthreads();
		total = (uint32_t)__builtin_amdgcn_readfirstlane((int)total);
		if (!total) continue;
		const LdsChunkList lst{s_list};
		uint32_t win_base = UINT32_MAX, win_len = 0;  // vertices held in s_head (block-uniform)
		uint32_t c = lst(0);
		PackSlot pk = t.pack ? pack_slot(t.pack, c, wv) : PackSlot{0u, 0u, 0u, 0u};
		uint32_t h[8];
		load_edges(pk.flags & 1u, t.heads, t.heads16, c, tid, true, true, h);
		for (uint32_t i = 0; i < total; ++i) {
			const ChunkMeta md = t.meta[c];
			// the chunk's rows, from a multiple of 4 vertices on
			const uint64_t b0 = (uint64_t)md.row_lo * t.W & ~3ull, b1 = min((uint64_t)(md.row_hi + 1) * t.W, (uint64_t)t.n);
			const bool inw = b1 - b0 <= kHopWin;
			if (inw && ((uint32_t)b0 != win_base || (uint32_t)(b1 - b0) > win_len)) {
				__syncthreads();  // every wave is done with the rows before
				win_base = (uint32_t)b0;
				win_len = (uint32_t)(b1 - b0);
				// 4 vertices per lane and load (the arrays are padded past n)
				for (uint32_t q = tid; q < (win_len + 3) / 4; q += kBlock) {
					const uint4 d = *reinterpret_cast<const uint4 *>(t.dist + win_base + 4 * q);
					const uint32_t st = *reinterpret_cast<const uint32_t *>(t.stamp + win_base + 4 * q);
					const uint32_t dd[4] = {d.x, d.y, d.z, d.w};
					uint32_t x[4];
#pragma unroll
					for (int i = 0; i < 4; ++i) {
						const uint8_t b = (uint8_t)(st >> (8 * i));
						x[i] = b == before || b == now ? dd[i] : kHopSkip;
					}
					s_head4[q] = make_uint4(x[0], x[1], x[2], x[3]);
				}
				__syncthreads();
			}
			decode_edges(pk.flags & 1u, pk.hbase, pk.hbase, h);
			uint32_t hd[8];
			if (inw) {
#pragma unroll
				for (int j = 0; j < 8; ++j) {
					const uint32_t x = h[j] - win_base;  // a padding edge (head n) falls outside
					hd[j] = h[j] < t.n && x < win_len ? s_head[x] : kHopSkip;
				}
			} else {
				uint8_t st[8];
#pragma unroll
				for (int j = 0; j < 8; ++j) {
					const uint32_t v = h[j] < t.n ? h[j] : 0u;
					st[j] = t.stamp[v];
					hd[j] = t.dist[v];
				}
#pragma unroll
				for (int j = 0; j < 8; ++j)
					if (h[j] >= t.n || (st[j] != before && st[j] != now)) hd[j] = kHopSkip;
			}
			uint32_t need = 0;
#pragma unroll
			for (int j = 0; j < 8; ++j) need |= (hd[j] != kHopSkip ? 1u : 0u) << j;
			// this chunk's tails, then the next one's heads, which arrive behind them
			uint32_t tl[8], dt[8];
			load_edges(pk.flags & 2u, t.tails, t.tails16, c, tid, need & 0x0Fu, need & 0xF0u, tl);
			const uint32_t cn = i + 1 < total ? lst(i + 1) : c;
			const PackSlot pn = t.pack ? pack_slot(t.pack, cn, wv) : PackSlot{0u, 0u, 0u, 0u};
			load_edges(pn.flags & 1u, t.heads, t.heads16, cn, tid, true, true, h);
			decode_edges(pk.flags & 2u, pk.tb0, pk.tb1, tl);
#pragma unroll
			for (int j = 0; j < 8; ++j) dt[j] = t.dist[(need >> j) & 1u ? tl[j] : 0u];
#pragma unroll
			for (int j = 0; j < 8; ++j) {
				// a tail lowered below the dist[t] read was lowered in this sweep
				if (((need >> j) & 1u) && (int32_t)(hd[j] + 1) < (int32_t)dt[j]) {
					atomicMin(t.dist + tl[j], hd[j] + 1);
					t.stamp[tl[j]] = now;
					t.row_sweep[tl[j] / t.W] = k + 1;
					lowered = true;
				}
			}
			c = cn;
			pk = pn;
		}
	}
	// a plain store of 1, not an atomic: every writer stores the same value
	if (__ballot(lowered) && lane_id() == 0) mine->fsize = 1u;
}

}  // namespace

int run_bellman_ford(gphi_graph *gr, uint32_t src, uint32_t max_sweeps, uint32_t *dist, uint32_t *sweeps_run,
                     float *ms)
{
	gphi_ctx *ctx = gr->ctx;
	DevGraph &G = gr->g;
	if (src >= G.n) return set_error(ctx, GPHI_E_RANGE, "source %u >= N %u", src, G.n);
	if (!G.has_tiles) return set_error(ctx, GPHI_E_STATE, "graph has no tile arrays");
	hipStream_t s = ctx->stream;
	int rc;
	if (!gr->dist && (rc = dmalloc(ctx, (void **)&gr->dist, (size_t)G.n_pad * 4, nullptr))) return rc;
	const size_t ring = kLevelRing * sizeof(LevelRec), rows = ((size_t)G.side * 4 + 255) / 256 * 256;
	if (!gr->hop && (rc = dmalloc(ctx, (void **)&gr->hop, ring + rows + G.n_pad, nullptr))) return rc;
	Hops t = {};
	t.n = G.n, t.n_pad = G.n_pad, t.W = G.W, t.nchunks = (uint32_t)G.nchunks;
	t.heads = G.heads, t.tails = G.tails, t.heads16 = G.heads16, t.tails16 = G.tails16;
	t.meta = G.meta, t.pack = G.heads16 ? G.pack : nullptr;
	t.dist = gr->dist;
	t.rec = reinterpret_cast<LevelRec *>(gr->hop);
	t.row_sweep = reinterpret_cast<uint32_t *>(gr->hop + ring);
	t.stamp = gr->hop + ring + rows;
	t.board = ctx->h_board;
	static const unsigned resident = resident_grid(reinterpret_cast<const void *>(hop_sweep_kernel));
	const unsigned grid = (unsigned)std::min<uint64_t>(resident, std::max<uint64_t>((G.nchunks + kHopRun - 1) / kHopRun, 1));
	if ((rc = reset_board(ctx))) return rc;
	hop_init_kernel<<<(unsigned)std::min<uint32_t>(G.n_pad / kBlock, 4096), kBlock, 0, s>>>(t, G.side, src);
	rc = follow_levels(ctx, [&](uint32_t i) {
		hop_sweep_kernel<<<grid, kBlock, 0, s>>>(t, i + 1, max_sweeps);
		return GPHI_OK;
	});
	if (rc) return rc;
	if (dist && (rc = out_dist(ctx, gr->dist, kHopInf, G.n, G.n_pad, dist))) return rc;
	if (ms) *ms = board_ms(ctx);
	if (sweeps_run) *sweeps_run = ctx->h_board->levels;
	return GPHI_OK;
}

}  // namespace gphi
