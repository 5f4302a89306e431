// sssp_batch.hip -- weighted SSSP from up to 16 sources in one traversal.
//
// The label-correcting relaxation of apps/sssp_simd/sssp.cpp (dist[t] =
// min(dist[t], dist[h] + w) over the frontier's edges, the frontier being the
// vertices whose distance dropped in the last step; :968-1100) run for k
// sources at once.  Each vertex holds 16 distances side by side (64 bytes, one
// sector), so a frontier edge reads its head's and its tail's distances with
// one random access each, for all sources, where k single-source runs would
// make k of each.  The frontier is the union over the sources; a step relaxes
// every source's distance along every union-frontier edge (a source whose
// distance at the head did not drop relaxes to no effect), and the traversal
// ends when no distance drops.  Label correction reaches the unique shortest
// distances whatever the order of the relaxations, so each row equals that
// source's single-source result (and Dijkstra's).
//
// The level loop is that of levels.h, two launches per level (expand,
// advance; state byte 1 = some distance dropped), with a direction rule on the
// union frontier of its own (|F| + sum deg > M / 2, see kSsspBatchDenseDiv).
// A sparse step is the CSR push over the union queue.  A dense step is a pull
// over the in-edges and their weights (build_in_weights), skipping heads
// outside the frontier bitmap, so that a tail's 16 distances take one write,
// not an atomic per improved source; vertices of few in-edges and the pieces
// of the others share the launch, the pieces first.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "levels.h"

namespace gphi {

namespace {

constexpr uint32_t kInf = 2147483647u;  // unreached, as sssp.cpp:994-998
constexpr unsigned kSsspGrid = 8192;  // most blocks of the push, and of each pull (grid-stride loops)
// A step is dense when the union frontier's |F| + sum deg(F) exceeds M / 2,
// not M / T_RATIO as in the single-source rule: a push step relaxes 16
// distances per frontier edge with one row gather, while a pull step reads
// every in-edge.  Measured over divisors 20, 5, 4, 2 and 1: 2 is fastest on
// rmat25-ef36 (106 against 112 ms for 16 sources) and on the serving mix's
// rmat22 and rmat24 graphs (6.9 against 7.7 ms, 23.0 against 24.5 ms).
constexpr uint64_t kSsspBatchDenseDiv = 2;

__device__ __forceinline__ void load_row(const uint32_t *__restrict__ dist, uint32_t v, uint32_t (&d)[kSsspBatchMax])
{
	const uint4 *p = reinterpret_cast<const uint4 *>(dist + (uint64_t)v * kSsspBatchMax);
#pragma unroll
	for (uint32_t i = 0; i < kSsspBatchMax / 4; ++i) {
		const uint4 x = p[i];
		d[4 * i] = x.x;
		d[4 * i + 1] = x.y;
		d[4 * i + 2] = x.z;
		d[4 * i + 3] = x.w;
	}
}

// every source's dist[t] = min(dist[t], dist[h] + w); true when one dropped.
// A distance that beats the dist[t] read lowers it with a return-free
// atomicMin, as the single-source sweep does: dist[t] then ends the step below
// a value read during it, so t improved this step.  The sum is taken in 64
// bits: a head unreached by a source (kInf) or a wide weight cannot wrap.
__device__ __forceinline__ bool relax_row(const uint32_t (&dh)[kSsspBatchMax], uint32_t w, uint32_t t,
                                          uint32_t *dist)
{
	uint32_t dt[kSsspBatchMax];
	load_row(dist, t, dt);
	bool better = false;
#pragma unroll
	for (int s = 0; s < (int)kSsspBatchMax; ++s) {
		const uint64_t nd = (uint64_t)dh[s] + w;
		if (dh[s] != kInf && nd < dt[s]) {
			atomicMin(dist + (uint64_t)t * kSsspBatchMax + s, (uint32_t)nd);
			better = true;
		}
	}
	return better;
}

// What the kernels of a traversal share.
struct SsspBatch : Frontier {
	uint32_t n, npieces, heavy_blocks;
	const uint32_t *row_off, *cols, *csr_w, *in_off, *in_src, *w32;
	const uint8_t *w8;
	const uint2 *pieces;
	uint32_t *dist;
};

// all distances kInf, state bytes and frontier bitmap clear, level records set
// for the advance that opens level 0 (that of the level before it, UINT32_MAX)
__global__ __launch_bounds__(kBlock) void ssspb_clear_kernel(SsspBatch t, uint32_t n_words)
{
	const uint64_t stride = (uint64_t)gridDim.x * kBlock;
	const uint64_t i0 = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
	if (i0 == 0) t.board->t_begin = wall_clock64();
	for (uint64_t i = i0; i < (uint64_t)t.n_pad * kSsspBatchMax / 4; i += stride)
		reinterpret_cast<uint4 *>(t.dist)[i] = make_uint4(kInf, kInf, kInf, kInf);
	for (uint64_t i = i0; i < t.n_pad / 16; i += stride) reinterpret_cast<uint4 *>(t.flag)[i] = make_uint4(0, 0, 0, 0);
	for (uint64_t i = i0; i < n_words; i += stride) t.cur[i] = 0;
	if (i0 < kLevelRing) {
		LevelRec r = {};
		if (i0 == UINT32_MAX % kLevelRing) r.fsize = 1;
		t.rec[i0] = r;
	}
}

// source i at slot i: distance 0, in the first frontier
struct SsspSeeds {
	uint32_t src[kSsspBatchMax];
};
__global__ void ssspb_seed_kernel(SsspBatch t, SsspSeeds seeds, uint32_t k)
{
	const uint32_t i = threadIdx.x;
	if (i >= k) return;
	t.dist[(uint64_t)seeds.src[i] * kSsspBatchMax + i] = 0;
	t.flag[seeds.src[i]] = 1;
}

// Sparse step: the edge-balanced CSR push over the union queue (tiles of
// kSparseTile edges from tile_lo, as the single-source push).
__device__ __forceinline__ void push_union(const SsspBatch &t, uint32_t level, const Step &st)
{
	__shared__ uint32_t s_off[kSparseTile + 2];
	__shared__ uint32_t s_u[kSparseTile + 2];
	__shared__ uint32_t s_base[kSparseTile + 2];
	const uint32_t *__restrict__ row_off = t.row_off, *__restrict__ cols = t.cols, *__restrict__ csr_w = t.csr_w;
	uint32_t *dist = t.dist;
	uint8_t *flag = t.flag;
	const uint32_t qsize = st.qsize, qdeg = st.fdeg;
	const uint32_t par = level & 1u;  // the half the advance wrote
	const uint32_t *__restrict__ queue = t.qb.queue + par * t.qb.qstride;
	const uint32_t *__restrict__ qoff = t.qb.qoff + par * t.qb.qstride;
	const uint32_t *__restrict__ tile_lo = t.qb.tile_lo + par * t.qb.tstride;
	const uint32_t ntile = (qdeg + kSparseTile - 1) / kSparseTile;
	for (uint32_t k = blockIdx.x; k < ntile; k += gridDim.x) {
		const uint32_t lo = tile_lo[k];
		uint32_t hi = (k + 1 < ntile) ? tile_lo[k + 1] : qsize - 1;
		if (hi > qsize - 1) hi = qsize - 1;
		const uint32_t cnt = hi - lo + 1;
		for (uint32_t j = threadIdx.x; j < cnt; j += kBlock) {
			const uint32_t u = queue[lo + j];
			s_off[j] = qoff[lo + j];
			s_u[j] = u;
			s_base[j] = row_off[u];
		}
		__syncthreads();
		const uint32_t e0 = k * kSparseTile, e1 = min(e0 + kSparseTile, qdeg);
		for (uint32_t e = e0 + threadIdx.x; e < e1; e += kBlock) {
			uint32_t a = 0, b = cnt;  // largest j with s_off[j] <= e
			while (b - a > 1) {
				const uint32_t mid = (a + b) >> 1;
				if (s_off[mid] <= e)
					a = mid;
				else
					b = mid;
			}
			const uint32_t idx = s_base[a] + (e - s_off[a]);
			const uint32_t v = cols[idx];
			uint32_t du[kSsspBatchMax];
			load_row(dist, s_u[a], du);
			if (relax_row(du, csr_w[idx], v, dist)) flag[v] = 1;
		}
		__syncthreads();
	}
}

// Dense step: a pull over the in-edges.  A tail takes, per source, the
// minimum of dist[h] + w over its in-edges from frontier heads, then lowers
// its own distances where that beats them; no atomics, where a push along
// the tiles makes one per improved (edge, source) pair (15-46 ms per dense
// step at scale 25 against 17 ms for a whole single-source query).  The sums
// are clamped to kInf, which never beats a distance.
constexpr uint32_t kPullRound = 4;  // in-edges per lane whose loads are issued together

template <bool kW8>
__device__ __forceinline__ void pull_edges(uint32_t e, uint32_t e_end, uint32_t stride,
                                           const uint32_t *__restrict__ in_src, const uint32_t *__restrict__ w32,
                                           const uint8_t *__restrict__ w8, const uint32_t *__restrict__ cur,
                                           const uint32_t *dist, uint32_t (&cand)[kSsspBatchMax])
{
	for (; e < e_end; e += kPullRound * stride) {
		uint32_t h[kPullRound], w[kPullRound];
		bool on[kPullRound];
#pragma unroll
		for (uint32_t u = 0; u < kPullRound; ++u) {
			const uint32_t x = e + u * stride;
			on[u] = x < e_end;
			h[u] = on[u] ? in_src[x] : 0u;
			w[u] = on[u] ? (kW8 ? (uint32_t)w8[x] : w32[x]) : 0u;
		}
#pragma unroll
		for (uint32_t u = 0; u < kPullRound; ++u) on[u] = on[u] && ((cur[h[u] >> 5] >> (h[u] & 31)) & 1u);
#pragma unroll
		for (uint32_t u = 0; u < kPullRound; ++u) {
			if (!on[u]) continue;
			uint32_t dh[kSsspBatchMax];
			load_row(dist, h[u], dh);
#pragma unroll
			for (int s = 0; s < (int)kSsspBatchMax; ++s) {
				const uint64_t nd = dh[s] == kInf ? (uint64_t)kInf : (uint64_t)dh[s] + w[u];
				const uint32_t c = nd < kInf ? (uint32_t)nd : kInf;
				cand[s] = c < cand[s] ? c : cand[s];
			}
		}
	}
}

// vertices with 1..kPullLight in-edges, a lane each (it owns the vertex:
// plain stores)
template <bool kW8>
__device__ __forceinline__ void pull_light(const SsspBatch &b, uint32_t bid, uint32_t nb)
{
	const uint32_t n = b.n;
	const uint32_t *__restrict__ in_off = b.in_off, *__restrict__ in_src = b.in_src, *__restrict__ w32 = b.w32;
	const uint32_t *__restrict__ cur = b.cur;
	const uint8_t *__restrict__ w8 = b.w8;
	uint32_t *dist = b.dist;
	uint8_t *flag = b.flag;
	for (uint32_t t = bid * kBlock + threadIdx.x; t < n; t += nb * kBlock) {
		const uint32_t e0 = in_off[t], e1 = in_off[t + 1];
		if (e1 == e0 || e1 - e0 > kPullLight) continue;
		uint32_t cand[kSsspBatchMax];
#pragma unroll
		for (int s = 0; s < (int)kSsspBatchMax; ++s) cand[s] = kInf;
		pull_edges<kW8>(e0, e1, 1, in_src, w32, w8, cur, dist, cand);
		uint32_t dt[kSsspBatchMax];
		load_row(dist, t, dt);
		bool better = false;
#pragma unroll
		for (int s = 0; s < (int)kSsspBatchMax; ++s)
			if (cand[s] < dt[s]) {
				dist[(uint64_t)t * kSsspBatchMax + s] = cand[s];
				better = true;
			}
		if (better) flag[t] = 1;
	}
}

// pieces of up to kPullPiece in-edges of the other vertices, a wavefront
// each: lane minima, a wavefront minimum per source, then lane s lowers
// source s's distance (atomicMin: a vertex's pieces may run at once)
template <bool kW8>
__device__ __forceinline__ void pull_heavy(const SsspBatch &b, uint32_t bid, uint32_t nb)
{
	const uint32_t *__restrict__ in_off = b.in_off, *__restrict__ in_src = b.in_src, *__restrict__ w32 = b.w32;
	const uint32_t *__restrict__ cur = b.cur;
	const uint8_t *__restrict__ w8 = b.w8;
	const uint2 *__restrict__ pieces = b.pieces;
	const uint32_t npieces = b.npieces;
	uint32_t *dist = b.dist;
	uint8_t *flag = b.flag;
	const uint32_t lane = threadIdx.x & 63, nwaves = (nb * kBlock) >> 6;
	for (uint32_t p = (bid * kBlock + threadIdx.x) >> 6; p < npieces; p += nwaves) {
		const uint2 pc = pieces[p];
		const uint32_t t = pc.x, e1 = min(pc.y + kPullPiece, in_off[t + 1]);
		uint32_t cand[kSsspBatchMax];
#pragma unroll
		for (int s = 0; s < (int)kSsspBatchMax; ++s) cand[s] = kInf;
		pull_edges<kW8>(pc.y + lane, e1, 64, in_src, w32, w8, cur, dist, cand);
		uint32_t mine = kInf;  // lane s < 16: source s's minimum over the wavefront
#pragma unroll
		for (int s = 0; s < (int)kSsspBatchMax; ++s) {
			uint32_t c = cand[s];
#pragma unroll
			for (int o = 32; o > 0; o >>= 1) {
				const uint32_t x = (uint32_t)__shfl_xor((int)c, o, 64);
				c = x < c ? x : c;
			}
			if ((int)lane == s) mine = c;
		}
		bool better = false;
		if (lane < kSsspBatchMax) {
			const uint64_t i = (uint64_t)t * kSsspBatchMax + lane;
			if (mine < dist[i]) {
				atomicMin(dist + i, mine);
				better = true;
			}
		}
		if (__ballot(better) && lane == 0) flag[t] = 1;
	}
}

template <bool kW8>
__global__ __launch_bounds__(kBlock) void ssspb_expand_kernel(SsspBatch t, uint32_t level)
{
	const Step st = step_of(t, level);
	if (blockIdx.x == 0 && threadIdx.x == 0) publish_level(t, level, st.fsize, st.fdeg, st.dense);
	if (st.fsize == 0) return;
	if (!st.dense)
		push_union(t, level, st);
	else if (blockIdx.x < t.heavy_blocks)
		pull_heavy<kW8>(t, blockIdx.x, t.heavy_blocks);
	else
		pull_light<kW8>(t, blockIdx.x - t.heavy_blocks, gridDim.x - t.heavy_blocks);
}

template <uint32_t kThreads>
__global__ __launch_bounds__(kThreads) void ssspb_advance_kernel(Frontier t, uint32_t level)
{
	advance_block<false, kThreads>(t, level);
}

}  // namespace

// The traversal state, in-edge arrays with their weights, and the distance
// array of an SSSP batch on gr (idempotent).
int sssp_batch_prepare(gphi_graph *gr)
{
	gphi_ctx *ctx = gr->ctx;
	const DevGraph &G = gr->g;
	if (!G.weighted) return set_error(ctx, GPHI_E_STATE, "graph carries no weights");
	if (!G.has_csr || !G.has_tiles) return set_error(ctx, GPHI_E_STATE, "graph needs CSR and tile arrays");
	int rc = ensure_traversal_state(gr);
	if (rc) return rc;
	if ((rc = build_in_edges(gr)) || (rc = build_in_weights(gr))) return rc;
	if (!gr->sb_dist) {
		const size_t bytes = (size_t)G.n_pad * kSsspBatchMax * 4;
		if (take_injected_alloc_failure())
			return set_error(ctx, GPHI_E_OOM, "hipMalloc(%zu bytes) failed: injected failure", bytes);
		if (hipMalloc((void **)&gr->sb_dist, bytes) != hipSuccess) {
			gr->sb_dist = nullptr;
			return set_error(ctx, GPHI_E_OOM, "hipMalloc(%zu bytes) for the SSSP batch failed", bytes);
		}
	}
	return GPHI_OK;
}

int run_sssp_batch(gphi_graph *gr, const uint32_t *srcs, uint32_t k, uint32_t *const *rows, gphi_stats *st)
{
	gphi_ctx *ctx = gr->ctx;
	const DevGraph &G = gr->g;
	if (k == 0 || k > kSsspBatchMax)
		return set_error(ctx, GPHI_E_ARG, "SSSP batch size %u not in [1, %u]", k, kSsspBatchMax);
	if (!srcs) return set_error(ctx, GPHI_E_ARG, "sources are NULL");
	for (uint32_t i = 0; i < k; ++i)
		if (srcs[i] >= G.n) return set_error(ctx, GPHI_E_RANGE, "source %u >= N %u", srcs[i], G.n);
	int rc = sssp_batch_prepare(gr);
	if (rc) return rc;
	if (st) memset(st, 0, sizeof(*st));
	hipStream_t s = ctx->stream;
	SsspBatch t = {};
	static_cast<Frontier &>(t) = make_frontier(gr, (uint32_t)(G.m / kSsspBatchDenseDiv));
	t.n = G.n, t.npieces = gr->npieces;
	t.row_off = G.row_off, t.cols = G.cols, t.csr_w = G.csr_w;
	t.in_off = gr->in_off, t.in_src = gr->in_src, t.w32 = gr->in_w32, t.w8 = gr->in_w8, t.pieces = gr->pieces;
	t.dist = gr->sb_dist;
	t.heavy_blocks = std::min<unsigned>((gr->npieces + 3) / 4, kSsspGrid);
	const unsigned light_blocks = std::min<unsigned>((G.n + kBlock - 1) / kBlock, kSsspGrid);
	const unsigned push_blocks = (unsigned)std::min<uint64_t>(G.m / kSparseTile + 1, kSsspGrid);
	const unsigned grid = std::max(t.heavy_blocks + light_blocks, push_blocks);
	const unsigned adv = advance_threads(G.n_pad), nblk = advance_blocks(G.n_pad);
	if ((rc = reset_board(ctx))) return rc;
	const uint64_t items = std::max<uint64_t>((uint64_t)G.n_pad * kSsspBatchMax / 4, G.n_words);
	ssspb_clear_kernel<<<(unsigned)std::min<uint64_t>((items + kBlock - 1) / kBlock, 16384), kBlock, 0, s>>>(t, G.n_words);
	SsspSeeds seeds = {};
	std::copy(srcs, srcs + k, seeds.src);
	ssspb_seed_kernel<<<1, 64, 0, s>>>(t, seeds, k);
	auto advance = [&](uint32_t level) {
		if (adv == 256)
			ssspb_advance_kernel<256><<<nblk, 256, 0, s>>>(t, level);
		else
			ssspb_advance_kernel<1024><<<nblk, 1024, 0, s>>>(t, level);
	};
	advance(UINT32_MAX);  // opens level 0: the sources
	// every step lowers some distance, and distances are bounded
	rc = follow_levels(ctx, [&](uint32_t level) -> int {
		if (level > (1u << 20)) return set_error(ctx, GPHI_E_STATE, "SSSP batch did not terminate");
		if (gr->in_w8)
			ssspb_expand_kernel<true><<<grid, kBlock, 0, s>>>(t, level);
		else
			ssspb_expand_kernel<false><<<grid, kBlock, 0, s>>>(t, level);
		advance(level);
		return GPHI_OK;
	});
	if (rc) return rc;
	bool any_row = false;
	for (uint32_t i = 0; rows && i < k; ++i) any_row |= rows[i] != nullptr;
	if (any_row && (rc = out_sssp_rows(gr, k, rows))) return rc;
	if (st) {
		st->steps = ctx->h_board->levels;
		st->total_ms = board_ms(ctx);
	}
	return GPHI_OK;
}

}  // namespace gphi
