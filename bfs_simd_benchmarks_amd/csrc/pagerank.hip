// pagerank.hip -- PageRank (FP32) over the in-edges, head band by head band.
//
// contrib = rank/deg; sum[t] += contrib[h] over the in-edges; rank = (1-d)/N +
// d*sum (apps/pageRank_simd/page_rank.cpp:128-199 gathers rank[h]/deg[h] into
// sum[t] over stripes of tile rows, each tile column owned by one thread;
// :428-446).  The bands, their segments and tiles are build_pr_bands's.
//
// The sweep of a band is one launch over tiles of kPrTile edges.  A block
// gathers a tile's contributions into LDS, all of its loads independent of
// where segments begin, and the heads of its next tile arrive meanwhile; then
// it adds up each segment's stretch of the tile, with as many lanes per segment
// as the tile's segments leave it, and a wavefront for one far longer than
// that.  Contributions of the first
// kPrHot heads (after the degree reordering, the ones most edges come from) are
// read from a copy in LDS: a gather from L2 costs a lane a cycle and CU, an LDS
// read a fraction.  A segment that lies in one tile goes straight into sum; the
// stretches of one that crosses tiles are left in two words per tile, and
// pr_cross_kernel adds them in tile order.
//
// What bounds it is the gathers that miss L1, about one L2 line per two cycles
// and CU: without the LDS copy an iteration takes 30 us more.  Before, segments
// were classed by length, each class with its kernel, and a wavefront took one
// long segment at a time, five dependent loads before its first add: 140 us an
// iteration on the pokec shape (31M edges) in nine launches, now 117 in three;
// 24 on 65536 vertices x 16, now 15.5; 355 on 4.2M x 16, now 309; 5.99 ms on
// rmat25 x 36, now 5.57.
//
// The FP32 additions run in a fixed order, so an iteration gives the same bits
// on every run: sum[t] = ((0 + band 0) + band 1) + ...; within a stretch each
// lane in turn, then a fixed butterfly, the number of lanes being the tile's.
// Every tail has one segment per band, so the adds of one band never meet on a
// tail.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "internal.h"

namespace gphi {

namespace {

// Three blocks per CU, by the LDS: 117 us an iteration on the pokec shape,
// where 1024 threads with tiles of 4096 and 14336 heads took 126, with 8192 and
// 31744 139, and 256 threads with tiles of 1024 and 4096 heads 129.
constexpr uint32_t kPrThreads = 512;
constexpr uint32_t kPrHot = 8000;
constexpr uint32_t kPrShort = 32;    // adds per lane before a stretch is given a wavefront (8: 30% slower; 64, 128: the same)
constexpr uint32_t kPrPer = kPrTile / kPrThreads;  // edges per lane and tile
static_assert(kPrPer % 4 == 0, "whole uint4s of heads per lane and tile");

__device__ __forceinline__ float wave_sum_f32(float x)
{
	// xor butterfly: lanes l and l^o add the same two values, so every lane
	// ends with the same bits
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
	return x;
}

__global__ void pr_prepare_kernel(uint32_t n, const float *__restrict__ rank, const uint32_t *__restrict__ deg,
                                  float *__restrict__ contrib, float *__restrict__ sum)
{
	uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
	if (v < n) {
		uint32_t d = deg[v];
		contrib[v] = d ? rank[v] / (float)d : 0.f;
		sum[v] = 0.f;
	}
}

// this lane's 4 heads of a tile (0xFFFFFFFF past the band's end)
__device__ __forceinline__ uint4 load_heads(const uint32_t *__restrict__ src, uint32_t e0, uint32_t at, uint32_t end)
{
	const uint32_t e = e0 + at, left = end - e0 > at ? end - e : 0u;  // (e may pass 2^32)
	if (left >= 4) return *reinterpret_cast<const uint4 *>(src + e);
	return make_uint4(left > 0 ? src[e] : ~0u, left > 1 ? src[e + 1] : ~0u, left > 2 ? src[e + 2] : ~0u, ~0u);
}

// What the reduction of a tile needs.
struct TileSums {
	uint32_t e0, e1, s0, s1, tile;
	const uint32_t *off, *tail;
	const float *val;  // LDS: the tile's contributions
	float *sum;
	float2 *part;
	// a stretch's sum: the segment's own if it lies in the tile, else the
	// tile's first or last part
	__device__ __forceinline__ void out(uint32_t s, uint32_t first, uint32_t last, float v) const
	{
		if (first < e0)
			part[tile].x = v;
		else if (last > e1)
			part[tile].y = v;
		else
			sum[tail[s]] += v;
	}
};

// Every segment's stretch of the tile, kLanes lanes each (a power of two), at
// most kPrShort adds per lane; the longer ones are listed for add_long.  The
// bounds of a lane's first segment were loaded ahead (first, last).
template <uint32_t kLanes>
__device__ __forceinline__ void add_segments(const TileSums &t, uint32_t tid, uint32_t first, uint32_t last, uint2 *s_long,
                                             uint32_t *s_nlong)
{
	const uint32_t g = tid % kLanes;
	for (uint32_t s = t.s0 + tid / kLanes;; ) {
		// the last segment may begin with the next tile
		const uint32_t lo = max(first, t.e0), hi = s <= t.s1 ? min(last, t.e1) : 0u;
		float acc = 0.f;
		const bool small = lo < hi && hi - lo <= kPrShort * kLanes;
		if (small) {
			const float *v = t.val + (lo - t.e0);
			const uint32_t n = hi - lo;
			float a[4] = {0.f, 0.f, 0.f, 0.f};
			uint32_t k = g;
			for (; k + 3 * kLanes < n; k += 4 * kLanes) {
#pragma unroll
				for (int j = 0; j < 4; ++j) a[j] += v[k + j * kLanes];
			}
			for (; k < n; k += kLanes) a[0] += v[k];
			acc = (a[0] + a[1]) + (a[2] + a[3]);
		} else if (lo < hi && g == 0) {
			s_long[atomicAdd(s_nlong, 1u)] = make_uint2(s, lo - t.e0 | (hi - t.e0) << 16);
		}
#pragma unroll
		for (int o = kLanes / 2; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
		if (small && g == 0) t.out(s, first, last, acc);
		s += kPrThreads / kLanes;
		if (__ballot(s <= t.s1) == 0) break;  // (whole groups: every lane takes part in the shuffles)
		if (s <= t.s1) {
			first = t.off[s];
			last = t.off[s + 1];
		}
	}
}

__global__ __launch_bounds__(kPrThreads) void pr_tile_kernel(PrBand b, const uint32_t *__restrict__ src,
                                                             const uint32_t *__restrict__ off,
                                                             const uint32_t *__restrict__ tail,
                                                             const uint32_t *__restrict__ tile_seg,
                                                             const float *__restrict__ contrib,
                                                             float *__restrict__ sum, float2 *__restrict__ part)
{
	__shared__ float s_hot[kPrHot];
	__shared__ float4 s_val4[kPrTile / 4];
	__shared__ uint2 s_long[kPrTile / kPrShort];
	__shared__ uint32_t s_nlong[2];  // of this tile and, cleared meanwhile, the next
	const float *s_val = reinterpret_cast<const float *>(s_val4);
	const uint32_t tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
	const uint32_t end = b.edge0 + b.nedges;
	const uint32_t hot = b.head_lo == 0 ? min(kPrHot, b.head_hi) : 0u;
	uint32_t i = blockIdx.x;
	if (i >= b.ntiles) return;
	// a lane's heads: 4 consecutive ones of each kPrThreads * 4 edges
	uint4 h[kPrPer / 4];
#pragma unroll
	for (uint32_t u = 0; u < kPrPer / 4; ++u)
		h[u] = load_heads(src, b.edge0 + i * kPrTile, 4 * (u * kPrThreads + tid), end);
	uint32_t s0 = tile_seg[b.tile0 + i], s1 = tile_seg[b.tile0 + i + 1];
	for (uint32_t k = tid; k < hot; k += kPrThreads) s_hot[k] = contrib[k];
	if (tid < 2) s_nlong[tid] = 0;
	for (uint32_t p = 0; i < b.ntiles; i += gridDim.x, p ^= 1) {
		const uint32_t e0 = b.edge0 + i * kPrTile, e1 = e0 + min(kPrTile, end - e0);
		// lanes per segment: as many as keep the block busy
		const uint32_t nseg = s1 - s0 + 1;
		uint32_t lg = 0;
		while (lg < 6 && (nseg << lg) * 4 <= kPrThreads) ++lg;
		const uint32_t mine = min(s0 + (tid >> lg), s1);
		const uint32_t first = off[mine], last = off[mine + 1];
		__syncthreads();  // the tile before is added up (and the first time, s_hot is filled)
		uint32_t hh[kPrPer];
		float c[kPrPer];
#pragma unroll
		for (uint32_t u = 0; u < kPrPer / 4; ++u)
			hh[4 * u] = h[u].x, hh[4 * u + 1] = h[u].y, hh[4 * u + 2] = h[u].z, hh[4 * u + 3] = h[u].w;
#pragma unroll
		for (uint32_t j = 0; j < kPrPer; ++j) c[j] = hh[j] >= hot && hh[j] != ~0u ? contrib[hh[j]] : 0.f;
#pragma unroll
		for (uint32_t j = 0; j < kPrPer; ++j)
			if (hh[j] < hot) c[j] = s_hot[hh[j]];
#pragma unroll
		for (uint32_t u = 0; u < kPrPer / 4; ++u)
			s_val4[u * kPrThreads + tid] = make_float4(c[4 * u], c[4 * u + 1], c[4 * u + 2], c[4 * u + 3]);
		const TileSums t{e0, e1, s0, s1, b.tile0 + i, off, tail, s_val, sum, part};
		if (i + gridDim.x < b.ntiles) {
#pragma unroll
			for (uint32_t u = 0; u < kPrPer / 4; ++u)
				h[u] = load_heads(src, e0 + gridDim.x * kPrTile, 4 * (u * kPrThreads + tid), end);
			s0 = tile_seg[b.tile0 + i + gridDim.x];
			s1 = tile_seg[b.tile0 + i + gridDim.x + 1];
		}
		if (tid == 0) s_nlong[p ^ 1] = 0;
		__syncthreads();
		switch (lg) {
		case 0: add_segments<1>(t, tid, first, last, s_long, &s_nlong[p]); break;
		case 1: add_segments<2>(t, tid, first, last, s_long, &s_nlong[p]); break;
		case 2: add_segments<4>(t, tid, first, last, s_long, &s_nlong[p]); break;
		case 3: add_segments<8>(t, tid, first, last, s_long, &s_nlong[p]); break;
		case 4: add_segments<16>(t, tid, first, last, s_long, &s_nlong[p]); break;
		case 5: add_segments<32>(t, tid, first, last, s_long, &s_nlong[p]); break;
		default: add_segments<64>(t, tid, first, last, s_long, &s_nlong[p]); break;
		}
		__syncthreads();
		// the long stretches, a wavefront each
		const uint32_t nlong = s_nlong[p];
		for (uint32_t q = wid; q < nlong; q += kPrThreads / 64) {
			const uint2 x = s_long[q];
			const uint32_t lo = x.y & 0xFFFFu, hi = x.y >> 16;
			float acc = 0.f;
			for (uint32_t e = lo + lane; e < hi; e += 64) acc += s_val[e];
			acc = wave_sum_f32(acc);
			if (lane == 0) t.out(x.x, off[x.x], off[x.x + 1], acc);
		}
	}
}

// The segments that cross tiles: a wavefront per tile, which owns the segment
// that begins in it and goes on in the next.
__global__ __launch_bounds__(kBlock) void pr_cross_kernel(PrBand b, const uint32_t *__restrict__ off,
                                                          const uint32_t *__restrict__ tail,
                                                          const uint32_t *__restrict__ tile_seg,
                                                          const float2 *__restrict__ part, float *__restrict__ sum)
{
	const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
	if (i + 1 >= b.ntiles) return;
	const uint32_t s = tile_seg[b.tile0 + i + 1], first = off[s], e0 = b.edge0 + i * kPrTile;
	if (first < e0 || first - e0 >= kPrTile) return;
	const uint32_t last = (off[s + 1] - 1 - b.edge0) / kPrTile;  // the tile it ends in
	// in 64 bits: the hubs, whose ranks are the largest, cross hundreds of tiles
	double acc = 0.;
	for (uint32_t k = i + 1 + lane; k <= last; k += 64) acc += (double)part[b.tile0 + k].x;
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
	if (lane == 0) sum[tail[s]] = (float)((double)sum[tail[s]] + (double)part[b.tile0 + i].y + acc);
}

// rank = (1-d)/N + d*sum (page_rank.cpp:428-446), the next iteration's
// contributions rank/deg, and sum cleared for it, in one pass; rank is kept
// after the last iteration only
__global__ void pr_apply_kernel(uint32_t n, float first, float damping, float *__restrict__ sum,
                                const uint32_t *__restrict__ deg, float *__restrict__ rank,
                                float *__restrict__ contrib)
{
	uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
	if (v < n) {
		const float r = first + damping * sum[v];
		if (rank) {
			rank[v] = r;
			return;
		}
		sum[v] = 0.f;
		const uint32_t d = deg[v];
		contrib[v] = d ? r / (float)d : 0.f;
	}
}

}  // namespace

int run_pagerank(gphi_graph *gr, uint32_t iters, float damping, float init, float *rank, float *ms)
{
	gphi_ctx *ctx = gr->ctx;
	DevGraph &G = gr->g;
	hipStream_t s = ctx->stream;
	int rc;
	if ((rc = build_in_edges(gr))) return rc;
	if ((rc = build_pr_bands(gr))) return rc;
	if (!gr->rank) {
		// rank, sum, contrib (n_pad each), then the parts of the crossing segments
		const size_t bytes = 3 * (size_t)G.n_pad * 4 + ((size_t)gr->pr_ntiles + 1) * 8;
		if ((rc = dmalloc(ctx, (void **)&gr->rank, bytes, nullptr))) return rc;
		gr->sum = gr->rank + G.n_pad;
		gr->contrib = gr->sum + G.n_pad;
	}
	float2 *part = reinterpret_cast<float2 *>(gr->contrib + G.n_pad);
	const float first = (1.0f - damping) / (float)G.n;
	const unsigned vgrid = (unsigned)((G.n + kBlock - 1) / kBlock);
	static const unsigned resident = resident_grid(reinterpret_cast<const void *>(pr_tile_kernel), kPrThreads);
	uint32_t bits;
	memcpy(&bits, &init, 4);
	fill_words(ctx, (uint32_t *)gr->rank, G.n, bits);
	if (ctx->ev_ok) GPHI_HIP(ctx, hipEventRecord(ctx->ev[0], s));
	pr_prepare_kernel<<<vgrid, kBlock, 0, s>>>(G.n, gr->rank, G.deg, gr->contrib, gr->sum);
	for (uint32_t it = 0; it < iters; ++it) {
		for (const PrBand &b : gr->pr_bands) {
			pr_tile_kernel<<<std::min(resident, b.ntiles), kPrThreads, 0, s>>>(b, gr->pr_src, gr->pr_off, gr->pr_tail,
			                                                                  gr->pr_tile, gr->contrib, gr->sum, part);
			if (b.ntiles > 1)
				pr_cross_kernel<<<(b.ntiles + kBlock / 64 - 1) / (kBlock / 64), kBlock, 0, s>>>(
				    b, gr->pr_off, gr->pr_tail, gr->pr_tile, part, gr->sum);
		}
		pr_apply_kernel<<<vgrid, kBlock, 0, s>>>(G.n, first, damping, gr->sum, G.deg, it + 1 == iters ? gr->rank : nullptr,
		                                         gr->contrib);
	}
	GPHI_HIP(ctx, hipGetLastError());
	if (ctx->ev_ok) GPHI_HIP(ctx, hipEventRecord(ctx->ev[1], s));
	if (rank && (rc = out_words(ctx, gr->rank, nullptr, G.n, rank))) return rc;
	if (ms) {
		GPHI_HIP(ctx, hipStreamSynchronize(s));
		float t = 0.f;
		*ms = ctx->ev_ok && hipEventElapsedTime(&t, ctx->ev[0], ctx->ev[1]) == hipSuccess ? t : 0.f;
	}
	return GPHI_OK;
}

}  // namespace gphi
