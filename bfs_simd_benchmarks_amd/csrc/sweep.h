// sweep.h -- device code shared by the traversal kernels: wavefront helpers,
// the LDS windows of the tile sweeps, the 16-bit edge forms, and the BFS and
// SSSP walks over a list of chunks.
#pragma once

#include <hip/hip_runtime.h>

#include "internal.h"

namespace gphi {

// ---------------------------------------------------------------------------
// wave helpers (wave64)
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

__device__ __forceinline__ uint32_t wave_sum(uint32_t x)
{
	for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
	return x;
}

// exclusive prefix sum across the wave; *total gets the wave sum
__device__ __forceinline__ uint32_t wave_excl_scan(uint32_t x, uint32_t *total)
{
	uint32_t lane = lane_id();
	uint32_t inc = x;
	for (int o = 1; o < 64; o <<= 1) {
		uint32_t y = __shfl_up(inc, o, 64);
		if (lane >= (uint32_t)o) inc += y;
	}
	*total = __shfl(inc, 63, 64);
	return inc - x;
}

__device__ __forceinline__ bool test_bit(const uint32_t *__restrict__ bm, uint32_t v)
{
	return (bm[v >> 5] >> (v & 31)) & 1u;
}

// A window: an aligned run of R tile rows (or columns) whose R*W vertices fit
// kWinWords bitmap words, i.e. 16-bit offsets (R*W <= 65536).
constexpr uint32_t kWinWords = 2048;

// tile rows per window for tile width W (0: no window fits)
inline uint32_t dense_window_rows(uint32_t W)
{
	if (W == 0) return 0;
	if ((W & (W - 1)) == 0 && W <= kWinWords * 32) return kWinWords * 32 / W;
	return W <= (kWinWords - 4) * 32 ? (kWinWords - 4) * 32 / W : 0;
}

// first vertex of the window that holds tile row (column) lo
__host__ __device__ __forceinline__ uint32_t window_base(uint32_t lo, uint32_t R, uint32_t W)
{
	return (uint32_t)((uint64_t)(lo - lo % R) * W);
}

typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
// streaming (non-temporal) 16-byte load: the tile arrays are read once per
// sweep and should not evict the bitmaps and state arrays from L2 / MALL
__device__ __forceinline__ uint4 ld_stream(const uint4 *p)
{
	const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t *>(p));
	return make_uint4(v.x, v.y, v.z, v.w);
}

// Frontier-bit lookups of the dense sweep go through LDS.  A chunk's heads
// lie in its tile-row range [row_lo, row_hi] (a column-stripe chunk stays in
// one stripe), so the frontier bitmap of an aligned run of R tile rows
// (kWinWords words) is copied into LDS once and serves every chunk of the
// block inside it; a chunk outside any such run looks its bits up in global
// memory.  Gathers cost address-unit cycles per lane, LDS reads do not.
constexpr uint32_t kDenseRun = 8;  // consecutive live-list entries per block run

// window [wlo, wlo + wlen) of bitmap words holding tile rows row_lo..row_hi,
// or false; wlo is a multiple of 4 and wlen <= kWinWords
__device__ __forceinline__ bool window_of(uint32_t row_lo, uint32_t row_hi, uint32_t R, uint32_t W,
                                          uint32_t n_words, uint32_t &wlo, uint32_t &wlen)
{
	if (R == 0) return false;
	const uint32_t r0 = row_lo - row_lo % R;
	if (row_hi - r0 >= R) return false;
	const uint64_t b0 = (uint64_t)r0 * W, b1 = (uint64_t)(r0 + R) * W;
	wlo = (uint32_t)(b0 >> 5) & ~3u;
	const uint32_t whi = (uint32_t)min((b1 + 31) >> 5, (uint64_t)n_words);
	wlen = whi - wlo;
	return true;
}

// block-wide copy of bitmap words [wlo, wlo + wlen) into LDS (n_words is a
// multiple of 4, so the rounded-up last uint4 stays inside the bitmap)
__device__ __forceinline__ void load_window(uint4 *s_win, const uint32_t *cur, uint32_t wlo, uint32_t wlen,
                                            uint32_t tid)
{
	const uint4 *src = reinterpret_cast<const uint4 *>(cur + wlo);
	const uint32_t nq = (wlen + 3) / 4;
	// one uint4 in flight per lane: window changes are rare, registers are not
#pragma nounroll
	for (uint32_t q = tid; q < nq; q += kBlock) s_win[q] = src[q];
}

// frontier bits of 8 heads; in the window every real head of the chunk is
// inside it, a padding head (id n) outside it reads as not in the frontier
__device__ __forceinline__ uint32_t frontier_bits(const uint32_t (&hh)[8], bool inw, const uint32_t *s_win,
                                                  uint32_t wlo, uint32_t wlen, const uint32_t *cur)
{
	uint32_t cw[8];
	if (inw) {
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const uint32_t wi = (hh[j] >> 5) - wlo;
			cw[j] = wi < wlen ? s_win[wi] : 0u;
		}
	} else {
#pragma unroll
		for (int j = 0; j < 8; ++j) cw[j] = cur[hh[j] >> 5];
	}
	uint32_t hit = 0;
#pragma unroll
	for (int j = 0; j < 8; ++j) hit |= ((cw[j] >> (hh[j] & 31)) & 1u) << j;
	return hit;
}

// Software-pipelined walk of this XCD's live-chunk list (runs of kDenseRun
// entries per block), 8 edges per lane per chunk.  While chunk k finishes
// (state bytes of its tails, writes), the frontier bits of chunk k+1 are
// looked up, and then its tails and the heads of chunk k+2 are requested, so
// each iteration waits on one HBM latency and one L2 round trip.  Every
// global load is unconditional (a lane with nothing to fetch reads a cached
// dummy word) so the compiler can count them.  Tails of a 4-edge quad are
// fetched only when one of its heads is in the frontier.
// Heads and tails come in their 16-bit forms wherever those are exact (half
// the bytes and memory requests); lane tid always owns edges 4tid..4tid+3
// and 1024+4tid..1024+4tid+3 of the chunk, in either form, so the tails of
// a wavefront's two quads decode from its two tail groups.
// One byte per vertex says whether a tail is new (state 0): "visited before
// this step" and "reached in this step" live in the same byte, so a
// candidate costs one lookup.  Every lane that sees state 0 writes parent and
// state 1 (benign races: every writer stores a valid frontier head and the
// same state; an earlier step's kVisited is never overwritten, since no lane
// of this step reads state 0 for such a vertex).
__device__ __forceinline__ void unpack8(const uint4 a, const uint4 b, uint32_t (&x)[8])
{
	x[0] = a.x, x[1] = a.y, x[2] = a.z, x[3] = a.w, x[4] = b.x, x[5] = b.y, x[6] = b.z, x[7] = b.w;
}

typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint2 ld_stream8(const uint2 *p)
{
	const u32x2_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x2_t *>(p));
	return make_uint2(v.x, v.y);
}

// Raw edge words of one array of chunk c as loaded: 8 ids, or (16-bit form)
// 4 words of two offsets each.  q0 / q1: fetch the first / second quad (a
// lane that skips one reads the array's first bytes instead).
__device__ __forceinline__ void load_edges(bool p16, const uint32_t *__restrict__ a32,
                                           const uint16_t *__restrict__ a16, uint64_t c, uint32_t tid, bool q0,
                                           bool q1, uint32_t (&raw)[8])
{
	if (p16) {
		const uint2 *A = reinterpret_cast<const uint2 *>(a16 + c * kChunk);
		const uint2 *D = reinterpret_cast<const uint2 *>(a16);
		const uint2 x = ld_stream8(q0 ? A + tid : D), y = ld_stream8(q1 ? A + tid + kBlock : D);
		raw[0] = x.x, raw[1] = x.y, raw[2] = y.x, raw[3] = y.y;
	} else {
		const uint4 *A = reinterpret_cast<const uint4 *>(a32 + c * kChunk);
		const uint4 *D = reinterpret_cast<const uint4 *>(a32);
		unpack8(ld_stream(q0 ? A + tid : D), ld_stream(q1 ? A + tid + kBlock : D), raw);
	}
}

// raw edge words -> 8 vertex ids (in place)
// (base0 for the lane's first quad, base1 for its second)
__device__ __forceinline__ void decode_edges(bool p16, uint32_t base0, uint32_t base1, uint32_t (&x)[8])
{
	if (p16) {
		const uint32_t w0 = x[0], w1 = x[1], w2 = x[2], w3 = x[3];
		x[0] = base0 + (w0 & 0xFFFFu), x[1] = base0 + (w0 >> 16);
		x[2] = base0 + (w1 & 0xFFFFu), x[3] = base0 + (w1 >> 16);
		x[4] = base1 + (w2 & 0xFFFFu), x[5] = base1 + (w2 >> 16);
		x[6] = base1 + (w3 & 0xFFFFu), x[7] = base1 + (w3 >> 16);
	}
}

// what the sweep needs of a chunk's ChunkPack: head base, flags, and the
// tail bases of this wavefront's two edge groups (wv and 4 + wv)
struct PackSlot {
	uint32_t hbase, flags, tb0, tb1;
};
__device__ __forceinline__ PackSlot pack_slot(const ChunkPack *__restrict__ pack, uint32_t c, uint32_t wv)
{
	return PackSlot{pack[c].hbase, pack[c].flags, pack[c].tbase[wv], pack[c].tbase[4 + wv]};
}

// The list of chunks a block walks: entries pos, ... below end, kDenseRun
// consecutive ones at a time, skip entries apart.  Entries come from a list
// in memory (uniform loads) or in LDS, where readfirstlane keeps the chunk
// ids, and with them the chunk summaries' loads, scalar.
struct ChunkList {
	const uint32_t *p;
	__device__ __forceinline__ uint32_t operator()(uint32_t i) const { return p[i]; }
};
struct LdsChunkList {
	const uint32_t *p;
	__device__ __forceinline__ uint32_t operator()(uint32_t i) const
	{
		return (uint32_t)__builtin_amdgcn_readfirstlane((int)p[i]);
	}
};

template <class List>
__device__ __forceinline__ void bfs_dense_walk(
    uint4 *s_win4 /* frontier bits of chunk k+1's rows */, uint4 *s_vwin4 /* visited / claimed bits of chunk k's columns */,
    List lst, uint32_t pos, uint32_t end, uint32_t skip, const uint32_t *__restrict__ heads,
    const uint32_t *__restrict__ tails, const uint16_t *__restrict__ heads16, const uint16_t *__restrict__ tails16,
    const ChunkMeta *__restrict__ meta, const ChunkPack *__restrict__ pack, const uint32_t *__restrict__ cur,
    const uint32_t *__restrict__ visited, uint32_t n_words, uint32_t W, uint32_t R, uint8_t *__restrict__ state,
    int32_t *__restrict__ parent)
{
	const uint32_t *s_win = reinterpret_cast<const uint32_t *>(s_win4);
	uint32_t *s_vwin = reinterpret_cast<uint32_t *>(s_vwin4);
	auto nxt = [&](uint32_t p) { return ((p + 1) % kDenseRun) ? p + 1 : p + 1 + skip; };
	if (pos >= end) return;
	const uint32_t tid = threadIdx.x;
	const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));  // wavefront in the block
	static_assert(kPackGroup == 4 * 64, "a wavefront's quad row is one tail group");
	// first words of the windows held in LDS (block-uniform)
	uint32_t win_lo = UINT32_MAX, vwin_lo = UINT32_MAX;
	// list entries: chunks k, k+1, k+2 (an absent one repeats chunk k's id, so
	// every address stays valid; its results are masked off)
	const uint32_t c0 = lst(pos);
	uint32_t p1 = nxt(pos), p2 = nxt(p1);
	bool v1 = p1 < end, v2 = p2 < end;
	uint32_t c1 = v1 ? lst(p1) : c0;
	uint32_t c2 = v2 ? lst(p2) : c0;
	// prologue: heads and frontier bits of chunk k, then heads of k+1 and tails of k
	PackSlot pk = pack_slot(pack, c0, wv), pk1 = pack_slot(pack, c1, wv);
	uint32_t h[8], hn[8], t[8];
	load_edges(pk.flags & 1u, heads, heads16, c0, tid, true, true, h);
	decode_edges(pk.flags & 1u, pk.hbase, pk.hbase, h);
	uint32_t hit;
	{
		const ChunkMeta m0 = meta[c0];
		uint32_t wlo = 0, wlen = 0;
		const bool inw = window_of(m0.row_lo, m0.row_hi, R, W, n_words, wlo, wlen);
		if (inw) {
			load_window(s_win4, cur, wlo, wlen, tid);
			__syncthreads();
			win_lo = wlo;
		}
		hit = frontier_bits(h, inw, s_win, wlo, wlen, cur);
	}
	load_edges(pk1.flags & 1u, heads, heads16, c1, tid, true, true, hn);
	load_edges(pk.flags & 2u, tails, tails16, c0, tid, hit & 0x0Fu, hit & 0xF0u, t);
	uint32_t ck = c0;  // chunk k
	for (;;) {
		// windows (block-uniform): frontier rows of chunk k+1, visited columns of chunk k
		bool inw_n = false;
		uint32_t wlo_n = 0, wlen_n = 0, vwlo = 0, vwlen = 0;
		if (v1) {
			const ChunkMeta mn = meta[c1];
			inw_n = window_of(mn.row_lo, mn.row_hi, R, W, n_words, wlo_n, wlen_n);
		}
		const ChunkMeta mk = meta[ck];
		const bool vin = window_of(mk.col_lo, mk.col_hi, R, W, n_words, vwlo, vwlen);
		const bool ld_c = inw_n && wlo_n != win_lo, ld_v = vin && vwlo != vwin_lo;
		if (ld_c || ld_v) {
			__syncthreads();  // every wave is done with the old windows
			if (ld_c) {
				load_window(s_win4, cur, wlo_n, wlen_n, tid);
				win_lo = wlo_n;
			}
			if (ld_v) {
				load_window(s_vwin4, visited, vwlo, vwlen, tid);
				vwin_lo = vwlo;
			}
			__syncthreads();
		}
		decode_edges(pk.flags & 2u, pk.tb0, pk.tb1, t);
		decode_edges(pk1.flags & 1u, pk1.hbase, pk1.hbase, hn);
		// stage A: states of chunk k's new frontier-edge tails, frontier bits of
		// chunk k+1.  In the column window each frontier edge claims its tail's
		// bit: a tail visited in an earlier step (bit set when the window was
		// loaded) or already claimed by another edge of this block in this step
		// needs no state lookup, so a block looks each new tail up once.
		uint32_t need = hit;
		if (vin) {
#pragma unroll
			for (int j = 0; j < 8; ++j) {
				const uint32_t wi = (t[j] >> 5) - vwlo, b = 1u << (t[j] & 31);
				if (((hit >> j) & 1u) && wi < vwlen && (atomicOr(s_vwin + wi, b) & b)) need &= ~(1u << j);
			}
		}
		uint32_t sv[8];
#pragma unroll
		for (int j = 0; j < 8; ++j) sv[j] = state[((need >> j) & 1u) ? t[j] : 0u];
		const uint32_t hit_n = v1 ? frontier_bits(hn, inw_n, s_win, wlo_n, wlen_n, cur) : 0u;
		uint32_t cand = 0;
#pragma unroll
		for (int j = 0; j < 8; ++j) cand |= (sv[j] == 0 ? 1u : 0u) << j;
		cand &= need;
		// stage B: chunk k's writes (few; issued first, so chunk k's heads and
		// tails are dead before the next requests take their registers)
#pragma unroll
		for (int j = 0; j < 8; ++j)
			if ((cand >> j) & 1u) {
				parent[t[j]] = (int32_t)h[j];
				state[t[j]] = 1;
			}
		// stage C: the HBM requests of the next iteration: tails of k+1, heads of k+2
		const PackSlot pk2 = pack_slot(pack, c2, wv);
		uint32_t tn[8], h2[8];
		load_edges(pk1.flags & 2u, tails, tails16, c1, tid, hit_n & 0x0Fu, hit_n & 0xF0u, tn);
		load_edges(pk2.flags & 1u, heads, heads16, c2, tid, true, true, h2);
		const uint32_t p3 = nxt(p2);
		const bool v3 = p3 < end;
		const uint32_t c3 = v3 ? lst(p3) : c0;
		if (!v1) break;
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			h[j] = hn[j];
			t[j] = tn[j];
			hn[j] = h2[j];
		}
		hit = hit_n;
		ck = c1;
		c1 = c2;
		c2 = c3;
		pk = pk1;
		pk1 = pk2;
		v1 = v2;
		v2 = v3;
		p2 = p3;
	}
}
static_assert(kChunk == 2 * 4 * kBlock, "dense sweep loads two uint4 per array per thread");

// SSSP relax (apps/sssp_simd/sssp.cpp:344-445): if mask[h] and dist[h]+w <
// dist[t] then lower dist[t] and mark t for the next frontier.  The walk of
// bfs_dense_kernel: runs of kDenseRun list entries per block, frontier bits
// from the LDS row window, heads and tails in their 16-bit forms where
// exact, and a three-chunk pipeline: while chunk k is relaxed, the frontier
// bits of chunk k+1 are looked up and its tails and weights (only for 4-edge
// quads with a frontier head) and the heads of chunk k+2 are requested.  A
// lane that sees dist[h]+w below the dist[t] it read issues an atomicMin (no
// return) and marks t: dist[t] then ends the step below the value read
// during it, i.e. t improved this step, which is exactly the condition for t
// to be in the next frontier.
// a lane's 8 weights of chunk c: 32-bit (8 registers) or, with kW8, the
// 1-byte copy (2 registers, 4 weights each); quads without a frontier head
// read the array's first bytes
template <bool kW8>
__device__ __forceinline__ void load_weights(const uint32_t *__restrict__ w32, const uint8_t *__restrict__ w8,
                                             uint64_t c, uint32_t tid, bool q0, bool q1,
                                             uint32_t (&w)[kW8 ? 2 : 8])
{
	if constexpr (kW8) {
		const uint32_t *A = reinterpret_cast<const uint32_t *>(w8 + c * kChunk);
		const uint32_t *D = reinterpret_cast<const uint32_t *>(w8);
		w[0] = q0 ? A[tid] : D[0];
		w[1] = q1 ? A[tid + kBlock] : D[0];
	} else {
		load_edges(false, w32, nullptr, c, tid, q0, q1, w);
	}
}
template <bool kW8>
__device__ __forceinline__ uint32_t weight_of(const uint32_t (&w)[kW8 ? 2 : 8], int j)
{
	if constexpr (kW8)
		return (w[j >> 2] >> (8 * (j & 3))) & 0xFFu;
	else
		return w[j];
}

template <bool kW8, class List>
__device__ __forceinline__ void sssp_dense_walk(
    uint4 *s_win4 /* frontier bits of chunk k+1's rows */, List lst, uint32_t first, uint32_t end, uint32_t skip, const uint32_t *__restrict__ heads,
    const uint32_t *__restrict__ tails, const uint16_t *__restrict__ heads16, const uint16_t *__restrict__ tails16,
    const uint32_t *__restrict__ wts, const uint8_t *__restrict__ wts8, const ChunkMeta *__restrict__ meta,
    const ChunkPack *__restrict__ pack, const uint32_t *__restrict__ cur, uint32_t n_words, uint32_t W, uint32_t R,
    uint32_t *dist, uint8_t *__restrict__ flag)
{
	const uint32_t *s_win = reinterpret_cast<const uint32_t *>(s_win4);
	auto nxt = [&](uint32_t p) { return ((p + 1) % kDenseRun) ? p + 1 : p + 1 + skip; };
	if (first >= end) return;
	const uint32_t tid = threadIdx.x;
	const uint32_t wv = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
	uint32_t win_lo = UINT32_MAX;  // first word of the window held in LDS (block-uniform)
	const uint32_t c0 = lst(first);
	uint32_t p2 = nxt(nxt(first));
	bool v1 = nxt(first) < end, v2 = p2 < end;
	uint32_t c1 = v1 ? lst(nxt(first)) : c0, c2 = v2 ? lst(p2) : c0;
	PackSlot pk = pack_slot(pack, c0, wv), pk1 = pack_slot(pack, c1, wv);
	uint32_t h[8], hn[8], t[8], w[kW8 ? 2 : 8];
	load_edges(pk.flags & 1u, heads, heads16, c0, tid, true, true, h);
	decode_edges(pk.flags & 1u, pk.hbase, pk.hbase, h);
	uint32_t hit;
	{
		const ChunkMeta m0 = meta[c0];
		uint32_t wlo = 0, wlen = 0;
		const bool inw = window_of(m0.row_lo, m0.row_hi, R, W, n_words, wlo, wlen);
		if (inw) {
			load_window(s_win4, cur, wlo, wlen, tid);
			__syncthreads();
			win_lo = wlo;
		}
		hit = frontier_bits(h, inw, s_win, wlo, wlen, cur);
	}
	{
		load_edges(pk1.flags & 1u, heads, heads16, c1, tid, true, true, hn);
		load_edges(pk.flags & 2u, tails, tails16, c0, tid, hit & 0x0Fu, hit & 0xF0u, t);
		load_weights<kW8>(wts, wts8, c0, tid, hit & 0x0Fu, hit & 0xF0u, w);
	}
	for (;;) {
		// window of chunk k+1 (a block-uniform branch)
		bool inw_n = false;
		uint32_t wlo_n = 0, wlen_n = 0;
		if (v1) {
			const ChunkMeta mn = meta[c1];
			inw_n = window_of(mn.row_lo, mn.row_hi, R, W, n_words, wlo_n, wlen_n);
			if (inw_n && wlo_n != win_lo) {
				__syncthreads();  // every wave is done with the old window
				load_window(s_win4, cur, wlo_n, wlen_n, tid);
				__syncthreads();
				win_lo = wlo_n;
			}
		}
		decode_edges(pk.flags & 2u, pk.tb0, pk.tb1, t);
		decode_edges(pk1.flags & 1u, pk1.hbase, pk1.hbase, hn);
		// stage A: distances at both ends of chunk k's frontier edges, frontier bits of chunk k+1
		uint32_t dh[8], dt[8];
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			const bool on = (hit >> j) & 1u;
			dh[j] = dist[on ? h[j] : 0u];
			dt[j] = dist[on ? t[j] : 0u];
		}
		const uint32_t hit_n = v1 ? frontier_bits(hn, inw_n, s_win, wlo_n, wlen_n, cur) : 0u;
		uint32_t better = 0;
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			// (a byte added to a distance stays below 2^32)
			const uint32_t x = weight_of<kW8>(w, j), nd = kW8 ? dh[j] + x : path_sum(dh[j], x);
			better |= (uint32_t)(nd < dt[j]) << j;
		}
		better &= hit;
		// stage B: chunk k's relaxations
#pragma unroll
		for (int j = 0; j < 8; ++j)
			if ((better >> j) & 1u) {
				atomicMin(dist + t[j], dh[j] + weight_of<kW8>(w, j));
				flag[t[j]] = 1;
			}
		// stage C: the requests of the next iteration
		const PackSlot pk2 = pack_slot(pack, c2, wv);
		uint32_t tn[8], wn[kW8 ? 2 : 8], h2[8];
		load_edges(pk1.flags & 2u, tails, tails16, c1, tid, hit_n & 0x0Fu, hit_n & 0xF0u, tn);
		load_weights<kW8>(wts, wts8, c1, tid, hit_n & 0x0Fu, hit_n & 0xF0u, wn);
		load_edges(pk2.flags & 1u, heads, heads16, c2, tid, true, true, h2);
		const uint32_t p3 = nxt(p2);
		const bool v3 = p3 < end;
		const uint32_t c3 = v3 ? lst(p3) : c0;
		if (!v1) break;
#pragma unroll
		for (int j = 0; j < 8; ++j) {
			h[j] = hn[j];
			t[j] = tn[j];
			hn[j] = h2[j];
		}
#pragma unroll
		for (int j = 0; j < (kW8 ? 2 : 8); ++j) w[j] = wn[j];
		hit = hit_n;
		c1 = c2;
		c2 = c3;
		pk = pk1;
		pk1 = pk2;
		v1 = v2;
		v2 = v3;
		p2 = p3;
	}
}

}  // namespace gphi
