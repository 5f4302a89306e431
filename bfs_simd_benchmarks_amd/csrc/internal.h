// internal.h -- shared declarations of libgphi (host C++ and HIP translation units).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/gphi.h"

namespace gphi {

// Edges of one sweep chunk.  The tiled COO arrays are padded to a multiple of
// this with sentinel edges (head = tail = n) whose frontier bit is never set.
constexpr uint32_t kChunk = 2048;
constexpr uint32_t kBlock = 256;
constexpr uint32_t kSparseTile = 1024;  // edges per block iteration of the CSR push
constexpr uint32_t kPadVerts = kBlock * 32;  // vertices per frontier-update block
constexpr uint32_t kPullLight = 64;     // pull steps: a lane per vertex up to this in-degree,
constexpr uint32_t kPullPiece = 4096;    // else a wavefront per piece of this many in-edges
constexpr uint8_t kVisited = 2;          // state byte of a vertex reached in an earlier step
constexpr int kNumXcd = 8;              // MI355X: 8 XCDs, blocks dispatched round-robin
// The per-XCD live-list counters, one 128-byte line apart so that their
// atomics do not queue on one line.
constexpr uint32_t kLiveCntStride = 32;
constexpr size_t kLiveCntBytes = (size_t)kNumXcd * kLiveCntStride * 4;

// dist[u] + w of a relaxation.  A weight is any 32-bit number, and a sum past
// 2^32 stays at the top, above every distance, where it lowers nothing.  (One
// that wrapped would pass for a short path, and the edges of a cycle could lower
// each other's ends for ever.)
__host__ __device__ inline uint32_t path_sum(uint32_t d, uint32_t w)
{
	const uint32_t x = d + w;
	return x < d ? UINT32_MAX : x;
}

// A traversal whose relaxations are sums as above has at most n frontiers; a
// loop that passes this many has lost its way and stops with GPHI_E_STATE.
__host__ __device__ inline uint64_t level_limit(uint32_t n) { return (uint64_t)n + 2; }

struct Error {
	int code;
	std::string msg;
};

// Per-chunk summary used to skip whole chunks of the tile sweep: the range of
// head tile-rows and tail tile-columns its (non-sentinel) edges touch.
struct ChunkMeta {
	uint32_t row_lo, row_hi, col_lo, col_hi;
};

// 16-bit forms of a chunk's heads and tails.  Heads: offsets from the first
// vertex of the aligned run of tile rows that holds the chunk's rows.  Tails:
// offsets from the smallest tail of each group of kPackGroup consecutive
// edges (a wavefront's quad row in the dense sweep).  flags bit 0 / bit 1:
// every head / tail of the chunk, padding included, fits in 16 bits, so the
// 16-bit form is valid.
constexpr uint32_t kPackGroup = 256;
struct ChunkPack {
	uint32_t hbase, flags, pad0, pad1;
	uint32_t tbase[8];  // per group of kPackGroup edges
};

// Control block of one traversal in the five-kernel loop (128 bytes).  The level loop runs
// on the device: every kernel of a level reads the direction, the level and
// the queue sizes here, and the host reads the block back only every few
// levels to see whether the traversal is done.
struct StepCtrl {
	uint32_t fsize;         // |F| of the frontier just produced
	uint32_t fdeg;          // sum of out-degrees of that frontier
	uint32_t qsize;         // queue entries (frontier vertices with outdeg > 0)
	uint32_t dir;           // direction chosen for expanding it
	uint32_t done;          // frontier empty
	uint32_t facc;          // accumulator: |F|
	unsigned long long qpack;  // accumulator: (queue count << 32) | degree sum
	uint32_t chunks;        // chunks on the live lists of the last dense sweep
	uint32_t level;         // the step being expanded (device-driven loop)
	uint32_t queued;        // BFS: the step expanded last built the next queue itself
	unsigned long long reached, traversed;  // sums of |F| and of sum deg(F) over the steps
	uint32_t col_stale;     // BFS: column counts miss the vertices of queue-building steps
	uint32_t pad[15];
};

// A BFS sparse step whose frontier's edges fill at most this many CSR-push
// tiles builds the next queue itself (its claims append to it); a larger one
// leaves the next frontier to the frontier update's pass over all vertices,
// which then costs less than the appends' reservations on one counter.
constexpr uint32_t kQueueStepTiles = 512;
__host__ __device__ inline bool queue_step(uint32_t dir, uint32_t fdeg)
{
	return dir == 0 && ((uint64_t)fdeg + kSparseTile - 1) / kSparseTile <= kQueueStepTiles;
}
static_assert(sizeof(StepCtrl) == 128, "StepCtrl is 128 bytes");

// The queue of a sparse step (vertices, degree prefix, first entry of each
// kSparseTile-edge tile) in two halves, one per level parity: the step that
// expands level L reads half L & 1, and the next frontier goes to the other.
struct QueueBufs {
	uint32_t *queue, *qoff, *tile_lo;  // half 0
	uint32_t qstride, tstride;         // half 1 starts this many entries later
};
// an entry per vertex is enough for one traversal; the sparse-source queue of
// batch.hip takes one per vertex and kSparseTile out-edges begun
inline uint32_t queue_stride(uint32_t n_pad, uint64_t m) { return n_pad + (uint32_t)(m / kSparseTile); }
inline uint32_t tile_lo_stride(uint64_t m) { return (uint32_t)(m / kSparseTile + 2); }

// Entries of one XCD's live-chunk list: chunk selection hands out chunks in
// groups of 64 (a wavefront's), group g to XCD g % 8.
inline uint32_t live_list_capacity(uint64_t nchunks)
{
	const uint64_t groups = (nchunks + kBlock - 1) / kBlock;
	return (uint32_t)((groups + kNumXcd - 1) / kNumXcd * kBlock);
}

// The direction rule of the level loop of levels.h, |F| + sum deg(F) > M /
// T_RATIO (apps/bfs_simd/bfs.cpp:829-834), with the sum in 64 bits: M may be
// anything below 2^32.  The advance drops the queue of a frontier whose degrees
// alone pass the threshold, so such a step has to be dense; in 32 bits |F| could
// take the sum past 2^32 and back under the threshold, and the step would read a
// queue that was never written.
__host__ __device__ inline bool queue_dropped(uint32_t fdeg, uint32_t threshold) { return fdeg > threshold; }
__host__ __device__ inline bool dense_step(uint32_t fsize, uint32_t fdeg, uint32_t threshold)
{
	return (uint64_t)fsize + fdeg > threshold;
}

// The level loop of levels.h.  LevelRec: a level's totals, the
// accumulators the level before adds to; a ring over the levels, whose entry
// half a ring ahead is cleared as a level starts.  LevelBoard: what the
// device tells the host, in pinned memory.
constexpr uint32_t kLevelRing = 16;
struct LevelRec {
	uint32_t fsize;            // |F|
	uint32_t chunks;           // chunks its dense sweep took
	unsigned long long reached, traversed;  // sums of |F| and of sum deg(F) up to this level
	uint32_t pad0[26];
	// on a line of its own: the advance's blocks each add to both lines
	unsigned long long qpack;  // (queue entries << 32) | sum of out-degrees
	uint32_t pad1[30];
};
static_assert(sizeof(LevelRec) == 256, "LevelRec is two lines");
struct LevelBoard {
	unsigned long long progress;  // (levels started << 1) | ended
	unsigned long long reached, traversed;
	// device wall clock: the first block of the kernel that sets the state up, as
	// it starts; the kernel that sees the end
	unsigned long long t_begin, t_end;
	uint32_t levels, err;
	unsigned long long live[4];         // multi-source: sources with a non-empty frontier,
	unsigned long long step_seq;        // as of the step (BatchRun::step) with this number
	uint4 trace[GPHI_MAX_STEPS];  // per step: direction, |F|, sum deg(F), chunks swept
};
// the ring lies in the memory of gphi_graph::trace, which only the five-kernel loop uses
static_assert(kLevelRing * sizeof(LevelRec) <= (GPHI_MAX_STEPS + 1) * sizeof(uint4), "the ring fits the trace");
// The graphs it serves (2048-edge chunks).  Measured against the five-kernel
// loop without output: BFS 214 -> 96 us at 2^10 vertices (edge factor 16),
// 326 -> 212 at 2^20, 549 -> 524 at 2^23 x 8, 840 -> 613 at 2^24 x 4, but 723 ->
// 742 at 2^23 x 24 and 937 -> 951 at 2^24 x 16, where the live lists' balance
// pays; SSSP 432 -> 167, 995 -> 773, 2914 -> 2557, 3539 -> 3319 and 4550 -> 4284,
// 5022 -> 4572 us.
constexpr uint32_t kTinyVerts = 8192, kTinyChunks = 32, kTinyThreads = 1024;  // one block runs all levels
constexpr uint32_t kSmallVerts = 1u << 24;
constexpr uint32_t kSmallChunksBfs = 1u << 15;
constexpr uint32_t kSmallChunksSssp = 1u << 17;

struct DevGraph {
	uint32_t n = 0;
	uint64_t m = 0;
	uint32_t W = 0, S = 0, side = 0;
	uint64_t ntiles = 0;
	int tile_order = GPHI_TILES_COL_STRIPE;
	uint32_t n_words = 0;      // 32-bit words of a vertex bitmap (covers id n)
	uint32_t n_pad = 0;        // padded vertex count (multiple of 32*kBlock, > n)
	uint64_t m_pad = 0;        // tile arrays padded to whole chunks
	uint64_t nchunks = 0;
	bool has_csr = false, has_tiles = false, weighted = false;
	// CSR (the _untiled files)
	uint32_t *row_off = nullptr;  // n+1
	uint32_t *cols = nullptr;     // m
	uint32_t *csr_w = nullptr;    // m or null
	uint32_t *deg = nullptr;      // n_pad
	// tiled COO (padded)
	uint32_t *heads = nullptr, *tails = nullptr, *coo_w = nullptr;
	ChunkMeta *meta = nullptr;
	uint16_t *heads16 = nullptr, *tails16 = nullptr;  // or null when no window fits (W too wide)
	ChunkPack *pack = nullptr;
	uint8_t *coo_w8 = nullptr;  // 8-bit tile-order weights when every weight is below 256
	uint64_t device_bytes = 0;
};

// No less than what a lane of the server allocates besides the graph: the
// single-source arrays (~42 bytes per vertex, the tile rows' and columns', and
// what grows with the edges: queue, tile partition, live-chunk lists), the
// multi-source masks, levels and bitmaps for max_batch sources, and the in-edge
// arrays of their pull steps (4 bytes per edge, 12 per vertex, pieces).
inline uint64_t lane_state_bytes(const DevGraph &G, uint32_t max_batch)
{
	const uint64_t nw = max_batch <= 64 ? 1 : max_batch <= 128 ? 2 : 4;
	const uint64_t in_edges = max_batch > 1 ? 4 * G.m + 12 * (uint64_t)G.n_pad + G.m / 256 : 0;
	const uint64_t queues = 4ull * 4 * (queue_stride(G.n_pad, G.m) - G.n_pad) + 2ull * 4 * tile_lo_stride(G.m) +
	                        4ull * kNumXcd * live_list_capacity(G.nchunks);
	return (uint64_t)G.n_pad * (42 + 3 * 8 * nw + 64 * nw + 1) + 8 * ((uint64_t)G.side + 1) + queues + in_edges;
}

// PageRank head bands (build_pr_bands).  The heads are cut into bands
// [head_lo, head_hi); within a band, the in-edges of a tail whose heads lie in
// it form a segment.  A band's segments are in tail order and its edges, in
// segment order with heads ascending, one contiguous run of pr_src, swept in
// tiles of kPrTile.  Indices are global over the band arrays; a band's
// segments end with a sentinel (its edge end), its tiles with the last segment.
constexpr uint32_t kSsspBatchMax = GPHI_SSSP_BATCH_MAX;  // distances per vertex of the SSSP batch
constexpr uint32_t kPrTile = 2048;
constexpr uint32_t kBandHeads = 1u << 19;  // heads per band window: 2 MiB of FP32 contributions
// vertices up to which one band is swept: two bands at 1.6M vertices x 21 take
// 124 us an iteration instead of 117, eight at 4.2M x 16 311 instead of 309, and
// twice the set-up
constexpr uint32_t kPrOneBand = 1u << 22;
struct PrBand {
	uint32_t head_lo, head_hi;
	uint32_t edge0, nedges;  // edge0 is a multiple of 4
	uint32_t seg0, nseg;
	uint32_t tile0, ntiles;
};

}  // namespace gphi

struct gphi_ctx {
	int device = 0;
	uint32_t t_ratio = 20;
	hipStream_t stream = nullptr;
	std::mutex mu;
	gphi::Error err{0, ""};
	std::string last;
	// pinned host copy of the control block
	gphi::StepCtrl *h_ctrl = nullptr;
	gphi::LevelBoard *h_board = nullptr;  // in h_ctrl's allocation, written by the kernels of levels.h
	bool board_busy = false;              // a traversal's kernels may still write the board
	double wall_clock_khz = 1e5;          // rate of the device wall clock
	uint32_t *d_word = nullptr;           // a device word of copyout.hip
	// per-step timing: [0] start, [1] init done, [2+2k] sweep k done, [3+2k] update k
	// done, [2*MAX+4+k] chunk selection of dense step k done
	hipEvent_t ev[3 * GPHI_MAX_STEPS + 4];
	bool ev_ok = false;
	bool level_timing = true;  // gphi_set_level_timing
};

struct gphi_graph {
	gphi_ctx *ctx = nullptr;
	gphi::DevGraph g;
	gphi_graph *base = nullptr;  // a view (gphi_graph_view) shares base's graph arrays
	// per-graph traversal state (allocated lazily, reused across calls)
	int32_t *level = nullptr;  // levels (BFS) ; dist (SSSP/BF) aliases via uint32
	int32_t *parent = nullptr;
	uint32_t *dist = nullptr;
	// per-vertex state byte: 0 not reached, 1 reached in the current step,
	// kVisited (BFS) reached in an earlier step; SSSP and multi-source use 0/1
	uint8_t *flag = nullptr;
	uint32_t *visited = nullptr;  // BFS: bitmap of the vertices reached in earlier steps
	uint32_t *cur = nullptr;      // frontier bitmap of the current step
	uint32_t *row_stamp = nullptr, *col_unvis = nullptr;
	// sparse-step queue, two halves each (QueueBufs): queue / qoff of
	// 2 * queue_len entries, tile_lo of 2 * (m / kSparseTile + 2)
	uint32_t *queue = nullptr, *qoff = nullptr, *tile_lo = nullptr;
	uint32_t queue_len = 0;
	gphi::QueueBufs queue_bufs() const
	{
		return gphi::QueueBufs{queue, qoff, tile_lo, queue_len, gphi::tile_lo_stride(g.m)};
	}
	gphi::StepCtrl *ctrl = nullptr;
	gphi::LevelRec *rec() const { return reinterpret_cast<gphi::LevelRec *>(trace); }  // kLevelRing entries
	uint4 *blk_cnt = nullptr;  // per update block: |F|, queue entries, degree sum
	uint2 *blk_base = nullptr; // per update block: queue and degree prefix
	uint2 *wave_cnt = nullptr; // per update wavefront: queue entries, degree sum
	uint32_t *live = nullptr;  // per-XCD lists of live chunks of a dense step
	uint32_t *live_cnt = nullptr;
	uint4 *trace = nullptr;    // five-kernel loop, per step: direction, |F|, sum deg(F), chunks swept
	// PageRank: one allocation holding rank, sum and contrib (n_pad each) and
	// two partial sums per tile
	float *rank = nullptr, *sum = nullptr, *contrib = nullptr;
	// PageRank head bands (build_pr_bands; built once, independent of W and S):
	// the heads band by band (pr_src; in_src itself when there is one band),
	// each segment's first edge and tail, and the segment of each tile's first
	// edge; one allocation, pr_mem
	std::vector<gphi::PrBand> pr_bands;
	void *pr_mem = nullptr;
	const uint32_t *pr_src = nullptr;
	uint32_t *pr_off = nullptr, *pr_tail = nullptr, *pr_tile = nullptr;
	uint32_t pr_ntiles = 0;
	// multi-source BFS (batch.hip): per-vertex source masks and uint8 levels
	uint32_t batch_words = 0;  // 64-bit words per vertex the buffers were sized for
	// leading mask words that front / next (and the touched bitmap) are known
	// to hold as zero: a traversal that runs to its end leaves them so
	uint64_t batch_clean_words = 0;
	unsigned long long *b_front = nullptr, *b_seen = nullptr, *b_next = nullptr;
	uint8_t *b_level = nullptr;
	unsigned long long *b_sums = nullptr;
	unsigned long long *b_live = nullptr;  // sources with a non-empty frontier, then the per-block slots
	uint32_t *b_touch = nullptr;           // bitmap: vertices whose next mask got a bit this step
	uint32_t *b_scount = nullptr;          // in b_touch's allocation: new vertices per source, per slot
	uint32_t *b_aux = nullptr;             // per-slot start levels, then the error flag
	// multi-source SSSP (sssp_batch.hip): kSsspBatchMax distances per vertex
	// (vertex-major, n_pad rows), then the sources
	uint32_t *sb_dist = nullptr;
	// hop relaxation (hops.hip): sweep records, row sweeps, vertex stamps
	uint8_t *hop = nullptr;
	// in-edge arrays of the pull steps (built once, independent of W and S)
	uint32_t *in_off = nullptr, *in_src = nullptr;
	// the weights of in_src's edges (build_in_weights): 1 byte when every
	// weight is below 256, else 4
	uint8_t *in_w8 = nullptr;
	uint32_t *in_w32 = nullptr;
	uint2 *pieces = nullptr;
	uint32_t npieces = 0;
	uint64_t in_bytes = 0;
};

namespace gphi {
int set_error(gphi_ctx *ctx, int code, const char *fmt, ...);
// true when an allocation failure injected by gphi_debug_fail_alloc is due now
bool take_injected_alloc_failure();
int hip_fail(gphi_ctx *ctx, hipError_t e, const char *what, const char *file, int line);

// device memory (GPHI_E_OOM when it is exhausted); *acc, if any, counts the bytes
int dmalloc(gphi_ctx *ctx, void **p, size_t bytes, uint64_t *acc);

void fill_words(gphi_ctx *ctx, uint32_t *p, uint64_t count, uint32_t value);  // on ctx's stream

// Pinned memory that kernels write while the host looks at it (the level board,
// staging slots and their flags): asked for as coherent, which a plain request
// is only if the environment's HIP_HOST_COHERENT does not say otherwise.
inline hipError_t pinned_alloc(void **p, size_t bytes)
{
	return hipHostMalloc(p, bytes, hipHostMallocPortable | hipHostMallocCoherent);
}

// device-side entry points (device.hip, hops.hip, pagerank.hip)
int upload_graph(gphi_ctx *ctx, const gphi_graph_desc *d, gphi_graph *gr);
void free_graph_device(gphi_graph *gr);
void free_traversal_state(gphi_graph *gr);
int retile_graph(gphi_graph *gr, uint32_t W, uint32_t S, int tile_order);
int build_in_edges(gphi_graph *gr);
int build_pr_bands(gphi_graph *gr);  // after build_in_edges
int build_in_weights(gphi_graph *gr);  // after build_in_edges; weighted graphs with CSR
int run_bfs(gphi_graph *gr, uint32_t src, int32_t *levels, int32_t *parents, gphi_stats *st);
int run_bfs_noalloc(gphi_graph *gr, uint32_t src, int32_t *levels_dev, int32_t *parents_dev, gphi_stats *st);
void noalloc_setup(int device);  // with `device` current, once per device (gphi_open)
int run_sssp(gphi_graph *gr, uint32_t src, uint32_t *dist, gphi_stats *st);
int run_pagerank(gphi_graph *gr, uint32_t iters, float damping, float init, float *rank,
                 float *ms);
int run_bellman_ford(gphi_graph *gr, uint32_t src, uint32_t max_sweeps, uint32_t *dist,
                     uint32_t *sweeps_run, float *ms);

int finish_tiles(gphi_ctx *ctx, gphi_graph *gr);
void free_chunk_summaries(DevGraph &G);  // meta and the 16-bit tile forms
int count_active_tiles(gphi_graph *gr, const int32_t *levels, const std::vector<uint32_t> &dense_steps,
                       std::vector<double> &e_act, std::vector<double> &t_act);
int tile_offsets(gphi_graph *gr, uint32_t *out);
int download_graph(gphi_graph *gr, uint32_t *deg, uint32_t *cols, uint32_t *cw, uint32_t *th,
                   uint32_t *tt, uint32_t *tw);

int ensure_traversal_state(gphi_graph *gr);
// the level loop of small graphs without per-level timing (small.hip); the
// traversal has ended, and st is filled in, when it returns
bool small_graph(const DevGraph &G, bool bfs);
template <bool kBfs>
int small_level_loop(gphi_graph *gr, uint32_t src, gphi_stats *st, uint32_t *steps);
// the BFS level loop of run_bfs on gr's state buffers (set up by the caller)
int bfs_level_loop(gphi_graph *gr, uint32_t src, gphi_stats *st);

// results to host arrays (copyout.hip); the caller's arrays are complete on return
// n 4-byte words; with state bytes, -1 where the byte is 0
int out_words(gphi_ctx *ctx, const void *dev, const uint8_t *state, uint32_t n, void *dst);
// BFS levels of gr's last traversal, none above `deepest`
int out_bfs_levels(gphi_graph *gr, uint32_t deepest, int32_t *levels);
// rows of the multi-source levels, row i that of slot slots[i]; unreached is
// 255 (uint8) or -1 (int32)
template <class T>
int out_batch_rows(gphi_graph *gr, const uint32_t *slots, uint32_t deepest, uint32_t nrows, T *const *rows);
// n distances of an array of n_pad, unreached ones `none` (in the padding too)
int out_dist(gphi_ctx *ctx, const uint32_t *dev, uint32_t none, uint32_t n, uint32_t n_pad, uint32_t *dst);
// the first k sources' distances of the multi-source SSSP (null rows are skipped)
int out_sssp_rows(gphi_graph *gr, uint32_t k, uint32_t *const *rows);
// gphi_open / gphi_close: the staging memory is freed with the last context
void out_context_opened();
void out_context_closed();
// blocks of `block` threads of a kernel that fit the device at once, a multiple of the XCD count
unsigned resident_grid(const void *kernel, unsigned block = kBlock);
int run_bfs_batch(gphi_graph *gr, const uint32_t *srcs, uint32_t k, uint8_t *levels, gphi_stats *st);
// the multi-source state of gr for nw mask words: traversal state, in-edge
// arrays, masks, levels (idempotent)
int batch_prepare(gphi_graph *gr, uint32_t nw);
// weighted SSSP from k <= kSsspBatchMax sources in one traversal
// (sssp_batch.hip); rows[i]: n distances of source i to copy out, or null
// (rows itself may be null)
int run_sssp_batch(gphi_graph *gr, const uint32_t *srcs, uint32_t k, uint32_t *const *rows, gphi_stats *st);
int sssp_batch_prepare(gphi_graph *gr);  // its state, in-edges and weights (idempotent)

// A multi-source traversal (batch.hip).  gphi_bfs_batch runs one to its end
// on the device; the serving loop advances one level by level, admitting new
// sources into free slots between levels and reading out the rows of the
// slots whose frontier has emptied.  Slot i is bit i of the masks.
constexpr uint32_t kBatchMaxSources = 256;
struct BatchRun {
	gphi_graph *gr = nullptr;
	uint32_t nw = 0;       // 64-bit mask words per vertex
	uint32_t cap = 0;      // slots (64 * nw)
	uint32_t used = 0;     // slots handed out (slots are not reused within a run)
	uint32_t levels = 0;   // levels expanded
	bool done = false;     // the union frontier is empty
	std::vector<uint32_t> slot_src, slot_start;  // per slot: source vertex, level it joined at
	uint64_t mask_words = 0;                     // n_pad * nw
	uint64_t prev_clean = 0;                     // gr->batch_clean_words when the run began
	unsigned long long live[4] = {0, 0, 0, 0};   // sources with a non-empty frontier (after step)
	unsigned long long pairs[2] = {0, 0};        // reached (source, vertex) pairs, their out-degrees
	// clears the state and seeds k sources (slots 0..k-1); capacity picks the
	// mask width (1..256 sources)
	int begin(gphi_graph *g, uint32_t capacity, const uint32_t *srcs, uint32_t k);
	// one level, then k new sources join (slots used..used+k-1); learns the
	// live mask and whether the traversal ended
	int step(const uint32_t *srcs, uint32_t k);
	int run_to_end(gphi_stats *st);  // the remaining levels, on the device
	// levels of the given slots into host rows of n (unreached: 255 in uint8 rows, -1 in int32 ones)
	template <class T>
	int copy_rows(const uint32_t *slots, uint32_t ns, T *const *rows);
	int seed(const uint32_t *srcs, uint32_t k, uint32_t start_level);
};

// generator + tool pipeline on the device (gen.hip)
int generate_graph(gphi_ctx *ctx, const gphi_rmat_spec *sp, uint32_t W, uint32_t S, int reorder,
                   const gphi_weight_spec *ws, int tile_order, gphi_graph *gr);
void glibc_rand_seq(uint32_t seed, uint64_t n, int32_t *out);
void random_perm_host(uint32_t n, uint64_t seed, uint32_t *perm);

// host text formats (formats.cpp)
// moves st[0..6] (degrees, csr, csr w, heads, tails, tile w, offsets) into a new host graph
int host_adopt(const gphi_graph_desc *d, std::vector<uint32_t> *st, gphi_host_graph **out);
int read_text_graph(gphi_ctx *ctx, const char *prefix, uint32_t W, uint32_t S, int weighted,
                    bool row_major, gphi_graph_desc *d, std::vector<uint32_t> *store);
}  // namespace gphi

#define GPHI_HIP(ctx, call)                                                    \
	do {                                                                       \
		hipError_t e_ = (call);                                                \
		if (e_ != hipSuccess) return gphi::hip_fail((ctx), e_, #call, __FILE__, __LINE__); \
	} while (0)
