// Device rings: frontier BFS levels and a counting sort by level (see levels.hpp).
#include "levels.hpp"

#include <algorithm>
#include <memory>
#include <mutex>
#include <type_traits>

#include "gp_internal.hpp"

namespace gp {

// BFS state: launch k expands the cnt[(k - 1) & 3] vertices queued by the one
// before (queue half k & 1) and queues the next ones in the other half through
// cnt[k & 3].  serial numbers the launches over the life of the state (the marks
// that keep a vertex from being queued twice by one launch); a launch reads it
// from slot (k - 1) & 3 and workgroup 0 publishes the next in slot k & 3.
struct LevelState {
	uint32_t serial[4];
	uint32_t cnt[4];
	uint32_t done, max_level;
};

__global__ void k_lv_zero(uint32_t *p, uint32_t n)
{
	for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) p[v] = 0;
}

// Levels before the first round: unreached everywhere.
__global__ void k_lv_clear(uint32_t *level, uint32_t n)
{
	for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += gridDim.x * blockDim.x) level[v] = GP_NIL;
}

// Seeds the BFS: sources src[first, ns) get level 0 and form the frontier of
// launch 0.
__global__ void k_lv_seed(const uint32_t *src, uint32_t first, uint32_t ns, uint32_t *level, uint32_t *queue,
                          LevelState *ls, uint32_t fresh)
{
	for (uint32_t q = first + threadIdx.x; q < ns; q += blockDim.x) {
		level[src[q]] = 0;
		queue[q - first] = src[q];
	}
	if (threadIdx.x == 0) {
		uint32_t s = 0;
		if (!fresh)
			for (uint32_t q = 0; q < 4; q++) s = max(s, ls->serial[q]);
		for (uint32_t q = 0; q < 4; q++) { ls->serial[q] = s; ls->cnt[q] = 0; }
		ls->cnt[3] = ns - first;
		ls->max_level = 0;
		ls->done = ns > first ? 0u : 1u;
	}
}

__global__ void k_link8(const uint32_t *fan_off, const uint32_t *fan, const uint8_t *closed, uint32_t nv,
                        uint32_t *link8)
{
	const size_t n8 = (size_t) nv * LINK_ROW;   // vertex ids stay below 2^31 (build_che)
	for (size_t q = blockIdx.x * blockDim.x + threadIdx.x; q < n8; q += gridDim.x * blockDim.x) {
		const uint32_t v = (uint32_t) (q / LINK_ROW), k = (uint32_t) (q % LINK_ROW);
		const uint32_t s = fan_off[v], c = fan_off[v + 1] - s;
		const uint32_t n = (c && closed[v]) ? c - 1 : c;
		uint32_t id = k < n ? fan[s + k] : GP_NIL;
		if (k == LINK_ROW - 1 && n > LINK_ROW) id |= LONG_LINK;
		link8[q] = id;
	}
}

// LV_DEPTH levels of the frontier in one launch.  A workgroup takes up to
// LV_CHUNK queued vertices into LDS and pushes level + 1 to their links, eight
// lanes a vertex; a vertex whose level dropped (exactly one atomicMin sees it
// drop) is expanded next by the workgroup that lowered it, from LDS, and the
// vertices of the last depth form the next launch's frontier.  A drop is always
// expanded, here or by a later launch, so the BFS ends at the hop distances in
// any order; as all workgroups start from one level, each vertex is lowered
// once but for the seams between workgroups.
//
// Bound by the round trips of a level.  A lane asks for its neighbour's own
// link with the atomic on its level, so the next level starts from LDS and a
// level costs one round trip (~1.3 us) instead of a launch and four (state,
// queue, fan offsets, fan, atomic).  1M-vertex mesh, one source: 992 launches
// of 5.9 us before (5.8 ms), 58 of 22 us now (1.29 ms); 201k vertices, 16
// sources: 1.23 -> 0.31 ms; 10k vertices: 0.39 -> 0.13 ms.  24 or 32
// levels a launch and 64, 128 or 512 threads were no faster on all three.
// (Running spatial tiles of 1,024 vertices to their end in LDS instead needs
// ~200 launches of 50-120 us on the 1M mesh: a tile entered from one side first
// is corrected again and again.)
constexpr uint32_t LV_T = 256, LV_CHUNK = LV_T / LINK_ROW, LV_DEPTH = 16, LV_Q = 512, LV_SPREAD = 512;

struct LvArgs {
	const uint32_t *link8, *fan_off, *fan;
	uint32_t *level, *queue, *mark;
	LevelState *ls;
	uint32_t nv;
};

__global__ __launch_bounds__(LV_T) void k_lv_step(LvArgs a, uint32_t k4)
{
	__shared__ uint32_t s_link[2][LV_Q][LINK_ROW], s_id[2][LV_Q], s_lev[2][LV_Q], s_n[3];
	LevelState *ls = a.ls;
	const uint32_t tid = threadIdx.x, lane = tid & 63u, slot = tid % LINK_ROW, group = tid / LINK_ROW;
	const uint32_t kp = (k4 + 3u) & 3u;
	const uint32_t n = ls->cnt[kp], serial = ls->serial[kp] + 1;
	const uint32_t *q_in = a.queue + (size_t) (k4 & 1u) * a.nv;
	uint32_t *q_out = a.queue + (size_t) ((k4 + 1u) & 1u) * a.nv;
	if (blockIdx.x == 0 && tid == 0) {
		ls->serial[k4] = serial;
		ls->cnt[(k4 + 1u) & 3u] = 0;
		if (n == 0) ls->done = 1;
	}
	// Vertex w to the next launch's frontier (every lane of the wave calls).
	auto queue_next = [&](bool want, uint32_t w) {
		const bool first = want && atomicExch(&a.mark[w], serial) != serial;
		const unsigned long long m = __ballot(first);
		if (!m) return;
		uint32_t base = 0;
		if (lane == 0) base = atomicAdd(&ls->cnt[k4], (uint32_t) __popcll(m));
		base = __shfl(base, 0);
		if (first) q_out[base + (uint32_t) __popcll(m & ((1ull << lane) - 1ull))] = w;
	};
	// A short frontier is spread over LV_SPREAD workgroups, one vertex each if
	// need be: the lists stay short (a 16-source seed by one workgroup: 190 us).
	const uint32_t chunk = max(1u, min(LV_CHUNK, n / LV_SPREAD));
	for (uint32_t c0 = blockIdx.x * chunk; c0 < n; c0 += gridDim.x * chunk) {
		if (tid == 0) { s_n[0] = min(chunk, n - c0); s_n[1] = 0; s_n[2] = 0; }
		{
			const uint32_t i = c0 + group;
			if (group < chunk && i < n) {
				const uint32_t v = q_in[i];
				s_link[0][group][slot] = a.link8[(size_t) v * LINK_ROW + slot];
				if (slot == 0) { s_id[0][group] = v; s_lev[0][group] = a.level[v]; }
			}
		}
		__syncthreads();
		for (uint32_t d = 0;; d++) {
			const uint32_t cur = d & 1u, nq = s_n[d % 3u];
			if (nq == 0) break;
			const bool last = d + 1 == LV_DEPTH;
			if (tid == 0) s_n[(d + 2) % 3u] = 0;   // read at depth d - 1, counted from depth d + 1
			for (uint32_t b = 0; b < nq; b += LV_T / LINK_ROW) {
				const uint32_t i = b + group;
				uint32_t w = i < nq ? s_link[cur][i][slot] : GP_NIL;
				const bool more = w != GP_NIL && (w & LONG_LINK);
				if (w != GP_NIL) w &= ~LONG_LINK;
				const uint32_t l1 = i < nq ? s_lev[cur][i] + 1 : 0u;
				bool won = false;
				uint4 r0 = make_uint4(0, 0, 0, 0), r1 = r0;
				if (w != GP_NIL) {
					const uint4 *row = (const uint4 *) (a.link8 + (size_t) w * LINK_ROW);
					r0 = row[0];
					r1 = row[1];
					won = atomicMin(&a.level[w], l1) > l1;
				}
				bool out = won && last;
				// Room in the next depth's list: one LDS counter add per wave.
				const unsigned long long m = last ? 0ull : __ballot(won);
				uint32_t at = 0;
				if (m) {
					if (lane == 0) at = atomicAdd(&s_n[(d + 1) % 3u], (uint32_t) __popcll(m));
					at = __shfl(at, 0) + (uint32_t) __popcll(m & ((1ull << lane) - 1ull));
				}
				if (won && !last) {
					if (at < LV_Q) {
						*(uint4 *) &s_link[cur ^ 1u][at][0] = r0;
						*(uint4 *) &s_link[cur ^ 1u][at][4] = r1;
						s_id[cur ^ 1u][at] = w;
						s_lev[cur ^ 1u][at] = l1;
					} else {
						out = true;   // no room: the next launch expands it
					}
				}
				queue_next(out, w);
				if (__ballot(more)) {
					// Links longer than a row: lane 7 of the vertex walks the
					// rest in the fan table.
					uint32_t e = 0, e1 = 0;
					if (more) {
						const uint32_t v = s_id[cur][i];
						e = a.fan_off[v] + LINK_ROW;
						e1 = a.fan_off[v + 1];
					}
					while (__ballot(e < e1)) {
						const bool act = e < e1;
						const uint32_t u = act ? a.fan[e] : 0u;
						queue_next(act && atomicMin(&a.level[u], l1) > l1, u);
						e++;
					}
				}
			}
			__syncthreads();
			if (tid == 0) s_n[(d + 1) % 3u] = last ? 0u : min(s_n[(d + 1) % 3u], LV_Q);
			__syncthreads();
		}
		__syncthreads();
	}
}

// Counting sort of the reached vertices by level and, inside a level, by slot
// count (longest fans first), so that a 64-position chunk of a ring holds fans
// of one length: histogram of the keys (and the largest level), exclusive scan
// into the cursors and limits (one workgroup), scatter into sorted[].  The
// order inside a level is free (a sweep relaxes whole rings from the previous
// buffer).  Global atomics on a few thousand counters serialise, so each
// workgroup counts a block of SORT_T * PER vertices in LDS bins (keys lo .. lo +
// SORT_BINS - 1 of the block; keys past them, rare, count globally) and adds
// or reserves one global count per key present in the block.  Small meshes are
// bound by a workgroup's own chain: with two vertices a thread, their keys held in
// registers, and only the bins in use cleared, histogram and scatter of 66k vertices
// take 4.9 and 5.3 us instead of 13.6 and 17.  Large ones are bound by the global
// counts, so by the number of blocks: eight a thread.  Histogram and scatter with
// two / eight vertices a thread, one source: 262k vertices 15.4 / 23.2 us, 410k
// 20.7 / 25.9, 608k 21.5 / 24.6, 810k 29.9 / 27.9, 1M 31.6 / 27.6; sixteen sources:
// 262k 14.3 / 22.2, 410k 18.8 / 22.0, 608k 26.7 / 25.2, 810k 33.4 / 26.0.
constexpr uint32_t SORT_SMALL = 1u << 19;
constexpr uint32_t SORT_BINS = 12288, SORT_T = 1024;

// Sort key of vertex v: level * KS + slot class (KS or more slots first, then
// KS - 1, ..., 1), NIL when unreached.
__device__ __forceinline__ uint32_t sort_key(const uint32_t *level, const uint32_t *fan_off, const uint8_t *closed,
                                             uint32_t v)
{
	const uint32_t l = level[v], n = fan_off[v + 1] - fan_off[v];
	const uint32_t c = closed[v];   // asked for with the others
	const uint32_t sl = (n && c) ? n - 1 : n;
	return l == GP_NIL ? GP_NIL : l * LEVEL_KEYS + (LEVEL_KEYS - min(max(sl, 1u), LEVEL_KEYS));
}

struct KeySrc {
	const uint32_t *level, *fan_off;
	const uint8_t *closed;
	__device__ uint32_t operator()(uint32_t v) const { return sort_key(level, fan_off, closed, v); }
};

// The keys of the workgroup's SORT_T * PER vertices, a thread's in registers (NIL
// past n); the smallest and largest of them in every thread.
template <uint32_t PER>
__device__ __forceinline__ void block_keys(const KeySrc &key, uint32_t n, uint32_t (&k)[PER], uint32_t *red, uint32_t &lo,
                                           uint32_t &hi)
{
	const uint32_t b0 = blockIdx.x * SORT_T * PER + threadIdx.x;
	lo = GP_NIL; hi = 0;
#pragma unroll
	for (uint32_t q = 0; q < PER; q++) k[q] = b0 + q * SORT_T < n ? key(b0 + q * SORT_T) : GP_NIL;
#pragma unroll
	for (uint32_t q = 0; q < PER; q++)
		if (k[q] != GP_NIL) { lo = min(lo, k[q]); hi = max(hi, k[q]); }
	for (uint32_t o = 32; o > 0; o >>= 1) {
		lo = min(lo, (uint32_t) __shfl_xor(lo, o));
		hi = max(hi, (uint32_t) __shfl_xor(hi, o));
	}
	const uint32_t w = threadIdx.x >> 6;
	if ((threadIdx.x & 63u) == 0) { red[w] = lo; red[16 + w] = hi; }
	__syncthreads();
	lo = GP_NIL; hi = 0;
	for (uint32_t q = 0; q < SORT_T / 64; q++) { lo = min(lo, red[q]); hi = max(hi, red[16 + q]); }
}

// LDS counts of the block's keys lo .. lo + range - 1; the others are
// counted in glob (when given).
template <uint32_t PER>
__device__ __forceinline__ void block_key_counts(const uint32_t (&k)[PER], uint32_t lo, uint32_t range, uint32_t *bins,
                                                 uint32_t *glob)
{
	for (uint32_t q = threadIdx.x; q < range; q += SORT_T) bins[q] = 0;
	__syncthreads();
#pragma unroll
	for (uint32_t q = 0; q < PER; q++) {
		if (k[q] == GP_NIL) continue;
		if (k[q] - lo < SORT_BINS) atomicAdd(&bins[k[q] - lo], 1u);
		else if (glob) atomicAdd(&glob[k[q]], 1u);
	}
	__syncthreads();
}

template <uint32_t PER>
__global__ __launch_bounds__(SORT_T) void k_lv_hist(KeySrc key, uint32_t n, uint32_t *hist, LevelState *ls)
{
	__shared__ uint32_t bins[SORT_BINS];
	__shared__ uint32_t red[32];
	uint32_t k[PER], lo, hi;
	block_keys<PER>(key, n, k, red, lo, hi);
	if (lo == GP_NIL) return;   // nothing reached in the block (uniform)
	const uint32_t range = min(SORT_BINS, hi - lo + 1);
	block_key_counts<PER>(k, lo, range, bins, hist);
	for (uint32_t q = threadIdx.x; q < range; q += SORT_T)
		if (bins[q]) atomicAdd(&hist[lo + q], bins[q]);
	if (threadIdx.x == 0) atomicMax(&ls->max_level, hi / LEVEL_KEYS);
}

// Exclusive scan of the key counts into the scatter cursors; limits[l] = the
// first position of level l, limits[max_level + 1] = the reached count.
__global__ __launch_bounds__(1024) void k_lv_scan(uint32_t *hist, uint32_t *limits, uint32_t *nl, const LevelState *ls)
{
	__shared__ uint32_t part[1024];
	const uint32_t nlev = ls->max_level + 1, nb = nlev * LEVEL_KEYS;
	uint32_t carry = 0;
	for (uint32_t b0 = 0; b0 < nb; b0 += 1024) {
		const uint32_t q = b0 + threadIdx.x;
		const uint32_t x = q < nb ? hist[q] : 0u;
		part[threadIdx.x] = x;
		__syncthreads();
		for (uint32_t o = 1; o < 1024; o <<= 1) {
			const uint32_t y = threadIdx.x >= o ? part[threadIdx.x - o] : 0u;
			__syncthreads();
			part[threadIdx.x] += y;
			__syncthreads();
		}
		const uint32_t excl = part[threadIdx.x] + carry - x;
		if (q < nb) {
			hist[q] = excl;   // becomes the scatter cursor of key q
			if (q % LEVEL_KEYS == 0) limits[q / LEVEL_KEYS] = excl;
		}
		const uint32_t tot = part[1023];
		__syncthreads();
		carry += tot;
	}
	if (threadIdx.x == 0) { limits[nlev] = carry; *nl = nlev + 1; }
}

template <uint32_t PER>
__global__ __launch_bounds__(SORT_T) void k_lv_scatter(KeySrc key, uint32_t n, uint32_t *cursor, uint32_t *sorted)
{
	__shared__ uint32_t bins[SORT_BINS];
	__shared__ uint32_t red[32];
	uint32_t k[PER], lo, hi;
	block_keys<PER>(key, n, k, red, lo, hi);
	if (lo == GP_NIL) return;
	const uint32_t range = min(SORT_BINS, hi - lo + 1);
	block_key_counts<PER>(k, lo, range, bins, nullptr);
	// Reserve the block's run of each key; the bins become its cursors.
	for (uint32_t q = threadIdx.x; q < range; q += SORT_T)
		if (bins[q]) bins[q] = atomicAdd(&cursor[lo + q], bins[q]);
	__syncthreads();
	const uint32_t b0 = blockIdx.x * SORT_T * PER + threadIdx.x;
#pragma unroll
	for (uint32_t q = 0; q < PER; q++) {
		if (k[q] == GP_NIL) continue;
		sorted[k[q] - lo < SORT_BINS ? atomicAdd(&bins[k[q] - lo], 1u) : atomicAdd(&cursor[k[q]], 1u)] = b0 + q * SORT_T;
	}
}

// Slot rows of each 64-position chunk of sorted[] (its longest fan; 0 past the
// reached vertices), one wave per chunk.
__global__ void k_lv_chunk_slots(const uint32_t *sorted, const uint32_t *limits, const uint32_t *nl,
                                 const uint32_t *fan_off, const uint8_t *closed, uint32_t nchunks, uint32_t *cslots)
{
	const uint32_t nr = limits[*nl - 1];
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t nw = (gridDim.x * blockDim.x) >> 6;
	for (uint32_t c = (blockIdx.x * blockDim.x + threadIdx.x) >> 6; c < nchunks; c += nw) {
		const uint32_t p = (c << 6) + lane;
		uint32_t sl = 0;
		if (p < nr) {
			const uint32_t v = sorted[p];
			const uint32_t n = fan_off[v + 1] - fan_off[v];
			sl = (n && closed[v]) ? n - 1 : n;
		}
		for (uint32_t o = 32; o > 0; o >>= 1) sl = max(sl, (uint32_t) __shfl_xor(sl, o));
		if (lane == 0) cslots[c] = sl;
	}
}

// out[q] = in[0] + ... + in[q - 1] for q <= n (one workgroup).
__global__ __launch_bounds__(1024) void k_exclusive_scan(const uint32_t *in, uint32_t n, uint32_t *out)
{
	__shared__ uint32_t part[1024];
	uint32_t carry = 0;
	for (uint32_t b0 = 0; b0 < n; b0 += 1024) {
		const uint32_t q = b0 + threadIdx.x;
		const uint32_t x = q < n ? in[q] : 0u;
		part[threadIdx.x] = x;
		__syncthreads();
		for (uint32_t o = 1; o < 1024; o <<= 1) {
			const uint32_t y = threadIdx.x >= o ? part[threadIdx.x - o] : 0u;
			__syncthreads();
			part[threadIdx.x] += y;
			__syncthreads();
		}
		if (q < n) out[q] = part[threadIdx.x] + carry - x;
		const uint32_t tot = part[1023];
		__syncthreads();
		carry += tot;
	}
	if (threadIdx.x == 0) out[n] = carry;
}

Levels::~Levels()
{
	if (stream) (void) hipStreamSynchronize(stream);
	for (void *p : { (void *) level, (void *) queue, (void *) mark, (void *) hist, (void *) sorted, (void *) limits,
	                 (void *) nl, (void *) ls, (void *) cslots, (void *) coff })
		(void) pool_free(p);
	pinned_free(h_ls);
	for (hipEvent_t e : ev)
		if (e) (void) hipEventDestroy(e);
}

static uint32_t fill_grid(uint32_t n) { return std::max<uint32_t>(1, std::min<uint32_t>(2048, (n + 255) / 256)); }

// The mesh's link rows, built once on first use (several threads may ask).
int link_rows(DeviceMesh *dm)
{
	static std::mutex mu;
	std::lock_guard<std::mutex> lock(mu);
	if (dm->link8) return GP_OK;
	uint32_t *p = nullptr;
	if (device_malloc(&p, 4ull * LINK_ROW * dm->nv) != hipSuccess)
		return fail(GP_ERR_NOMEM, "levels: device allocation failed");
	k_link8<<<fill_grid(dm->nv), 256>>>(dm->fan_off, dm->fan, dm->closed, dm->nv, p);
	const hipError_t e = hipGetLastError() != hipSuccess ? hipErrorUnknown : hipDeviceSynchronize();
	if (e != hipSuccess) {
		(void) hipFree(p);
		return fail(GP_ERR_HIP, "levels: link rows: %s", hipGetErrorString(e));
	}
	dm->link8 = p;
	return GP_OK;
}

int Levels::create(DeviceMesh *mesh, hipStream_t s)
{
	dm = mesh;
	nv = mesh->nv;
	stream = s;
	if (int rc = link_rows(mesh)) return rc;
	if (pool_malloc(&level, 4ull * nv) != hipSuccess || pool_malloc(&queue, 8ull * nv) != hipSuccess ||
	    pool_malloc(&mark, 4ull * nv) != hipSuccess ||
	    pool_malloc(&hist, 4ull * ((size_t) nv * LEVEL_KEYS + 1)) != hipSuccess ||
	    pool_malloc(&sorted, 4ull * nv) != hipSuccess || pool_malloc(&cslots, 4ull * (nchunks() + 1)) != hipSuccess ||
	    pool_malloc(&coff, 4ull * (nchunks() + 1)) != hipSuccess ||
	    pool_malloc(&limits, 4ull * (nv + 2)) != hipSuccess || pool_malloc(&nl, 4) != hipSuccess ||
	    pool_malloc(&ls, sizeof(LevelState)) != hipSuccess || pinned_malloc(&h_ls, 3 * sizeof(LevelState)) != hipSuccess)
		return fail(GP_ERR_NOMEM, "levels: device allocation failed");
	static_assert(sizeof(LevelInfo) <= sizeof(LevelState), "the sizes take a third snapshot's room");
	h_info = (LevelInfo *) (h_ls + 2);
	GP_HIP(hipEventCreateWithFlags(&ev[0], hipEventDisableTiming));
	GP_HIP(hipEventCreateWithFlags(&ev[1], hipEventDisableTiming));
	k_lv_zero<<<fill_grid(nv), 256, 0, stream>>>(mark, nv);
	GP_HIP(hipGetLastError());
	// One workgroup per LV_CHUNK frontier vertices; frontiers past the grid loop.
	lv_grid = std::max<uint32_t>(1, std::min<uint32_t>(1024, (nv + LV_CHUNK - 1) / LV_CHUNK));
	fresh = true;
	return GP_OK;
}

void Levels::clear() { k_lv_clear<<<fill_grid(nv), 256, 0, stream>>>(level, nv); }

void Levels::seed(const uint32_t *d_src, uint32_t first, uint32_t ns)
{
	k_lv_seed<<<1, 256, 0, stream>>>(d_src, first, ns, level, queue, ls, fresh ? 1u : 0u);
	fresh = false;
}

// Launches in rounds of LV until the state reports done, two rounds in flight:
// each round is followed by a kernel that writes the state into its pinned
// snapshot and an event; the host waits for the older round while the newer one
// runs (a round queued behind the one that finishes finds nothing queued).  Few
// and long launches: one by one on the stream, no graph to build.
constexpr uint32_t LV = 4;   // a multiple of 4 (the state slots)

int Levels::expand()
{
	GP_HIP(hipGetLastError());
	const LvArgs a{ dm->link8, dm->fan_off, dm->fan, level, queue, mark, ls, nv };
	auto round = [&](uint32_t s) -> int {
		for (uint32_t q = 0; q < LV; q++) k_lv_step<<<lv_grid, LV_T, 0, stream>>>(a, q & 3u);
		snapshot(ls, h_ls + s, stream);
		GP_HIP(hipGetLastError());
		GP_HIP(hipEventRecord(ev[s], stream));
		return GP_OK;
	};
	int rc = round(0);
	if (rc) return rc;
	for (uint32_t reps = 0, cur = 0;; reps++, cur ^= 1u) {
		// Every launch but the last lowers at least one vertex.
		if (reps > nv / LV + 2) return fail(GP_ERR_KERNEL, "levels: BFS did not finish");
		if ((rc = round(cur ^ 1u))) return rc;
		GP_HIP(hipEventSynchronize(ev[cur]));
		if (h_ls[cur].done) break;
	}
	GP_HIP(hipStreamSynchronize(stream));
	return GP_OK;
}

void Levels::sort()
{
	const uint32_t nk = nv * LEVEL_KEYS + 1;
	const uint32_t g = fill_grid(nk);
	const KeySrc key{ level, dm->fan_off, dm->closed };
	k_lv_zero<<<g, 256, 0, stream>>>(hist, nk);
	if (nv <= SORT_SMALL) {
		const uint32_t gb = (nv + 2 * SORT_T - 1) / (2 * SORT_T);
		k_lv_hist<2><<<gb, SORT_T, 0, stream>>>(key, nv, hist, ls);
		k_lv_scan<<<1, 1024, 0, stream>>>(hist, limits, nl, ls);
		k_lv_scatter<2><<<gb, SORT_T, 0, stream>>>(key, nv, hist, sorted);
	} else {
		const uint32_t gb = (nv + 8 * SORT_T - 1) / (8 * SORT_T);
		k_lv_hist<8><<<gb, SORT_T, 0, stream>>>(key, nv, hist, ls);
		k_lv_scan<<<1, 1024, 0, stream>>>(hist, limits, nl, ls);
		k_lv_scatter<8><<<gb, SORT_T, 0, stream>>>(key, nv, hist, sorted);
	}
	const uint32_t nc = nchunks();
	k_lv_chunk_slots<<<fill_grid(64 * nc), 256, 0, stream>>>(sorted, limits, nl, dm->fan_off, dm->closed, nc, cslots);
	k_exclusive_scan<<<1, 1024, 0, stream>>>(cslots, nc, coff);
}

// The four sizes a plan is built from, in one wait instead of a copy each.
__global__ __launch_bounds__(1024) void k_lv_info(const uint32_t *limits, const uint32_t *nl, const uint32_t *coff,
                                                  uint32_t max_nl, LevelInfo *out)
{
	__shared__ uint32_t red[16];
	const uint32_t n = min(*nl, max_nl);
	uint32_t m = 0;
	for (uint32_t q = 1 + threadIdx.x; q < n; q += 1024) m = max(m, limits[q] - limits[q - 1]);
	for (uint32_t o = 32; o > 0; o >>= 1) m = max(m, (uint32_t) __shfl_xor(m, o));
	if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = m;
	__syncthreads();
	if (threadIdx.x != 0) return;
	for (uint32_t q = 1; q < 16; q++) m = max(m, red[q]);
	const uint32_t nr = n ? limits[n - 1] : 0u;
	*out = LevelInfo{ *nl, nr, coff[(nr + 63) / 64], m };
}

int Levels::info(LevelInfo &out)
{
	k_lv_info<<<1, 1024, 0, stream>>>(limits, nl, coff, nv + 2, h_info);
	GP_HIP(hipGetLastError());
	GP_HIP(hipStreamSynchronize(stream));
	out = *h_info;
	if (out.nl < 2 || out.nl > nv + 1 || out.nr > nv)
		return fail(GP_ERR_KERNEL, "levels: bad ring count %u", out.nl);
	return GP_OK;
}

// BFS levels of the sources (NIL where unreached) on the device, copied into
// levels[nv]: the same sets as the host toplesets' levels.
int levels_gpu(Che &m, const uint32_t *src, uint32_t ns, uint32_t *levels)
{
	if (!ns) return fail(GP_ERR_INVALID, "levels: no sources");
	for (uint32_t q = 0; q < ns; q++)
		if (src[q] >= m.nv) return fail(GP_ERR_INVALID, "levels: source %u out of range", src[q]);
	int rc = upload_mesh(m);
	if (rc) return rc;
	PoolStream ps;
	GP_HIP(ps.create());
	const hipStream_t stream = ps.s;
	PoolBuf<uint32_t> srcb(stream);
	if (srcb.alloc(4ull * ns) != hipSuccess) return fail(GP_ERR_NOMEM, "levels: device allocation failed");
	uint32_t *const d_src = srcb.p;
	GP_HIP(hipMemcpy(d_src, src, 4ull * ns, hipMemcpyHostToDevice));
	Levels lv;
	if ((rc = lv.create(m.dev, stream))) return rc;
	lv.clear();
	lv.seed(d_src, 0, ns);
	if ((rc = lv.expand())) return rc;
	GP_HIP(hipMemcpyAsync(levels, lv.level, 4ull * m.nv, hipMemcpyDeviceToHost, stream));
	GP_HIP(hipStreamSynchronize(stream));
	return GP_OK;
}

}  // namespace gp
