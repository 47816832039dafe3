// Batched PTP: many (mesh, source) fields of uneven size in one persistent
// launch behind the reset of its queue: two launches on the stream, for which a
// graph has nothing to save (a launch runs for milliseconds; 1,024 fields 27 ms).
//
// Each 1024-thread workgroup repeatedly takes the next job from an atomic
// queue (jobs sorted by decreasing cost V^1.5, so the grid drains evenly), and
// runs it entirely by itself: the ring build (bfs_bits, its visited bits and
// frontier in LDS, with barriers that wait for LDS only; meshes of more than
// 262,144 vertices take the ordered BFS, bfs_block), then the reference window
// schedule (K/2 band limit, PTP_TOL test, 2*|limits| cap, last-written buffer)
// with one __syncthreads a sweep as the only barrier,
// on the rings of the reference's non-coalesced driver
// (src/cuda/geodesics_ptp.cu:174-299).  Each mesh is stored vertex-major (a
// vertex's slots are contiguous) in Morton order; after its BFS the workgroup
// gathers the field's own ring-ordered tables into its scratch (64 positions
// to a chunk, one lane per vertex, neighbour ids mapped to positions, as the
// coalesced driver renumbers the mesh, src/geodesics_ptp.cpp:15-38), so every
// slot load of a sweep is one contiguous access; the FP64 geometry of flagged
// triangles is read from the mesh's tables through the slot's index there.
// The gather keeps every fan's order, hence the rings and the arithmetic, and
// the output is scattered back.  Every workgroup leaves the loop when the
// queue is exhausted, so the launch always drains.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>
#include <numeric>
#include <vector>

#include "device.hpp"
#include "levels.hpp"
#include "rings_dev.hpp"
#include "sweep_dev.hpp"

namespace gp {

struct BMesh {
	const uint32_t *fan_off, *fan, *link8;
	const uint8_t *closed;
	const uint32_t *coff, *cid;
	const float2 *cgeo;
	const double4 *cgeo64;
	const Edge64 *cx64;
	const uint32_t *perm;   // Morton position -> original vertex id
	float h, inv_h;
	uint32_t nv, ms;        // ms: the longest fan (slots of a field's chunk)
};

struct BJob {
	uint32_t mesh, source, sweeps, pad;
	unsigned long long out, relax;
};

struct BArgs {
	const BMesh *meshes;
	BJob *jobs;
	uint32_t njobs, max_nv;
	uint32_t *queue;
	uint32_t *level, *sorted, *limits, *nlim;
	unsigned long long *key;
	float *dist;
	float *out;
	double tol;
	// Per-workgroup field tables (fslots slots each): ids in positions, FP32
	// geometry, the slot's index in the mesh's tables; inv: vertex -> position.
	uint32_t *fcid, *fmidx, *finv;
	float2 *fgeo;
	size_t fslots;
	uint32_t bit_words;   // LDS words of the BFS's visited bits; 0: bfs_block
};

// Pointers that the kernel reads from memory: without the address space their
// loads are flat ones, which wait for LDS too.
template <typename T>
__device__ __forceinline__ const __attribute__((address_space(1))) T *in_global(const T *p)
{
	return (const __attribute__((address_space(1))) T *) p;
}

// The field's tables as relax_lane reads them.
struct FieldTables {
	const uint32_t *cid;
	const float2 *cgeo;
	GeoRemap64 cgeo64;
	const Edge64 *cx64;
	float h, inv_h;
};

__global__ void k_batch_reset(uint32_t *queue) { *queue = 0; }

// Barrier for data in LDS: stores to memory stay in flight (__syncthreads waits
// for them).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// BFS of one source by the whole workgroup: rings, limits and the vertices'
// positions.  The visited bits and the frontier are in LDS, eight lanes expand a
// vertex from its 32-byte link row, so a level is one round trip to the row and
// two LDS barriers; frontiers past BQ vertices are read back from sorted[].  No
// value depends on the order inside a ring, but it follows the frontier's (the
// waves' counts are scanned), so that the 64 vertices of a chunk lie side by side
// and a sweep's neighbour loads share their lines.  The ordered BFS (bfs_block)
// reads each level's links twice and keys every neighbour with a 64-bit atomic in
// memory: with the gather of the tables 7.9 of the 30.1 ms of 1,024 fields of
// 2k-58k vertices (1,024 threads a field), now 1.9 of 26.7.
constexpr uint32_t BQ = 1024, BFS_UNROLL = 4;   // BQ: whole passes of the loop below
constexpr uint32_t MAX_BIT_WORDS = 8192;        // 32 KB: meshes to 262,144 vertices

template <uint32_t NT>
__device__ __forceinline__ uint32_t bfs_bits(const BMesh &M, uint32_t src, uint32_t *bits, uint32_t (*s_q)[BQ],
                                             uint32_t *s_cnt, uint32_t *s_end, uint32_t *sorted, uint32_t *inv,
                                             uint32_t *limits)
{
	constexpr uint32_t GROUPS = NT / LINK_ROW, NW = NT / 64;
	static_assert(BQ % (GROUPS * BFS_UNROLL) == 0, "a pass reads the frontier from one place");
	static_assert(NW * BFS_UNROLL <= 64, "one lane a count");
	const uint32_t tid = threadIdx.x, lane = tid & 63u, slot = tid % LINK_ROW, group = tid / LINK_ROW;
	const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const auto *link8 = in_global(M.link8);
	for (uint32_t w = tid; w < (M.nv + 31) / 32; w += NT) bits[w] = 0;
	__syncthreads();
	if (tid == 0) {
		bits[src >> 5] = 1u << (src & 31u);
		s_q[0][0] = src;
		sorted[0] = src;
		inv[src] = 0;
		limits[0] = 0;
		limits[1] = 1;
	}
	__syncthreads();
	uint32_t fb = 0, fe = 1, nl = 2;   // the frontier is sorted[fb, fe)
	for (uint32_t cur = 0;; cur ^= 1u) {
		const uint32_t n = fe - fb;
		uint32_t p = fe;               // the next ring is sorted[fe, p)
		auto claim = [&](uint32_t u) -> bool {
			const uint32_t bit = 1u << (u & 31u);
			return u != GP_NIL && !(atomicOr(&bits[u >> 5], bit) & bit);
		};
		auto append = [&](uint32_t u, uint32_t at) {
			if (at - fe < BQ) s_q[cur ^ 1u][at - fe] = u;
			sorted[at] = u;
			inv[u] = at;
		};
		for (uint32_t c0 = 0; c0 < n; c0 += GROUPS * BFS_UNROLL) {
			uint32_t id[BFS_UNROLL];
			unsigned long long got[BFS_UNROLL];
			uint32_t more = 0;         // bit r: the link of pass r goes on (lane of entry 7)
#pragma unroll
			for (uint32_t r = 0; r < BFS_UNROLL; r++) {
				const uint32_t c = c0 + r * GROUPS + group;
				id[r] = GP_NIL;
				if (c < n) {
					uint32_t v;
					if (c0 < BQ) v = s_q[cur][c];
					else v = sorted[fb + c];
					id[r] = link8[(size_t) v * LINK_ROW + slot];
				}
			}
#pragma unroll
			for (uint32_t r = 0; r < BFS_UNROLL; r++) {
				if (id[r] != GP_NIL && (id[r] & LONG_LINK)) {
					id[r] &= ~LONG_LINK;
					more |= 1u << r;
				}
				got[r] = __ballot(claim(id[r]));
				if (lane == 0) s_cnt[r * NW + wave] = (uint32_t) __popcll(got[r]);
				if (more >> r & 1u) s_cnt[r * NW + wave] = (uint32_t) __popcll(got[r]) | LONG_LINK;
			}
			lds_barrier();
			// Every wave scans the pass's counts, one a lane.
			uint32_t x = lane < NW * BFS_UNROLL ? s_cnt[lane] : 0u;
			const bool any_more = __ballot((x & LONG_LINK) != 0u) != 0;
			x &= ~LONG_LINK;
			uint32_t inc = x;
			for (uint32_t o = 1; o < 64; o <<= 1) {
				const uint32_t y = __shfl_up(inc, o);
				if (lane >= o) inc += y;
			}
#pragma unroll
			for (uint32_t r = 0; r < BFS_UNROLL; r++) {
				const uint32_t at = p + __shfl(inc - x, (int) (r * NW + wave));
				if (got[r] >> lane & 1ull) append(id[r], at + (uint32_t) __popcll(got[r] & ((1ull << lane) - 1)));
			}
			p += __shfl(inc, 63);
			if (any_more) {
				// The entries past eight, from the fan table, as they come.
				if (tid == 0) *s_end = p;
				lds_barrier();
				for (uint32_t r = 0; r < BFS_UNROLL; r++) {
					uint32_t k = 0, e = 0;
					if (__shfl((int) more, (int) (lane | (LINK_ROW - 1))) >> r & 1) {
						const uint32_t c = c0 + r * GROUPS + group;
						uint32_t v;
						if (c0 < BQ) v = s_q[cur][c];
						else v = sorted[fb + c];
						k = M.fan_off[v] + LINK_ROW + slot;
						e = M.fan_off[v + 1] - (M.closed[v] ? 1u : 0u);
					}
					for (; __ballot(k < e); k += LINK_ROW) {
						const uint32_t u = k < e ? M.fan[k] & ID_MASK : GP_NIL;
						const bool take = claim(u);
						const unsigned long long m = __ballot(take);
						if (!m) continue;
						const int first = __builtin_ctzll(m);
						uint32_t at = 0;
						if (lane == (uint32_t) first) at = atomicAdd(s_end, (uint32_t) __popcll(m));
						at = __shfl(at, first) + (uint32_t) __popcll(m & ((1ull << lane) - 1));
						if (take) append(u, at);
					}
				}
				lds_barrier();
				p = __builtin_amdgcn_readfirstlane(*s_end);
			}
			lds_barrier();
		}
		if (p == fe) break;
		if (p - fe > BQ) __syncthreads();   // sorted[] is read back
		fb = fe;
		fe = p;
		if (tid == 0) limits[nl] = fe;
		nl++;
	}
	__syncthreads();
	return nl;
}

// NT threads per field (a multiple of 64, at most 1024).
//
// The sweeps, 25 of 27 ms, run 16 waves a CU (128 registers a lane), each taking
// one chunk after the other: rows from memory (43 GB in all; 79 % of the requests
// miss L2, as 32 fields share one), neighbours' values, ~510 vector instructions
// (the units are busy 46 % of the time), a chain that four waves a SIMD cover in
// part.  Two fields a CU of 512 threads take longer (38 ms) as they need twice
// the cache, and asking for a chunk's rows one chunk ahead does too (29 ms).
//
// Four waves a SIMD is the most that is asked for.  A build of this kernel forced to
// eight (64 registers, 304 bytes of spills a lane) ended in a GPU memory fault with
// 1,024 threads a field; every index is bounded alike in both builds and no cause was
// found, so it was not run again.
constexpr uint32_t BL = 1024;   // ring limits kept in LDS

template <uint32_t NT, uint32_t MS>
__global__ __launch_bounds__(NT, 4) void k_batch(BArgs a)
{
	extern __shared__ uint32_t s_bits[];
	__shared__ uint32_t s_job, s_bad[3], s_cnt[64], s_end, s_q[2][BQ], s_lim[BL];
	const uint32_t tid = threadIdx.x, nt = NT, wg = blockIdx.x;
	const size_t mv = a.max_nv;
	uint32_t *sorted = a.sorted + wg * mv;
	uint32_t *limits = a.limits + wg * (mv + 2);
	float *d0 = a.dist + 2 * wg * mv, *d1 = d0 + mv;
	uint32_t *fcid = a.fcid + wg * a.fslots, *fmidx = a.fmidx + wg * a.fslots, *finv = a.finv + wg * mv;
	float2 *fgeo = a.fgeo + wg * a.fslots;
	// Values every thread of the workgroup holds alike (the wave index, the
	// job, the ring-test count) are taken from the first lane, so the
	// compiler keeps them and what follows from them (the mesh, the window,
	// the chunk index, the slot count) in scalar registers.
	const uint32_t lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwave = NT >> 6;
	for (;;) {
		if (tid == 0) s_job = atomicAdd(a.queue, 1u);
		__syncthreads();
		const uint32_t job = __builtin_amdgcn_readfirstlane(s_job);
		__syncthreads();
		if (job >= a.njobs) break;
		const BMesh M = a.meshes[a.jobs[job].mesh];
		const uint32_t nv = M.nv;
		for (uint32_t v = tid; v < nv; v += nt) {
			finv[v] = GP_NIL;
			d0[v] = INFINITY; d1[v] = INFINITY;
		}
		__syncthreads();
		uint32_t nl;
		if (a.bit_words) {
			nl = bfs_bits<NT>(M, a.jobs[job].source, s_bits, s_q, s_cnt, &s_end, sorted, finv, limits);
		} else {
			uint32_t *level = a.level + wg * mv;
			unsigned long long *key = a.key + wg * mv;
			for (uint32_t v = tid; v < nv; v += nt) { level[v] = GP_NIL; key[v] = ~0ull; sorted[v] = GP_NIL; }
			__syncthreads();
			const BfsJob bj{ &a.jobs[job].source, 1u, level, key, sorted, limits, a.nlim + wg };
			bfs_block(M.fan_off, M.fan, M.closed, bj);
			nl = __builtin_amdgcn_readfirstlane(__hip_atomic_load(a.nlim + wg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
			for (uint32_t q = tid; q < limits[nl - 1]; q += nt) finv[sorted[q]] = q;
		}
		for (uint32_t q = tid; q < min(nl, BL); q += nt) s_lim[q] = limits[q];
		auto lim = [&](uint32_t q) { return __builtin_amdgcn_readfirstlane(q < BL ? s_lim[q] : limits[q]); };
		__syncthreads();
		// The field's ring-ordered tables: position p holds vertex sorted[p]
		// (the source is position 0).
		const uint32_t nr = lim(nl - 1);
		const auto *mcoff = in_global(M.coff), *mcid = in_global(M.cid);
		const auto *mgeo = in_global(M.cgeo);
		const auto *perm = in_global(M.perm);
		const uint32_t S = M.ms, npos = (nr + 63u) & ~63u;
		for (uint32_t q = tid; q < npos; q += nt) {
			const size_t fb = (size_t) (q >> 6) * S * 64 + (q & 63u);
			uint32_t mb = 0, n = 0;
			if (q < nr) {
				const uint32_t v = sorted[q];
				mb = mcoff[v];
				n = mcoff[v + 1] - mb;
			}
			// Eight slots at a time: their ids, then the positions and the
			// geometry they lead to, in flight together.
			for (uint32_t k0 = 0; k0 < S; k0 += 8) {
				uint32_t id[8], at[8], p[8];
				float2 g[8];
#pragma unroll
				for (uint32_t k = 0; k < 8; k++) {
					at[k] = k0 + k < n ? mb + k0 + k : 0u;
					id[k] = mcid[at[k]];
					if (k0 + k >= n) id[k] = 0;
				}
#pragma unroll
				for (uint32_t k = 0; k < 8; k++) { p[k] = finv[id[k] & SLOT_ID_MASK]; g[k] = float2{ mgeo[at[k]].x, mgeo[at[k]].y }; }
#pragma unroll
				for (uint32_t k = 0; k < 8; k++)
					if (k0 + k < S) {
						const bool has = k0 + k < n;
						const size_t to = fb + 64 * (size_t) (k0 + k);
						fcid[to] = has ? p[k] | (id[k] & ~SLOT_ID_MASK) : q | SLOT_EMPTY;
						fgeo[to] = has ? g[k] : make_float2(0.f, 0.f);
						fmidx[to] = has ? at[k] : 0u;
					}
			}
		}
		if (tid == 0 && nr) { d0[0] = 0.f; d1[0] = 0.f; }
		if (tid < 3) s_bad[tid] = 0;
		__syncthreads();
		const FieldTables F{ fcid, fgeo, GeoRemap64{ M.cgeo64, fmidx }, nullptr, M.h, M.inv_h };
		uint32_t i = 1, j = 2, d = 0, iter = 0, turn = 0;
		unsigned long long relax = 0;
		const uint32_t max_iter = nl << 1;
		bool done = nl < 3;
		// One barrier a sweep: the ring test counts into one of three words in
		// turn, the word after next cleared meanwhile.
		while (!done) {
			const uint32_t ii = i < (j >> 1) ? (j >> 1) : i;
			const uint32_t start = lim(ii), end = lim(j), cend = lim(ii + 1);
			const float *od = d ? d1 : d0;
			float *nd = d ? d0 : d1;
			uint32_t bad = 0;
			for (uint32_t c = (start >> 6) + wave; c < ((end + 63u) >> 6); c += nwave) {
				const uint32_t pos = (c << 6) + lane;
				bool lbad = false;
				if (pos >= start && pos < end) {
					const float old = od[pos];
					const float best = relax_lane<false, 64, false, false, MS>(F, (size_t) c * S * 64 + lane, S, od, old);
					nd[pos] = best;
					if (pos < cend) lbad = !(fabs((double) best - (double) old) / (double) old < a.tol);
				}
				bad += (uint32_t) __popcll(__ballot(lbad));
			}
			if (lane == 0 && bad) atomicAdd(&s_bad[turn], bad);
			__syncthreads();
			const uint32_t nbad = __builtin_amdgcn_readfirstlane(s_bad[turn]);
			turn = turn == 2 ? 0 : turn + 1;
			if (tid == 0) s_bad[turn == 2 ? 0 : turn + 1] = 0;
			relax += end - start;
			i = ii + (nbad == 0 ? 1u : 0u);
			if (j < nl - 1) j++;
			d ^= 1u;
			iter++;
			done = !(i < j) || !(iter < max_iter);
		}
		const float *res = d ? d1 : d0;            // the buffer the last sweep wrote
		float *out = a.out + a.jobs[job].out;
		for (uint32_t v = tid; v < nv; v += nt) out[perm[v]] = finv[v] != GP_NIL ? res[finv[v]] : INFINITY;
		if (tid == 0) { a.jobs[job].sweeps = iter; a.jobs[job].relax = relax; }
		__syncthreads();
	}
}

}  // namespace gp

// ---------------------------------------------------------------------------

struct gp_batch {
	struct MeshTables {
		std::unique_ptr<gp::Che> ren;   // Morton-numbered copy of the mesh
		std::vector<uint32_t> inv;      // original -> Morton numbering
		uint32_t *coff = nullptr, *cid = nullptr, *perm = nullptr;
		float2 *cgeo = nullptr;
		double4 *cgeo64 = nullptr;
	};
	std::vector<MeshTables> tabs;
	std::vector<unsigned long long> out_off;   // user job -> offset of its field
	std::vector<uint32_t> job_nv;              // user job -> vertices
	std::vector<uint32_t> slot_of;             // user job -> queue slot
	// Read back under the lock: the fields of the last run around the one asked
	// for, as the caller takes them, and the jobs' sweep counts.
	std::mutex mu;
	double *h_win = nullptr;
	unsigned long long win_at = 0, next_at = 0;   // next_at: behind the field read last
	uint32_t win_n = 0;
	std::vector<gp::BJob> jobs;                // of the last run (empty: not read yet)
	gp::BMesh *d_meshes = nullptr;
	gp::BJob *d_jobs = nullptr;
	uint32_t *d_queue = nullptr;
	float *d_out = nullptr;
	// Per-workgroup scratch, sized for the current configuration.
	uint32_t *d_level = nullptr, *d_sorted = nullptr, *d_limits = nullptr, *d_nlim = nullptr;
	unsigned long long *d_key = nullptr;
	float *d_dist = nullptr;
	uint32_t *d_fcid = nullptr, *d_fmidx = nullptr, *d_finv = nullptr;
	float2 *d_fgeo = nullptr;
	uint32_t njobs = 0, max_nv = 0, max_slots = 0, grid = 0, block = 0;
	unsigned long long total_out = 0;
	double tol = GP_PTP_TOL;
	hipStream_t stream = nullptr;
	gp::BArgs args{};
	const void *fn = nullptr;
	hipEvent_t e0 = nullptr, e1 = nullptr;

	void free_scratch()
	{
		for (void *p : { (void *) d_level, (void *) d_sorted, (void *) d_limits, (void *) d_nlim, (void *) d_key,
		                 (void *) d_dist, (void *) d_fcid, (void *) d_fmidx, (void *) d_finv, (void *) d_fgeo })
			(void) hipFree(p);
		d_level = d_sorted = d_limits = d_nlim = nullptr;
		d_key = nullptr;
		d_dist = nullptr;
		d_fcid = d_fmidx = d_finv = nullptr;
		d_fgeo = nullptr;
	}
	~gp_batch()
	{
		free_scratch();
		for (auto &t : tabs)
			for (void *p : { (void *) t.coff, (void *) t.cid, (void *) t.cgeo, (void *) t.cgeo64, (void *) t.perm })
				(void) hipFree(p);
		for (void *p : { (void *) d_meshes, (void *) d_jobs, (void *) d_queue, (void *) d_out }) (void) hipFree(p);
		gp::pinned_free(h_win);
		if (e0) (void) hipEventDestroy(e0);
		if (e1) (void) hipEventDestroy(e1);
		if (stream) (void) hipStreamDestroy(stream);
	}
};

namespace gp {

template <typename V>
static int up(V *&dst, const V *src, size_t n)
{
	if (device_malloc(&dst, sizeof(V) * std::max<size_t>(n, 1)) != hipSuccess) return fail(GP_ERR_NOMEM, "batch: allocation failed");
	if (n) GP_HIP(hipMemcpy(dst, src, sizeof(V) * n, hipMemcpyHostToDevice));
	return GP_OK;
}

// Fields whose fans all fit 8 slots run the 8-slot register path.
template <uint32_t NT>
static int launch_shape(uint32_t njobs, bool ms8, uint32_t lds, uint32_t &grid, const void *&fn)
{
	int dev = 0, ncu = 0, occ = 0;
	GP_HIP(hipGetDevice(&dev));
	GP_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev));
	fn = ms8 ? (const void *) k_batch<NT, 8> : (const void *) k_batch<NT, MAXS>;
	GP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, fn, NT, lds));
	grid = std::max<uint32_t>(1, std::min<uint32_t>(njobs, (uint32_t) ncu * (uint32_t) std::max(1, occ)));
	return GP_OK;
}

// Sizes the per-workgroup scratch for `block` threads per field.
static int batch_configure(gp_batch *b, uint32_t block)
{
	b->free_scratch();
	uint32_t grid = 0;
	const void *fn = nullptr;
	int rc;
	const uint32_t words = (b->max_nv + 31) / 32, bit_words = words <= MAX_BIT_WORDS ? words : 0;
	switch (block) {
	case 256: rc = launch_shape<256>(b->njobs, b->max_slots <= 8, 4 * bit_words, grid, fn); break;
	case 512: rc = launch_shape<512>(b->njobs, b->max_slots <= 8, 4 * bit_words, grid, fn); break;
	case 1024: rc = launch_shape<1024>(b->njobs, b->max_slots <= 8, 4 * bit_words, grid, fn); break;
	default: return fail(GP_ERR_INVALID, "batch: block must be 256, 512 or 1024 (got %u)", block);
	}
	if (rc) return rc;
	const size_t mv = b->max_nv;
	// Field tables: the largest field's chunks at the longest fan's width.
	const size_t fslots = ((mv + 63) / 64) * 64 * (size_t) b->max_slots;
	const size_t bfs_mv = bit_words ? 0 : mv;   // the ordered BFS's levels and keys
	const size_t per_wg = 4 * mv * 2 + 4 * (mv + 2) + 12 * bfs_mv + 8 * mv + fslots * (4 + 4 + sizeof(float2));
	// At most 32 GiB of scratch: a wider grid than that would take no more
	// fields at once than the workgroups that fit.
	const size_t cap = std::max<size_t>(1, (32ull << 30) / std::max<size_t>(per_wg, 1));
	grid = (uint32_t) std::min<size_t>(grid, cap);
	const size_t g = grid;
	if (device_malloc(&b->d_level, std::max<size_t>(4, 4 * bfs_mv * g)) != hipSuccess || device_malloc(&b->d_sorted, 4 * mv * g) != hipSuccess ||
	    device_malloc(&b->d_limits, 4 * (mv + 2) * g) != hipSuccess || device_malloc(&b->d_nlim, 4 * g) != hipSuccess ||
	    device_malloc(&b->d_key, std::max<size_t>(8, 8 * bfs_mv * g)) != hipSuccess || device_malloc(&b->d_dist, 8 * mv * g) != hipSuccess ||
	    device_malloc(&b->d_finv, 4 * mv * g) != hipSuccess || device_malloc(&b->d_fcid, 4 * fslots * g) != hipSuccess ||
	    device_malloc(&b->d_fmidx, 4 * fslots * g) != hipSuccess || device_malloc(&b->d_fgeo, sizeof(float2) * fslots * g) != hipSuccess) {
		b->free_scratch();
		return fail(GP_ERR_NOMEM, "batch: scratch allocation failed (%u workgroups x %u vertices)", grid, b->max_nv);
	}
	BArgs a{ b->d_meshes, b->d_jobs, b->njobs, b->max_nv, b->d_queue, b->d_level, b->d_sorted, b->d_limits, b->d_nlim,
	         b->d_key, b->d_dist, b->d_out, b->tol, b->d_fcid, b->d_fmidx, b->d_finv, b->d_fgeo, fslots, bit_words };
	b->args = a;
	b->fn = fn;
	b->grid = grid;
	b->block = block;
	return GP_OK;
}

static int batch_launch(gp_batch *b, float *ms)
{
	std::lock_guard<std::mutex> lock(b->mu);
	b->win_n = 0;
	b->next_at = 0;
	b->jobs.clear();
	GP_HIP(hipEventRecord(b->e0, b->stream));
	void *kargs[] = { &b->args };
	k_batch_reset<<<1, 1, 0, b->stream>>>(b->d_queue);
	GP_HIP(hipLaunchKernel(b->fn, dim3(b->grid), dim3(b->block), kargs, 4 * b->args.bit_words, b->stream));
	GP_HIP(hipEventRecord(b->e1, b->stream));
	GP_HIP(hipStreamSynchronize(b->stream));
	GP_HIP(hipEventElapsedTime(ms, b->e0, b->e1));
	return GP_OK;
}

int batch_create(Che *const *meshes, uint32_t nmeshes, const uint32_t *job_mesh, const uint32_t *job_source,
                 uint32_t njobs, double tol, uint32_t block, gp_batch **out)
{
	*out = nullptr;
	if (!meshes || !nmeshes || !job_mesh || !job_source || !njobs) return fail(GP_ERR_INVALID, "batch: empty input");
	if (!(tol > 0)) return fail(GP_ERR_INVALID, "batch: tol must be positive");
	for (uint32_t k = 0; k < nmeshes; k++)
		if (!meshes[k]) return fail(GP_ERR_INVALID, "batch: mesh %u is null", k);
	for (uint32_t q = 0; q < njobs; q++) {
		if (job_mesh[q] >= nmeshes) return fail(GP_ERR_INVALID, "batch: job %u mesh out of range", q);
		if (job_source[q] >= meshes[job_mesh[q]]->nv) return fail(GP_ERR_INVALID, "batch: job %u source out of range", q);
	}
	auto b = std::make_unique<gp_batch>();
	b->njobs = njobs;
	b->tol = tol;
	std::vector<BMesh> bm(nmeshes);
	b->tabs.resize(nmeshes);
	for (uint32_t k = 0; k < nmeshes; k++) {
		const Che &m0 = *meshes[k];
		if (m0.nv >= SLOT_WRAP) return fail(GP_ERR_CAPACITY, "batch: mesh %u has too many vertices", k);
		for (uint32_t v = 0; v < m0.nv; v++)
			if (m0.fan_off[v + 1] - m0.fan_off[v] > MAX_LINK)
				return fail(GP_ERR_CAPACITY, "batch: mesh %u vertex %u: link over %u", k, v, MAX_LINK);
		auto &t = b->tabs[k];
		std::vector<uint32_t> order;
		morton_order(m0, order);
		t.ren = std::make_unique<Che>();
		int rc = coalesce(m0, order.data(), m0.nv, *t.ren, t.inv);
		if (rc) return rc;
		Che &m = *t.ren;
		m.mean_edge = m0.mean_edge;      // the same h as the mesh itself
		if ((rc = upload_mesh(m)) || (rc = link_rows(m.dev))) return rc;
		Layout L;
		if ((rc = build_layout(m, nullptr, m.nv, false, L, 0, 1, 0, true))) return rc;
		if ((rc = up(t.coff, L.coff.data(), L.coff.size())) || (rc = up(t.cid, L.cid.data(), L.cid.size())) ||
		    (rc = up(t.cgeo, reinterpret_cast<const float2 *>(L.cgeo.data()), L.cgeo.size())) ||
		    (rc = up(t.cgeo64, reinterpret_cast<const double4 *>(L.cgeo64.data()), L.cgeo64.size())) ||
		    (rc = up(t.perm, order.data(), order.size())))
			return rc;
		bm[k] = BMesh{ m.dev->fan_off, m.dev->fan, m.dev->link8, m.dev->closed, t.coff, t.cid, t.cgeo, t.cgeo64, nullptr, t.perm,
		               m.dev->h, m.dev->inv_h, m.nv, L.max_slots };
		b->max_nv = std::max(b->max_nv, m.nv);
		b->max_slots = std::max(b->max_slots, L.max_slots);
	}
	// Queue order: longest fields first (work of a field grows ~ V^1.5), so
	// the last jobs taken are the short ones and the grid drains evenly.
	std::vector<uint32_t> order(njobs);
	std::iota(order.begin(), order.end(), 0u);
	std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) {
		return meshes[job_mesh[x]]->nv > meshes[job_mesh[y]]->nv;
	});
	b->slot_of.resize(njobs);
	b->out_off.resize(njobs);
	b->job_nv.resize(njobs);
	std::vector<BJob> jobs(njobs);
	unsigned long long off = 0;
	for (uint32_t q = 0; q < njobs; q++) {   // fields in the caller's order
		b->out_off[q] = off;
		b->job_nv[q] = meshes[job_mesh[q]]->nv;
		off += b->job_nv[q];
	}
	for (uint32_t s = 0; s < njobs; s++) {
		const uint32_t q = order[s];
		b->slot_of[q] = s;
		jobs[s] = BJob{ job_mesh[q], b->tabs[job_mesh[q]].inv[job_source[q]], 0, 0, b->out_off[q], 0 };
	}
	b->total_out = off;
	int rc;
	if ((rc = up(b->d_meshes, bm.data(), bm.size())) || (rc = up(b->d_jobs, jobs.data(), jobs.size()))) return rc;
	if (device_malloc(&b->d_queue, 4) != hipSuccess || device_malloc(&b->d_out, 4 * std::max<size_t>(off, 1)) != hipSuccess)
		return fail(GP_ERR_NOMEM, "batch: output allocation failed (%llu values)", off);
	GP_HIP(hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking));
	GP_HIP(hipEventCreate(&b->e0));
	GP_HIP(hipEventCreate(&b->e1));
	if (block) {
		if ((rc = batch_configure(b.get(), block))) return rc;
	} else {
		// Autotune threads per field: one timed run of the whole batch per
		// candidate after one warm-up run, keep the fastest.
		float best = INFINITY;
		uint32_t best_block = 1024;
		for (uint32_t cand : { 256u, 512u, 1024u }) {
			float ms = 0;
			if ((rc = batch_configure(b.get(), cand)) || (rc = batch_launch(b.get(), &ms)) ||
			    (rc = batch_launch(b.get(), &ms)))
				return rc;
			if (ms < best) { best = ms; best_block = cand; }
		}
		if (b->block != best_block && (rc = batch_configure(b.get(), best_block))) return rc;
	}
	*out = b.release();
	return GP_OK;
}

// The jobs' counts of the last run (lock held).
static int batch_jobs(gp_batch *b)
{
	if (!b->jobs.empty()) return GP_OK;
	std::vector<BJob> jobs(b->njobs);
	GP_HIP(hipMemcpy(jobs.data(), b->d_jobs, sizeof(BJob) * b->njobs, hipMemcpyDeviceToHost));
	b->jobs.swap(jobs);
	return GP_OK;
}

int batch_run(gp_batch *b, gp_batch_stats *st)
{
	if (!b) return fail(GP_ERR_INVALID, "batch is null");
	float ms = 0;
	int rc = batch_launch(b, &ms);
	if (rc) return rc;
	if (st) {
		std::lock_guard<std::mutex> lock(b->mu);
		if ((rc = batch_jobs(b))) return rc;
		unsigned long long s = 0, r = 0;
		for (auto &j : b->jobs) { s += j.sweeps; r += j.relax; }
		st->sweeps = s;
		st->relaxations = r;
		st->vertex_fields = b->total_out;
		st->block = b->block;
		st->grid = b->grid;
		st->kernel_ms = ms;
	}
	return GP_OK;
}

__global__ void k_widen(const float *in, uint32_t n, double *out)
{
	for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) out[q] = in[q];
}

// Fields are read back one by one, in order as a rule: the device widens a field
// straight into pinned memory, the WIN values from there on where the last one
// read lies just before it, and the calls that follow copy out of there (two hipMemcpy of pageable memory a field
// before: 59 us a field of 17k doubles, 28 now, most of it the caller's fresh pages).
constexpr uint32_t WIN = 1u << 19;

int batch_result(gp_batch *b, uint32_t job, double *dist, uint32_t cap, uint32_t *sweeps)
{
	if (!b || !dist) return fail(GP_ERR_INVALID, "null argument");
	if (job >= b->njobs) return fail(GP_ERR_INVALID, "batch: job %u out of range", job);
	const uint32_t n = b->job_nv[job];
	if (cap < n) return fail(GP_ERR_CAPACITY, "batch: result of job %u needs %u entries", job, n);
	std::lock_guard<std::mutex> lock(b->mu);
	const unsigned long long off = b->out_off[job];
	for (uint32_t at = 0; at < n;) {
		const unsigned long long from = off + at;
		if (from < b->win_at || from >= b->win_at + b->win_n) {
			if (!b->h_win && pinned_malloc(&b->h_win, sizeof(double) * std::min<unsigned long long>(WIN, b->total_out)) != hipSuccess) {
				// None to be had: this field by a pageable copy.
				std::vector<float> field(n);
				GP_HIP(hipMemcpy(field.data(), b->d_out + off, sizeof(float) * n, hipMemcpyDeviceToHost));
				for (uint32_t v = 0; v < n; v++) dist[v] = field[v];
				break;
			}
			const uint32_t m = (uint32_t) std::min<unsigned long long>(WIN, from == b->next_at ? b->total_out - from : n - at);
			b->win_n = 0;
			k_widen<<<std::min<uint32_t>(256, (m + 255) / 256), 256, 0, b->stream>>>(b->d_out + from, m, b->h_win);
			GP_HIP(hipGetLastError());
			GP_HIP(hipStreamSynchronize(b->stream));
			b->win_at = from;
			b->win_n = m;
		}
		const uint32_t skip = (uint32_t) (from - b->win_at), m = std::min(n - at, b->win_n - skip);
		copy_out(dist + at, b->h_win + skip, sizeof(double) * m);
		at += m;
		b->next_at = off + at;
	}
	if (sweeps) {
		if (int rc = batch_jobs(b)) return rc;
		*sweeps = b->jobs[b->slot_of[job]].sweeps;
	}
	return GP_OK;
}

}  // namespace gp

extern "C" void gp_batch_destroy(gp_batch *b) { delete b; }
