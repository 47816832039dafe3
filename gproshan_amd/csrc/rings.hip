// Toplesets (BFS rings) on the GPU, bit-identical to che::compute_toplesets
// (src/che.cpp:546-593).
//
// Ring membership is the hop distance: the levels and the rings as sets come
// from levels.hip.  The order inside a ring is the reference's discovery order:
// the serial BFS appends u when it first meets it while scanning the ring
// before in sorted order and, within a vertex, in link order.  So u takes the
// smallest (rank of the discovering vertex in its ring, slot in its link), and
// the new ring is in the order of those keys.  The ranks of a ring need those
// of the ring before, so one workgroup walks the rings (k_ring_order); what
// does not depend on ranks -- each vertex's link entries in the next ring -- is
// laid out by all workgroups beforehand (k_ring_children).
//
// Meshes with a link over ORDER_MAX_LINK take the one-workgroup BFS
// (k_rings_bfs): a newly reached u takes the smallest key (position of the
// discovering vertex in sorted) * 1024 + (slot in its link) by a 64-bit
// atomicMin, and the owner (pos, slot) of each u emits it, with a workgroup
// prefix sum over the frontier in (pos, slot) order.
#include "device.hpp"
#include "levels.hpp"
#include "rings_dev.hpp"

#include <algorithm>
#include <memory>
#include <type_traits>
#include <vector>

namespace gp {

// Children of each position q of the rings as sets: the link entries of
// sorted[q] one level down, as (index in the next ring) * 32 + slot, CHILD_ROWS
// to a position (NIL past them); CHILD_MORE in the last when there are more (the
// walk then reads the link itself).
constexpr uint32_t CHILD_ROWS = 8, CHILD_MORE = GP_NIL - 1u;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

struct OrderArgs {
	const uint32_t *sorted, *limits, *level, *inv, *fan_off, *fan;
	const uint8_t *closed;
	uint32_t nl, nr;
	uint32_t *child;         // [nr][CHILD_ROWS]
	const uint32_t *rank0;   // ring 0: index among the sources
	uint32_t *out;
};

__global__ void k_ring_children(OrderArgs a)
{
	for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < a.nr; q += gridDim.x * blockDim.x) {
		const uint32_t v = a.sorted[q], l1 = a.level[v] + 1;
		const uint32_t s = a.fan_off[v], c = a.fan_off[v + 1] - s;
		const uint32_t n = (c && a.closed[v]) ? c - 1 : c;
		const uint32_t first = l1 < a.nl - 1 ? a.limits[l1] : 0u;
		uint32_t e[CHILD_ROWS], m = 0;
#pragma unroll
		for (uint32_t k = 0; k < CHILD_ROWS; k++) e[k] = GP_NIL;
		for (uint32_t k = 0; k < n; k++) {
			const uint32_t u = a.fan[s + k];
			if (a.level[u] != l1) continue;
			const uint32_t x = ((a.inv[u] - first) << 5) | k;
#pragma unroll
			for (uint32_t j = 0; j < CHILD_ROWS; j++)
				if (m == j) e[j] = x;
			m++;
		}
		if (m > CHILD_ROWS) e[CHILD_ROWS - 1] = CHILD_MORE;
		uint4 *row = (uint4 *) (a.child + (size_t) q * CHILD_ROWS);
		row[0] = make_uint4(e[0], e[1], e[2], e[3]);
		row[1] = make_uint4(e[4], e[5], e[6], e[7]);
	}
}

__global__ void k_ring_rank0(const uint32_t *src, uint32_t ns, const uint32_t *inv, uint32_t *rank0)
{
	for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < ns; q += gridDim.x * blockDim.x) rank0[inv[src[q]]] = q;
}

__global__ void k_ring_inv(const uint32_t *sorted, uint32_t nr, uint32_t *inv)
{
	for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < nr; q += gridDim.x * blockDim.x) inv[sorted[q]] = q;
}

// Inclusive sum over the wave's lanes (row shifts, then the rows' totals).
__device__ __forceinline__ uint32_t wave_scan(uint32_t x)
{
	x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x111, 0xF, 0xF, true);    // row_shr:1
	x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x112, 0xF, 0xF, true);    // row_shr:2
	x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x114, 0xF, 0xF, true);    // row_shr:4
	x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x118, 0xF, 0xF, true);    // row_shr:8
	x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x142, 0xA, 0xF, false);   // row_bcast:15 into rows 1, 3
	x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x143, 0xC, 0xF, false);   // row_bcast:31 into rows 2, 3
	return x;
}

// Barrier of the walk.  LDS arrays: only the LDS accesses are waited for, so
// the next ring's loads and this ring's stores stay in flight across it (nobody
// in the workgroup reads what another thread stored to memory).
template <bool LDS>
__device__ __forceinline__ void order_barrier()
{
	if constexpr (LDS) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
	else __syncthreads();
}

// Walks the rings: the ranks of ring r give every vertex of ring r + 1 its
// smallest (parent rank, slot) (an atomic minimum by the parents' children),
// the slots taken of each parent as a bit mask, a prefix sum of the masks' bit
// counts over the parents in rank order, and so the ranks of ring r + 1, its
// vertices written in that order.  One workgroup, as every ring waits for the
// one before; the keys, masks, sums and ranks of rings up to R vertices stay in
// LDS, and the next ring's children (its first 2 NT vertices) are on their way
// before this ring is done, so a ring costs a few LDS passes: 2.2 us a ring
// of the 1M-vertex mesh (1,010 rings, 2.2 ms; the one-workgroup BFS 40 ms, the
// host 30 ms), 1.7 us with 256 threads on rings of 200.  R == 0: rings of any width, the arrays in global memory.
template <uint32_t NT, uint32_t R>
__global__ __launch_bounds__(NT) void k_ring_order(OrderArgs a, uint32_t *work, uint32_t wide)
{
	constexpr bool LDS = R > 0;
	constexpr uint32_t RA = LDS ? R : 1, AHEAD = 2;
	using Rank = typename std::conditional<LDS, uint16_t, uint32_t>::type;
	__shared__ uint32_t s_key[RA], s_mask[RA], part[2][NT / 64];
	__shared__ Rank s_rank[RA], s_base[RA];
	uint32_t *key, *mask;
	Rank *rank, *base;
	if constexpr (LDS) {
		key = s_key; mask = s_mask; rank = s_rank; base = s_base;
	} else {
		key = work; mask = work + wide; rank = work + 2 * (size_t) wide; base = work + 3 * (size_t) wide;
	}
	// Global arrays are read and written past the vector cache, as other lanes'
	// atomics change them.
	auto ld = [](const auto *p) {
		if constexpr (LDS) return *p;
		else return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	};
	auto st = [](auto *p, uint32_t x) {
		if constexpr (LDS) *p = (typename std::remove_reference<decltype(*p)>::type) x;
		else __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	};
	const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
	uint32_t b0 = 0, b1 = a.limits[1], b2 = a.nl > 2 ? a.limits[2] : b1;
	for (uint32_t i = tid; i < b1; i += NT) {
		const uint32_t r = a.rank0[i];
		st(&rank[i], r);
		a.out[r] = a.sorted[i];
	}
	for (uint32_t i = tid; i < b1; i += NT) st(&mask[i], 0u);
	for (uint32_t i = tid; i < b2 - b1; i += NT) st(&key[i], GP_NIL);
	// Children and vertices of a ring's first AHEAD * NT positions, and the end
	// of the ring after it
	struct Ahead {
		uint32_t end2, v[AHEAD];
		u32x4 c[AHEAD][2];
	};
	// (no bounds: a position past the ring reads another's and is not used).
	auto fetch = [&](Ahead &s, uint32_t from, uint32_t ring) {
		s.end2 = a.limits[min(ring + 2, a.nl - 1)];
#pragma unroll
		for (uint32_t j = 0; j < AHEAD; j++) {
			const uint32_t q = min(from + j * NT + tid, a.nr - 1);
			const u32x4 *row = (const u32x4 *) (a.child + (size_t) q * CHILD_ROWS);
			s.v[j] = a.sorted[q];
			s.c[j][0] = row[0];
			s.c[j][1] = row[1];
		}
	};
	auto push = [&](uint32_t i, const u32x4 c0, const u32x4 c1) {
		const uint32_t rk = (uint32_t) ld(&rank[i]) << 5;
		if (c1.w != CHILD_MORE) {
			const uint32_t e[CHILD_ROWS] = { c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w };
#pragma unroll
			for (uint32_t k = 0; k < CHILD_ROWS; k++)
				if (e[k] != GP_NIL) atomicMin(&key[e[k] >> 5], rk | (e[k] & 31u));
		} else {
			const uint32_t v = a.sorted[b0 + i], s = a.fan_off[v], c = a.fan_off[v + 1] - s;
			const uint32_t n = (c && a.closed[v]) ? c - 1 : c, l1 = a.level[v] + 1;
			for (uint32_t k = 0; k < n; k++) {
				const uint32_t u = a.fan[s + k];
				if (a.level[u] == l1) atomicMin(&key[a.inv[u] - b1], rk | k);
			}
		}
	};
	// Ring r -> r + 1: `cur` holds ring r, `nxt` ring r + 1; once ring r's
	// children are pushed, `cur` is refilled with ring r + 2, almost two rings
	// ahead of its use.
	auto step = [&](Ahead &cur, const Ahead &nxt, uint32_t r) {
		const uint32_t n0 = b1 - b0, n1 = b2 - b1;
#pragma unroll
		for (uint32_t j = 0; j < AHEAD; j++)
			if (j * NT + tid < n0) push(j * NT + tid, cur.c[j][0], cur.c[j][1]);
		for (uint32_t i = AHEAD * NT + tid; i < n0; i += NT) {
			const u32x4 *row = (const u32x4 *) (a.child + (size_t) (b0 + i) * CHILD_ROWS);
			push(i, row[0], row[1]);
		}
		const uint32_t b3 = __builtin_amdgcn_readfirstlane(nxt.end2);
		fetch(cur, b2, r + 2);
		order_barrier<LDS>();
		for (uint32_t i = tid; i < n1; i += NT) {
			const uint32_t k = ld(&key[i]);
			atomicOr(&mask[k >> 5], 1u << (k & 31u));
		}
		order_barrier<LDS>();
		// Exclusive sums of the bit counts, NT parents at a time; the halves of
		// part[] alternate, so one barrier a pass is enough.
		uint32_t carry = 0;
		for (uint32_t i0 = 0, h = 0; i0 < n0; i0 += NT, h ^= 1u) {
			const uint32_t i = i0 + tid;
			const uint32_t x = i < n0 ? (uint32_t) __popc(ld(&mask[i])) : 0u;
			const uint32_t inc = wave_scan(x);
			if (lane == 63) part[h][wave] = inc;
			order_barrier<LDS>();
			uint32_t before = 0, total = 0;
#pragma unroll
			for (uint32_t q = 0; q < NT / 64; q++) {
				const uint32_t t = part[h][q];
				before += q < wave ? t : 0u;
				total += t;
			}
			if (i < n0) st(&base[i], carry + before + inc - x);
			carry += total;
		}
		order_barrier<LDS>();
		for (uint32_t i = tid, j = 0; i < n1; i += NT, j++) {
			const uint32_t k = ld(&key[i]), p = k >> 5;
			const uint32_t at = (uint32_t) ld(&base[p]) + (uint32_t) __popc(ld(&mask[p]) & ((1u << (k & 31u)) - 1u));
			st(&rank[i], at);
			a.out[b1 + at] = j == 0 ? nxt.v[0] : j == 1 ? nxt.v[1] : a.sorted[b1 + i];
		}
		order_barrier<LDS>();
		// Lists of the next ring (its parents are this ring's children).
		for (uint32_t i = tid; i < b3 - b2; i += NT) st(&key[i], GP_NIL);
		for (uint32_t i = tid; i < n1; i += NT) st(&mask[i], 0u);
		order_barrier<LDS>();
		b0 = b1; b1 = b2; b2 = b3;
	};
	Ahead s0, s1;
	fetch(s0, b0, 0);
	fetch(s1, b1, 1);
	order_barrier<LDS>();
	for (uint32_t r = 0; r + 2 < a.nl; r += 2) {
		step(s0, s1, r);
		if (r + 3 >= a.nl) break;
		step(s1, s0, r + 1);
	}
}

__global__ void k_order_tail(uint32_t *out, uint32_t from, uint32_t n)
{
	for (uint32_t q = from + blockIdx.x * blockDim.x + threadIdx.x; q < n; q += gridDim.x * blockDim.x) out[q] = GP_NIL;
}

static uint32_t fill_grid(uint32_t n) { return std::max<uint32_t>(1, std::min<uint32_t>(2048, (n + 255) / 256)); }

// Widest rings whose arrays (12 bytes a vertex) fit in LDS.  Small rings run
// with fewer waves, whose barriers are cheaper.
constexpr uint32_t ORDER_LDS_SMALL = 1024, ORDER_LDS = 12288;

int RingOrder::queue(const Levels &lv, const LevelInfo &li, const uint32_t *limits, const uint32_t *inv,
                     const uint32_t *d_src, uint32_t ns, hipStream_t on)
{
	stream = on;
	const bool wide = li.max_ring > ORDER_LDS;
	if (pool_malloc(&child, 4ull * CHILD_ROWS * li.nr) != hipSuccess || pool_malloc(&rank0, 4ull * ns) != hipSuccess ||
	    pool_malloc(&out, 4ull * lv.nv) != hipSuccess ||
	    (wide && pool_malloc(&work, 16ull * li.max_ring) != hipSuccess))
		return fail(GP_ERR_NOMEM, "rings: device allocation failed");
	const DeviceMesh *dm = lv.dm;
	const OrderArgs a{ lv.sorted, limits, lv.level, inv, dm->fan_off, dm->fan, dm->closed, li.nl, li.nr, child, rank0, out };
	k_ring_rank0<<<fill_grid(ns), 256, 0, stream>>>(d_src, ns, inv, rank0);
	k_ring_children<<<fill_grid(li.nr), 256, 0, stream>>>(a);
	if (li.nr < lv.nv) k_order_tail<<<fill_grid(lv.nv - li.nr), 256, 0, stream>>>(out, li.nr, lv.nv);
	if (wide) k_ring_order<1024, 0><<<1, 1024, 0, stream>>>(a, work, li.max_ring);
	else if (li.max_ring > ORDER_LDS_SMALL) k_ring_order<1024, ORDER_LDS><<<1, 1024, 0, stream>>>(a, nullptr, 0);
	else k_ring_order<256, ORDER_LDS_SMALL><<<1, 256, 0, stream>>>(a, nullptr, 0);
	GP_HIP(hipGetLastError());
	return GP_OK;
}

__global__ void k_rings_init(uint32_t *level, unsigned long long *key, uint32_t *sorted, uint32_t nv)
{
	for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < nv; v += gridDim.x * blockDim.x) {
		level[v] = GP_NIL;
		key[v] = ~0ull;
		sorted[v] = GP_NIL;
	}
}

__global__ __launch_bounds__(BFS_THREADS) void k_rings_bfs(const uint32_t *fan_off, const uint32_t *fan,
                                                           const uint8_t *closed, const BfsJob *jobs)
{
	bfs_block(fan_off, fan, closed, jobs[blockIdx.x]);
}

// The one-workgroup BFS, for meshes with links over ORDER_MAX_LINK.
static int toplesets_bfs(Che &m, const uint32_t *src, uint32_t ns, uint32_t *levels, uint32_t *sorted,
                         std::vector<uint32_t> &limits)
{
	for (uint32_t v = 0; v < m.nv; v++)
		if (m.fan_off[v + 1] - m.fan_off[v] > MAX_LINK) return fail(GP_ERR_CAPACITY, "vertex %u: link over %u", v, MAX_LINK);
	int rc = upload_mesh(m);
	if (rc) return rc;
	const DeviceMesh *dm = m.dev;
	const uint32_t nv = m.nv;
	uint32_t *d_level = nullptr, *d_sorted = nullptr, *d_limits = nullptr, *d_nl = nullptr, *d_src = nullptr;
	unsigned long long *d_key = nullptr;
	BfsJob *d_job = nullptr;
	struct Free {
		std::vector<void *> p;
		~Free() { for (void *q : p) (void) hipFree(q); }
	} fr;
	if (device_malloc(&d_level, 4ull * nv) != hipSuccess || device_malloc(&d_sorted, 4ull * nv) != hipSuccess ||
	    device_malloc(&d_limits, 4ull * (nv + 2)) != hipSuccess || device_malloc(&d_nl, 4) != hipSuccess ||
	    device_malloc(&d_src, 4ull * ns) != hipSuccess || device_malloc(&d_key, 8ull * nv) != hipSuccess ||
	    device_malloc(&d_job, sizeof(BfsJob)) != hipSuccess) {
		fr.p = { d_level, d_sorted, d_limits, d_nl, d_src, d_key, d_job };
		return fail(GP_ERR_NOMEM, "toplesets_gpu: allocation failed");
	}
	fr.p = { d_level, d_sorted, d_limits, d_nl, d_src, d_key, d_job };
	BfsJob job{ d_src, ns, d_level, d_key, d_sorted, d_limits, d_nl };
	GP_HIP(hipMemcpy(d_src, src, 4ull * ns, hipMemcpyHostToDevice));
	GP_HIP(hipMemcpy(d_job, &job, sizeof(job), hipMemcpyHostToDevice));
	const uint32_t g = std::max<uint32_t>(1, std::min<uint32_t>(2048, (nv + 255) / 256));
	k_rings_init<<<g, 256>>>(d_level, d_key, d_sorted, nv);
	GP_HIP(hipGetLastError());
	k_rings_bfs<<<1, BFS_THREADS>>>(dm->fan_off, dm->fan, dm->closed, d_job);
	GP_HIP(hipGetLastError());
	GP_HIP(hipDeviceSynchronize());
	uint32_t nl = 0;
	GP_HIP(hipMemcpy(&nl, d_nl, 4, hipMemcpyDeviceToHost));
	if (nl < 2 || nl > nv + 2) return fail(GP_ERR_KERNEL, "toplesets_gpu: bad ring count %u", nl);
	limits.resize(nl);
	GP_HIP(hipMemcpy(limits.data(), d_limits, 4ull * nl, hipMemcpyDeviceToHost));
	GP_HIP(hipMemcpy(levels, d_level, 4ull * nv, hipMemcpyDeviceToHost));
	GP_HIP(hipMemcpy(sorted, d_sorted, 4ull * nv, hipMemcpyDeviceToHost));
	return GP_OK;
}

int toplesets_gpu(Che &m, const uint32_t *src, uint32_t ns, uint32_t *levels, uint32_t *sorted,
                  std::vector<uint32_t> &limits)
{
	limits.clear();
	if (ns == 0) return GP_OK;
	std::vector<uint8_t> seen(m.nv, 0);
	for (uint32_t q = 0; q < ns; q++) {
		if (src[q] >= m.nv) return fail(GP_ERR_INVALID, "toplesets: source %u out of range", src[q]);
		if (seen[src[q]]) return fail(GP_ERR_DUPLICATE_SOURCE, "toplesets: source %u listed twice", src[q]);
		seen[src[q]] = 1;
	}
	if (m.max_link > ORDER_MAX_LINK) return toplesets_bfs(m, src, ns, levels, sorted, limits);
	int rc = upload_mesh(m);
	if (rc) return rc;
	const uint32_t nv = m.nv;
	PoolStream ps;
	GP_HIP(ps.create());
	const hipStream_t stream = ps.s;
	PoolBuf<uint32_t> srcb(stream), invb(stream);
	if (srcb.alloc(4ull * ns) != hipSuccess || invb.alloc(4ull * nv) != hipSuccess)
		return fail(GP_ERR_NOMEM, "toplesets_gpu: allocation failed");
	uint32_t *const d_src = srcb.p, *const d_inv = invb.p;
	GP_HIP(hipMemcpy(d_src, src, 4ull * ns, hipMemcpyHostToDevice));
	Levels lv;
	if ((rc = lv.create(m.dev, stream))) return rc;
	lv.clear();
	lv.seed(d_src, 0, ns);
	if ((rc = lv.expand())) return rc;
	lv.sort();
	LevelInfo li;
	if ((rc = lv.info(li))) return rc;
	k_ring_inv<<<fill_grid(li.nr), 256, 0, stream>>>(lv.sorted, li.nr, d_inv);
	RingOrder ord;
	if ((rc = ord.queue(lv, li, lv.limits, d_inv, d_src, ns, stream))) return rc;
	limits.resize(li.nl);
	GP_HIP(hipMemcpyAsync(limits.data(), lv.limits, 4ull * li.nl, hipMemcpyDeviceToHost, stream));
	GP_HIP(hipMemcpyAsync(levels, lv.level, 4ull * nv, hipMemcpyDeviceToHost, stream));
	GP_HIP(hipMemcpyAsync(sorted, ord.out, 4ull * nv, hipMemcpyDeviceToHost, stream));
	GP_HIP(hipStreamSynchronize(stream));
	return GP_OK;
}

}  // namespace gp
