// Multi-source BFS levels on the device and the vertices sorted by level (the
// rings of parallel_toplesets_propagation, che::compute_toplesets,
// src/che.cpp:546-593, as sets).  A frontier BFS over all workgroups (each
// launch takes the frontier LV_DEPTH levels further, the host polling a done
// flag) lowers the levels from the seeded sources, stopping where the levels
// are already as low -- so seeding one more source into existing levels updates
// them incrementally -- and a counting sort by level and, inside a level, by
// slot count (longest fans first) rebuilds sorted[], limits and the slot rows
// of each 64-position chunk.  The order inside a ring is not the reference's
// discovery order (the window sweeps relax whole rings, so it changes no
// value).
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"

namespace gp {

// First 8 link entries of each vertex in 32 bytes (NIL past the link; LONG_LINK
// on entry 7 when the link goes on in the fan table): DeviceMesh::link8.
constexpr uint32_t LONG_LINK = 0x80000000u, LINK_ROW = 8;
int link_rows(DeviceMesh *dm);

struct LevelState;

constexpr uint32_t LEVEL_KEYS = 8;   // slot classes per level in the sort key

// Sizes of sorted rings: |limits|, reached vertices, their chunks' slot rows,
// the widest ring.
struct LevelInfo {
	uint32_t nl, nr, rows, max_ring;
};

struct Levels {
	uint32_t nv = 0;
	uint32_t *level = nullptr;    // [nv], NIL = unreached
	uint32_t *queue = nullptr;    // [2][nv] frontier of this launch and the next
	uint32_t *mark = nullptr;     // [nv] number of the last launch that queued the vertex
	uint32_t lv_grid = 1;
	bool fresh = true;            // the state has not been seeded yet
	uint32_t *hist = nullptr;     // [nv * LEVEL_KEYS + 1]  key counts, then cursors
	uint32_t *sorted = nullptr;   // [nv]   vertices by level, longest fans first in a level
	uint32_t *limits = nullptr;   // [nv + 2]
	uint32_t *nl = nullptr;       // |limits| (device)
	uint32_t *cslots = nullptr;   // [nchunks() + 1] slot rows of each 64-position chunk of sorted
	uint32_t *coff = nullptr;     // [nchunks() + 1] their exclusive prefix (chunk c at row coff[c])
	LevelState *ls = nullptr, *h_ls = nullptr;   // h_ls: two pinned snapshots
	LevelInfo *h_info = nullptr;  // pinned (behind the snapshots)
	hipEvent_t ev[2] = { nullptr, nullptr };
	hipStream_t stream = nullptr;   // borrowed
	DeviceMesh *dm = nullptr;

	Levels() = default;
	Levels(const Levels &) = delete;
	Levels &operator=(const Levels &) = delete;
	~Levels();
	int create(DeviceMesh *mesh, hipStream_t s);
	void clear();                                               // every level unreached
	void seed(const uint32_t *d_src, uint32_t first, uint32_t ns);   // d_src[first, ns) to level 0
	int expand();                                               // BFS to completion
	void sort();                                                // sorted, limits, nl, coff on the device
	int info(LevelInfo &out);                                   // sizes of the last sort (waits for it)
	uint32_t nchunks() const { return (nv + 63) / 64; }
};

// Reference order of the sorted rings (rings.hip): ring_order_queue enqueues the
// kernels that write sorted_out[nv] (device; NIL past the reached vertices) in
// the discovery order of che::compute_toplesets from rings sorted as sets
// (lv.sorted, lv.limits, lv.level and inv[nv], the position of each vertex in
// lv.sorted; d_src: the sources in the caller's order).  Everything passed stays
// unchanged and allocated until the stream has run them.
constexpr uint32_t ORDER_MAX_LINK = GP_ORDERED_LINK;   // longer links: the one-workgroup BFS of rings.hip

struct RingOrder {
	uint32_t *child = nullptr, *rank0 = nullptr, *work = nullptr, *out = nullptr;
	hipStream_t stream = nullptr;   // the one it was queued on
	~RingOrder()
	{
		if (stream) (void) hipStreamSynchronize(stream);
		for (void *p : { (void *) child, (void *) rank0, (void *) work, (void *) out }) (void) pool_free(p);
	}
	int queue(const Levels &lv, const LevelInfo &li, const uint32_t *limits, const uint32_t *inv, const uint32_t *d_src,
	          uint32_t ns, hipStream_t on);
};

}  // namespace gp
