// Device memory, pinned host memory and streams kept between calls.
//
// A solve makes and drops about forty device buffers, three pinned records and
// a stream or two; at 1M vertices hipMalloc and hipFree took 2.6-5 ms of a 23 ms
// solve (hipFree waits for the device), at 10k vertices streams and pinned
// records 0.3 of 1.2 ms.  So what a call drops goes on a list here and the next
// call takes it from there: with results by way of pinned memory a 1M FP64 solve
// went from 21.8 to 18.7 ms, a 10k one from 1.21 to 1.06, a learned 1M plan from
// 28.0 to 21.9.
//
// The lists are process-wide, per device and locked.  They hold at most
// POOL_BYTES of device memory (the oldest blocks go back first) and are emptied
// when the last mesh with device tables is destroyed, or when an allocation
// fails.  A block comes with whatever it held before.  Whoever drops a block
// has waited for every stream that uses it: the owners here synchronise their
// stream first.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace gp {

constexpr size_t POOL_BYTES = size_t(1) << 30;     // device memory kept, at most
constexpr size_t POOL_PINNED = size_t(64) << 20;   // pinned memory kept, at most

hipError_t device_malloc_bytes(void **p, size_t bytes);   // not kept: hipMalloc, the lists emptied if it fails
hipError_t pool_malloc_bytes(void **p, size_t bytes);
hipError_t pool_free(void *p);
hipError_t pinned_malloc_bytes(void **p, size_t bytes);
void pinned_free(void *p);
hipError_t pool_stream(hipStream_t *s);            // non-blocking, default priority
void pool_stream_free(hipStream_t s);              // idle

// Meshes with device tables: the lists are emptied with the last one.
void pool_mesh_added();
void pool_mesh_removed();

template <typename T>
hipError_t device_malloc(T **p, size_t bytes)
{
	return device_malloc_bytes((void **) p, bytes);
}
template <typename T>
hipError_t pool_malloc(T **p, size_t bytes)
{
	return pool_malloc_bytes((void **) p, bytes);
}
template <typename T>
hipError_t pinned_malloc(T **p, size_t bytes)
{
	return pinned_malloc_bytes((void **) p, bytes);
}

// A stream and its place back in the pool.
struct PoolStream {
	hipStream_t s = nullptr;
	PoolStream() = default;
	PoolStream(const PoolStream &) = delete;
	PoolStream &operator=(const PoolStream &) = delete;
	hipError_t create() { return pool_stream(&s); }
	~PoolStream()
	{
		if (!s) return;
		(void) hipStreamSynchronize(s);
		pool_stream_free(s);
	}
};

// A device buffer used on one stream (null: the null stream).
template <typename T>
struct PoolBuf {
	T *p = nullptr;
	hipStream_t s;
	explicit PoolBuf(hipStream_t stream) : s(stream) {}
	PoolBuf(const PoolBuf &) = delete;
	PoolBuf &operator=(const PoolBuf &) = delete;
	hipError_t alloc(size_t bytes) { return pool_malloc(&p, bytes); }
	~PoolBuf()
	{
		if (!p) return;
		(void) hipStreamSynchronize(s);
		(void) pool_free(p);
	}
};

}  // namespace gp
