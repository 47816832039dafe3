// Stand-in for the HIP runtime's memory and stream calls, on the host: counts what
// is allocated, in what order it is freed, and fails on demand.
#pragma once

#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <map>
#include <set>
#include <vector>

typedef int hipError_t;
typedef struct FakeStream *hipStream_t;
enum { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum { hipStreamNonBlocking = 1 };

namespace fake {
struct Heap {
	std::map<void *, size_t> live;
	std::vector<void *> freed;
	size_t bytes = 0, limit = SIZE_MAX;
	int fail = 0;   // calls to refuse
	uintptr_t next = 4096;
	hipError_t get(void **p, size_t n)
	{
		*p = nullptr;
		if (fail > 0) { fail--; return hipErrorOutOfMemory; }
		if (bytes + n > limit) return hipErrorOutOfMemory;
		*p = (void *) next;
		next += n + 4096;
		live[*p] = n;
		bytes += n;
		return hipSuccess;
	}
	hipError_t put(void *p)
	{
		auto it = live.find(p);
		if (it == live.end()) std::abort();   // freed twice, or never allocated
		bytes -= it->second;
		live.erase(it);
		freed.push_back(p);
		return hipSuccess;
	}
};
inline Heap device, pinned;
inline std::set<hipStream_t> streams;
inline uintptr_t next_stream = 1;
}  // namespace fake

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMalloc(void **p, size_t n) { return fake::device.get(p, n); }
inline hipError_t hipFree(void *p) { return p ? fake::device.put(p) : hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n) { return fake::pinned.get(p, n); }
inline hipError_t hipHostFree(void *p) { return fake::pinned.put(p); }
inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
	*s = (hipStream_t) fake::next_stream++;
	fake::streams.insert(*s);
	return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s)
{
	if (!fake::streams.erase(s)) std::abort();
	return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t, int *d) { *d = 0; return hipSuccess; }
