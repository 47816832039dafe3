// Device memory, pinned host memory and streams kept between calls (pool.hpp).
#include "pool.hpp"

#include <algorithm>
#include <deque>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

namespace gp {

namespace {

struct Block {
	void *p;
	size_t bytes;
	int dev;
};

struct Lists {
	std::mutex mu;
	std::map<void *, std::pair<size_t, int>> used;   // device blocks handed out: size, device
	std::deque<Block> free_dev;                      // oldest first
	size_t free_bytes = 0;
	std::map<void *, size_t> used_pinned;
	std::deque<Block> free_pinned;
	size_t pinned_bytes = 0;
	std::vector<std::pair<hipStream_t, int>> streams;
	size_t meshes = 0;
};

// Never destroyed: objects of the process may outlive static destructors, and
// the runtime takes its memory back by itself.
Lists &lists()
{
	static Lists *l = new Lists;
	return *l;
}

constexpr size_t MAX_STREAMS = 16;

// Sizes in steps of an eighth of their power of two, so that meshes of nearly
// one size share blocks.
size_t round_up(size_t n)
{
	size_t step = 256;
	while (step * 16 < n) step *= 2;
	return (std::max<size_t>(n, 1) + step - 1) / step * step;
}

// Everything kept goes back to the runtime (lock held).
void empty(Lists &l)
{
	int cur = 0;
	(void) hipGetDevice(&cur);
	for (const Block &b : l.free_dev) {
		(void) hipSetDevice(b.dev);
		(void) hipFree(b.p);
	}
	l.free_dev.clear();
	l.free_bytes = 0;
	for (const Block &b : l.free_pinned) (void) hipHostFree(b.p);
	l.free_pinned.clear();
	l.pinned_bytes = 0;
	for (const auto &s : l.streams) {
		(void) hipSetDevice(s.second);
		(void) hipStreamDestroy(s.first);
	}
	l.streams.clear();
	(void) hipSetDevice(cur);
}

// Smallest kept block of the device that holds `bytes` without wasting more than
// half of itself.
std::deque<Block>::iterator best_fit(std::deque<Block> &v, size_t bytes, int dev)
{
	auto best = v.end();
	for (auto it = v.begin(); it != v.end(); ++it)
		if (it->dev == dev && it->bytes >= bytes && it->bytes <= 2 * bytes && (best == v.end() || it->bytes < best->bytes))
			best = it;
	return best;
}

}  // namespace

hipError_t device_malloc_bytes(void **p, size_t bytes)
{
	hipError_t e = hipMalloc(p, bytes);
	if (e != hipSuccess) {
		(void) hipGetLastError();
		std::lock_guard<std::mutex> lock(lists().mu);
		empty(lists());
		e = hipMalloc(p, bytes);
	}
	return e;
}

hipError_t pool_malloc_bytes(void **p, size_t bytes)
{
	*p = nullptr;
	int dev = 0;
	hipError_t e = hipGetDevice(&dev);
	if (e != hipSuccess) return e;
	bytes = round_up(bytes);
	Lists &l = lists();
	{
		std::lock_guard<std::mutex> lock(l.mu);
		auto it = best_fit(l.free_dev, bytes, dev);
		if (it != l.free_dev.end()) {
			*p = it->p;
			l.used[it->p] = { it->bytes, dev };
			l.free_bytes -= it->bytes;
			l.free_dev.erase(it);
			return hipSuccess;
		}
	}
	if ((e = device_malloc_bytes(p, bytes)) != hipSuccess) return e;
	std::lock_guard<std::mutex> lock(l.mu);
	l.used[*p] = { bytes, dev };
	return hipSuccess;
}

hipError_t pool_free(void *p)
{
	if (!p) return hipSuccess;
	Lists &l = lists();
	std::vector<Block> drop;
	{
		std::lock_guard<std::mutex> lock(l.mu);
		auto it = l.used.find(p);
		if (it == l.used.end()) return hipErrorInvalidValue;
		const Block b{ p, it->second.first, it->second.second };
		l.used.erase(it);
		if (b.bytes > POOL_BYTES || l.meshes == 0) {
			drop.push_back(b);
		} else {
			l.free_dev.push_back(b);
			l.free_bytes += b.bytes;
			while (l.free_bytes > POOL_BYTES) {
				drop.push_back(l.free_dev.front());
				l.free_bytes -= l.free_dev.front().bytes;
				l.free_dev.pop_front();
			}
		}
	}
	for (const Block &b : drop) (void) hipFree(b.p);
	return hipSuccess;
}

hipError_t pinned_malloc_bytes(void **p, size_t bytes)
{
	*p = nullptr;
	bytes = round_up(bytes);
	Lists &l = lists();
	{
		std::lock_guard<std::mutex> lock(l.mu);
		auto it = best_fit(l.free_pinned, bytes, 0);
		if (it != l.free_pinned.end()) {
			*p = it->p;
			l.used_pinned[it->p] = it->bytes;
			l.pinned_bytes -= it->bytes;
			l.free_pinned.erase(it);
			return hipSuccess;
		}
	}
	hipError_t e = hipHostMalloc(p, bytes);
	if (e != hipSuccess) {
		(void) hipGetLastError();
		{
			std::lock_guard<std::mutex> lock(l.mu);
			empty(l);
		}
		e = hipHostMalloc(p, bytes);
	}
	if (e != hipSuccess) {
		(void) hipGetLastError();
		*p = nullptr;
		return e;
	}
	std::lock_guard<std::mutex> lock(l.mu);
	l.used_pinned[*p] = bytes;
	return hipSuccess;
}

void pinned_free(void *p)
{
	if (!p) return;
	Lists &l = lists();
	std::vector<void *> drop;
	{
		std::lock_guard<std::mutex> lock(l.mu);
		auto it = l.used_pinned.find(p);
		if (it == l.used_pinned.end()) return;
		const size_t bytes = it->second;
		l.used_pinned.erase(it);
		if (bytes > POOL_PINNED || l.meshes == 0) {
			drop.push_back(p);
		} else {
			l.free_pinned.push_back(Block{ p, bytes, 0 });
			l.pinned_bytes += bytes;
			while (l.pinned_bytes > POOL_PINNED) {
				drop.push_back(l.free_pinned.front().p);
				l.pinned_bytes -= l.free_pinned.front().bytes;
				l.free_pinned.pop_front();
			}
		}
	}
	for (void *q : drop) (void) hipHostFree(q);
}

hipError_t pool_stream(hipStream_t *s)
{
	int dev = 0;
	hipError_t e = hipGetDevice(&dev);
	if (e != hipSuccess) return e;
	Lists &l = lists();
	{
		std::lock_guard<std::mutex> lock(l.mu);
		for (size_t q = l.streams.size(); q-- > 0;)
			if (l.streams[q].second == dev) {
				*s = l.streams[q].first;
				l.streams.erase(l.streams.begin() + (long) q);
				return hipSuccess;
			}
	}
	return hipStreamCreateWithFlags(s, hipStreamNonBlocking);
}

void pool_stream_free(hipStream_t s)
{
	if (!s) return;
	int dev = 0;
	Lists &l = lists();
	if (hipStreamGetDevice(s, &dev) == hipSuccess) {
		std::lock_guard<std::mutex> lock(l.mu);
		if (l.meshes && l.streams.size() < MAX_STREAMS) {
			l.streams.push_back({ s, dev });
			return;
		}
	}
	(void) hipStreamDestroy(s);
}

void pool_mesh_added()
{
	std::lock_guard<std::mutex> lock(lists().mu);
	lists().meshes++;
}

void pool_mesh_removed()
{
	Lists &l = lists();
	std::lock_guard<std::mutex> lock(l.mu);
	if (l.meshes && --l.meshes == 0) empty(l);
}

}  // namespace gp
