// The pool of device memory, pinned memory and streams on a stand-in of the HIP
// runtime: what it keeps, in what order it gives it back, and what it does when an
// allocation fails.  argv[1] names the check; exit status 1 and a line where it fails.
#include "../../gproshan_amd/csrc/pool.hip"

#include <cstdio>
#include <cstring>

using namespace gp;

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

constexpr size_t MB = size_t(1) << 20;

static void *dev(size_t n)
{
	void *p = nullptr;
	return pool_malloc_bytes(&p, n) == hipSuccess ? p : nullptr;
}
static void *pin(size_t n)
{
	void *p = nullptr;
	return pinned_malloc_bytes(&p, n) == hipSuccess ? p : nullptr;
}

// 20 blocks of 128 MiB dropped one after the other: POOL_BYTES stay, the newest.
static int device_bound()
{
	pool_mesh_added();
	std::vector<void *> b;
	for (int q = 0; q < 20; q++) {
		b.push_back(dev(128 * MB));
		CHECK(b.back());
	}
	for (void *p : b) {
		CHECK(pool_free(p) == hipSuccess);
		size_t used = 0;
		for (void *q : b)
			if (q > p && fake::device.live.count(q)) used += 128 * MB;
		CHECK(fake::device.bytes - used <= POOL_BYTES);
	}
	CHECK(fake::device.bytes == POOL_BYTES);
	CHECK(fake::device.freed.size() == 12);
	for (int q = 0; q < 12; q++) CHECK(fake::device.freed[q] == b[q]);
	CHECK(pool_free(b[19]) != hipSuccess);         // twice
	void *p = dev(POOL_BYTES + MB);                // larger than the pool: not kept
	CHECK(p && pool_free(p) == hipSuccess && fake::device.bytes == POOL_BYTES);
	p = dev(100 * MB);                             // from the list
	CHECK(fake::device.live.count(p) && fake::device.bytes == POOL_BYTES);
	CHECK(dev(50 * MB) && fake::device.bytes > POOL_BYTES);   // half of a kept block would be wasted
	pool_mesh_removed();
	CHECK(fake::device.live.size() == 2);          // those in use
	CHECK(pool_free(p) == hipSuccess && fake::device.live.size() == 1);   // no mesh: not kept
	return 0;
}

static int pinned_bound()
{
	pool_mesh_added();
	std::vector<void *> b;
	for (int q = 0; q < 20; q++) b.push_back(pin(8 * MB));
	for (void *p : b) pinned_free(p);
	CHECK(fake::pinned.bytes == POOL_PINNED);
	for (int q = 0; q < 12; q++) CHECK(fake::pinned.freed[q] == b[q]);
	void *p = pin(POOL_PINNED + MB);
	CHECK(p);
	pinned_free(p);
	CHECK(fake::pinned.bytes == POOL_PINNED);
	pool_mesh_removed();
	CHECK(fake::pinned.live.empty());
	return 0;
}

// A failed allocation, device or pinned: everything kept goes back, and it is
// tried once more.
static int fails(bool pinned)
{
	fake::Heap &h = pinned ? fake::pinned : fake::device;
	pool_mesh_added();
	hipStream_t s;
	CHECK(pool_stream(&s) == hipSuccess);
	pool_stream_free(s);
	CHECK(fake::streams.size() == 1);
	void *d = dev(MB), *k = pin(MB), *keep = pin(3 * MB);
	CHECK(d && k && keep);
	pool_free(d);
	pinned_free(k);
	h.limit = h.bytes + 7 * MB;                    // room for 8 MB only without the kept one
	void *p = pinned ? pin(8 * MB) : dev(8 * MB);
	CHECK(p);
	CHECK(fake::streams.empty());
	CHECK(fake::device.live.size() == (pinned ? 0u : 1u));
	CHECK(fake::pinned.live.size() == (pinned ? 2u : 1u));
	p = pinned ? pin(64 * MB) : dev(64 * MB);      // no room at all: refused, nothing lost
	CHECK(!p);
	pinned_free(keep);
	h.limit = SIZE_MAX;
	CHECK(pinned ? pin(64 * MB) : dev(64 * MB));
	return 0;
}

int main(int argc, char **argv)
{
	const char *what = argc > 1 ? argv[1] : "";
	if (!std::strcmp(what, "device_bound")) return device_bound();
	if (!std::strcmp(what, "pinned_bound")) return pinned_bound();
	if (!std::strcmp(what, "device_fails")) return fails(false);
	if (!std::strcmp(what, "pinned_fails")) return fails(true);
	return 2;
}
