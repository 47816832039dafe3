// Refuses pinned host memory over a number of bytes: loaded before the library,
// this hipHostMalloc is the one it calls.
#include <cstddef>
#include <dlfcn.h>

extern "C" {

size_t pinned_limit = (size_t) -1;
size_t pinned_refused = 0;

int hipHostMalloc(void **p, size_t bytes, unsigned flags)
{
	static int (*real)(void **, size_t, unsigned) = (int (*)(void **, size_t, unsigned)) dlsym(RTLD_NEXT, "hipHostMalloc");
	if (!real) return 999;
	if (bytes <= pinned_limit) return real(p, bytes, flags);
	pinned_refused++;
	*p = nullptr;
	return 2;   // hipErrorOutOfMemory
}

}
