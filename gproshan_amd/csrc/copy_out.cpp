// Copies out of pinned staging memory on several threads: most of the time of
// filling a caller's fresh array is the kernel handing out its pages.
#include "gp_internal.hpp"

#include <omp.h>

#include <algorithm>
#include <cstring>

namespace gp {

void copy_out(void *dst, const void *src, size_t bytes)
{
	constexpr size_t PIECE = size_t(256) << 10;
	const int64_t n = (int64_t) ((bytes + PIECE - 1) / PIECE);
	const int threads = (int) std::min<int64_t>({ n, 8, (int64_t) omp_get_max_threads() });
	if (threads < 2) {
		std::memcpy(dst, src, bytes);
		return;
	}
	#pragma omp parallel for schedule(static) num_threads(threads)
	for (int64_t q = 0; q < n; q++) {
		const size_t at = (size_t) q * PIECE;
		std::memcpy((char *) dst + at, (const char *) src + at, std::min(PIECE, bytes - at));
	}
}

}  // namespace gp
