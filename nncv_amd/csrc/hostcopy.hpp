// Host-side copies between the caller's pageable memory and pinned staging memory on a few threads (the reference ABI hands
// over pageable host buffers: examples/Res18/main.cpp:79-99).
#pragma once
#include <cstddef>

namespace nncv_hip {

// dst[0..bytes) = src[0..bytes), split over the calling thread and the pool's workers (started on first use, kept for the
// life of the process).  Callers are serialised by the library's mutex.
void parallel_copy(void* dst, const void* src, size_t bytes);

}  // namespace nncv_hip
