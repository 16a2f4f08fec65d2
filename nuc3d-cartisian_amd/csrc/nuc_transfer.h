// nuc_transfer.h -- copies between pageable host arrays and device buffers.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace nuctransfer {

// Copies `bytes` between host and device memory, ordered after the earlier
// work of `s`; returns when the copy is complete.  Any host pointer
// hipMemcpyAsync takes is accepted.
hipError_t copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t s);

// The staging memory is kept while someone holds it: every context and every
// serving loop (whose contexts come and go) does, once.
void retain();
void release();

}  // namespace nuctransfer
