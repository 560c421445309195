// Declarations shared between the copy kernels' host code.
#pragma once
#include <hip/hip_runtime.h>

#include "mhip_internal.h"

namespace mhip {

// Launches the LDS-tiled transposing copy when the canonical slice calls for it (the
// memory-contiguous dimension is not the innermost iteration dimension).  Returns false
// when the direct chunk copy should be used instead; otherwise *rc holds the launch status.
template <bool PACK>
bool try_transpose_copy(char* base, char* packed, const CanonSlice& c, uint32_t unit, hipStream_t stream, int* rc);

// The same for views with a side of at most 512 bytes and for small views; `cd` is the memory-contiguous dimension of
// `c`, nbatch the product of the dimensions before it and Q of those after it.  Returns false for other views.
template <bool PACK>
bool try_narrow_transpose(char* base, char* packed, const CanonSlice& c, int cd, uint64_t nbatch, uint32_t Q, uint32_t unit,
                          hipStream_t stream, int* rc);

}  // namespace mhip
