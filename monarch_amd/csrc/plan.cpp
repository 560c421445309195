// Host-side planning: turn a Slice into the few numbers a copy kernel needs.
#include "mhip_internal.h"

namespace mhip {

static inline uint32_t pow2_factor(uint64_t v, uint32_t cap) {
    // largest power of two <= cap dividing v (v == 0 divides by everything)
    uint32_t u = cap;
    while (u > 1 && (v & (u - 1))) u >>= 1;
    return u;
}

bool canonicalize(const mhip_slice_t& s, uint32_t elem_size, uint64_t align_mask, uint32_t max_unit,
                  CanonSlice* out, uint32_t* unit, uint64_t* skew) {
    uint64_t len = 1;
    for (uint32_t k = 0; k < s.ndim; ++k) len *= s.sizes[k];
    if (len == 0 || elem_size == 0) return false;

    // (size, byte stride), outermost first; the element itself is the innermost dimension.
    // Neighbours that walk one linear run are merged on the way.
    CanonDim* const dims = out->dims;
    int n = 0;
    auto add = [&](uint64_t size, uint64_t stride) {
        if (n > 0 && dims[n - 1].stride == stride * size) {
            // previous (outer) dimension steps by exactly the extent of this one
            dims[n - 1].size *= size;
            dims[n - 1].stride = stride;
        } else {
            dims[n++] = {size, stride};
        }
    };
    for (uint32_t k = 0; k < s.ndim; ++k)
        if (s.sizes[k] > 1) add(s.sizes[k], s.strides[k] * elem_size);
    if (elem_size > 1) add(elem_size, 1);

    uint64_t run_bytes = 1;
    if (n > 0 && dims[n - 1].stride == 1) run_bytes = dims[--n].size;

    uint64_t mask = align_mask | run_bytes | (skew ? 0 : s.offset * elem_size);
    for (int k = 0; k < n; ++k) mask |= dims[k].stride;
    const uint32_t u = pow2_factor(mask, max_unit);

    out->offset = s.offset * elem_size / u;
    if (skew) *skew = s.offset * elem_size % u;
    out->total = len * elem_size / u;
    out->run = run_bytes / u;
    out->ndim = n;
    for (int k = 0; k < n; ++k) dims[k].stride /= u;
    *unit = u;
    return true;
}

// Bytes of lines from which the strided side of a copy unit by unit is streamed: from there on the lines do not stay in
// the Infinity Cache between one pass over them and the next.
constexpr uint64_t kStreamUnitsFromBytes = 92ull << 20;

bool streams_units(const CanonSlice& c, uint32_t unit) {
    if (c.ndim == 0 || c.run != 1) return false;
    const uint64_t step = c.dims[c.ndim - 1].stride;
    for (int k = 0; k < c.ndim; ++k)
        if (c.dims[k].stride < step) return false;  // its units lie between the innermost dimension's: shared lines
    const uint64_t line = 128 / unit;
    return c.total >= kStreamUnitsFromBytes / unit / (step < line ? step : line);
}

bool gathers_units(const CanonSlice& c, uint32_t unit) {
    if (c.ndim < 2 || c.run != 1 || c.total < (6ull << 20) / unit) return false;
    const CanonDim& last = c.dims[c.ndim - 1];
    if (last.size < 4 || last.size > 7) return false;
    for (int k = 0; k < c.ndim - 1; ++k)
        if (c.dims[k].stride < last.stride) return true;
    return false;
}

bool same_shape(const CanonSlice& a, const CanonSlice& b) {
    if (a.ndim != b.ndim || a.run != b.run || a.total != b.total) return false;
    for (int k = 0; k < a.ndim; ++k)
        if (a.dims[k].size != b.dims[k].size || a.dims[k].stride != b.dims[k].stride) return false;
    return true;
}

}  // namespace mhip
