// Prints what the copy planner (plan.cpp) decides about a view copied unit by unit.  Input, one view per line:
//   element_size offset ndim sizes... strides...     (elements)
// Output, one line per view: unit in bytes, streams_units, gathers_units.  No GPU, no HIP headers.
#include <cstdio>
#include <iostream>

#include "../../monarch_amd/csrc/mhip_internal.h"

int main() {
    uint32_t elem_size, ndim;
    uint64_t offset, sizes[MHIP_MAX_DIMS], strides[MHIP_MAX_DIMS];
    while (std::cin >> elem_size >> offset >> ndim && ndim <= MHIP_MAX_DIMS) {
        for (uint32_t k = 0; k < ndim; ++k) std::cin >> sizes[k];
        for (uint32_t k = 0; k < ndim; ++k) std::cin >> strides[k];
        const mhip_slice_t s{offset, ndim, sizes, strides};
        mhip::CanonSlice c;
        uint32_t unit = 0;
        if (!mhip::canonicalize(s, elem_size, 0, 16, &c, &unit)) return 1;
        std::printf("%u %d %d\n", unit, mhip::streams_units(c, unit), mhip::gathers_units(c, unit));
    }
    return 0;
}
