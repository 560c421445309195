/* Prints the kernels that a pack or an unpack launches, without a GPU: this program's hipLaunchKernel takes the place of the
 * runtime's, records a launch and starts nothing.  Input, one view per line:
 *   pack element_size offset ndim sizes... strides...     (pack 1 or 0; sizes in elements)
 * Output, one line per view: status, then for every kernel in the order of its first launch its workgroups and its name. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stdio.h>
#include <string.h>

#include "monarch_hip.h"

typedef struct { uint32_t x, y, z; } launch_size_t; /* dim3 */

enum { kMost = 8 };
static struct { const void* kernel; unsigned long long workgroups; } seen[kMost];
static int n_seen;

int hipLaunchKernel(const void* kernel, launch_size_t grid, launch_size_t block, void** args, size_t lds, void* stream) {
    (void)block; (void)args; (void)lds; (void)stream;
    int k = 0;
    while (k < n_seen && seen[k].kernel != kernel) ++k;
    if (k == kMost) return 1;
    if (k == n_seen) {
        seen[n_seen].kernel = kernel;
        seen[n_seen++].workgroups = 0;
    }
    seen[k].workgroups += (unsigned long long)grid.x * grid.y * grid.z;
    return 0;
}

int main(void) {
    unsigned pack, size, ndim;
    unsigned long long offset, v;
    while (scanf("%u %u %llu %u", &pack, &size, &offset, &ndim) == 4 && ndim <= MHIP_MAX_DIMS) {
        uint64_t sizes[MHIP_MAX_DIMS], strides[MHIP_MAX_DIMS];
        for (unsigned k = 0; k < 2 * ndim; ++k) {
            if (scanf("%llu", &v) != 1) return 1;
            if (k < ndim) sizes[k] = v;
            else strides[k - ndim] = v;
        }
        const mhip_slice_t s = {offset, ndim, sizes, strides};
        char* const memory = (char*)((uintptr_t)1 << 40); /* addresses that nothing reads */
        char* const packed = (char*)((uintptr_t)1 << 45);
        n_seen = 0;
        const int rc = pack ? mhip_slice_pack(packed, memory, &s, size, NULL) : mhip_slice_unpack(memory, packed, &s, size, NULL);
        printf("%d", rc);
        for (int k = 0; k < n_seen; ++k) {
            Dl_info info;
            printf(" %llu %s", seen[k].workgroups, dladdr(seen[k].kernel, &info) && info.dli_sname ? info.dli_sname : "?");
        }
        printf("\n");
    }
    return 0;
}
