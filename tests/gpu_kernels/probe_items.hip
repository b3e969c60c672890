// Test-only entry: the work items of a probe batch (spec_tiles.h), on the host.
// Built into tests/_build/libhvx_testkernels.so.
#include <hip/hip_runtime.h>

#include "../../hellovulkan_amd/csrc/spec_tiles.h"

// out_faces, mips: n of each; items: room for cap x (probe, mip, first, count).
// Returns the items made (at most cap are written), the variant in *one.
extern "C" uint32_t hvxt_probe_items(const uint32_t* out_faces, const uint32_t* mips, uint32_t n, uint32_t samples,
                                     uint32_t texels, uint32_t slots, uint32_t* items, uint32_t cap,
                                     uint32_t* xcd_begin, uint32_t* one) {
    std::vector<hvx::ProbeJob> jobs(n);
    for (uint32_t p = 0; p < n; ++p) {
        jobs[p] = hvx::ProbeJob{};
        jobs[p].So = out_faces[p];
        jobs[p].mips = mips[p];
        jobs[p].n = samples;
    }
    std::vector<hvx::ProbeItem> made;
    *one = hvx::make_probe_items(jobs.data(), n, texels, slots, made, xcd_begin) ? 1u : 0u;
    static_assert(sizeof(hvx::ProbeItem) == 16, "four words an item");
    std::copy(made.begin(), made.begin() + std::min<size_t>(made.size(), cap), reinterpret_cast<hvx::ProbeItem*>(items));
    return (uint32_t)made.size();
}
