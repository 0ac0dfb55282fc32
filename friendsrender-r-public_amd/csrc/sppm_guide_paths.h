// sppm_guide_paths.h -- buffers of a guided render per path and per photon.
#pragma once
#include <stddef.h>

namespace sppm {

// All four are there or none: sppm_guide_set and sppm_begin both fill them,
// and a pass writes through each of them.
struct GuidePaths {
    int* cell = nullptr;               // emission cell per path, 2 x paths (block = step parity)
    float* ratio = nullptr;            // q / p_plain per path, like cell
    unsigned long long* dep = nullptr; // deposited luminance per flattened photon (guide_fix)
    // the pass's photon offsets and stored count (paths + 1), copied by the
    // build for the gather's deposits and the training records, which run
    // while the next pass stages its photons
    int* off = nullptr;
    bool whole() const { return cell && ratio && dep && off; }
};

// drop(void*) frees one buffer.
template <class Drop>
void guide_paths_free(GuidePaths& p, Drop&& drop) {
    for (void* q : {(void*)p.cell, (void*)p.ratio, (void*)p.dep, (void*)p.off})
        if (q) drop(q);
    p = GuidePaths();
}
// get(void**, bytes) allocates one buffer, 0 on success.  Buffers that are
// there are kept (the caller frees them when the sizes change); on a failure
// none is left.
template <class Get, class Drop>
int guide_paths_alloc(GuidePaths& p, size_t paths, size_t photons, Get&& get, Drop&& drop) {
    if (p.whole()) return 0;
    guide_paths_free(p, drop);
    int rc;
    if ((rc = get((void**)&p.cell, 2 * paths * sizeof *p.cell)) ||
        (rc = get((void**)&p.ratio, 2 * paths * sizeof *p.ratio)) ||
        (rc = get((void**)&p.dep, photons * sizeof *p.dep)) || (rc = get((void**)&p.off, (paths + 1) * sizeof *p.off))) {
        guide_paths_free(p, drop);
        return rc;
    }
    return 0;
}

}  // namespace sppm
