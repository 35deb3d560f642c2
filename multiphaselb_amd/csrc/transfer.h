// Large field transfers (transfer.hip).
#pragma once

#include <cstddef>
#include <cstdint>

struct mplb_case;

namespace mplb {

// A field large enough for the pinned ring, and the ring is there (allocated at the first such
// field); without it the caller copies through pageable memory.
bool stage_wanted(mplb_case* c, int64_t N, int comps);
// planes [comps][N] of the case's scalar type <-> host [N][comps] doubles, complete on return
int stage_transfer(mplb_case* c, void* planes, int64_t N, int comps, double* host, bool to_device);
void stage_free(mplb_case* c);

}  // namespace mplb
