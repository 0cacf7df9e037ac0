// cellsort_device.hpp - the counting half of the cell sort (cellsort.hip), for
// the kernels that make the keys (one system, or a batch of them).
#pragma once

#include "common.hpp"

namespace cmag {

// an entry of the sort: the particle number, below the bucket of its row in
// the sub-cell walk order (0 without it)
constexpr int ENTRY_BUCKET_SHIFT = 27;
constexpr uint32_t ENTRY_INDEX = (1u << ENTRY_BUCKET_SHIFT) - 1u;

// Count particle i (cell key) into its cell and note its place among the
// cell's arrivals.  Arrival order depends on the order the atomics land in and
// is sorted out by the reorder, so it need only be a numbering.
// Neighbouring particles often share a cell: only the first lane of each run
// of equal keys adds, the run's length.
// Every lane of the wave calls this; valid lanes come first.
__device__ __forceinline__ void count_particle(uint32_t* __restrict__ cell_count, uint32_t* __restrict__ place,
                                               uint32_t i, uint32_t key, uint32_t bucket, bool valid) {
    const int lane = __lane_id();
    const int lanes = __popcll(__ballot(valid));
    const uint64_t upto = lane == 63 ? ~0ull : (1ull << (lane + 1)) - 1ull;
    const uint32_t prev = __shfl_up(key, 1, 64);
    const bool head = valid && (lane == 0 || prev != key);
    const uint64_t heads = __ballot(head);
    const uint64_t mine = heads & upto, later = heads & ~upto;
    const int start = mine ? 63 - __clzll((long long)mine) : 0;
    const int end = later ? __ffsll((unsigned long long)later) - 1 : lanes;
    uint32_t base = 0;
    if (head) base = atomicAdd(&cell_count[key], (uint32_t)(end - start));
    base = __shfl(base, start, 64);
    if (valid) place[i] = (base + (uint32_t)(lane - start)) | (bucket << ENTRY_BUCKET_SHIFT);
}

}  // namespace cmag
