// cellsort.hip - particles into cell order by counting (gfx950).
//
// A step's keys are cells, its values the particle numbers 0..n-1, so the
// stable sort_by_key of the reference (fluidSystem.cu:94-99) followed by its
// reorder and cell ranges (fluid_kernel.cu:50-97) is "particles by cell, and
// within a cell by number".  Four launches make it, however many bits the keys
// have:
//   hash      key of every particle; counts per cell by atomics, which also
//             hand out places within the cell
//   offsets   first[c] = particles in cells < c, and the cellStart array.  A
//             workgroup takes one tile of cells; in a grid of a few tiles it sums
//             the counts before its own itself, in a larger one it sums the
//             tile totals that a launch in front made: nothing waits on another
//             workgroup
//   place     perm[first[cell] + place] = particle
//   reorder   a row finds its particle's rank among its cell's (a handful of)
//             entries, which undoes the atomics' arrival order: hash, index and
//             the sorted rows come out as the stable sort gives them, on every
//             run.  DamBreak systems rank their rows in the sub-cell walk
//             order in the same loop and write that copy too.  The counts of
//             the cells it meets go back to zero for the next step
//
// What bounds them: launches up to some 100,000 particles (a captured launch
// costs 4 to 5 us whatever it does; a three-digit radix sort with the reorder
// and the offset scan was 15 of them: a 200,000-particle channel's two steps
// went from 136 to 90 us), memory above (16M dam break, 20.07M rows, 2^24 cells:
// hash 192 us, offsets 17 + 53, place 91, reorder of both orders 588 us, 2.6 GB;
// radix sort, reorder, offset scan and the separate walk-order copy 1,320 us).
// Counts per tile by atomics in the hash kernel instead of their own launch
// met on too few addresses: hash 460 us at 16M, 793 us at 1.6M.  The radix sort
// of sort.hip remains for callers' own keys (cmag_sort_by_key).
#include <hip/hip_runtime.h>

#include "cellsort_device.hpp"
#include "integrate_device.hpp"
#include "kernels.hpp"
#include "scan_device.hpp"
#include "step_state.hpp"

namespace cmag {

constexpr int OFF_ITEMS = 16;  // cells per thread: four 16-byte words, one occupancy half-word
static_assert(WALK_MAX_PARTICLES == 1u << ENTRY_BUCKET_SHIFT, "entries hold the particle number below the bucket");
// A grid of up to OFF_SMALL_TILES tiles of 1024 threads reads the counts before
// its tile itself (at most 28 16-byte loads a thread): one launch of 4.5 us at
// 2^12 cells, 7.3 at 2^14, 9.0 at 2^16 and 10.8 at 2^17, against two of 4.5 us at
// each.  It saves eager steps a launch of the host's (17,500-particle channel,
// 2^14 cells, one update 23.5 against 26.9 us; 2,240 particles, 10 captured steps
// 117 against 120 us) and costs captured steps of large grids time (17,000
// particles, 10 steps by themselves: 2^13 cells 416 against 419 us, 2^14 401 / 382,
// 2^16 420 / 386, 2^17 437 / 386; the 200-step gradient on 2^17 cells 23.7 / 22.0 ms)
constexpr int OFF_NT_SMALL = 1024, OFF_NT = 256;
constexpr uint32_t OFF_SMALL_TILES = 8;
// tile totals a workgroup of a larger grid sums itself (at most 32 a thread,
// from L2); beyond that they are scanned first
constexpr uint32_t OFF_TILES_DIRECT = 8192;

constexpr size_t off_tile(int nt) { return (size_t)nt * OFF_ITEMS; }
static bool small_grid(size_t cells) { return cells <= OFF_SMALL_TILES * off_tile(OFF_NT_SMALL); }
static uint32_t cell_tiles(size_t cells) { return (uint32_t)((cells + off_tile(OFF_NT) - 1) / off_tile(OFF_NT)); }

// keys of one system; Peristalsis walls move to the boundary configuration's
// height first when this step's state record says so (configureBoundaryD,
// PeristalsisKernel.cu:144-171).  The record itself is advanced by the offset
// kernel: every thread here works from its own advanced copy.
template <bool BUCKET>
__global__ __launch_bounds__(256) void hash_count_kernel(const cmag_params P, float4* __restrict__ pos,
                                                         const StepState* __restrict__ state,
                                                         uint32_t* __restrict__ key, uint32_t* __restrict__ place,
                                                         uint32_t* __restrict__ cell_count, uint32_t n) {
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    uint32_t k = 0, bucket = 0;
    if (valid) {
        float4 p = pos[i];
        if (state) {
            StepState st = *state;
            advance_step_state(P, st);
            if (st.configure_now && (p.w > 0.0f || p.w < 0.0f)) {
                p = make_float4(p.x, wall_y(P, p.x, p.w, st.configure_height, 0.0f), p.z, p.w);
                pos[i] = p;
            }
        }
        const Cell c = grid_pos(P, p.x, p.y, p.z);
        k = grid_hash(P, c.x, c.y, c.z);
        key[i] = k;
        if (BUCKET) bucket = (uint32_t)(p.w != CMAG_DB_FLUID ? X_SUBS : x_sub(P, p.x));
    }
    count_particle(cell_count, place, i, k, bucket, valid);
}

__device__ __forceinline__ uint32_t sum4(const uint4 x) { return (x.x + x.y) + (x.z + x.w); }

// total of each tile of cells
__global__ __launch_bounds__(OFF_NT) void cell_totals_kernel(const uint32_t* __restrict__ cell_count, size_t cells,
                                                             uint32_t* __restrict__ total) {
    __shared__ uint32_t lds[OFF_NT / 64];
    const size_t c0 = (size_t)blockIdx.x * off_tile(OFF_NT);
    uint32_t sum = 0;
    if (c0 + off_tile(OFF_NT) <= cells) {
        const uint4* w = reinterpret_cast<const uint4*>(cell_count + c0);
#pragma unroll
        for (int q = 0; q < OFF_ITEMS / 4; ++q) sum += sum4(w[q * OFF_NT + threadIdx.x]);
    } else {
        for (size_t c = c0 + threadIdx.x; c < cells; c += OFF_NT) sum += cell_count[c];
    }
    uint32_t tot;
    (void)block_exclusive_scan<OFF_NT>(sum, lds, &tot);
    if (threadIdx.x == 0) total[blockIdx.x] = tot;
}

// One tile of cells per workgroup: exclusive scan of the tile's counts from its
// base: carry[tile], or the sum of the totals of the tiles before it, or
// (neither given) of their counts.  Also advances the m state records (params:
// one block per record), and with pre keeps the sub-cell counts of empty cells
// at zero: occ holds one bit per cell, set where the last step left counts, so
// only cells that became empty are cleared (clearing all is 16 B a cell, 48 us
// at 2^24 cells).
template <int NT>
__global__ __launch_bounds__(NT) void cell_offsets_kernel(const uint32_t* __restrict__ cell_count,
                                                          const uint32_t* __restrict__ total,
                                                          const uint32_t* __restrict__ carry, size_t cells, uint32_t n,
                                                          uint32_t* __restrict__ first,
                                                          uint32_t* __restrict__ cellStart, uint4* __restrict__ pre,
                                                          uint16_t* __restrict__ occ,
                                                          const cmag_params* __restrict__ params, const cmag_params P0,
                                                          StepState* __restrict__ state, uint32_t m) {
    __shared__ uint32_t lds[NT / 64];
    const uint32_t tile = blockIdx.x;
    if (state) {
        for (uint32_t k = tile * NT + threadIdx.x; k < m; k += gridDim.x * NT) {
            StepState s = state[k];
            advance_step_state(params ? params[k] : P0, s);
            state[k] = s;
        }
    }
    uint32_t base = 0;
    if (carry) {
        base = carry[tile];
    } else {
        uint32_t sum = 0;
        if (total) {
            for (uint32_t t = threadIdx.x; t < tile; t += NT) sum += total[t];
        } else {
            // whole tiles in front: whole 16-byte words
            const uint4* w = reinterpret_cast<const uint4*>(cell_count);
            const size_t words = (size_t)tile * off_tile(NT) / 4;
#pragma unroll 14
            for (size_t q = threadIdx.x; q < words; q += NT) sum += sum4(w[q]);
        }
        (void)block_exclusive_scan<NT>(sum, lds, &base);
    }
    const size_t c0 = (size_t)tile * off_tile(NT) + (size_t)threadIdx.x * OFF_ITEMS;
    const bool whole = c0 + OFF_ITEMS <= cells;
    uint32_t v[OFF_ITEMS];
    if (whole) {
#pragma unroll
        for (int q = 0; q < OFF_ITEMS / 4; ++q) {
            const uint4 x = reinterpret_cast<const uint4*>(cell_count + c0)[q];
            v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < OFF_ITEMS; ++k) v[k] = c0 + k < cells ? cell_count[c0 + k] : 0u;
    }
    uint32_t sum = 0, filled = 0;
#pragma unroll
    for (int k = 0; k < OFF_ITEMS; ++k) {
        sum += v[k];
        filled |= (v[k] != 0u ? 1u : 0u) << k;
    }
    uint32_t tot;
    uint32_t run = base + block_exclusive_scan<NT>(sum, lds, &tot);
    uint32_t o[OFF_ITEMS];
#pragma unroll
    for (int k = 0; k < OFF_ITEMS; ++k) {
        o[k] = run;
        run += v[k];
    }
    if (whole) {
#pragma unroll
        for (int q = 0; q < OFF_ITEMS / 4; ++q) {
            const uint32_t* a = o + 4 * q;
            const uint32_t* b = v + 4 * q;
            reinterpret_cast<uint4*>(first + c0)[q] = make_uint4(a[0], a[1], a[2], a[3]);
            reinterpret_cast<uint4*>(cellStart + c0)[q] =
                make_uint4(b[0] ? a[0] : CMAG_CELL_EMPTY, b[1] ? a[1] : CMAG_CELL_EMPTY,
                           b[2] ? a[2] : CMAG_CELL_EMPTY, b[3] ? a[3] : CMAG_CELL_EMPTY);
        }
    } else {
#pragma unroll
        for (int k = 0; k < OFF_ITEMS; ++k)
            if (c0 + k < cells) {
                first[c0 + k] = o[k];
                cellStart[c0 + k] = v[k] ? o[k] : CMAG_CELL_EMPTY;
            }
    }
    if (tile == gridDim.x - 1 && threadIdx.x == 0) first[cells] = n;
    if (pre && c0 < cells) {
        uint16_t* half = occ + c0 / OFF_ITEMS;
        uint32_t gone = *half & ~filled;
        while (gone) {
            const uint32_t k = (uint32_t)__ffs((int)gone) - 1u;
            gone &= gone - 1u;
            pre[c0 + k] = make_uint4(0u, 0u, 0u, 0u);
        }
        *half = (uint16_t)filled;
    }
}

// the particles at their places
__global__ __launch_bounds__(256) void place_kernel(const uint32_t* __restrict__ key,
                                                    const uint32_t* __restrict__ place,
                                                    const uint32_t* __restrict__ first, uint32_t* __restrict__ perm,
                                                    uint32_t n, uint32_t index_mask) {
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = place[i];
    const uint32_t at = first[key[i]] + (p & index_mask);
    if (at < n) perm[at] = i | (p & ~index_mask);
}

// Row r of the arrival order goes to its place in the reference order (and in
// the sub-cell walk order: SUB).  An entry compares by bucket, then number, so
// both ranks come from one pass over the cell's entries; `bytes` counts
// entries of eighths <= t in byte t, eight at a time, for the cell's running
// counts.  O(cell size) per row: 1 entry in the 2-D cells of one spacing, ~18 in
// the 3-D cells of 2h; the loads are 16 bytes and hit the row's own cache line.
template <bool SUB>
__global__ __launch_bounds__(256) void reorder_cells_kernel(
    const uint32_t* __restrict__ perm, const uint32_t* __restrict__ key, const uint32_t* __restrict__ first,
    uint32_t* __restrict__ cell_count, uint32_t n, const float4* __restrict__ pos, const float4* __restrict__ vel, uint32_t* __restrict__ hash,
    uint32_t* __restrict__ index, uint32_t* __restrict__ cellEnd, float4* __restrict__ sortedPos,
    float4* __restrict__ sortedVel, uint4* __restrict__ pre, float4* __restrict__ posW, float4* __restrict__ velW,
    uint32_t* __restrict__ indexW, uint32_t* __restrict__ w2r) {
    const uint32_t r = xcd_block() * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const uint32_t e = perm[r];
    const uint32_t i = SUB ? e & ENTRY_INDEX : e;
    if (i >= n) return;  // inconsistent counts only
    const float4 p = pos[i], u = vel[i];
    const uint32_t c = key[i];
    const uint32_t a = first[c], b = min(first[c + 1], n);
    uint32_t before = 0, below = 0;  // rank in the reference order, in the walk order
    uint32_t cnt[X_SUBS] = {};
    for (uint32_t k4 = a & ~3u; k4 < b;) {
        uint64_t bytes = 0;
        for (int q = 0; q < 8 && k4 < b; ++q, k4 += 4u) {
            const uint4 v = *reinterpret_cast<const uint4*>(perm + k4);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool in = k4 + (uint32_t)j >= a && k4 + (uint32_t)j < b;
                if (SUB) {
                    before += (in && (w[j] & ENTRY_INDEX) < i) ? 1u : 0u;
                    below += (in && w[j] < e) ? 1u : 0u;
                    const uint32_t bk = w[j] >> ENTRY_BUCKET_SHIFT;
                    bytes += in && bk < (uint32_t)X_SUBS ? 0x0101010101010101ull << (8u * bk) : 0ull;
                } else {
                    before += (in && w[j] < i) ? 1u : 0u;
                }
            }
        }
        if (SUB) {
#pragma unroll
            for (int t = 0; t < X_SUBS; ++t) cnt[t] += (uint32_t)(bytes >> (8 * t)) & 0xffu;
        }
    }
    const uint32_t row = a + before;
    if (row >= n) return;  // inconsistent counts only
    hash[row] = c;
    index[row] = i;
    sortedPos[row] = p;
    sortedVel[row] = u;
    if (before == 0) {
        cellEnd[c] = b;
        cell_count[c] = 0u;
    }
    if (SUB) {
        const uint32_t w = a + below;
        if (w >= n) return;
        // the walk tells walls from fluid by the sign bit of w (the density
        // pass stores -rho in fluid rows): every non-fluid row, whatever its
        // type code (-0.0 and negative codes included), gets the tag +0
        posW[w] = make_float4(p.x, p.y, p.z, p.w != CMAG_DB_FLUID ? 0.0f : p.w);
        velW[w] = u;
        indexW[w] = i;
        w2r[w] = row;
        // 16-bit counts, capped: a cell of more than 65,535 rows (no physical
        // state has one) keeps its runs inside the cell
        if (below == 0) {
            uint32_t h[X_SUBS];
#pragma unroll
            for (int t = 0; t < X_SUBS; ++t) h[t] = min(cnt[t], 0xffffu);
            pre[c] = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
        }
    }
}

// ---- buffers ------------------------------------------------------------------
int CellSort::alloc(size_t cells_, uint32_t n_, hipStream_t s) {
    cells = cells_;
    n = n_;
    // one allocation, its parts on 256-byte boundaries (perm is read four entries at a time)
    auto part = [](size_t words) { return (sizeof(uint32_t) * (words ? words : 1) + 255) & ~(size_t)255; };
    const uint32_t tiles = cell_tiles(cells);
    const bool scanned = tiles > OFF_TILES_DIRECT;
    const size_t sizes[] = {part(n), part(n), part(n), part(cells), part(small_grid(cells) ? 0 : tiles),
                            part(scanned ? tiles : 0), part(scanned ? scan_levels_words(tiles) + 1 : 0)};
    uint32_t** bufs[] = {&key, &place, &perm, &cell_count, &total, &carry, &scan_ws};
    size_t bytes = 0;
    for (size_t z : sizes) bytes += z;
    CMAG_HIP_TRY(hipMalloc(&arena, bytes));
    char* at = static_cast<char*>(arena);
    for (size_t k = 0; k < sizeof(sizes) / sizeof(sizes[0]); at += sizes[k], ++k)
        *bufs[k] = reinterpret_cast<uint32_t*>(at);
    if (!scanned) carry = nullptr;
    return clear(s);
}

int CellSort::alloc_walk(hipStream_t s) {
    if (pre) return CMAG_OK;
    // pre, then occ, in one allocation that starts as zeros
    const size_t counts = sizeof(uint32_t) * 4 * cells, halves = (cells + OFF_ITEMS - 1) / OFF_ITEMS;
    const size_t bytes = counts + sizeof(uint16_t) * halves;
    CMAG_HIP_TRY(hipMalloc((void**)&pre, bytes));
    occ = reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(pre) + counts);
    CMAG_HIP_TRY(hipMemsetAsync(pre, 0, bytes, s));
    return CMAG_OK;
}

void CellSort::release() {
    void* bufs[] = {arena, pre};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
}

int CellSort::clear(hipStream_t s) {
    CMAG_TRY(launch_fill_u32(cell_count, 0u, cells, s));
    counts_clean = true;
    return CMAG_OK;
}

int CellSort::begin(hipStream_t s) {
    CMAG_TRY(ready(s));
    counts_clean = false;
    return CMAG_OK;
}

int CellSort::hash(const cmag_params& P, float* pos, const StepState* state, bool walk, hipStream_t s) {
    CMAG_TRY(begin(s));
    if (n == 0) return CMAG_OK;
    const dim3 g(div_up(n, 256)), b(256);
    float4* p4 = reinterpret_cast<float4*>(pos);
    if (walk)
        hipLaunchKernelGGL(hash_count_kernel<true>, g, b, 0, s, P, p4, state, key, place, cell_count, n);
    else
        hipLaunchKernelGGL(hash_count_kernel<false>, g, b, 0, s, P, p4, state, key, place, cell_count, n);
    return check_launch("hash_count_kernel");
}

int CellSort::offsets(uint32_t* first, uint32_t* cellStart, bool walk, const cmag_params* params,
                      const cmag_params& P0, StepState* state, uint32_t m, hipStream_t s) {
    uint4* pre4 = walk ? reinterpret_cast<uint4*>(pre) : nullptr;
    if (small_grid(cells)) {
        const uint32_t tiles = (uint32_t)((cells + off_tile(OFF_NT_SMALL) - 1) / off_tile(OFF_NT_SMALL));
        hipLaunchKernelGGL(cell_offsets_kernel<OFF_NT_SMALL>, dim3(tiles), dim3(OFF_NT_SMALL), 0, s, cell_count,
                           nullptr, nullptr, cells, n, first, cellStart, pre4, occ, params, P0, state, m);
    } else {
        const uint32_t tiles = cell_tiles(cells);
        hipLaunchKernelGGL(cell_totals_kernel, dim3(tiles), dim3(OFF_NT), 0, s, cell_count, cells, total);
        CMAG_TRY(check_launch("cell_totals_kernel"));
        if (carry) CMAG_TRY(exclusive_scan_u32(total, carry, tiles, scan_ws, s));
        hipLaunchKernelGGL(cell_offsets_kernel<OFF_NT>, dim3(tiles), dim3(OFF_NT), 0, s, cell_count, total, carry,
                           cells, n, first, cellStart, pre4, occ, params, P0, state, m);
    }
    CMAG_TRY(check_launch("cell_offsets_kernel"));
    if (n) {
        hipLaunchKernelGGL(place_kernel, dim3(div_up(n, 256)), dim3(256), 0, s, key, place, first, perm, n,
                           walk ? ENTRY_INDEX : 0xffffffffu);
        CMAG_TRY(check_launch("place_kernel"));
    }
    return CMAG_OK;
}

int CellSort::reorder(const float* pos, const float* vel, const uint32_t* first, uint32_t* hash_out, uint32_t* index,
                      uint32_t* cellEnd, float* sortedPos, float* sortedVel, const WalkRows* walk, hipStream_t s) {
    if (n == 0) {
        counts_clean = true;
        return CMAG_OK;
    }
    auto f4 = [](float* q) { return reinterpret_cast<float4*>(q); };
    auto c4 = [](const float* q) { return reinterpret_cast<const float4*>(q); };
    const dim3 g(div_up(n, 256)), b(256);
    if (walk)
        hipLaunchKernelGGL(reorder_cells_kernel<true>, g, b, 0, s, perm, key, first, cell_count, n, c4(pos), c4(vel), hash_out,
                           index, cellEnd, f4(sortedPos), f4(sortedVel), reinterpret_cast<uint4*>(pre), f4(walk->pos),
                           f4(walk->vel), walk->index, walk->to_ref);
    else
        hipLaunchKernelGGL(reorder_cells_kernel<false>, g, b, 0, s, perm, key, first, cell_count, n, c4(pos), c4(vel), hash_out,
                           index, cellEnd, f4(sortedPos), f4(sortedVel), nullptr, nullptr, nullptr, nullptr, nullptr);
    CMAG_TRY(check_launch("reorder_cells_kernel"));
    counts_clean = true;
    return CMAG_OK;
}

}  // namespace cmag
