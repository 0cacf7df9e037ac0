// kernels.hpp - launchers shared between the translation units of libcmag_hip.so.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "cmag_hip.h"

namespace cmag {

struct StepState;

int launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t s);
// the demos' colour buffer of a system's kind (render.hip)
int launch_fill_colors(const cmag_params& P, const float* pos4, float* color4, uint32_t n, hipStream_t s);
int launch_copy_u32(uint32_t* dst, const uint32_t* src, size_t n, hipStream_t s);
int launch_calc_hash(const cmag_params& P, const float* pos4, uint32_t* hash, uint32_t* index,
                     uint32_t n, hipStream_t s);
int launch_reorder(uint32_t* cellStart, uint32_t* cellEnd, float* sortedPos, float* sortedVel,
                   const uint32_t* hash, const uint32_t* index, const float* oldPos,
                   const float* oldVel, uint32_t n, uint32_t numCells, hipStream_t s);

// out = exclusive_scan(in) (in place allowed); ws holds scan_levels_words(len) words
size_t scan_levels_words(size_t len);
int exclusive_scan_u32(const uint32_t* in, uint32_t* out, size_t len, uint32_t* ws, hipStream_t s);
// particles of a system in sub-cell walk order: an entry of its sort holds the particle number in 27 bits
constexpr uint32_t WALK_MAX_PARTICLES = 1u << 27;

// the sub-cell walk order's copy of the sorted rows (DamBreak): pos, vel and
// particle number of every row, and its row in the reference order
struct WalkRows {
    float *pos, *vel;
    uint32_t *index, *to_ref;
};

// A step's particles into cell order by counting (cellsort.hip): hash(), then
// offsets(), then reorder(), on one stream.  The counters are zero between
// sorts.  first[c] = number of particles in cells < c, first[C] = n, is what the
// neighbour walkers read: a run of cells with consecutive keys is one range
// [first[k0], first[k1 + 1]) without any empty-cell test.
struct CellSort {
    size_t cells = 0;
    uint32_t n = 0;
    void* arena = nullptr;
    uint32_t *key = nullptr, *place = nullptr, *perm = nullptr;  // per particle; perm: per row
    uint32_t *cell_count = nullptr, *total = nullptr, *carry = nullptr, *scan_ws = nullptr;
    uint16_t* occ = nullptr;  // cells that hold sub-cell counts, one bit each
    uint32_t* pre = nullptr;  // the sub-cell walk's running counts, 16 B a cell
    bool counts_clean = false;

    int alloc(size_t cells, uint32_t n, hipStream_t s);
    int alloc_walk(hipStream_t s);
    void release();
    int clear(hipStream_t s);
    // zero counters: they are left so by every sort, one that ended early leaves them to be cleared
    int ready(hipStream_t s) { return counts_clean ? CMAG_OK : clear(s); }
    // call in front of a kernel that counts
    int begin(hipStream_t s);
    // keys and counts; state: the Peristalsis time record (walls are configured from it)
    int hash(const cmag_params& P, float* pos, const StepState* state, bool walk, hipStream_t s);
    // also advances the m records of state by one step (params: a block per record, or P0)
    int offsets(uint32_t* first, uint32_t* cellStart, bool walk, const cmag_params* params, const cmag_params& P0,
                StepState* state, uint32_t m, hipStream_t s);
    int reorder(const float* pos, const float* vel, const uint32_t* first, uint32_t* hash, uint32_t* index,
                uint32_t* cellEnd, float* sortedPos, float* sortedVel, const WalkRows* walk, hipStream_t s);
};

// stable LSD radix sort.  Sorts (keys, vals) using (alt_keys, alt_vals) as the
// ping-pong buffers; *result_in_alt tells where the sorted pair ended up.
size_t radix_sort_workspace_bytes(uint32_t n);
int radix_sort_pairs(uint32_t* keys, uint32_t* vals, uint32_t* alt_keys, uint32_t* alt_vals,
                     uint32_t n, int key_bits, void* workspace, size_t workspace_bytes,
                     bool* result_in_alt, hipStream_t s);

// neighbour passes.  cellFirst (optional, from CellSort) selects the
// compact-offset walker; without it the reference cellStart/cellEnd are walked.
// With cellFirst the rows of sortedPos are followed by two of padding, and the
// channels' density pass leaves pair values (2 floats a row) and, with
// row_masks, in-range masks (ROW_MASK_ROWS words a row) for the force pass.
constexpr int ROW_MASK_ROWS = 7;  // stencils of up to 3 cells a side
__host__ __device__ inline bool row_masks_apply(const cmag_params& P) {
    return P.dim == 2 && P.system != CMAG_SYS_DAMBREAK && P.hash_order == CMAG_HASH_LINEAR &&
           2 * P.cellcount + 1 <= ROW_MASK_ROWS;
}
// Dam-break targets are shared between four lanes up to this many rows.
// Two steps of a 3-D dam break by itself / of four at once on their own streams,
// a lane to a target against four: 25,168 rows 395 / 104 us against 169 / 56,
// 54,508: 412 / 115 against 260 / 95, 82,188: 399 / 126 against 261 / 120,
// 117,260: 414 / 136 against 310 / 159 (four at once fill the chip either way,
// and a shared target costs more work); 160,492: 466 / 161 against 389 / 223.
// The stage launchers over a caller's arrays: 54,508 rows 214 against 137 us,
// 82,188: 210 against 186, 117,260: 223 against 237.
constexpr uint32_t SHARED_TARGETS = 3u << 15;
// where a step's force pass integrates its targets (in place, at their particle
// numbers); pos null: it only writes the accelerations
struct StepArrays {
    float4 *pos = nullptr, *vel = nullptr, *velLF = nullptr;
    const StepState* state = nullptr;  // Peristalsis: the time record(s)
};
int launch_density(const cmag_params& P, float* measures, const float* sortedPos,
                   const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n, hipStream_t s,
                   const uint32_t* cellFirst = nullptr, float* pairs = nullptr, uint32_t* row_masks = nullptr);
// sub-cell walk order (DamBreak; the copies and pre from CellSort): density and
// force over it; density writes the reference-order measures through w2r and
// leaves, for the force pass, -rho (fluid rows) in posW.w and p / rho^2 times the
// pair terms' common factor in velW.w; keys: the sorted cell keys
// masks (optional, 2 * MASK_ROWS words per particle): density leaves the
// in-range masks of staged blocks there and force reads them
int launch_density_sub(const cmag_params& P, float* measures, const uint32_t* keys, const uint32_t* w2r, float* posW,
                       float* velW, const uint32_t* cellFirst, const uint32_t* pre, uint32_t n, hipStream_t s,
                       uint32_t* masks = nullptr);
int launch_force_sub(const cmag_params& P, float* acc, const float* posW, const float* velW,
                     const uint32_t* indexW, const uint32_t* keys, const uint32_t* cellFirst, const uint32_t* pre,
                     uint32_t n, hipStream_t s, const uint32_t* masks = nullptr, const StepArrays& step = {});
int launch_force(const cmag_params& P, float* acc, const float* measures, const float* sortedPos,
                 const float* sortedVel, const uint32_t* index, const uint32_t* cellStart,
                 const uint32_t* cellEnd, uint32_t n, hipStream_t s,
                 const uint32_t* cellFirst = nullptr, const float* pairs = nullptr,
                 const uint32_t* row_masks = nullptr, const StepArrays& step = {});
int launch_peristalsis_forces(const cmag_params& P, float* viscF, float* presF, const float* measures,
                              const float* sortedPos, const float* sortedVel, const uint32_t* index,
                              const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n,
                              hipStream_t s, const uint32_t* cellFirst = nullptr, const float* pairs = nullptr,
                              const uint32_t* row_masks = nullptr, const StepArrays& step = {});
int launch_pressure_force(const cmag_params& P, float* presF, const float* measures,
                          const float* sortedPos, const uint32_t* index, const uint32_t* cellStart,
                          const uint32_t* cellEnd, uint32_t n, hipStream_t s);
int launch_viscous_force(const cmag_params& P, float* viscF, const float* measures,
                         const float* sortedPos, const float* sortedVel, const uint32_t* index,
                         const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n,
                         hipStream_t s);
// with a state record (step_state.hpp) the wave time and configuration phase
// come from it on the device, else from wave_time and P
int launch_integrate(const cmag_params& P, float* pos, float* vel, float* velLF, const float* acc,
                     const float* presF, float wave_time, uint32_t n, hipStream_t s,
                     const StepState* state = nullptr);
int launch_configure_boundary(const cmag_params& P, float* pos, float wave_height, uint32_t n,
                              hipStream_t s);
int launch_shift_right_boundary(const cmag_params& P, float* pos, uint32_t n, hipStream_t s);
int launch_remove_right_boundary(const cmag_params& P, float* pos, uint32_t n, hipStream_t s);

// adjoints of the Poiseuille step (adjoint.hip)
int launch_integrate_vjp(const cmag_params& P, const float* pos, float* gpos, float* gvel, float* gvelLF,
                         float* gacc, double* ggrav, uint32_t n, hipStream_t s);
// integrate_vjp by sorted row: gaccS, and terms (2 floats a row) for launch_force_vjp
int launch_step_vjp(const cmag_params& P, const float* sortedPos, const float* measures, const uint32_t* index,
                    float* gpos, float* gvel, float* gvelLF, float* gaccS, float* terms, double* ggrav, uint32_t n,
                    hipStream_t s);
int launch_force_vjp(const cmag_params& P, float* gposS, float* gvelS, float* grho, float* gmu, double* gmu_acc,
                     const float* gaccS, const float* measures, const float* sortedPos, const float* sortedVel,
                     const uint32_t* cellStart, const uint32_t* cellEnd, const uint32_t* cellFirst, uint32_t n,
                     const float* terms, hipStream_t s);
int launch_density_vjp(const cmag_params& P, float* gposS, const float* grho, const float* sortedPos,
                       const uint32_t* cellStart, const uint32_t* cellEnd, const uint32_t* cellFirst, uint32_t n,
                       const uint32_t* index, const float* gvelS, float* gpos, float* gvelLF, hipStream_t s);

}  // namespace cmag
