// sph.hip - neighbour-pass kernels of one system and their launchers.
// The per-particle bodies live in sph_device.hpp (shared with batch.hip).
#include <type_traits>

#include "kernels.hpp"
#include "sph_device.hpp"

namespace cmag {

template <int SYS, int DIM, int HASH, typename Cells, int LANES = 1>
__global__ __launch_bounds__(256) void density_kernel(const cmag_params P, float4* __restrict__ measures,
                                                       const float4* __restrict__ sortedPos, const Cells cells,
                                                       uint32_t n, float2* __restrict__ pairs,
                                                       uint32_t* __restrict__ row_masks) {
    const uint32_t i = xcd_block() * (256 / LANES) + threadIdx.x / LANES;
    if (i >= n) return;
    density_body<SYS, DIM, HASH, LANES>(P, i, measures, sortedPos, cells, pairs, row_masks, n, threadIdx.x % LANES);
}

template <int SYS, int DIM, int HASH, typename Cells, int LANES = 1>
__global__ __launch_bounds__(256) void force_kernel(const cmag_params P, float4* __restrict__ acc,
                                                     const float4* __restrict__ measures,
                                                     const float4* __restrict__ sortedPos,
                                                     const float4* __restrict__ sortedVel,
                                                     const uint32_t* __restrict__ index, const Cells cells,
                                                     uint32_t n, const float2* __restrict__ pairs,
                                                     const uint32_t* __restrict__ row_masks, const StepArrays step) {
    __shared__ uint32_t nbl[256 / 64][NB_CAP][64];
    const uint32_t i = xcd_block() * (256 / LANES) + threadIdx.x / LANES;
    if (i >= n) return;
    force_body<SYS, DIM, HASH, Cells, NB_CAP, LANES>(P, i, acc, measures, sortedPos, sortedVel, index, cells, n,
                                                     nbl[threadIdx.x >> 6], nullptr, false, nullptr, n, pairs,
                                                     row_masks, step, threadIdx.x % LANES);
}

// Peristalsis: pressure and viscous passes; the fused variant produces both
// from one neighbour walk (same per-pair arithmetic as the split kernels)
template <int DIM, int HASH, bool WANT_VISC, bool WANT_PRES, typename Cells>
__global__ __launch_bounds__(256) void peristalsis_force_kernel(
    const cmag_params P, float4* __restrict__ viscF, float4* __restrict__ presF,
    const float4* __restrict__ measures, const float4* __restrict__ sortedPos,
    const float4* __restrict__ sortedVel, const uint32_t* __restrict__ index, const Cells cells,
    uint32_t n, const float2* __restrict__ pairs, const uint32_t* __restrict__ row_masks, const StepArrays step) {
    __shared__ uint32_t nbl[256 / 64][NB_CAP][64];
    const uint32_t i = xcd_block() * blockDim.x + threadIdx.x;
    if (i >= n) return;
    peristalsis_force_body<DIM, HASH, WANT_VISC, WANT_PRES>(P, i, viscF, presF, measures, sortedPos, sortedVel,
                                                            index, cells, n, nbl[threadIdx.x >> 6], pairs, row_masks,
                                                            n, step);
}

// in-range neighbours (j != i, r^2 < 4h^2) of each sorted particle: the pair
// count behind the neighbour-pair interactions/s figure
template <int SYS, int DIM, int HASH, typename Cells>
__global__ __launch_bounds__(256) void count_kernel(const cmag_params P, uint32_t* __restrict__ counts,
                                                     const float4* __restrict__ sortedPos, const Cells cells,
                                                     uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float4 pi = sortedPos[i];
    const Cell gp = grid_pos(P, pi.x, pi.y, pi.z);
    const float r2max = 4.0f * P.smoothing_radius * P.smoothing_radius;
    uint32_t c = 0;
    walk_stencil<DIM, HASH>(P, pi, gp, cells, [&](uint32_t j, float px, float py, float pz, int) {
        const float4 pj = sortedPos[j];
        const float rx = px - pj.x, ry = py - pj.y, rz = pz - pj.z;
        c += (j != i && norm2(rx, ry, rz) < r2max) ? 1u : 0u;
    });
    counts[i] = c;
}

// ---- launchers --------------------------------------------------------------
// every kernel is instantiated per (system, dimension, hash order, range policy)
template <template <int, int, int> class K, typename... Args>
static void dispatch3(const cmag_params& P, Args&&... args) {
    const bool m = P.hash_order == CMAG_HASH_MORTON;
#define CMAG_GO(SYS, DIM, H) K<SYS, DIM, H>::go(args...)
    if (P.dim == 3) {
        if (P.system == CMAG_SYS_DAMBREAK) { if (m) CMAG_GO(0, 3, 1); else CMAG_GO(0, 3, 0); }
        else if (P.system == CMAG_SYS_POISEUILLE) { if (m) CMAG_GO(1, 3, 1); else CMAG_GO(1, 3, 0); }
        else { if (m) CMAG_GO(2, 3, 1); else CMAG_GO(2, 3, 0); }
    } else {
        if (P.system == CMAG_SYS_DAMBREAK) { if (m) CMAG_GO(0, 2, 1); else CMAG_GO(0, 2, 0); }
        else if (P.system == CMAG_SYS_POISEUILLE) { if (m) CMAG_GO(1, 2, 1); else CMAG_GO(1, 2, 0); }
        else { if (m) CMAG_GO(2, 2, 1); else CMAG_GO(2, 2, 0); }
    }
#undef CMAG_GO
}

template <int SYS, int DIM, int H>
struct DensityGo {
    template <int LANES = 1, typename Cells>
    static void run(const cmag_params& P, float* measures, const float* sortedPos, const Cells& cells,
                    uint32_t n, float* pairs, uint32_t* row_masks, hipStream_t s) {
        hipLaunchKernelGGL((density_kernel<SYS, DIM, H, Cells, LANES>), dim3(div_up(n, 256 / LANES)), dim3(256), 0, s, P,
                           reinterpret_cast<float4*>(measures), reinterpret_cast<const float4*>(sortedPos),
                           cells, n, reinterpret_cast<float2*>(pairs), row_masks);
    }
    static void go(const cmag_params& P, float* measures, const float* sortedPos, const uint32_t* cellStart,
                   const uint32_t* cellEnd, const uint32_t* cellFirst, uint32_t n, float* pairs, uint32_t* row_masks,
                   hipStream_t s) {
        constexpr int SHARE = SYS == CMAG_SYS_DAMBREAK ? TARGET_LANES : 1;
        const RefCells ref{cellStart, cellEnd, n};
        if (cellFirst) run(P, measures, sortedPos, FirstCells{cellFirst}, n, pairs, row_masks, s);
        else if (n <= SHARED_TARGETS) run<SHARE>(P, measures, sortedPos, ref, n, nullptr, nullptr, s);
        else run(P, measures, sortedPos, ref, n, nullptr, nullptr, s);
    }
};

int launch_density(const cmag_params& P, float* measures, const float* sortedPos,
                   const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n, hipStream_t s,
                   const uint32_t* cellFirst, float* pairs, uint32_t* row_masks) {
    if (n == 0) return CMAG_OK;
    dispatch3<DensityGo>(P, P, measures, sortedPos, cellStart, cellEnd, cellFirst, n, pairs,
                         row_masks && row_masks_apply(P) ? row_masks : nullptr, s);
    return check_launch("density_kernel");
}

template <int SYS, int DIM, int H>
struct CountGo {
    static void go(const cmag_params& P, uint32_t* counts, const float* sortedPos, const uint32_t* cellStart,
                   const uint32_t* cellEnd, uint32_t n, hipStream_t s) {
        hipLaunchKernelGGL((count_kernel<SYS, DIM, H, RefCells>), dim3(div_up(n, 256)), dim3(256), 0, s, P,
                           counts, reinterpret_cast<const float4*>(sortedPos), RefCells{cellStart, cellEnd, n}, n);
    }
};

template <int SYS, int DIM, int H>
struct ForceGo {
    template <int LANES = 1, typename Cells>
    static void run(const cmag_params& P, float* acc, const float* measures, const float* sortedPos,
                    const float* sortedVel, const uint32_t* index, const Cells& cells, uint32_t n,
                    const float* pairs, const uint32_t* row_masks, const StepArrays& step, hipStream_t s) {
        if constexpr (SYS != CMAG_SYS_PERISTALSIS)
            hipLaunchKernelGGL((force_kernel<SYS, DIM, H, Cells, LANES>), dim3(div_up(n, 256 / LANES)), dim3(256), 0, s, P,
                               reinterpret_cast<float4*>(acc), reinterpret_cast<const float4*>(measures),
                               reinterpret_cast<const float4*>(sortedPos),
                               reinterpret_cast<const float4*>(sortedVel), index, cells, n,
                               reinterpret_cast<const float2*>(pairs), row_masks, step);
    }
    static void go(const cmag_params& P, float* acc, const float* measures, const float* sortedPos,
                   const float* sortedVel, const uint32_t* index, const uint32_t* cellStart,
                   const uint32_t* cellEnd, const uint32_t* cellFirst, uint32_t n, const float* pairs,
                   const uint32_t* row_masks, const StepArrays& step, hipStream_t s) {
        constexpr int SHARE = SYS == CMAG_SYS_DAMBREAK ? TARGET_LANES : 1;
        const RefCells ref{cellStart, cellEnd, n};
        if (cellFirst)
            run(P, acc, measures, sortedPos, sortedVel, index, FirstCells{cellFirst}, n, pairs, row_masks, step, s);
        else if (n <= SHARED_TARGETS)
            run<SHARE>(P, acc, measures, sortedPos, sortedVel, index, ref, n, nullptr, nullptr, StepArrays{}, s);
        else
            run(P, acc, measures, sortedPos, sortedVel, index, ref, n, nullptr, nullptr, StepArrays{}, s);
    }
};

int launch_force(const cmag_params& P, float* acc, const float* measures, const float* sortedPos,
                 const float* sortedVel, const uint32_t* index, const uint32_t* cellStart,
                 const uint32_t* cellEnd, uint32_t n, hipStream_t s, const uint32_t* cellFirst, const float* pairs,
                 const uint32_t* row_masks, const StepArrays& step) {
    if (n == 0) return CMAG_OK;
    if (n >= (1u << NB_SHIFT_BITS)) return fail(CMAG_E_INVALID, "force passes take at most 2^27 particles");
    if (P.system == CMAG_SYS_PERISTALSIS)
        return fail(CMAG_E_INVALID, "Peristalsis uses the split pressure/viscous passes");
    if (cellFirst && P.system != CMAG_SYS_DAMBREAK && !pairs)
        return fail(CMAG_E_INVALID, "the force pass over compact offsets takes the density pass's pair values");
    dispatch3<ForceGo>(P, P, acc, measures, sortedPos, sortedVel, index, cellStart, cellEnd, cellFirst, n, pairs,
                       row_masks && row_masks_apply(P) ? row_masks : nullptr, step, s);
    return check_launch("force_kernel");
}

// ---- sub-cell walk order (DamBreak) ---------------------------------------------
// Density in sub-cell order (cell lookups staged in LDS as in force_sub_kernel,
// and the candidate positions of four stencil rows as well).
// The result goes to the reference-order row
// measures[w2r[i]] and, for a fluid row, into the sub-cell copies that the
// force pass reads: -rho in posW[i].w and db_scale p / rho^2 in velW[i].w.
// Other threads read posW rows during this pass, but only their x, y, z; a
// thread writes the w of its own row only, after its walk.
// With masks, staged blocks also leave the in-range masks of their rows for
// the force pass (masks[r * n + i]).
template <int DIM, int HASH, int LANES>
__global__ __launch_bounds__(256) void density_sub_kernel(const cmag_params P, float4* __restrict__ measures,
                                                           const uint32_t* __restrict__ keys,
                                                           const uint32_t* __restrict__ w2r, float4* posW,
                                                           float4* velW, const SubCells cells, uint32_t n,
                                                           uint2* __restrict__ masks) {
    __shared__ LookupPlan lp;
    __shared__ LookupTables lt;
    const uint32_t b0 = xcd_block() * (256 / LANES);
    const uint32_t i = b0 + threadIdx.x / LANES, part = threadIdx.x % LANES;
    // the lanes of a shared target are in different rows: none of theirs is staged
    constexpr bool ROWS = LANES == 1;
    using Stage = std::conditional_t<ROWS, RowStage, char>;
    using Rows = std::conditional_t<ROWS, RowLds, char>;
    __shared__ Stage stage;
    __shared__ Rows rows;
    const RowStage* rs = nullptr;
    const RowLds* rl = nullptr;
    const bool staged = stage_lookups<DIM, HASH>(P, keys, cells, n, b0, 256 / LANES, lp, lt);
    if constexpr (ROWS) {
        if (staged) stage_rows<DIM>(lp, lt, posW, rows, stage);
        rs = &stage;
        rl = &rows;
    }
    if (i >= n) return;
    const float4 pi = posW[i];
    float dens;
    if (!staged) {
        dens = density_sum<CMAG_SYS_DAMBREAK, DIM, HASH, LANES>(P, pi, posW, cells, part);
    } else {
        const LookupView v = lookup_view<DIM>(lp, lt, keys[i], key_masks<HASH>(P).x);
        dens = masks ? density_sum_masks<DIM, LANES>(P, pi, v, rs, rl, posW, masks, i, n, part)
                     : density_sum_lookup<DIM, LANES>(P, pi, v, rs, rl, posW, part);
    }
    if (part != 0) return;
    const float p = eos(P, dens);
    reinterpret_cast<float2*>(measures)[2 * (size_t)w2r[i]] = make_float2(dens, p);
    if (pi.w == CMAG_DB_FLUID) {
        reinterpret_cast<float*>(posW)[4 * (size_t)i + 3] = -dens;
        reinterpret_cast<float*>(velW)[4 * (size_t)i + 3] = p / (dens * dens) * db_scale(P);
    }
}

int launch_density_sub(const cmag_params& P, float* measures, const uint32_t* keys, const uint32_t* w2r, float* posW,
                       float* velW, const uint32_t* cellFirst, const uint32_t* pre, uint32_t n, hipStream_t s,
                       uint32_t* masks) {
    if (n == 0) return CMAG_OK;
    if (P.system != CMAG_SYS_DAMBREAK) return fail(CMAG_E_INVALID, "the sub-cell walk is DamBreak's");
    const SubCells cells{cellFirst, reinterpret_cast<const uint4*>(pre)};
    float4* m4 = reinterpret_cast<float4*>(measures);
    float4* pw = reinterpret_cast<float4*>(posW);
    float4* vw = reinterpret_cast<float4*>(velW);
    uint2* mk = reinterpret_cast<uint2*>(masks);
    const bool m = P.hash_order == CMAG_HASH_MORTON;
    auto run = [&](auto lanes) {
        constexpr int LANES = decltype(lanes)::value;
        const dim3 g(div_up(n, 256 / LANES)), b(256);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, g, b, 0, s, P, m4, keys, w2r, pw, vw, cells, n, mk);
        };
        if (P.dim == 3) {
            if (m) go(density_sub_kernel<3, 1, LANES>);
            else go(density_sub_kernel<3, 0, LANES>);
        } else {
            if (m) go(density_sub_kernel<2, 1, LANES>);
            else go(density_sub_kernel<2, 0, LANES>);
        }
    };
    if (n <= SHARED_TARGETS) run(std::integral_constant<int, TARGET_LANES>{});
    else run(std::integral_constant<int, 1>{});
    return check_launch("density_sub_kernel");
}

// Force in sub-cell order; a block whose targets share one row of cells finds
// its runs through the cell lookups staged in LDS (the same runs as the
// global walk).  CAP: neighbour queue depth; with the in-range masks only
// walked rows and blocks without staged lookups queue neighbours, and a
// shallower queue leaves more LDS to the CU.  What bounds it: the rows gathered
// for the pair terms (the data-return path of L1 is busy 88 % of the time, vector
// issue about half of it), 32 B a neighbour.  Z-order cells, 16M dam break: 3.54 ms
// with registers held so that six waves share a SIMD, 3.75 ms with seven (a spill
// inside the pair loop), 3.56 ms with five.  Linear cells, a whole step of the 1M
// one (1.6M rows): 679 us with six, though that spills, 702 with five and 744
// with four, neither of which does.
template <int DIM, int HASH, int CAP, int LANES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(CAP <= 8 && LANES == 1 ? 6 : 1, 8))) void force_sub_kernel(
    const cmag_params P, float4* __restrict__ acc, const float4* __restrict__ posW, const float4* __restrict__ velW,
    const uint32_t* __restrict__ indexW, const uint32_t* __restrict__ keys, const SubCells cells, uint32_t n,
    const uint2* __restrict__ masks, const StepArrays step) {
    __shared__ uint32_t nbl[256 / 64][CAP][64];
    __shared__ LookupPlan lp;
    __shared__ LookupTables lt;
    const uint32_t b0 = xcd_block() * (256 / LANES);
    const uint32_t i = b0 + threadIdx.x / LANES;
    const bool staged = stage_lookups<DIM, HASH>(P, keys, cells, n, b0, 256 / LANES, lp, lt);
    if (i >= n) return;
    // made in every block, so that the tables stay LDS addresses; used when staged
    const LookupView v = lookup_view<DIM>(lp, lt, keys[i], key_masks<HASH>(P).x);
    force_body<CMAG_SYS_DAMBREAK, DIM, HASH, SubCells, CAP, LANES>(P, i, acc, nullptr, posW, velW, indexW, cells, n,
                                                                   nbl[threadIdx.x >> 6], &v, staged, masks, n,
                                                                   nullptr, nullptr, step, threadIdx.x % LANES);
}

int launch_force_sub(const cmag_params& P, float* acc, const float* posW, const float* velW,
                     const uint32_t* indexW, const uint32_t* keys, const uint32_t* cellFirst, const uint32_t* pre,
                     uint32_t n, hipStream_t s, const uint32_t* masks, const StepArrays& step) {
    if (n == 0) return CMAG_OK;
    if (step.pos && n > SHARED_TARGETS)
        return fail(CMAG_E_INVALID, "the sub-cell force pass integrates shared targets only");
    if (n >= (1u << NB_SHIFT_BITS)) return fail(CMAG_E_INVALID, "force passes take at most 2^27 particles");
    if (P.system != CMAG_SYS_DAMBREAK) return fail(CMAG_E_INVALID, "the sub-cell walk is DamBreak's");
    const SubCells cells{cellFirst, reinterpret_cast<const uint4*>(pre)};
    auto run = [&](auto dim, auto hash, auto lanes) {
        constexpr int D = decltype(dim)::value, H = decltype(hash)::value, LANES = decltype(lanes)::value;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(div_up(n, 256 / LANES)), dim3(256), 0, s, P, reinterpret_cast<float4*>(acc),
                               reinterpret_cast<const float4*>(posW), reinterpret_cast<const float4*>(velW), indexW,
                               keys, cells, n, reinterpret_cast<const uint2*>(masks), step);
        };
        if (masks) go(force_sub_kernel<D, H, 8, LANES>);
        else go(force_sub_kernel<D, H, NB_CAP, LANES>);
    };
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    auto pick = [&](auto lanes) {
        const bool m = P.hash_order == CMAG_HASH_MORTON;
        if (P.dim == 3) { if (m) run(I3{}, H1{}, lanes); else run(I3{}, H0{}, lanes); }
        else { if (m) run(I2{}, H1{}, lanes); else run(I2{}, H0{}, lanes); }
    };
    if (n <= SHARED_TARGETS) pick(std::integral_constant<int, TARGET_LANES>{});
    else pick(std::integral_constant<int, 1>{});
    return check_launch("force_sub_kernel");
}

template <bool V, bool PR, typename Cells>
static void go_peri_cells(const cmag_params& P, float* viscF, float* presF, const float* measures,
                          const float* sortedPos, const float* sortedVel, const uint32_t* index,
                          const Cells& cells, uint32_t n, const float* pairs, const uint32_t* row_masks,
                          const StepArrays& step, hipStream_t s) {
    const bool m = P.hash_order == CMAG_HASH_MORTON;
    auto launch = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(div_up(n, 256)), dim3(256), 0, s, P, reinterpret_cast<float4*>(viscF),
                           reinterpret_cast<float4*>(presF), reinterpret_cast<const float4*>(measures),
                           reinterpret_cast<const float4*>(sortedPos), reinterpret_cast<const float4*>(sortedVel),
                           index, cells, n, reinterpret_cast<const float2*>(pairs), row_masks, step);
    };
    if (P.dim == 3) {
        if (m) launch(peristalsis_force_kernel<3, 1, V, PR, Cells>);
        else launch(peristalsis_force_kernel<3, 0, V, PR, Cells>);
    } else {
        if (m) launch(peristalsis_force_kernel<2, 1, V, PR, Cells>);
        else launch(peristalsis_force_kernel<2, 0, V, PR, Cells>);
    }
}

template <bool V, bool PR>
static void go_peri(const cmag_params& P, float* viscF, float* presF, const float* measures,
                    const float* sortedPos, const float* sortedVel, const uint32_t* index,
                    const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n, hipStream_t s) {
    if (n >= (1u << NB_SHIFT_BITS)) return;  // rejected by the callers
    go_peri_cells<V, PR>(P, viscF, presF, measures, sortedPos, sortedVel, index, RefCells{cellStart, cellEnd, n}, n,
                         nullptr, nullptr, StepArrays{}, s);
}

int launch_pressure_force(const cmag_params& P, float* presF, const float* measures,
                          const float* sortedPos, const uint32_t* index, const uint32_t* cellStart,
                          const uint32_t* cellEnd, uint32_t n, hipStream_t s) {
    if (n == 0) return CMAG_OK;
    if (n >= (1u << NB_SHIFT_BITS)) return fail(CMAG_E_INVALID, "force passes take at most 2^27 particles");
    go_peri<false, true>(P, nullptr, presF, measures, sortedPos, nullptr, index, cellStart, cellEnd, n, s);
    return check_launch("peristalsis_force_kernel<pressure>");
}

int launch_viscous_force(const cmag_params& P, float* viscF, const float* measures,
                         const float* sortedPos, const float* sortedVel, const uint32_t* index,
                         const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n,
                         hipStream_t s) {
    if (n == 0) return CMAG_OK;
    if (n >= (1u << NB_SHIFT_BITS)) return fail(CMAG_E_INVALID, "force passes take at most 2^27 particles");
    go_peri<true, false>(P, viscF, nullptr, measures, sortedPos, sortedVel, index, cellStart, cellEnd, n, s);
    return check_launch("peristalsis_force_kernel<viscous>");
}

int launch_peristalsis_forces(const cmag_params& P, float* viscF, float* presF, const float* measures,
                              const float* sortedPos, const float* sortedVel, const uint32_t* index,
                              const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n,
                              hipStream_t s, const uint32_t* cellFirst, const float* pairs,
                              const uint32_t* row_masks, const StepArrays& step) {
    if (n == 0) return CMAG_OK;
    if (n >= (1u << NB_SHIFT_BITS)) return fail(CMAG_E_INVALID, "force passes take at most 2^27 particles");
    if (!cellFirst) {
        go_peri<true, true>(P, viscF, presF, measures, sortedPos, sortedVel, index, cellStart, cellEnd, n, s);
        return check_launch("peristalsis_force_kernel<fused>");
    }
    if (!pairs) return fail(CMAG_E_INVALID, "the force pass over compact offsets takes the density pass's pair values");
    go_peri_cells<true, true>(P, viscF, presF, measures, sortedPos, sortedVel, index, FirstCells{cellFirst}, n, pairs,
                              row_masks && row_masks_apply(P) ? row_masks : nullptr, step, s);
    return check_launch("peristalsis_force_kernel<fused>");
}

}  // namespace cmag

using namespace cmag;

extern "C" {

int cmag_density(const cmag_params* p, float* measures, const float* sortedPos,
                 const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n,
                 cmag_stream_t stream) {
    CMAG_TRY(validate_params(p));
    if (n && (!measures || !sortedPos || !cellStart || !cellEnd))
        return fail(CMAG_E_INVALID, "cmag_density: null pointer");
    return launch_density(*p, measures, sortedPos, cellStart, cellEnd, n, as_stream(stream));
}

int cmag_count_neighbours(const cmag_params* p, uint32_t* counts, const float* sortedPos,
                          const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n,
                          cmag_stream_t stream) {
    CMAG_TRY(validate_params(p));
    if (n && (!counts || !sortedPos || !cellStart || !cellEnd))
        return fail(CMAG_E_INVALID, "cmag_count_neighbours: null pointer");
    if (n == 0) return CMAG_OK;
    dispatch3<CountGo>(*p, *p, counts, sortedPos, cellStart, cellEnd, n, as_stream(stream));
    return check_launch("count_kernel");
}

int cmag_force(const cmag_params* p, float* acc, const float* measures, const float* sortedPos,
               const float* sortedVel, const uint32_t* index, const uint32_t* cellStart,
               const uint32_t* cellEnd, uint32_t n, cmag_stream_t stream) {
    CMAG_TRY(validate_params(p));
    if (n && (!acc || !measures || !sortedPos || !sortedVel || !index || !cellStart || !cellEnd))
        return fail(CMAG_E_INVALID, "cmag_force: null pointer");
    return launch_force(*p, acc, measures, sortedPos, sortedVel, index, cellStart, cellEnd, n,
                        as_stream(stream));
}

int cmag_pressure_force(const cmag_params* p, float* presF, const float* measures,
                        const float* sortedPos, const uint32_t* index, const uint32_t* cellStart,
                        const uint32_t* cellEnd, uint32_t n, cmag_stream_t stream) {
    CMAG_TRY(validate_params(p));
    if (n && (!presF || !measures || !sortedPos || !index || !cellStart || !cellEnd))
        return fail(CMAG_E_INVALID, "cmag_pressure_force: null pointer");
    return launch_pressure_force(*p, presF, measures, sortedPos, index, cellStart, cellEnd, n,
                                 as_stream(stream));
}

int cmag_viscous_force(const cmag_params* p, float* viscF, const float* measures,
                       const float* sortedPos, const float* sortedVel, const uint32_t* index,
                       const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n,
                       cmag_stream_t stream) {
    CMAG_TRY(validate_params(p));
    if (n && (!viscF || !measures || !sortedPos || !sortedVel || !index || !cellStart || !cellEnd))
        return fail(CMAG_E_INVALID, "cmag_viscous_force: null pointer");
    return launch_viscous_force(*p, viscF, measures, sortedPos, sortedVel, index, cellStart, cellEnd,
                                n, as_stream(stream));
}

}  // extern "C"
