// sph_device.hpp - per-particle bodies of the neighbour passes (gfx950, wave64,
// FP32), shared by the single-system kernels (sph.hip) and the batched
// persistent kernels (batch.hip).
//
// The stencil of (2*cellcount+1)^dim cells is walked in the reference's z, y, x
// order and each cell's particles in sorted order, so sums accumulate in the
// reference's order.  Candidates are culled on r^2 < 4h^2 before any square
// root; inner-loop reciprocals use the hardware v_rcp/v_sqrt (1 ulp), the
// per-particle divisions stay IEEE.
//
//   density       fluid_kernel.cu:99-169, poiseuilleFlowKernel.cu:99-182,
//                 PeristalsisDensity.cu:3-79
//   force         fluid_kernel.cu:172-292 (DamBreak: pressure + Monaghan AV,
//                 Lennard-Jones walls), poiseuilleFlowKernel.cu:184-309
//                 (pressure + Morris viscosity with wall extrapolation)
//   pressure /    PeristalsisPressureForce.cu:3-90,
//   viscous       PeristalsisViscousForce.cu:143-241
#pragma once

#include "common.hpp"
#include "integrate_device.hpp"
#include "kernels.hpp"
#include "step_state.hpp"

// Every fused multiply-add below is written out (fmaf) and no other is formed:
// the same sum then rounds the same way in every kernel that inlines it
// (walker or neighbour list, single system or batch), which keeps those
// paths bit-identical.
#pragma clang fp contract(off)

namespace cmag {

// |r|^2 as (x*x) then two fused steps
__device__ __forceinline__ float norm2(float rx, float ry, float rz) {
    return fmaf(rz, rz, fmaf(ry, ry, rx * rx));
}


__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float frsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

// integer power by squaring (gamma is an integer in [1,15])
__device__ __forceinline__ float pow_int(float x, int e) {
    float r = 1.0f, b = x;
    while (e) {
        if (e & 1) r *= b;
        b *= b;
        e >>= 1;
    }
    return r;
}

__device__ __forceinline__ float eos(const cmag_params& P, float dens) {
    if (P.eos == CMAG_EOS_TAIT) return P.B * (pow_int(dens / P.rest_density, (int)P.gamma) - 1.0f);
    if (P.eos == CMAG_EOS_LINEAR_C2) return P.soundspeed * P.soundspeed * dens;
    return 50.0f * P.soundspeed * dens;
}

// Range policies of the stencil walker.  A run holds the cells with keys
// k0..k1 (consecutive keys are contiguous in the sorted arrays).
//   RefCells   the reference arrays: first non-empty cellStart and last
//              cellEnd of the run (empty cells hold 0xffffffff)
//   FirstCells compact offsets first[c] (cells before c), one pair of loads
struct RefCells {
    static constexpr bool SUB = false;
    static constexpr bool PADDED = false;  // a caller's rows: nothing is read past them
    const uint32_t* __restrict__ cellStart;
    const uint32_t* __restrict__ cellEnd;
    uint32_t n;
    __device__ __forceinline__ bool range(uint32_t k0, uint32_t k1, uint32_t& s, uint32_t& e) const {
        // up to three cells (a stencil of one cell a side) with their loads side
        // by side; e clamped to the particle count: consistent cell arrays
        // never need it, inconsistent ones cannot read past n
        if (k1 - k0 <= 2u) {
            const uint32_t km = min(k0 + 1u, k1);
            const uint32_t s0 = cellStart[k0], s1 = cellStart[km], s2 = cellStart[k1];
            const uint32_t e0 = cellEnd[k0], e1 = cellEnd[km], e2 = cellEnd[k1];
            s = s0 != CMAG_CELL_EMPTY ? s0 : s1 != CMAG_CELL_EMPTY ? s1 : s2;
            e = min(s2 != CMAG_CELL_EMPTY ? e2 : s1 != CMAG_CELL_EMPTY ? e1 : e0, n);
            return s != CMAG_CELL_EMPTY && s < e;
        }
        s = CMAG_CELL_EMPTY;
        e = 0;
        for (uint32_t k = k0; k <= k1; ++k) {
            const uint32_t st = cellStart[k];
            if (st == CMAG_CELL_EMPTY) continue;
            if (s == CMAG_CELL_EMPTY) s = st;
            e = min(cellEnd[k], n);
        }
        return s != CMAG_CELL_EMPTY && s < e;
    }
};

struct FirstCells {
    static constexpr bool SUB = false;
    static constexpr bool PADDED = true;  // rows of a System or batch: two may be read past the last
    const uint32_t* __restrict__ first;
    __device__ __forceinline__ bool range(uint32_t k0, uint32_t k1, uint32_t& s, uint32_t& e) const {
        s = first[k0];
        e = first[k1 + 1];
        return s < e;
    }
};

// ---- sub-cell walk order (DamBreak) ---------------------------------------------
// Inside each cell the particles can be kept in a second, internal order: by
// bucket, then in reference order, with buckets 0..7 the fluid particles of
// each eighth of the cell along x and bucket 8 the wall particles.  A target
// in eighth q of its cell needs, of the stencil's first cell along x, only the
// fluid of eighths >= q (the rest lies more than cellcount cells away, beyond
// 2h), and of the last cell only the eighths <= q.  Wall particles sit in
// their own bucket and are always walked: DamBreak's Lennard-Jones term acts
// on every wall particle of the stencil.  x_sub (common.hpp) is the target's /
// particle's eighth.

// SubCells: cell offsets first[] as FirstCells plus, per cell, the running
// counts pre[c]: eight 16-bit counts, #buckets <= t for t = 0..7 (t = 7: the
// cell's fluid), two to a word, low half first; cells without particles hold
// zeros
struct SubCells {
    static constexpr bool SUB = true;
    static constexpr bool PADDED = true;
    const uint32_t* __restrict__ first;
    const uint4* __restrict__ pre;
    // count t (0..7) of a cell's entry, read as one 16-bit value (the eighth
    // differs between the lanes of a wave)
    __device__ __forceinline__ static uint32_t count(const uint4* c, int t) {
        return reinterpret_cast<const uint16_t*>(c)[t];
    }
    // the fluid of eighths <= q, of eighths < q, and all of it
    __device__ __forceinline__ static uint32_t through(const uint4* c, int q) { return count(c, q); }
    __device__ __forceinline__ static uint32_t below(const uint4* c, int q) {
        const uint32_t v = count(c, q > 0 ? q - 1 : 0);
        return q > 0 ? v : 0u;
    }
    __device__ __forceinline__ static uint32_t fluid(const uint4* c) { return count(c, X_SUBS - 1); }
    // the run k0..k1 trimmed for a target in eighth q: lo (k0 is the
    // stencil's first cell along x) drops k0's fluid eighths < q, hi (k1 is
    // the last) ends at k1's eighth q and returns k1's walls as [ws, we)
    __device__ __forceinline__ void range_sub(uint32_t k0, uint32_t k1, bool lo, bool hi, int q, uint32_t& s,
                                              uint32_t& e, uint32_t& ws, uint32_t& we) const {
        s = first[k0];
        if (lo) s += below(pre + k0, q);
        ws = we = 0;
        if (hi) {
            const uint32_t f1 = first[k1];
            e = f1 + through(pre + k1, q);
            ws = f1 + fluid(pre + k1);
            we = first[k1 + 1];
        } else {
            e = first[k1 + 1];
        }
    }
};

// A run of key-consecutive cells: a contiguous range of the sorted arrays,
// with the target position minus the run's periodic image offset and the
// image-shift code (sx+1) + 3(sy+1) + 9(sz+1) (13: no shift).
struct Run {
    uint32_t s, len;
    float px;
    int code;
};

// The order in which the force pass takes the stencil rows (row r = (dz + 1)
// * 3 + (dy + 1)): rows of opposite offsets in pairs -- the diagonal corners
// (y - 1, z - 1) with (y + 1, z + 1) and (y + 1, z - 1) with (y - 1, z + 1),
// then y - 1 with y + 1 and z - 1 with z + 1 -- and the centre row last.  A
// lane's in-range neighbours are spread unevenly between opposite rows (a
// target near the top of its cell has most of them above), so taking a pair's
// mask bits as one sequence per lane evens the lanes' work out; the walks
// without masks take the rows in the same order, so the sums are the same.
struct RowList {
    uint64_t rows;  // four bits each, first lowest
    int count;
    __device__ __forceinline__ int operator[](int k) const { return (int)((rows >> (4 * k)) & 15u); }
};

// Targets shared between lanes.  A neighbour pass is one serial chain per
// target; with few targets the chip waits for it (20,000 rows fill a third of
// the SIMDs with one wave).  TARGET_LANES lanes then share a target, each with
// some of its stencil rows, and fold their sums: pairs of lanes first, then
// both pairs.  The same lanes take the same rows in the same order wherever
// the neighbours come from (global walk, staged lookups, masks).
constexpr int TARGET_LANES = 4;
__device__ __forceinline__ float quad_sum(float v) {
    // quad_perm [1,0,3,2], then [2,3,0,1]
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, true));
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, true));
    return v;
}

// the rows of lane `part` of LANES in the force pass.  Shared: two edge pairs,
// each with one row of a corner pair, the centre row, and the other corner
// pair: about 24, 24, 16 and 10 of the 74 in-range neighbours, in two turns
template <int LANES>
__device__ __forceinline__ RowList force_rows(int dim, uint32_t part) {
    static_assert(LANES == 1 || LANES == TARGET_LANES, "one lane or a quad");
    // 3-D: 0 8 2 6 3 5 1 7 4; 2-D: 0 2 1
    if (LANES == 1) return dim == 3 ? RowList{0x471536280ull, 9} : RowList{0x120ull, 3};
    if (dim == 3) {
        const uint64_t rows = part == 0 ? 0x253ull : part == 1 ? 0x671ull : part == 2 ? 0x4ull : 0x80ull;
        return RowList{rows, part < 2 ? 3 : part == 2 ? 1 : 2};
    }
    return RowList{part == 0 ? 0x0ull : part == 1 ? 0x2ull : 0x1ull, part < 3 ? 1 : 0};
}

// Walk the stencil of gp in z, y, x order and call cand(j, qx, qy, qz, code)
// for every candidate j in the reference's order.  Along x, cells with
// consecutive keys form one run (linear order: the whole row; brick Z order:
// the part inside one brick; plain Z order: an even/odd pair); a row has at
// most two runs except at periodic seams.  The runs of a row are gathered
// first and then walked as one loop, so every lane of a wave spends the row in
// the same loop whatever its x position -- lanes whose row splits at a
// different x would otherwise serialise the wave.
// PERIODIC = false compiles the image shifts out (DamBreak has none).
//
// In the linear order a target inside the grid along x has the same one or two
// runs of cells (two where its stencil crosses the seam) relative to every row,
// so they are found once: a wave all of whose targets are so takes each row
// with two to four offset loads.  Stepping through a row's cells instead cost
// more than half the instructions of the 2-D passes (7 x 7 cells of one
// spacing, 4.1M particles in 256 channels: density 2,647 VALU instructions per
// wave of 64 targets and 264 us, force 4,582 and 552 us).
//
// walk_rows does the walk and hands each row's runs to row(a, b, qy, qz, whole);
// whole: the whole row comes in this one call (in every lane of the wave).
// walk_stencil and walk_stencil_pf turn them into candidate calls.  With
// FORCE_ORDER and one cell per stencil side, the rows come in force_rows order.
// With LANES > 1 that many lanes share the target: this one takes the rows
// part, part + LANES, ...
template <int DIM, int HASH, bool PERIODIC = true, bool FORCE_ORDER = false, int LANES = 1, typename Cells, typename R>
__device__ __forceinline__ void walk_rows(const cmag_params& P, const float4& pi, const Cell& gp,
                                          const Cells& cells, R&& run_pair, uint32_t part = 0) {
    const int cc = P.cellcount;
    const int sub = Cells::SUB ? x_sub(P, pi.x) : 0;
    const uint32_t gxm = P.grid_size[0] - 1u, gym = P.grid_size[1] - 1u, gzm = P.grid_size[2] - 1u;
    const uint32_t Mx = P.morton_mask[0], My = P.morton_mask[1], Mz = P.morton_mask[2];
    const bool perx = PERIODIC && (P.periodic_mask & 1), pery = PERIODIC && (P.periodic_mask & 2),
               perz = PERIODIC && (P.periodic_mask & 4);
    uint32_t kx0 = 0, ky0 = 0, kz0 = 0;
    if (HASH == CMAG_HASH_MORTON) {
        const uint32_t own = grid_hash(P, gp.x, gp.y, gp.z);
        kx0 = own & Mx;
        ky0 = own & My;
        kz0 = own & Mz;
        for (int k = 0; k < cc; ++k) {
            kx0 = dilated_dec(kx0, Mx);
            ky0 = dilated_dec(ky0, My);
            if (DIM == 3) kz0 = dilated_dec(kz0, Mz);
        }
    }
    // linear order: the same cells [a0, a1], then [b0, b1] (none: b0 > b1),
    // relative to every row; any_b: some lane has both
    bool rows_alike = false, any_b = false;
    int a0 = 0, a1 = 0, b0 = 1, b1 = 0;
    float apx = pi.x, bpx = pi.x;
    int acx = 1, bcx = 1;
    if (HASH == CMAG_HASH_LINEAR && Cells::PADDED) {
        const int gx = (int)P.grid_size[0], lo = gp.x - cc, hi = gp.x + cc;
        const bool inside = lo >= 0 && hi < gx;
        rows_alike = __ballot(!(inside || (gp.x >= 0 && gp.x < gx && 2 * cc + 1 <= gx))) == 0ull;
        any_b = __ballot(!inside) != 0ull;
        if (lo < 0) {
            a0 = lo + gx; a1 = gx - 1; b0 = 0; b1 = hi;
            if (perx) { apx = pi.x + P.world_size[0]; acx = 0; }
        } else if (hi >= gx) {
            a0 = lo; a1 = gx - 1; b0 = 0; b1 = hi - gx;
            if (perx) { bpx = pi.x - P.world_size[0]; bcx = 2; }
        } else {
            a0 = lo; a1 = hi;
        }
    }
    // one stencil row (dy, dz); ky, kz: its Morton key parts
    auto row_body = [&](int dy, int dz, uint32_t ky, uint32_t kz) {
        const int nz = gp.z + dz;
        const int sz = perz ? image_shift(nz, P.grid_size[2]) : 0;
        const float pz = perz ? pi.z - (float)sz * P.world_size[2] : pi.z;
        const int ny = gp.y + dy;
        const int sy = pery ? image_shift(ny, P.grid_size[1]) : 0;
        const float py = pery ? pi.y - (float)sy * P.world_size[1] : pi.y;
        const int code_yz = 3 * (sy + 1) + 9 * (sz + 1);
        const uint32_t row = (HASH == CMAG_HASH_LINEAR)
                                 ? (((uint32_t)nz & gzm) * P.grid_size[1] + ((uint32_t)ny & gym)) * P.grid_size[0]
                                 : (kz | ky);
        if constexpr (HASH == CMAG_HASH_LINEAR && Cells::PADDED) {
            // one call of run_pair in the code (it is large): a row that is not
            // alike comes cell by cell, the sub-cell walk's last walls by themselves
            auto run = [](uint32_t s, uint32_t e, float px, int code) { return Run{s, e > s ? e - s : 0u, px, code}; };
            const Run none{0u, 0u, pi.x, 13};
            const int parts = rows_alike ? (Cells::SUB && any_b ? 2 : 1) : 2 * cc + 1;
            uint32_t ws = 0, we = 0;
            for (int part = 0; part < parts; ++part) {
                Run a = none, b = none;
                uint32_t s, e;
                if (!rows_alike) {
                    const int nx = gp.x + part - cc;
                    const int sx = perx ? image_shift(nx, P.grid_size[0]) : 0;
                    const float px = perx ? pi.x - (float)sx * P.world_size[0] : pi.x;
                    const uint32_t key = row + ((uint32_t)nx & gxm);
                    const int code = (sx + 1) + code_yz;
                    if constexpr (Cells::SUB) {
                        cells.range_sub(key, key, part == 0, part == 2 * cc, sub, s, e, ws, we);
                        b = run(ws, we, px, code);
                    } else {
                        (void)cells.range(key, key, s, e);
                    }
                    a = run(s, e, px, code);
                } else if constexpr (Cells::SUB) {
                    const bool both = any_b && b0 <= b1;
                    if (part == 0) {
                        cells.range_sub(row + (uint32_t)a0, row + (uint32_t)a1, true, !both, sub, s, e, ws, we);
                        a = run(s, e, pi.x, code_yz + 1);
                        if (both) {
                            cells.range_sub(row + (uint32_t)b0, row + (uint32_t)b1, false, true, sub, s, e, ws, we);
                            b = run(s, e, pi.x, code_yz + 1);
                        } else {
                            b = run(ws, we, pi.x, code_yz + 1);
                            ws = we = 0u;
                        }
                    } else {
                        a = run(ws, we, pi.x, code_yz + 1);
                    }
                } else {
                    (void)cells.range(row + (uint32_t)a0, row + (uint32_t)a1, s, e);
                    a = run(s, e, apx, acx + code_yz);
                    if (any_b && b0 <= b1) {
                        (void)cells.range(row + (uint32_t)b0, row + (uint32_t)b1, s, e);
                        b = run(s, e, bpx, bcx + code_yz);
                    }
                }
                run_pair(a, b, py, pz, !Cells::SUB && rows_alike);
            }
            return;
        }
        Run a{0u, 0u, pi.x, 13}, b{0u, 0u, pi.x, 13};
        bool have_a = false;
        auto push = [&](uint32_t s, uint32_t e, float px, int code) {
            const Run r{s, e - s, px, code};
            if (!have_a) {
                a = r;
                have_a = true;
            } else if (b.len == 0) {
                b = r;
            } else {  // a third run in one row (periodic seam with plain Z order, or walls)
                run_pair(a, b, py, pz, false);
                a = r;
                b.len = 0;
            }
        };
        // lo / hi: the run starts at the stencil's first cell / ends at its last
        auto emit = [&](uint32_t k0, uint32_t k1, float px, int code, bool lo, bool hi) {
            uint32_t s, e;
            if constexpr (Cells::SUB) {
                uint32_t ws, we;
                cells.range_sub(k0, k1, lo, hi, sub, s, e, ws, we);
                if (s < e) push(s, e, px, code);
                if (ws < we) push(ws, we, px, code);
            } else {
                if (cells.range(k0, k1, s, e)) push(s, e, px, code);
            }
        };
        uint32_t k0 = 0, k1 = 0;
        float run_px = pi.x;
        int run_sx = 0;
        bool run_lo = true;
        uint32_t kx = kx0;
        for (int dx = -cc; dx <= cc; ++dx) {
            const int nx = gp.x + dx;
            const int sx = perx ? image_shift(nx, P.grid_size[0]) : 0;
            const float px = perx ? pi.x - (float)sx * P.world_size[0] : pi.x;
            const uint32_t key = (HASH == CMAG_HASH_LINEAR) ? row + ((uint32_t)nx & gxm) : (row | kx);
            if (dx == -cc) {
                k0 = k1 = key;
                run_px = px;
                run_sx = sx;
            } else if (key == k1 + 1u && sx == run_sx) {
                k1 = key;
            } else {
                emit(k0, k1, run_px, (run_sx + 1) + code_yz, run_lo, false);
                k0 = k1 = key;
                run_px = px;
                run_sx = sx;
                run_lo = false;
            }
            if (HASH == CMAG_HASH_MORTON) kx = dilated_inc(kx, Mx);
        }
        emit(k0, k1, run_px, (run_sx + 1) + code_yz, run_lo, true);
        run_pair(a, b, py, pz, false);
    };
    const int zlo = DIM == 2 ? 0 : -cc, zhi = DIM == 2 ? 0 : cc;
    if (FORCE_ORDER && cc == 1) {
        // the force pass's row order (force_rows), as its staged blocks take it;
        // the Morton key parts are stepped from the stencil's first row each time
        const RowList list = force_rows<LANES>(DIM, part);
        for (int k = 0; k < list.count; ++k) {
            const int r = list[k];
            const int iy = r % 3, iz = DIM == 3 ? r / 3 : 0;
            uint32_t ky = ky0, kz = kz0;
            if (HASH == CMAG_HASH_MORTON) {
                for (int t = 0; t < iy; ++t) ky = dilated_inc(ky, My);
                for (int t = 0; t < iz; ++t) kz = dilated_inc(kz, Mz);
            }
            row_body(iy - 1, DIM == 3 ? iz - 1 : 0, ky, kz);
        }
        return;
    }
    if (LANES > 1) {
        const int side = 2 * cc + 1, rows = DIM == 2 ? side : side * side;
        for (int r = (int)part; r < rows; r += LANES) {
            const int iz = DIM == 2 ? 0 : r / side, iy = r - iz * side;
            uint32_t ky = ky0, kz = kz0;
            if (HASH == CMAG_HASH_MORTON) {
                for (int t = 0; t < iy; ++t) ky = dilated_inc(ky, My);
                for (int t = 0; t < iz; ++t) kz = dilated_inc(kz, Mz);
            }
            row_body(iy - cc, DIM == 2 ? 0 : iz - cc, ky, kz);
        }
        return;
    }
    uint32_t kz = kz0;
    for (int dz = zlo; dz <= zhi; ++dz) {
        uint32_t ky = ky0;
        for (int dy = -cc; dy <= cc; ++dy) {
            row_body(dy, dz, ky, kz);
            if (HASH == CMAG_HASH_MORTON) ky = dilated_inc(ky, My);
        }
        if (HASH == CMAG_HASH_MORTON) kz = dilated_inc(kz, Mz);
    }
}

// row j of a float4 array through a 32-bit byte offset (j < 2^28), which
// lets the load take the array base from scalar registers
__device__ __forceinline__ float4 row4(const float4* __restrict__ base, uint32_t j) {
    return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(base) + (j << 4));
}

template <int DIM, int HASH, bool PERIODIC = true, typename Cells, typename C>
__device__ __forceinline__ void walk_stencil(const cmag_params& P, const float4& pi, const Cell& gp,
                                             const Cells& cells, C&& cand) {
    walk_rows<DIM, HASH, PERIODIC>(P, pi, gp, cells, [&](const Run& a, const Run& b, float py, float pz, bool) {
        const uint32_t total = a.len + b.len;
        for (uint32_t t = 0; t < total; ++t) {
            const bool second = t >= a.len;
            const uint32_t j = second ? b.s + (t - a.len) : a.s + t;
            cand(j, second ? b.px : a.px, py, pz, second ? b.code : a.code);
        }
    });
}

// walk_stencil with the candidates' sorted positions loaded ahead:
// cand(j, pos[j], valid, qx, qy, qz, code).  The loop is unrolled by two; the
// load of candidate t + 1 is issued before candidate t is evaluated and the
// load for the next pass before candidate t + 1, so each wait covers loads
// that were issued a candidate earlier.  Loads and calls are unconditional
// (indices clamped to the run's last row, and the second call flagged
// valid = false when it lies past the run: the candidate must then contribute
// nothing), which keeps the loads out of divergent branches.
// the rows [s, e) of a sub-cell copy as one loop over a byte offset, two rows
// per iteration, each load issued one candidate ahead of its use; it reads up
// to two rows past the run (the copies carry padding rows)
template <typename C>
__device__ __forceinline__ void walk_run_sub(const float4* __restrict__ pos, uint32_t s, uint32_t e, float px,
                                             float py, float pz, int code, C&& cand) {
    const char* base = reinterpret_cast<const char*>(pos);
    auto ld = [&](uint32_t off) { return *reinterpret_cast<const float4*>(base + off); };
    const uint32_t end = e << 4, end1 = end - 16u;
    uint32_t off = s << 4;
    if (off >= end) return;
    float4 p0 = ld(off);
    do {
        const float4 p1 = ld(off + 16u);
        cand(off >> 4, p0, true, px, py, pz, code);
        p0 = ld(off + 32u);
        cand((off >> 4) + 1u, p1, off < end1, px, py, pz, code);
        off += 32u;
    } while (off < end);
}

// one row of walk_stencil_pf
template <bool PADDED, typename C>
__device__ __forceinline__ void walk_row_pf(const Run& a, const Run& b, float py, float pz,
                                            const float4* __restrict__ pos, C&& cand) {
    const uint32_t total = a.len + b.len;
    if (total == 0) return;
    const uint32_t off_b = b.s - a.len;
    auto row = [&](uint32_t t) { return (t >= a.len ? off_b : a.s) + t; };
    auto visit = [&](uint32_t t, uint32_t j, const float4& pj, bool valid) {
        const bool second = t >= a.len;
        cand(j, pj, valid, second ? b.px : a.px, py, pz, second ? b.code : a.code);
    };
    const uint32_t last = total - 1u;
    // padded: up to two rows past the row's last run are read (and flagged)
    auto next = [&](uint32_t t) { return PADDED ? t : min(t, last); };
    uint32_t j0 = row(0);
    float4 p0 = row4(pos, j0);
    for (uint32_t t = 0; t < total; t += 2) {
        const uint32_t t1 = next(t + 1u);
        const uint32_t j1 = row(t1);
        const float4 p1 = row4(pos, j1);
        visit(t, j0, p0, true);
        j0 = row(next(t + 2u));
        p0 = row4(pos, j0);
        visit(t1, j1, p1, t + 1u < total);
    }
}

// one row's candidates two at a time, for a pass that needs only their
// positions: f(p0, px0, p1, px1, valid1).  A wave none of whose targets has a
// second run (no seam near) steps a byte offset; the others choose between
// their two runs per candidate.  Rows of a System or batch: up to two rows past
// the last run are read (and flagged).
template <typename F>
__device__ __forceinline__ void walk_row_two(const Run& a, const Run& b, const float4* __restrict__ pos, F&& f) {
    if (__ballot(b.len != 0u) == 0ull) {
        const char* base = reinterpret_cast<const char*>(pos);
        const uint32_t end = (a.s + a.len) << 4, end1 = end - 16u;
        for (uint32_t off = a.s << 4; off < end; off += 32u) {
            const float4 p0 = *reinterpret_cast<const float4*>(base + off);
            const float4 p1 = *reinterpret_cast<const float4*>(base + off + 16u);
            f(p0, a.px, p1, a.px, off < end1);
        }
        return;
    }
    const uint32_t total = a.len + b.len, off_b = b.s - a.len;
    for (uint32_t t = 0; t < total; t += 2) {
        const bool s0 = t >= a.len, s1 = t + 1u >= a.len;
        const float4 p0 = row4(pos, (s0 ? off_b : a.s) + t);
        const float4 p1 = row4(pos, (s1 ? off_b : a.s) + t + 1u);
        f(p0, s0 ? b.px : a.px, p1, s1 ? b.px : a.px, t + 1u < total);
    }
}

template <int DIM, int HASH, bool PERIODIC = true, bool FORCE_ORDER = false, int LANES = 1, typename Cells, typename C>
__device__ __forceinline__ void walk_stencil_pf(const cmag_params& P, const float4& pi, const Cell& gp,
                                                const Cells& cells, const float4* __restrict__ pos, C&& cand,
                                                uint32_t part = 0) {
    if constexpr (Cells::SUB) {
        walk_rows<DIM, HASH, PERIODIC, FORCE_ORDER, LANES>(P, pi, gp, cells,
                                                    [&](const Run& a, const Run& b, float py, float pz, bool) {
            walk_run_sub(pos, a.s, a.s + a.len, a.px, py, pz, a.code, cand);
            walk_run_sub(pos, b.s, b.s + b.len, b.px, py, pz, b.code, cand);
        }, part);
        return;
    }
    walk_rows<DIM, HASH, PERIODIC, false, LANES>(P, pi, gp, cells,
                                                 [&](const Run& a, const Run& b, float py, float pz, bool) {
        walk_row_pf<Cells::PADDED>(a, b, py, pz, pos, cand);
    }, part);
}

// ---- cell lookups staged in LDS (sub-cell walk) -----------------------------
// A block whose targets lie in one row of cells along x, or in two rows (the
// end of one and the start of the next in key order), with each row's stencil
// x-range [cx0 - 1, cx1 + 1] inside the grid, on consecutive keys and at most
// LK_W cells wide (both rows together when there are two), copies the compact offsets
// and eighth counts of those cells in the 9 (2-D: 3) stencil rows of each of
// its rows into LDS once; its targets then find their runs there instead of
// with five loads per stencil row.  The runs and their order are the global
// walk's, so the sums are the same bit for bit.
constexpr int LK_W = 32;

struct LookupPlan {
    uint32_t row[2];    // each part's row of cells: the key without its x bits
    uint32_t x0[2];     // x bits of the key of the part's first target
    uint32_t width[2];  // cells per stencil row segment
    int parts;          // 0: not staged, 1 or 2 rows
};

// part p (width w_p) keeps its stencil rows r at first[f_p + r * (w_p + 1) + c]
// and pre[q_p + r * w_p + c]: f_0 = q_0 = 0, part 1 after part 0 (f_1 =
// R (w_0 + 1), q_1 = R w_0); w_0 + w_1 <= LK_W
struct LookupTables {
    uint32_t first[18 * (LK_W / 2 + 1)];
    uint4 pre[9 * LK_W];
};

// a target's view of the staged tables: entries from its cell x - 1 on, per
// stencil row
struct LookupView {
    const uint32_t* first;
    const uint4* pre;
    uint32_t fs, ps;
    __device__ __forceinline__ uint32_t F(int r, uint32_t c) const { return first[(uint32_t)r * fs + c]; }
    __device__ __forceinline__ const uint4* Pr(int r, uint32_t c) const { return pre + (uint32_t)r * ps + c; }
};

// the bits of each axis in a cell key; the linear order's are fields, so its
// keys step by dilated_inc / dilated_dec too
struct KeyMasks {
    uint32_t x, y, z;
};
template <int HASH>
__device__ __forceinline__ KeyMasks key_masks(const cmag_params& P) {
    if (HASH == CMAG_HASH_MORTON) return KeyMasks{P.morton_mask[0], P.morton_mask[1], P.morton_mask[2]};
    const uint32_t bx = P.grid_bits[0], by = P.grid_bits[1];
    return KeyMasks{P.grid_size[0] - 1u, (P.grid_size[1] - 1u) << bx, (P.grid_size[2] - 1u) << (bx + by)};
}

// the view of a target whose cell has this key
template <int DIM>
__device__ __forceinline__ LookupView lookup_view(const LookupPlan& lp, const LookupTables& lt, uint32_t key,
                                                  uint32_t xmask) {
    constexpr int R = DIM == 3 ? 9 : 3;
    const int part = (lp.parts == 2 && (key & ~xmask) == lp.row[1]) ? 1 : 0;
    const uint32_t w0 = lp.width[0], w = part ? lp.width[1] : w0;
    const uint32_t dx = (key & xmask) - lp.x0[part];  // consecutive keys: cells
    LookupView v;
    v.fs = w + 1u;
    v.ps = w;
    v.first = lt.first + (part ? (uint32_t)R * (w0 + 1u) : 0u) + dx;
    v.pre = lt.pre + (part ? (uint32_t)R * w0 : 0u) + dx;
    return v;
}

// All threads of the block (whole waves, at most four) call this for its
// targets b0, b0 + 1, ... (at most one a thread); returns whether the block's
// lookups are staged.  keys: the sorted cell keys (a sub-cell row lies in the same cell as
// the reference-order row of its number).  Everything is found from the keys'
// bits by every thread at once: one barrier and one pass of loads until the
// tables are filled.  (When one thread worked out the block's 22 keys from
// positions, with a division per coordinate and a bit deposit per key, that
// chain was a tenth of a block's life.)
template <int DIM, int HASH>
__device__ __forceinline__ bool stage_lookups(const cmag_params& P, const uint32_t* __restrict__ keys,
                                              const SubCells& cells, uint32_t n, uint32_t b0, uint32_t targets,
                                              LookupPlan& lp, LookupTables& lt) {
    constexpr int R = DIM == 3 ? 9 : 3;
    if (P.cellcount != 1 || b0 >= n) return false;
    const KeyMasks M = key_masks<HASH>(P);
    const uint32_t count = min(targets, n - b0);
    const uint32_t tid = threadIdx.x;
    const uint32_t mine = keys[b0 + min(tid, count - 1u)];
    const uint32_t k0 = keys[b0], k1 = keys[b0 + count - 1u];
    const uint32_t rowa = k0 & ~M.x, rowb = k1 & ~M.x;
    const uint32_t prev = tid == 0 ? k0 : keys[b0 + min(tid, count) - 1u];
    // the only step between rows that may occur is one from the first target's
    // to the last target's
    const bool step = (prev & ~M.x) != (mine & ~M.x);
    __shared__ uint32_t split_key[2];  // x bits of the last target of part 0, the first of part 1
    if (step) {
        split_key[0] = prev & M.x;
        split_key[1] = mine & M.x;
    }
    __shared__ uint32_t bad_step[256 / 64];
    const uint64_t bad = __ballot(step && ((prev & ~M.x) != rowa || (mine & ~M.x) != rowb));
    if ((tid & 63u) == 0u) bad_step[tid >> 6] = bad != 0u ? 1u : 0u;
    __syncthreads();
    for (uint32_t w = 0; w < blockDim.x >> 6; ++w)
        if (bad_step[w]) return false;
    const int parts = rowa == rowb ? 1 : 2;
    // cells x - 1 of the part's first target to x + 1 of its last: inside the
    // grid and on consecutive keys (x bits that are the key's lowest)
    auto part_width = [&](uint32_t a, uint32_t b) -> uint32_t {
        if (a == 0u || b == M.x) return 0u;
        const uint32_t lo = dilated_dec(a, M.x), hi = dilated_inc(b, M.x);
        const uint32_t low = M.x & ~(M.x + 1u);  // the run of ones at the bottom
        if (((lo ^ hi) & ~low) != 0u) return 0u;
        const uint32_t w = hi - lo + 1u;
        return w <= (uint32_t)LK_W ? w : 0u;
    };
    const uint32_t xa = k0 & M.x, xb = parts == 2 ? split_key[1] : 0u;
    const uint32_t w0 = part_width(xa, parts == 2 ? split_key[0] : k1 & M.x);
    const uint32_t w1 = parts == 2 ? part_width(xb, k1 & M.x) : 0u;
    if (w0 == 0u || (parts == 2 && w1 == 0u) || w0 + w1 > (uint32_t)LK_W) return false;
    if (tid == 0) {
        lp.row[0] = rowa;
        lp.row[1] = rowb;
        lp.x0[0] = xa;
        lp.x0[1] = xb;
        lp.width[0] = w0;
        lp.width[1] = w1;
        lp.parts = parts;
    }
    // part 0's entries first, then part 1's; entry t of first[] is t
    const uint32_t n0 = (uint32_t)R * (w0 + 1u), total = n0 + (parts == 2 ? (uint32_t)R * (w1 + 1u) : 0u);
    for (uint32_t t = tid; t < total; t += blockDim.x) {
        const uint32_t pt = t >= n0 ? 1u : 0u, loc = pt ? t - n0 : t, w = pt ? w1 : w0;
        const uint32_t r = loc / (w + 1u), c = loc - r * (w + 1u);
        const uint32_t rk = pt ? rowb : rowa;
        uint32_t ky = rk & M.y, kz = rk & M.z;
        const uint32_t iy = r % 3u, iz = DIM == 3 ? r / 3u : 1u;
        if (iy == 0u) ky = dilated_dec(ky, M.y);
        else if (iy == 2u) ky = dilated_inc(ky, M.y);
        if (iz == 0u) kz = dilated_dec(kz, M.z);
        else if (iz == 2u) kz = dilated_inc(kz, M.z);
        const uint32_t key = (ky | kz | dilated_dec(pt ? xb : xa, M.x)) + c;
        lt.first[t] = cells.first[key];
        if (c < w) lt.pre[(pt ? (uint32_t)R * w0 : 0u) + r * w + c] = cells.pre[key];
    }
    __syncthreads();
    return true;
}

// The density pass also stages candidate rows: after the lookups, the
// positions of the rows of four stencil rows of cells (r = 3..6: the three of
// dz = 0 and the first of dz = +1 in 3-D), up to ROW_STAGE_CAP rows, are copied
// into LDS (12 B a row, 16 KB) and read from there.
// 16 KB keeps seven blocks per CU; more rows cost more in occupancy than they
// save in loads.  A row's 12 bytes lie together, so one address serves a
// candidate.  The force pass stages none: its lanes read one row each, at
// unlike places, and the copies cost it waves.
constexpr int ROW_STAGE_FIRST = 3, ROW_STAGE_ROWS = 4, ROW_STAGE_CAP = 1365;

struct RowStage {
    int32_t off[ROW_STAGE_ROWS];  // LDS row of sorted row j of staged stencil row r: j + off
    int ok;
};

// ROW_STAGE_CAP + 1 rows: the walk reads one row past a run.  12 bytes a row,
// together, so that one address serves a candidate
struct RowLds {
    struct Row {
        float x, y, z;
    };
    Row row[ROW_STAGE_CAP + 1];
};

// all threads of a staged block call this after stage_lookups
template <int DIM>
__device__ __forceinline__ void stage_rows(const LookupPlan& lp, const LookupTables& lt,
                                           const float4* __restrict__ pos, RowLds& lds, RowStage& rs) {
    // blocks staged over one row of cells only (its rows are at stride width + 1)
    const uint32_t FS = lp.width[0] + 1u;
    if (threadIdx.x == 0) {
        int32_t tot = 0;
        for (int k = 0; k < ROW_STAGE_ROWS; ++k) {
            const uint32_t r = (uint32_t)(ROW_STAGE_FIRST + k);
            const uint32_t s = lt.first[r * FS], e = lt.first[r * FS + lp.width[0]];
            rs.off[k] = tot - (int32_t)s;
            tot += (int32_t)(e - s);
        }
        rs.ok = DIM == 3 && lp.parts == 1 && tot <= ROW_STAGE_CAP;
    }
    __syncthreads();
    if (!rs.ok) return;
    for (int k = 0; k < ROW_STAGE_ROWS; ++k) {
        const uint32_t r = (uint32_t)(ROW_STAGE_FIRST + k);
        const uint32_t s = lt.first[r * FS], e = lt.first[r * FS + lp.width[0]];
        const int32_t d0 = (int32_t)s + rs.off[k];
        for (uint32_t t = threadIdx.x; t < e - s; t += blockDim.x) {
            const float4 v = pos[s + t];
            lds.row[d0 + t] = RowLds::Row{v.x, v.y, v.z};
        }
    }
    __syncthreads();
}

// the candidates of target pi through its view of the staged
// lookups, as walk_stencil_pf hands them; with ROWS, the stencil rows that
// stage_rows copied are read from LDS; with FORCE_ORDER, rows in force_rows order
template <int DIM, bool ROWS = false, bool FORCE_ORDER = false, int LANES = 1, typename C>
__device__ __forceinline__ void walk_lookup(const cmag_params& P, const float4& pi, const LookupView& v,
                                            const float4* __restrict__ pos, C&& cand, const RowStage* rs = nullptr,
                                            const RowLds* lds = nullptr, uint32_t part = 0) {
    constexpr int R = DIM == 3 ? 9 : 3;
    const int q = x_sub(P, pi.x);
    auto run_lds = [&](uint32_t s, uint32_t e, int32_t off) {
        for (uint32_t j = s; j < e; j += 2u) {
            const int32_t l = (int32_t)j + off;  // in [0, staged rows]
            const RowLds::Row a0 = lds->row[l], a1 = lds->row[l + 1];
            const float4 p0 = make_float4(a0.x, a0.y, a0.z, 0.0f);
            const float4 p1 = make_float4(a1.x, a1.y, a1.z, 0.0f);
            cand(j, p0, true, pi.x, pi.y, pi.z, 13);
            cand(j + 1u, p1, j + 1u < e, pi.x, pi.y, pi.z, 13);
        }
    };
    const RowList list = force_rows<LANES>(DIM, part);
    const int k0 = FORCE_ORDER ? 0 : (int)part, k1 = FORCE_ORDER ? list.count : R;
    for (int k = k0; k < k1; k += FORCE_ORDER ? 1 : LANES) {
        const int r = FORCE_ORDER ? list[k] : k;
        const uint32_t s = v.F(r, 0) + SubCells::below(v.Pr(r, 0), q);
        const uint32_t f1 = v.F(r, 2);
        const uint4* c1 = v.Pr(r, 2);
        const uint32_t e = f1 + SubCells::through(c1, q), ws = f1 + SubCells::fluid(c1), we = v.F(r, 3);
        if (ROWS && rs->ok && r >= ROW_STAGE_FIRST && r < ROW_STAGE_FIRST + ROW_STAGE_ROWS) {
            run_lds(s, e, rs->off[r - ROW_STAGE_FIRST]);
            run_lds(ws, we, rs->off[r - ROW_STAGE_FIRST]);
        } else {
            walk_run_sub(pos, s, e, pi.x, pi.y, pi.z, 13, cand);
            walk_run_sub(pos, ws, we, pi.x, pi.y, pi.z, 13, cand);
        }
    }
}

// ---- in-range masks (staged blocks of the sub-cell walk) ---------------------
// The density pass tests every candidate of a staged block anyway; it leaves,
// per target and stencil row r, a 64-bit mask of which fluid candidates of the
// row's main run [s, e) lie within 2h (r^2 < 4h^2, the force pass's own test
// on the same float operations; the walls in the run, which are those of its
// first two cells, are cleared).  The force pass then pushes the row's in-range
// fluid neighbours straight from the mask, in the walk's order, without loading
// or testing those candidates, and walks the walls apart.  Masks are stored
// row-major, [r][target] (uint2: low word first); a row whose run is longer
// than MASK_BITS is walked as before.
// Layout: two words, bit t of the first for candidate t < 32 of the run, bit t
// of the second for candidate 32 + t.  The scan takes the run's candidates in
// pairs, the first 32 into one word, the rest into the other: a subtraction and
// a funnel shift a candidate, and one more a pair (shift_in_less below).  (One
// 64-bit word shifted by two bits a pair took four and a half instructions a
// candidate, of which v_lshlrev_b64 and the selects most.)
constexpr int MASK_BITS = 64;
constexpr int MASK_ROWS = 9;

// bits [lo, hi), hi <= 64
__device__ __forceinline__ uint64_t mask_bits(uint32_t lo, uint32_t hi) {
    if (hi <= lo) return 0ull;
    const uint32_t len = hi - lo;
    return (len >= 64u ? ~0ull : (1ull << len) - 1ull) << lo;
}

// m shifted left, with the bit a < b below (a >= 0 or NaN): the sign of |a| - b,
// which is exact, and 0 for a NaN; a subtraction and a funnel shift, without
// the wait a comparison's mask needs before it can be read
__device__ __forceinline__ uint32_t shift_in_less(uint32_t m, float a, float b) {
    return __builtin_amdgcn_alignbit(m, __float_as_uint(__builtin_fabsf(a) - b), 31u);
}

// density of the target pi over a staged block's lookups, as
// density_sum_lookup, writing the in-range masks of its rows' main runs to
// masks[r * stride + i] (fluid targets only)
template <int DIM, int LANES>
__device__ __forceinline__ float density_sum_masks(const cmag_params& P, const float4& pi, const LookupView& v,
                                                   const RowStage* rs, const RowLds* lds,
                                                   const float4* __restrict__ pos, uint2* __restrict__ masks,
                                                   uint32_t i, uint32_t stride, uint32_t part) {
    constexpr int R = DIM == 3 ? 9 : 3;
    const int q = x_sub(P, pi.x);
    const float half_inv_h = -0.5f / P.smoothing_radius;
    const float r2max = 4.0f * P.smoothing_radius * P.smoothing_radius;
    // the force pass reads the masks of fluid targets only
    const bool fluid = pi.w == CMAG_DB_FLUID;
    float sum = 0.0f;
    auto term = [&](float r2) {
        const float t = fminf(fmaxf(fmaf(half_inv_h, fsqrt(r2), 1.0f), 0.0f), 1.0f);
        const float t2 = t * t;
        sum = fmaf(t2 * t2, fmaf(-4.0f, t, 5.0f), sum);
    };
    auto d2 = [&](const float4& pj) { return norm2(pi.x - pj.x, pi.y - pj.y, pi.z - pj.z); };
    auto cand = [&](uint32_t, const float4& pj, bool valid, float, float, float, int) {
        term(valid ? d2(pj) : 1e30f);
    };
    for (int r = (int)part; r < R; r += LANES) {
        const uint4* c0 = v.Pr(r, 0);
        const uint32_t f0 = v.F(r, 0);
        const uint32_t s = f0 + SubCells::below(c0, q);
        const uint32_t f1 = v.F(r, 2);
        const uint4* c1 = v.Pr(r, 2);
        const uint32_t e = f1 + SubCells::through(c1, q), ws = f1 + SubCells::fluid(c1), we = v.F(r, 3);
        uint32_t m0 = 0, m1 = 0;
        const bool in_lds = DIM == 3 && LANES == 1 && rs->ok && r >= ROW_STAGE_FIRST && r < ROW_STAGE_FIRST + ROW_STAGE_ROWS;
        // two candidates per step; `at` steps through the run by `row` a candidate
        auto scan = [&](auto at, auto row, auto&& ld) {
            const auto end = at + (e - s) * row, last = end - row;
            auto bits = [&](float ra, float rb) {
                m1 = __builtin_amdgcn_alignbit(m1, m0, 30u);
                m0 = shift_in_less(shift_in_less(m0, ra, r2max), rb, r2max);
            };
            // four at a time, then two
            for (; at + 2u * row < end; at += 4u * row) {
                float4 p0, p1, p2, p3;
                ld(at, p0, p1);
                ld(at + 2u * row, p2, p3);
                const float ra = d2(p0), rb = d2(p1), rc = d2(p2);
                const float rd = at + 2u * row < last ? d2(p3) : 1e30f;
                term(ra);
                term(rb);
                term(rc);
                term(rd);
                bits(ra, rb);
                bits(rc, rd);
            }
            if (at < end) {
                float4 p0, p1;
                ld(at, p0, p1);
                const float ra = d2(p0);
                const float rb = at < last ? d2(p1) : 1e30f;
                term(ra);
                term(rb);
                bits(ra, rb);
            }
        };
        if (in_lds) {
            scan(lds->row + ((int32_t)s + rs->off[r - ROW_STAGE_FIRST]), 1u,
                 [&](const RowLds::Row* q, float4& p0, float4& p1) {
                     p0 = make_float4(q[0].x, q[0].y, q[0].z, 0.0f);
                     p1 = make_float4(q[1].x, q[1].y, q[1].z, 0.0f);
                 });
        } else {
            scan(s << 4, 16u, [&](uint32_t off, float4& p0, float4& p1) {
                const char* base = reinterpret_cast<const char*>(pos);
                const RowLds::Row a = *reinterpret_cast<const RowLds::Row*>(base + off);
                const RowLds::Row b = *reinterpret_cast<const RowLds::Row*>(base + (off + 16u));
                p0 = make_float4(a.x, a.y, a.z, 0.0f);
                p1 = make_float4(b.x, b.y, b.z, 0.0f);
            });
        }
        // candidate t of K was shifted in K - 1 - t places from the right of m1:m0
        const uint32_t len = e > s ? e - s : 0u, K = min((len + 1u) & ~1u, (uint32_t)MASK_BITS);
        const uint64_t m = K ? __builtin_bitreverse64((uint64_t)m1 << 32 | m0) >> (64u - K) : 0ull;
        uint32_t lo = (uint32_t)m, hi = (uint32_t)(m >> 32);
        // the walls of the run's first two cells are walked by the force pass
        // (every wall of the stencil acts): their bits are cleared
        const uint32_t fx = v.F(r, 1), cxw = SubCells::fluid(v.Pr(r, 1));
        if ((f1 - f0) - SubCells::fluid(c0) - cxw != 0u && len <= (uint32_t)MASK_BITS) {
            const uint64_t w = mask_bits(f0 + SubCells::fluid(c0) - s, fx - s) | mask_bits(fx + cxw - s, f1 - s);
            lo &= ~(uint32_t)w;
            hi &= ~(uint32_t)(w >> 32);
        }
        if (fluid) masks[(size_t)r * stride + i] = make_uint2(lo, hi);
        if (in_lds) {
            const int32_t off = rs->off[r - ROW_STAGE_FIRST];
            for (uint32_t j = ws; j < we; j += 2u) {
                const int32_t l = (int32_t)j + off;
                const RowLds::Row a0 = lds->row[l], a1 = lds->row[l + 1];
                cand(j, make_float4(a0.x, a0.y, a0.z, 0.0f), true, 0.f, 0.f, 0.f, 13);
                cand(j + 1u, make_float4(a1.x, a1.y, a1.z, 0.0f), j + 1u < we, 0.f, 0.f, 0.f, 13);
            }
        } else {
            walk_run_sub(pos, ws, we, pi.x, pi.y, pi.z, 13, cand);
        }
    }
    if (LANES > 1) sum = quad_sum(sum);
    return sum * P.kernel_coeff * P.particle_mass;
}

// queue depth and drain size (compile-time; -D overrides for tuning builds)
#ifndef CMAG_NB_CAP
#define CMAG_NB_CAP 16
#endif
#ifndef CMAG_NB_DRAIN
#define CMAG_NB_DRAIN 2
#endif
constexpr int NB_CAP = CMAG_NB_CAP;
constexpr int NB_SHIFT_BITS = 27;  // entry = j | (image-shift code << 27)

struct NbEntry {
    __device__ static __forceinline__ uint32_t pack(uint32_t j, int code) {
        return j | ((uint32_t)code << NB_SHIFT_BITS);
    }
    __device__ static __forceinline__ uint32_t index(uint32_t e) { return e & ((1u << NB_SHIFT_BITS) - 1u); }
    __device__ static __forceinline__ int code(uint32_t e) { return (int)(e >> NB_SHIFT_BITS); }
};

// A per-lane queue of CAP (a power of two) neighbour entries in LDS, one
// [CAP][64] block per wave.  Entries leave in the order they came, so pair
// terms are summed in walk order whatever the queue depth and drain sizes.
// The walk pushes; when any lane's queue is full every active lane drains its
// NB_DRAIN oldest entries (fewer if it has fewer), which keeps all lanes busy
// in the pair loop instead of waiting for the fullest one; a final drain
// empties the queues.  push() has no room check: every site that pushes
// leaves each queue below CAP before the next site may push.
constexpr int NB_DRAIN = CMAG_NB_DRAIN;

template <int CAP>
struct NbQueue {
    static_assert((CAP & (CAP - 1)) == 0 && CAP >= 2, "queue depth: a power of two");
    uint32_t (*q)[64];
    int lane;
    int head = 0, count = 0;
    __device__ __forceinline__ NbQueue(uint32_t (*q_)[64], int lane_) : q(q_), lane(lane_) {}
    __device__ __forceinline__ void push(uint32_t e) {
        q[(head + count) & (CAP - 1)][lane] = e;
        ++count;
    }
    __device__ __forceinline__ bool full() const { return count == CAP; }
    // f(e0, e1, second): the oldest entries two at a time; a lane with an odd
    // number left repeats its last entry with second = false (contributing
    // nothing), so both entries' rows can be loaded before either is used
    template <typename F>
    __device__ __forceinline__ void drain(int upto, F&& f) {
        for (int k = 0; k < upto; k += 2) {
            if (k >= count) break;
            const uint32_t e0 = q[(head + k) & (CAP - 1)][lane];
            const uint32_t e1 = q[(head + min(k + 1, count - 1)) & (CAP - 1)][lane];
            f(e0, e1, k + 1 < count);
        }
        const int d = min(upto, count);
        head = (head + d) & (CAP - 1);
        count -= d;
    }
};

// ---------------------------------------------------------------------------
// the density of the particle at pi: the mass-weighted kernel sum over the
// stencil (the particle itself included)
template <int SYS, int DIM, int HASH, int LANES = 1, typename Cells>
__device__ __forceinline__ float density_sum(const cmag_params& P, const float4& pi,
                                             const float4* __restrict__ sortedPos, const Cells& cells,
                                             uint32_t part = 0) {
    const Cell gp = grid_pos(P, pi.x, pi.y, pi.z);
    const float half_inv_h = -0.5f / P.smoothing_radius;
    float sum = 0.0f;
    walk_stencil_pf<DIM, HASH, SYS != CMAG_SYS_DAMBREAK, false, LANES>(P, pi, gp, cells, sortedPos,
                                                         [&](uint32_t, const float4& pj, bool valid, float px,
                                                             float py, float pz, int) {
        // a candidate past the run sits at r^2 = 1e30: t = 0 and it adds +0
        const float r2 = valid ? norm2(px - pj.x, py - pj.y, pz - pj.z) : 1e30f;
        // t = 1 - q/2 with q = r/h, clamped at 0 (nothing beyond 2h, no
        // branch); 1 - q/2 <= 1, so the clamp to [0, 1] is max(0, .) and folds
        // into the fma.  (1 - q/2)^4 (2q + 1) = t^4 (5 - 4t)
        const float t = fminf(fmaxf(fmaf(half_inv_h, fsqrt(r2), 1.0f), 0.0f), 1.0f);
        const float t2 = t * t;
        sum = fmaf(t2 * t2, fmaf(-4.0f, t, 5.0f), sum);
    }, part);
    if (LANES > 1) sum = quad_sum(sum);
    return sum * P.kernel_coeff * P.particle_mass;
}

template <int DIM, int LANES>
__device__ __forceinline__ float density_sum_lookup(const cmag_params& P, const float4& pi, const LookupView& v,
                                                    const RowStage* rs, const RowLds* lds,
                                                    const float4* __restrict__ pos, uint32_t part) {
    const float half_inv_h = -0.5f / P.smoothing_radius;
    float sum = 0.0f;
    walk_lookup<DIM, LANES == 1, false, LANES>(P, pi, v, pos,
                           [&](uint32_t, const float4& pj, bool valid, float px, float py, float pz, int) {
        const float r2 = valid ? norm2(px - pj.x, py - pj.y, pz - pj.z) : 1e30f;
        const float t = fminf(fmaxf(fmaf(half_inv_h, fsqrt(r2), 1.0f), 0.0f), 1.0f);
        const float t2 = t * t;
        sum = fmaf(t2 * t2, fmaf(-4.0f, t, 5.0f), sum);
    }, rs, lds, part);
    if (LANES > 1) sum = quad_sum(sum);
    return sum * P.kernel_coeff * P.particle_mass;
}

// ---- in-range masks of the 2-D channel passes ---------------------------------
// The density pass tests every candidate; for each target and stencil row that
// walk_rows hands out whole it keeps a 32-bit mask, bit t set when candidate t of
// the row lies within 2h (r^2 < 4h^2, the force pass's own test on the same
// float operations).  The force pass then queues the set bits' candidates, in
// the walk's order, without loading or testing the others: about 21 (h = 1.3
// spacings) or 28 (h = 1.5) of 49 on cells of one spacing.  A row of more than
// 32 candidates is walked.  Layout [row][target], 4 bytes, coalesced; both
// passes map targets to lanes alike, so a wave that gets its rows whole in one
// gets them whole in the other.
constexpr int ROW_MASK_BITS = 32;

// density_sum over whole rows two candidates at a time; with masks, leaving
// the rows' in-range masks at masks[row * stride + i]
template <int SYS, int DIM, int HASH, bool MASKS, typename Cells>
__device__ __forceinline__ float density_sum_rows(const cmag_params& P, const float4& pi,
                                                  const float4* __restrict__ sortedPos, const Cells& cells,
                                                  uint32_t* __restrict__ masks, uint32_t i, uint32_t stride) {
    const Cell gp = grid_pos(P, pi.x, pi.y, pi.z);
    const float half_inv_h = -0.5f / P.smoothing_radius;
    const float r2max = 4.0f * P.smoothing_radius * P.smoothing_radius;
    float sum = 0.0f, total_sum = 0.0f;
    uint32_t* out = MASKS ? masks + i : nullptr;
    walk_rows<DIM, HASH, SYS != CMAG_SYS_DAMBREAK>(P, pi, gp, cells,
                                                   [&](const Run& a, const Run& b, float py, float pz, bool whole) {
        uint32_t m = 0;
        walk_row_two(a, b, sortedPos, [&](const float4& p0, float px0, const float4& p1, float px1, bool valid1) {
            auto term = [&](float r2) {
                const float t = fminf(fmaxf(fmaf(half_inv_h, fsqrt(r2), 1.0f), 0.0f), 1.0f);
                const float t2 = t * t;
                sum = fmaf(t2 * t2, fmaf(-4.0f, t, 5.0f), sum);
            };
            const float ra = norm2(px0 - p0.x, py - p0.y, pz - p0.z);
            const float rb = valid1 ? norm2(px1 - p1.x, py - p1.y, pz - p1.z) : 1e30f;
            term(ra);
            term(rb);
            if (MASKS) {
                m = shift_in_less(m, ra, r2max);
                m = shift_in_less(m, rb, r2max);
            }
        });
        // the dam break's 100 to 500 candidates a target: a sum per row, as the
        // lanes of a shared target form them, keeps the error at a row's
        if (SYS == CMAG_SYS_DAMBREAK) {
            total_sum += sum;
            sum = 0.0f;
        }
        if (MASKS && whole) {
            // candidate t was shifted in K - 1 - t places from the right, K even
            const uint32_t total = a.len + b.len, K = (total + 1u) & ~1u;
            if (total != 0u && total <= (uint32_t)ROW_MASK_BITS) *out = __brev(m) >> (32u - K);
            else *out = 0u;
            out += stride;
        }
    });
    if (SYS == CMAG_SYS_DAMBREAK) sum = total_sum;
    return sum * P.kernel_coeff * P.particle_mass;
}

// pairs (optional): what a neighbour's pair terms need of the density pass,
// (p / rho, 1 / rho) in the reciprocal the terms use; masks (optional): as above
template <int SYS, int DIM, int HASH, int LANES = 1, typename Cells>
__device__ __forceinline__ void density_body(const cmag_params& P, uint32_t i, float4* __restrict__ measures,
                                             const float4* __restrict__ sortedPos, const Cells& cells,
                                             float2* __restrict__ pairs = nullptr,
                                             uint32_t* __restrict__ masks = nullptr, uint32_t stride = 0,
                                             uint32_t part = 0) {
    const float4 pi = sortedPos[i];
    float2* m2 = reinterpret_cast<float2*>(measures);
    const bool rest = SYS == CMAG_SYS_POISEUILLE && pi.w == CMAG_PO_WALL;
    float dens = 0.0f;
    if constexpr (Cells::PADDED && !Cells::SUB) {
        // with masks a wall walks too: the force pass takes it as a target
        if (SYS != CMAG_SYS_DAMBREAK && DIM == 2 && HASH == CMAG_HASH_LINEAR && masks)
            dens = density_sum_rows<SYS, DIM, HASH, true>(P, pi, sortedPos, cells, masks, i, stride);
        else if (!rest)
            dens = density_sum_rows<SYS, DIM, HASH, false>(P, pi, sortedPos, cells, nullptr, i, stride);
    } else {
        if (!rest) dens = density_sum<SYS, DIM, HASH, LANES>(P, pi, sortedPos, cells, part);
    }
    if (LANES > 1 && part != 0) return;
    if (rest) dens = P.rest_density;
    const float p = eos(P, dens);
    if (SYS == CMAG_SYS_PERISTALSIS) {
        measures[i] = make_float4(dens, p, 0.0f, pi.w);
    } else {
        m2[2 * (size_t)i] = make_float2(dens, p);
    }
    if (SYS != CMAG_SYS_DAMBREAK && pairs) {
        const float inv = frcp(dens);
        pairs[i] = make_float2(p * inv, inv);
    }
}

// getVelocityDiff, poiseuilleFlowKernel.cu:184-208
__device__ __forceinline__ float3 vel_diff_poiseuille(const cmag_params& P, const float4& vi,
                                                      const float4& pi, const float4& vj,
                                                      const float4& pj) {
    if (pj.w == CMAG_PO_WALL && pj.y > P.wall_top) {
        float beta = fminf(P.beta_max, 1.0f + (pj.y - P.wall_top) / (P.wall_top - pi.y));
        return make_float3(beta * vi.x, beta * vi.y, beta * vi.z);
    }
    if (pj.w == CMAG_PO_WALL && pj.y < P.wall_bottom) {
        float beta = fminf(P.beta_max, 1.0f + (P.wall_bottom - pj.y) / (pi.y - P.wall_bottom));
        return make_float3(beta * vi.x, beta * vi.y, beta * vi.z);
    }
    return make_float3(vi.x - vj.x, vi.y - vj.y, vi.z - vj.z);
}

// target position minus the periodic image offset named by code, computed with
// the same float operations as walk_stencil
template <bool PERIODIC = true>
__device__ __forceinline__ float3 image_target(const cmag_params& P, const float4& pi, int code) {
    if (!PERIODIC) return make_float3(pi.x, pi.y, pi.z);
    if ((P.periodic_mask & 6) == 0)  // images along x only: code = 13 + sx
        return make_float3((P.periodic_mask & 1) ? pi.x - (float)(code - 13) * P.world_size[0] : pi.x, pi.y, pi.z);
    const int sx = code % 3 - 1, sy = (code / 3) % 3 - 1, sz = code / 9 - 1;
    float3 q;
    q.x = (P.periodic_mask & 1) ? pi.x - (float)sx * P.world_size[0] : pi.x;
    q.y = (P.periodic_mask & 2) ? pi.y - (float)sy * P.world_size[1] : pi.y;
    q.z = (P.periodic_mask & 4) ? pi.z - (float)sz * P.world_size[2] : pi.z;
    return q;
}

// ---- fused force (DamBreak, Poiseuille) -------------------------------------------
// Per-target state of the force sum.  Pair terms accumulate in f in walk
// order; DamBreak's wall terms go to w as they are met, and f + w is formed
// once at the end, so the result does not depend on how the neighbours were
// staged (list depth, which particles share the wave, lists from the density
// pass).

// the DamBreak pair terms' common factor (ForceSum::pair_db), 5 m gc / (2h)
__device__ __forceinline__ float db_scale(const cmag_params& P) {
    return 2.5f * P.particle_mass * P.grad_coeff / P.smoothing_radius;
}

template <int SYS>
struct ForceSum {
    const cmag_params& P;
    float4 pi, vi;
    float dens, inv_dens, pterm_i, inv_h, m, gc, av_c, av_eps, visc_k, t_k, cterm_i;
    float fx = 0.f, fy = 0.f, fz = 0.f, wx = 0.f, wy = 0.f, wz = 0.f;

    // rho, pterm: the target's density and p / rho^2 (DamBreak: times db_scale)
    __device__ __forceinline__ ForceSum(const cmag_params& P_, const float4& pi_, const float4& vi_, float rho,
                                        float pterm)
        : P(P_), pi(pi_), vi(vi_) {
        dens = rho;
        inv_dens = 1.0f / dens;
        pterm_i = pterm;
        const float h = P.smoothing_radius;
        inv_h = 1.0f / h;
        m = P.particle_mass;
        gc = P.grad_coeff;
        cterm_i = pterm;
        av_c = -2.0f * P.alpha * h * P.soundspeed * db_scale(P);  // of nu * (rho_i + rho_j)
        av_eps = 0.001f * h * h;
        visc_k = m * (P.mu + P.mu);
        t_k = -0.5f * inv_h;
    }

    // Lennard-Jones wall term (DamBreak), fluid_kernel.cu:199-208
    __device__ __forceinline__ void wall(float rx, float ry, float rz, float r2) {
        const float inv_d = frsq(r2);
        const float ad = P.lj_a * inv_d;
        const float ad2 = ad * ad;
        const float ad6 = ad2 * ad2 * ad2;
        const float sc = P.lj_D * (ad6 * ad6 - ad6) * (inv_d * inv_d);
        wx = fmaf(sc, rx, wx); wy = fmaf(sc, ry, wy); wz = fmaf(sc, rz, wz);
    }

    // DamBreak pressure + artificial viscosity of an in-range fluid neighbour
    // (fluid_kernel.cu:210-262) with density rho_j and cp_j = db_scale p_j /
    // rho_j^2.  With t = 1 - q/2 the kernel gradient over the distance,
    // ((1-q/2)^4 - (1-q/2)^3 (2q+1)) / d = 5 t^3 (t - 1) / d, is -5 t^3 / (2h), so
    // with the -m gc factors it is db_scale t^3, and db_scale is folded into
    // the pressure and viscosity terms ahead of the pairs.  The viscosity
    // term is branch-free (min(v.r, 0) makes it +0 for separating pairs), which
    // also keeps rho_j's load with the rest of its row.  One reciprocal square
    // root and one reciprocal per pair.  valid = false adds +0 (the term is
    // computed and dropped: a skipped term would move its row loads into a
    // branch).  28 VALU instructions; with the gradient as 5 t^3 (t - 1) and the
    // constants in the pair it was 33.
    __device__ __forceinline__ void pair_db(const float3& q, const float4& pj, const float4& vj, float rho_j,
                                            float cp_j, bool valid = true) {
        const float rx = q.x - pj.x, ry = q.y - pj.y, rz = q.z - pj.z;
        const float r2 = norm2(rx, ry, rz);
        const float t = fmaf(t_k, r2 * frsq(r2), 1.0f);
        const float vr = fmaf(vi.z - vj.z, rz, fmaf(vi.y - vj.y, ry, (vi.x - vj.x) * rx));
        const float av = fminf(vr, 0.0f) * frcp((dens + rho_j) * (r2 + av_eps));
        const float s = fmaf(av_c, av, cterm_i + cp_j);
        const float k = s * (t * t * t);
        const float kk = valid ? k : 0.0f;
        fx = fmaf(kk, rx, fx); fy = fmaf(kk, ry, fy); fz = fmaf(kk, rz, fz);
    }

    // Poiseuille pressure + Morris viscosity of an in-range neighbour
    // (poiseuilleFlowKernel.cu:184-270); mj = (p_j / rho_j, 1 / rho_j); one
    // reciprocal square root per pair; valid = false adds nothing
    __device__ __forceinline__ void pair(const float3& q, const float4& pj, const float2& mj, const float4& vj,
                                         bool valid = true) {
        const float rx = q.x - pj.x, ry = q.y - pj.y, rz = q.z - pj.z;
        const float r2 = norm2(rx, ry, rz);
        const float inv_d = frsq(r2);
        const float dist = r2 * inv_d;
        const float qq = dist * inv_h;
        const float t = fmaf(-0.5f, qq, 1.0f);
        const float t2 = t * t;
        const float temp = gc * fmaf(t2, t2, -(t2 * t) * fmaf(2.0f, qq, 1.0f));
        const float inv_dj = mj.y;
        const float s = fmaf(mj.x, inv_dj, pterm_i);
        const float3 V = vel_diff_poiseuille(P, vi, pi, vj, pj);
        const float kk = valid ? -m * s * inv_d * temp : 0.0f;
        const float kv = valid ? visc_k * inv_dens * inv_dj * inv_d * temp : 0.0f;
        fx += fmaf(kk, rx, kv * V.x);
        fy += fmaf(kk, ry, kv * V.y);
        fz += fmaf(kk, rz, kv * V.z);
    }
};

// the walk of a 2-D channel's force pass: rows that come whole give their
// in-range candidates from the density pass's masks (the target itself left
// out), the others are tested by cand
template <int HASH, int CAP, typename Cells, typename C, typename Q>
__device__ __forceinline__ void walk_row_masks(const cmag_params& P, uint32_t i, const float4& pi, const Cell& gp,
                                               const Cells& cells, const float4* __restrict__ pos,
                                               const uint32_t* __restrict__ masks, uint32_t stride, NbQueue<CAP>& nq,
                                               C&& cand, Q&& pairs) {
    const uint32_t* in = masks + i;
    int left = P.cellcount;  // rows until the target's own
    // a grid of no more cells along y than the stencil reaches brings the
    // target's own row back as other rows: then it is looked for in each (in
    // every grid that cost a 200,003-particle channel 2 %: 62.4 -> 63.5 us)
    const bool repeated = P.grid_size[1] <= (uint32_t)P.cellcount;
    walk_rows<2, HASH>(P, pi, gp, cells, [&](const Run& a, const Run& b, float py, float pz, bool whole) {
        const uint32_t total = a.len + b.len, off_b = b.s - a.len;
        uint32_t m = 0;
        if (whole) {
            m = *in;
            in += stride;
            if (left-- == 0 || repeated) {
                const uint32_t da = i - a.s, db = i - b.s;
                const uint32_t t = da < a.len ? da : db < b.len ? a.len + db : 32u;
                m &= ~(t < 32u ? 1u << t : 0u);
            }
        }
        if (!whole || __ballot(total > (uint32_t)ROW_MASK_BITS)) {
            // no mask, or a long row in some lane: all of them test this one
            for (uint32_t t = 0; t < total; ++t) {
                const bool second = t >= a.len;
                const uint32_t j = (second ? off_b : a.s) + t;
                cand(j, row4(pos, j), true, second ? b.px : a.px, py, pz, second ? b.code : a.code);
            }
            return;
        }
        while (m != 0u) {
            const uint32_t t = (uint32_t)__ffs((int)m) - 1u;
            m &= m - 1u;
            const bool second = t >= a.len;
            nq.push(NbEntry::pack((second ? off_b : a.s) + t, second ? b.code : a.code));
            if (__ballot(nq.full())) nq.drain(NB_DRAIN, pairs);
        }
    });
}

// (p / rho, 1 / rho) of sorted row j: as the density pass left it (STORED), or
// from measures, with the same operations
template <bool STORED>
__device__ __forceinline__ float2 pair_values(const float2* __restrict__ pairs, const float4* __restrict__ measures,
                                              uint32_t j) {
    if (STORED) return *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(pairs) + (j << 3));
    const float4 m = row4(measures, j);
    const float inv = frcp(m.x);
    return make_float2(m.y * inv, inv);
}

// ---- force passes: two phases per target ------------------------------------
// Phase 1 walks the stencil and only tests candidates (r^2 < 4h^2), appending
// the in-range ones to a per-lane list in LDS; phase 2 evaluates the pair
// terms of the listed neighbours.  Without the split, the ~50-instruction pair
// term would run for every candidate (some lane of the wave is almost always
// in range), i.e. ~475 times per particle instead of ~74.  The list is an
// NbQueue of CAP entries per lane (NB_CAP unless a caller picks another
// depth); pair terms take entries two at a time with all their row loads
// (four in the sub-cell walk, six otherwise) issued before either term.
// nbl: this wave's queues in LDS, [CAP][64]
// In the sub-cell walk (Cells::SUB, DamBreak) the row copies carry the
// density pass's results: a fluid row holds -rho in pos.w, sign bit set (a wall
// row keeps its type flag, 0..3, sign bit clear) and db_scale p / rho^2 in vel.w, so a
// pair term gathers two rows instead of three and measures is not read.
// With masks (staged blocks of the sub-cell walk), the in-range fluid
// neighbours of a row whose main run holds at most MASK_BITS candidates come
// from the density pass's mask instead of a walk, and their pair terms are
// evaluated at once, two at a time, after whatever earlier rows left in the
// queue; the walls of the row's first two cells are walked on their own.  Pair
// terms keep the walk's order and wall terms accumulate apart, so the sums are
// the same bit for bit.
template <int SYS, int DIM, int HASH, typename Cells, int CAP = NB_CAP, int LANES = 1>
__device__ __forceinline__ void force_body(const cmag_params& P, uint32_t i, float4* __restrict__ acc,
                                           const float4* __restrict__ measures,
                                           const float4* __restrict__ sortedPos,
                                           const float4* __restrict__ sortedVel,
                                           const uint32_t* __restrict__ index, const Cells& cells, uint32_t n,
                                           uint32_t (*nbl)[64], const LookupView* lp = nullptr, bool staged = false,
                                           const uint2* __restrict__ masks = nullptr, uint32_t stride = 0,
                                           const float2* __restrict__ pv = nullptr,
                                           const uint32_t* __restrict__ row_masks = nullptr,
                                           const StepArrays& step = {}, uint32_t part = 0) {
    const int lane = threadIdx.x & 63;
    constexpr bool PACKED = SYS == CMAG_SYS_DAMBREAK && Cells::SUB;
    auto is_wall = [](float w) { return PACKED ? __float_as_int(w) >= 0 : w != CMAG_DB_FLUID; };
    const float4 pi = sortedPos[i];
    if (SYS == CMAG_SYS_DAMBREAK && is_wall(pi.w)) return;
    const float4 vi = sortedVel[i];
    float rho_i, pterm_i;
    if (PACKED) {
        rho_i = -pi.w;
        pterm_i = vi.w;
    } else {
        const float4 mi = measures[i];
        rho_i = mi.x;
        pterm_i = mi.y / (mi.x * mi.x);
        if (SYS == CMAG_SYS_DAMBREAK) pterm_i *= db_scale(P);
    }
    ForceSum<SYS> F(P, pi, vi, rho_i, pterm_i);
    const Cell gp = grid_pos(P, pi.x, pi.y, pi.z);
    const float r2max = 4.0f * P.smoothing_radius * P.smoothing_radius;
    NbQueue<CAP> nq(nbl, lane);
    auto pairs = [&](uint32_t j0, uint32_t j1, bool second) {
        const float4 p0 = row4(sortedPos, j0), v0 = row4(sortedVel, j0);
        const float4 p1 = row4(sortedPos, j1), v1 = row4(sortedVel, j1);
        const float3 q = make_float3(pi.x, pi.y, pi.z);
        if (PACKED) {
            F.pair_db(q, p0, v0, -p0.w, v0.w);
            F.pair_db(q, p1, v1, -p1.w, v1.w, second);
        } else {
            const float4 m0 = row4(measures, j0), m1 = row4(measures, j1);
            const float i0 = frcp(m0.x), i1 = frcp(m1.x), sc = db_scale(P);
            F.pair_db(q, p0, v0, m0.x, m0.y * i0 * i0 * sc);
            F.pair_db(q, p1, v1, m1.x, m1.y * i1 * i1 * sc, second);
        }
    };
    auto queued_pairs = [&](uint32_t e0, uint32_t e1, bool second) {
        const uint32_t j0 = NbEntry::index(e0), j1 = NbEntry::index(e1);
        if constexpr (SYS == CMAG_SYS_DAMBREAK) {
            pairs(j0, j1, second);
        } else {
            const float4 p0 = row4(sortedPos, j0), v0 = row4(sortedVel, j0);
            const float4 p1 = row4(sortedPos, j1), v1 = row4(sortedVel, j1);
            const float2 m0 = pair_values<Cells::PADDED>(pv, measures, j0), m1 = pair_values<Cells::PADDED>(pv, measures, j1);
            F.pair(image_target(P, pi, NbEntry::code(e0)), p0, m0, v0);
            F.pair(image_target(P, pi, NbEntry::code(e1)), p1, m1, v1, second);
        }
    };

    auto cand = [&](uint32_t j, const float4& pj, bool valid, float px, float py, float pz, int code) {
        const float rx = px - pj.x, ry = py - pj.y, rz = pz - pj.z;
        const float r2 = norm2(rx, ry, rz);
        if (valid && j != i) {
            if (SYS == CMAG_SYS_DAMBREAK && is_wall(pj.w)) {
                // Lennard-Jones wall term: every wall particle of the stencil acts
                F.wall(rx, ry, rz, r2);
            } else if (r2 < r2max) {
                nq.push(NbEntry::pack(j, code));
            }
        }
        if (__ballot(nq.full())) nq.drain(NB_DRAIN, queued_pairs);
    };
    // a run of wall rows only: every one acts (Lennard-Jones), none is queued
    auto wall_only = [&](uint32_t, const float4& pj, bool valid, float px, float py, float pz, int) {
        if (valid) {
            const float rx = px - pj.x, ry = py - pj.y, rz = pz - pj.z;
            F.wall(rx, ry, rz, norm2(rx, ry, rz));
        }
    };
    if constexpr (Cells::SUB) {
        if (staged && masks) {
            const LookupView& v = *lp;
            const int q = x_sub(P, pi.x);
            // the main run [s, e) of row r: cells x - 1 (from eighth q) to
            // x + 1 (through eighth q)
            auto main_run = [&](int r, uint32_t& s, uint32_t& e) {
                s = v.F(r, 0) + SubCells::below(v.Pr(r, 0), q);
                e = v.F(r, 2) + SubCells::through(v.Pr(r, 2), q);
            };
            // the walls of a main run (those of its first two cells, in run
            // order) when the run itself is not walked: the mask holds fluid only
            auto run_walls = [&](int r) {
                const uint4* c0 = v.Pr(r, 0);
                const uint32_t f0 = v.F(r, 0), fx = v.F(r, 1), f1 = v.F(r, 2), cxw = SubCells::fluid(v.Pr(r, 1));
                if ((f1 - f0) - SubCells::fluid(c0) - cxw != 0u) {
                    walk_run_sub(sortedPos, f0 + SubCells::fluid(c0), fx, pi.x, pi.y, pi.z, 13, wall_only);
                    walk_run_sub(sortedPos, fx + cxw, f1, pi.x, pi.y, pi.z, 13, wall_only);
                }
            };
            // the last cell's walls [ws, we)
            auto last_walls = [&](int r) {
                walk_run_sub(sortedPos, v.F(r, 2) + SubCells::fluid(v.Pr(r, 2)), v.F(r, 3), pi.x, pi.y, pi.z, 13, cand);
            };
            // a row's mask without the target's own bit
            auto row_mask = [&](uint2 w, uint32_t s) {
                const uint32_t d = i - s;
                w.x &= ~(d < 32u ? 1u << d : 0u);
                w.y &= ~(d - 32u < 32u ? 1u << (d - 32u) : 0u);
                return w;
            };
            // pair terms straight from masks, two neighbours per iteration in
            // walk order (a missing second repeats the first and adds nothing),
            // without the queue: the words of row a's mask, then row b's.  A
            // word at a time keeps the bit arithmetic in 32 bits; an iteration
            // takes both its neighbours from one word.
            auto mask_pairs = [&](uint2 a, uint32_t sa, uint2 b, uint32_t sb) {
                uint32_t m0 = a.x, m1 = a.y, m2 = b.x, m3 = b.y;
                uint32_t s0 = sa, s1 = sa + 32u, s2 = sb, s3 = sb + 32u;
                // empty words out of the way: every shift below then finds a
                // word with bits, or the end
                if (m2 == 0u) { m2 = m3; s2 = s3; m3 = 0u; }
                if (m1 == 0u) { m1 = m2; s1 = s2; m2 = m3; s2 = s3; m3 = 0u; }
                if (m0 == 0u) { m0 = m1; s0 = s1; m1 = m2; s1 = s2; m2 = m3; s2 = s3; m3 = 0u; }
                while (m0 != 0u) {
                    const uint32_t j0 = s0 + (uint32_t)__builtin_ctz(m0);
                    m0 &= m0 - 1u;
                    const bool two = m0 != 0u;
                    const uint32_t j1 = two ? s0 + (uint32_t)__builtin_ctz(m0) : j0;
                    m0 &= m0 - 1u;  // 0 stays 0
                    if (m0 == 0u) {
                        m0 = m1; s0 = s1;
                        m1 = m2; s1 = s2;
                        m2 = m3; s2 = s3;
                        m3 = 0u;
                    }
                    pairs(j0, j1, two);
                }
            };
            // rows in force_rows order, two at a time (the last alone)
            const RowList list = force_rows<LANES>(DIM, part);
            for (int k = 0; k < list.count; k += 2) {
                const int ra = list[k], rb = k + 1 < list.count ? list[k + 1] : -1;
                // both masks are loaded ahead of the walls (a walked row's is not used)
                const uint2 wa = masks[(size_t)ra * stride + i];
                const uint2 wb = rb >= 0 ? masks[(size_t)rb * stride + i] : make_uint2(0u, 0u);
                uint32_t s, e, sa = 0u, sb = 0u;
                uint2 mA = make_uint2(0u, 0u), mB = mA;
                main_run(ra, s, e);
                const bool walk_a = e - s > (uint32_t)MASK_BITS;
                if (walk_a) {
                    walk_run_sub(sortedPos, s, e, pi.x, pi.y, pi.z, 13, cand);
                } else {
                    run_walls(ra);
                    mA = row_mask(wa, s);
                    sa = s;
                }
                last_walls(ra);
                if (rb >= 0) {
                    main_run(rb, s, e);
                    if (e - s > (uint32_t)MASK_BITS) {
                        // row a's pair terms come before the ones row b queues
                        if (!walk_a) {
                            if (nq.count != 0) nq.drain(CAP, queued_pairs);
                            mask_pairs(mA, sa, make_uint2(0u, 0u), 0u);
                            mA = make_uint2(0u, 0u);
                        }
                        walk_run_sub(sortedPos, s, e, pi.x, pi.y, pi.z, 13, cand);
                    } else {
                        run_walls(rb);
                        mB = row_mask(wb, s);
                        sb = s;
                    }
                    last_walls(rb);
                }
                if (__ballot((mA.x | mA.y | mB.x | mB.y) != 0u)) {
                    // neighbours queued by earlier walked rows come first
                    if (__ballot(nq.count != 0)) nq.drain(CAP, queued_pairs);
                    mask_pairs(mA, sa, mB, sb);
                }
            }
        } else if (staged) {
            walk_lookup<DIM, false, true, LANES>(P, pi, *lp, sortedPos, cand, nullptr, nullptr, part);
        } else {
            walk_stencil_pf<DIM, HASH, false, true, LANES>(P, pi, gp, cells, sortedPos, cand, part);
        }
    } else if (SYS != CMAG_SYS_DAMBREAK && DIM == 2 && HASH == CMAG_HASH_LINEAR && Cells::PADDED && row_masks) {
        walk_row_masks<HASH>(P, i, pi, gp, cells, sortedPos, row_masks, stride, nq, cand, queued_pairs);
    } else {
        walk_stencil_pf<DIM, HASH, SYS != CMAG_SYS_DAMBREAK, false, LANES>(P, pi, gp, cells, sortedPos, cand, part);
    }
    nq.drain(CAP, queued_pairs);
    if (LANES > 1) {
        F.fx = quad_sum(F.fx); F.fy = quad_sum(F.fy); F.fz = quad_sum(F.fz);
        F.wx = quad_sum(F.wx); F.wy = quad_sum(F.wy); F.wz = quad_sum(F.wz);
        if (part != 0) return;
    }
    const uint32_t k = index[i];
    if (k >= n) return;
    const float4 a = make_float4(F.fx + F.wx, F.fy + F.wy, F.fz + F.wz, 0.0f);
    acc[k] = a;
    // Integrating the target here takes a launch (2 to 4 us) and the reads of
    // position, acceleration and leapfrog velocity out of the step: the row
    // holds them (4.1M particles in 256 channels: 810 -> 774 us a step; a
    // 17,500-particle channel: 28.4 -> 24.5 us).  The pass reads the sorted copies
    // only, so its targets' own rows may change under it.
    if (Cells::PADDED && (!Cells::SUB || LANES > 1) && step.pos) {
        // packed rows hold -rho and the pressure term in the w of their copies
        const float4 p = PACKED ? make_float4(pi.x, pi.y, pi.z, CMAG_DB_FLUID) : pi;
        integrate_row<SYS>(P, k, p, PACKED ? step.velLF[k].w : vi.w, a, a, step.pos, step.vel, step.velLF, 0.0f, 0);
    }
}

// ---- Peristalsis: pressure and viscous passes -------------------------------------
// The fused variant produces both from one neighbour walk (same per-pair
// arithmetic as the split kernels)
template <bool WANT_VISC, bool WANT_PRES>
struct PeriSum {
    const cmag_params& P;
    float4 pi, vi;
    float dens, inv_dens, pterm_i, inv_h, m, gc, visc_k;
    float vx = 0.f, vy = 0.f, vz = 0.f, px = 0.f, py = 0.f, pz = 0.f;
    __device__ __forceinline__ PeriSum(const cmag_params& P_, const float4& pi_, const float4& vi_, const float4& mi)
        : P(P_), pi(pi_), vi(vi_) {
        dens = mi.x;
        inv_dens = 1.0f / dens;
        pterm_i = mi.y / (dens * dens);
        inv_h = 1.0f / P.smoothing_radius;
        m = P.particle_mass;
        gc = P.grad_coeff;
        visc_k = m * (P.mu + P.mu);
    }
    // mj = (p_j / rho_j, 1 / rho_j); valid = false adds nothing
    __device__ __forceinline__ void pair(const float3& q, const float4& pj, const float2& mj, const float4& vj,
                                         bool valid = true) {
        const float rx = q.x - pj.x, ry = q.y - pj.y, rz = q.z - pj.z;
        const float r2 = norm2(rx, ry, rz);
        const float inv_d = frsq(r2);
        const float dist = r2 * inv_d;
        const float qq = dist * inv_h;
        const float t = fmaf(-0.5f, qq, 1.0f);
        const float t2 = t * t;
        const float temp = gc * fmaf(t2, t2, -(t2 * t) * fmaf(2.0f, qq, 1.0f));
        const float inv_dj = mj.y;
        if (WANT_PRES) {
            const float kk = valid ? -m * temp * fmaf(mj.x, inv_dj, pterm_i) * inv_d : 0.0f;
            px = fmaf(kk, rx, px); py = fmaf(kk, ry, py); pz = fmaf(kk, rz, pz);
        }
        if (WANT_VISC) {
            const float kv = valid ? visc_k * temp * inv_dens * inv_dj * inv_d : 0.0f;
            vx = fmaf(kv, vi.x - vj.x, vx); vy = fmaf(kv, vi.y - vj.y, vy); vz = fmaf(kv, vi.z - vj.z, vz);
        }
    }
};

template <int DIM, int HASH, bool WANT_VISC, bool WANT_PRES, typename Cells, int CAP = NB_CAP>
__device__ __forceinline__ void peristalsis_force_body(
    const cmag_params& P, uint32_t i, float4* __restrict__ viscF, float4* __restrict__ presF,
    const float4* __restrict__ measures, const float4* __restrict__ sortedPos,
    const float4* __restrict__ sortedVel, const uint32_t* __restrict__ index, const Cells& cells, uint32_t n,
    uint32_t (*nbl)[64], const float2* __restrict__ pv = nullptr, const uint32_t* __restrict__ row_masks = nullptr,
    uint32_t stride = 0, const StepArrays& step = {}) {
    const int lane = threadIdx.x & 63;
    const float4 pi = sortedPos[i];
    PeriSum<WANT_VISC, WANT_PRES> F(P, pi, WANT_VISC ? sortedVel[i] : make_float4(0.f, 0.f, 0.f, 0.f),
                                    measures[i]);
    const Cell gp = grid_pos(P, pi.x, pi.y, pi.z);
    const float r2max = 4.0f * P.smoothing_radius * P.smoothing_radius;
    NbQueue<CAP> nq(nbl, lane);
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    auto pairs = [&](uint32_t e0, uint32_t e1, bool second) {
        const uint32_t j0 = NbEntry::index(e0), j1 = NbEntry::index(e1);
        const float2 m0 = pair_values<Cells::PADDED>(pv, measures, j0), m1 = pair_values<Cells::PADDED>(pv, measures, j1);
        const float4 p0 = row4(sortedPos, j0), p1 = row4(sortedPos, j1);
        const float4 v0 = WANT_VISC ? row4(sortedVel, j0) : zero4;
        const float4 v1 = WANT_VISC ? row4(sortedVel, j1) : zero4;
        F.pair(image_target(P, pi, NbEntry::code(e0)), p0, m0, v0);
        F.pair(image_target(P, pi, NbEntry::code(e1)), p1, m1, v1, second);
    };

    auto cand = [&](uint32_t j, const float4& pj, bool valid, float qx, float qy, float qz, int code) {
        const float rx = qx - pj.x, ry = qy - pj.y, rz = qz - pj.z;
        const float r2 = norm2(rx, ry, rz);
        if (valid && j != i && r2 < r2max) nq.push(NbEntry::pack(j, code));
        if (__ballot(nq.full())) nq.drain(NB_DRAIN, pairs);
    };
    if (DIM == 2 && HASH == CMAG_HASH_LINEAR && Cells::PADDED && row_masks)
        walk_row_masks<HASH>(P, i, pi, gp, cells, sortedPos, row_masks, stride, nq, cand, pairs);
    else
        walk_stencil_pf<DIM, HASH>(P, pi, gp, cells, sortedPos, cand);
    nq.drain(CAP, pairs);
    const uint32_t k = index[i];
    if (k >= n) return;
    const float4 a = make_float4(F.vx, F.vy, F.vz, 0.0f), pr = make_float4(F.px, F.py, F.pz, 0.0f);
    if (WANT_VISC) viscF[k] = a;
    if (WANT_PRES) presF[k] = pr;
    if (Cells::PADDED && WANT_VISC && WANT_PRES && step.pos)  // as in force_body
        integrate_row<CMAG_SYS_PERISTALSIS>(P, k, pi, F.vi.w, a, pr, step.pos, step.vel, step.velLF,
                                            step.state->t_w, step.state->is_config);
}

}  // namespace cmag
