// adjoint.hip - hand-written vector-Jacobian products of the Poiseuille step
// (gfx950, FP32 with FP64 parameter accumulators).
//
// The reference has no adjoint.  These differentiate this library's forward
// passes with the neighbour structure (sort order, cell lists) of the step
// held fixed, as it is piecewise constant:
//   density_vjp    density + EOS      poiseuilleFlowKernel.cu:99-182
//   force_vjp      pressure + Morris viscous force with the wall
//                  extrapolation      poiseuilleFlowKernel.cu:184-309
//   integrate_vjp  integratePoiseuilleSystemD  poiseuilleFlowKernel.cu:311-348
// Walls (w == 1) are not state: their density is the constant rho0 and their
// adjoints are zero.
//
// Pair notation (target k, neighbour j, r = x_k - x_j after the image shift,
// d = |r|, G = (dW/dr)/d, G' = dG/dd, pi = p/rho^2):
//   a_k = sum_j [ -m (pi_k + pi_j) G r + c_kj V_kj ],  c_kj = 2 m mu G/(rho_k rho_j),
//   V_kj = l_k - l_j, or beta l_k for a wall neighbour beyond its wall plane.
// A pair enters k's adjoint once as target and once as neighbour; with
// D = abar_k - abar_j (abar of walls is zero) both collapse into one term, so
// every pass gathers over the same stencil as the forward pass, with no
// atomics:
//   pibar_k  = sum -m G (r . D)
//   rhobar_k = pibar_k dpi/drho - (1/rho_k) sum c (V . D)
//   lbar_k   = sum c (beta~ abar_k - abar_j)        (beta~ = beta or 1)
//   xbar_k   = sum A [G D + (G'/d) r (r . D)] + B (G'/d) r (V . D)
//              (+ c (abar_k . l_k) dbeta/dy_k for wall neighbours)
//   mubar    = sum_k sum_j 2 m G/(rho_k rho_j) (abar_k . V_kj)
//   density: xbar_k += sum_j m G r (rhobar_k + rhobar_j)
#include <string>
#include <type_traits>

#include "kernels.hpp"
#include "sph_device.hpp"

namespace cmag {

// With q = d / h and t = 1 - q/2, the dW/dr bracket t^4 - t^3 (2q + 1) is
// 5 t^3 (t - 1) = -2.5 q t^3, so
//   G    = (dW/dr) / d = g_k t^3,     g_k  = -2.5 grad_coeff / h
//   G'/d = (dG/dd) / d = gp_k t^2 / d, gp_k = 3.75 grad_coeff / h^2
// without the differences of the bracket's own form, and with one division a
// pair instead of six.
struct GradKernel {
    float t_k, g_k, gp_k, r2max;
    __device__ __forceinline__ explicit GradKernel(const cmag_params& P) {
        const float h = P.smoothing_radius, gc = P.grad_coeff;
        t_k = -0.5f / h;
        g_k = -2.5f * gc / h;
        gp_k = 3.75f * gc / (h * h);
        r2max = 4.0f * h * h;
    }
};

// p / rho^2 and 1 / rho of a row
__device__ __forceinline__ float2 row_terms(const float4& m) { return make_float2(m.y / (m.x * m.x), 1.0f / m.x); }

// target and lane of a thread: the lanes of a target are neighbours
__device__ __forceinline__ void vjp_target(uint32_t& i, uint32_t& part) {
    i = xcd_block() * (blockDim.x / TARGET_LANES) + threadIdx.x / TARGET_LANES;
    part = threadIdx.x % TARGET_LANES;
}

// d p / d rho of the equation of state
__device__ __forceinline__ float deos(const cmag_params& P, float dens) {
    if (P.eos == CMAG_EOS_TAIT)
        return P.B * P.gamma * pow_int(dens / P.rest_density, (int)P.gamma - 1) / P.rest_density;
    if (P.eos == CMAG_EOS_LINEAR_C2) return P.soundspeed * P.soundspeed;
    return 50.0f * P.soundspeed;
}

__device__ __forceinline__ float dot3(float ax, float ay, float az, float bx, float by, float bz) {
    return ax * bx + ay * by + az * bz;
}

// ---- integrate ----------------------------------------------------------------
// gpos/gvel/gvelLF: adjoints of the step outputs in, of its inputs out (velLF is
// no input of integrate); returns the acceleration's; ggrav[i] += share of
// the body-force adjoint
__device__ __forceinline__ float4 integrate_vjp_row(const cmag_params& P, uint32_t i, bool wall,
                                                    float4* __restrict__ gpos, float4* __restrict__ gvel,
                                                    float4* __restrict__ gvelLF, double* __restrict__ ggrav) {
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
    if (wall) {
        gpos[i] = z;
        gvel[i] = z;
        gvelLF[i] = z;
        return z;
    }
    const float dt = P.delta_time;
    const float4 gx = gpos[i], gv = gvel[i], gl = gvelLF[i];
    const float ux = gv.x + 0.5f * gl.x + dt * gx.x;
    const float uy = gv.y + 0.5f * gl.y + dt * gx.y;
    const float uz = gv.z + 0.5f * gl.z + dt * gx.z;
    gvel[i] = make_float4(ux + 0.5f * gl.x, uy + 0.5f * gl.y, uz + 0.5f * gl.z, 0.f);
    gvelLF[i] = z;
    if (ggrav) {
        ggrav[4 * (size_t)i] += (double)(dt * ux);
        ggrav[4 * (size_t)i + 1] += (double)(dt * uy);
        ggrav[4 * (size_t)i + 2] += (double)(dt * uz);
    }
    return make_float4(dt * ux, dt * uy, dt * uz, 0.f);
}

// unsorted order
__global__ __launch_bounds__(256) void integrate_vjp_kernel(const cmag_params P, const float4* __restrict__ pos,
                                                            float4* __restrict__ gpos, float4* __restrict__ gvel,
                                                            float4* __restrict__ gvelLF, float4* __restrict__ gacc,
                                                            double* __restrict__ ggrav, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    gacc[i] = integrate_vjp_row(P, i, pos[i].w == CMAG_PO_WALL, gpos, gvel, gvelLF, ggrav);
}

// The same by sorted row, for a step whose density has run: the acceleration
// adjoint goes to the row itself, and the row's terms of the pair sums are
// formed once.  A launch and a pass over gacc less than integrate_vjp and a
// gather, and no division by a neighbour's density in the pair loops.
__global__ __launch_bounds__(256) void step_vjp_kernel(const cmag_params P, const float4* __restrict__ sortedPos,
                                                       const float4* __restrict__ measures,
                                                       const uint32_t* __restrict__ index, float4* __restrict__ gpos,
                                                       float4* __restrict__ gvel, float4* __restrict__ gvelLF,
                                                       float4* __restrict__ gaccS, float2* __restrict__ terms,
                                                       double* __restrict__ ggrav, uint32_t n) {
    const uint32_t r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    terms[r] = row_terms(measures[r]);
    const uint32_t i = index[r];
    if (i >= n) {
        gaccS[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        return;
    }
    const bool wall = sortedPos[r].w == CMAG_PO_WALL;
    gaccS[r] = integrate_vjp_row(P, i, wall, gpos, gvel, gvelLF, ggrav);
}

// ---- force ----------------------------------------------------------------------
// sorted order.  gmu_acc (optional) += the target's share of d/d mu in FP64;
// gmu (optional) = the same share in FP32; terms: row_terms of every row, or
// null (a caller's rows: formed here)
//
// Both neighbour passes give a target to TARGET_LANES lanes, each with every
// fourth stencil row (the rows of 5 + 1, 5, 5 + 1 and 5 in-range neighbours at h =
// 1.5 spacings), and fold their sums: the passes are one serial chain per
// target, too long for the few waves of a channel.  A row's loads are issued
// one candidate ahead.
template <int DIM, int HASH, typename Cells>
__global__ __launch_bounds__(256) void force_vjp_kernel(const cmag_params P, float4* __restrict__ gpos,
                                                        float4* __restrict__ gvel, float* __restrict__ grho,
                                                        float* __restrict__ gmu, double* __restrict__ gmu_acc,
                                                        const float4* __restrict__ gacc,
                                                        const float4* __restrict__ measures,
                                                        const float4* __restrict__ sortedPos,
                                                        const float4* __restrict__ sortedVel, const Cells cells,
                                                        uint32_t n, const float2* __restrict__ terms) {
    uint32_t i, part;
    vjp_target(i, part);
    if (i >= n) return;
    const float4 pi = sortedPos[i];
    const float4 z = make_float4(0.f, 0.f, 0.f, 0.f);
    if (pi.w == CMAG_PO_WALL) {
        if (part == 0) {
            gpos[i] = z;
            gvel[i] = z;
            grho[i] = 0.f;
            if (gmu) gmu[i] = 0.f;
        }
        return;
    }
    const float4 li = sortedVel[i], ai = gacc[i], mi = measures[i];
    const float2 ti = row_terms(mi);
    const float rho_i = mi.x;
    const float m = P.particle_mass;
    const GradKernel K(P);
    const float top = P.wall_top, bottom = P.wall_bottom;
    const float mu2 = 2.f * m * ti.y;  // 2 m / rho_i
    float pibar = 0.f, vd = 0.f, mubar = 0.f;
    float gx = 0.f, gy = 0.f, gz = 0.f, lx = 0.f, ly = 0.f, lz = 0.f;
    struct Row {
        float4 p, l, a;
        float2 t;
    };
    auto load = [&](uint32_t j) {
        return Row{sortedPos[j], sortedVel[j], gacc[j], Cells::PADDED ? terms[j] : row_terms(measures[j])};
    };
    auto pair = [&](uint32_t j, const Row& J, float qx, float qy, float qz) {
        const float rx = qx - J.p.x, ry = qy - J.p.y, rz = qz - J.p.z;
        const float r2 = rx * rx + ry * ry + rz * rz;
        if (j == i || !(r2 < K.r2max)) return;
        const float dist = sqrtf(r2);
        const float t = fmaf(K.t_k, dist, 1.0f);
        const float t2 = t * t;
        const float G = K.g_k * (t2 * t);
        const float Gpd = K.gp_k * t2 / dist;
        float bt = 1.f, dbeta = 0.f;
        bool wall_beyond = false;
        if (J.p.w == CMAG_PO_WALL && (J.p.y > top || J.p.y < bottom)) {
            const bool up = J.p.y > top;
            const float dA = up ? top - pi.y : pi.y - bottom, dB = up ? J.p.y - top : bottom - J.p.y;
            const float b = 1.f + dB / dA;
            wall_beyond = true;
            bt = fminf(P.beta_max, b);
            if (b < P.beta_max) dbeta = up ? dB / (dA * dA) : -dB / (dA * dA);
        }
        const float Vx = wall_beyond ? bt * li.x : li.x - J.l.x;
        const float Vy = wall_beyond ? bt * li.y : li.y - J.l.y;
        const float Vz = wall_beyond ? bt * li.z : li.z - J.l.z;
        const float Dx = ai.x - J.a.x, Dy = ai.y - J.a.y, Dz = ai.z - J.a.z;
        const float A = -m * (ti.x + J.t.x);
        const float B0 = mu2 * J.t.y;  // 2 m / (rho_i rho_j)
        const float B = B0 * P.mu;
        const float c = B * G;
        const float rD = dot3(rx, ry, rz, Dx, Dy, Dz);
        const float VD = dot3(Vx, Vy, Vz, Dx, Dy, Dz);
        pibar = fmaf(G, rD, pibar);
        vd = fmaf(c, VD, vd);
        mubar = fmaf(B0 * G, dot3(ai.x, ai.y, ai.z, Vx, Vy, Vz), mubar);
        lx = fmaf(c, bt * ai.x - J.a.x, lx);
        ly = fmaf(c, bt * ai.y - J.a.y, ly);
        lz = fmaf(c, bt * ai.z - J.a.z, lz);
        const float k1 = A * G, k2 = (A * rD + B * VD) * Gpd;
        gx += k1 * Dx + k2 * rx;
        gy += k1 * Dy + k2 * ry;
        gz += k1 * Dz + k2 * rz;
        if (wall_beyond) gy += c * dot3(ai.x, ai.y, ai.z, li.x, li.y, li.z) * dbeta;
    };
    const Cell gp = grid_pos(P, pi.x, pi.y, pi.z);
    walk_rows<DIM, HASH, true, false, TARGET_LANES>(P, pi, gp, cells,
                                                 [&](const Run& a, const Run& b, float py, float pz, bool) {
        const uint32_t total = a.len + b.len, off_b = b.s - a.len;
        if (total == 0) return;
        auto row = [&](uint32_t t) { return (t >= a.len ? off_b : a.s) + t; };
        uint32_t j = row(0);
        Row J = load(j);
        for (uint32_t t = 0; t < total; ++t) {
            const uint32_t jn = row(min(t + 1u, total - 1u));
            const Row N = load(jn);
            pair(j, J, t >= a.len ? b.px : a.px, py, pz);
            j = jn;
            J = N;
        }
    }, part);
    pibar = quad_sum(pibar); vd = quad_sum(vd); mubar = quad_sum(mubar);
    gx = quad_sum(gx); gy = quad_sum(gy); gz = quad_sum(gz);
    lx = quad_sum(lx); ly = quad_sum(ly); lz = quad_sum(lz);
    if (part != 0) return;
    const float dpi = deos(P, rho_i) / (rho_i * rho_i) - 2.f * mi.y / (rho_i * rho_i * rho_i);
    gpos[i] = make_float4(gx, gy, gz, 0.f);
    gvel[i] = make_float4(lx, ly, lz, 0.f);
    grho[i] = -m * pibar * dpi - ti.y * vd;
    if (gmu) gmu[i] = mubar;
    if (gmu_acc) gmu_acc[i] += (double)mubar;
}

// ---- density ------------------------------------------------------------------
// sorted order: gposS[k] += sum_j m G r (grho_k + grho_j) for non-walls.  With
// index, the total goes to the unsorted adjoints: gpos[index[k]] += gposS[k],
// gvelLF[index[k]] = gvelS[k] (the step's output adjoints already consumed)
template <int DIM, int HASH, typename Cells>
__global__ __launch_bounds__(256) void density_vjp_kernel(const cmag_params P, float4* __restrict__ gposS,
                                                          const float* __restrict__ grho,
                                                          const float4* __restrict__ sortedPos, const Cells cells,
                                                          uint32_t n, const uint32_t* __restrict__ index,
                                                          const float4* __restrict__ gvelS,
                                                          float4* __restrict__ gpos, float4* __restrict__ gvelLF) {
    uint32_t i, part;
    vjp_target(i, part);
    if (i >= n) return;
    const float4 pi = sortedPos[i];
    if (pi.w == CMAG_PO_WALL) return;
    const GradKernel K(P);
    const float gi = grho[i];
    float gx = 0.f, gy = 0.f, gz = 0.f;
    const Cell gp = grid_pos(P, pi.x, pi.y, pi.z);
    walk_rows<DIM, HASH, true, false, TARGET_LANES>(P, pi, gp, cells,
                                                 [&](const Run& a, const Run& b, float py, float pz, bool) {
        const uint32_t total = a.len + b.len, off_b = b.s - a.len;
        if (total == 0) return;
        auto row = [&](uint32_t t) { return (t >= a.len ? off_b : a.s) + t; };
        uint32_t j = row(0);
        float4 pj = sortedPos[j];
        float gj = grho[j];
        for (uint32_t t = 0; t < total; ++t) {
            const uint32_t jn = row(min(t + 1u, total - 1u));
            const float4 pn = sortedPos[jn];
            const float gn = grho[jn];
            const float rx = (t >= a.len ? b.px : a.px) - pj.x, ry = py - pj.y, rz = pz - pj.z;
            const float r2 = rx * rx + ry * ry + rz * rz;
            if (j != i && r2 < K.r2max) {
                const float w = fmaf(K.t_k, sqrtf(r2), 1.0f);
                const float c = w * w * w * (gi + gj);
                gx = fmaf(c, rx, gx); gy = fmaf(c, ry, gy); gz = fmaf(c, rz, gz);
            }
            j = jn;
            pj = pn;
            gj = gn;
        }
    }, part);
    gx = quad_sum(gx); gy = quad_sum(gy); gz = quad_sum(gz);
    if (part != 0) return;
    const float mg = P.particle_mass * K.g_k;
    float4 g = gposS[i];
    g.x = fmaf(mg, gx, g.x); g.y = fmaf(mg, gy, g.y); g.z = fmaf(mg, gz, g.z);
    if (!index) {
        gposS[i] = g;
        return;
    }
    const uint32_t k = index[i];
    if (k >= n) return;
    float4 t = gpos[k];
    gpos[k] = make_float4(t.x + g.x, t.y + g.y, t.z + g.z, t.w);
    gvelLF[k] = gvelS[i];
}

// ---- launchers ------------------------------------------------------------------
template <typename F>
static int dispatch_dh(const cmag_params& P, F&& f) {
    const bool mo = P.hash_order == CMAG_HASH_MORTON;
    if (P.dim == 3) {
        if (mo) f(std::integral_constant<int, 3>{}, std::integral_constant<int, 1>{});
        else f(std::integral_constant<int, 3>{}, std::integral_constant<int, 0>{});
    } else {
        if (mo) f(std::integral_constant<int, 2>{}, std::integral_constant<int, 1>{});
        else f(std::integral_constant<int, 2>{}, std::integral_constant<int, 0>{});
    }
    return CMAG_OK;
}

static int need_poiseuille(const cmag_params& P, const char* who) {
    if (P.system != CMAG_SYS_POISEUILLE)
        return fail(CMAG_E_INVALID, std::string(who) + ": the adjoint covers the Poiseuille system");
    return CMAG_OK;
}

int launch_integrate_vjp(const cmag_params& P, const float* pos, float* gpos, float* gvel, float* gvelLF,
                         float* gacc, double* ggrav, uint32_t n, hipStream_t s) {
    CMAG_TRY(need_poiseuille(P, "integrate_vjp"));
    if (n == 0) return CMAG_OK;
    hipLaunchKernelGGL(integrate_vjp_kernel, dim3(div_up(n, 256)), dim3(256), 0, s, P,
                       reinterpret_cast<const float4*>(pos), reinterpret_cast<float4*>(gpos),
                       reinterpret_cast<float4*>(gvel), reinterpret_cast<float4*>(gvelLF),
                       reinterpret_cast<float4*>(gacc), ggrav, n);
    return check_launch("integrate_vjp_kernel");
}

int launch_step_vjp(const cmag_params& P, const float* sortedPos, const float* measures, const uint32_t* index,
                    float* gpos, float* gvel, float* gvelLF, float* gaccS, float* terms, double* ggrav, uint32_t n,
                    hipStream_t s) {
    CMAG_TRY(need_poiseuille(P, "step_vjp"));
    if (n == 0) return CMAG_OK;
    hipLaunchKernelGGL(step_vjp_kernel, dim3(div_up(n, 256)), dim3(256), 0, s, P,
                       reinterpret_cast<const float4*>(sortedPos), reinterpret_cast<const float4*>(measures), index,
                       reinterpret_cast<float4*>(gpos), reinterpret_cast<float4*>(gvel),
                       reinterpret_cast<float4*>(gvelLF), reinterpret_cast<float4*>(gaccS),
                       reinterpret_cast<float2*>(terms), ggrav, n);
    return check_launch("step_vjp_kernel");
}

int launch_force_vjp(const cmag_params& P, float* gposS, float* gvelS, float* grho, float* gmu, double* gmu_acc,
                     const float* gaccS, const float* measures, const float* sortedPos, const float* sortedVel,
                     const uint32_t* cellStart, const uint32_t* cellEnd, const uint32_t* cellFirst, uint32_t n,
                     const float* terms, hipStream_t s) {
    CMAG_TRY(need_poiseuille(P, "force_vjp"));
    if (n == 0) return CMAG_OK;
    if (cellFirst && !terms) return fail(CMAG_E_INVALID, "force_vjp over compact offsets takes the rows' terms");
    auto f4 = [](float* q) { return reinterpret_cast<float4*>(q); };
    auto c4 = [](const float* q) { return reinterpret_cast<const float4*>(q); };
    dispatch_dh(P, [&](auto D, auto H) {
        constexpr int DIM = decltype(D)::value, HASH = decltype(H)::value;
        if (cellFirst)
            hipLaunchKernelGGL((force_vjp_kernel<DIM, HASH, FirstCells>), dim3(div_up(n, 256 / TARGET_LANES)), dim3(256), 0, s,
                               P, f4(gposS), f4(gvelS), grho, gmu, gmu_acc, c4(gaccS), c4(measures), c4(sortedPos),
                               c4(sortedVel), FirstCells{cellFirst}, n, reinterpret_cast<const float2*>(terms));
        else
            hipLaunchKernelGGL((force_vjp_kernel<DIM, HASH, RefCells>), dim3(div_up(n, 256 / TARGET_LANES)), dim3(256), 0, s, P,
                               f4(gposS), f4(gvelS), grho, gmu, gmu_acc, c4(gaccS), c4(measures), c4(sortedPos),
                               c4(sortedVel), RefCells{cellStart, cellEnd, n}, n, nullptr);
    });
    return check_launch("force_vjp_kernel");
}

int launch_density_vjp(const cmag_params& P, float* gposS, const float* grho, const float* sortedPos,
                       const uint32_t* cellStart, const uint32_t* cellEnd, const uint32_t* cellFirst, uint32_t n,
                       const uint32_t* index, const float* gvelS, float* gpos, float* gvelLF, hipStream_t s) {
    CMAG_TRY(need_poiseuille(P, "density_vjp"));
    if (n == 0) return CMAG_OK;
    auto f4 = [](float* q) { return reinterpret_cast<float4*>(q); };
    auto c4 = [](const float* q) { return reinterpret_cast<const float4*>(q); };
    dispatch_dh(P, [&](auto D, auto H) {
        constexpr int DIM = decltype(D)::value, HASH = decltype(H)::value;
        if (cellFirst)
            hipLaunchKernelGGL((density_vjp_kernel<DIM, HASH, FirstCells>), dim3(div_up(n, 256 / TARGET_LANES)), dim3(256), 0, s,
                               P, f4(gposS), grho, c4(sortedPos), FirstCells{cellFirst}, n, index, c4(gvelS),
                               f4(gpos), f4(gvelLF));
        else
            hipLaunchKernelGGL((density_vjp_kernel<DIM, HASH, RefCells>), dim3(div_up(n, 256 / TARGET_LANES)), dim3(256), 0, s, P,
                               f4(gposS), grho, c4(sortedPos), RefCells{cellStart, cellEnd, n}, n, index,
                               c4(gvelS), f4(gpos), f4(gvelLF));
    });
    return check_launch("density_vjp_kernel");
}

}  // namespace cmag

using namespace cmag;

extern "C" {

int cmag_integrate_vjp(const cmag_params* p, const float* pos, float* gpos, float* gvel, float* gvelLF,
                       float* gacc, double* ggrav, uint32_t n, cmag_stream_t stream) {
    CMAG_TRY(validate_params(p));
    if (n && (!pos || !gpos || !gvel || !gvelLF || !gacc))
        return fail(CMAG_E_INVALID, "cmag_integrate_vjp: null pointer");
    return launch_integrate_vjp(*p, pos, gpos, gvel, gvelLF, gacc, ggrav, n, as_stream(stream));
}

int cmag_force_vjp(const cmag_params* p, float* gposS, float* gvelS, float* grho, float* gmu, const float* gaccS,
                   const float* measures, const float* sortedPos, const float* sortedVel,
                   const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n, cmag_stream_t stream) {
    CMAG_TRY(validate_params(p));
    if (n && (!gposS || !gvelS || !grho || !gaccS || !measures || !sortedPos || !sortedVel || !cellStart ||
              !cellEnd))
        return fail(CMAG_E_INVALID, "cmag_force_vjp: null pointer");
    return launch_force_vjp(*p, gposS, gvelS, grho, gmu, nullptr, gaccS, measures, sortedPos, sortedVel, cellStart,
                            cellEnd, nullptr, n, nullptr, as_stream(stream));
}

int cmag_density_vjp(const cmag_params* p, float* gposS, const float* grho, const float* sortedPos,
                     const uint32_t* cellStart, const uint32_t* cellEnd, uint32_t n, cmag_stream_t stream) {
    CMAG_TRY(validate_params(p));
    if (n && (!gposS || !grho || !sortedPos || !cellStart || !cellEnd))
        return fail(CMAG_E_INVALID, "cmag_density_vjp: null pointer");
    return launch_density_vjp(*p, gposS, grho, sortedPos, cellStart, cellEnd, nullptr, n, nullptr, nullptr, nullptr,
                              nullptr, as_stream(stream));
}

}  // extern "C"
