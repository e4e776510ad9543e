// terms.h - the neighbour sums and per-particle terms of the step, shared by the launched kernels (dfsph.hip) and the
// resident solvers (solve.hip). A sum takes the particle's own value and a loader that hands it each neighbour's
// records, so that both forms run the same arithmetic in the same list order.
#pragma once

#include "device.h"
#include "kernels.h"

namespace vfd {

__device__ __forceinline__ KTab ktab(const KTabHost& h) { return KTab{h.tab, h.R, h.R2, h.invStep, h.W0}; }
__device__ __forceinline__ uint32_t nbr(const Fields& F, uint32_t cap, uint32_t i, uint32_t j) {
    return F.nbrList[list_at(i, j)];
}
__device__ __forceinline__ HaloView halo(const Fields& F) { return HaloView{F.haloCount, F.haloIds}; }
__device__ __forceinline__ NbrSrc global_src(const Fields& F, uint32_t cap) {
    return NbrSrc{nullptr, F.nbrLocal, F.nbrList, F.nbrCount, cap};
}

// Every gradient-loop kernel stages the G table in LDS, followed by the halo records of the current group.
#define VFD_HALO_KERNEL_PROLOGUE(kh)                                   \
    extern __shared__ float4 lds[];                                    \
    float* sG = reinterpret_cast<float*>(lds);                         \
    load_table_g(sG, (kh).tab);                                        \
    const KLds K{sG, (kh).R, (kh).invStep};                            \
    float* rec = reinterpret_cast<float*>(lds + kLdsG / sizeof(float4));

// ---- shared neighbour sums --------------------------------------------------------------------------------------
// sum_j (u_i - u_j).gradW_ij * V + sum_b V_b u_i.gradW_ib: the velocity divergence (DFSPHKernels.cu:233-278, :483-529)
// and, of the pressure accelerations, ComputeDensityPressureForce (:280-315); records lo = {x_j}, hi = {u_j}
template <class Load>
__device__ __forceinline__ float field_divergence(const SceneParams& p, const KLds& k, const Fields& F, uint32_t cap,
                                                  uint32_t i, f3 ui, const Load& load, const NbrSrc& src) {
    const f3 xi = ld3(F.pos[i]);
    float d = 0.0f;
    each_neighbor_rec<2>(src, i, k.R, k.invStep, xi, k.sG, load, [&](float4 lo, float4 hi, float g) {
        d += dot3(ui - ld3(hi), g * (xi - ld3(lo)));
    });
    d *= p.V;
    for (uint32_t b = 0; b < p.bodyCount; ++b) {
        const float vb = F.vb[(size_t)b * cap + i];
        if (vb > 0.0f) d += vb * dot3(ui, gradW(k, xi - ld3(F.xb[(size_t)b * cap + i])));
    }
    return d;
}

// pressure acceleration from kappa (ComputePressureAccelerationKernel :342-386 and its three siblings);
// records lo = {x_j, kappa_j}
template <class Load>
__device__ __forceinline__ f3 pressure_accel(const SceneParams& p, const KLds& k, const Fields& F, uint32_t cap,
                                             uint32_t i, float ki, const Load& load, const NbrSrc& src) {
    const f3 xi = ld3(F.pos[i]);
    const float negV = -p.V;  // read before the loop: a global read inside it would wait for the list prefetch
    f3 a = mk3(0.0f, 0.0f, 0.0f);
    each_neighbor_rec<1>(src, i, k.R, k.invStep, xi, k.sG, load, [&](float4 lo, float4, float g) {
        const float s = ki + lo.w;
        if (above_eps(fabsf(s))) {
            const f3 gj = negV * (g * (xi - ld3(lo)));
            a = a + s * gj;
        }
    });
    if (above_eps(fabsf(ki))) {
        for (uint32_t b = 0; b < p.bodyCount; ++b) {
            const float vb = F.vb[(size_t)b * cap + i];
            if (vb > 0.0f) {
                const f3 gj = (-vb) * gradW(k, xi - ld3(F.xb[(size_t)b * cap + i]));
                a = a + ki * gj;
            }
        }
    }
    return a;
}

// ---- implicit viscosity (ComputeViscosity, DFSPHImplementation.cu:577-615; Weiler et al. 2018) ------------------
struct M3 {
    float m[9];  // row-major
};
__device__ __forceinline__ M3 inverse3(const M3& A) {
    const float a = A.m[0], b = A.m[1], c = A.m[2];
    const float d = A.m[3], e = A.m[4], f = A.m[5];
    const float g = A.m[6], h = A.m[7], i = A.m[8];
    const float c00 = e * i - f * h, c01 = f * g - d * i, c02 = d * h - e * g;
    const float det = a * c00 + b * c01 + c * c02;
    const float s = 1.0f / det;
    M3 r;
    r.m[0] = c00 * s;
    r.m[1] = (c * h - b * i) * s;
    r.m[2] = (b * f - c * e) * s;
    r.m[3] = c01 * s;
    r.m[4] = (a * i - c * g) * s;
    r.m[5] = (c * d - a * f) * s;
    r.m[6] = c02 * s;
    r.m[7] = (b * g - a * h) * s;
    r.m[8] = (a * e - b * d) * s;
    return r;
}
__device__ __forceinline__ f3 minv_mul(const float* __restrict__ minv, uint32_t cap, uint32_t i, f3 v) {
    float m[9];
#pragma unroll
    for (int e = 0; e < 9; ++e) m[e] = minv[(size_t)e * cap + i];
    return mk3(m[0] * v.x + m[1] * v.y + m[2] * v.z, m[3] * v.x + m[4] * v.y + m[5] * v.z,
               m[6] * v.x + m[7] * v.y + m[8] * v.z);
}

// GetOrthogonalVectors (Core/Math/Math.h:19-33)
__device__ __forceinline__ void orthogonal_vectors(f3 vec, f3& x, f3& y) {
    f3 v = mk3(1.0f, 0.0f, 0.0f);
    if ((double)fabsf(dot3(v, vec)) > 0.999) v = mk3(0.0f, 1.0f, 0.0f);
    x = cross(vec, v);
    y = cross(vec, x);
    x = normalize(x);
    y = normalize(y);
}

// four tangential boundary samples (DFSPHKernels.cu:643-671, 713-742, 800-829)
struct Tangential {
    f3 pd[4];
    f3 gw[4];
    float vol;
};
__device__ __forceinline__ bool tangential(const SceneParams& p, const KLds& k, f3 xi, f3 xb, float vb, Tangential& t) {
    f3 normal = -(xi - xb);
    const float nl = length(normal);
    if (!(nl > 0.0001f)) return false;
    normal = normal / nl;
    f3 t1, t2;
    orthogonal_vectors(normal, t1, t2);
    const f3 pos[4] = {xb - t1 * p.td, xb + t1 * p.td, xb - t2 * p.td, xb + t2 * p.td};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        t.pd[q] = xi - pos[q];
        t.gw[q] = gradW(k, t.pd[q]);
    }
    t.vol = 0.25f * vb;
    return true;
}

// ComputeViscosityPreconditionerKernel (:604-684): the inverse of the system's diagonal block of particle i;
// records lo = {x_j, m / rho_j}
template <class Load>
__device__ __forceinline__ M3 visc_precond(const SceneParams& p, const KLds& k, const Fields& F, uint32_t cap,
                                           uint32_t i, float dt, const Load& load, const NbrSrc& src) {
    const f3 xi = ld3(F.pos[i]);
    const float d001 = 0.01f * p.R2;
    const float mu10 = 10.0f * p.mu;  // read before the loop (see pressure_accel)
    float M[9];
#pragma unroll
    for (int e = 0; e < 9; ++e) M[e] = 0.0f;
    each_neighbor_rec<1>(src, i, k.R, k.invStep, xi, k.sG, load, [&](float4 lo, float4, float gt) {
        const f3 xij = xi - ld3(lo);
        const f3 gw = gt * xij;
        const float s = mu10 * lo.w / (length2(xij) + d001);
        const float a[3] = {xij.x, xij.y, xij.z}, g[3] = {gw.x, gw.y, gw.z};
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
            for (int cc = 0; cc < 3; ++cc) M[3 * r + cc] += s * (a[r] * g[cc]);
    });
    if (p.muB != 0.0f) {
        for (uint32_t b = 0; b < p.bodyCount; ++b) {
            const float vb = F.vb[(size_t)b * cap + i];
            if (!(vb > 0.0f)) continue;
            Tangential t;
            if (!tangential(p, k, xi, ld3(F.xb[(size_t)b * cap + i]), vb, t)) continue;
            const float a[3] = {t.pd[0].x, t.pd[0].y, t.pd[0].z};  // the reference uses direction 1 for all four
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float s = 10.0f * p.muB * t.vol / (length2(t.pd[q]) + d001);
                const float g[3] = {t.gw[q].x, t.gw[q].y, t.gw[q].z};
#pragma unroll
                for (int r = 0; r < 3; ++r)
#pragma unroll
                    for (int cc = 0; cc < 3; ++cc) M[3 * r + cc] += s * (a[r] * g[cc]);
            }
        }
    }
    const float f = dt / F.density[i];
    M3 A;
#pragma unroll
    for (int e = 0; e < 9; ++e) A.m[e] = (e % 4 == 0 ? 1.0f : 0.0f) - f * M[e];
    return inverse3(A);
}

// ComputeMatrixVecProdFunctionKernel (:758-842): y_i = u_i - dt/rho_i * (viscous acceleration of u)
// records lo = {x_j, m / rho_j}, hi = {u_j}
template <class Load>
__device__ __forceinline__ f3 visc_matvec(const SceneParams& p, const KLds& k, const Fields& F, uint32_t cap,
                                          uint32_t i, f3 vi, float dt, const Load& load, const NbrSrc& src) {
    const f3 xi = ld3(F.pos[i]);
    const float d001 = 0.01f * p.R2;
    const float mu10 = 10.0f * p.mu;  // read before the loop (see pressure_accel)
    f3 acc = mk3(0.0f, 0.0f, 0.0f);
    each_neighbor_rec<2>(src, i, k.R, k.invStep, xi, k.sG, load, [&](float4 lo, float4 hi, float g) {
        const f3 xij = xi - ld3(lo);
        const f3 gw = g * xij;
        const float s = mu10 * lo.w * dot3(vi - ld3(hi), xij) / (length2(xij) + d001);
        acc = acc + s * gw;
    });
    if (p.muB != 0.0f) {
        for (uint32_t b = 0; b < p.bodyCount; ++b) {
            const float vb = F.vb[(size_t)b * cap + i];
            if (!(vb > 0.0f)) continue;
            Tangential t;
            if (!tangential(p, k, xi, ld3(F.xb[(size_t)b * cap + i]), vb, t)) continue;
            f3 s4;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float s = 10.0f * p.muB * t.vol * dot3(vi, t.pd[q]) / (length2(t.pd[q]) + d001);
                s4 = q == 0 ? s * t.gw[q] : s4 + s * t.gw[q];
            }
            acc = acc + s4;
        }
    }
    return vi - (dt / F.density[i]) * acc;
}

}  // namespace vfd
