// sphk_walk_pairs.h -- pair arithmetic and per-particle epilogues of the two SPH walks, shared
// by every walk shape: one definition, so that every walk forms the same bits.
#pragma once

#include "sphk_walk_common.h"

namespace sphk {

namespace {

// The cubic spline (CubicSplineKernel::W_3d, src/kernels.cpp:58-66) as one expression:
// 6 W(q) / sigma = (2 - q)^3 - 4 (1 - q)^3 for q <= 1
// and (2 - q)^3 for 1 < q <= 2, i.e. t^3 - 4 s^3 with t = max(2 - q, 0), s = max(1 - q, 0).
// The walk sums an eighth of it, u^3 + s^2 (-s / 2) with u = t / 2 = max(1 - q / 2, 0): every
// rounding is that of the t-form scaled by 2^-3 (terms below 2^-126 aside), so the sums are
// the same bits / 8; u and s lie in [0, 1], where the max is the instructions' clamp bit
// (seven operations, no select).  The sum is scaled by 8 sigma / 6 at the end.
__device__ __forceinline__ float w6_shape8(float r, float half_inv_h, float inv_h) {
    const float u = __builtin_amdgcn_fmed3f(__builtin_fmaf(-half_inv_h, r, 1.0f), 0.0f, 1.0f);
    const float s = __builtin_amdgcn_fmed3f(__builtin_fmaf(-inv_h, r, 1.0f), 0.0f, 1.0f);
    return __builtin_fmaf(s * s, -0.5f * s, u * u * u);
}

// One neighbour's 6 W / 8 sigma.  Pairs the filter let through beyond the radius: with
// a radius of at least 2h they have q >= 2 (up to the rounding of sqrt, which leaves a shape
// below 2^-75) and weigh nothing, so d^2 may be formed with fused multiply-adds; with a smaller
// radius (kCut) the reference's test d^2 <= r^2, on the reference's unfused d^2, drops them.
// (The neighbour count, which needs the reference's test on every pair, is taken by the force
// walk: this walk is bound by VALU issue, the force walk by its row gathers.)
template <bool kCut>
__device__ __forceinline__ float density_weight(const float4& pi, const float4& q,
                                                const StepConsts& c, float half_inv_h) {
    float d2;
    if (kCut) {
        d2 = dist2_exact(pi.x, pi.y, pi.z, q.x, q.y, q.z);
    } else {
        const float dx = pi.x - q.x, dy = pi.y - q.y, dz = pi.z - q.z;
        d2 = __builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz));
    }
    float w = w6_shape8(__builtin_amdgcn_sqrtf(d2), half_inv_h, c.inv_h);
    if (kCut) w = d2 <= c.r2 ? w : 0.0f;
    return w;
}
template <bool kCut>
__device__ __forceinline__ float density_pair(const float4& pi, const float4& q,
                                              const StepConsts& c, float half_inv_h, float acc) {
    return __builtin_fmaf(q.w, density_weight<kCut>(pi, q, c, half_inv_h), acc);
}

// Density, the force rows of the particle (B = m/rho and C = B P / 4, so that
// m_j (P_i + P_j) / (2 rho_j) = 2 ((P_i / 4) B_j + C_j); the 2 rides on dW/dq) and rho in
// svr.w.
__device__ __forceinline__ void density_epilogue(float sum, const float4& pi, uint32_t s,
                                                 const StepConsts& c, float4* __restrict__ svr,
                                                 ForceRow* __restrict__ rows) {
    const float rho = c.sigma * (sum * (8.0f / 6.0f));  // 8.0f / 6.0f == 8 * (1.0f / 6.0f)
    float4 v = svr[s];
    v.w = rho;
    svr[s] = v;
    const float B = pi.w / rho;
    const float P = c.k_gas * (rho - c.rho0);
    rows[s].a = make_float4(pi.x, pi.y, pi.z, B);
    rows[s].b = make_float4(v.x, v.y, v.z, 0.25f * B * P);
}

__device__ __forceinline__ void integrate_clamp(float4& p, float3& v, float3 a, float dt,
                                                const StepConsts& c, const float* lo,
                                                const float* hi) {
#pragma clang fp contract(off)
    float hx = 0.5f * a.x, hy = 0.5f * a.y, hz = 0.5f * a.z;
    v.x = v.x + hx * dt;
    v.y = v.y + hy * dt;
    v.z = v.z + hz * dt;
    p.x = p.x + v.x * dt;
    p.y = p.y + v.y * dt;
    p.z = p.z + v.z * dt;
    v.x = v.x + hx * dt;
    v.y = v.y + hy * dt;
    v.z = v.z + hz * dt;
    v.x = v.x * c.damping;
    v.y = v.y * c.damping;
    v.z = v.z * c.damping;
    const float wd = -0.8f;
    if (p.x < lo[0]) {
        p.x = lo[0];
        v.x = v.x * wd;
    } else if (p.x > hi[0]) {
        p.x = hi[0];
        v.x = v.x * wd;
    }
    if (p.y < lo[1]) {
        p.y = lo[1];
        v.y = v.y * wd;
    } else if (p.y > hi[1]) {
        p.y = hi[1];
        v.y = v.y * wd;
    }
    if (p.z < lo[2]) {
        p.z = lo[2];
        v.z = v.z * wd;
    } else if (p.z > hi[2]) {
        p.z = hi[2];
        v.z = v.z * wd;
    }
}

__device__ __forceinline__ float3 final_accel(float3 fp, float3 fv, float m_i, float rho_i,
                                              const StepConsts& c) {
    // explicit fused forms: left to contraction, the choice of which product to fuse can
    // differ between the kernels that inline this, and so would their bits
    const float fx = __builtin_fmaf(fp.x, c.grad_scale, fv.x * c.lap_scale);
    const float fy = __builtin_fmaf(fp.y, c.grad_scale, fv.y * c.lap_scale);
    const float fz = __builtin_fmaf(fp.z, c.grad_scale, fv.z * c.lap_scale);
    const float m = c.formulation == 1 ? rho_i : m_i;
    const float inv_m = 1.0f / m;
    return make_float3(fx * inv_m, __builtin_fmaf(c.grav, m, fy) * inv_m, fz * inv_m);
}

// Pressure and viscosity sums of one target over neighbour rows (ForceRow a, b).
// The self pair (r = 0, v_j = v_i) and the padding slot (B = C = 0) add exactly zero.  Pairs
// the filter let through beyond the radius: with a radius of at least 2h they have q >= 2 (up
// to rounding, which leaves a Laplacian factor below 3e-8 of a neighbour's) and add nothing;
// with a smaller radius (kCut) the reference's test on its own d^2 drops them: d^2 is pushed
// to 1e30, where both kernel factors clamp to zero.
// One pair's factors: the sums are fp -= coef r and fv += cv dv, each term one fused
// multiply-add.
struct ForcePair {
    float coef, cv;
    float3 r, dv;
};

// `cnt` counts the pairs that pass the reference's test d^2 <= r^2 on the reference's
// unfused d^2 (the particle itself included): the engine's neighbour statistics.
template <bool kCut>
__device__ __forceinline__ ForcePair force_pair(const float4& pi, const float3& vi,
                                                float p_quarter, const float4& a, const float4& b,
                                                const StepConsts& c, uint32_t& cnt) {
    ForcePair o;
    o.r = make_float3(pi.x - a.x, pi.y - a.y, pi.z - a.z);
    float d2 = dist2_exact(pi.x, pi.y, pi.z, a.x, a.y, a.z);
    const bool in = d2 <= c.r2;
    cnt += in ? 1u : 0u;
    if (kCut) d2 = in ? d2 : 1e30f;
    const float rinv = __builtin_amdgcn_rsqf(fmaxf(d2, 1e-30f));
    const float rl = d2 * rinv;
    // u = (2 - q) / 2 and s = 1 - q, clamped to [0, 1] by the instructions' clamp bit
    // (seven operations, no select): dwq = (s - u)(s + u) = s^2 - u^2 is q (3q - 4) / 4
    // for q <= 1 and -(2 - q)^2 / 4 beyond, proportional to dW/dq; lap = u - 2 s is
    // (3q - 2) / 2 and (2 - q) / 2.  grad_scale and lap_scale carry the constant factors.
    const float u = __builtin_amdgcn_fmed3f(__builtin_fmaf(-0.5f * c.inv_h, rl, 1.0f), 0.0f, 1.0f);
    const float s = __builtin_amdgcn_fmed3f(__builtin_fmaf(-c.inv_h, rl, 1.0f), 0.0f, 1.0f);
    const float dwq = (s - u) * (s + u);
    const float lap = __builtin_fmaf(-2.0f, s, u);
    // gradW is zero below |r| = 1e-6 (src/kernels.cpp:96-98)
    const float dw = rl >= 1e-6f ? dwq : 0.0f;
    o.coef = __builtin_fmaf(p_quarter, a.w, b.w) * dw * rinv;
    o.cv = a.w * lap;
    o.dv = make_float3(b.x - vi.x, b.y - vi.y, b.z - vi.z);
    return o;
}

struct ForceSums {
    float3 fp = make_float3(0.f, 0.f, 0.f);
    float3 fv = make_float3(0.f, 0.f, 0.f);
    template <bool kCut>
    __device__ __forceinline__ void add(const float4& pi, const float3& vi, float p_quarter,
                                        const float4& a, const float4& b, const StepConsts& c,
                                        uint32_t& cnt) {
        const ForcePair p = force_pair<kCut>(pi, vi, p_quarter, a, b, c, cnt);
        fp.x = __builtin_fmaf(-p.coef, p.r.x, fp.x);
        fp.y = __builtin_fmaf(-p.coef, p.r.y, fp.y);
        fp.z = __builtin_fmaf(-p.coef, p.r.z, fp.z);
        fv.x = __builtin_fmaf(p.cv, p.dv.x, fv.x);
        fv.y = __builtin_fmaf(p.cv, p.dv.y, fv.y);
        fv.z = __builtin_fmaf(p.cv, p.dv.z, fv.z);
    }
    // the sums (and the count) formed here, before whatever follows (see pinned)
    __device__ __forceinline__ void pin(uint32_t& cnt) {
        asm volatile("" : "+v"(fp.x), "+v"(fp.y), "+v"(fp.z), "+v"(fv.x), "+v"(fv.y),
                     "+v"(fv.z), "+v"(cnt));
    }
};

// Acceleration, leapfrog, clamp and the caller-order writes of one target.
__device__ __forceinline__ void force_epilogue(const ForceSums& f, float4 pi, float3 vi,
                                               float rho_i, float P_i, uint32_t s,
                                               const SceneGrid& g, const StepConsts& c,
                                               const uint32_t* __restrict__ sid,
                                               const float* __restrict__ dt_dev, float dt_arg,
                                               float4* __restrict__ pm, float4* __restrict__ vel,
                                               float4* __restrict__ acc_out,
                                               float* __restrict__ rho_out,
                                               float* __restrict__ prs_out) {
    const float3 a = final_accel(f.fp, f.fv, pi.w, rho_i, c);
    const float dt = dt_dev ? *dt_dev : dt_arg;
    float3 v = vi;
    float4 p = pi;
    integrate_clamp(p, v, a, dt, c, g.lo, g.hi);
    const uint32_t id = sid[s];
    pm[id] = p;
    vel[id] = make_float4(v.x, v.y, v.z, 0.0f);
    acc_out[id] = make_float4(a.x, a.y, a.z, 0.0f);
    rho_out[id] = rho_i;
    prs_out[id] = P_i;
}

}  // namespace

}  // namespace sphk
