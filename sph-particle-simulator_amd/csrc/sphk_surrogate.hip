// sphk_surrogate.hip -- kernels of the learned macro-step surrogate: operand packing, the
// edge pass (message layer 1 on MFMA over the stored neighbour words), the row GEMMs of the
// node MLP and of the backward pass, weight-gradient reductions, loss, Adam, and the
// macro-step integration.  Network and layouts: sphk_surrogate.h.
#include <hip/hip_runtime.h>

#include "sphk_surrogate.h"
#include "sphk_walk_common.h"

namespace sphk {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16 mfma16(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 load8(const __bf16* p) {
    return *reinterpret_cast<const bf16x8*>(p);
}

__device__ __forceinline__ bf16x8 zero8() {
    bf16x8 z;
#pragma unroll
    for (int i = 0; i < 8; ++i) z[i] = (__bf16)0.0f;
    return z;
}

__device__ __forceinline__ f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.0f;
    return z;
}

// Row of accumulator register v for lane half h.
__device__ __forceinline__ uint32_t acc_row(int v, uint32_t h) {
    return (uint32_t)((v >> 2) * 8 + (v & 3)) + 4u * h;
}

// W(|r|) / W(0) of the cubic spline.  kOrdered: in the operation order of the oracle (no
// contraction).  Otherwise by clamped cubes, 2 (u^3 - s^3 / 2) with u = max(1 - q / 2, 0) and
// s = max(1 - q, 0) (the density walk's form: 8 operations, no select, against 13; each bracket of
// the piecewise form is this polynomial, to FP32 rounding).
template <bool kOrdered>
__device__ __forceinline__ float w_feature(float r, float inv_h) {
#pragma clang fp contract(off)
    if (kOrdered) {
        const float q = r * inv_h;
        const float q2 = q * q;
        const float win = (2.0f / 3.0f - q2) + 0.5f * q2 * q;
        const float t = 2.0f - q;
        const float wout = (1.0f / 6.0f) * t * t * t;
        return 1.5f * (q <= 1.0f ? win : (q <= 2.0f ? wout : 0.0f));
    }
    const float u = __builtin_amdgcn_fmed3f(__builtin_fmaf(-0.5f * inv_h, r, 1.0f), 0.0f, 1.0f);
    const float s = __builtin_amdgcn_fmed3f(__builtin_fmaf(-inv_h, r, 1.0f), 0.0f, 1.0f);
    return 2.0f * __builtin_fmaf(s * s, -0.5f * s, u * u * u);
}

// Edge features of one pair in FP32 (any values for a non-edge: the caller zeroes them).
template <bool kOrdered>
__device__ __forceinline__ void edge_values(float4 pi, float4 vi, float4 pj, float4 vj,
                                            float d2, const SurScales& sc, float (&f)[9]) {
#pragma clang fp contract(off)
    const float rx = pi.x - pj.x, ry = pi.y - pj.y, rz = pi.z - pj.z;
    const float rl = __builtin_amdgcn_sqrtf(d2);
    f[0] = rx * sc.inv_r;
    f[1] = ry * sc.inv_r;
    f[2] = rz * sc.inv_r;
    f[3] = (vi.x - vj.x) * sc.inv_v;
    f[4] = (vi.y - vj.y) * sc.inv_v;
    f[5] = (vi.z - vj.z) * sc.inv_v;
    f[6] = rl * sc.inv_r;
    f[7] = w_feature<kOrdered>(rl, sc.inv_h);
    f[8] = (vj.w - sc.rho0) * sc.rho_scale;
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Edge features of one pair rounded to bf16 (round to nearest even, two per conversion),
// zero when `edge` is false: features 0..7, and [1, feature 8] (neighbour density) packed.
template <bool kOrdered>
__device__ __forceinline__ void edge_features(bool edge, float4 pi, float4 vi, float4 pj,
                                              float4 vj, float d2, const SurScales& sc,
                                              uint32_t (&e)[4], uint32_t& ext) {
    float f[9];
    edge_values<kOrdered>(pi, vi, pj, vj, d2, sc, f);
    auto pack = [&](float a, float b) {
        const f32x2 v = {a, b};
        const uint32_t bits = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
        return edge ? bits : 0u;
    };
#pragma unroll
    for (int k = 0; k < 4; ++k) e[k] = pack(f[2 * k], f[2 * k + 1]);
    ext = pack(1.0f, f[8]);
}

__device__ __forceinline__ uint32_t bits16(__bf16 x) {
    return (uint32_t)__builtin_bit_cast(uint16_t, x);
}

// B operands of message layer 1 for hidden tile hb (n = 32 hb + l % 32).  The K range of an
// MFMA is 16: the lower lanes supply W1 columns 0..7, the upper ones [b1, W1 column 8, 0 ...]
// (k = 8, 9), so W1 e + b1 is one product.  kSwapped: the two halves of K the other way round.
template <bool kSwapped = false>
__device__ __forceinline__ void load_layer1(const __bf16* __restrict__ pk, uint32_t lane,
                                            bf16x8 (&B)[4]) {
    const uint32_t col = lane & 31u;
    const bool hi = kSwapped ? lane < 32u : lane >= 32u;
#pragma unroll
    for (int hb = 0; hb < 4; ++hb) {
        const uint32_t n = 32u * hb + col;
        const bf16x8 w = load8(pk + kPkW1 + n * 8u);
        bf16x8 b = zero8();
        b[0] = pk[kPkB1 + n];
        b[1] = pk[kPkW1r + n];
        B[hb] = hi ? b : w;
    }
}

// A operands: row r of block b is the edge of lane 32 b + r, its features 0..7 in the lower
// lanes (k = 0..7) and [1, feature 8, 0 ...] in the upper ones (zeros for a padding row, which is
// then exactly zero).  One v_permlane32_swap per dword trades the upper lanes' features for
// the lower lanes' tail, which is both operands at once.  kSwapped: block 1 has the halves of
// K the other way round (from a second swap), for B operands loaded so.
template <bool kSwapped>
__device__ __forceinline__ void layer1_a(const uint32_t (&e)[4], uint32_t ext, bf16x8& a0,
                                         bf16x8& a1) {
    uint4 x, y;
    uint32_t* xp = &x.x;
    uint32_t* yp = &y.x;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const uint32_t t = k == 0 ? ext : 0u;
        const auto r = __builtin_amdgcn_permlane32_swap(e[k], t, false, false);
        xp[k] = r[0];
        yp[k] = kSwapped ? __builtin_amdgcn_permlane32_swap(t, e[k], false, false)[1] : r[1];
    }
    a0 = __builtin_bit_cast(bf16x8, x);
    a1 = __builtin_bit_cast(bf16x8, y);
}

typedef short short2v __attribute__((ext_vector_type(2)));

// All eight values with their sign flipped.
__device__ __forceinline__ bf16x8 negated(bf16x8 x) {
    uint4 w = __builtin_bit_cast(uint4, x);
    w.x ^= 0x80008000u;
    w.y ^= 0x80008000u;
    w.z ^= 0x80008000u;
    w.w ^= 0x80008000u;
    return __builtin_bit_cast(bf16x8, w);
}

// 16-bit masks of a pair: all ones where the value's sign bit is set (a in the low half).
__device__ __forceinline__ uint32_t neg_masks(float a, float b) {
    const uint32_t hi =
        __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(short2v, hi) >> (short)15);
}

constexpr int kEdgeWaves = 2;   // one chunk per workgroup: 32 targets per wavefront
constexpr int kStage = 136;     // LDS row stride (bf16) of staged 128-wide rows
constexpr int kStageX = 152;    // LDS row stride (bf16) of staged node-input rows

// One macro-step of a particle: v' = d^k v + a T, x' = x + T (v + v') / 2, then the wall
// clamp of the plain step (src/particle.cpp:122-153).
__device__ __forceinline__ void macro_integrate(float4& p, float3& v1, float3 v0, float3 a,
                                                float T, float dk, const SceneGrid& g) {
#pragma clang fp contract(off)
    v1 = make_float3(dk * v0.x + a.x * T, dk * v0.y + a.y * T, dk * v0.z + a.z * T);
    p.x = p.x + (0.5f * T) * (v0.x + v1.x);
    p.y = p.y + (0.5f * T) * (v0.y + v1.y);
    p.z = p.z + (0.5f * T) * (v0.z + v1.z);
    const float wd = -0.8f;
    if (p.x < g.lo[0]) { p.x = g.lo[0]; v1.x = v1.x * wd; } else if (p.x > g.hi[0]) { p.x = g.hi[0]; v1.x = v1.x * wd; }
    if (p.y < g.lo[1]) { p.y = g.lo[1]; v1.y = v1.y * wd; } else if (p.y > g.hi[1]) { p.y = g.hi[1]; v1.y = v1.y * wd; }
    if (p.z < g.lo[2]) { p.z = g.lo[2]; v1.z = v1.z * wd; } else if (p.z > g.hi[2]) { p.z = g.hi[2]; v1.z = v1.z * wd; }
}

// Row-tile GEMM of one wavefront: D[t][n] (+)= sum_k A[t][k] Bt[n][k] for the 32 target rows
// of A (LDS, row stride lda) and the 4 output tiles of Bt (global, row stride ldb), K = 16 ks.
__device__ __forceinline__ void tile_gemm(f32x16 (&d)[4], const __bf16* A, int lda,
                                          const __bf16* __restrict__ Bt, int ldb, int ks,
                                          int ntiles, uint32_t lane) {
    const uint32_t col = lane & 31u, h = lane >> 5;
    for (int k = 0; k < ks; ++k) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(A + col * lda + 16 * k + 8 * h);
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (t < ntiles)
                d[t] = mfma16(a, load8(Bt + (size_t)(32 * t + col) * ldb + 16 * k + 8 * h), d[t]);
    }
}

// Activation staging of one wavefront (reuses the list once the walk is done).
struct EpiLds {
    __bf16 s[32 * kStage];      // S, later z (row stride kStage)
    __bf16 x[32 * kStageX];     // node input (row stride kStageX)
};

static_assert(sizeof(EpiLds) <= sizeof(WalkLds), "activation staging reuses the list");

}  // namespace

// ---------------------------------------------------------------------------
// operand packing
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_sur_pack(const float* __restrict__ p,
                                                  __bf16* __restrict__ pk,
                                                  float* __restrict__ pf) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < kPkTotal) {
        float v;
        if (i < kPkB1) {
            v = p[kOffW1 + (i / 8u) * kSurNF + i % 8u];
        } else if (i < kPkW1r) {
            v = p[kOffB1 + (i - kPkB1)];
        } else if (i < kPkW2) {
            v = p[kOffW1 + (i - kPkW1r) * kSurNF + 8u];
        } else if (i < kPkW2T) {
            v = p[kOffW2 + (i - kPkW2)];
        } else if (i < kPkWn1) {
            const uint32_t t = i - kPkW2T, in = t / 128u, out = t % 128u;
            v = p[kOffW2 + out * 128u + in];
        } else if (i < kPkWn1T) {
            const uint32_t t = i - kPkWn1, out = t / kSurRow, in = t % kSurRow;
            v = in < (uint32_t)kSurNodeIn ? p[kOffWn1 + out * kSurNodeIn + in] : 0.0f;
        } else if (i < kPkWn2) {
            const uint32_t t = i - kPkWn1T, in = t / 128u, out = t % 128u;
            v = in < (uint32_t)kSurNodeIn ? p[kOffWn1 + out * kSurNodeIn + in] : 0.0f;
        } else if (i < kPkWn2T) {
            const uint32_t t = i - kPkWn2, out = t / 128u, in = t % 128u;
            v = out < 3u ? p[kOffWn2 + out * 128u + in] : 0.0f;
        } else {
            const uint32_t t = i - kPkWn2T, in = t / 32u, out = t % 32u;
            v = out < 3u ? p[kOffWn2 + out * 128u + in] : 0.0f;
        }
        pk[i] = (__bf16)v;
    }
    if (i < kFTotal) {
        float v;
        if (i < kFB1) v = p[kOffW1 + i];
        else if (i < kFB2) v = p[kOffB1 + (i - kFB1)];
        else if (i < kFBn1) v = p[kOffB2 + (i - kFB2)];
        else if (i < kFBn2) v = p[kOffBn1 + (i - kFBn1)];
        else v = (i - kFBn2) < 3u ? p[kOffBn2 + (i - kFBn2)] : 0.0f;
        pf[i] = (float)(__bf16)v;
    }
}

// ---------------------------------------------------------------------------
// forward pass.  Per chunk (two wavefronts of 32 targets):
//   edge walk: S_i = c * sum_j ReLU(W1 e_ij + b1) through
//       sum ReLU(u) = (sum u + sum |u|) / 2,  sum_j u_ij = W1 (sum_j e_ij) + n_i b1,
//     so the per-edge work after the MFMA is one add with an |.| modifier per value.  The
//     two MFMA blocks of a step hold the two lanes' edges of the same 32 targets.
//   node MLP on MFMA from LDS: m = W2 S + c n b2, z = ReLU(Wn1 x + bn1), out = Wn2 z + bn2.
// kIntegrate: the macro-step is applied and written to the caller-order state.  Otherwise
// the S, X, Z and OUT rows are written for the backward pass (batch: rows 64 b + lane;
// no batch: rows = sorted slots).
// Bound by VALU issue (two wavefronts per SIMD, 204 operations beside the 8 products of a step
// of 64 edges, 128 of them the sums of |u|).  The inference walk takes what is cheapest: long
// windows, the operands of both blocks from one swap, the shape by clamped cubes, and the
// sums of a product under the next product.  The rows for the backward pass keep the order of
// edges, products and sums they have always had: a sum rounded another way flips some of the
// bf16 roundings behind it (gradients then move by up to 1e-3 of their largest).
// Macro-step of 295,000 particles 759 -> 664 us.
// ---------------------------------------------------------------------------
template <bool kIntegrate>
__global__ __launch_bounds__(64 * kEdgeWaves) __attribute__((amdgpu_waves_per_eu(2))) void
k_sur_forward(WalkBuffers wb, const uint32_t* __restrict__ batch, uint32_t nbatch,
              const float4* __restrict__ spm, const float4* __restrict__ svr,
              const uint32_t* __restrict__ skey, const uint32_t* __restrict__ sid,
              const uint32_t* __restrict__ cs, StepConsts c, const SceneGrid* __restrict__ scenes,
              const __bf16* __restrict__ pk, const float* __restrict__ pf, SurScales sc,
              SurRows rows, SurStep step) {
    __shared__ WalkLds lds_all[kEdgeWaves];
    __shared__ float lout_all[kEdgeWaves][32][4];
    __shared__ float lcnt_all[kEdgeWaves][32];
    const uint32_t half = uni(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t col = lane & 31u, h = lane >> 5;
    WalkLds& L = lds_all[half];
    const uint32_t b_idx = xcd_unit(batch ? nbatch : uni(wb.nitems[0]), 1, 0);
    if (b_idx == ~0u) return;
    const uint32_t item = batch ? uni(batch[b_idx]) : b_idx;
    const uint32_t clane = 32u * half + col;  // this lane's target within the chunk
    Chunk ch;
    uint32_t s;
    bool active;
    float4 pi;
    if (!load_chunk(item, wb.items, wb.desc, wb.nitems, skey, spm, c, scenes, clane, ch, s, active,
                    pi))
        return;
    const float4 vi = active ? svr[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    constexpr bool kOrdered = !kIntegrate;
    bf16x8 B[4], B1[4];
    load_layer1(pk, lane, B);
    if constexpr (kOrdered) load_layer1<true>(pk, lane, B1);
    f32x16 acc[4];
#pragma unroll
    for (int hb = 0; hb < 4; ++hb) acc[hb] = zero16();
    // sum_j (e_ij, 1) of this lane's edges, of the values the layer-1 product sees (sum u is
    // subtracted from sum |u| for hidden units that are mostly inactive).  On the VALU: an MFMA
    // against a unit matrix was 2 % faster here, but its accumulation rounds less exactly
    // (gradients 4e-4 off instead of 3e-7).
    float se[10];
#pragma unroll
    for (int k = 0; k < 10; ++k) se[k] = 0.0f;
    walk_pairs<kIntegrate>(item, ch, s, active, pi, clane, wb, spm, svr, cs, c, L, lane,
               [&](bool edge, float4 pj, float4 vj, float d2) {
                   uint32_t fe[4], ext;
                   edge_features<kOrdered>(edge, pi, vi, pj, vj, d2, sc, fe, ext);
                   bf16x8 a[2];
                   layer1_a<kOrdered>(fe, ext, a[0], a[1]);
#pragma unroll
                   for (int k = 0; k < 5; ++k) {
                       const uint32_t w = k < 4 ? fe[k] : ext;
                       se[2 * k] += __uint_as_float(w << 16);
                       se[2 * k + 1] += __uint_as_float(w & 0xffff0000u);
                   }
                   if constexpr (kOrdered) {
#pragma unroll
                       for (int hb = 0; hb < 4; ++hb) {
                           const f32x16 d0 = mfma16(a[0], B[hb], zero16());
                           const f32x16 d1 = mfma16(a[1], B1[hb], zero16());
#pragma unroll
                           for (int v = 0; v < 16; ++v) acc[hb][v] += fabsf(d0[v]) + fabsf(d1[v]);
                       }
                   } else {
                       f32x16 d[2];
                       d[0] = mfma16(a[0], B[0], zero16());
#pragma unroll
                       for (int k = 0; k < 8; ++k) {
                           const int n = k + 1;
                           if (n < 8) d[n & 1] = mfma16(a[n & 1], B[n >> 1], zero16());
                           __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                           for (int v = 0; v < 16; ++v) acc[k >> 1][v] += fabsf(d[k & 1][v]);
                           __builtin_amdgcn_sched_barrier(0);
                       }
                   }
               });
    // sum u + sum |u| = [sum e, n] W1aug^T + acc, on MFMA with the accumulators as C.  The
    // sums enter as three bf16 parts (x = x0 + x1 + x2 to about 2^-27 relative): sum u is
    // cancelled against sum |u| for hidden units that are mostly inactive.
    // both lanes of a target hold half of its sums: 0..7, n, 8
#pragma unroll
    for (int k = 0; k < 10; ++k) se[k] += __shfl_xor(se[k], 32);
    const float ne = se[8];
    float* lcnt = lcnt_all[half];
    if (h == 0u) lcnt[col] = ne;
    {
        // lanes 0..31 supply k = 0..7 (feature sums 0..7), lanes 32..63 k = 8, 9 (the edge
        // count, which meets b1, and feature sum 8, which meets W1 column 8)
        float x[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) x[k] = h == 0u ? se[k] : k < 2 ? se[8 + k] : 0.0f;
#pragma unroll
        for (int part = 0; part < 3; ++part) {
            bf16x8 a;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                a[k] = (__bf16)x[k];
                x[k] = x[k] - (float)a[k];
            }
#pragma unroll
            for (int hb = 0; hb < 4; ++hb) acc[hb] = mfma16(a, B[hb], acc[hb]);
        }
    }
    wave_sync();  // the list is free from here on
    EpiLds& E = *reinterpret_cast<EpiLds*>(&L);
    const float half_c = 0.5f * sc.msg_scale;
#pragma unroll
    for (int hb = 0; hb < 4; ++hb)
#pragma unroll
        for (int v = 0; v < 16; ++v)
            E.s[acc_row(v, h) * kStage + 32u * hb + col] = (__bf16)(half_c * acc[hb][v]);
    // node input tail: [rho, v, 1, 0 ...] (column 132 = 1 is the bias column of dbn1)
    if (h == 0u) {
#pragma clang fp contract(off)
        const bool a = active;
        __bf16* xr = E.x + col * kStageX + 128;
        xr[0] = (__bf16)(a ? (vi.w - sc.rho0) * sc.rho_scale : 0.0f);
        xr[1] = (__bf16)(a ? vi.x * sc.inv_v : 0.0f);
        xr[2] = (__bf16)(a ? vi.y * sc.inv_v : 0.0f);
        xr[3] = (__bf16)(a ? vi.z * sc.inv_v : 0.0f);
        xr[4] = (__bf16)(a ? 1.0f : 0.0f);
#pragma unroll
        for (int k = 5; k < 16; ++k) xr[k] = (__bf16)0.0f;
    }
    wave_sync();
    // m = W2 S + c n b2 -> X[:, :128]
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = zero16();
    tile_gemm(acc, E.s, kStage, pk + kPkW2, 128, 8, 4, lane);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint32_t n = 32u * t + col;
        const float b2 = pf[kFB2 + n];
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t r = acc_row(v, h);
            E.x[r * kStageX + n] = (__bf16)(acc[t][v] + sc.msg_scale * lcnt[r] * b2);
        }
    }
    wave_sync();
    // rows for the backward pass: S (and its c n column) before z overwrites it
    const uint32_t len = ch.s_end - ch.s0;
    const bool all_rows = batch != nullptr;
    const size_t row0 = batch ? 64u * (size_t)b_idx : (size_t)ch.s0;
    if constexpr (!kIntegrate) {
        for (uint32_t idx = lane; idx < 32u * 18u; idx += 64u) {
            const uint32_t tl = idx / 18u, part = idx % 18u;
            const uint32_t cl = 32u * half + tl;
            if (!all_rows && cl >= len) continue;
            uint4 val = make_uint4(0u, 0u, 0u, 0u);
            if (part < 16u) {
                val = *reinterpret_cast<const uint4*>(E.s + tl * kStage + part * 8u);
            } else if (part == 16u && cl < len) {
                val.x = bits16((__bf16)(sc.msg_scale * lcnt[tl]));
            }
            *reinterpret_cast<uint4*>(rows.S + (row0 + cl) * kSurRow + part * 8u) = val;
            uint4 xv = make_uint4(0u, 0u, 0u, 0u);
            if (cl < len) xv = *reinterpret_cast<const uint4*>(E.x + tl * kStageX + part * 8u);
            *reinterpret_cast<uint4*>(rows.X + (row0 + cl) * kSurRow + part * 8u) = xv;
        }
        wave_sync();
    }
    // z = ReLU(Wn1 x + bn1) -> E.s
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = zero16();
    tile_gemm(acc, E.x, kStageX, pk + kPkWn1, kSurRow, 9, 4, lane);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const uint32_t n = 32u * t + col;
        const float bn1 = pf[kFBn1 + n];
#pragma unroll
        for (int v = 0; v < 16; ++v)
            E.s[acc_row(v, h) * kStage + n] = (__bf16)fmaxf(acc[t][v] + bn1, 0.0f);
    }
    wave_sync();
    // out = Wn2 z + bn2
    acc[0] = zero16();
    tile_gemm(acc, E.s, kStage, pk + kPkWn2, 128, 8, 1, lane);
    float(*lout)[4] = lout_all[half];
    if (col < 3u) {
        const float bn2 = pf[kFBn2 + col];
#pragma unroll
        for (int v = 0; v < 16; ++v) lout[acc_row(v, h)][col] = acc[0][v] + bn2;
    }
    wave_sync();
    if constexpr (kIntegrate) {
        if (h == 0u && active) {
            const float3 a = make_float3(sc.acc_scale * lout[col][0], sc.acc_scale * lout[col][1],
                                         sc.acc_scale * lout[col][2]);
            float4 p = pi;
            float3 v1;
            const SceneGrid& g = scenes[ch.scene];
            macro_integrate(p, v1, make_float3(vi.x, vi.y, vi.z), a, step.T, step.dk, g);
            const uint32_t id = sid[s];
            step.pm[id] = p;
            step.vel[id] = make_float4(v1.x, v1.y, v1.z, 0.0f);
            step.acc[id] = make_float4(a.x, a.y, a.z, 0.0f);
            step.rho[id] = vi.w;
            step.prs[id] = c.k_gas * (vi.w - c.rho0);
        }
    } else {
        // Z rows (+ bias column) and OUT rows
        for (uint32_t idx = lane; idx < 32u * 18u; idx += 64u) {
            const uint32_t tl = idx / 18u, part = idx % 18u;
            const uint32_t cl = 32u * half + tl;
            if (!all_rows && cl >= len) continue;
            uint4 val = make_uint4(0u, 0u, 0u, 0u);
            if (cl < len) {
                if (part < 16u) val = *reinterpret_cast<const uint4*>(E.s + tl * kStage + part * 8u);
                else if (part == 16u) val.x = bits16((__bf16)1.0f);
            }
            *reinterpret_cast<uint4*>(rows.Z + (row0 + cl) * kSurRow + part * 8u) = val;
        }
        if (h == 0u && (all_rows || active)) {
            const size_t row = row0 + clane;
            rows.OUT[row] = active ? make_float4(lout[col][0], lout[col][1], lout[col][2], 0.0f)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
            rows.cnt[row] = active ? sc.msg_scale * ne : 0.0f;
            rows.rowslot[row] = active ? s : kSurNoSlot;
        }
    }
}

// ---------------------------------------------------------------------------
// Loss and the backward pass through the node MLP and the hoisted message layer, 32 batch rows
// per wavefront:
//   d = OUT - target (zero without a slot), DOUT = 2 d, DZ = (Wn2^T DOUT) [Z > 0],
//   DM = Wn1^T DZ, DS = c W2^T DM.
// One launch instead of a loss kernel and three row GEMMs: the rows stay in one LDS tile per
// wavefront, which feeds the next product's A operand and the 16-byte row stores, and Z is the
// only activation read.  Bound by memory: 0.3 KB read and 0.8 KB written a row.
// 65,536 rows: loss and products 61 -> 32 us.
// Per workgroup: the partial sum of squared errors and the number of rows with a slot.
// ---------------------------------------------------------------------------
constexpr uint32_t kNodeWaves = 4;

__global__ __launch_bounds__(64 * kNodeWaves) void k_sur_node_bwd(
    const float4* __restrict__ out, const uint32_t* __restrict__ rowslot,
    const uint32_t* __restrict__ sid, const float4* __restrict__ target, uint32_t R,
    const __bf16* __restrict__ Z, const __bf16* __restrict__ pk, float msg_scale, SurGradRows g,
    float* __restrict__ loss_part) {
    __shared__ alignas(16) __bf16 stage_all[kNodeWaves][32 * kStage];
    __shared__ float red[kNodeWaves], redc[kNodeWaves];
    const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    const uint32_t h = lane >> 5, col = lane & 31u;
    const uint32_t row0 = (blockIdx.x * kNodeWaves + wave) * 32u;
    __bf16* E = stage_all[wave];
    float l = 0.0f, cnt = 0.0f;
    if (row0 < R) {  // R is a multiple of 32
        const uint32_t row = row0 + col;
        // 16-byte pieces of 128-wide rows: lane l takes pieces l, l + 64, ... of the 32 x 16
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t r = 4u * k + (lane >> 4), piece = lane & 15u;
            *reinterpret_cast<uint4*>(E + r * kStage + 8u * piece) =
                *reinterpret_cast<const uint4*>(Z + (size_t)(row0 + r) * kSurRow + 8u * piece);
        }
        bf16x8 a = zero8();
        if (h == 0u) {
            const uint32_t slot = rowslot[row];
            float d0 = 0.0f, d1 = 0.0f, d2 = 0.0f;
            if (slot != kSurNoSlot) {
                cnt = 1.0f;
                const float4 t = target[sid[slot]];
                const float4 o = out[row];
                d0 = o.x - t.x;
                d1 = o.y - t.y;
                d2 = o.z - t.z;
                l = (d0 * d0 + d1 * d1) + d2 * d2;
            }
            a[0] = (__bf16)(2.0f * d0);
            a[1] = (__bf16)(2.0f * d1);
            a[2] = (__bf16)(2.0f * d2);
            const uint4 w = __builtin_bit_cast(uint4, a);
            *reinterpret_cast<uint2*>(g.DOUT + (size_t)row * kSurOutRow) = make_uint2(w.x, w.y);
        }
        wave_sync();
        f32x16 acc[4];
        // rows of the tile to global memory, 16 bytes a lane
        auto store_rows = [&](__bf16* dst) {
            wave_sync();
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                const uint32_t r = 4u * k + (lane >> 4), piece = lane & 15u;
                *reinterpret_cast<uint4*>(dst + (size_t)(row0 + r) * 128u + 8u * piece) =
                    *reinterpret_cast<const uint4*>(E + r * kStage + 8u * piece);
            }
        };
        // DZ: the three output gradients are one K step (k = 0..2)
#pragma unroll
        for (int t = 0; t < 4; ++t)
            acc[t] = mfma16(a, load8(pk + kPkWn2T + (32u * t + col) * 32u + 8u * h), zero16());
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                __bf16* e = E + acc_row(v, h) * kStage + 32u * t + col;
                *e = (__bf16)((float)*e > 0.0f ? acc[t][v] : 0.0f);
            }
        store_rows(g.DZ);
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = zero16();
        tile_gemm(acc, E, kStage, pk + kPkWn1T, 128, 8, 4, lane);
        wave_sync();
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                E[acc_row(v, h) * kStage + 32u * t + col] = (__bf16)acc[t][v];
        store_rows(g.DM);
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = zero16();
        tile_gemm(acc, E, kStage, pk + kPkW2T, 128, 8, 4, lane);
        wave_sync();
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                E[acc_row(v, h) * kStage + 32u * t + col] = (__bf16)(msg_scale * acc[t][v]);
        store_rows(g.DS);
    }
    for (int off = 32; off > 0; off >>= 1) {
        l += __shfl_xor(l, off);
        cnt += __shfl_xor(cnt, off);
    }
    if (lane == 0) {
        red[wave] = l;
        redc[wave] = cnt;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        loss_part[2 * blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
        loss_part[2 * blockIdx.x + 1] = (redc[0] + redc[1]) + (redc[2] + redc[3]);
    }
}

// ---------------------------------------------------------------------------
// weight-gradient partials P^T Q of a slab of kSurSlabRows rows (K = rows), one workgroup per
// slab and product.  An operand needs 8 consecutive rows of one column; which columns form a
// 32-wide tile is free, so a lane loads the 2 (P) or 4 (Q) neighbouring columns of 8 rows with
// wide, coalesced loads and its column t belongs to tile t: a byte permute per operand dword
// does the transpose, no LDS.  The 16 columns of Q beyond 128 (the bias columns and the last
// node inputs) are a fifth tile.  The next K step's rows are requested before this one's
// products.  Bound by the read of the rows (a K step of 16: 4 KB of P, 0.1 KB in the output
// layer, and 4.6 KB of Q): 65,536 rows,
// three products 218 -> 25 us, against one 32 x 32 tile per wavefront with 2-byte loads.
// kMT 2: P has 128 columns; two wavefronts split them, two pairs split the rows.
// kMT 1: P is the output gradient (3 of 4 columns); the four wavefronts split the rows.
// ---------------------------------------------------------------------------
struct WgradStep {
    uint32_t p[8];
    uint2 q[8];
    uint32_t x[8];
};

template <int kMT>
__device__ __forceinline__ void wgrad_load(WgradStep& w, const __bf16* __restrict__ P,
                                           const __bf16* __restrict__ Q, uint32_t r,
                                           uint32_t lane) {
    const uint32_t h = lane >> 5, col = lane & 31u;
#pragma unroll
    for (uint32_t i = 0; i < 8u; ++i) {
        const size_t row = r + 8u * h + i;
        if (kMT == 2)
            w.p[i] = *reinterpret_cast<const uint32_t*>(P + row * 128u + 2u * col);
        else
            w.p[i] = bits16(P[row * kSurOutRow + min(col, 3u)]);  // column 3 is zero
        w.q[i] = *reinterpret_cast<const uint2*>(Q + row * kSurRow + 4u * col);
        w.x[i] = bits16(Q[row * kSurRow + 128u + min(col, 15u)]);
    }
}

// Operand of one column from 8 rows' dwords: its low (kHi false) or high halves.
template <bool kHi>
__device__ __forceinline__ bf16x8 column8(const uint32_t (&d)[8]) {
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        w[k] = __builtin_amdgcn_perm(d[2 * k + 1], d[2 * k], kHi ? 0x07060302u : 0x05040100u);
    return __builtin_bit_cast(bf16x8, make_uint4(w[0], w[1], w[2], w[3]));
}

template <int kMT>
__device__ __forceinline__ void wgrad_mfma(const WgradStep& w, f32x16 (&acc)[kMT][5]) {
    bf16x8 a[kMT];
    a[0] = column8<false>(w.p);
    if (kMT == 2) a[kMT - 1] = column8<true>(w.p);
    uint32_t lo[8], hi[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        lo[i] = w.q[i].x;
        hi[i] = w.q[i].y;
    }
    const bf16x8 b[5] = {column8<false>(lo), column8<true>(lo), column8<false>(hi),
                         column8<true>(hi), column8<false>(w.x)};
#pragma unroll
    for (int m = 0; m < kMT; ++m)
#pragma unroll
        for (int n = 0; n < 5; ++n) acc[m][n] = mfma16(a[m], b[n], acc[m][n]);
}

template <int kMT>
__device__ __forceinline__ void wgrad_slab(const __bf16* __restrict__ P,
                                           const __bf16* __restrict__ Q, uint32_t R,
                                           uint32_t slab, float* __restrict__ part,
                                           float* __restrict__ fold) {
    constexpr uint32_t kParts = kMT == 2 ? 2u : 4u;  // row parts of the slab
    constexpr uint32_t kRows = kSurSlabRows / kParts;
    static_assert(kRows % 32u == 0u, "K steps are taken in pairs");
    const uint32_t wave = uni(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    const uint32_t h = lane >> 5, col = lane & 31u;
    const uint32_t mhalf = kMT == 2 ? wave & 1u : 0u;
    const uint32_t rp = kMT == 2 ? wave >> 1 : wave;
    const uint32_t r_begin = slab * kSurSlabRows + rp * kRows;
    const uint32_t r_end = min(R, r_begin + kRows);  // R is a multiple of 64
    f32x16 acc[kMT][5];
#pragma unroll
    for (int m = 0; m < kMT; ++m)
#pragma unroll
        for (int n = 0; n < 5; ++n) acc[m][n] = zero16();
    if (r_begin < r_end) {
        const __bf16* Pw = P + 64u * mhalf;
        WgradStep w0, w1;
        wgrad_load<kMT>(w0, Pw, Q, r_begin, lane);
        for (uint32_t r = r_begin; r < r_end; r += 32u) {
            wgrad_load<kMT>(w1, Pw, Q, r + 16u, lane);
            wgrad_mfma<kMT>(w0, acc);
            wgrad_load<kMT>(w0, Pw, Q, r + 32u < r_end ? r + 32u : r, lane);
            wgrad_mfma<kMT>(w1, acc);
        }
    }
    // row parts in order: parts 1.. go through LDS to part 0's wavefront
    constexpr uint32_t kVals = kMT * 5u * 16u;
    if (rp > 0u) {
        float* f = fold + (size_t)((rp - 1u) * (kMT == 2 ? 2u : 1u) + mhalf) * kVals * 64u;
#pragma unroll
        for (int m = 0; m < kMT; ++m)
#pragma unroll
            for (int n = 0; n < 5; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    f[((m * 5 + n) * 16 + v) * 64 + lane] = acc[m][n][v];
    }
    __syncthreads();
    if (rp > 0u) return;
#pragma unroll
    for (uint32_t q = 0; q + 1u < kParts; ++q) {
        const float* f = fold + (size_t)(q * (kMT == 2 ? 2u : 1u) + mhalf) * kVals * 64u;
#pragma unroll
        for (int m = 0; m < kMT; ++m)
#pragma unroll
            for (int n = 0; n < 5; ++n)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[m][n][v] += f[((m * 5 + n) * 16 + v) * 64 + lane];
    }
#pragma unroll
    for (int m = 0; m < kMT; ++m)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t i = acc_row(v, h);
            const uint32_t row = kMT == 2 ? 64u * mhalf + 2u * i + m : i;
            if (kMT == 1 && row >= 3u) continue;
            float* o = part + (size_t)row * kSurRow;
            *reinterpret_cast<float4*>(o + 4u * col) =
                make_float4(acc[m][0][v], acc[m][1][v], acc[m][2][v], acc[m][3][v]);
            if (col < 16u) o[128u + col] = acc[m][4][v];
        }
}

__global__ __launch_bounds__(256) void k_sur_wgrad(SurGradRows g, const __bf16* __restrict__ S,
                                                   const __bf16* __restrict__ X,
                                                   const __bf16* __restrict__ Z, uint32_t R,
                                                   SurParts parts) {
    __shared__ float fold[2 * 160 * 64];
    const uint32_t slab = blockIdx.x;
    if (blockIdx.y == 0)
        wgrad_slab<2>(g.DZ, X, R, slab, parts.Wn1 + (size_t)slab * 128u * kSurRow, fold);
    else if (blockIdx.y == 1)
        wgrad_slab<2>(g.DM, S, R, slab, parts.W2 + (size_t)slab * 128u * kSurRow, fold);
    else
        wgrad_slab<1>(g.DOUT, Z, R, slab, parts.Wn2 + (size_t)slab * 3u * kSurRow, fold);
}

// ---------------------------------------------------------------------------
// edge pass (backward): d(W1|b1) = sum_i sum_j (dS_i * [u_ij > 0]) (e_ij | 1)^T.  The masked
// gradient is formed in the accumulator layout of the recomputed layer-1 product and fed
// back as an A operand (K = edges); the edge features reach the B operand through LDS.  One
// workgroup per batch chunk, 32 targets per wavefront.
//
// Bound by VALU issue and the latency of its LDS and MFMA chain (two wavefronts per SIMD).
//  - The layer-1 product is taken with negated weights, so u > 0 is the sign bit of the
//    result: per pair of values one byte permute (the two high halves), one packed 16-bit shift
//    (two masks) and one AND with the bf16 gradient pair, instead of two compares, two
//    selects and a conversion.
//  - The features are written to LDS as ten rows of 64 edges, in the order the B operand takes
//    them (the accumulator's row order), so an operand is one 16-byte read instead of eight
//    2-byte ones and their packing.
// The features and the layer-1 product are the forward pass's to the bit.  W(r) by clamped cubes
// (5 us of a call of 880 faster) now and then rounds to the next bf16 value, in the ReLU masks and
// in dW1; operands with the halves of K the same way round in both blocks (no time) give the sums
// that lie within a rounding of zero another sign, some of 2e9 a call: one such mask moved a
// small scene's gradient by 5e-6 of its norm.
// 1,024 chunks: 600 -> 241 us.
// ---------------------------------------------------------------------------
constexpr uint32_t kEdgeRow = 72;  // LDS row stride (bf16) of one feature over 64 edges

__global__ __launch_bounds__(64 * kEdgeWaves) __attribute__((amdgpu_waves_per_eu(2))) void
k_sur_edges_bwd(
    WalkBuffers wb, const uint32_t* __restrict__ batch, uint32_t nbatch,
    const float4* __restrict__ spm, const float4* __restrict__ svr,
    const uint32_t* __restrict__ skey, const uint32_t* __restrict__ cs, StepConsts c,
    const SceneGrid* __restrict__ scenes, const __bf16* __restrict__ pk, SurScales sc,
    const __bf16* __restrict__ DS, float* __restrict__ part) {
    __shared__ WalkLds lds_all[kEdgeWaves];
    __shared__ alignas(16) uint16_t le_all[kEdgeWaves][10 * kEdgeRow];
    const uint32_t half = uni(threadIdx.x >> 6);
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t col = lane & 31u, h = lane >> 5;
    WalkLds& L = lds_all[half];
    uint16_t* le = le_all[half];
    const uint32_t b = blockIdx.x;
    if (b >= nbatch) return;
    const uint32_t item = uni(batch[b]);
    const uint32_t clane = 32u * half + col;
    Chunk ch;
    uint32_t s;
    bool active;
    float4 pi;
    if (!load_chunk(item, wb.items, wb.desc, wb.nitems, skey, spm, c, scenes, clane, ch, s, active,
                    pi))
        return;
    const float4 vi = active ? svr[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    bf16x8 B[2][4];
    load_layer1(pk, lane, B[0]);
    load_layer1<true>(pk, lane, B[1]);
#pragma unroll
    for (int hb = 0; hb < 4; ++hb) {
        B[0][hb] = negated(B[0][hb]);
        B[1][hb] = negated(B[1][hb]);
    }
    // dS of this lane's hidden units for the 16 accumulator rows, as bf16 pairs (rows v, v + 1)
    uint32_t ds[4][8];
#pragma unroll
    for (int hb = 0; hb < 4; ++hb)
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const size_t row = 64u * (size_t)b + 32u * half;
            const __bf16* d = DS + 32u * hb + col;
            ds[hb][k] = bits16(d[(row + acc_row(2 * k, h)) * 128u]) |
                        bits16(d[(row + acc_row(2 * k + 1, h)) * 128u]) << 16;
        }
    // where this lane's edge goes in a feature row: operand (block, g), lane half, element
    const uint32_t epos =
        (lane & 32u) + (col & 16u) + ((col >> 2) & 1u) * 8u + ((col >> 3) & 1u) * 4u + (col & 3u);
    // this lane's feature row (columns from 10 on are garbage that is never stored)
    const __bf16* erow = reinterpret_cast<const __bf16*>(le) + min(col, 9u) * kEdgeRow + 8u * h;
    f32x16 accw[4];
#pragma unroll
    for (int hb = 0; hb < 4; ++hb) accw[hb] = zero16();
    walk_pairs<true>(item, ch, s, active, pi, clane, wb, spm, svr, cs, c, L, lane,
               [&](bool edge, float4 pj, float4 vj, float d2) {
                   uint32_t fe[4], ext;
                   edge_features<true>(edge, pi, vi, pj, vj, d2, sc, fe, ext);
                   // features 0..8 and 1 of this lane's edge
#pragma unroll
                   for (int k = 0; k < 4; ++k) {
                       le[2 * k * kEdgeRow + epos] = (uint16_t)fe[k];
                       le[(2 * k + 1) * kEdgeRow + epos] = (uint16_t)(fe[k] >> 16);
                   }
                   le[8 * kEdgeRow + epos] = (uint16_t)(ext >> 16);
                   le[9 * kEdgeRow + epos] = (uint16_t)ext;
                   wave_sync();
                   bf16x8 a[2];
                   layer1_a<true>(fe, ext, a[0], a[1]);
#pragma unroll
                   for (int blk = 0; blk < 2; ++blk) {
                       const bf16x8 e0 = load8(erow + 32 * blk);
                       const bf16x8 e1 = load8(erow + 32 * blk + 16);
#pragma unroll
                       for (int hb = 0; hb < 4; ++hb) {
                           // -u of 16 edges
                           const f32x16 d = mfma16(a[blk], B[blk][hb], zero16());
                           uint32_t g[8];
#pragma unroll
                           for (int k = 0; k < 8; ++k)
                               g[k] = ds[hb][k] & neg_masks(d[2 * k], d[2 * k + 1]);
                           accw[hb] = mfma16(
                               __builtin_bit_cast(bf16x8, make_uint4(g[0], g[1], g[2], g[3])), e0,
                               accw[hb]);
                           accw[hb] = mfma16(
                               __builtin_bit_cast(bf16x8, make_uint4(g[4], g[5], g[6], g[7])), e1,
                               accw[hb]);
                       }
                   }
                   wave_sync();
               });
    // the chunk's partial: half 0 plus half 1 (through LDS, the list is free)
    float* fold = reinterpret_cast<float*>(&lds_all[1]);  // [64 values][64 lanes]
    if (half == 1u) {
#pragma unroll
        for (int hb = 0; hb < 4; ++hb)
#pragma unroll
            for (int v = 0; v < 16; ++v) fold[(hb * 16 + v) * 64 + lane] = accw[hb][v];
    }
    __syncthreads();
    if (half == 1u || col >= 16u) return;
#pragma unroll
    for (int hb = 0; hb < 4; ++hb)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t m = 32u * hb + acc_row(v, h);
            part[((size_t)b * 128u + m) * 16u + col] =
                accw[hb][v] + fold[(hb * 16 + v) * 64 + lane];
        }
}

// ---------------------------------------------------------------------------
// small element-wise kernels
// ---------------------------------------------------------------------------
// Gradient of every parameter from the partials of all four products, one launch: a workgroup
// sums 16 columns of one partial row, 16 threads per column, each a sixteenth of the slabs in
// order, then folds the sixteen in order.  Scaled by 1 / (3 rows), rows counted in the loss
// partials (0 when no row has a slot).  Bound by the read of the partials: a chain of 8 slabs
// (weights) or 64 (edges) per thread instead of one thread per parameter over all of them:
// 1,024 chunks, four reductions 532 -> 13 us.
struct SurReduceTask {
    const float* part;
    uint32_t slabs, rows, ld;  // partials [slabs][rows][ld]
    uint32_t ncols;            // columns of the weight; column ncols is the bias
    uint32_t dst, bias_dst;
    uint32_t first;            // first workgroup of the task
};
struct SurReduceTasks {
    SurReduceTask t[4];
};

__global__ __launch_bounds__(256) void k_sur_reduce(SurReduceTasks tasks,
                                                    const float* __restrict__ loss_part,
                                                    uint32_t nparts, float* __restrict__ grad) {
    __shared__ float sums[16][17];
    __shared__ uint32_t lrows[4];
    int ti = 0;
    while (ti < 3 && blockIdx.x >= tasks.t[ti + 1].first) ++ti;
    const SurReduceTask& t = tasks.t[ti];
    const uint32_t cblocks = (t.ncols + 16u) / 16u;  // of ncols + 1 columns
    const uint32_t wg = blockIdx.x - t.first;
    const uint32_t m = wg / cblocks, n = (wg % cblocks) * 16u + (threadIdx.x & 15u);
    const uint32_t grp = threadIdx.x >> 4;
    const uint32_t per = (t.slabs + 15u) / 16u;
    const uint32_t sl0 = min(grp * per, t.slabs), sl1 = min(sl0 + per, t.slabs);
    const float* p = t.part + (size_t)m * t.ld + n;  // ld is a multiple of 16
    const size_t stride = (size_t)t.rows * t.ld;
    float sum = 0.0f;
#pragma unroll 8
    for (uint32_t sl = sl0; sl < sl1; ++sl) sum += p[sl * stride];
    sums[grp][threadIdx.x & 15u] = sum;
    uint32_t cnt = 0;
    for (uint32_t b = threadIdx.x; b < nparts; b += 256u) cnt += (uint32_t)loss_part[2u * b + 1u];
    for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off);
    if ((threadIdx.x & 63u) == 0u) lrows[threadIdx.x >> 6] = cnt;
    __syncthreads();
    if (grp != 0u || n > t.ncols) return;
    const uint32_t rows = (lrows[0] + lrows[1]) + (lrows[2] + lrows[3]);
    const float scale = rows ? (float)(1.0 / (3.0 * (double)rows)) : 0.0f;
    float tot = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) tot += sums[k][threadIdx.x];
    if (n < t.ncols) grad[t.dst + m * t.ncols + n] = scale * tot;
    else grad[t.bias_dst + m] = scale * tot;
}

__device__ __forceinline__ float block_sum_256(float x, float* red) {
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(256) void k_sur_targets(const float4* __restrict__ v0,
                                                     const float4* __restrict__ v4, uint32_t n,
                                                     float dk, float inv_Tas,
                                                     float4* __restrict__ target) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const float4 a = v0[i], b = v4[i];
    target[i] = make_float4((b.x - dk * a.x) * inv_Tas, (b.y - dk * a.y) * inv_Tas,
                            (b.z - dk * a.z) * inv_Tas, 0.0f);
}

__global__ __launch_bounds__(256) void k_sur_scale_rows(const float* __restrict__ rows,
                                                        uint32_t n, float scale,
                                                        float4* __restrict__ dst) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    const float* r = rows + 3 * (size_t)i;
    dst[i] = make_float4(r[0] * scale, r[1] * scale, r[2] * scale, 0.0f);
}

__global__ __launch_bounds__(256) void k_sur_mask(const uint32_t* __restrict__ rowslot,
                                                  uint32_t R, const uint32_t* __restrict__ sid,
                                                  uint8_t* __restrict__ mask) {
    const uint32_t r = blockIdx.x * 256u + threadIdx.x;
    if (r >= R) return;
    const uint32_t slot = rowslot[r];
    if (slot != kSurNoSlot) mask[sid[slot]] = 1;
}

// Particles with a non-finite coordinate (dense index G) have no neighbours: free fall over
// the macro-step, as in the plain step.
__global__ __launch_bounds__(256) void k_sur_nonfinite(const float4* __restrict__ spm,
                                                       const float4* __restrict__ svr,
                                                       const uint32_t* __restrict__ sid,
                                                       const uint32_t* __restrict__ cs,
                                                       uint32_t n, StepConsts c,
                                                       const SceneGrid* __restrict__ scenes,
                                                       SurStep step) {
    const uint32_t s = cs[c.G] + blockIdx.x * 256u + threadIdx.x;
    if (s >= n) return;
    const float4 vr = svr[s];
    const uint32_t id = sid[s];
    float4 p = spm[s];
    const float3 a = make_float3(0.0f, c.grav, 0.0f);
    float3 v1;
    macro_integrate(p, v1, make_float3(vr.x, vr.y, vr.z), a, step.T, step.dk,
                    scenes[scene_of_particle(scenes, c.nscenes, id)]);
    const float rho_i = p.w * c.w0;
    step.pm[id] = p;
    step.vel[id] = make_float4(v1.x, v1.y, v1.z, 0.0f);
    step.acc[id] = make_float4(a.x, a.y, a.z, 0.0f);
    step.rho[id] = rho_i;
    step.prs[id] = c.k_gas * (rho_i - c.rho0);
}

__global__ __launch_bounds__(256) void k_sur_adam(float* __restrict__ w, float* __restrict__ m,
                                                  float* __restrict__ v,
                                                  const float* __restrict__ g, uint32_t np,
                                                  float lr, float beta1, float beta2, float eps,
                                                  float bc1, float bc2) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= np) return;
    const float gi = g[i];
    const float mi = beta1 * m[i] + (1.0f - beta1) * gi;
    const float vi = beta2 * v[i] + (1.0f - beta2) * (gi * gi);
    m[i] = mi;
    v[i] = vi;
    const float mh = __fdiv_rn(mi, bc1), vh = __fdiv_rn(vi, bc2);
    w[i] = w[i] - __fdiv_rn(lr * mh, __fsqrt_rn(vh) + eps);
}

__global__ __launch_bounds__(256) void k_sur_rho_diff(const float* __restrict__ a,
                                                      const float* __restrict__ b, uint32_t n,
                                                      float* __restrict__ part) {
    __shared__ float red[4];
    __shared__ float redm[4];
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const float d = i < n ? fabsf(a[i] - b[i]) : 0.0f;
    float mx = d;
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    if ((threadIdx.x & 63u) == 0) redm[threadIdx.x >> 6] = mx;
    const float tot = block_sum_256(d, red);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = tot;
        part[2 * blockIdx.x + 1] = fmaxf(fmaxf(redm[0], redm[1]), fmaxf(redm[2], redm[3]));
    }
}

// Densities of the sorted state in caller order (non-finite particles: m W(0)).
__global__ __launch_bounds__(256) void k_sur_rho_home(const float4* __restrict__ spm,
                                                      const float4* __restrict__ svr,
                                                      const uint32_t* __restrict__ sid,
                                                      const uint32_t* __restrict__ cs,
                                                      uint32_t n, StepConsts c,
                                                      float* __restrict__ out) {
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= n) return;
    out[sid[s]] = s < cs[c.G] ? svr[s].w : spm[s].w * c.w0;
}

// Network accelerations a = a_s out in caller order (non-finite particles: (0, g, 0)).
__global__ __launch_bounds__(256) void k_sur_scatter_out(const float* __restrict__ out,
                                                         const uint32_t* __restrict__ sid,
                                                         const uint32_t* __restrict__ cs,
                                                         uint32_t n, StepConsts c,
                                                         float acc_scale,
                                                         float4* __restrict__ dst) {
    const uint32_t s = blockIdx.x * 256u + threadIdx.x;
    if (s >= n) return;
    float4 a = make_float4(0.0f, c.grav, 0.0f, 0.0f);
    if (s < cs[c.G])
        a = make_float4(acc_scale * out[4 * (size_t)s], acc_scale * out[4 * (size_t)s + 1],
                        acc_scale * out[4 * (size_t)s + 2], 0.0f);
    dst[sid[s]] = a;
}

// ---------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------
hipError_t launch_sur_rho_home(const float4* spm, const float4* svr, const uint32_t* sid,
                               const uint32_t* cs, uint32_t n, const StepConsts& c, float* out,
                               hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sur_rho_home, dim3((n + 255) / 256), dim3(256), 0, st, spm, svr, sid, cs,
                       n, c, out);
    return hipGetLastError();
}

hipError_t launch_sur_scatter_out(const float* out, const uint32_t* sid, const uint32_t* cs,
                                  uint32_t n, const StepConsts& c, float acc_scale, float4* dst,
                                  hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sur_scatter_out, dim3((n + 255) / 256), dim3(256), 0, st, out, sid, cs,
                       n, c, acc_scale, dst);
    return hipGetLastError();
}

hipError_t launch_sur_pack(const float* params, __bf16* pk, float* pf, hipStream_t st) {
    hipLaunchKernelGGL(k_sur_pack, dim3((kPkTotal + 255) / 256), dim3(256), 0, st, params, pk, pf);
    return hipGetLastError();
}

hipError_t launch_sur_forward(bool integrate, const WalkBuffers& wb, const uint32_t* batch,
                              uint32_t nbatch, uint32_t max_items, const float4* spm,
                              const float4* svr, const uint32_t* skey, const uint32_t* sid,
                              const uint32_t* cs, uint32_t n, const StepConsts& c,
                              const SceneGrid* scenes, const __bf16* pk, const float* pf,
                              const SurScales& sc, const SurRows& rows, const SurStep& step,
                              hipStream_t st) {
    const uint32_t chunks = batch ? nbatch : max_items;
    if (chunks == 0) return hipSuccess;
    const uint32_t blocks = (chunks + kXcds - 1) / kXcds * kXcds;  // xcd_unit() needs it
    if (integrate) {
        hipLaunchKernelGGL(k_sur_forward<true>, dim3(blocks), dim3(64 * kEdgeWaves), 0, st, wb,
                           batch, nbatch, spm, svr, skey, sid, cs, c, scenes, pk, pf, sc, rows,
                           step);
        // the non-finite bin holds at most n particles; the kernel reads its start on the device
        hipLaunchKernelGGL(k_sur_nonfinite, dim3((n + 255) / 256), dim3(256), 0, st, spm, svr,
                           sid, cs, n, c, scenes, step);
    } else {
        hipLaunchKernelGGL(k_sur_forward<false>, dim3(blocks), dim3(64 * kEdgeWaves), 0, st, wb,
                           batch, nbatch, spm, svr, skey, sid, cs, c, scenes, pk, pf, sc, rows,
                           step);
    }
    return hipGetLastError();
}

hipError_t launch_sur_node_bwd(const float4* out, const uint32_t* rowslot, const uint32_t* sid,
                               const float4* target, uint32_t R, const __bf16* Z,
                               const __bf16* pk, float msg_scale, const SurGradRows& g,
                               float* loss_part, hipStream_t st) {
    hipLaunchKernelGGL(k_sur_node_bwd, dim3(sur_loss_parts(R)), dim3(64 * kNodeWaves), 0, st, out,
                       rowslot, sid, target, R, Z, pk, msg_scale, g, loss_part);
    return hipGetLastError();
}

hipError_t launch_sur_wgrad(const SurGradRows& g, const __bf16* S, const __bf16* X,
                            const __bf16* Z, uint32_t R, const SurParts& parts, hipStream_t st) {
    hipLaunchKernelGGL(k_sur_wgrad, dim3(sur_slabs(R), 3), dim3(256), 0, st, g, S, X, Z, R, parts);
    return hipGetLastError();
}

hipError_t launch_sur_edges_bwd(const WalkBuffers& wb, const uint32_t* batch, uint32_t nbatch,
                                const float4* spm, const float4* svr, const uint32_t* skey,
                                const uint32_t* cs, const StepConsts& c,
                                const SceneGrid* scenes, const __bf16* pk, const SurScales& sc,
                                const __bf16* DS, float* part, hipStream_t st) {
    if (nbatch == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sur_edges_bwd, dim3(nbatch), dim3(64 * kEdgeWaves), 0, st, wb, batch,
                       nbatch, spm, svr, skey, cs, c, scenes, pk, sc, DS, part);
    return hipGetLastError();
}

hipError_t launch_sur_reduce(const SurParts& parts, uint32_t R, uint32_t nbatch,
                             const float* loss_part, float* grad, hipStream_t st) {
    const uint32_t slabs = sur_slabs(R);
    SurReduceTasks k;
    k.t[0] = {parts.Wn1, slabs, 128, kSurRow, kSurNodeIn, kOffWn1, kOffBn1, 0};
    k.t[1] = {parts.W2, slabs, 128, kSurRow, 128, kOffW2, kOffB2, 0};
    k.t[2] = {parts.Wn2, slabs, 3, kSurRow, 128, kOffWn2, kOffBn2, 0};
    k.t[3] = {parts.W1, nbatch, 128, 16, kSurNF, kOffW1, kOffB1, 0};
    uint32_t wgs = 0;
    for (auto& t : k.t) {
        t.first = wgs;
        wgs += t.rows * ((t.ncols + 16u) / 16u);
    }
    hipLaunchKernelGGL(k_sur_reduce, dim3(wgs), dim3(256), 0, st, k, loss_part, sur_loss_parts(R),
                       grad);
    return hipGetLastError();
}

hipError_t launch_sur_scale_rows(const float* rows, uint32_t n, float scale, float4* dst,
                                 hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sur_scale_rows, dim3((n + 255) / 256), dim3(256), 0, st, rows, n, scale,
                       dst);
    return hipGetLastError();
}

hipError_t launch_sur_mask(const uint32_t* rowslot, uint32_t R, const uint32_t* sid, uint32_t n,
                           uint8_t* mask, hipStream_t st) {
    hipError_t e = launch_fill_u32(reinterpret_cast<uint32_t*>(mask), 0u, (n + 3u) / 4u, st);
    if (e != hipSuccess || R == 0) return e;
    hipLaunchKernelGGL(k_sur_mask, dim3((R + 255) / 256), dim3(256), 0, st, rowslot, R, sid, mask);
    return hipGetLastError();
}

hipError_t launch_sur_targets(const float4* v0, const float4* v4, uint32_t n, float dk,
                              float inv_Tas, float4* target, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sur_targets, dim3((n + 255) / 256), dim3(256), 0, st, v0, v4, n, dk,
                       inv_Tas, target);
    return hipGetLastError();
}

hipError_t launch_sur_adam(float* w, float* m, float* v, const float* g, uint32_t np, float lr,
                           float beta1, float beta2, float eps, float bc1, float bc2,
                           hipStream_t st) {
    hipLaunchKernelGGL(k_sur_adam, dim3((np + 255) / 256), dim3(256), 0, st, w, m, v, g, np, lr,
                       beta1, beta2, eps, bc1, bc2);
    return hipGetLastError();
}

hipError_t launch_sur_rho_diff(const float* a, const float* b, uint32_t n, float* part,
                               uint32_t* nparts, hipStream_t st) {
    const uint32_t blocks = (n + 255u) / 256u;
    *nparts = blocks;
    if (blocks == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sur_rho_diff, dim3(blocks), dim3(256), 0, st, a, b, n, part);
    return hipGetLastError();
}

}  // namespace sphk
