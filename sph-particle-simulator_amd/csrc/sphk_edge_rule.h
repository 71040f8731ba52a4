// sphk_edge_rule.h -- which particles may have a neighbour two cells away along an axis: the exact
// rule and the quick test that spares most particles it.  Plain C++ besides the function
// attributes, so that a host program can run the same lines.
#pragma once

#include <cstring>

#ifdef __HIP__
#define SPHK_EDGE_RULE __host__ __device__ __forceinline__
#else
#define SPHK_EDGE_RULE inline
#endif

namespace sphk {

namespace {

SPHK_EDGE_RULE int float_bits(float x) {
    int i;
    memcpy(&i, &x, sizeof i);
    return i;
}

SPHK_EDGE_RULE float bits_float(int i) {
    float x;
    memcpy(&x, &i, sizeof x);
    return x;
}

SPHK_EDGE_RULE float next_up(float x) {
    if (x == 0.0f) return bits_float(1);
    const int i = float_bits(x);
    return bits_float(x > 0.0f ? i + 1 : i - 1);
}

SPHK_EDGE_RULE float next_down(float x) {
    if (x == 0.0f) return -bits_float(1);
    const int i = float_bits(x);
    return bits_float(x > 0.0f ? i - 1 : i + 1);
}

// Can a particle at coordinate x (cell c = floor(fl(x*inv))) have a neighbour in cell c+2
// (bit 1) or c-2 (bit 0)?  A neighbour needs fl(fl(b-x)^2) <= r2 on this axis alone, and
// fl(b-x) grows with b, so it suffices to test the float b nearest to x that lands in cell
// c+2 (resp. c-2).  Exact; conservative (flag set) if the bracket search does not settle.
SPHK_EDGE_RULE int axis_edge_flags(float x, float inv, float r2) {
#pragma clang fp contract(off)
    float c = __builtin_floorf(x * inv);
    int flags = 0;
    {
        float t = c + 2.0f;
        float b = t / inv;
        int ok = 0;
        for (int k = 0; k < 6; ++k) {
            if (b * inv >= t) {
                ok = 1;
                break;
            }
            b = next_up(b);
        }
        if (ok) {
            for (int k = 0; k < 6; ++k) {
                float bd = next_down(b);
                if (bd * inv >= t) {
                    b = bd;
                } else {
                    ok = 2;
                    break;
                }
            }
        }
        float d = b - x;
        if (ok != 2 || d * d <= r2) flags |= 2;
    }
    {
        float t = c - 1.0f;
        float b = t / inv;
        int ok = 0;
        for (int k = 0; k < 6; ++k) {
            if (b * inv < t) {
                ok = 1;
                break;
            }
            b = next_down(b);
        }
        if (ok) {
            for (int k = 0; k < 6; ++k) {
                float bu = next_up(b);
                if (bu * inv < t) {
                    b = bu;
                } else {
                    ok = 2;
                    break;
                }
            }
        }
        float d = x - b;
        if (ok != 2 || d * d <= r2) flags |= 1;
    }
    return flags;
}

// Whether axis_edge_flags(x, inv, r2) can set a flag at all (r2 = fl(R^2), inv = fl(1 / R)).
// With u = 2^-24 and t = fl(x inv), c = floor(t): a neighbour b in cell c + 2 has
// b / R >= c + 2 - 2.1 u |c + 2| and b - x <= R (1 + 3 u), so t >= c + 1 - 5 u (|c| + 3); in
// cell c - 2, by the same bounds, t <= c + 5 u (|c| + 3).  Tested with 32 u for 5 u.  The
// bracket searches of the exact flags (six divisions a lane) are then skipped by every chunk
// without such a lane: 1M step 1.086 -> 1.081 ms, 9.6M 0.8 % faster, and every wavefront of a
// walk pays them.
SPHK_EDGE_RULE bool axis_edge_near(float x, float inv) {
#pragma clang fp contract(off)
    const float t = x * inv;
    const float c = __builtin_floorf(t);
    const float margin = (__builtin_fabsf(c) + 3.0f) * 0x1p-19f;
    const float f = t - c;
    // (written so that a NaN counts as near)
    return !(f > margin && f < 1.0f - margin);
}

}  // namespace

}  // namespace sphk

#undef SPHK_EDGE_RULE
