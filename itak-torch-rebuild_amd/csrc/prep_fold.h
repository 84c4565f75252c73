// Norm and rotation of Q and of new K rows inside the kernels that read them (one-row steps and
// speculative blocks at head_dim 128).
#pragma once

#include "internal.h"
#include "mfma_common.h"

#include <math.h>

namespace itak {

namespace {

// ---- preparation folded into the step (PREP instantiations) -----------------------------
// The reference's model norms and rotates Q and K between their projections and attention
// (per-head RMSNorm, crates/torch-math/src/norm.rs:40-51; RoPE, rope_interleaved.rs:103-114 /
// rope.rs:99-114; order of calls crates/muse-glimmer/src/model.rs:445-451). A decode step is a
// few thousand elements, so as a launch of its own that work costs a launch; here every
// workgroup prepares the 16 query vectors it stages anyway, and the workgroup that appends
// the new K rows prepares those. A 128-channel head row lies across 32 consecutive lanes, four
// channels each (c4 = 4 * (lane % 32)), which is how Q and the new rows are loaded.
//
// Arithmetic: the angle position * base^(-2i/rot) is formed and reduced to [-pi, pi] in f64
// (an f32 angle is off by 8e-3 rad at position 100,000); norm, sine, cosine and rotation are
// f32. The results feed f16 storage and f16 MFMA operands, so they differ from the
// reference's f64 chain by parts in 1e7 before that rounding: at most one f16 step after it.
struct PrepTrig {
    float c[4], s[4];  // per pair held by this lane: 2 (interleaved) or 4 (half split)
};

__device__ __forceinline__ void prep_trig(PrepTrig &t, double position, const double (&freq)[4],
                                          int pairs) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (i >= pairs) break;
        // The angle in turns, reduced to [-1/2, 1/2] exactly in f64; the sine and cosine
        // instructions take turns. Their error (about 1e-6 absolute) is a five-hundredth of
        // the f16 step the results are rounded to.
        const double turns = position * freq[i] * 0.15915494309189535;
        const float frac = float(turns - rint(turns));
        t.s[i] = __builtin_amdgcn_sinf(frac);
        t.c[i] = __builtin_amdgcn_cosf(frac);
    }
}

// Sum over the 32 lanes that share a head row: four DPP steps inside each row of 16 lanes
// (neighbour, other pair, mirrored half, mirrored row), then the row 16 lanes away.
__device__ __forceinline__ float row_sum32(float v) {
    v += dpp_lane<0xB1>(v);   // quad_perm [1,0,3,2]
    v += dpp_lane<0x4E>(v);   // quad_perm [2,3,0,1]
    v += dpp_lane<0x141>(v);  // row_half_mirror
    v += dpp_lane<0x140>(v);  // row_mirror
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// x = channels c4 .. c4+3 of a head row, w = the norm weight's same channels.
__device__ __forceinline__ float4 prep_chunk(float4 x, bool norm, float4 w, float eps, uint32_t c4,
                                             uint32_t lane, uint32_t rot, bool interleaved,
                                             const PrepTrig &t) {
    if (norm) {
        const float ss = row_sum32(x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w);
        const float inv = __builtin_amdgcn_rsqf(ss * (1.0f / kD) + eps);
        x = make_float4(x.x * inv * w.x, x.y * inv * w.y, x.z * inv * w.z, x.w * inv * w.w);
    }
    if (rot == 0) return x;
    if (interleaved) {  // pairs (c4, c4+1) and (c4+2, c4+3)
        float4 y = x;
        if (c4 < rot) {
            y.x = x.x * t.c[0] - x.y * t.s[0];
            y.y = x.x * t.s[0] + x.y * t.c[0];
        }
        if (c4 + 2 < rot) {
            y.z = x.z * t.c[1] - x.w * t.s[1];
            y.w = x.z * t.s[1] + x.w * t.c[1];
        }
        return y;
    }
    // Half split: channel c < rot/2 turns with channel c + rot/2, four lanes-of-four apart.
    const uint32_t half = rot >> 1;
    const bool low = c4 < half, turn = c4 < rot;
    const uint32_t partner = (lane & 32u) | (((lane & 31u) + (low ? half / 4 : 32u - half / 4)) & 31u);
    const float4 o = make_float4(__shfl(x.x, partner), __shfl(x.y, partner), __shfl(x.z, partner),
                                 __shfl(x.w, partner));
    if (!turn) return x;
    if (low)
        return make_float4(x.x * t.c[0] - o.x * t.s[0], x.y * t.c[1] - o.y * t.s[1],
                           x.z * t.c[2] - o.z * t.s[2], x.w * t.c[3] - o.w * t.s[3]);
    return make_float4(o.x * t.s[0] + x.x * t.c[0], o.y * t.s[1] + x.y * t.c[1],
                       o.z * t.s[2] + x.z * t.c[2], o.w * t.s[3] + x.w * t.c[3]);
}

}  // namespace

}  // namespace itak
