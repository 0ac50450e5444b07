// valu_metrics.h -- the element steps of the metrics that run on the vector ALUs (knn_valu.hip,
// knn_rows.hip), in the direct form of the reference CPU engine (scalar.rs:81-263).
#pragma once

#include "vh_common.h"

namespace vh {

// k-means Hellinger: centroids are means of the raw data, so sqrt(|x|) of the centroid
// side is taken in the loop (the point side holds sqrt(|p|)).
constexpr int HELL_RAW = 11;

template <int M>
__device__ __forceinline__ void accum(float &a, float &b, float q, float x) {
    if constexpr (M == HELL_RAW) {
        const float d = q - sqrtf(fabsf(x));
        a = fmaf(d, d, a);
    } else if constexpr (M == L1) {
        a += fabsf(q - x);
    } else if constexpr (M == L2 || M == MAHA || M == HELL) {
        const float d = q - x;
        a = fmaf(d, d, a);
    } else if constexpr (M == LINF) {
        a = fmaxf(a, fabsf(q - x));
    } else if constexpr (M == MINK) {
        const float d = fabsf(q - x);
        a = fmaf(d * d, d, a);
    } else if constexpr (M == HAMF) {
        a += fabsf(q - x) > 1e-6f ? 1.0f : 0.0f;
    } else if constexpr (M == DOT) {
        a = fmaf(q, x, a);
    } else if constexpr (M == COS) {  // dot product and the row's squared norm
        a = fmaf(q, x, a);
        b = fmaf(x, x, b);
    } else {  // JACC: q holds |q|
        const float ax = fabsf(x);
        a += fminf(q, ax);
        b += fmaxf(q, ax);
    }
}

// Two consecutive elements; L-inf takes both in one max of three (|.| source modifiers).
template <int M>
__device__ __forceinline__ void accum2(float &a, float &b, float q0, float q1, float x0, float x1) {
    if constexpr (M == LINF) {
        a = fmaxf(a, fmaxf(fabsf(q0 - x0), fabsf(q1 - x1)));
    } else {
        accum<M>(a, b, q0, x0);
        accum<M>(a, b, q1, x1);
    }
}

template <int M>
__device__ __forceinline__ float finish(float a, float b) {
    if constexpr (M == MINK) return cbrtf(a);
    else if constexpr (M == MAHA) return sqrtf(a);
    else if constexpr (M == HELL || M == HELL_RAW) return sqrtf(0.5f * a);
    else if constexpr (M == JACC) return b <= 1e-9f ? 0.0f : 1.0f - a / b;
    else return a;
}

}  // namespace vh
