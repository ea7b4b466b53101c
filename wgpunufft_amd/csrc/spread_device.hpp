// Device helpers shared by the spreaders: the exponential-of-semicircle
// weight and the bin intervals that reach a block of cells.
#pragma once

#include <hip/hip_runtime.h>

#include "nufft_internal.hpp"
#include "tile_index.hpp"

namespace mnufft {
namespace {

template <typename T>
__device__ inline T es_weight(T d, int w, T beta)
{
    T s = (T)2 * d / (T)w;
    T q = (T)1 - s * s;
    if (!(q > (T)0)) return (T)0;
    if constexpr (sizeof(T) == 4)
        return expf(beta * (sqrtf(q) - 1.0f));
    else
        return exp(beta * (sqrt(q) - 1.0));
}

// Coefficients read by scalar loads: the same address for every lane.
template <typename T>
using UniformPtr = const __attribute__((address_space(4))) T *;

template <typename T>
__device__ inline UniformPtr<T> panel_coefficients(const GridParams &g)
{
    return (UniformPtr<T>)(uintptr_t)g.panels;
}

// The weight of a support's first or last cell, at distance d: directly, for
// W known (no division).  FP32 takes the hardware square root and base-2
// exponential, up to width 4 of -beta s^2 / (1 + sqrt q), which does not
// cancel near the centre; wider kernels weigh these cells so little that the
// cancellation in sqrt(q) - 1 stays below the rounding of the other cells.
// Largest errors at upsampling factor 2, es_weight / sqrt(q) - 1 on the
// hardware units / this: width 2 18e-8 / 18e-8 / 8e-8, 3 24e-8 / 28e-8 /
// 10e-8, 4 14e-8 / 17e-8 / 6e-8, 5 7e-8 / 7e-8, 6 2e-8 / 4e-8, 7 1e-8 / 1e-8.
// SPLIT: weights that become FP16 or BF16 operands, rounded to 2^-21 at best,
// take the shorter form at every width (width 4, 9.3e6 points: an execute 873
// us, 884 with the other).
template <typename T, int W, bool SPLIT>
__device__ inline T es_edge_weight(T d, T beta)
{
    const T s = d * (T)(2.0 / W);
    const T q = (T)1 - s * s;
    if constexpr (sizeof(T) == 4) {
        const float bl = 1.44269504f * beta;
        float e;
        if constexpr (W <= 4 && !SPLIT)
            e = -bl * (s * s) *
                __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_sqrtf(fmaxf(q, 0.0f)));
        else
            e = __builtin_fmaf(__builtin_amdgcn_sqrtf(q), bl, -bl);
        return q > 0.0f ? __builtin_amdgcn_exp2f(e) : 0.0f;
    } else {
        return q > 0.0 ? exp(beta * (sqrt(q) - 1.0)) : 0.0;
    }
}

// Whether an offset is that of a point's support (at most 1 - w/2, which is
// at most zero) and not of one out of the fold's reach (kOutsideOffset, the
// same on every axis), which weighs zero.
template <typename T>
__device__ inline bool on_support(T off)
{
    return off < (T)1;
}

// The W weights of one axis of a point, put(t, weight) for cell t of its
// support, from its offset (start - position, in [-W/2, 1 - W/2)).  Inner
// cells come in pairs from the panel polynomials (about 5 FMAs a weight in
// FP32 and 8 in FP64, where sqrt and exp take 30 and 60 instructions),
// accurate to the type's rounding; the end cells directly.  The polynomials
// hold on the support alone: an offset that is not on_support is the caller's
// to leave out (a tile takes no such record, the interpolations write zero:
// one test a point, where zero weights cost the FP64 tiles 4%).
template <typename T, int W, bool SPLIT = false, typename Put>
__device__ __forceinline__ void es_axis_weights(T off, T beta, UniformPtr<T> c, Put put)
{
    constexpr int NE = panel_even(sizeof(T) == 8, W), NO = panel_odd(sizeof(T) == 8, W);
    const T x = off + (T)(0.5 * (W - 1));
    const T x2 = x * x;
    put(0, es_edge_weight<T, W, SPLIT>(off, beta));
    put(W - 1, es_edge_weight<T, W, SPLIT>(off + (T)(W - 1), beta));
#pragma unroll
    for (int t = 1; t <= (W - 1) / 2; ++t) {
        UniformPtr<T> e = c + (t - 1) * (NE + NO), o = e + NE;
        T even = e[NE - 1];
#pragma unroll
        for (int i = NE - 2; i >= 0; --i) even = __builtin_elementwise_fma(even, x2, e[i]);
        if (2 * t == W - 1) {
            put(t, even);
        } else {
            T odd = o[NO - 1];
#pragma unroll
            for (int i = NO - 2; i >= 0; --i) odd = __builtin_elementwise_fma(odd, x2, o[i]);
            put(t, __builtin_elementwise_fma(x, odd, even));
            put(W - 1 - t, __builtin_elementwise_fma(-x, odd, even));
        }
    }
}

// The FP32 weight from the hardware square root and base-2 exponential
// (v_sqrt_f32, v_exp_f32): a few ulp where the weight is near one and an
// absolute error below 1e-12 at the support edges (weight about e^-beta),
// against the correctly rounded sqrtf/expf sequence above.  Used where the
// weights feed FP32 sums of many terms (interpolation) or operands rounded
// to FP16 (matrix-core spread).
__device__ inline float es_weight_fast(float d, float two_over_w, float beta_log2e)
{
    const float s = d * two_over_w;
    const float q = 1.0f - s * s;
    if (!(q > 0.0f)) return 0.0f;
    return __builtin_amdgcn_exp2f(beta_log2e * (__builtin_amdgcn_sqrtf(q) - 1.0f));
}

}  // namespace
}  // namespace mnufft
