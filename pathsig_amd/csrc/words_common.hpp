// Device helpers shared by the per-word signature kernels (lanes on words, and lanes on paths).
#pragma once

#include "common.hpp"

namespace psig {
namespace {

template <typename T>
__device__ __forceinline__ T fma_t(T a, T b, T c);
template <>
__device__ __forceinline__ float fma_t<float>(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
template <>
__device__ __forceinline__ double fma_t<double>(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

__device__ __forceinline__ int find_level(const LevelPlan &plan, int64_t blk) {
    int deg = 1;
    while (deg < plan.depth && blk >= plan.block_begin[deg + 1]) ++deg;
    return deg;
}

struct WindowSpan {
    int64_t start, steps;
};

__device__ __forceinline__ WindowSpan window_span(const SigShape &shape, int64_t w) {
    int64_t start = 0, end = shape.L;
    if (shape.windows) {
        start = shape.windows[2 * w];
        end = shape.windows[2 * w + 1];
        start = start < 0 ? 0 : (start > shape.L ? shape.L : start);
        end = end < 0 ? 0 : (end > shape.L ? shape.L : end);
    }
    int64_t steps = end - start - 1;
    return {start, steps < 0 ? 0 : steps};
}

template <int DEG>
__device__ __forceinline__ void decode_letters(uint64_t code, uint64_t d, int (&l)[DEG]) {
#pragma unroll
    for (int pos = DEG - 1; pos >= 0; --pos) {
        const uint64_t q = code / d;
        l[pos] = (int)(code - q * d);
        code = q;
    }
}

// Horner values of target level M over what their next product asks for: with r_0 = 1/M and T_J = S(w_1..w_J) + r_(J-1) dl_J,
// r_J = T_J / (M - J) for J < M; S_new(w_1..w_M) = S(w_1..w_M) + r_(M-1) dl_M.  Two instructions for M - J > 1 and one for M - J = 1,
// as many as letters at the M scales that a word asks for would take, and constants in place of those.  (1/(M - J)! in place of
// 1/(M - J), with r_0 = 1/M!, takes as many: the first of them are 5040 times smaller at depth 8, and a word that begins with
// an increment below 5e-34 then lost digits to the smallest floats.)
template <typename T, int M, int DEG, int J = 1>
__device__ __forceinline__ void horner_values(const T (&p)[DEG + 1], const T (&dl)[DEG], T (&r)[DEG + 1]) {
    if constexpr (J == 1) r[0] = Recip<T>::of(M);
    if constexpr (J < M) {
        r[J] = fma_t<T>(r[J - 1], dl[J - 1], p[J]);
        if constexpr (M - J > 1) r[J] *= Recip<T>::of(M - J);
        horner_values<T, M, DEG, J + 1>(p, dl, r);
    }
}

// one forward Horner/Chen step on the chain p[0..TOP]
template <typename T, int DEG, int TOP>
__device__ __forceinline__ void chain_step(T (&p)[DEG + 1], const T (&dl)[DEG]) {
    if constexpr (TOP >= 1) {
        T r[DEG + 1];
        horner_values<T, TOP, DEG>(p, dl, r);
        p[TOP] = TOP == 1 ? p[1] + dl[0] : fma_t<T>(r[TOP - 1], dl[TOP - 1], p[TOP]);
        chain_step<T, DEG, TOP - 1>(p, dl);
    }
}

// One Chen step on the chain back, and its adjoint.  p is the chain after the step (levels < DEG) and becomes the one
// before it; h, the adjoint of the chain after the step, becomes the one before it, and gl[k] holds the step's
// dL/d(dl[k]).  Targets ascend: h[M] is still the adjoint after the step when target M reads it, and the levels below
// M have been taken back, so the Horner values of target M are those of the forward step: they serve the adjoint and
// take level M back, S(w_1..w_M) -= r_(M-1) dl_M.  The adjoint of T_J is v_J = v_(J+1) dl_(J+1) / (M - J): the chain gets
// v_J of it and letter J v_J r_(J-1).  v and r are divided at every node, so that both stay within what ends up in a
// result: with products of letters in place of v, divided once at the end, a word of eight letters overflowed 5040 times
// earlier than its gradient.  The divisions take 10 of 91 vector instructions of a word of six letters (101 with the letters
// at every scale in their place) and 15 of 781 us a step, 256 paths of 512 points, 16 letters, 2320 words up to length 6, fp32.
template <typename T, int DEG, int M = 1>
__device__ __forceinline__ void chain_step_adjoint(T (&p)[DEG + 1], T (&h)[DEG + 1], const T (&dl)[DEG], T (&gl)[DEG]) {
    if constexpr (M <= DEG) {
        T r[DEG + 1];
        horner_values<T, M, DEG>(p, dl, r);
        if (M < DEG) p[M] = M == 1 ? p[1] - dl[0] : fma_t<T>(-r[M - 1], dl[M - 1], p[M]);
        T v = h[M];
        gl[M - 1] = M == 1 ? v : v * r[M - 1];
#pragma unroll
        for (int j = M - 1; j >= 1; --j) {
            if (M - j > 1) v *= Recip<T>::of(M - j);
            v *= dl[j];
            h[j] += v;
            gl[j - 1] = fma_t<T>(v, r[j - 1], gl[j - 1]);
        }
        chain_step_adjoint<T, DEG, M + 1>(p, h, dl, gl);
    }
}

}  // namespace
}  // namespace psig
