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

// Increments of time chunk c of a span.
__device__ __forceinline__ WindowSpan chunk_of_span(const WindowSpan &span, int chunks, int c) {
    const int64_t begin = span.steps * c / chunks;
    return {span.start + begin, span.steps * (c + 1) / chunks - begin};
}

// place of w_(i+1) .. w_j among the factors of a word of length n
__host__ __device__ constexpr int factor_at(int n, int i, int j) { return i * n - i * (i - 1) / 2 + j - i - 1; }

// A lane sweeps its word, BLOCK lanes to a block.  FACTORS: `sig` is the table of a call in time chunks (words_chunks.hip),
// `row` counts the chunks of all paths, and the lane's word is a suffix of length DEG of one of the words of the levels
// DEG .. depth, whose chain it leaves in the table.
template <typename T, int DEG, int BLOCK, bool FACTORS = false>
__device__ void forward_body(const T *__restrict__ path, T *__restrict__ sig, const SigShape &shape,
                             const LevelPlan &plan, const int64_t *__restrict__ codes, int64_t row, int64_t blk_in_level,
                             int tile, T *sdx, const WordChunks *wc = nullptr) {
    const int tid = threadIdx.x;
    const int64_t d = shape.d;
    int64_t word_idx = blk_in_level * BLOCK + tid;
    bool active = word_idx < plan.size[DEG];
    int n = DEG;  // length of the word
    if constexpr (FACTORS) {
        while (!active && n < plan.depth) {
            word_idx -= plan.size[n++];
            active = word_idx < plan.size[n];
        }
    }
    uint64_t code = 0;
    if (active) code = plan.code_off[n] >= 0 ? (uint64_t)codes[plan.code_off[n] + word_idx] : (uint64_t)word_idx;
    int l[DEG];
    decode_letters<DEG>(code, (uint64_t)d, l);

    const int64_t per_path = FACTORS ? wc->chunks : shape.W;
    const int64_t b = row / per_path, w = row - b * per_path;
    WindowSpan span;
    if constexpr (FACTORS) span = chunk_of_span(window_span(shape, 0), wc->chunks, (int)w);
    else span = window_span(shape, w);
    const T *x = path + (b * shape.L + span.start) * d;

    T p[DEG + 1];
    p[0] = T(1);
#pragma unroll
    for (int k = 1; k <= DEG; ++k) p[k] = T(0);

    // Increments are staged in pairs, [pair][letter][increment of the pair]: a read, and the address that it takes, bring a
    // letter of two of them, which matters because a word of length n takes n reads beside some n^2 instructions of its chain.
    // Forward launch, one increment / two to a read: 256 paths of 512 points, 16 letters, 2320 words up to length 6, fp32
    // 205 / 181 us, fp64 345 / 313; 200 paths of 700, 1020 words up to length 8 over 12 letters, 300 / 279.  (The letter and pair
    // of an element are carried along: a division for each costs 3 of 34 us over 100 letters, 2000 words, 256 paths of 128.)
    typedef T Pair __attribute__((ext_vector_type(2)));
    const int width = (int)d;
    const int first_letter = tid % width, first_pair = tid / width;
    int at[DEG];
#pragma unroll
    for (int k = 0; k < DEG; ++k) at[k] = 2 * l[k];
    for (int64_t t0 = 0; t0 < span.steps; t0 += tile) {
        const int nt = (int)((span.steps - t0) < tile ? (span.steps - t0) : tile);
        const T *xw = x + t0 * d;
        __syncthreads();
        int letter = first_letter, pair = first_pair;  // of element idx
        for (int idx = tid; idx < (nt + 1) / 2 * width; idx += BLOCK, letter += BLOCK % width, pair += BLOCK / width) {
            if (letter >= width) {
                letter -= width;
                ++pair;
            }
            const T *from = xw + (int64_t)pair * 2 * d + letter;
            const T mid = from[d], first = mid - from[0];
            const T second = 2 * pair + 1 < nt ? from[2 * d] - mid : T(0);
            reinterpret_cast<Pair *>(sdx)[idx] = Pair{first, second};
        }
        __syncthreads();
        if (active) {
            const T *dxr = sdx;
            T dl[DEG];
            for (int tt = 0; tt + 1 < nt; tt += 2, dxr += 2 * width) {
                Pair both[DEG];
#pragma unroll
                for (int k = 0; k < DEG; ++k) both[k] = *reinterpret_cast<const Pair *>(dxr + at[k]);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
#pragma unroll
                    for (int k = 0; k < DEG; ++k) dl[k] = both[k][i];
                    chain_step<T, DEG, DEG>(p, dl);
                }
            }
            if (nt % 2) {
#pragma unroll
                for (int k = 0; k < DEG; ++k) dl[k] = dxr[at[k]];
                chain_step<T, DEG, DEG>(p, dl);
            }
        }
    }
    if constexpr (FACTORS) {
        if (active) {
            T *to = sig + row * wc->table_size + wc->table_off[n] + (int64_t)factor_at(n, n - DEG, n - DEG + 1) * plan.size[n] +
                    word_idx;
#pragma unroll
            for (int k = 1; k <= DEG; ++k) to[(k - 1) * plan.size[n]] = p[k];
        }
        return;
    }
    if (active) {
        sig[row * plan.sig_size + plan.out_off[DEG] + word_idx] = p[DEG];
        if (plan.keep && plan.keep_off[DEG] >= 0) {
            T *kept = (T *)plan.keep + row * plan.keep_size + plan.keep_off[DEG] + word_idx * (DEG - 1);
#pragma unroll
            for (int k = 1; k < DEG; ++k) kept[k - 1] = p[k];
        }
    }
}

// Chain and adjoint of a word at the right edge of a time chunk (unit: row * chunks + chunk): h[DEG] holds the upstream
// gradient.  (Nothing follows the last chunk, and a product with what is zero there would turn an infinite gradient into NaN.)
template <typename T, int DEG>
__device__ __forceinline__ void word_chunk_edges(const WordChunks &wc, const LevelPlan &plan, int64_t unit, int64_t word,
                                                 T (&p)[DEG + 1], T (&h)[DEG + 1]) {
    const int64_t size = plan.size[DEG], at = unit * wc.edge_size + wc.edge_off[DEG] + word;
    const T *left = (const T *)wc.left + at, *right = (const T *)wc.right + at;
    const bool last = unit % wc.chunks == wc.chunks - 1;
#pragma unroll
    for (int k = 1; k < DEG; ++k) {
        p[k] = left[(k - 1) * size];
        h[k] = last ? T(0) : h[DEG] * right[(k - 1) * size];
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
