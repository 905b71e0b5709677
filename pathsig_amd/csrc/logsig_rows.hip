// Log-signature of small layouts (d^depth <= 4096), one block per row with everything the row needs in LDS, compiled
// for the alphabet and the depth.  The formulas are those at the head of logsig_kernels.hip; what changes is the form:
//   * a top-level word needs the powers of the log-signature only through
//         Qc(u) = -sum_{k=2}^{|u|+1} Q_{k-1}(u) / k! ,      L(w) = S(w) + sum_j Qc(w_1..w_j) L(w_{j+1}..w_N),
//     N - 1 products instead of N (N - 1) / 2, and only wanted words are computed;
//   * the adjoint builds the powers again from the log-signature instead of reading them (a row of (6, 4): 1 kB
//     instead of 5), so the forward writes nothing but its outputs and the log-signature below the top level;
//   * the sums over the top level start in registers: a thread takes the d words below one prefix of length N - 1 for
//     all sums over suffixes, and the d words above one suffix of length N - 1 for all sums over prefixes, one value
//     per thread and sum; what is left are sums of those values.
// A row is a few thousand multiply-adds, so the kernels are bound by LDS traffic and by the latency of their 2 N
// passes; the general kernels spent most of their time on index arithmetic with a run-time alphabet and on generic
// reductions ((6, 4), 4064 rows: 36 + 72 + 13 us for the adjoint there, 23 us for the forward).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.hpp"

#ifndef PSIG_ROWS_TYPE
#define PSIG_ROWS_TYPE float
#endif

namespace psig {

namespace {

constexpr int ipow(int b, int e) { return e <= 0 ? 1 : b * ipow(b, e - 1); }

template <int Begin, int End, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (Begin < End) {
        f(std::integral_constant<int, Begin>{});
        static_for<Begin + 1, End>(f);
    }
}

template <typename T>
__device__ __forceinline__ constexpr T inv_factorial(int k) {
    T r = T(1);
    for (int i = 2; i <= k; ++i) r /= T(i);
    return r;
}

template <typename T, int D, int N>
struct Rows {
    static constexpr int off(int k) { return k <= 1 ? 0 : off(k - 1) + ipow(D, k - 1); }  // first column of level k
    static constexpr int kLow = off(N);        // columns below the top level
    static constexpr int kTop = ipow(D, N);
    static constexpr int kPre = ipow(D, N - 1);  // prefixes (suffixes) of length N - 1
    // a thread for each of these, up to 512; for a tiny layout a wave
    static constexpr int kThreads = kPre >= 512 ? 512 : (kPre + kWave - 1) / kWave * kWave;
    static constexpr int kPowers = N >= 3 ? N - 2 : 0;  // Q_2 .. Q_{N-1}
    static constexpr int kForward = (2 + kPowers) * kLow;
    // adjoint: the top level; L, Qc, R, T and the gradient below it; Q_k; a_k, in the place of the per-thread sums
    static constexpr int kSums = 2 * kPowers * kPre, kAdj = kPowers * kLow;
    static constexpr int kBackward = kTop + 5 * kLow + kPowers * kLow + (kSums > kAdj ? kSums : kAdj);
    static constexpr bool kUsable = kTop <= 4096 && (size_t)kBackward * sizeof(T) <= 150 * 1024;
};

// Q_k(w) of a word of level n from Q_{k-1} and L
template <typename T, int D, int N, int n, int k>
__device__ __forceinline__ T power_of_word(const T *L, const T *Q, int i) {
    using R = Rows<T, D, N>;
    T q = T(0);
    static_for<k - 1, n>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        constexpr int tail = ipow(D, n - j);
        const T *left = k == 2 ? L : Q + (k - 3) * R::kLow;
        q += left[R::off(j) + i / tail] * L[R::off(n - j) + i % tail];
    });
    return q;
}

// Qc from the powers
template <typename T, int D, int N, int n>
__device__ __forceinline__ T weight_of_word(const T *L, const T *Q, int col) {
    using R = Rows<T, D, N>;
    T c = -inv_factorial<T>(2) * L[col];
    static_for<2, n + 1>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        c -= inv_factorial<T>(k + 1) * Q[(k - 2) * R::kLow + col];
    });
    return c;
}

// sig: dense rows; lg (may be null): [rows, kLow] log-signature below the top level; out: [rows, n_out].
// picked: hybrid column of every output (null: all columns, dense); top_words: top_size codes of a listed top level.
// The gridDim.y blocks of a row share its outputs (each computes the levels below the top for itself).
template <typename T, int D, int N>
__global__ void __launch_bounds__((Rows<T, D, N>::kThreads))
    log_rows_forward_kernel(const T *__restrict__ sig, T *__restrict__ lg, T *__restrict__ out, int n_out, int64_t top_size,
                            const int64_t *__restrict__ top_words, const int64_t *__restrict__ picked) {
    using R = Rows<T, D, N>;
    __shared__ T mem[R::kForward];
    T *L = mem, *Qc = mem + R::kLow, *Q = mem + 2 * R::kLow;
    const int64_t row = blockIdx.x;
    const T *s = sig + row * (R::kLow + R::kTop);
    const int tid = (int)threadIdx.x;
    static_for<1, N>([&](auto nc) {
        constexpr int n = decltype(nc)::value;
        for (int i = tid; i < ipow(D, n); i += R::kThreads) {
            const int col = R::off(n) + i;
            T acc = s[col];
            static_for<2, n + 1>([&](auto kc) {
                constexpr int k = decltype(kc)::value;
                const T q = power_of_word<T, D, N, n, k>(L, Q, i);
                acc -= inv_factorial<T>(k) * q;
                Q[(k - 2) * R::kLow + col] = q;
            });
            L[col] = acc;
            Qc[col] = weight_of_word<T, D, N, n>(L, Q, col);
            if (lg && blockIdx.y == 0) lg[row * R::kLow + col] = acc;
        }
        __syncthreads();
    });
    T *o = out + row * n_out;
    const int first = (int)blockIdx.y * R::kThreads + tid, stride = (int)gridDim.y * R::kThreads;
    if (!picked) {
        // everything: a thread takes the words below one prefix of length N - 1
        for (int col = first; col < R::kLow; col += stride) o[col] = L[col];
        for (int p = first; p < R::kPre; p += stride) {
            T acc[D];
#pragma unroll
            for (int b = 0; b < D; ++b) acc[b] = s[R::kLow + p * D + b];
            static_for<1, N>([&](auto jc) {
                constexpr int j = decltype(jc)::value;
                const T c = Qc[R::off(j) + p / ipow(D, N - 1 - j)];
                const T *l = L + R::off(N - j) + (p % ipow(D, N - 1 - j)) * D;
#pragma unroll
                for (int b = 0; b < D; ++b) acc[b] += c * l[b];
            });
#pragma unroll
            for (int b = 0; b < D; ++b) o[R::kLow + p * D + b] = acc[b];
        }
        return;
    }
    for (int j = first; j < n_out; j += stride) {
        const int at = (int)picked_column(picked[j], top_words, R::kLow, R::kLow + top_size, R::kTop);
        if (at < 0) {
            o[j] = (T)NAN;
        } else if (at < R::kLow) {
            o[j] = L[at];
        } else {
            const int w = at - R::kLow;
            T acc = s[R::kLow + w];
            static_for<1, N>([&](auto jc) {
                constexpr int p = decltype(jc)::value;
                constexpr int tail = ipow(D, N - p);
                acc += Qc[R::off(p) + w / tail] * L[R::off(N - p) + w % tail];
            });
            o[j] = acc;
        }
    }
}

// largest power of two of lanes that can share one of `outputs` sums of `terms` terms
constexpr int lanes_per_sum(int threads, int outputs, int terms) {
    int g = 1;
    while (2 * g * outputs <= threads && 2 * g <= terms && 2 * g <= kWave) g *= 2;
    return g;
}

template <int G, typename T>
__device__ __forceinline__ T sum_of_lanes(T v) {
#pragma unroll
    for (int off = G / 2; off >= 1; off /= 2) v += __shfl_xor(v, off);
    return v;
}

// grad: [rows, n_out]; dense: [rows, kLow + kTop], the gradient of the dense signature rows (every column written)
template <typename T, int D, int N>
__global__ void __launch_bounds__((Rows<T, D, N>::kThreads))
    log_rows_adjoint_kernel(const T *__restrict__ lg, const T *__restrict__ grad, T *__restrict__ dense, int n_out, int64_t top_size,
                            const int64_t *__restrict__ top_words, const int64_t *__restrict__ picked) {
    using R = Rows<T, D, N>;
    extern __shared__ __align__(16) unsigned char rows_smem[];
    T *g = reinterpret_cast<T *>(rows_smem);  // top level of the gradient
    T *lam = g + R::kTop;                     // gradient below it, in the end that of the signature
    T *L = lam + R::kLow, *Qc = L + R::kLow, *Rs = Qc + R::kLow, *Ts = Rs + R::kLow, *Q = Ts + R::kLow;
    T *z = Q + R::kPowers * R::kLow, *y = z + R::kPowers * R::kPre;  // the per-thread sums
    T *a = z;                                                        // a_k, k >= 2 (z and y are read no more then)
    const int64_t row = blockIdx.x;
    const int tid = (int)threadIdx.x;
    const T *gin = grad + row * n_out;
    if (picked) {
        for (int i = tid; i < R::kTop + R::kLow; i += R::kThreads) g[i] = T(0);
    } else {
        for (int i = tid; i < R::kTop; i += R::kThreads) g[i] = gin[R::kLow + i];
        for (int i = tid; i < R::kLow; i += R::kThreads) lam[i] = gin[i];
    }
    for (int i = tid; i < R::kLow; i += R::kThreads) L[i] = lg[row * R::kLow + i];
    __syncthreads();
    if (picked) {
        for (int j = tid; j < n_out; j += R::kThreads) {
            const int at = (int)picked_column(picked[j], top_words, R::kLow, R::kLow + top_size, R::kTop);
            // (an output may be asked for twice)
            if (at >= R::kLow) atomicAdd(&g[at - R::kLow], gin[j]);
            else if (at >= 0) atomicAdd(&lam[at], gin[j]);
        }
    }
    static_for<2, N>([&](auto kc) {
        constexpr int k = decltype(kc)::value;
        static_for<k, N>([&](auto nc) {
            constexpr int n = decltype(nc)::value;
            for (int i = tid; i < ipow(D, n); i += R::kThreads)
                Q[(k - 2) * R::kLow + R::off(n) + i] = power_of_word<T, D, N, n, k>(L, Q, i);
        });
        __syncthreads();
    });
    static_for<1, N>([&](auto nc) {
        constexpr int n = decltype(nc)::value;
        for (int i = tid; i < ipow(D, n); i += R::kThreads)
            Qc[R::off(n) + i] = weight_of_word<T, D, N, n>(L, Q, R::off(n) + i);
    });
    __syncthreads();
    // sums over the top level, the part of one prefix and of one suffix of length N - 1
    for (int p = tid; p < R::kPre; p += R::kThreads) {
        T v[D];
#pragma unroll
        for (int b = 0; b < D; ++b) v[b] = g[p * D + b];
        static_for<1, N>([&](auto jc) {
            constexpr int j = decltype(jc)::value;  // R(u), |u| = j: the rest of p and the last letter are its suffix
            const T *l = L + R::off(N - j) + (p % ipow(D, N - 1 - j)) * D;
            T sum = T(0);
#pragma unroll
            for (int b = 0; b < D; ++b) sum += v[b] * l[b];
            if constexpr (j == N - 1) Rs[R::off(j) + p] = sum;
            else z[(j - 1) * R::kPre + p] = sum;
        });
#pragma unroll
        for (int b = 0; b < D; ++b) v[b] = g[b * R::kPre + p];
        static_for<1, N>([&](auto ic) {
            constexpr int i = decltype(ic)::value;  // T(v), |v| = i: the first letter and the head of p are its prefix
            const T *c = Qc + R::off(N - i) + p / ipow(D, i);
            T sum = T(0);
#pragma unroll
            for (int b = 0; b < D; ++b) sum += v[b] * c[b * ipow(D, N - 1 - i)];
            if constexpr (i == N - 1) Ts[R::off(i) + p] = sum;
            else y[(i - 1) * R::kPre + p] = sum;
        });
    }
    __syncthreads();
    static_for<1, N - 1>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        constexpr int outs = ipow(D, j), terms = ipow(D, N - 1 - j), G = lanes_per_sum(R::kThreads / 2, outs, terms);
        // half of the block to either side where a wave is not split by that
        for (int o = tid / G; o < 2 * outs; o += R::kThreads / G) {
            const bool suffix = o >= outs;
            const int w = suffix ? o - outs : o;
            T sum = T(0);
            if (suffix)
                for (int t = tid % G; t < terms; t += G) sum += y[(j - 1) * R::kPre + t * outs + w];
            else
                for (int t = tid % G; t < terms; t += G) sum += z[(j - 1) * R::kPre + w * terms + t];
            sum = sum_of_lanes<G>(sum);
            if (tid % G == 0) (suffix ? Ts : Rs)[R::off(j) + w] = sum;
        }
    });
    __syncthreads();
    // the levels below the top, going down
    static_for<1, N>([&](auto mc) {
        constexpr int n = N - decltype(mc)::value;
        constexpr int words = ipow(D, n), between = N - 1 - n;
        constexpr int G = between == 0 ? 1 : lanes_per_sum(R::kThreads, words, ipow(D, between));
        for (int w = tid / G; w < words; w += R::kThreads / G) {
            const int part = tid % G, col = R::off(n) + w;
            T A[n + 1];  // A[k] = sum_v a_{k+1}(w v) L(v), k = 1 .. n, over the levels between this one and the top
            T U = T(0);  // sum_u sum_k a_k(u w) Q_{k-1}(u)
#pragma unroll
            for (int k = 0; k <= n; ++k) A[k] = T(0);
            static_for<1, between + 1>([&](auto ic) {
                constexpr int i = decltype(ic)::value;
                for (int v = part; v < ipow(D, i); v += G) {
                    const T lv = L[R::off(i) + v];
                    const int at = R::off(n + i) + w * ipow(D, i) + v;
#pragma unroll
                    for (int k = 1; k <= n; ++k) A[k] += a[(k - 1) * R::kLow + at] * lv;
                }
                for (int u = part; u < ipow(D, i); u += G) {
                    const int at = R::off(n + i) + u * words + w, from = R::off(i) + u;
                    U += a[at] * L[from];
#pragma unroll
                    for (int k = 3; k <= i + 1; ++k) U += a[(k - 2) * R::kLow + at] * Q[(k - 3) * R::kLow + from];
                }
            });
            if constexpr (G > 1) {
#pragma unroll
                for (int k = 1; k <= n; ++k) A[k] = sum_of_lanes<G>(A[k]);
                U = sum_of_lanes<G>(U);
            }
            if (part == 0) {
                const T r = Rs[col];
                const T total = lam[col] + (A[1] - inv_factorial<T>(2) * r) + Ts[col] + U;
                lam[col] = total;
#pragma unroll
                for (int k = 2; k <= n; ++k)
                    a[(k - 2) * R::kLow + col] = A[k] - inv_factorial<T>(k + 1) * r - inv_factorial<T>(k) * total;
            }
        }
        __syncthreads();
    });
    T *o = dense + row * (R::kLow + R::kTop);
    for (int i = tid; i < R::kLow; i += R::kThreads) o[i] = lam[i];
    for (int i = tid; i < R::kTop; i += R::kThreads) o[R::kLow + i] = g[i];
}

// f(integral_constant d, integral_constant depth) for the compiled layout, or `otherwise`
template <typename T, int D, int N, typename F, typename E>
E with_layout(int64_t d, int depth, F &&f, E otherwise) {
    if constexpr (D > 16) {
        return otherwise;
    } else if constexpr (N > 8 || ipow(D, N) > 4096) {
        return with_layout<T, D + 1, 2>(d, depth, f, otherwise);
    } else {
        if (d == D && depth == N) {
            if constexpr (Rows<T, D, N>::kUsable)
                return f(std::integral_constant<int, D>{}, std::integral_constant<int, N>{});
            else return otherwise;
        }
        return with_layout<T, D, N + 1>(d, depth, f, otherwise);
    }
}

}  // namespace

template <>
bool log_rows_possible<PSIG_ROWS_TYPE>(int64_t d, int depth) {
    return with_layout<PSIG_ROWS_TYPE, 2, 2>(d, depth, [](auto, auto) { return true; }, false);
}

template <>
hipError_t launch_log_rows_forward<PSIG_ROWS_TYPE>(const PSIG_ROWS_TYPE *sig, PSIG_ROWS_TYPE *lg, PSIG_ROWS_TYPE *out,
                                                   int64_t n_out, int64_t rows, int64_t d, int depth, int64_t top_size,
                                                   const int64_t *top_words, const int64_t *picked, hipStream_t stream) {
    return with_layout<PSIG_ROWS_TYPE, 2, 2>(
        d, depth,
        [&](auto dc, auto nc) {
            using R = Rows<PSIG_ROWS_TYPE, decltype(dc)::value, decltype(nc)::value>;
            // few rows: several blocks share the outputs of one, as long as each has a round of its own
            const int64_t rounds = ((picked ? n_out : (int64_t)R::kPre) + R::kThreads - 1) / R::kThreads;
            const int64_t slices = rows >= 512 ? 1 : std::max<int64_t>(1, std::min<int64_t>(rounds, 512 / rows));
            hipLaunchKernelGGL((log_rows_forward_kernel<PSIG_ROWS_TYPE, decltype(dc)::value, decltype(nc)::value>),
                               dim3((unsigned)rows, (unsigned)slices), dim3(R::kThreads), 0, stream, sig, lg, out,
                               (int)n_out, top_size, top_words, picked);
            return hipGetLastError();
        },
        hipErrorNotSupported);
}

template <>
hipError_t launch_log_rows_adjoint<PSIG_ROWS_TYPE>(const PSIG_ROWS_TYPE *lg, const PSIG_ROWS_TYPE *grad,
                                                   PSIG_ROWS_TYPE *dense, int64_t n_out, int64_t rows, int64_t d, int depth,
                                                   int64_t top_size, const int64_t *top_words, const int64_t *picked, hipStream_t stream) {
    return with_layout<PSIG_ROWS_TYPE, 2, 2>(
        d, depth,
        [&](auto dc, auto nc) {
            constexpr int D = decltype(dc)::value, N = decltype(nc)::value;
            using R = Rows<PSIG_ROWS_TYPE, D, N>;
            constexpr size_t bytes = (size_t)R::kBackward * sizeof(PSIG_ROWS_TYPE);
            if constexpr (bytes > 32 * 1024) {
                const hipError_t e = allow_dynamic_lds<log_rows_adjoint_kernel<PSIG_ROWS_TYPE, D, N>>(bytes);
                if (e != hipSuccess) return e;
            }
            hipLaunchKernelGGL((log_rows_adjoint_kernel<PSIG_ROWS_TYPE, D, N>), dim3((unsigned)rows), dim3(R::kThreads),
                               bytes, stream, lg, grad, dense, (int)n_out, top_size, top_words, picked);
            return hipGetLastError();
        },
        hipErrorNotSupported);
}

}  // namespace psig
