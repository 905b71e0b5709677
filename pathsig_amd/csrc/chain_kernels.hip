// Products of long chains of signatures: the time chunks of a few long paths.
//
// Few rows fill the device only when each is cut into hundreds of chunks, and then the products of the chunks, one
// after the other (dense_scan_kernel, combine_staged), take longer than the sweeps: about 1 us per product.  Here
// they are formed in log_R(n) launches instead, every launch a step of a parallel prefix product over all chunks of
// all rows and both directions at once (Kogge-Stone with radix R):
//     x_c <- x_{c-(R-1)s} (x) .. (x) x_{c-s} (x) x_c,    s = 1, R, R^2, ..
// The top level of the whole product is left out of the steps: given the products L_c of everything left of chunk c
// below the top level, it is a plain sum over the chunks, one thread per word and slice of chunks
// (chain_top_kernel):
//     S(w) = sum_c [ x_c(w) + sum_k L_c(w_1..w_k) x_c(w_{k+1}..w_N) ].
// Bound by the latency of the loads and of the launches, not by arithmetic or bandwidth (an element is a few kB), so
// nothing here is tiled or compiled for a shape: one thread per word, words taken apart by multiplication.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace psig {

namespace {

struct ChainLevels {
    int depth;                     // levels of the full layout; the products below hold the levels 1 .. depth - 1
    uint32_t low;                  // words of the levels 1 .. depth - 1
    uint32_t off[kMaxDepth + 1];   // first column of a level
    uint32_t width[kMaxDepth + 1];  // d^k
    uint32_t magic[kMaxDepth + 1];  // floor(2^32 / d^k) + 1: i / d^k = umulhi(i, magic) for the words that occur
};

// the words of a level: i < 2^32 / (2 d^k) holds for every (i, k) used when d^depth d^(depth - 1) < 2^31
bool chain_levels(int64_t d, int depth, ChainLevels *lv) {
    lv->depth = depth;
    double most = 1;
    for (int k = 0; k < 2 * depth - 1; ++k) most *= (double)d;
    if (d < 2 || most >= 2147483648.0) return false;
    uint32_t off = 0, w = 1;
    lv->width[0] = 1;
    lv->magic[0] = 0;
    for (int k = 1; k <= depth; ++k) {
        w *= (uint32_t)d;
        lv->off[k] = off;
        lv->width[k] = w;
        lv->magic[k] = (uint32_t)((uint64_t(1) << 32) / w) + 1;
        if (k == depth) lv->low = off;
        off += w;
    }
    return true;
}

// put(column, (A (x) B)(word)) for the words of the levels 1 .. LEVELS that belong to this thread.  The levels are
// unrolled: with a level looked up per word, its offsets are loads from the argument segment at lane-dependent
// places (measured 21 us per step for (3, 6) instead of 6).
template <typename T, int LEVELS, typename Put>
__device__ __forceinline__ void chain_product(const T *A, const T *B, uint32_t begin, uint32_t stride,
                                              const ChainLevels &lv, Put &&put) {
    if constexpr (LEVELS >= 1) {
        // the longest level first: it has work for all threads
        for (uint32_t i = begin; i < lv.width[LEVELS]; i += stride) {
            const uint32_t col = lv.off[LEVELS] + i;
            T acc = A[col] + B[col];
#pragma unroll
            for (int r = 1; r < LEVELS; ++r) {
                const uint32_t q = __umulhi(i, lv.magic[r]);  // the first LEVELS - r letters; the other r are the rest
                acc += A[lv.off[LEVELS - r] + q] * B[lv.off[r] + (i - q * lv.width[r])];
            }
            put(col, acc);
        }
        chain_product<T, LEVELS - 1>(A, B, begin, stride, lv, put);
    }
}

constexpr int kChainThreads = 256;

// Where the results of the last step go (they are not the scan's own array then): direction 0 to left[c]
// (inclusive) or left[c + 1] (exclusive; entry 0 stays unwritten), direction 1 to right[c - 1], with the identity
// at right[n - 1]; total receives x_0 (x) .. (x) x_{n-1}.
template <typename T>
struct ChainEnds {
    T *left, *right, *total;
    int64_t total_stride;
    bool inclusive;
};

// One step.  Grid: x over (row, element), y over the directions, z over slices of the words (RADIX 2 only).
// RADIX 4: the up to four factors of the element are brought to LDS in one burst, the two halves are multiplied side
// by side, then their products.  RADIX 2: straight from memory (rows too large for six of them in LDS).
template <typename T, int N, int RADIX>
__global__ void __launch_bounds__(kChainThreads)
    chain_step_kernel(const T *__restrict__ src0, const T *__restrict__ src1, int64_t src_stride, T *__restrict__ dst0,
                      T *__restrict__ dst1, int n, int s, ChainLevels lv, bool last_step, ChainEnds<T> ends) {
    extern __shared__ __align__(16) unsigned char chain_smem[];
    const uint32_t row = blockIdx.x / (uint32_t)n;
    const int c = (int)(blockIdx.x - row * (uint32_t)n);
    const bool down = blockIdx.y == 1;
    const uint32_t low = lv.low;
    const T *src = (down ? src1 : src0) + (int64_t)row * n * src_stride;
    // factors from the left: f[0] is element `first`, the next ones s elements further right
    int count = down ? (n - 1 - c) / s + 1 : c / s + 1;
    if (count > RADIX) count = RADIX;
    const int first = down ? c : c - (count - 1) * s;
    T *to = nullptr, *also = nullptr;
    if (!last_step) {
        to = (down ? dst1 : dst0) + ((int64_t)row * n + c) * low;
    } else if (down) {
        if (c > 0) to = ends.right + ((int64_t)row * n + c - 1) * low;
    } else {
        const int at = ends.inclusive ? c : c + 1;
        if (at < n) to = ends.left + ((int64_t)row * n + at) * low;
        if (c == n - 1 && ends.total) also = ends.total + (int64_t)row * ends.total_stride;
    }
    const uint32_t begin = blockIdx.z * kChainThreads + threadIdx.x, stride = gridDim.z * kChainThreads;
    if (last_step && down && c == 0) {
        T *identity = ends.right + ((int64_t)row * n + n - 1) * low;
        for (uint32_t i = begin; i < low; i += stride) identity[i] = T(0);
    }
    if (!to && !also) return;
    auto put = [&](uint32_t i, T v) {
        if (to) to[i] = v;
        if (also) also[i] = v;
    };
    const T *f0 = src + (int64_t)first * src_stride;
    const int64_t apart = (int64_t)s * src_stride;
    if (count == 1) {
        for (uint32_t i = begin; i < low; i += stride) put(i, f0[i]);
        return;
    }
    if constexpr (RADIX == 2) {
        chain_product<T, N - 1>(f0, f0 + apart, begin, stride, lv, put);
    } else {
        T *f = reinterpret_cast<T *>(chain_smem);  // four factors, then the products of the halves
        T *p = f + 4 * (int64_t)low;
        for (uint32_t i = threadIdx.x; i < low; i += kChainThreads) {
            T v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = f0[(int64_t)(q < count ? q : 0) * apart + i];
#pragma unroll
            for (int q = 0; q < 4; ++q) f[(uint32_t)q * low + i] = v[q];
        }
        __syncthreads();
        if (count == 2) {
            chain_product<T, N - 1>(f, f + low, threadIdx.x, kChainThreads, lv, put);
            return;
        }
        // (half of the block to each of the two products)
        constexpr uint32_t kHalf = kChainThreads / 2;
        const uint32_t which = threadIdx.x / kHalf;
        if (which == 0 || count == 4) {
            const T *A = f + which * 2 * low;
            T *to_half = p + which * low;
            chain_product<T, N - 1>(A, A + low, threadIdx.x % kHalf, kHalf, lv, [&](uint32_t i, T v) { to_half[i] = v; });
        }
        __syncthreads();
        chain_product<T, N - 1>(p, count == 4 ? p + low : f + 2 * low, threadIdx.x, kChainThreads, lv, put);
    }
}

// Top level of the product of n elements (rows of `stride` columns, full layout) from the products of everything to
// the left of every element (ChainLeft).  A wave takes V runs of 64 words (so that 2 N V loads are in flight), the
// waves of a block share the elements.  left.total: the rows of the product of all below the top level are copied to
// `out` too.
constexpr int kTopWaves = 16;  // at most
template <typename T, int N, int V>
__global__ void __launch_bounds__(kTopWaves *kWave)
    chain_top_kernel(const T *__restrict__ elements, int64_t stride, ChainLeft<T> left, T *__restrict__ out,
                     int64_t out_stride, int n, ChainLevels lv) {
    __shared__ T part[kTopWaves][V][kWave];
    const int lane = (int)threadIdx.x % kWave, wave = (int)threadIdx.x / kWave, waves = (int)blockDim.x / kWave;
    const int64_t row = blockIdx.y;
    const uint32_t top = lv.width[N], first = blockIdx.x * (V * kWave) + lane;
    T acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = T(0);
    for (int c = wave; c < n; c += waves) {
        const T *x = elements + (row * n + c) * stride;
        const T *L = left.first + (row * left.per_row + (int64_t)c * left.step + left.shift) * (int64_t)lv.low;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint32_t w = first + v * kWave;
            const uint32_t i = w < top ? w : top - 1;
            T sum = x[lv.off[N] + i];
            if (c > 0) {
#pragma unroll
                for (int r = 1; r < N; ++r) {
                    const uint32_t q = __umulhi(i, lv.magic[r]);
                    sum += L[lv.off[N - r] + q] * x[lv.off[r] + (i - q * lv.width[r])];
                }
            }
            acc[v] += sum;
        }
    }
    if (waves > 1) {
#pragma unroll
        for (int v = 0; v < V; ++v) part[wave][v][lane] = acc[v];
        __syncthreads();
        if (wave == 0) {
            for (int k = 1; k < waves; ++k)
#pragma unroll
                for (int v = 0; v < V; ++v) acc[v] += part[k][v][lane];
        }
    }
    if (wave == 0) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const uint32_t w = first + v * kWave;
            if (w < top) out[row * out_stride + lv.off[N] + w] = acc[v];
            // (there are fewer words below the top level than on it, so every one has a thread)
            if (left.total && w < lv.low)
                out[row * out_stride + w] = left.first[(row * left.per_row + left.per_row - 1) * (int64_t)lv.low + w];
        }
    }
}

// Adjoints of the chunks.  Grid: x over (row, chunk), y over slices of the words.  A word of level m sums over the d + d^2 +
// .. + d^(depth - m) words that continue it: by a block, or by a group of lanes, as many as that number keeps at work, the
// more the fewer words a level has.  Bandwidth of L2: every level is read once per shorter level.
template <typename T>
__global__ void __launch_bounds__(kChainThreads)
    chunk_adjoints_kernel(const T *__restrict__ grad, const T *__restrict__ right, T *__restrict__ out, int n, ChainLevels lv) {
    const uint32_t unit = blockIdx.x, row = unit / (uint32_t)n;
    const int depth = lv.depth;
    const int64_t all = (int64_t)lv.low + lv.width[depth];
    const T *g = grad + row * all;
    const T *z = right + (int64_t)unit * lv.low;
    T *to = out + (int64_t)unit * all;
    const uint32_t tid = blockIdx.y * kChainThreads + threadIdx.x, threads = gridDim.y * kChainThreads;
    if (unit - row * (uint32_t)n == (uint32_t)n - 1) {
        // nothing follows the last chunk (and a product with what is zero there would turn an infinite gradient into NaN)
        for (int64_t i = tid; i < all; i += threads) to[i] = g[i];
        return;
    }
    for (uint32_t i = tid; i < lv.width[depth]; i += threads) to[lv.low + i] = g[lv.low + i];
    __shared__ T part_sums[kChainThreads / kWave];
    uint32_t longer = 0;
    for (int m = depth - 1; m >= 1; --m) {
        longer += lv.width[depth - m];
        if (longer >= 1024) {
            // the short words: a block each, four products of a lane in flight
            for (uint32_t w = blockIdx.y; w < lv.width[m]; w += gridDim.y) {
                T sum = T(0);
                for (int q = 1; q <= depth - m; ++q) {
                    const T *from = g + lv.off[m + q] + w * lv.width[q], *by = z + lv.off[q];
                    T level[4] = {T(0), T(0), T(0), T(0)};
                    uint32_t s = threadIdx.x;
                    for (; s + 3 * kChainThreads < lv.width[q]; s += 4 * kChainThreads)
#pragma unroll
                        for (int r = 0; r < 4; ++r) level[r] += from[s + r * kChainThreads] * by[s + r * kChainThreads];
                    for (; s < lv.width[q]; s += kChainThreads) level[0] += from[s] * by[s];
                    sum += (level[0] + level[1]) + (level[2] + level[3]);
                }
                for (uint32_t o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, (int)o, kWave);
                if (threadIdx.x % kWave == 0) part_sums[threadIdx.x / kWave] = sum;
                __syncthreads();
                if (threadIdx.x == 0) {
                    for (int v = 1; v < kChainThreads / kWave; ++v) sum += part_sums[v];
                    to[lv.off[m] + w] = g[lv.off[m] + w] + sum;
                }
                __syncthreads();
            }
            continue;
        }
        const uint32_t lanes = longer >= 256 ? kWave : longer >= 32 ? 16 : longer >= 8 ? 4 : 1;
        const uint32_t part = tid % lanes, step = threads / lanes;
        // (whole waves stay together: the shuffles below need all lanes of a group)
        for (uint32_t w = tid / lanes; w < (lv.width[m] + step - 1) / step * step; w += step) {
            T sum = T(0);
            if (w < lv.width[m]) {
                for (int q = 1; q <= depth - m; ++q) {
                    const T *from = g + lv.off[m + q] + w * lv.width[q], *by = z + lv.off[q];
                    T level = T(0);
                    for (uint32_t s = part; s < lv.width[q]; s += lanes) level += from[s] * by[s];
                    sum += level;
                }
            }
            for (uint32_t o = lanes / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, (int)o, kWave);
            if (part == 0 && w < lv.width[m]) to[lv.off[m] + w] = g[lv.off[m] + w] + sum;
        }
    }
}

}  // namespace

namespace {
// (two blocks to a CU at least)
int chain_radix(size_t elem, uint32_t low) { return 6 * (size_t)low * elem <= 78 * 1024 ? 4 : 2; }
int chain_steps(int n, int radix) {
    int steps = 0;
    for (int64_t s = 1; s < n; s *= radix) ++steps;
    return steps;
}
}  // namespace

bool chain_possible(int64_t rows, int n, int64_t d, int depth) {
    ChainLevels lv;
    return depth >= 2 && n >= 6 && rows * n < (int64_t(1) << 31) && rows < 65536 && chain_levels(d, depth, &lv);
}

// A step takes 4 us plus, with many rows, what it has to compute: 4 us per million words in fp32, 8 in fp64
// ((4, 6) in fp64, 32 rows of 32: 16.5 us; (6, 5) in fp32, 32 rows of 8: 7.1 us).
double chain_us(size_t elem, int64_t rows, int n, int64_t d, int depth, int directions) {
    ChainLevels lv;
    if (!chain_possible(rows, n, d, depth) || !chain_levels(d, depth, &lv)) return 1e9;
    const double words = 1e-6 * (double)rows * n * directions * lv.low;
    return chain_steps(n, chain_radix(elem, lv.low)) * (4.0 + (double)elem * words);
}

// The sum over the elements: 3 us plus 0.17 us per million bytes of operands, two per level and word ((4, 6) in fp64,
// 32 rows of 32: 29 us; (6, 5) in fp32, 32 rows of 8: 12 us).
double chain_top_us(size_t elem, int64_t rows, int n, int64_t d, int depth) {
    ChainLevels lv;
    if (!chain_possible(rows, n, d, depth) || !chain_levels(d, depth, &lv)) return 1e9;
    return 3.0 + 0.17e-6 * (double)rows * n * lv.width[depth] * depth * (double)elem;
}

namespace {
template <typename T, int N>
hipError_t chain_of_depth(const T *src, int64_t src_stride, int64_t rows, int n, int64_t d, T *left,
                          bool left_inclusive, T *right, T *total, int64_t total_stride, T *temp, int64_t temp_elems,
                          hipStream_t stream) {
    ChainLevels lv;
    if (!chain_levels(d, N, &lv)) return hipErrorNotSupported;
    const size_t lds = 6 * (size_t)lv.low * sizeof(T);
    const int radix = chain_radix(sizeof(T), lv.low);
    const int steps = chain_steps(n, radix);
    const ChainEnds<T> ends{left, right, total, total_stride, left_inclusive};
    const T *from0 = src, *from1 = src;
    int64_t from_stride = src_stride;
    int64_t s = 1;
    for (int k = 0; k < steps; ++k, s *= radix) {
        const bool last = k == steps - 1;
        // the arrays that the last step writes serve as the other half of a double buffer on the way there
        const bool in_temp = (steps - 1 - k) % 2 == 1;
        T *to0 = in_temp ? temp : left, *to1 = in_temp ? temp + temp_elems : right;
        const dim3 grid((unsigned)(rows * n), right ? 2 : 1,
                        radix == 2 ? (unsigned)((lv.low + 4 * kChainThreads - 1) / (4 * kChainThreads)) : 1);
        if (radix == 4) {
            if (lds > 32 * 1024) {
                hipError_t e = allow_dynamic_lds<chain_step_kernel<T, N, 4>>(lds);
                if (e != hipSuccess) return e;
            }
            hipLaunchKernelGGL((chain_step_kernel<T, N, 4>), grid, dim3(kChainThreads), lds, stream, from0, from1,
                               from_stride, to0, to1, n, (int)s, lv, last, ends);
        } else {
            hipLaunchKernelGGL((chain_step_kernel<T, N, 2>), grid, dim3(kChainThreads), 0, stream, from0, from1,
                               from_stride, to0, to1, n, (int)s, lv, last, ends);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        from0 = to0;
        from1 = to1;
        from_stride = lv.low;
    }
    return hipSuccess;
}

// f(std::integral_constant<int, depth>)
template <int N = 2, typename F>
hipError_t with_depth(int depth, F &&f) {
    if constexpr (N > kMaxDepth) {
        return hipErrorNotSupported;
    } else {
        return depth == N ? f(std::integral_constant<int, N>{}) : with_depth<N + 1>(depth, f);
    }
}
}  // namespace

template <typename T>
hipError_t launch_chain(const T *src, int64_t src_stride, int64_t rows, int n, int64_t d, int depth, T *left,
                        bool left_inclusive, T *right, T *total, int64_t total_stride, T *temp, int64_t temp_elems,
                        hipStream_t stream) {
    return with_depth(depth, [&](auto nc) {
        return chain_of_depth<T, decltype(nc)::value>(src, src_stride, rows, n, d, left, left_inclusive, right, total,
                                                      total_stride, temp, temp_elems, stream);
    });
}

template <typename T>
hipError_t launch_chain_top(const T *elements, int64_t stride, const ChainLeft<T> &left, T *out, int64_t out_stride,
                            int64_t rows, int n, int64_t d, int depth, hipStream_t stream) {
    ChainLevels lv;
    if (!chain_levels(d, depth, &lv)) return hipErrorNotSupported;
    return with_depth(depth, [&](auto nc) {
        constexpr int N = decltype(nc)::value;
        // four runs to a wave when that leaves two waves to a SIMD; the elements are split until there are four
        const int64_t runs = (lv.width[depth] + kWave - 1) / kWave;
        const bool wide = rows * runs >= 8192;
        const int64_t blocks = wide ? (runs + 3) / 4 : runs;
        int waves = 1;
        while (waves < kTopWaves && 2 * waves <= n && rows * blocks * waves < 4096) waves *= 2;
        auto launch = [&](auto vc) {
            hipLaunchKernelGGL((chain_top_kernel<T, N, decltype(vc)::value>), dim3((unsigned)blocks, (unsigned)rows),
                               dim3(waves * kWave), 0, stream, elements, stride, left, out, out_stride, n, lv);
        };
        if (wide) launch(std::integral_constant<int, 4>{});
        else launch(std::integral_constant<int, 1>{});
        return hipGetLastError();
    });
}

namespace {
// blocks to a chunk: enough for a few thousand waves, none without 1024 words of its own
unsigned adjoint_slices(int64_t units, uint32_t top) {
    int64_t slices = 1;
    while (slices * units < 2048 && slices * 2048 <= (int64_t)top) slices *= 2;
    return (unsigned)slices;
}
}  // namespace

template <typename T>
hipError_t launch_chunk_adjoints(const T *grad, const T *right, T *out, int64_t rows, int n, int64_t d, int depth,
                                 hipStream_t stream) {
    ChainLevels lv;
    if (!chain_levels(d, depth, &lv)) return hipErrorNotSupported;
    hipLaunchKernelGGL(chunk_adjoints_kernel<T>, dim3((unsigned)(rows * n), adjoint_slices(rows * n, lv.width[depth])),
                       dim3(kChainThreads), 0, stream, grad, right, out, n, lv);
    return hipGetLastError();
}

// 4 us, and what it reads and writes at 4 TB/s
double chunk_adjoints_us(size_t elem, int64_t rows, int n, int64_t d, int depth) {
    ChainLevels lv;
    if (!chain_levels(d, depth, &lv)) return 1e9;
    return 4.0 + 0.25e-6 * (double)rows * n * lv.width[depth] * (depth + 1) * (double)elem;
}

#define PSIG_INSTANTIATE(T)                                                                                         \
    template hipError_t launch_chunk_adjoints<T>(const T *, const T *, T *, int64_t, int, int64_t, int, hipStream_t); \
    template hipError_t launch_chain<T>(const T *, int64_t, int64_t, int, int64_t, int, T *, bool, T *, T *, int64_t, \
                                        T *, int64_t, hipStream_t);                                                 \
    template hipError_t launch_chain_top<T>(const T *, int64_t, const ChainLeft<T> &, T *, int64_t, int64_t, int, int64_t, int, \
                                            hipStream_t);
PSIG_INSTANTIATE(float)
PSIG_INSTANTIATE(double)
#undef PSIG_INSTANTIATE

}  // namespace psig
