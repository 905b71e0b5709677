// Time chunks for the per-word kernels: calls of few paths and words.
//
// A word needs nothing but its own prefixes, so such a call is a few waves that sweep a path one increment after the other,
// whatever the number of words.  Cut into chunks, the signature of a word is a product over the chunks c of the
// unitriangular matrices
//     M_c[i][j] = S_c(w_(i+1) .. w_j),    S(w) = (M_0 M_1 ..)[0][n],
// whose entries are prefixes of the word's suffixes: a lane sweeps a chunk for one suffix (word_factors_kernel, n lanes for
// a word of length n, about (n + 2) / 3 times the work of the word alone), and the product is taken as the row
// e_0 M_0 M_1 .., one chunk after the other, by a lane per word (word_products_kernel).  The rows on the way are the prefix
// values at the chunks' right edges; the columns .. M_(C-1) e_n, made beside them, hold what the word's adjoint is there but
// for the upstream gradient.  With the two, the backward kernels sweep every chunk on its own.
// Bound by the latency of the chain of increments, which is what the chunks shorten, and of the products.  us, in one piece / in
// chunks: a step, 24 to 2000 words: 1 path of 300 points, 16 letters, depth 6, 2000 words, 216 / 70; fp64, 1 of 806, 12
// letters, depth 8, 245 words, 697 / 80; 16 of 2000, 16 letters, depth 8, 64 words, 1980 / 128; 40 of 500, 16 letters, depth
// 6, 300 words, fp64, 573 / 146; 270 of 1146, 11 letters, depth 8, 101 words, 1328 / 489; a forward, 77 of 1134, 5 letters,
// depth 8, 24 words, 315 / 38; 248 of 2869, 6 letters, depth 8, 457 / 184.
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "words_common.hpp"

namespace psig {

namespace {

// The waves of word_factors_kernel: suffixes of one length side by side, whatever the length of their words.  (A wave for
// each length of word and suffix left most lanes of a call with few words idle.)
struct FactorBlocks {
    int depth;
    int64_t begin[kMaxDepth + 2];  // first block of the suffixes of length m (the longest first)
};

// Grid: consecutive blocks work on the same suffixes of the chunks of all paths, the longest suffixes first.
template <typename T, int MAXDEG>
__global__ void __launch_bounds__(kWave)
    word_factors_kernel(const T *__restrict__ path, T *__restrict__ table, SigShape shape, LevelPlan plan,
                        const int64_t *__restrict__ codes, WordChunks wc, FactorBlocks fb, unsigned units, int tile) {
    extern __shared__ __align__(16) unsigned char smem[];
    const unsigned blk = blockIdx.x / units, unit = blockIdx.x - blk * units;
    int m = fb.depth;
    while (m > 1 && blk >= fb.begin[m - 1]) --m;
    switch (m) {
#define PSIG_CASE(N)                                                                                                \
    case N:                                                                                                         \
        if constexpr (N <= MAXDEG)                                                                                  \
            forward_body<T, N, kWave, true>(path, table, shape, plan, codes, unit, blk - fb.begin[N], tile,         \
                                            reinterpret_cast<T *>(smem), &wc);                                      \
        break;
        PSIG_CASE(1) PSIG_CASE(2) PSIG_CASE(3) PSIG_CASE(4) PSIG_CASE(5) PSIG_CASE(6) PSIG_CASE(7) PSIG_CASE(8)
#undef PSIG_CASE
        default: break;
    }
}

// DOWN: columns from the last chunk on (right), else rows from the first (left, sig).  The factors of the next chunk are
// read while those of one are multiplied.
template <typename T, int DEG, bool DOWN>
__device__ __forceinline__ void products_body(T *__restrict__ sig, const T *__restrict__ table, T *__restrict__ edge,
                                              const LevelPlan &plan, const WordChunks &wc, int64_t word, int64_t b) {
    constexpr int kFactors = DEG * (DEG + 1) / 2;
    const int64_t size = plan.size[DEG];
    if (word >= size) return;
    const int chunks = wc.chunks;
    const int64_t first = b * chunks + (DOWN ? chunks - 1 : 0);
    const T *from = table + first * wc.table_size + wc.table_off[DEG] + word;
    const int64_t step = DOWN ? -wc.table_size : wc.table_size;
    T *to = edge ? edge + first * wc.edge_size + wc.edge_off[DEG] + word : nullptr;
    const int64_t edge_step = DOWN ? -wc.edge_size : wc.edge_size;
    T v[DEG + 1], next[kFactors];
#pragma unroll
    for (int k = 0; k <= DEG; ++k) v[k] = k == (DOWN ? DEG : 0) ? T(1) : T(0);
    auto read = [&]() {
#pragma unroll
        for (int f = 0; f < kFactors; ++f) next[f] = from[f * size];
    };
    auto store = [&]() {
        if (to) {
#pragma unroll
            for (int k = 1; k <= DEG; ++k) to[(k - 1) * size] = v[k];
            to += edge_step;
        }
    };
    read();
    for (int c = 0; c < chunks; ++c) {
        T m[kFactors];
#pragma unroll
        for (int f = 0; f < kFactors; ++f) m[f] = next[f];
        if (c + 1 < chunks) from += step;
        read();
        if constexpr (DOWN) {
            store();  // (of what follows the chunk)
#pragma unroll
            for (int i = 1; i < DEG; ++i)
#pragma unroll
                for (int j = i + 1; j <= DEG; ++j) v[i] = fma_t<T>(m[factor_at(DEG, i, j)], v[j], v[i]);
        } else {
#pragma unroll
            for (int j = DEG; j >= 1; --j)
#pragma unroll
                for (int i = 0; i < j; ++i) v[j] = fma_t<T>(v[i], m[factor_at(DEG, i, j)], v[j]);
            store();
        }
    }
    if constexpr (!DOWN)
        if (sig) sig[b * plan.sig_size + plan.out_off[DEG] + word] = v[DEG];
}

// Grid: x over the waves of words (block_begin of the plan: 64 words each), y over the paths, z over the directions.
template <typename T, int MAXDEG>
__global__ void __launch_bounds__(kWave)
    word_products_kernel(T *__restrict__ sig, const T *__restrict__ table, T *__restrict__ left, T *__restrict__ right,
                         LevelPlan plan, WordChunks wc, int64_t B) {
    const int n = find_level(plan, blockIdx.x);
    const int64_t word = (blockIdx.x - plan.block_begin[n]) * kWave + threadIdx.x;
    for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
        switch (n) {
#define PSIG_CASE(N)                                                                                                \
    case N:                                                                                                         \
        if constexpr (N <= MAXDEG) {                                                                                \
            if (blockIdx.z == 0) products_body<T, N, false>(sig, table, left, plan, wc, word, b);                   \
            else products_body<T, N, true>(sig, table, right, plan, wc, word, b);                                   \
        }                                                                                                           \
        break;
            PSIG_CASE(1) PSIG_CASE(2) PSIG_CASE(3) PSIG_CASE(4) PSIG_CASE(5) PSIG_CASE(6) PSIG_CASE(7) PSIG_CASE(8)
#undef PSIG_CASE
            default: break;
        }
    }
}

constexpr int64_t kChunkSteps = 16;  // increments of a chunk, at least

}  // namespace

// Chunks of sixteen increments and more, at most 64 and no more than fill the GPU, if the forward gains by them (a backward
// gains more).  In one piece an increment takes 0.010 us and 0.019 for every letter of the longest words, or what keeps the
// SIMDs busy; in chunks that latency is divided, but suffixes and the staging of all letters for blocks of one wave keep them
// busy for longer, the launches take 4.5 us more, the products 0.15 (depth 1) to 0.5 us (depth 8) a chunk, and the table is written and
// read (1 us a megabyte, of short paths more than they sweep).  (With 0.3 us an increment, staging and table left out, a
// forward lost in 23 of 240 random calls, now in one, by 3 us: fp32, 3 paths of 2436 points, 58 057 words of (38, 4), 174 / 515 us; fp64, 2 of 105, 31 029 words of
// (31, 4), 11 / 27.)  fp32 rows of more than 4096 increments keep to one piece, as those of the dense kernels keep to 64 chunks.
WordChunks word_chunks(size_t elem, int64_t B, int64_t L, int64_t d, int depth, const int64_t *level_sizes, bool windowed) {
    WordChunks wc{};
    if (windowed || !level_sizes || depth > 8 || B < 1 || L - 1 < 2 * kChunkSteps || (elem == 4 && L - 1 > 4096)) return wc;
    int longest = 0;
    int64_t waves = 0, longer = 0;
    double work = 0, factor_work = 0, staged_work = 0;  // us of a SIMD per increment, of one path
    for (int n = depth; n >= 1; --n) {
        const int64_t size = level_sizes[n], of_level = (size + kWave - 1) / kWave;
        if (size > (int64_t(1) << 24)) return wc;
        // (1 ns to an instruction, twice that in fp64)
        const double us = 1e-3 * (10.0 + 0.85 * n * (n + 1) + n) * ((double)elem / 4);
        if (longest == 0 && size > 0) longest = n;
        longer += size;
        waves += of_level;
        work += us * (double)of_level;
        factor_work += us * (double)((longer + kWave - 1) / kWave);
        staged_work += (0.8 * us + 0.3e-3 * (double)d * ((double)elem / 4)) * (double)((longer + kWave - 1) / kWave);
        wc.table_off[n] = wc.table_size;
        wc.edge_off[n] = wc.edge_size;
        wc.table_size += size * n * (n + 1) / 2;
        wc.edge_size += size * n;
    }
    if (waves == 0 || B * waves >= 8192) return WordChunks{};
    const bool lists = batch_backward_usable(elem, B, d, 1);
    if (lists && d > 16) return WordChunks{};
    const int64_t backward = lists ? list_waves(B, depth, level_sizes) : B * waves;
    int64_t c = (L - 1) / kChunkSteps;
    if (c > 64) c = 64;
    // (a product is made in the forward and again in the backward; an increment takes both sweeps 1.4 us)
    const double product_us = 0.1 + 0.05 * depth;
    c = std::min(c, (int64_t)std::sqrt(0.7 * (double)(L - 1) / product_us));
    // (so many that the SIMDs, 1024, have what an increment's latency leaves room for; reverse sweeps four to a SIMD)
    const double room = 0.3 * 1024 / ((double)B * factor_work);
    if ((double)c > 1.0 + room) c = (int64_t)(1.0 + room);
    if (c > 1 + 4096 / backward) c = 1 + 4096 / backward;
    // (a quarter of a gigabyte of factors, which a forward keeps for its backward; grids and rows of the lists below 2^16)
    if (c * B * wc.table_size * (int64_t)elem > (int64_t(1) << 28)) c = (int64_t(1) << 28) / (B * wc.table_size * (int64_t)elem);
    if (c * ((B + 15) / 16) > 65535) c = 65535 / ((B + 15) / 16);
    if (c < 2) return WordChunks{};
    const double steps = (double)(L - 1), simds = 1.0 / 1024, latency = 0.010 + 0.019 * longest;
    const double one_piece = 3.0 + steps * std::max(latency, (double)B * work * simds);
    const double in_chunks = 7.5 + product_us * (double)c + steps * std::max(latency / (double)c, (double)B * staged_work * simds) +
                             1e-6 * (double)c * (double)B * (double)wc.table_size * (double)elem;
    if (in_chunks > one_piece) return WordChunks{};
    wc.chunks = (int)c;
    return wc;
}

template <typename T>
hipError_t launch_word_factors(const T *path, T *table, const SigShape &shape, const LevelPlan &plan, const int64_t *codes,
                               const WordChunks &wc, hipStream_t stream) {
    FactorBlocks fb{};
    fb.depth = plan.depth;
    int64_t blocks = 0, longer = 0;  // longer: words of length m and more
    for (int m = plan.depth; m >= 1; --m) {
        longer += plan.size[m];
        fb.begin[m] = blocks;
        blocks += (longer + kWave - 1) / kWave;
    }
    const int64_t units = shape.B * wc.chunks;
    if (blocks == 0 || units == 0) return hipSuccess;
    if (blocks * units >= (int64_t(1) << 31)) return hipErrorInvalidValue;
    // whole pairs of increments, 8 KB at most (a pair of rows of letters takes more where there are a great many)
    int64_t tile = 8192 / (2 * shape.d * (int64_t)sizeof(T)) * 2;
    const int64_t longest = (shape.L - 1 + wc.chunks - 1) / wc.chunks;
    if (tile > longest) tile = (longest + 1) / 2 * 2;
    if (tile < 2) tile = 2;
    const size_t lds = (size_t)(tile * shape.d) * sizeof(T);
#define PSIG_LAUNCH(MAXDEG)                                                                                           \
    hipLaunchKernelGGL((word_factors_kernel<T, MAXDEG>), dim3((unsigned)(blocks * units)), dim3(kWave), lds, stream, path, \
                       table, shape, plan, codes, wc, fb, (unsigned)units, (int)tile)
    if (plan.depth <= 4) PSIG_LAUNCH(4);
    else if (plan.depth <= 6) PSIG_LAUNCH(6);
    else if (plan.depth <= 8) PSIG_LAUNCH(8);
    else return hipErrorInvalidValue;
#undef PSIG_LAUNCH
    return hipGetLastError();
}

template <typename T>
hipError_t launch_word_products(const T *table, T *sig, T *left, T *right, const SigShape &shape, const LevelPlan &plan_in,
                                const WordChunks &wc, hipStream_t stream) {
    LevelPlan plan = plan_in;
    int64_t blocks = 0;
    for (int n = 1; n <= plan.depth; ++n) {
        plan.block_begin[n] = blocks;
        blocks += (plan.size[n] + kWave - 1) / kWave;
    }
    plan.block_begin[plan.depth + 1] = blocks;
    if (blocks == 0 || shape.B == 0) return hipSuccess;
    const dim3 grid((unsigned)blocks, (unsigned)(shape.B < 65535 ? shape.B : 65535), right ? 2 : 1);
#define PSIG_LAUNCH(MAXDEG)                                                                                       \
    hipLaunchKernelGGL((word_products_kernel<T, MAXDEG>), grid, dim3(kWave), 0, stream, sig, table, left, right, plan, wc, \
                       shape.B)
    if (plan.depth <= 4) PSIG_LAUNCH(4);
    else if (plan.depth <= 6) PSIG_LAUNCH(6);
    else if (plan.depth <= 8) PSIG_LAUNCH(8);
    else return hipErrorInvalidValue;
#undef PSIG_LAUNCH
    return hipGetLastError();
}

#define PSIG_INSTANTIATE(T)                                                                                            \
    template hipError_t launch_word_factors<T>(const T *, T *, const SigShape &, const LevelPlan &, const int64_t *,   \
                                               const WordChunks &, hipStream_t);                                       \
    template hipError_t launch_word_products<T>(const T *, T *, T *, T *, const SigShape &, const LevelPlan &,         \
                                                const WordChunks &, hipStream_t);
PSIG_INSTANTIATE(float)
PSIG_INSTANTIATE(double)
#undef PSIG_INSTANTIATE

}  // namespace psig
