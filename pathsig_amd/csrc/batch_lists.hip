// Signature backward for word projections with lanes on paths, over at most sixteen letters.
//
// As in batch_kernels.hip a lane holds one path and sweeps a few words, which leaves it with one gradient per position
// of every word ("entry") and increment; an increment needs their sums per letter.  Added to LDS cells as they come, an
// entry is a read, an add and a store, each waiting for the one before (two entries may share a letter), and the cells
// of eight waves fill the LDS of a CU.  Here the entries of an increment are stored as they are, plainly and without
// waiting, [entry][path]; which of them belong to a letter does not change over time, so the block sorts its entries
// by letter once, into rows of at most kRowLen entries of one letter, and after every kTile increments its waves add
// up the rows: a lane takes four paths of a row, sixteen bytes of an entry at a time.  A letter that most words share
// takes more rows, so the time does not depend on the words.  The sums of the rows are stored in LDS, added up per
// letter and sent to memory by atomics in the order of the output, whole cache lines at a time (atomics from the lanes
// that add the rows, four paths and a few letters to an instruction, took a third of the kernel's time).
//
// 256 paths of 512 points, 16 letters, 2320 words up to length 6, fp32: 599 us against 959 us with the cells (fp64,
// forward and backward, 1631 against 2368 us).  Not bound by memory, nor by the vector ALU's own rate: four resident waves can issue a vector
// instruction every 0.9 ns.  Two barriers per two increments and blocks of unequal length (912 on 1024 places) add to the
// chains.  The same sums on the matrix cores (16x16x4 fp32, the entries times a matrix of zeros and ones) were built and
// are slower: fp32 matrix instructions take as long as the vector ALU would for sixteen letters and do not run beside it.
#include <type_traits>

#include "common.hpp"
#include "words_common.hpp"

namespace psig {

namespace {

constexpr int kGroup = 16;    // paths of a wave
constexpr int kSlots = 4;     // words side by side in a wave
constexpr int kWaves = 4;     // waves of a block: they share paths and increments, each with its own words
constexpr int kThreads = kWaves * kWave;
constexpr int kLetters = 16;  // at most
constexpr int kTile = 2;      // increments between barriers: two waves add up the rows of each
constexpr int kRows = 32;     // rows of entries: sixteen lanes' worth for two waves
// Staged increments: [pair][letter][path][increment of the pair].  In fp32 half a wave reads the pairs of two words at once,
// 32 LDS banks for each: they lie there twice, in the lower 32 banks for the even words of a wave and in the upper 32 for the
// odd ones, and the paths of a letter are rotated by the letter, so that the lanes that stage neighbouring letters store to
// different banks.  (Once, 34 elements apart, so that the parity of a letter chose its half of the banks, half the reads met in
// one: step of the example above 815 us, in both halves 796; LDS clocks lost to conflicts 78 -> 59 M of 216 -> 201 M, the rest of
// them where the rows of entries are read and stored.)  In fp64 a word's sixteen
// pairs fill the banks by themselves.
template <typename T>
struct Staged {
    static constexpr int kCopies = sizeof(T) == 4 ? 2 : 1;
    static constexpr int kStage = 8 / kCopies;  // increments staged at once: the same room for both types
    static constexpr int kLetterRow = kCopies == 2 ? 4 * kGroup : 2 * kGroup + 2;
    static constexpr int kPair = kLetters * kLetterRow;  // from one pair of staged increments to the next
    static_assert(kStage % kTile == 0 && kStage * kLetters % kWave == 0, "whole tiles and whole waves");
    // element of the pair of a letter and path that the words of parity `copy` read
    static __device__ __forceinline__ int at(int letter, int path, int copy) {
        return kCopies == 2 ? letter * kLetterRow + 2 * kGroup * copy + 2 * ((path + letter) % kGroup)
                            : letter * kLetterRow + 2 * path;
    }
};
static_assert(kTile == 2, "the increments of a tile are read as a pair");
static_assert(kTile * kRows * 4 == kThreads, "a thread per increment of the tile, row and four paths");

// Entries of a lane: with twelve, four blocks share a CU's LDS and the registers of four waves to a SIMD suffice
// (eighteen, three blocks: 4 % slower in the example above).
constexpr int kEntries = 12;
constexpr int kBlockEntries = kWaves * kSlots * kEntries;
// The rows suffice however the entries fall to the letters: a letter with n entries leaves at most kRowLen - 1 places
// of its last row unused.
constexpr int kRowLen = 12;
static_assert(kLetters * (kRowLen - 1) + kBlockEntries <= kRows * kRowLen && kRowLen % 4 == 0, "rows suffice");

// Words swept at once by one lane: about the same number of entries at every length
constexpr int list_words(int deg) { return kEntries / deg; }

template <typename T>
struct alignas(32) Increment {
    T entry[kWaves][kEntries][kWave];  // (lane: word of the four, path of the sixteen)
    T zero[kGroup];                            // what the unused places of a row add
};

template <typename T>
struct ListShared {
    Increment<T> inc[kTile];
    alignas(16) T steps[Staged<T>::kStage / 2][Staged<T>::kPair];
    alignas(16) uint32_t place[kRows][kRowLen];    // byte offsets of entries in an increment
    alignas(32) T sums[kTile][kRows][kGroup + 4];       // of the rows, for every path
    int count[kLetters], first_row[kLetters];
};

template <typename T, int DEG, typename ACC, bool CHUNKED>
__device__ __forceinline__ void list_backward_body(const T *__restrict__ path, const T *__restrict__ sig,
                                                   const T *__restrict__ grad_sig, ACC *__restrict__ grad_inc,
                                                   const SigShape &shape, const LevelPlan &plan,
                                                   const int64_t *__restrict__ codes, int64_t blk_in_level,
                                                   int64_t unit, ListShared<T> &sh, const WordChunks &wc) {
    constexpr int WPL = list_words(DEG);
    constexpr int kPaths = kGroup / kWaves;  // paths that a wave stages
    constexpr int kStage = Staged<T>::kStage, kPair = Staged<T>::kPair, kCopies = Staged<T>::kCopies;
    typedef T Pair __attribute__((ext_vector_type(2)));
    const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const int slot = lane / kGroup, pl = lane % kGroup;
    const int d = (int)shape.d;
    // (a unit is a window of a group of paths, or a time chunk of paths without windows)
    const int64_t per_group = CHUNKED ? wc.chunks : shape.W;
    const int64_t group = unit / per_group, part = unit - group * per_group;
    const int64_t w = CHUNKED ? 0 : part;
    const int64_t b0 = group * kGroup;
    const bool path_ok = b0 + pl < shape.B;
    const int64_t b = path_ok ? b0 + pl : shape.B - 1;
    WindowSpan span = window_span(shape, w);
    if constexpr (CHUNKED) span = chunk_of_span(span, wc.chunks, (int)part);
    const int64_t row = b * shape.W + w;
    const T *srow = sig + row * plan.sig_size;
    const T *grow = grad_sig + row * plan.sig_size;

    for (int i = tid; i < kRows * kRowLen; i += kThreads)
        (&sh.place[0][0])[i] = (uint32_t)(kBlockEntries * kGroup * sizeof(T));
    if (tid < kLetters) sh.count[tid] = 0;
    if (tid < kTile * kGroup) sh.inc[tid / kGroup].zero[tid % kGroup] = T(0);
    __syncthreads();

    // per word: offsets of the lane's increments, chain at the right end of the window, chain adjoint
    const bool kept_chain = DEG > 1 && !CHUNKED && !plan.from_saved[DEG] && plan.keep != nullptr && plan.keep_off[DEG] >= 0;
    const int64_t word0 = ((blk_in_level * kWaves + wave) * kSlots + slot) * WPL;
    int aoff[WPL][DEG], nth[WPL][DEG];
    T p[WPL][DEG + 1], h[WPL][DEG + 1];
#pragma unroll
    for (int i = 0; i < WPL; ++i) {
        const int64_t word_idx = word0 + i;
        const bool have = word_idx < plan.size[DEG];
        uint64_t code = 0;
        if (have) code = plan.code_off[DEG] >= 0 ? (uint64_t)codes[plan.code_off[DEG] + word_idx] : (uint64_t)word_idx;
        int l[DEG];
        decode_letters<DEG>(code, (uint64_t)d, l);
        p[i][0] = T(1);
#pragma unroll
        for (int k = 0; k < DEG; ++k) {
            aoff[i][k] = Staged<T>::at(l[k], pl, slot % kCopies);
            nth[i][k] = have && pl == 0 ? atomicAdd(&sh.count[l[k]], 1) : -1;
            p[i][k + 1] = T(0);
            h[i][k] = T(0);
        }
        h[i][DEG] = (have && path_ok) ? grow[plan.out_off[DEG] + word_idx] : T(0);
        if (CHUNKED) {
            if (have && path_ok) word_chunk_edges<T, DEG>(wc, plan, row * wc.chunks + part, word_idx, p[i], h[i]);
        } else if (plan.from_saved[DEG] && have) {
            uint64_t off = 0, width = (uint64_t)d, pref = 0;
#pragma unroll
            for (int k = 1; k < DEG; ++k) {
                pref = pref * (uint64_t)d + (uint64_t)l[k - 1];
                p[i][k] = srow[off + pref];
                off += width;
                width *= (uint64_t)d;
            }
        } else if (kept_chain && have && path_ok) {
            // the forward of this call kept the chain
            const T *kept = (const T *)plan.keep + row * plan.keep_size + plan.keep_off[DEG] + word_idx * (DEG - 1);
#pragma unroll
            for (int k = 1; k < DEG; ++k) p[i][k] = kept[k - 1];
        }
    }
    __syncthreads();
    if (tid < kLetters) {
        int at = 0;
        for (int a = 0; a < tid; ++a) at += (sh.count[a] + kRowLen - 1) / kRowLen;
        sh.first_row[tid] = at;
    }
    __syncthreads();
    if (pl == 0) {
#pragma unroll
        for (int i = 0; i < WPL; ++i)
#pragma unroll
            for (int k = 0; k < DEG; ++k)
                if (nth[i][k] >= 0) {
                    const int to = sh.first_row[aoff[i][k] / Staged<T>::kLetterRow] * kRowLen + nth[i][k];
                    (&sh.place[0][0])[to] =
                        (uint32_t)(((wave * kEntries + i * DEG + k) * kWave + slot * kGroup) * (int)sizeof(T));
                }
    }

    // Staging: the wave brings paths wave, wave + kWaves, .. and its lanes run along time and letters.  The points of
    // the next kStage increments are fetched into registers before the current ones are worked on and become
    // increments in LDS after them.  (kStage is larger than kTile because a wait for these loads is one for the atomics
    // issued before them too.)
    constexpr int kChunks = kStage * kLetters / kWave;
    T hi[kPaths][kChunks], lo[kPaths][kChunks];
    int stage_at[kChunks], stage_step[kChunks], stage_letter[kChunks];
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
        const int j = lane + c * kWave, st = j / d;
        stage_step[c] = st;
        stage_letter[c] = j - st * d;
        stage_at[c] = (st / 2) * kPair + st % 2;
    }
    auto fetch = [&](int64_t t0, int nt) {
#pragma unroll
        for (int pp = 0; pp < kPaths; ++pp) {
            const int64_t q = b0 + wave + pp * kWaves;
            const T *xq = path + ((q < shape.B ? q : 0) * shape.L + span.start + t0) * d;
#pragma unroll
            for (int c = 0; c < kChunks; ++c) {
                const int at = stage_step[c] < nt ? lane + c * kWave : 0;
                hi[pp][c] = xq[at + d];
                lo[pp][c] = xq[at];
            }
        }
    };
    T *steps = &sh.steps[0][0];
    auto commit = [&](int nt) {
#pragma unroll
        for (int c = 0; c < kChunks; ++c)
            if (stage_step[c] < nt)
#pragma unroll
                for (int pp = 0; pp < kPaths; ++pp) {
                    const T dx = b0 + wave + pp * kWaves < shape.B ? hi[pp][c] - lo[pp][c] : T(0);
#pragma unroll
                    for (int copy = 0; copy < kCopies; ++copy)
                        steps[stage_at[c] + Staged<T>::at(stage_letter[c], wave + pp * kWaves, copy)] = dx;
                }
    };
    const int64_t nstages = (span.steps + kStage - 1) / kStage;
    auto stage_steps = [&](int64_t si) {
        const int64_t left = span.steps - si * kStage;
        return (int)(left < kStage ? left : kStage);
    };

    if (!plan.from_saved[DEG] && DEG > 1 && nstages > 0 && !kept_chain && !CHUNKED) {
        // chain at the right end of the window by a forward sweep (levels < DEG)
        fetch(0, stage_steps(0));
        commit(stage_steps(0));
        for (int64_t si = 0; si < nstages; ++si) {
            const int nt = stage_steps(si);
            lds_barrier();
            if (si + 1 < nstages) fetch((si + 1) * kStage, stage_steps(si + 1));
            for (int tt = 0; tt < nt; ++tt) {
#pragma unroll
                for (int i = 0; i < WPL; ++i) {
                    T dl[DEG];
#pragma unroll
                    for (int k = 0; k < DEG; ++k) dl[k] = steps[aoff[i][k] + (tt / 2) * kPair + tt % 2];
                    chain_step<T, DEG, DEG - 1>(p[i], dl);
                }
            }
            lds_barrier();
            if (si + 1 < nstages) commit(stage_steps(si + 1));
        }
    }

    // the thread's part of the sums: increment, row, four paths
    const int sum_step = wave / (kWaves / kTile);
    const int sum_row = (wave % (kWaves / kTile)) * (kWave / 4) + lane / 4, quad = lane % 4;
    __syncthreads();
    // .. and its outputs: path out_path and the one half a group further on, an increment, a letter.  A path's 2 d
    // outputs of a tile lie together: the atomics of a wave fill the cache lines that they touch.
    constexpr int kHalf = kGroup / 2;
    const int letter = lane % kLetters, out_step = lane / kLetters % kTile;
    const int out_path = wave * (kHalf / kWaves) + lane / (kLetters * kTile);
    const int first_row = sh.first_row[letter], end_row = first_row + (sh.count[letter] + kRowLen - 1) / kRowLen;
    const int64_t per_path = (shape.L - 1) * d;
    ACC *out = grad_inc + (b0 + out_path) * per_path + (span.start + out_step) * d + letter;
    auto flush = [&](int64_t tile, int nt) {
        if (out_step >= nt) return;
        T v[2] = {T(0), T(0)};
        for (int r = first_row; r < end_row; ++r)
#pragma unroll
            for (int c = 0; c < 2; ++c) v[c] += sh.sums[out_step][r][out_path + c * kHalf];
#pragma unroll
        for (int c = 0; c < 2; ++c)
            if (b0 + out_path + c * kHalf < shape.B && v[c] != T(0))
                atomicAdd(out + tile * kTile * d + c * kHalf * per_path, (ACC)v[c]);
    };

    if (nstages > 0) {
        fetch((nstages - 1) * kStage, stage_steps(nstages - 1));
        commit(stage_steps(nstages - 1));
    }
    int64_t ti = (span.steps + kTile - 1) / kTile - 1;
    int pair = ti < 0 ? 0 : (int)(ti % (kStage / kTile));
    const T *at_pair = steps + pair * kPair;
    if (ti >= kStage / kTile) fetch((nstages - 2) * kStage, kStage);
    int last_nt = 0;
    for (; ti >= 0; --ti) {
        const int64_t left = span.steps - ti * kTile;
        const int nt = (int)(left < kTile ? left : kTile);
        lds_barrier();
        if (last_nt) flush(ti + 1, last_nt);  // of the tile before
        last_nt = nt;
        Pair both[WPL][DEG];
#pragma unroll
        for (int i = 0; i < WPL; ++i)
#pragma unroll
            for (int k = 0; k < DEG; ++k) both[i][k] = *reinterpret_cast<const Pair *>(at_pair + aoff[i][k]);
#pragma unroll
        for (int tt = kTile - 1; tt >= 0; --tt) {
            if (tt >= nt) continue;
            T *to = &sh.inc[tt].entry[wave][0][lane];
#pragma unroll
            for (int i = 0; i < WPL; ++i) {
                T dl[DEG], gl[DEG];
#pragma unroll
                for (int k = 0; k < DEG; ++k) dl[k] = both[i][k][tt];
                // S_t = S_{t+1} (x) exp(-dx_t) on the chain (levels < DEG are all the adjoint needs), and the adjoint
                chain_step_adjoint<T, DEG>(p[i], h[i], dl, gl);
#pragma unroll
                for (int k = 0; k < DEG; ++k) to[(i * DEG + k) * kWave] = gl[k];
            }
        }
        lds_barrier();
        if (pair > 0) {
            --pair;
            at_pair -= kPair;
        } else if (ti > 0) {
            // the increments before these: fetched while this stage was worked on
            commit(kStage);
            pair = kStage / kTile - 1;
            at_pair = steps + pair * kPair;
            if (ti > kStage / kTile) fetch((ti / (kStage / kTile) - 2) * kStage, kStage);
        }
        if (sum_step < nt) {
            typedef T V __attribute__((ext_vector_type(4)));
            V sum = {T(0), T(0), T(0), T(0)};
            const uint32_t *list = sh.place[sum_row];
            auto add_row = [&](auto stepc) {
                const unsigned char *from =
                    reinterpret_cast<const unsigned char *>(&sh.inc[decltype(stepc)::value]) + quad * 4 * sizeof(T);
#pragma unroll
                for (int j = 0; j < kRowLen; ++j) sum += *reinterpret_cast<const V *>(from + list[j]);
            };
            if (sum_step == 0)
                add_row(std::integral_constant<int, 0>{});
            else
                add_row(std::integral_constant<int, 1>{});
            *reinterpret_cast<V *>(&sh.sums[sum_step][sum_row][4 * quad]) = sum;
        }
    }
    lds_barrier();
    if (last_nt) flush(0, last_nt);
}

// level of block `blk`; the levels are laid out from the deepest down (block_begin[0]: all blocks)
__device__ __forceinline__ int level_of_block(const LevelPlan &plan, int64_t blk) {
    int deg = plan.depth;
    while (deg > 1 && blk >= plan.block_begin[deg - 1]) --deg;
    return deg;
}

// Consecutive blocks work on the same words of consecutive groups of paths: the blocks of the longest words, which
// take longest, start first and spread over the device.
template <typename T, int MAXDEG, typename ACC, bool CHUNKED>
__global__ void __launch_bounds__(kThreads, sizeof(T) == 8 || MAXDEG > 8 ? 2 : MAXDEG > 6 ? 3 : 4)
    list_backward_kernel(const T *__restrict__ path, const T *__restrict__ sig, const T *__restrict__ grad_sig,
                         ACC *__restrict__ grad_inc, SigShape shape, LevelPlan plan,
                         const int64_t *__restrict__ codes, WordChunks wc) {
    __shared__ ListShared<T> sh;
    const int64_t linear = (int64_t)blockIdx.y * gridDim.x + blockIdx.x;
    const int64_t blk = linear / gridDim.y, unit = linear - blk * gridDim.y;
    const int deg = level_of_block(plan, blk);
    const int64_t bl = blk - plan.block_begin[deg];
    switch (deg) {
#define PSIG_CASE(N)                                                                                               \
    case N:                                                                                                        \
        if constexpr (N <= MAXDEG)                                                                                 \
            list_backward_body<T, N, ACC, CHUNKED>(path, sig, grad_sig, grad_inc, shape, plan, codes, bl, unit, sh, wc);    \
        break;
        PSIG_CASE(1) PSIG_CASE(2) PSIG_CASE(3) PSIG_CASE(4) PSIG_CASE(5) PSIG_CASE(6)
        PSIG_CASE(7) PSIG_CASE(8) PSIG_CASE(9) PSIG_CASE(10) PSIG_CASE(11) PSIG_CASE(12)
#undef PSIG_CASE
        default: break;
    }
}

}  // namespace

template <typename T, typename ACC>
hipError_t launch_batch_lists(const T *path, const T *sig, const T *grad_sig, ACC *grad_inc, const SigShape &shape,
                              const LevelPlan &plan_in, const int64_t *codes, const WordChunks &wc, hipStream_t stream) {
    LevelPlan plan = plan_in;
    const int64_t units = (shape.B + kGroup - 1) / kGroup * (wc.chunks ? wc.chunks : shape.W);
    int64_t blocks = 0;
    for (int k = plan.depth; k >= 1; --k) {
        const int64_t per_block = (int64_t)kWaves * kSlots * list_words(k);
        plan.block_begin[k] = blocks;
        blocks += (plan.size[k] + per_block - 1) / per_block;
    }
    plan.block_begin[0] = blocks;
    if (blocks == 0 || units == 0) return hipSuccess;
    if (shape.d > kLetters || blocks >= (int64_t(1) << 31) || units > 65535) return hipErrorInvalidValue;
    const dim3 grid((unsigned)blocks, (unsigned)units);
#define PSIG_LAUNCH(MAXDEG)                                                                                         \
    if (wc.chunks)                                                                                                  \
        hipLaunchKernelGGL((list_backward_kernel<T, MAXDEG, ACC, true>), grid, dim3(kThreads), 0, stream, path, sig, \
                           grad_sig, grad_inc, shape, plan, codes, wc);                                             \
    else                                                                                                            \
        hipLaunchKernelGGL((list_backward_kernel<T, MAXDEG, ACC, false>), grid, dim3(kThreads), 0, stream, path, sig, \
                           grad_sig, grad_inc, shape, plan, codes, wc)
    if (plan.depth <= 4)
        PSIG_LAUNCH(4);
    else if (plan.depth <= 6)
        PSIG_LAUNCH(6);
    else if (plan.depth <= 8)
        PSIG_LAUNCH(8);
    else
        PSIG_LAUNCH(12);
#undef PSIG_LAUNCH
    return hipGetLastError();
}

#define PSIG_INSTANCE(T, ACC)                                                                                     \
    template hipError_t launch_batch_lists<T, ACC>(const T *, const T *, const T *, ACC *, const SigShape &,      \
                                                   const LevelPlan &, const int64_t *, const WordChunks &, hipStream_t);
PSIG_INSTANCE(float, float)
PSIG_INSTANCE(float, double)
PSIG_INSTANCE(double, double)
#undef PSIG_INSTANCE

int64_t list_waves(int64_t B, int depth, const int64_t *level_sizes) {
    int64_t blocks = 0;
    for (int k = 1; k <= depth; ++k) {
        const int64_t per_block = (int64_t)kWaves * kSlots * list_words(k);
        blocks += (level_sizes[k] + per_block - 1) / per_block;
    }
    return blocks * kWaves * ((B + kGroup - 1) / kGroup);
}

}  // namespace psig
