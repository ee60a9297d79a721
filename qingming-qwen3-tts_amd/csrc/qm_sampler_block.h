// qm_sampler_block.h — the top-k categorical sampler (and arg-max) as the work of one block, shared by the
// sampler's own kernel and the predictor's frame kernel.
//
// Reference: gpu_sample_topk_f32_kernel / gpu_sample_topk_bf16_kernel (R17:7407-7518) and the final-head score
// processing in front of it (R17:14025-14143).
//
// What fixes the result.  The reference sorts all scores by (score descending, id ascending)
// with a 4 096-wide sorting network in LDS; that order is total (no two entries compare equal),
// so the first `keep` entries of the sorted sequence are a property of the scores, not of the
// sorting algorithm.  Thread 0 then sums exp(score / T - maximum) over them in double, in that
// order, draws one SplitMix64 number and walks the running sum.  Here the first `keep` entries
// are found without sorting the rest: every score becomes a key (order-preserving image
// of the float above, inverted id below); a bound that at least `keep` keys reach is found by a radix select
// (histogram passes of 12 bits, sixteen bins per thread, ended as soon as few enough keys lie at or above it to be
// ranked), those keys are gathered and ranked by counting, several threads to a key where there are threads for it, and
// the first `keep` ranks are the sequence.  The select looks at each thread's largest key first: the keep-th largest of
// those is such a bound, with an eighth of the additions to LDS; only where it would let too many keys through (`keep` beyond half of the
// threads) or does (one thread holding many of the largest) are all keys looked at, in passes of 8 bits.  The exponentials are computed by
// `keep` threads at once; the sums are added in the reference's order: the running sum of the second loop repeats the partial sums of the first, so one pass
// gives both.
// Bound: a chain of LDS exchanges.  Cycles for 50 of 2048 16-bit scores: 14 400 with 64-bit keys, 8-bit digits of all keys until the bin is
// wanted whole, a thread per key and the sums of one thread through LDS; 9 900 as it stands.  (us a draw of many in a row, 200 of 2048: 16-bit scores
// 14.5 so at first, 13.0 from the largest keys and then from all, 11.5 from all at once; 32-bit ones 11.5, 14.4 and 11.7.)
// One block of 256 threads; vocab <= 4096 (the reference's sort size), top_k <= 256.
#pragma once

#include "qm_device.h"

namespace qm {

constexpr int kSmpThreads = 256;
constexpr int kSmpMaxVocab = 4096;                       // kGpuSamplerSortSize, R17:7336
constexpr int kSmpPerThread = kSmpMaxVocab / kSmpThreads;
constexpr int kSmpMaxKeep = 256;
constexpr int kSmpBins = 4096;                           // of a histogram pass: 16-bit counters, two to a word
constexpr int kSmpWords = kSmpBins / 2 / kSmpThreads;    // counter words of a thread
// Most entries that the select finds from each thread's largest key.  Of random scores the keep-th largest of 256 maxima lets through about
// -256 ln(1 - keep / 256) keys, 177 for 128 and more than can be ranked from 160 on: its passes would be for nothing.
constexpr int kSmpFromLargest = 128;

struct SamplerParams {
    const void* logits;          // float or bf16 bits
    int is_bf16;
    int offset;                  // first element (last_row_offset of the bf16 kernel)
    int vocab;
    int top_k;                   // <= 0: arg-max
    float temperature;
    unsigned long long* rng_state;
    int32_t* output_id;
    // final-head processing in front of the selection (process != 0; logits are bf16)
    int process;
    int32_t* history;            // read [0, history_count); the code is appended at [append_index] if >= 0
    int history_count;
    int append_index;
    int generation_index;
    int eos;
    int suppressed_tail;
    float penalty;
    float reciprocal;            // float(1) / float(penalty)
    float* scores_out;           // processed scores, or NULL
    int process_only;            // stop after writing scores_out
};

// Order-preserving image of a float: a > b  <=>  image(a) > image(b)  (-0 counted as +0).
__device__ __forceinline__ uint32_t ordered_bits(float v) {
    const uint32_t bits = __float_as_uint(v + 0.0f);
    return (bits & 0x80000000U) ? ~bits : (bits | 0x80000000U);
}
__device__ __forceinline__ float from_ordered_bits(uint32_t image) {
    return __uint_as_float((image & 0x80000000U) ? (image & 0x7fffffffU) : ~image);
}

__device__ __forceinline__ unsigned long long splitmix64_next(unsigned long long* state) {
    unsigned long long z = *state + 0x9e3779b97f4a7c15ULL;
    *state = z;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    return z ^ (z >> 31);
}

// Inclusive prefix sum over the 64 lanes of a wave: four DPP row shifts inside the 16-lane rows, then the
// three row totals (no LDS traffic; a shuffle-based scan costs an LDS round trip per step).
__device__ __forceinline__ int wave_inclusive_scan(int v, int lane) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
    const int t0 = __builtin_amdgcn_readlane(v, 15);
    const int t1 = __builtin_amdgcn_readlane(v, 31);
    const int t2 = __builtin_amdgcn_readlane(v, 47);
    if (lane >= 16) v += t0;
    if (lane >= 32) v += t1;
    if (lane >= 48) v += t2;
    return v;
}

// A score and its id as one number: larger key = earlier in the order; 0 is below every key.  kPasses radix digits of 12 bits (`mask(p)`)
// from bit `shift(p)` on cover the significant bits, or kBytePasses of 8 (`byte_mask(p)`, `byte_shift(p)`); those that no pass looks at (kFree)
// are set in every key.
template <bool NARROW>
struct SamplerKey;
template <>
struct SamplerKey<false> {                               // any score: 32 bits of it, and of the inverted id the low 12 (ids < 4096)
    using type = unsigned long long;
    static constexpr int kPasses = 4;
    static constexpr type kFree = 0xfffff000ULL;
    static __device__ __forceinline__ int shift(int p) { return p == 0 ? 52 : p == 1 ? 40 : p == 2 ? 32 : 0; }
    static __device__ __forceinline__ unsigned mask(int p) { return p == 2 ? 0xffU : 0xfffU; }
    static constexpr int kBytePasses = 6;
    static __device__ __forceinline__ int byte_shift(int p) { return p < 4 ? 56 - 8 * p : p == 4 ? 4 : 0; }
    static __device__ __forceinline__ unsigned byte_mask(int p) { return p == 5 ? 0xfU : 0xffU; }
    static __device__ __forceinline__ type make(float v, int id) {
        return (static_cast<type>(ordered_bits(v)) << 32) | (0xffffffffU - static_cast<uint32_t>(id));
    }
    static __device__ __forceinline__ float score(type k) { return from_ordered_bits(static_cast<uint32_t>(k >> 32)); }
    static __device__ __forceinline__ int32_t id(type k) { return static_cast<int32_t>(0xffffffffU - static_cast<uint32_t>(k)); }
};
template <>
struct SamplerKey<true> {                                // scores that are bf16 values: the other half of their image says nothing
    using type = uint32_t;
    static constexpr int kPasses = 3;
    static constexpr type kFree = 0xf000U;
    static __device__ __forceinline__ int shift(int p) { return p == 0 ? 20 : p == 1 ? 16 : 0; }
    static __device__ __forceinline__ unsigned mask(int p) { return p == 1 ? 0xfU : 0xfffU; }
    static constexpr int kBytePasses = 4;
    static __device__ __forceinline__ int byte_shift(int p) { return p == 0 ? 24 : p == 1 ? 16 : p == 2 ? 4 : 0; }
    static __device__ __forceinline__ unsigned byte_mask(int p) { return p == 3 ? 0xfU : 0xffU; }
    static __device__ __forceinline__ type make(float v, int id) {
        return (ordered_bits(v) & 0xffff0000U) | (0xffffU - static_cast<uint32_t>(id));
    }
    static __device__ __forceinline__ float score(type k) {
        return from_ordered_bits((k & 0xffff0000U) | ((k & 0x80000000U) ? 0U : 0xffffU));
    }
    static __device__ __forceinline__ int32_t id(type k) { return static_cast<int32_t>(0xffffU - (k & 0xffffU)); }
};

// The block's scratch memory (LDS): 14.6 KiB.
struct SamplerScratch {
    uint32_t seen[kSmpMaxVocab / 32];                    // tokens present in the history
    __attribute__((aligned(16))) uint32_t hist[kSmpBins / 2];    // bin 2 w in the low half of word w, or bin b in words 8 b ..; later the parts of the ranks
    int wave_total[4], wave_first[4];
    int digit, remaining, count;
    __attribute__((aligned(16))) unsigned long long cand[kSmpMaxKeep];
    unsigned long long sorted[kSmpMaxKeep];
    __attribute__((aligned(16))) double exp_terms[kSmpMaxKeep];  // the terms, then their running sums
    double target;
};

// The selection by one block of kSmpThreads threads, all of which call it: score[j] is the score of id
// tid + 256 j (ids beyond the vocabulary are ignored), rng the generator's state (read and advanced by thread 0
// only, when a draw happens).  Returns the chosen id in thread 0 (anything in the others), or -2 in every
// thread when prm.process_only stops after the processed scores.  Nothing is read from prm.logits or
// prm.rng_state and nothing written to prm.output_id / prm.history / prm.rng_state: that is the caller's.
// `sync` is the barrier of the kSmpThreads calling threads (the block's barrier where they are the whole block).
// NARROW: every score is a bf16 value and prm.process is 0.  COMPACT: all keys go through the passes of the largest ones instead of their own, for a
// kernel that has other uses for its registers (the second loop made the predictor's frame 1.7 % longer, 1132 -> 1151 us, with 50 entries).
template <bool NARROW, bool COMPACT, class Sync>
__device__ __forceinline__ int32_t sampler_block(const SamplerParams& prm, SamplerScratch& sh, const float (&score)[kSmpPerThread],
                                                 unsigned long long& rng, Sync&& sync) {
    using Key = SamplerKey<NARROW>;
    using key_t = typename Key::type;
    uint32_t* const sh_seen = sh.seen;
    uint32_t* const sh_hist = sh.hist;
    int* const sh_wave_total = sh.wave_total;
    int* const sh_wave_first = sh.wave_first;
    int& sh_digit = sh.digit;
    int& sh_remaining = sh.remaining;
    int& sh_count = sh.count;
    key_t* const sh_cand = reinterpret_cast<key_t*>(sh.cand);
    key_t* const sh_sorted = reinterpret_cast<key_t*>(sh.sorted);
    double* const sh_exp = sh.exp_terms;
    double& sh_target = sh.target;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int vocab = prm.vocab;
    uint4* const own_words = reinterpret_cast<uint4*>(sh_hist + tid * kSmpWords);    // (a thread only ever reads and clears its own bins)
    static_assert(kSmpWords == 8, "two 16-byte pieces");
    own_words[0] = own_words[1] = make_uint4(0, 0, 0, 0);

    // ---- which tokens were generated before (R17:14046-14052, as a bitmap) -----------------------------
    if (prm.process) {
        for (int i = tid; i < kSmpMaxVocab / 32; i += kSmpThreads) sh_seen[i] = 0;
        sync();
        for (int i = tid; i < prm.history_count; i += kSmpThreads) {
            const int token = prm.history[i];
            if (token >= 0 && token < vocab) atomicOr(&sh_seen[token >> 5], 1U << (token & 31));
        }
        sync();
    }

    // ---- the scores as keys: larger key = earlier in the order -------------------------------------------
    key_t key[kSmpPerThread];
#pragma unroll
    for (int j = 0; j < kSmpPerThread; ++j) {
        const int id = tid + kSmpThreads * j;
        key[j] = 0;                                        // below every real key
        if (id < vocab) {
            float value = score[j];
            if (prm.process) {
                if ((sh_seen[id >> 5] >> (id & 31)) & 1U) value = value < 0.0f ? value * prm.penalty : value * prm.reciprocal;
                if (id == prm.eos && prm.generation_index < 2) value = -INFINITY;
                if (id >= vocab - prm.suppressed_tail && id != prm.eos) value = -INFINITY;
                if (prm.scores_out) prm.scores_out[id] = value;
            }
            key[j] = Key::make(value, id);
        }
    }

    if (prm.process_only) return -2;
    const int keep = prm.top_k <= 0 ? 1 : min(prm.top_k, vocab);

    // ---- a bound that `keep` keys or some more reach: the keep-th largest of the threads' largest keys, or of all keys, as far as
    // its digits have been looked at, most significant first.  Equal scores are told apart by their ids when they are ranked, not in
    // passes over bits that they share.  (Half a block's threads rank 128 keys in less time than a pass takes.) ----
    const int rankable = keep <= 64 ? 128 : kSmpMaxKeep;
    key_t largest = 0;
#pragma unroll
    for (int j = 0; j < kSmpPerThread; ++j) largest = key[j] > largest ? key[j] : largest;
    key_t prefix = 0, prefix_mask = 0, threshold = 0;
    int remaining = keep, candidates = kSmpMaxVocab + 1, place = 0;
    bool all_keys = keep > kSmpFromLargest;
    // (kept as a loop: unrolled, the compiler computes the digits of all passes ahead and runs out of registers)
#pragma unroll 1
    for (int pass = COMPACT || !all_keys ? 0 : Key::kPasses; (COMPACT || pass < Key::kPasses) && candidates > rankable; ++pass) {
        const int shift = Key::shift(pass);
        const unsigned digit_mask = Key::mask(pass);
        sync();                                   // the bins are clear (and, later, the last pass's results read)
        auto count = [&](key_t k) __attribute__((always_inline)) {
            if (k != 0 && (k & prefix_mask) == prefix) {
                const unsigned digit = static_cast<unsigned>(k >> shift) & digit_mask;
                atomicAdd(&sh_hist[digit >> 1], 1U << (16 * (digit & 1U)));          // (at most 4096 in a counter)
            }
        };
        if (COMPACT && all_keys) {
#pragma unroll
            for (int j = 0; j < kSmpPerThread; ++j) count(key[j]);
        } else {
            count(largest);
        }
        sync();
        // keys in bins above this thread's sixteen: inside the wave from a prefix sum, then the waves above
        const uint4 low = own_words[0], high = own_words[1];
        own_words[0] = own_words[1] = make_uint4(0, 0, 0, 0);
        const uint32_t high_pairs = (high.x + high.y) + (high.z + high.w);
        const uint32_t all_pairs = (low.x + low.y) + (low.z + low.w) + high_pairs;
        auto both = [](uint32_t pair) { return static_cast<int>((pair & 0xffffU) + (pair >> 16)); };
        const int own = both(all_pairs);
        const int upto = wave_inclusive_scan(own, lane);
        const int wave_sum = __builtin_amdgcn_readlane(upto, 63);
        if (lane == 0) sh_wave_total[wave] = wave_sum;
        sync();
        int above = wave_sum - upto;
#pragma unroll
        for (int w = 1; w < 4; ++w) above += w > wave ? sh_wave_total[w] : 0;
        if (above < remaining && remaining <= above + own) {       // exactly one thread; its bins by halves, from the top
            int rest = remaining - above, digit = 16 * tid;
            bool upper = rest <= both(high_pairs);
            if (!upper) rest -= both(high_pairs);
            digit += upper ? 8 : 0;
            const uint32_t w0 = upper ? high.x : low.x, w1 = upper ? high.y : low.y, w2 = upper ? high.z : low.z, w3 = upper ? high.w : low.w;
            upper = rest <= both(w2 + w3);
            if (!upper) rest -= both(w2 + w3);
            digit += upper ? 4 : 0;
            const uint32_t v0 = upper ? w2 : w0, v1 = upper ? w3 : w1;
            upper = rest <= both(v1);
            if (!upper) rest -= both(v1);
            digit += upper ? 2 : 0;
            const uint32_t word = upper ? v1 : v0;
            upper = rest <= static_cast<int>(word >> 16);
            if (!upper) rest -= static_cast<int>(word >> 16);
            digit += upper ? 1 : 0;
            sh_digit = digit;
            sh_remaining = rest;
        }
        sync();
        prefix |= static_cast<key_t>(sh_digit) << shift;
        prefix_mask |= static_cast<key_t>(digit_mask) << shift;
        remaining = sh_remaining;
        // the bound starts with the digits in `prefix`; those not looked at are free (zero here)
        threshold = prefix | Key::kFree;
        // how many keys reach it, and where this thread's go (a prefix sum over the block: no counter to queue at)
        int mine = 0;
#pragma unroll
        for (int j = 0; j < kSmpPerThread; ++j) mine += key[j] >= threshold ? 1 : 0;
        const int upto_mine = wave_inclusive_scan(mine, lane);
        if (lane == 63) sh_wave_first[wave] = upto_mine;
        sync();
        place = upto_mine - mine;
        candidates = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            place += w < wave ? sh_wave_first[w] : 0;
            candidates += sh_wave_first[w];
        }
        // (the largest keys have told all they can, and too many keys reach the bound: from all of them; the last pass of that tells all
        // keys apart and leaves `keep`)
        if (COMPACT && !all_keys && pass + 1 == Key::kPasses && candidates > rankable) {
            all_keys = true;
            pass = -1;
            prefix = prefix_mask = 0;
            remaining = keep;
        }
    }
    // From all keys: a bin to a thread, and eight counters to a bin, since scores share their leading bits and additions to one word take turns.
    // (The last pass tells all keys apart and leaves `keep`.)
    if (!COMPACT && __builtin_expect(candidates > rankable, false)) {
        prefix = prefix_mask = 0;
        remaining = keep;
#pragma unroll 1
        for (int pass = 0; candidates > rankable; ++pass) {
            const int shift = Key::byte_shift(pass);
            const unsigned digit_mask = Key::byte_mask(pass);
            sync();
#pragma unroll
            for (int j = 0; j < kSmpPerThread; ++j)
                if (key[j] != 0 && (key[j] & prefix_mask) == prefix)
                    atomicAdd(&sh_hist[(static_cast<unsigned>(key[j] >> shift) & digit_mask) * kSmpWords + (lane & (kSmpWords - 1))], 1U);
            sync();
            const uint4 low = own_words[0], high = own_words[1];
            own_words[0] = own_words[1] = make_uint4(0, 0, 0, 0);
            const int own = static_cast<int>(((low.x + low.y) + (low.z + low.w)) + ((high.x + high.y) + (high.z + high.w)));
            const int upto = wave_inclusive_scan(own, lane);
            const int wave_sum = __builtin_amdgcn_readlane(upto, 63);
            if (lane == 0) sh_wave_total[wave] = wave_sum;
            sync();
            int above = wave_sum - upto;
            for (int w = wave + 1; w < 4; ++w) above += sh_wave_total[w];
            if (above < remaining && remaining <= above + own) {
                sh_digit = tid;
                sh_remaining = remaining - above;
                sh_count = keep - (remaining - above) + own;       // so many reach the bin
            }
            sync();
            prefix |= static_cast<key_t>(sh_digit) << shift;
            prefix_mask |= static_cast<key_t>(digit_mask) << shift;
            remaining = sh_remaining;
            candidates = sh_count;
        }
        threshold = prefix | Key::kFree;
        int mine = 0;
#pragma unroll
        for (int j = 0; j < kSmpPerThread; ++j) mine += key[j] >= threshold ? 1 : 0;
        const int upto = wave_inclusive_scan(mine, lane);
        if (lane == 63) sh_wave_first[wave] = upto;
        sync();
        place = upto - mine;
        for (int w = 0; w < wave; ++w) place += sh_wave_first[w];
    }

    // ---- gather the keys that reach the bound, rank them by counting ----------------------------------------
#pragma unroll
    for (int j = 0; j < kSmpPerThread; ++j)
        if (key[j] >= threshold) sh_cand[place++] = key[j];
    if (tid >= candidates && tid < ((candidates + 7) & ~7)) sh_cand[tid] = 0;          // (padding of the last batch below)
    sync();
    {
        // `sharers` threads to a key, in different waves, each against every sharers-th batch of eight
        const int sharers = candidates <= 64 ? 4 : candidates <= 128 ? 2 : 1;
        const int keys = kSmpThreads / sharers;
        const int part = __builtin_amdgcn_readfirstlane(tid / keys);
        const key_t mine = sh_cand[tid & (keys - 1)];
        int rank = 0;
        for (int j = 8 * part; j < candidates; j += 8 * sharers) {
            typedef key_t batch_t __attribute__((ext_vector_type(16 / sizeof(key_t))));
            constexpr int kPieces = 8 * sizeof(key_t) / 16;
            batch_t batch[kPieces];
#pragma unroll
            for (int u = 0; u < kPieces; ++u) batch[u] = *reinterpret_cast<const batch_t*>(sh_cand + j + u * (16 / sizeof(key_t)));
#pragma unroll
            for (int u = 0; u < kPieces; ++u)
#pragma unroll
                for (int e = 0; e < static_cast<int>(16 / sizeof(key_t)); ++e) rank += batch[u][e] > mine ? 1 : 0;
        }
        sh_hist[tid] = static_cast<uint32_t>(rank);
        sync();
        if (tid < candidates) {                            // (candidates <= keys: the first part's thread)
            const uint32_t other1 = sh_hist[(tid + keys) & (kSmpThreads - 1)], other2 = sh_hist[(tid + 2 * keys) & (kSmpThreads - 1)],
                           other3 = sh_hist[(tid + 3 * keys) & (kSmpThreads - 1)];
            if (sharers >= 2) rank += static_cast<int>(other1);
            if (sharers == 4) rank += static_cast<int>(other2 + other3);
            if (rank < keep) sh_sorted[rank] = mine;
        }
    }
    sync();

    // ---- sample (R17:7431-7460) ----------------------------------------------------------------------------
    const double inv_t = 1.0 / static_cast<double>(prm.temperature);
    auto id_of = [&](int i) { return Key::id(sh_sorted[i]); };
    if (prm.top_k > 0 && keep <= 64) {
        // One wave has a lane for every term.  Lane i's running sum is that of terms 0 .. i in their order (the terms behind its own
        // come as + 0, and a sum of exponentials is not -0); every lane reads all terms, the next eight on their way.
        if (wave != 0) return 0;
        const double maximum = static_cast<double>(Key::score(sh_sorted[0])) * inv_t;
        const double value = static_cast<double>(Key::score(sh_sorted[min(lane, keep - 1)]));
        sh_exp[lane] = exp(value * inv_t - maximum);       // (terms past `keep` reach lanes past `keep` only)
        typedef double f64x2_t __attribute__((ext_vector_type(2)));
        const f64x2_t* terms = reinterpret_cast<const f64x2_t*>(sh_exp);
        f64x2_t next[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) next[u] = terms[u];
        double running = 0.0;
#pragma unroll 1
        for (int i0 = 0; i0 < keep; i0 += 8) {
            f64x2_t term[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) term[u] = next[u];
#pragma unroll
            for (int u = 0; u < 4; ++u) next[u] = terms[(min(i0 + 8, 56)) / 2 + u];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                running += lane >= i0 + 2 * u ? term[u].x : 0.0;
                running += lane >= i0 + 2 * u + 1 ? term[u].y : 0.0;
            }
        }
        const unsigned long long all = __builtin_bit_cast(unsigned long long, running);
        const double total = __builtin_bit_cast(double, static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(all), keep - 1))
            | static_cast<unsigned long long>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(all >> 32), keep - 1))) << 32);
        if (!(total > 0.0)) return id_of(0);               // no draw
        double target = 0.0;
        if (tid == 0) target = static_cast<double>(splitmix64_next(&rng) >> 11) * (1.0 / 9007199254740992.0) * total;
        const unsigned long long wanted = __builtin_bit_cast(unsigned long long, target);
        target = __builtin_bit_cast(double, static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(wanted)))
            | static_cast<unsigned long long>(static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(wanted >> 32)))) << 32);
        const unsigned long long lanes = __builtin_amdgcn_ballot_w64(lane < keep && target < running);
        return id_of(lanes ? __builtin_ctzll(lanes) : keep - 1);
    }
    if (prm.top_k > 0 && tid < keep) {
        const double maximum = static_cast<double>(Key::score(sh_sorted[0])) * inv_t;
        const double value = static_cast<double>(Key::score(sh_sorted[tid]));
        sh_exp[tid] = exp(value * inv_t - maximum);
    } else if (tid < ((keep + 15) & ~15)) {
        sh_exp[tid] = 0.0;                                 // (padding of the last batch of sixteen below: x + 0 is x)
    }
    sync();
    // The running sums, added by one thread in the reference's order (its second loop repeats
    // the partial sums of its first: one pass serves both); the terms come sixteen at a time, the next
    // sixteen already on their way, so that the chain waits for additions, not for LDS.
    if (prm.top_k > 0 && tid == 0) {
        typedef double f64x2_t __attribute__((ext_vector_type(2)));
        const f64x2_t* terms = reinterpret_cast<const f64x2_t*>(sh_exp);
        f64x2_t* sums = reinterpret_cast<f64x2_t*>(sh_exp);
        double running = 0.0;
        f64x2_t next[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) next[u] = terms[u];
        for (int i0 = 0; i0 < keep; i0 += 16) {
            f64x2_t term[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) term[u] = next[u];
            if (i0 + 16 < keep) {
#pragma unroll
                for (int u = 0; u < 8; ++u) next[u] = terms[(i0 + 16) / 2 + u];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                running += term[u].x;
                term[u].x = running;
                running += term[u].y;
                term[u].y = running;
                sums[i0 / 2 + u] = term[u];
            }
        }
        const double total = running;
        sh_count = -1;                                     // no draw
        if (total > 0.0) {
            const double uniform = static_cast<double>(splitmix64_next(&rng) >> 11) * (1.0 / 9007199254740992.0);
            sh_target = uniform * total;
            sh_count = keep - 1;                           // the answer if no running sum exceeds the target
        }
    }
    sync();
    // first index whose running sum exceeds the target: the lowest such lane of each wave, then the lowest wave
    {
        const bool beyond = prm.top_k > 0 && sh_count >= 0 && tid < keep && sh_target < sh_exp[tid];
        const unsigned long long lanes = __builtin_amdgcn_ballot_w64(beyond);
        if (lane == 0) sh_wave_first[wave] = lanes ? 64 * wave + __builtin_ctzll(lanes) : 0x7fffffff;
    }
    sync();
    int32_t chosen = id_of(0);
    if (tid == 0 && prm.top_k > 0 && sh_count >= 0) {
        const int first = min(min(sh_wave_first[0], sh_wave_first[1]), min(sh_wave_first[2], sh_wave_first[3]));
        chosen = id_of(min(first, sh_count));              // sh_count = keep - 1: the answer if no sum exceeds the target
    }
    return chosen;
}

struct WholeBlockBarrier {
    __device__ __forceinline__ void operator()() const { __syncthreads(); }
};
template <bool NARROW, bool COMPACT = false>
__device__ __forceinline__ int32_t sampler_block(const SamplerParams& prm, SamplerScratch& sh, const float (&score)[kSmpPerThread],
                                                 unsigned long long& rng) {
    return sampler_block<NARROW, COMPACT>(prm, sh, score, rng, WholeBlockBarrier());
}

}  // namespace qm
