// qm_decoder_attention_mfma.hip — the chunked attention of a prompt's rows on the bf16 matrix cores (gfx950).
//
// A block of four or eight waves takes 32 query rows of one key/value head (a query row is a position and one of the head's
// query heads: they share keys and values); the waves take turns at the tiles of 32 keys that any of them sees and combine
// at the end.  A wave's keys and values are its own: it brings them straight into its part of the LDS
// (buffer_load ... lds, a tile of keys and a tile of values) and asks for the next keys when the products with these have read
// them, for the next values likewise, so that nothing waits for another wave and either is under way during the other's
// product; two blocks of four waves share a CU (not of 256 channels, 129 KiB).  Blocks of one key/value head share a die's L2 (block numbers go round the dies).
//
// Scores are S^T = K Q^T (v_mfma_f32_32x32x16_bf16): a lane then holds sixteen keys of one query, the softmax is in the lane
// but for one exchange with the other half of the wave, and the weights stand where the second product O^T = V^T P^T wants
// its operand, if it takes the keys of a block in the order the scores left them.  Scores and weights are fp32; the second
// product takes a weight as the sum of two bf16 numbers (its rounding and the rounding of what is left: 16 bits).  Values
// are transposed on their way out of LDS (ds_read_b64_tr_b16).  Bound: the chain of a tile in its wave (two products, the
// softmax between them); flops 2 (dim + vdim) per visible key and query (the second product's doubled weights not counted).
// (us, by blocks of eight waves that staged 128 keys for 64 rows through registers, values transposed on the way in, two barriers a
// tile / so, one shape again and again behind its rotation: 8 heads of 192 and 128 channels, 777 rows 25.8 / 13.1; 16 query heads on 8 of 128, 1024
// rows 28.0 / 15.4, of 64, 1000 rows 18.8 / 10.5; 32 heads of 128, 1500 rows 74 / 44; 4 on 2 of 250, 200 rows 32 / 14.  In a prompt of several layers the
// first two take 14.0 and 16.6.)
#include <algorithm>
#include <utility>

#include "../qm_host.h"
#include "qm_decoder_device.h"

namespace qm {

typedef float dec_f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t dec_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t dec_u32x2 __attribute__((ext_vector_type(2)));

constexpr int kFlashKeys = 32;                 // keys per tile of a wave
constexpr int kFlashRows = 32;                 // query rows per block
constexpr int kFlashHigh = 65535;              // blocks of a key/value head in one layer of the grid
constexpr int64_t kFlashMostRows = int64_t{64} * kFlashHigh;    // query rows of a key/value head (two layers)
constexpr float kFlashSlack = 8.0f;            // (powers of two)

// A tile in LDS: rows of CHANNELS bf16, in 16-byte pieces; piece c of row r stands in slot c ^ key(r).
// KEYS: the sixteen rows whose piece c a fragment read takes in a cycle stand in different banks; else the four rows of a
// transposing read do (it takes two pieces of each).
template <int CHANNELS, bool KEYS>
struct FlashTile {
    static constexpr int kPieces = CHANNELS / 8, kRowBytes = CHANNELS * 2, kBytes = kFlashKeys * kRowBytes;
    static constexpr int kRequests = kBytes / 1024;                            // instructions of a wave
    static constexpr int kPeriod = kPieces % 16 == 0 ? 1 : kPieces % 8 == 0 ? 2 : 4;    // rows to 256 bytes' multiple
    static constexpr int kSwap = KEYS ? 16 / kPeriod : 1;                      // (keys) pieces that change places with one another
    static __device__ __forceinline__ int key(int row) {
        if (KEYS) return row / kPeriod & (kSwap - 1);
        return kPeriod == 1 ? 4 * (row & 3) : kPeriod == 2 ? 4 * (row >> 1 & 1) : 0;
    }
    // instructions after which a lane's row has the same key: their offsets differ by rows only
    static constexpr int kOffsets = kRequests > kPieces / 4 ? kPieces / 4 : kRequests;
    static constexpr int kOffsetRows = kOffsets * 64 / kPieces;
    static_assert(kOffsets >= 1 && kOffsetRows % 16 == 0 && kRequests % kOffsets == 0, "");
};

template <int CK, int CV, int PARTS>
struct FlashShape {
    using Keys = FlashTile<CK, true>;
    using Values = FlashTile<CV, false>;
    static constexpr int kWaveBytes = Keys::kBytes + Values::kBytes;
    // the parts' sums meet in LDS, and the scores that their weights are taken of and sums of weights
    static constexpr int kSumBytes = PARTS * (CV / 32) * 4096, kCombineBytes = kSumBytes + PARTS * 2 * 32 * 4;
    static constexpr int kLds = PARTS * kWaveBytes > kCombineBytes ? PARTS * kWaveBytes : kCombineBytes;
};

template <class F, int... I>
__device__ __forceinline__ void flash_each_of(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void flash_each(F&& f) { flash_each_of(f, std::make_integer_sequence<int, N>{}); }

// LDS reads and the waits for them, as assembly: the compiler would have each read wait for all requests under way
template <int OFFSET>
__device__ __forceinline__ void flash_read(dec_u32x4& to, uint32_t at) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(at), "n"(OFFSET)); }
template <int OFFSET>
__device__ __forceinline__ void flash_read_transposed(dec_u32x2& to, uint32_t at) {
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(to) : "v"(at), "n"(OFFSET));
}
template <int LATER>
__device__ __forceinline__ void flash_arrived(dec_u32x4& a, dec_u32x4& b) { asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a), "+v"(b) : "n"(LATER) : "memory"); }
__device__ __forceinline__ void flash_arrived(dec_u32x2 (&v)[4]) { asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])::"memory"); }
template <int LATER>
__device__ __forceinline__ void flash_landed() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory"); }

template <int CK, int CV, int PARTS>
__global__ __launch_bounds__(64 * PARTS, PARTS == 8 || CK <= 192 ? 2 : 1) void chunk_attention_mfma_kernel(ChunkAttentionParams prm) {
    using Shape = FlashShape<CK, CV, PARTS>;
    using Keys = typename Shape::Keys;
    using Values = typename Shape::Values;
    request_arguments(prm);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    constexpr int kKb = CK / 16, kVt = CV / 32;
    const int tid = threadIdx.x, lane = tid & 63;
    const int part = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5;
    const int kv_head = static_cast<int>(blockIdx.x);
    // (What divisions and a median leave in vector registers is the same in every lane, but a descriptor made of it would be taken lane by lane, in a loop
    // around each request: 1024 rows of 16 query heads 19.5 us, so 15.8.)
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    const int group = uniform(prm.heads / prm.kv_heads);
    const int total = prm.rows * group;
    // late rows, which may see more keys, first
    const int row0 = ((total + kFlashRows - 1) / kFlashRows - 1 - static_cast<int>(blockIdx.z * gridDim.y + blockIdx.y)) * kFlashRows;
    if (row0 < 0) return;
    auto chunk_start = [&](int position) { return position - position % prm.chunk; };
    // what the block and this lane see: keys [.., ..]
    const int first_position = uniform(prm.position + row0 / group), last_position = uniform(prm.position + min(row0 + kFlashRows - 1, total - 1) / group);
    const int block_lo = uniform(chunk_start(first_position)), block_lo_most = uniform(chunk_start(last_position));
    const int query_row = min(row0 + (lane & 31), total - 1);
    const int local = query_row / group;
    const int position = prm.position + local;
    const int lo = block_lo == block_lo_most ? block_lo : chunk_start(position);

    // ---- requests: a tile goes out through a descriptor that begins at its first key and ends behind the last one that the block sees: a lane's
    // offset is the same for every tile, what lies past the last key or past a row's channels is out of range and reads as zero.  Past a wave's last
    // tile the requests stay (the waits count them) and ask for nothing. ----
    const uint16_t* k_head = static_cast<const uint16_t*>(prm.k_cache) + static_cast<int64_t>(kv_head) * prm.ring * prm.k_stride;
    const uint16_t* v_head = static_cast<const uint16_t*>(prm.v_cache) + static_cast<int64_t>(kv_head) * prm.ring * prm.v_stride;
    constexpr uint32_t kOutOfRange = 0x7ffffff0U;
    auto offsets_of = [&](auto tile_, int stride, auto& off) __attribute__((always_inline)) {
        using Tile = decltype(tile_);
#pragma unroll
        for (int i = 0; i < Tile::kOffsets; ++i) {
            const int at = 64 * i + lane, row = at / Tile::kPieces, c = 8 * (at % Tile::kPieces ^ Tile::key(row));
            off[i] = c < stride ? static_cast<uint32_t>(row * stride + c) * 2u : kOutOfRange;
        }
    };
    uint32_t k_off[Keys::kOffsets], v_off[Values::kOffsets];
    offsets_of(Keys{}, prm.k_stride, k_off);
    offsets_of(Values{}, prm.v_stride, v_off);
    unsigned char* const k_lds = smem + part * Shape::kWaveBytes;
    unsigned char* const v_lds = k_lds + Keys::kBytes;
    auto request = [&](auto tile_, const uint16_t* head_rows, int stride, const auto& off, unsigned char* to, int k0, int base) __attribute__((always_inline)) {
        using Tile = decltype(tile_);
        const int keys = uniform(max(min(last_position + 1 - k0, kFlashKeys), 0)), ahead = prm.ring - base;
        auto rows_from = [&](const uint16_t* first, int count) {
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(first), 0, count * stride * 2, 0x00020000);
        };
        auto bring = [&](const __amdgpu_buffer_rsrc_t& rsrc, int i, uint32_t from) __attribute__((always_inline)) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(to + 1024 * i), 16, static_cast<int>(from), 0, 0, 0);
        };
        const __amdgpu_buffer_rsrc_t rsrc = rows_from(head_rows + static_cast<int64_t>(base) * stride, min(keys, ahead));
        if (keys <= ahead) {
#pragma unroll
            for (int i = 0; i < Tile::kRequests; ++i)
                bring(rsrc, i, off[i % Tile::kOffsets] + static_cast<uint32_t>(i / Tile::kOffsets * Tile::kOffsetRows * stride * 2));
            return;
        }
        // (the rest at the ring's beginning, by other lanes of two instructions for one: the waits take that as longer ones)
        const __amdgpu_buffer_rsrc_t rest = rows_from(head_rows, keys - ahead);
#pragma unroll
        for (int i = 0; i < Tile::kRequests; ++i) {
            const int row = (64 * i + lane) / Tile::kPieces;
            const uint32_t from = off[i % Tile::kOffsets] + static_cast<uint32_t>(i / Tile::kOffsets * Tile::kOffsetRows * stride * 2);
            if (row < ahead) bring(rsrc, i, from);
            else bring(rest, i, from - static_cast<uint32_t>(ahead * stride * 2));
        }
    };
    auto request_keys = [&](int k0, int slot) __attribute__((always_inline)) { request(Keys{}, k_head, prm.k_stride, k_off, k_lds, k0, slot); };
    auto request_values = [&](int k0, int slot) __attribute__((always_inline)) { request(Values{}, v_head, prm.v_stride, v_off, v_lds, k0, slot); };

    // ---- fragment reads ----
    auto lds_of = [](unsigned char* at) { return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)at)); };
    // keys: lane's row lane % 32, piece 2 kb + half
    constexpr int kSwapKb = Keys::kSwap / 2;
    uint32_t k_at[kSwapKb];
#pragma unroll
    for (int i = 0; i < kSwapKb; ++i)
        k_at[i] = lds_of(k_lds) + static_cast<uint32_t>((lane & 31) * Keys::kRowBytes + 16 * (2 * i ^ half ^ Keys::key(lane & 31)));
    // queries: rows as a tile of keys, in KiB dealt to the waves' value tiles, every wave's piece brought by itself (straight into a matrix operand's
    // order a load goes to 32 rows, one lane a cycle: 24 KiB took a block 3000 cycles)
    auto query_lds = [&](int i) { return smem + i % PARTS * Shape::kWaveBytes + Keys::kBytes + i / PARTS * 1024; };
    {
        const int first_local = first_position - prm.position, locals = last_position - first_position + 1;
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(static_cast<const uint16_t*>(prm.q_rot) + static_cast<int64_t>(first_local) * prm.heads * prm.k_stride), 0,
            locals * prm.heads * prm.k_stride * 2, 0x00020000);
#pragma unroll
        for (int n = 0; n < (Keys::kRequests + PARTS - 1) / PARTS; ++n) {
            const int i = PARTS * n + part;
            if (i >= Keys::kRequests) break;
            const int at = 64 * i + lane, row = at / Keys::kPieces, c = 8 * (at % Keys::kPieces ^ Keys::key(row)), query = min(row0 + row, total - 1);
            const int from = (query / group - first_local) * prm.heads + kv_head * group + query % group;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)query_lds(i), 16,
                                                     static_cast<int>(c < prm.k_stride ? static_cast<uint32_t>(from * prm.k_stride + c) * 2u : kOutOfRange), 0, 0, 0);
        }
    }
    const int first_key = block_lo + kFlashKeys * part;
    int slot = uniform(first_key % prm.ring);
    request_keys(first_key, slot);
    flash_landed<Keys::kRequests>();
    asm volatile("s_barrier" ::: "memory");
    dec_u32x4 q[kKb];
    flash_each<kKb>([&](auto kb) {
        constexpr int i = decltype(kb)::value;
        const int at = (lane & 31) * Keys::kRowBytes + 16 * ((2 * i ^ half) ^ Keys::key(lane & 31));
        flash_read<0>(q[i], lds_of(smem) + static_cast<uint32_t>((at >> 10) % PARTS * Shape::kWaveBytes + Keys::kBytes + (at >> 10) / PARTS * 1024 + (at & 1023)));
    });
    flash_each<kKb / 2>([&](auto pair) { flash_arrived<0>(q[2 * decltype(pair)::value], q[2 * decltype(pair)::value + 1]); });
    asm volatile("s_barrier" ::: "memory");
    request_values(first_key, slot);
    // values: sixteen lanes take four keys x sixteen channels, lane 4 j + q of them channels 4 q .. of key j, and lane i gets the keys of channel i.
    // The product's k index 8 half + e of 16 keys is key 8 (e / 4) + 4 half + e % 4 (the order the scores left them in): two such reads.
    uint32_t v_at[kVt];
    const int v_row = 4 * half + (lane >> 2 & 3);
#pragma unroll
    for (int t = 0; t < kVt; ++t)
        v_at[t] = lds_of(v_lds) + static_cast<uint32_t>(v_row * Values::kRowBytes + 16 * ((4 * t + 2 * (lane >> 4 & 1) + (lane >> 1 & 1)) ^ Values::key(v_row)) + 8 * (lane & 1));

    dec_f32x16 o[kVt];
#pragma unroll
    for (int t = 0; t < kVt; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
    float m = -INFINITY, l = 0.0f;
    // (of scores times a positive factor the largest is the largest score's; others are multiplied first)
    const float to_log2 = prm.scale * kLog2e, factor_of_score = to_log2 > 0.0f ? to_log2 : 1.0f;

    for (int k0 = first_key; k0 <= last_position; k0 += PARTS * kFlashKeys) {
        const int next = k0 + PARTS * kFlashKeys;
        slot += PARTS * kFlashKeys;
        if (slot >= prm.ring) slot = uniform(slot % prm.ring);
        flash_landed<Values::kRequests>();
        dec_u32x4 key[kKb];
        flash_each<kKb>([&](auto kb) {
            constexpr int i = decltype(kb)::value;
            flash_read<16 * Keys::kSwap * (i / kSwapKb)>(key[i], k_at[i % kSwapKb]);
        });
        dec_f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.0f;
        flash_each<kKb / 2>([&](auto pair) {
            constexpr int i = 2 * decltype(pair)::value;
            flash_arrived<kKb - 2 - i>(key[i], key[i + 1]);
            if constexpr (i + 2 == kKb) request_keys(next, slot);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, key[i]), __builtin_bit_cast(bf16x8_t, q[i]), s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, key[i + 1]), __builtin_bit_cast(bf16x8_t, q[i + 1]), s, 0, 0, 0);
        });
        flash_landed<Keys::kRequests>();
        dec_u32x2 value[kVt][4];
        flash_each<kVt>([&](auto tile) {
            constexpr int t = decltype(tile)::value;
            flash_read_transposed<0>(value[t][0], v_at[t]);
            flash_read_transposed<8 * Values::kRowBytes>(value[t][1], v_at[t]);
            flash_read_transposed<16 * Values::kRowBytes>(value[t][2], v_at[t]);
            flash_read_transposed<24 * Values::kRowBytes>(value[t][3], v_at[t]);
        });
        // register r is key k0 + 8 (r / 4) + 4 half + r % 4
        const bool whole = k0 >= block_lo_most && k0 + kFlashKeys - 1 <= first_position;
        if (!(to_log2 > 0.0f)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] *= to_log2;
        }
        if (!whole) {
            const int first = lo - k0 - 4 * half, last = position - k0 - 4 * half;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 8 * (r / 4) + r % 4 >= first && 8 * (r / 4) + r % 4 <= last ? s[r] : -INFINITY;
        }
        float largest = fmaxf(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3])), fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7])));
        largest = fmaxf(largest, fmaxf(fmaxf(fmaxf(s[8], s[9]), fmaxf(s[10], s[11])), fmaxf(fmaxf(s[12], s[13]), fmaxf(s[14], s[15]))));
        largest = xor32_max(largest) * factor_of_score;
        // (weights are taken of a score up to kFlashSlack above the largest so far: where one exceeds that, it is raised and the sums so far are lowered.
        // 1024 rows of 16 query heads 15.8 -> 14.7 us.  Weights stay at one or below, so that no sum leaves the range that its result is in; what lies 2^118 below
        // the largest is zero.)
        if (__any(largest > m)) {
            const float before = m;
            m = fmaxf(m, largest + kFlashSlack);
            const float alpha = m == -INFINITY ? 1.0f : fast_exp2(before - m);
            l *= alpha;
#pragma unroll
            for (int t = 0; t < kVt; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[t][r] *= alpha;
        }
        const float reference = m == -INFINITY ? 0.0f : m;         // (a row that has seen no key yet: all its weights are zero)
#pragma unroll
        for (int t = 0; t < kVt; ++t) flash_arrived(value[t]);
        request_values(next, slot);
        float p[16], sum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            p[r] = fast_exp2(s[r] * factor_of_score - reference);       // (of rounded products, as the reference is: finite scores of any size come to zero at most; fused, 0.3 us less of 15)
            sum += p[r];
        }
        l += sum;
        dec_u32x4 high[2], low[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x = p[8 * b + 2 * e], y = p[8 * b + 2 * e + 1];
                const uint32_t pair_of = pack_bf16_pair(x, y);
                high[b][e] = pair_of;
                low[b][e] = pack_bf16_pair(x - lo_bf16(pair_of), y - hi_bf16(pair_of));
            }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
#pragma unroll
            for (int t = 0; t < 2 * kVt; ++t) {                    // (a sum is not asked for again right behind its last product)
                const dec_u32x2 *v = value[t % kVt] + 2 * b;
                const dec_u32x4 a = {v[0][0], v[0][1], v[1][0], v[1][1]};
                o[t % kVt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, t < kVt ? high[b] : low[b]), o[t % kVt], 0, 0, 0);
            }
        }
    }

    // The parts of the keys, combined: all leave their sums in LDS, and each takes its share of the rows.
    l = xor32_sum(l);
    flash_landed<0>();               // (the requests past the last tile)
    __syncthreads();
    float* sums = reinterpret_cast<float*>(smem);                  // [parts][kVt][register / 4][lane][4]
    float* ml = reinterpret_cast<float*>(smem + Shape::kSumBytes); // [parts][2][32]
#pragma unroll
    for (int t = 0; t < kVt; ++t)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<float4*>(sums + (((part * kVt + t) * 4 + g) * 64 + lane) * 4) = make_float4(o[t][4 * g], o[t][4 * g + 1], o[t][4 * g + 2], o[t][4 * g + 3]);
    if (lane < 32) {
        ml[part * 64 + lane] = m;
        ml[part * 64 + 32 + lane] = l;
    }
    __syncthreads();
    constexpr int kLanes = 2 * PARTS;                              // to a row
    const int mine = 32 / PARTS * part + lane / kLanes, mine_row = row0 + mine;
    if (mine_row < total) {
        float most = ml[mine], factor[PARTS], total_l = 0.0f;
#pragma unroll
        for (int p = 1; p < PARTS; ++p) most = fmaxf(most, ml[p * 64 + mine]);
#pragma unroll
        for (int p = 0; p < PARTS; ++p) {
            factor[p] = fast_exp2(ml[p * 64 + mine] - most);
            total_l = fmaf(ml[p * 64 + 32 + mine], factor[p], total_l);
        }
        const float scale = 1.0f / total_l;
        uint16_t* out = static_cast<uint16_t*>(prm.out) + mine_row / group * prm.ld_out + (kv_head * group + mine_row % group) * prm.vdim;
#pragma unroll
        for (int i = 0; i < (CV / 4 + kLanes - 1) / kLanes; ++i) {
            const int c = 4 * (kLanes * i + lane % kLanes);
            if (c >= prm.vdim) break;
            float v[4] = {};
#pragma unroll
            for (int p = 0; p < PARTS; ++p) {
                const float4 x = *reinterpret_cast<const float4*>(sums + ((p * (CV / 8) + (c >> 3)) * 64 + mine + 32 * (c >> 2 & 1)) * 4);
                v[0] = fmaf(x.x, factor[p], v[0]);
                v[1] = fmaf(x.y, factor[p], v[1]);
                v[2] = fmaf(x.z, factor[p], v[2]);
                v[3] = fmaf(x.w, factor[p], v[3]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] *= scale;
            if (prm.vdim % 4 == 0) {
                *reinterpret_cast<uint2*>(out + c) = make_uint2(pack_bf16_pair(v[0], v[1]), pack_bf16_pair(v[2], v[3]));
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (c + e < prm.vdim) out[c + e] = f2bf(v[e]);
            }
        }
    }
    // zeros behind the heads' columns, by the last head's blocks
    if (kv_head == prm.kv_heads - 1) {
        const int first = row0 / group, last = min(row0 + kFlashRows - 1, total - 1) / group;
        const int from = prm.heads * prm.vdim, behind = static_cast<int>(prm.ld_out) - from;
        for (int i = tid; i < (last - first + 1) * behind; i += 64 * PARTS)
            static_cast<uint16_t*>(prm.out)[(first + i / behind) * prm.ld_out + from + i % behind] = 0;
    }
}

template <int CK, int CV, int PARTS>
static int32_t flash_of(const ChunkAttentionParams& prm, unsigned blocks, hipStream_t stream) {
    using Shape = FlashShape<CK, CV, PARTS>;
    static std::atomic<bool> raised[kMaxDevices];
    const int32_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(chunk_attention_mfma_kernel<CK, CV, PARTS>), Shape::kLds, raised);
    if (rc != QM_OK) return rc;
    const unsigned layers = (blocks + kFlashHigh - 1) / kFlashHigh;
    hipLaunchKernelGGL((chunk_attention_mfma_kernel<CK, CV, PARTS>), dim3(prm.kv_heads, (blocks + layers - 1) / layers, layers), dim3(64 * PARTS), Shape::kLds, stream, prm);
    return launch_status();
}
// Eight waves where the grid leaves CUs without a second block and a block walks long: half the steps, for a longer combination (us, four waves /
// eight, 8 heads of 192 and 128: 100 rows behind 0, 500, 900, 1500 and 4000 keys 6.6 / 8.4, 10.6 / 11.1, 13.4 / 13.6, 18.4 / 16.9 and 35.7 / 28.6, 300 rows behind 1000
// 16.7 / 15.5; 16 query heads on 8 of 128, 100 rows behind 900 11.9 / 12.0, 500 behind 1500 21.2 / 20.2, 850 rows, 432 blocks, 13.2 / 18.3).
constexpr int kFlashLongWalk = 1200, kFlashCus = 256;
template <int CK, int CV>
static int32_t flash_as(const ChunkAttentionParams& prm, hipStream_t stream) {
    const int64_t blocks = (static_cast<int64_t>(prm.rows) * (prm.heads / prm.kv_heads) + kFlashRows - 1) / kFlashRows;
    if constexpr (FlashShape<CK, CV, 8>::kLds <= 160 * 1024)
        if (blocks * prm.kv_heads <= kFlashCus && std::min<int64_t>(prm.chunk, static_cast<int64_t>(prm.position) + prm.rows) >= kFlashLongWalk)
            return flash_of<CK, CV, 8>(prm, static_cast<unsigned>(blocks), stream);
    return flash_of<CK, CV, 4>(prm, static_cast<unsigned>(blocks), stream);
}

int32_t check_chunk_attention_mfma(const ChunkAttentionParams& prm) {
    if (prm.ld_out % 4 || (reinterpret_cast<uintptr_t>(prm.out) & 7)) return QM_ERR_GEOMETRY;
    return static_cast<int64_t>(prm.rows) * (prm.heads / prm.kv_heads) > kFlashMostRows ? QM_ERR_GEOMETRY : QM_OK;
}
int32_t launch_chunk_attention_mfma(const ChunkAttentionParams& prm, hipStream_t stream) {
    const int32_t rc = check_chunk_attention_mfma(prm);
    if (rc != QM_OK) return rc;
    const int c = prm.dim > prm.vdim ? prm.dim : prm.vdim;
    if (c <= 32) return flash_as<32, 32>(prm, stream);
    if (c <= 64) return flash_as<64, 64>(prm, stream);
    if (c <= 128) return flash_as<128, 128>(prm, stream);
    if (prm.dim <= 192 && prm.vdim <= 128) return flash_as<192, 128>(prm, stream);
    return flash_as<256, 256>(prm, stream);
}

}  // namespace qm
