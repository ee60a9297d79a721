// qm_decoder_attention_f32.hip — the chunked attention of a prompt's fp32 rows on the fp32 matrix cores (gfx950).
//
// A block takes 16 query rows of one key/value head (a query row is a position and one of the head's query heads: they share
// keys and values); its waves go round the steps of 16 keys that any of the rows sees and combine through LDS at the end.
// Scores are S^T = K Q^T (v_mfma_f32_16x16x4_f32): a lane then holds four keys of one query, where the second product
// O^T = V^T P^T wants its right operand, so that a wave needs nothing from another while it walks and keys and values go from
// L2 to registers once.  Bound: the chain of a wave's steps (a step's two products are 32 instructions of 32 cycles at heads of
// 64 channels, behind one trip to L2); flops 2 (dim + vdim) per key and query.
// No sum has longer chains than in the kernel of few rows: scores are kept in sixteen sums, and a step's share of the values
// is summed apart, in two, before it joins the rest.  Root mean square error against 64 bits, 16 query heads over 8 key/value
// heads of 64 channels, chunks of 512: 1.04e-7 at 16 rows, 1.18e-7 at 300 (the kernel of few rows: 1.07e-7, 1.21e-7).
#include <algorithm>

#include "../qm_host.h"
#include "qm_decoder_mfma32.h"

namespace qm {

constexpr int kF32AttentionRows = 16;          // query rows per block
constexpr int kF32AttentionSums = 16;          // sums per score

__host__ __device__ constexpr int f32_attention_lds(int waves, int channels) {
    return 4 * waves * (kF32AttentionRows * (channels + 4) + 2 * kF32AttentionRows);
}

// C: channels of a key and of a value, rounded up to a multiple of 64
template <int C, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void chunk_attention_f32_kernel(ChunkAttentionParams prm) {
    extern __shared__ __attribute__((aligned(16))) float sh_sums[];            // [waves][rows][C + 4]; [waves][2][rows]
    constexpr int kStride = C + 4;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kv_head = static_cast<int>(blockIdx.x);
    const int group = prm.heads / prm.kv_heads;
    const int total = prm.rows * group;
    const int row0 = static_cast<int>(gridDim.y - 1 - blockIdx.y) * kF32AttentionRows;    // (late rows, which may see more keys, first)
    auto position_at = [&](int query_row) { return prm.position + min(query_row, total - 1) / group; };
    auto chunk_start = [&](int position) { return position - position % prm.chunk; };
    const int first_position = position_at(row0), last_position = position_at(row0 + kF32AttentionRows - 1);
    const int block_lo = chunk_start(first_position), lo_most = chunk_start(last_position);
    const int query_row = min(row0 + l16, total - 1);
    const int position = position_at(query_row), lo = chunk_start(position);

    float4 q[C / 16];                          // (channels past the head: zeros here and in the keys, whose clamped loads repeat the last four)
    const float* q_row = static_cast<const float*>(prm.q_rot) +
                         (static_cast<int64_t>(query_row / group) * prm.heads + kv_head * group + query_row % group) * prm.k_stride;
#pragma unroll
    for (int kb = 0; kb < C / 16; ++kb) {
        const int c = 16 * kb + 4 * g;
        const float4 read = *reinterpret_cast<const float4*>(q_row + min(c, prm.k_stride - 4));
        q[kb] = c < prm.k_stride ? read : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    const float* k_head = static_cast<const float*>(prm.k_cache) + static_cast<int64_t>(kv_head) * prm.ring * prm.k_stride;
    const float* v_head = static_cast<const float*>(prm.v_cache) + static_cast<int64_t>(kv_head) * prm.ring * prm.v_stride;
    const int base = block_lo % prm.ring;
    auto slot_of = [&](int key) {              // (keys past the block's last repeat it: masked)
        const int s = base + min(key, last_position) - block_lo;
        return static_cast<int64_t>(s >= prm.ring ? s - prm.ring : s);
    };
    float4 k[C / 16];
    auto request = [&](int k0) __attribute__((always_inline)) {
        const float* k_row = k_head + slot_of(k0 + l16) * prm.k_stride;
#pragma unroll
        for (int kb = 0; kb < C / 16; ++kb) k[kb] = *reinterpret_cast<const float4*>(k_row + min(16 * kb + 4 * g, prm.k_stride - 4));
    };

    const f32x4_t none = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4_t o[C / 64][4];                      // row i of tile t of a group of 64 channels is channel 4 i + t
#pragma unroll
    for (int x = 0; x < C / 64; ++x)
#pragma unroll
        for (int t = 0; t < 4; ++t) o[x][t] = none;
    float m = -INFINITY, l = 0.0f;
    const int begin = block_lo + 16 * wave;
    if (begin <= last_position) request(begin);
    for (int k0 = begin; k0 <= last_position; k0 += 16 * WAVES) {
        float4 v[C / 64][4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float* v_row = v_head + slot_of(k0 + 4 * g + r) * prm.v_stride;
#pragma unroll
            for (int x = 0; x < C / 64; ++x) v[x][r] = *reinterpret_cast<const float4*>(v_row + min(64 * x + 4 * l16, prm.v_stride - 4));
        }
        f32x4_t s[kF32AttentionSums];
#pragma unroll
        for (int i = 0; i < kF32AttentionSums; ++i) s[i] = none;
        if (prm.k_stride < C) {
#pragma unroll
            for (int kb = 0; kb < C / 16; ++kb)
                if (16 * kb + 4 * g >= prm.k_stride) k[kb] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
#pragma unroll
        for (int kb = 0; kb < C / 16; ++kb) {
            f32x4_t* sums = s + 4 * (kb & 3);
            sums[0] = mfma32(k[kb].x, q[kb].x, sums[0]);
            sums[1] = mfma32(k[kb].y, q[kb].y, sums[1]);
            sums[2] = mfma32(k[kb].z, q[kb].z, sums[2]);
            sums[3] = mfma32(k[kb].w, q[kb].w, sums[3]);
        }
        request(min(k0 + 16 * WAVES, last_position));
        const bool whole = k0 >= lo_most && k0 + 15 <= first_position;     // every row sees every key
        float p[4], largest = -INFINITY;       // register r is key k0 + 4 g + r
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int key = k0 + 4 * g + r;
            float part[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) part[i] = (s[4 * i][r] + s[4 * i + 1][r]) + (s[4 * i + 2][r] + s[4 * i + 3][r]);
            const float score = ((part[0] + part[1]) + (part[2] + part[3])) * prm.scale;
            p[r] = whole || (key >= lo && key <= position) ? score : -INFINITY;
            largest = fmaxf(largest, p[r]);
        }
        largest = xor16_max(largest);
        largest = xor32_max(largest);
        const float before = m;
        m = fmaxf(m, largest);
        const float reference = m == -INFINITY ? 0.0f : m;                 // (a row that has seen no key yet: all its weights are zero)
        const float alpha = expf(before - reference);
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = expf(p[r] - reference);
        l = l * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
        // A weight of zero does not silence a value that is no number.  Where a row sees some of the step's keys only, its
        // others must not reach it whatever they hold.
        bool finite = true;
        if (!whole) {
#pragma unroll
            for (int x = 0; x < C / 64; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    finite = finite && fmaxf(fmaxf(fabsf(v[x][r].x), fabsf(v[x][r].y)), fmaxf(fabsf(v[x][r].z), fabsf(v[x][r].w))) < INFINITY &&
                             v[x][r].x == v[x][r].x && v[x][r].y == v[x][r].y && v[x][r].z == v[x][r].z && v[x][r].w == v[x][r].w;
        }
        if (__all(finite)) {
#pragma unroll
            for (int x = 0; x < C / 64; ++x) {
                f32x4_t step[2][4] = {{none, none, none, none}, {none, none, none, none}};
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    f32x4_t* sums = step[r & 1];
                    sums[0] = mfma32(v[x][r].x, p[r], sums[0]);
                    sums[1] = mfma32(v[x][r].y, p[r], sums[1]);
                    sums[2] = mfma32(v[x][r].z, p[r], sums[2]);
                    sums[3] = mfma32(v[x][r].w, p[r], sums[3]);
                }
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[x][t][r] = fmaf(o[x][t][r], alpha, step[0][t][r] + step[1][t][r]);
            }
        } else {
#pragma unroll
            for (int x = 0; x < C / 64; ++x)
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[x][t][r] *= alpha;
#pragma unroll 1
            for (int i = 0; i < 16; ++i) {
                const int key = k0 + i;
                const float weight = __shfl(i & 2 ? (i & 1 ? p[3] : p[2]) : (i & 1 ? p[1] : p[0]), 4 * (i & 12) + l16, 64);
                const bool seen = key >= lo && key <= position;
                const float* v_row = v_head + slot_of(key) * prm.v_stride;
#pragma unroll
                for (int x = 0; x < C / 64; ++x)
#pragma unroll
                    for (int t = 0; t < 4; ++t)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            if (seen) o[x][t][e] = fmaf(weight, v_row[min(64 * x + 4 * (4 * g + e) + t, prm.v_stride - 1)], o[x][t][e]);
            }
        }
    }

    // the waves' shares of the keys, combined by all threads
    l = xor16_sum(l);
    l = xor32_sum(l);
    float* sh_ml = sh_sums + WAVES * kF32AttentionRows * kStride;
    float* own = sh_sums + (wave * kF32AttentionRows + l16) * kStride + 16 * g;
#pragma unroll
    for (int x = 0; x < C / 64; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) *reinterpret_cast<float4*>(own + 64 * x + 4 * r) = make_float4(o[x][0][r], o[x][1][r], o[x][2][r], o[x][3][r]);
    if (g == 0) {
        sh_ml[2 * kF32AttentionRows * wave + l16] = m;
        sh_ml[2 * kF32AttentionRows * wave + kF32AttentionRows + l16] = l;
    }
    __syncthreads();
    for (int i = tid; i < kF32AttentionRows * (C / 4); i += WAVES * 64) {
        const int row = i / (C / 4), c = i % (C / 4) * 4;
        if (row0 + row >= total || c >= prm.vdim) continue;
        float most = sh_ml[row];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) most = fmaxf(most, sh_ml[2 * kF32AttentionRows * w + row]);
        float4 sum[2] = {};
        float weights[2] = {};
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {      // (a wave without keys for the row: factor zero; its sums are zeros)
            const float factor = expf(sh_ml[2 * kF32AttentionRows * w + row] - most);
            const float4 share = *reinterpret_cast<const float4*>(sh_sums + (w * kF32AttentionRows + row) * kStride + c);
            float4& to = sum[w & 1];
            weights[w & 1] = fmaf(sh_ml[2 * kF32AttentionRows * w + kF32AttentionRows + row], factor, weights[w & 1]);
            to.x = fmaf(share.x, factor, to.x); to.y = fmaf(share.y, factor, to.y);
            to.z = fmaf(share.z, factor, to.z); to.w = fmaf(share.w, factor, to.w);
        }
        const float scale = 1.0f / (weights[0] + weights[1]);
        const float values[4] = {(sum[0].x + sum[1].x) * scale, (sum[0].y + sum[1].y) * scale, (sum[0].z + sum[1].z) * scale,
                                 (sum[0].w + sum[1].w) * scale};
        const int local = (row0 + row) / group, head = kv_head * group + (row0 + row) % group;
        float* out = static_cast<float*>(prm.out) + local * prm.ld_out + head * prm.vdim + c;
        if (prm.vdim % 4 == 0) *reinterpret_cast<float4*>(out) = make_float4(values[0], values[1], values[2], values[3]);
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (c + e < prm.vdim) out[e] = values[e];
        }
    }
    // zeros behind the heads' columns, by the last head's blocks
    if (kv_head == prm.kv_heads - 1) {
        const int first = row0 / group, last = min(row0 + kF32AttentionRows - 1, total - 1) / group;
        const int from = prm.heads * prm.vdim, behind = static_cast<int>(prm.ld_out) - from;
        for (int i = tid; i < (last - first + 1) * behind; i += WAVES * 64)
            static_cast<float*>(prm.out)[(first + i / behind) * prm.ld_out + from + i % behind] = 0.0f;
    }
}

template <int C, int WAVES>
static int32_t attention_f32_as(const ChunkAttentionParams& prm, hipStream_t stream) {
    constexpr int kLds = f32_attention_lds(WAVES, C);
    static std::atomic<bool> raised[kMaxDevices];
    const int32_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(chunk_attention_f32_kernel<C, WAVES>), kLds, raised);
    if (rc != QM_OK) return rc;
    const int64_t blocks = (static_cast<int64_t>(prm.rows) * (prm.heads / prm.kv_heads) + kF32AttentionRows - 1) / kF32AttentionRows;
    hipLaunchKernelGGL((chunk_attention_f32_kernel<C, WAVES>), dim3(prm.kv_heads, static_cast<unsigned>(blocks)), dim3(WAVES * 64), kLds, stream, prm);
    return launch_status();
}

// Whether the rows take this kernel: its time against that of the kernel of few rows, which deals a row's keys to several blocks if
// the caller cut them.  Both are a start and a block's chain, in tenths of a microsecond as measured, times the rounds of blocks: here
// a step of 64 keys 14 (heads of more than 64 channels: 21) and a block per CU; there a pass of 128 keys 30 for up to two query heads
// of a key/value head, 39 for every four, two blocks per CU, and 0.07 for every block launched beyond that.
// Measured with the rotation's launch (us, here / kernel of few rows).  16 query heads over 8 of 64 channels, chunks of 512: 9.2 / 15.5
// at 16 rows, 10.5 / 23.0 at 100, 15.8 / 54.4 at 300, 43.5 / 172 at 1024; of 128 channels 11.6 / 16.8 at 16 rows, 68.5 / 180 at 1024.
// The last 16 rows of 1016, two heads over one of 128 channels: 41 / 31.  16 rows at position 8000 in a chunk of 8192, 16 heads over 8
// of 64 channels: 175 / 177 uncut and 65 in four pieces, of 128 channels 263 / 187 and 68; 4 heads over one of 64: 174 / 247 and 29 in
// sixteen; 150 rows 180 / 255 and 115.
// Heads past 128 channels stay with the kernel of few rows: the registers of 256 spill (4 query heads over one of 256 channels, 300
// rows: 54 / 51).
bool attention_f32_pays(const ChunkAttentionParams& prm) {
    const int64_t group = prm.heads / prm.kv_heads, chunk = prm.chunk;
    auto pieces = [](int64_t n, int64_t of) { return (n + of - 1) / of; };
    if (prm.rows < kAttentionMatrixRows || prm.dim > 128 || prm.vdim > 128 || pieces(prm.rows * group, kF32AttentionRows) > 65535 ||
        (reinterpret_cast<uintptr_t>(prm.out) & 15) != 0)
        return false;
    const int64_t before = prm.position % chunk;
    const int64_t keys = std::min(before + prm.rows, chunk);       // the most that a row sees
    const int64_t first = std::min<int64_t>(prm.rows, chunk - before), more = prm.rows - first, last = more % chunk;
    const int64_t all_keys = first * before + first * (first + 1) / 2 + more / chunk * (chunk * (chunk + 1) / 2) + last * (last + 1) / 2;
    const int64_t rows = pieces(all_keys, keys);                   // as many as see that many for the same work
    const int64_t here = 75 + pieces(keys, 64) * (std::max(prm.dim, prm.vdim) <= 64 ? 14 : 21) *
                                  pieces(pieces(rows * group, kF32AttentionRows) * prm.kv_heads, 256);
    const int64_t piece = std::min<int64_t>(keys, prm.part.keys_per_split);
    const int64_t there = 120 + pieces(piece, 128) * (group <= 2 ? 30 : 39 * pieces(group, 4)) * pieces(pieces(keys, piece) * prm.kv_heads * rows, 512) +
                          std::max<int64_t>(static_cast<int64_t>(prm.part.splits) * prm.kv_heads * prm.rows - 512, 0) * 7 / 100;
    return here <= there;
}

int32_t launch_chunk_attention_f32(const ChunkAttentionParams& prm, hipStream_t stream) {
    const int c = prm.dim > prm.vdim ? prm.dim : prm.vdim;
    if (c <= 64) return attention_f32_as<64, 4>(prm, stream);
    return attention_f32_as<128, 4>(prm, stream);
}

}  // namespace qm
