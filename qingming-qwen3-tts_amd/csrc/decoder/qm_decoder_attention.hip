// qm_decoder_attention.hip — softmax attention inside chunks of positions (position i sees j <= i with the same
// floor(. / chunk)), grouped query heads, over a ring cache of keys and values, for gfx950.
//
// Chunks count from position 0 of the sequence, so a query needs at most `chunk` keys, all of them in the cache however the
// prompt was cut.  Three kernels: few rows (decode) deal a chunk's keys to several blocks per key/value head and combine the
// partial results; many bf16 rows take the matrix-core kernel of qm_decoder_attention_mfma.hip, many fp32 rows, where it ends first, that of
// qm_decoder_attention_f32.hip.
#include "../qm_host.h"
#include "qm_decoder_attention.h"

namespace qm {

// Rotation of the rows' queries and keys, keys and values into the ring: one block per row.  The row's projections pass
// through LDS; a thread puts out eight channels at a time.
__device__ __forceinline__ void store8(uint16_t* to, const float (&v)[8]) {
    *reinterpret_cast<uint4*>(to) = make_uint4(pack_bf16_pair(v[0], v[1]), pack_bf16_pair(v[2], v[3]), pack_bf16_pair(v[4], v[5]), pack_bf16_pair(v[6], v[7]));
}
__device__ __forceinline__ void store8(float* to, const float (&v)[8]) {
    reinterpret_cast<float4*>(to)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4*>(to)[1] = make_float4(v[4], v[5], v[6], v[7]);
}

template <class T>
__global__ __launch_bounds__(kDecThreads) void rope_cache_kernel(ChunkAttentionParams prm) {
    extern __shared__ __attribute__((aligned(16))) float sh_row[];             // q, k, v; cosines; sines
    const int tid = threadIdx.x;
    const int row = static_cast<int>(blockIdx.x);
    const int position = position_of(prm.position_dev, prm.position) + row;
    const int half = prm.rot_dims >> 1, q_n = prm.heads * prm.dim, k_n = prm.kv_heads * prm.dim, v_n = prm.kv_heads * prm.vdim;
    float* sh_cos = sh_row + q_n + k_n + v_n;
    float* sh_sin = sh_cos + half;
    const float* proj = prm.proj + row * prm.ld_proj;
#pragma unroll 4
    for (int i = tid; i < q_n; i += kDecThreads) sh_row[i] = proj[i];
#pragma unroll 4
    for (int i = tid; i < k_n; i += kDecThreads) sh_row[q_n + i] = proj[prm.k_column + i];
#pragma unroll 4
    for (int i = tid; i < v_n; i += kDecThreads) sh_row[q_n + k_n + i] = proj[prm.v_column + i];
    for (int i = tid; i < half; i += kDecThreads) rotary(position, prm.frequency[i], sh_cos[i], sh_sin[i]);
    __syncthreads();
    auto rotated = [&](const float* head, int c0, float (&v)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int c = c0 + e;
            const int pair = c < half ? c : c - half;
            const bool turns = c < prm.rot_dims;
            const float own = c < prm.dim ? head[c] : 0.0f;
            const float other = turns ? head[c < half ? c + half : pair] : 0.0f;
            const float cosine = turns ? sh_cos[pair] : 1.0f, sine = turns ? sh_sin[pair] : 0.0f;
            v[e] = c < half ? own * cosine - other * sine : own * cosine + other * sine;
        }
    };
    const int64_t slot = position % prm.ring;
    const int k_pieces = prm.k_stride >> 3, v_pieces = prm.v_stride >> 3;
    for (int i = tid; i < (prm.heads + prm.kv_heads) * k_pieces; i += kDecThreads) {
        const int h = i / k_pieces, c = (i - h * k_pieces) * 8;
        float v[8];
        rotated(sh_row + h * prm.dim, c, v);                                   // (the key heads follow the query heads)
        store8(h < prm.heads ? static_cast<T*>(prm.q_rot) + (static_cast<int64_t>(row) * prm.heads + h) * prm.k_stride + c
                             : static_cast<T*>(prm.k_cache) + (static_cast<int64_t>(h - prm.heads) * prm.ring + slot) * prm.k_stride + c, v);
    }
    for (int i = tid; i < prm.kv_heads * v_pieces; i += kDecThreads) {
        const int h = i / v_pieces, c = (i - h * v_pieces) * 8;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = c + e < prm.vdim ? sh_row[q_n + k_n + h * prm.vdim + c + e] : 0.0f;
        store8(static_cast<T*>(prm.v_cache) + (static_cast<int64_t>(h) * prm.ring + slot) * prm.v_stride + c, v);
    }
}

// The same for heads of whole pieces of eight channels whose halves turn in fours, projections of whole float4s: a thread holds four channels of both
// halves of a head, asked for before the row's angles are known, and nothing but those passes through LDS.  Bound by memory: 16 + 8 heads of 128 and as
// many values over 1024 rows, 25 MB, 11.2 -> 6.6 us (3.8 TB/s); 16 + 8 of 64 over 300 fp32 rows 7.0 -> 4.8, most of it the launch.  (Above, a value a
// load, eight LDS reads of a stride of eight banks for a piece, a condition for each channel.)
__device__ __forceinline__ float4 turned(float4 own, float4 other, float4 cosine, float4 sine, float sign) {
    return make_float4(own.x * cosine.x + sign * other.x * sine.x, own.y * cosine.y + sign * other.y * sine.y,
                       own.z * cosine.z + sign * other.z * sine.z, own.w * cosine.w + sign * other.w * sine.w);
}
template <class T>
__global__ __launch_bounds__(kDecThreads) void rope_cache_vectors_kernel(ChunkAttentionParams prm) {
    __shared__ __attribute__((aligned(16))) float sh_cos[kDecMaxHead / 2], sh_sin[kDecMaxHead / 2];
    const int tid = threadIdx.x, row = static_cast<int>(blockIdx.x);
    const int position = position_of(prm.position_dev, prm.position) + row;
    const int half = prm.rot_dims >> 1, heads = prm.heads + prm.kv_heads;
    const int64_t slot = position % prm.ring;
    const float* proj = prm.proj + row * prm.ld_proj;
    auto from = [&](int h) { return proj + (h < prm.heads ? h * prm.dim : prm.k_column + (h - prm.heads) * prm.dim); };
    auto to = [&](int h) {
        return h < prm.heads ? static_cast<T*>(prm.q_rot) + (static_cast<int64_t>(row) * prm.heads + h) * prm.dim
                             : static_cast<T*>(prm.k_cache) + (static_cast<int64_t>(h - prm.heads) * prm.ring + slot) * prm.dim;
    };
    const int pairs = half >> 2, turning = heads * pairs, value_pieces = prm.vdim >> 2, values = prm.kv_heads * value_pieces;
    constexpr int kHeld = 2;
    float4 low[kHeld], high[kHeld], value[kHeld];
    auto request = [&](int first) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < kHeld; ++n) {
            const int i = min(first + n * kDecThreads, turning - 1), h = i / pairs, c = (i - h * pairs) * 4;
            low[n] = *reinterpret_cast<const float4*>(from(h) + c);
            high[n] = *reinterpret_cast<const float4*>(from(h) + c + half);
        }
    };
    auto request_values = [&](int first) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < kHeld; ++n) value[n] = *reinterpret_cast<const float4*>(proj + prm.v_column + min(first + n * kDecThreads, values - 1) * 4);
    };
    if (turning > 0) request(tid);
    request_values(tid);
    for (int i = tid; i < half; i += kDecThreads) rotary(position, prm.frequency[i], sh_cos[i], sh_sin[i]);
    for (int first = tid; first < values; first += kHeld * kDecThreads) {
        if (first != tid) request_values(first);
#pragma unroll
        for (int n = 0; n < kHeld; ++n) {
            const int i = first + n * kDecThreads, h = i / value_pieces;
            if (i < values)
                store4(static_cast<T*>(prm.v_cache) + (static_cast<int64_t>(h) * prm.ring + slot) * prm.vdim, i - h * value_pieces, value[n].x, value[n].y,
                       value[n].z, value[n].w);
        }
    }
    const int still = (prm.dim - prm.rot_dims) >> 2;
    for (int i = tid; i < heads * still; i += kDecThreads) {
        const int h = i / still, v = (prm.rot_dims >> 2) + i - h * still;
        const float4 x = reinterpret_cast<const float4*>(from(h))[v];
        store4(to(h), v, x.x, x.y, x.z, x.w);
    }
    __syncthreads();
    for (int first = tid; first < turning; first += kHeld * kDecThreads) {
        if (first != tid) request(first);
#pragma unroll
        for (int n = 0; n < kHeld; ++n) {
            const int i = first + n * kDecThreads, h = i / pairs, c = (i - h * pairs) * 4;
            if (i >= turning) break;
            const float4 cosine = *reinterpret_cast<const float4*>(sh_cos + c), sine = *reinterpret_cast<const float4*>(sh_sin + c);
            const float4 u = turned(low[n], high[n], cosine, sine, -1.0f), v = turned(high[n], low[n], cosine, sine, 1.0f);
            store4(to(h), c >> 2, u.x, u.y, u.z, u.w);
            store4(to(h), (c + half) >> 2, v.x, v.y, v.z, v.w);
        }
    }
}
static bool rope_in_vectors(const ChunkAttentionParams& p) {
    return p.dim % 8 == 0 && p.vdim % 8 == 0 && p.rot_dims % 8 == 0 && p.ld_proj % 4 == 0 && p.k_column % 4 == 0 && p.v_column % 4 == 0 &&
           reinterpret_cast<uintptr_t>(p.proj) % 16 == 0;
}

template <class T, int GQ, int VC>
__global__ __launch_bounds__(kDecThreads) void chunk_attention_kernel(ChunkAttentionParams prm) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    chunk_attention_block<T, GQ, VC, false>(prm, static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), static_cast<int>(blockIdx.z), lds);
}

template <class T>
__global__ __launch_bounds__(kDecThreads) void merge_attention_kernel(ChunkAttentionParams prm) {
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int64_t row = blockIdx.x;
    const int position = position_of(prm.position_dev, prm.position) + static_cast<int>(row);
    merge_attention_row<T>(prm.part, row, attention_active_splits(position, prm.chunk, prm.part.keys_per_split), lds,
                           static_cast<T*>(prm.out) + row * prm.ld_out, prm.ld_out);
}

int32_t check_attention(const ChunkAttentionParams& p) {
    if (p.rows < 0 || p.position < 0) return QM_ERR_ARGUMENT;
    if (!p.proj || !p.k_cache || !p.v_cache || !p.out || !p.part.ml || !p.part.acc || (p.rot_dims > 0 && !p.frequency)) return QM_ERR_NULL;
    if (p.heads <= 0 || p.kv_heads <= 0 || p.heads % p.kv_heads || p.dim <= 0 || p.vdim <= 0 || p.dim > kDecMaxHead || p.vdim > kDecMaxHead)
        return QM_ERR_GEOMETRY;
    if (p.k_stride != (p.dim + 7) / 8 * 8 || p.v_stride != (p.vdim + 7) / 8 * 8) return QM_ERR_GEOMETRY;
    if (p.rot_dims < 0 || p.rot_dims > p.dim || p.rot_dims % 2 || p.chunk <= 0 || p.ring <= 0) return QM_ERR_GEOMETRY;
    if (p.part.heads != p.heads || p.part.vdim != p.vdim || p.part.splits < 1 || p.part.splits > kDecMaxSplits) return QM_ERR_GEOMETRY;
    if (p.part.keys_per_split <= 0 || static_cast<int64_t>(p.part.keys_per_split) * p.part.splits < p.chunk) return QM_ERR_GEOMETRY;
    if (p.ld_out < static_cast<int64_t>(p.heads) * p.vdim || p.rows > 65535 || p.ld_out % 4) return QM_ERR_GEOMETRY;
    if (static_cast<int64_t>(p.heads) * p.part.splits > kDecMaxMerge) return QM_ERR_GEOMETRY;
    return QM_OK;
}

template <class T>
static int32_t rope_cache(const ChunkAttentionParams& prm, hipStream_t stream) {
    const size_t lds = sizeof(float) * (static_cast<size_t>(prm.heads + prm.kv_heads) * prm.dim + static_cast<size_t>(prm.kv_heads) * prm.vdim + prm.rot_dims);
    static std::atomic<bool> raised[kMaxDevices];
    const int32_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(rope_cache_kernel<T>), kDotLdsMost, raised);
    if (rc != QM_OK) return rc;
    if (lds > static_cast<size_t>(kDotLdsMost)) return QM_ERR_GEOMETRY;
    if (rope_in_vectors(prm)) {
        hipLaunchKernelGGL(rope_cache_vectors_kernel<T>, dim3(prm.rows), dim3(kDecThreads), 0, stream, prm);
        return launch_status();
    }
    hipLaunchKernelGGL(rope_cache_kernel<T>, dim3(prm.rows), dim3(kDecThreads), lds, stream, prm);
    return launch_status();
}

template <class T, int GQ>
static int32_t launch_rows(const ChunkAttentionParams& prm, hipStream_t stream) {
    const dim3 grid(prm.part.splits, prm.kv_heads, prm.rows);
    const size_t lds = sizeof(float) * attention_lds_floats(GQ, prm.k_stride, prm.v_stride);
    if (prm.v_stride <= 128 && prm.k_stride <= 128) hipLaunchKernelGGL((chunk_attention_kernel<T, GQ, 1>), grid, dim3(kDecThreads), lds, stream, prm);
    else hipLaunchKernelGGL((chunk_attention_kernel<T, GQ, 2>), grid, dim3(kDecThreads), lds, stream, prm);
    int32_t rc = launch_status();
    if (rc != QM_OK) return rc;
    hipLaunchKernelGGL(merge_attention_kernel<T>, dim3(prm.rows), dim3(kDecThreads), sizeof(float) * prm.heads * prm.part.splits, stream, prm);
    return launch_status();
}

template <class T>
static int32_t attention_rows(const ChunkAttentionParams& prm, hipStream_t stream) {
    const int group = prm.heads / prm.kv_heads;
    return group == 1 ? launch_rows<T, 1>(prm, stream) : group == 2 ? launch_rows<T, 2>(prm, stream) : launch_rows<T, 4>(prm, stream);
}

int32_t launch_chunk_attention(const ChunkAttentionParams& prm, int f32, hipStream_t stream) {
    int32_t rc = check_attention(prm);
    if (rc != QM_OK || prm.rows == 0) return rc;
    if (!prm.q_rot) return QM_ERR_NULL;
    // (positions that only the device knows belong to one-token steps)
    const bool many = !prm.position_dev && !(prm.options & QM_ATTENTION_ROWS), matrix = many && !f32 && prm.rows >= kAttentionMatrixRows;
    if (matrix) rc = check_chunk_attention_mfma(prm);              // (in front of the rotation, which writes the caches)
    if (rc != QM_OK) return rc;
    rc = f32 ? rope_cache<float>(prm, stream) : rope_cache<uint16_t>(prm, stream);
    if (rc != QM_OK) return rc;
    if (matrix) return launch_chunk_attention_mfma(prm, stream);
    if (f32 && many && attention_f32_pays(prm)) return launch_chunk_attention_f32(prm, stream);
    return f32 ? attention_rows<float>(prm, stream) : attention_rows<uint16_t>(prm, stream);
}

}  // namespace qm
