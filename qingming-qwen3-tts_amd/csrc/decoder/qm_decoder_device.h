// qm_decoder_device.h — device helpers shared by the decoder language models' kernels (gfx950, wave64).
//
// Activations that a matrix product reads are bf16 (T = uint16_t) when the model is served and fp32 (T = float) in the
// 32-bit mode; weights are bf16 in both (the checkpoint's own format, so nothing is lost).  Everything else — the residual
// stream, projections on their way into a mixer, norms, scores, recurrent state — is fp32 throughout.
#pragma once

#include "../qm_device.h"
#include "qm_decoder_ops.h"

namespace qm {

constexpr int kDecThreads = 256;

__device__ __forceinline__ float to_f32(uint16_t v) { return bf2f(v); }
__device__ __forceinline__ float to_f32(float v) { return v; }
template <class T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ uint16_t from_f32<uint16_t>(float v) { return f2bf(v); }
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }

// (v_exp_f32 and v_rcp_f32 are good to one unit in the last place)
__device__ __forceinline__ float reciprocal(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float sigmoid_f32(float z) { return reciprocal(1.0f + fast_exp2(-z * kLog2e)); }
__device__ __forceinline__ float silu_f32(float z) { return z * sigmoid_f32(z); }

// Sum / maximum over the 64 lanes of a wave, in every lane.
__device__ __forceinline__ float wave_sum(float v) {
    v = row16_allreduce_sum(v);
    v = xor16_sum(v);
    v = xor32_sum(v);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, row_ror<8>(v));
    v = fmaxf(v, row_ror<4>(v));
    v = fmaxf(v, row_ror<2>(v));
    v = fmaxf(v, row_ror<1>(v));
    return xor32_max(xor16_max(v));
}

// N sums over the 256 threads of a block at once, in every thread.  sh: 4 * N floats of LDS, free again for the next call
// after the caller's next barrier (two calls in a row take two areas).
template <int N>
__device__ __forceinline__ void block_sums(float (&v)[N], float* sh) {
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        v[i] = wave_sum(v[i]);
        if ((threadIdx.x & 63) == 0) sh[i * 4 + wave] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = (sh[i * 4] + sh[i * 4 + 1]) + (sh[i * 4 + 2] + sh[i * 4 + 3]);
}

// A position is known to the host, or lives in device memory where a captured graph finds it.
__device__ __forceinline__ int position_of(const int32_t* device, int host) { return device ? *device : host; }

// The residual sum and its norm for one row by a block of 256 threads.  Rows are padded with zeros to ld_h columns, and a
// thread owns the float4s tid, tid + 256, ... of a row (NV of them): everything the row needs is requested before the first
// sum waits.  sh_red: 16 floats of LDS; h may be LDS or global memory.  The caller puts a barrier between this and any use
// of sh_red or h by other threads.
__device__ __forceinline__ float4 load4(const float* p, int v) { return reinterpret_cast<const float4*>(p)[v]; }
__device__ __forceinline__ float4 load4(const uint16_t* p, int v) {
    const uint2 w = reinterpret_cast<const uint2*>(p)[v];
    return make_float4(lo_bf16(w.x), hi_bf16(w.x), lo_bf16(w.y), hi_bf16(w.y));
}
__device__ __forceinline__ void store4(float* p, int v, float a, float b, float c, float d) { reinterpret_cast<float4*>(p)[v] = make_float4(a, b, c, d); }
__device__ __forceinline__ void store4(uint16_t* p, int v, float a, float b, float c, float d) {
    reinterpret_cast<uint2*>(p)[v] = make_uint2(pack_bf16_pair(a, b), pack_bf16_pair(c, d));
}
__device__ __forceinline__ float square_sum(float4 v, float sum) { return fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, sum)))); }
// Element v, or zeros where it is not wanted: the load is made either way (from the first element), because a load under a
// condition would wait its turn behind a branch.
template <class P>
__device__ __forceinline__ float4 load4_if(bool wanted, const P* p, int v) {
    const float4 x = load4(p, wanted ? v : 0);
    return make_float4(wanted ? x.x : 0.0f, wanted ? x.y : 0.0f, wanted ? x.z : 0.0f, wanted ? x.w : 0.0f);
}
// acc + f * y * w
__device__ __forceinline__ float4 weighted(float4 acc, float f, float4 y, float4 w) {
    return make_float4(fmaf(f * y.x, w.x, acc.x), fmaf(f * y.y, w.y, acc.y), fmaf(f * y.z, w.z, acc.z), fmaf(f * y.w, w.w, acc.w));
}

// `behind` is called when the row's loads have been asked for: a wave's loads come back in the order they were made, and what it asks for
// (weights, by the megabyte) the sums do not wait for.  EARLY: the norms' weights are among the first loads too (registers).
struct NothingBehind {
    __device__ __forceinline__ void operator()() const {}
};
// The upper eight significant bits of x as a bf16 in the upper half of a word, and what is left of x.  (Infinities and NaNs
// stay what they are, with nothing left.)
__device__ __forceinline__ uint32_t take_upper(float& x) {
    const uint32_t bits = __float_as_uint(x);
    const bool finite = (bits & 0x7f800000U) != 0x7f800000U;
    const uint32_t nan = (bits & 0x7fffffffU) > 0x7f800000U ? 0x00400000U : 0U;
    const uint32_t upper = (bits | nan) & 0xffff0000U;
    x = finite ? x - __uint_as_float(upper) : 0.0f;
    return upper;
}

// A row of fp32 that is also left split into its three parts, `plane` elements apart.
struct SplitRow {
    float* whole;
    uint16_t* parts;
    int64_t plane;
};
__device__ __forceinline__ void store4(const SplitRow& to, int v, float a, float b, float c, float d) {
    store4(to.whole, v, a, b, c, d);
#pragma unroll
    for (int part = 0; part < 3; ++part) {
        auto next = [&](float& x) { return part < 2 ? take_upper(x) : __float_as_uint(x); };
        const uint32_t wa = next(a), wb = next(b), wc = next(c), wd = next(d);
        reinterpret_cast<uint2*>(to.parts + part * to.plane)[v] =
            make_uint2(__builtin_amdgcn_perm(wb, wa, 0x07060302U), __builtin_amdgcn_perm(wd, wc, 0x07060302U));
    }
}

// MORE: the last term's further pieces are added to it.  H: where the norm's output goes.
template <class T, int NV, bool EARLY = false, bool MORE = false, class Behind = NothingBehind, class H = T*>
__device__ __forceinline__ void residual_norm_row(const ResidualParams& prm, int row, float* sh_red, H h, bool write_x, Behind&& behind = Behind(),
                                                  const MoreOfTerm& more = MoreOfTerm()) {
    const int tid = threadIdx.x;
    const int64_t src = prm.row_map ? prm.row_map[row] : row;
    const int vectors = static_cast<int>(prm.ld_h >> 2);
    const float* y_row[3];
    bool normed[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        y_row[i] = i < prm.terms ? prm.term[i].y + src * prm.term[i].ld : nullptr;
        normed[i] = i < prm.terms && prm.term[i].norm_w;
    }
    const uint16_t *embedding = nullptr, *bigram = nullptr;
    if (!prm.x_in) {
        const int64_t token = min(max(prm.tokens[src], 0), prm.vocab - 1);
        embedding = prm.embed + token * prm.ld_h;
        if (prm.buckets > 0) {
            const int64_t before = prm.tokens[src - 1];
            bigram = prm.bigram + (before < 0 ? prm.buckets : (before * prm.mul_prev + token * prm.mul_cur) % prm.buckets) * prm.ld_h;
        }
    }
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f), one = make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    float4 x[NV], y[3][NV], pieces[MORE ? kMorePlanes : 1][MORE ? NV : 1];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int v = tid + i * kDecThreads;
        const bool in = v < vectors;
        x[i] = embedding ? load4_if(in, embedding, v) : load4_if(in, prm.x_in + src * prm.ld_h, v);
        if (bigram) x[i] = weighted(x[i], 1.0f, load4_if(in, bigram, v), one);
#pragma unroll
        for (int t = 0; t < 3; ++t) y[t][i] = y_row[t] ? load4_if(in, y_row[t], v) : zero;
        if constexpr (MORE) {
            const float* piece = more.sums + src * prm.term[prm.terms - 1].ld;
#pragma unroll
            for (int p = 0; p < kMorePlanes; ++p) pieces[p][i] = p < more.planes ? load4_if(in, piece + p * more.plane, v) : zero;
        }
    }
    float4 y_weight[3][EARLY ? NV : 1], step_vec[EARLY ? NV : 1], weight[EARLY ? NV : 1];
    if constexpr (EARLY) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int v = tid + i * kDecThreads, from = v < vectors ? v : 0;
#pragma unroll
            for (int t = 0; t < 3; ++t) y_weight[t][i] = normed[t] ? load4(prm.term[t].norm_w, from) : one;
            step_vec[i] = prm.step_vec ? load4(prm.step_vec, from) : zero;
            weight[i] = load4(prm.norm_w, from);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    behind();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (MORE) {
#pragma unroll
        for (int t = 0; t < 3; ++t)
            if (t == prm.terms - 1) {
#pragma unroll
                for (int i = 0; i < NV; ++i)
#pragma unroll
                    for (int p = 0; p < kMorePlanes; ++p) y[t][i] = weighted(y[t][i], 1.0f, pieces[p][i], one);
            }
    }
    const float inv_width = 1.0f / static_cast<float>(prm.width);
    float factor[3] = {0.0f, 0.0f, 0.0f};
    if (normed[0] || normed[1] || normed[2]) {
#pragma unroll
        for (int t = 0; t < 3; ++t)
#pragma unroll
            for (int i = 0; i < NV; ++i) factor[t] = square_sum(y[t][i], factor[t]);
        block_sums<3>(factor, sh_red);
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        const float inverse = normed[t] ? 1.0f / sqrtf(factor[t] * inv_width + prm.eps) : 1.0f;
        factor[t] = t < prm.terms ? prm.term[t].scale * inverse : 0.0f;
    }
    float total[1] = {0.0f};
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int v = tid + i * kDecThreads;
        if (v >= vectors) continue;
        float4 add = zero;
#pragma unroll
        for (int t = 0; t < 3; ++t)
            if (y_row[t]) add = weighted(add, factor[t], y[t][i], EARLY ? y_weight[t][EARLY ? i : 0] : normed[t] ? load4(prm.term[t].norm_w, v) : one);
        x[i] = weighted(x[i], 1.0f, add, one);
        if (prm.step_vec) x[i] = weighted(x[i], 1.0f, EARLY ? step_vec[EARLY ? i : 0] : load4(prm.step_vec, v), one);
        if (write_x && prm.x_out) reinterpret_cast<float4*>(prm.x_out + static_cast<int64_t>(row) * prm.ld_h)[v] = x[i];
        total[0] = square_sum(x[i], total[0]);
    }
    block_sums<1>(total, sh_red + 12);
    const float inverse = 1.0f / sqrtf(total[0] * inv_width + prm.eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int v = tid + i * kDecThreads;
        if (v >= vectors) continue;
        const float4 w = EARLY ? weight[EARLY ? i : 0] : load4(prm.norm_w, v);
        store4(h, v, x[i].x * inverse * w.x, x[i].y * inverse * w.y, x[i].z * inverse * w.z, x[i].w * inverse * w.w);
    }
}

// The factor that a gate's projection g becomes.
__device__ __forceinline__ float gate_f32(float g, bool silu) { return silu ? silu_f32(g) : sigmoid_f32(g); }

// One row of the gated norm's slices, a wave per slice, a slice of up to 256 values held by its lanes.  The values of AT_ONCE slices are
// asked for at once, and with more than one their weights.
template <class T, int AT_ONCE, class Behind>
__device__ __forceinline__ void gated_norm_slices(const GatedNormParams& prm, const float* o, const float* gate, T* out, Behind&& behind) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const bool silu = prm.silu != 0;
    const float inv_size = 1.0f / static_cast<float>(prm.size);
    auto weight_at = [&](int at) { return prm.weight ? prm.weight[at] : 1.0f; };
    for (int g0 = wave; g0 < prm.groups; g0 += AT_ONCE * (kDecThreads / 64)) {
        float held[AT_ONCE][4], gates[AT_ONCE][4], weights[AT_ONCE][4];
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j) {
            const int g = min(g0 + j * (kDecThreads / 64), prm.groups - 1);   // (past the last: repeated, not stored)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = lane + 64 * i;
                const bool in = c < prm.size;
                const int at = g * prm.size + (in ? c : 0);
                const float value = o[at];
                gates[j][i] = gate[at];
                if (AT_ONCE > 1) weights[j][i] = weight_at(at);
                held[j][i] = in ? value : 0.0f;
            }
        }
        if (g0 == wave) behind();
#pragma unroll
        for (int j = 0; j < AT_ONCE; ++j) {
            const int g = g0 + j * (kDecThreads / 64);
            if (g >= prm.groups) break;
            float sq = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) sq = fmaf(held[j][i], held[j][i], sq);
            for (int c = lane + 256; c < prm.size; c += 64) sq = fmaf(o[g * prm.size + c], o[g * prm.size + c], sq);
            const float inverse = 1.0f / sqrtf(wave_sum(sq) * inv_size + prm.eps);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int c = lane + 64 * i, at = g * prm.size + c;
                if (c < prm.size) out[at] = from_f32<T>(held[j][i] * inverse * (AT_ONCE > 1 ? weights[j][i] : weight_at(at)) * gate_f32(gates[j][i], silu));
            }
            for (int c = lane + 256; c < prm.size; c += 64) {
                const int at = g * prm.size + c;
                out[at] = from_f32<T>(o[at] * inverse * weight_at(at) * gate_f32(gate[at], silu));
            }
        }
    }
}

// Whether a wave asks for up to four of its slices at once: where more than four values a lane come of it, and for few rows, each a
// chain of round trips, from three slices on.  One by one a kernel has registers for more waves, which hides as much where rows are
// many; slices past 256 values are read twice then, from caches that fewer waves spare.  (us, one by one / four: 16 x 128 of 1 row
// 4.1 / 3.4, of 1024 7.9 / 6.5; 8 x 256 of 12 rows 3.7 / 3.0, of 4000 16.4 / 14.3; 16 x 64 of 12 rows 3.8 / 3.5, of 1024 5.1 / 5.2; 8 x
// 128 of 12 rows 3.0 / 2.9, of 1024 4.0 / 4.5; 8 x 64 of 1024 3.5 / 4.2; 8 x 512 of 1024 rows 13.3 / 11.2, of 2048 17.5 / 19.8.)
inline bool gated_norm_many(const GatedNormParams& prm, int rows) {
    const int slices = (prm.groups + 3) / 4;
    const bool wide = (slices < 4 ? slices : 4) * (prm.size < 256 ? prm.size : 256) > 256;
    return (wide && (prm.size <= 256 || rows <= 1024)) || (slices >= 3 && rows <= 512);
}

// One row of the gated norm by a block of 256 threads; sh_red: 4 floats of LDS.  AT_ONCE: how slices are taken; 0: in a
// one-token step, where they go by four and a single slice's weights are asked for with its values as well (the block has few waves
// beside it whatever its registers: 48 tokens of the second design 7990 us, 8160 by the rule for rows).  `behind` is called by every wave once,
// where that can be when its first loads have been asked for.
template <class T, int AT_ONCE = 0, class Behind = NothingBehind>
__device__ __forceinline__ void gated_norm_row(const GatedNormParams& prm, int64_t row, float* sh_red, T* out, Behind&& behind = Behind()) {
    const int tid = threadIdx.x;
    const float* o = prm.o + row * prm.ld_o;
    const float* gate = prm.gate + row * prm.ld_gate;
    const bool silu = prm.silu != 0;
    const int total = prm.groups * prm.size;
    const float inv_size = 1.0f / static_cast<float>(prm.size);
    auto weight_at = [&](int at) { return prm.weight ? prm.weight[at] : 1.0f; };
    constexpr int kHeld = 4;                   // float4s a thread holds between its two uses of a value
    if (AT_ONCE <= 1 && prm.groups == 1 && total % 4 == 0 && prm.ld_o % 4 == 0 && total <= kHeld * 4 * kDecThreads) {
        const int vectors = total >> 2;
        auto weight4 = [&](int v) { return prm.weight ? load4_if(v < vectors, prm.weight, v) : make_float4(1.0f, 1.0f, 1.0f, 1.0f); };
        float4 held[kHeld], g[kHeld], weight[kHeld];
        float sq[1] = {0.0f};
#pragma unroll
        for (int i = 0; i < kHeld; ++i) {
            const int v = tid + i * kDecThreads;
            held[i] = load4_if(v < vectors, o, v);
            g[i] = load4_if(v < vectors, gate, v);
            if (AT_ONCE == 0) weight[i] = weight4(v);
        }
        behind();
#pragma unroll
        for (int i = 0; i < kHeld; ++i) sq[0] = square_sum(held[i], sq[0]);
        block_sums<1>(sq, sh_red);
        const float inverse = 1.0f / sqrtf(sq[0] * inv_size + prm.eps);
#pragma unroll
        for (int i = 0; i < kHeld; ++i) {
            const int v = tid + i * kDecThreads;
            if (v >= vectors) continue;
            const float4 w = AT_ONCE == 0 ? weight[i] : weight4(v);
            store4(out, v, held[i].x * inverse * w.x * gate_f32(g[i].x, silu), held[i].y * inverse * w.y * gate_f32(g[i].y, silu),
                   held[i].z * inverse * w.z * gate_f32(g[i].z, silu), held[i].w * inverse * w.w * gate_f32(g[i].w, silu));
        }
    } else if (AT_ONCE <= 1 && prm.groups == 1) {
        behind();
        float sq[1] = {0.0f};
        for (int c = tid; c < total; c += kDecThreads) sq[0] = fmaf(o[c], o[c], sq[0]);
        block_sums<1>(sq, sh_red);
        const float inverse = 1.0f / sqrtf(sq[0] * inv_size + prm.eps);
        for (int c = tid; c < total; c += kDecThreads)
            out[c] = from_f32<T>(o[c] * inverse * weight_at(c) * gate_f32(gate[c], silu));
    } else {
        if (static_cast<int>(threadIdx.x >> 6) >= prm.groups) behind();        // (a wave without a slice)
        gated_norm_slices<T, AT_ONCE == 1 ? 1 : 4>(prm, o, gate, out, behind);
    }
    for (int c = total + tid; c < prm.ld_out; c += kDecThreads) out[c] = from_f32<T>(0.0f);
}

// One row's heads, combined, by a block of 256 threads; `active` splits hold keys.  sh_w: heads * active floats of LDS.  The statistics of four
// heads a wave and the values of eight splits for two vectors a thread are asked for first, `behind` is called then.
template <class T, class Behind = NothingBehind>
__device__ __forceinline__ void merge_attention_row(const AttentionPartials& p, int64_t row, int active, float* sh_w, T* out, int64_t ld_out,
                                                    Behind&& behind = Behind()) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = p.heads * p.vdim;
    const float* acc = p.acc + row * p.heads * p.splits * p.vdim;
    const bool vectors = p.vdim % 4 == 0;
    const int per_head = p.vdim >> 2, all = n >> 2;
    constexpr int kHeads = 4, kVectors = 2, kSplits = 8;
    float m_read[kHeads], l_read[kHeads];
    auto read_heads = [&](int h0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kHeads; ++j) {                         // (past the last: repeated, not stored)
            const int h = min(h0 + j * (kDecThreads / 64), p.heads - 1);
            const int64_t at = ((row * p.heads + h) * p.splits + min(lane, active - 1)) * 2;
            m_read[j] = p.ml[at];
            l_read[j] = p.ml[at + 1];
        }
    };
    float4 v[kVectors][kSplits];
    auto read_vectors = [&](int i0, int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < kVectors; ++j) {                       // (splits past the last: the last one, with factor zero)
            const int i = min(i0 + j * kDecThreads, all - 1), h = i / per_head;
            const float4* from = reinterpret_cast<const float4*>(acc + static_cast<int64_t>(h) * p.splits * p.vdim) + (i - h * per_head);
#pragma unroll
            for (int s = 0; s < kSplits; ++s) v[j][s] = from[min(s0 + s, active - 1) * per_head];
        }
    };
    read_heads(wave);
    if (vectors) read_vectors(static_cast<int>(threadIdx.x), 0);
    __builtin_amdgcn_sched_barrier(0);
    behind();
    __builtin_amdgcn_sched_barrier(0);
    for (int h0 = wave; h0 < p.heads; h0 += kHeads * (kDecThreads / 64)) {     // each split's factor: a wave per head, a lane per split
        if (h0 != wave) read_heads(h0);
#pragma unroll
        for (int j = 0; j < kHeads; ++j) {
            const int h = h0 + j * (kDecThreads / 64);
            const float m = lane < active ? m_read[j] : -INFINITY, l = lane < active ? l_read[j] : 0.0f;
            const float w = fast_exp2((m - wave_max(m)) * kLog2e);
            const float total = wave_sum(w * l);
            if (lane < active && h < p.heads) sh_w[h * active + lane] = w / total;
        }
    }
    __syncthreads();
    if (vectors) {
        for (int i0 = threadIdx.x; i0 < all; i0 += kVectors * kDecThreads) {
            float4 sum[kVectors];
#pragma unroll
            for (int j = 0; j < kVectors; ++j) sum[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            for (int s0 = 0; s0 < active; s0 += kSplits) {
                if (i0 != static_cast<int>(threadIdx.x) || s0 != 0) read_vectors(i0, s0);
#pragma unroll
                for (int j = 0; j < kVectors; ++j) {
                    const int h = min(i0 + j * kDecThreads, all - 1) / per_head;
#pragma unroll
                    for (int s = 0; s < kSplits; ++s) {
                        const float w = s0 + s < active ? sh_w[h * active + min(s0 + s, active - 1)] : 0.0f;
                        sum[j].x = fmaf(w, v[j][s].x, sum[j].x); sum[j].y = fmaf(w, v[j][s].y, sum[j].y);
                        sum[j].z = fmaf(w, v[j][s].z, sum[j].z); sum[j].w = fmaf(w, v[j][s].w, sum[j].w);
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < kVectors; ++j)
                if (i0 + j * kDecThreads < all) store4(out, i0 + j * kDecThreads, sum[j].x, sum[j].y, sum[j].z, sum[j].w);
        }
    } else {
        for (int i = threadIdx.x; i < n; i += kDecThreads) {
            const int h = i / p.vdim, e = i - h * p.vdim;
            float sum = 0.0f;
            for (int s = 0; s < active; ++s) sum = fmaf(sh_w[h * active + s], acc[(static_cast<int64_t>(h) * p.splits + s) * p.vdim + e], sum);
            out[i] = from_f32<T>(sum);
        }
    }
    for (int c = n + threadIdx.x; c < ld_out; c += kDecThreads) out[c] = from_f32<T>(0.0f);
}

// Rotary factors of pair i at a position: the angle in double (position * frequency, reduced to one turn), its sine and
// cosine in fp32.
__device__ __forceinline__ void rotary(int position, double frequency, float& cosine, float& sine) {
    const double angle = static_cast<double>(position) * frequency;
    const double turns = rint(angle * 0.15915494309189535);
    const float reduced = static_cast<float>(fma(-turns, 6.283185307179586, angle));
    sincosf(reduced, &sine, &cosine);
}

// n values divided by their root mean square and weighted, by a block of 256 threads, zeros behind them up to `padded`;
// sh_red: 4 floats of LDS.
template <class T, class Behind = NothingBehind>
__device__ __forceinline__ void slice_norm_row(const float* x, const float* weight, int n, int64_t padded, float eps, float* sh_red, T* out,
                                               Behind&& behind = Behind()) {
    const int tid = threadIdx.x;
    constexpr int kHeld = 4;
    float held[kHeld], weights[kHeld], sq[1] = {0.0f};
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
        const int c = min(tid + i * kDecThreads, n - 1);
        held[i] = x[c];
        weights[i] = weight[c];
    }
    behind();
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
        held[i] = tid + i * kDecThreads < n ? held[i] : 0.0f;
        sq[0] = fmaf(held[i], held[i], sq[0]);
    }
    for (int c = tid + kHeld * kDecThreads; c < n; c += kDecThreads) sq[0] = fmaf(x[c], x[c], sq[0]);
    block_sums<1>(sq, sh_red);
    const float inverse = 1.0f / sqrtf(sq[0] / static_cast<float>(n) + eps);
#pragma unroll
    for (int i = 0; i < kHeld; ++i) {
        const int c = tid + i * kDecThreads;
        if (c < n) out[c] = from_f32<T>(held[i] * inverse * weights[i]);
    }
    for (int c = tid + kHeld * kDecThreads; c < n; c += kDecThreads) out[c] = from_f32<T>(x[c] * inverse * weight[c]);
    for (int64_t c = n + tid; c < padded; c += kDecThreads) out[c] = from_f32<T>(0.0f);
}

}  // namespace qm
