// qm_decoder_linear_f32.hip — linears of the 32-bit mode over several token rows on the bf16 matrix cores (gfx950).
//
// An fp32 input of at least 2^-110 is the exact sum of three bf16 numbers (its upper eight significant bits, the next eight, the
// last eight: splitting a number over several narrow products is the common way to a wide product on narrow matrix cores) and the
// weights are bf16 as they are, so three bf16 products with fp32 accumulation form what fp32 products form: every product is exact.
// Of a smaller input what lies under 2^-133 is lost, so outputs so small that it could tell are formed again in fp32.  The sums are
// taken in two levels — 64 terms, the smallest parts first, then those sums one after the other — which keeps the chains of
// roundings as short as a wave's lanes keep them in the dot-product kernel.
//
// A block of four waves takes 16 BT token rows and 64 TN weight rows (a gate/up pair: 32 TN channels, gate and up rows in the
// same lanes), 64 k a step.  Weights are a wave's own and go straight to its registers, requested two steps ahead, a row's
// 64 bytes per instruction; inputs are read once per block, split by the threads that fetched them and shared through two
// LDS stages (a row's 16-byte pieces swizzled over the banks).  Bound: three times the bf16 matrix-core flops of the shape.
#include <algorithm>

#include "../qm_host.h"
#include "qm_decoder_dot.h"

namespace qm {

constexpr int kF32Step = 64;                   // k per step
constexpr float kF32Small = 0x1p-80f;          // what inputs lose under 2^-133 is no 2^-24th of this for weights that sum to 2^29

typedef uint32_t split_u32x4_t __attribute__((ext_vector_type(4)));

struct SplitLinearParams {
    DecLinearParams linears;
    int first_tile[kDecGroups + 1];            // column tiles in front of each linear
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

// x . w in one chain.
__device__ __forceinline__ float plain_dot(const float* x, const uint16_t* w, int k) {
    float sum = 0.0f;
    for (int c = 0; c < k; c += 8) sum = dot8(*reinterpret_cast<const uint4*>(w + c), x + c, sum);
    return sum;
}

template <int BT, int TN, int KS>
__global__ __launch_bounds__(kDecThreads * KS, KS > 2 ? KS : 2) void split_linear_kernel(SplitLinearParams prm) {
    request_arguments(prm);
    constexpr int kRows = 16 * BT;
    constexpr int kPlane = kRows * kF32Step * 2;                   // LDS bytes of one part of a stage's rows
    constexpr int kPieces = kRows * 8;                             // pieces of eight k per stage
    constexpr int kOwn = (kPieces + kDecThreads - 1) / kDecThreads;
    extern __shared__ __attribute__((aligned(16))) unsigned char all_smem[];   // [KS][2][3][kPlane]
    const int tid = threadIdx.x % kDecThreads, lane = tid & 63, g = lane >> 4, l16 = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), share = __builtin_amdgcn_readfirstlane(threadIdx.x / kDecThreads);
    unsigned char* const smem = all_smem + share * (2 * 3 * kPlane);
    int which = 0;
    while (which + 1 < prm.linears.groups && static_cast<int>(blockIdx.x) >= prm.first_tile[which + 1]) ++which;
    const DecLinearGroup& group = prm.linears.group[which];
    const int tile = static_cast<int>(blockIdx.x) - prm.first_tile[which];
    const int k = group.k, row0 = static_cast<int>(blockIdx.y) * kRows, rows = prm.linears.rows;
    const bool pair = TN == 2 && group.w_up;
    // this wave's weight rows: 16 channels a tile; a pair's second tile is the same channels of the up matrix
    const int channel0 = tile * (pair ? 64 : 64 * TN) + wave * (pair ? 16 : 16 * TN);
    const uint16_t* w_at[TN];
#pragma unroll
    for (int a = 0; a < TN; ++a) {
        const int channel = min(channel0 + (pair ? 0 : 16 * a), group.n - 16) + l16;   // (past the last: repeated, never stored)
        w_at[a] = (a == 1 && pair ? group.w_up : group.w) + static_cast<int64_t>(channel) * k + 8 * g;
    }
    // this thread's pieces of a stage's rows
    const float* x_at[kOwn];
    uint32_t x_to[kOwn];
#pragma unroll
    for (int i = 0; i < kOwn; ++i) {
        const int p = tid + i * kDecThreads, row = (p >> 3) % kRows;
        x_at[i] = static_cast<const float*>(group.x) + static_cast<int64_t>(min(row0 + row, rows - 1)) * group.ldx + 8 * (p & 7);
        x_to[i] = static_cast<uint32_t>(row * 128 + (((p & 7) ^ ((row >> 1) & 7)) << 4));
    }
    const bool fetches = kPieces >= kDecThreads || tid < kPieces;
    uint32_t x_from[2];                                            // a fragment's place: row l16 of tile 0, k block 0 and 1
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) x_from[kb] = static_cast<uint32_t>(l16 * 128 + (((4 * kb + g) ^ ((l16 >> 1) & 7)) << 4));

    split_u32x4_t w[3][2][TN];
    float4 x[3][kOwn][2];
    const int steps = k / (kF32Step * KS);
    auto request_w = [&](int step, auto set_) __attribute__((always_inline)) {
        constexpr int S = decltype(set_)::value;
        const int at = (min(step, steps - 1) * KS + share) * kF32Step;
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) w[S][kb][a] = *reinterpret_cast<const split_u32x4_t*>(w_at[a] + at + 32 * kb);
    };
    auto request_x = [&](int step, auto set_) __attribute__((always_inline)) {
        constexpr int S = decltype(set_)::value;
        const int at = (min(step, steps - 1) * KS + share) * kF32Step;
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            x[S][i][0] = *reinterpret_cast<const float4*>(x_at[i] + at);
            x[S][i][1] = *reinterpret_cast<const float4*>(x_at[i] + at + 4);
        }
    };
    auto store_x = [&](int stage, auto set_) __attribute__((always_inline)) {
        constexpr int S = decltype(set_)::value;
        if (!fetches) return;
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
            float v[8] = {x[S][i][0].x, x[S][i][0].y, x[S][i][0].z, x[S][i][0].w, x[S][i][1].x, x[S][i][1].y, x[S][i][1].z, x[S][i][1].w};
#pragma unroll
            for (int part = 0; part < 3; ++part) {
                uint32_t upper[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) upper[e] = part < 2 ? take_upper(v[e]) : __float_as_uint(v[e]);
                split_u32x4_t packed;
#pragma unroll
                for (int e = 0; e < 4; ++e) packed[e] = __builtin_amdgcn_perm(upper[2 * e + 1], upper[2 * e], 0x07060302U);
                *reinterpret_cast<split_u32x4_t*>(smem + (stage * 3 + part) * kPlane + x_to[i]) = packed;
            }
        }
    };
    f32x4_t sum[TN][BT] = {};
    auto one_step = [&](int step, auto set_) __attribute__((always_inline)) {
        constexpr int S = decltype(set_)::value;
        using next = std::integral_constant<int, (S + 1) % 3>;
        using after = std::integral_constant<int, (S + 2) % 3>;
        __syncthreads();
        request_x(step + 2, after{});
        request_w(step + 2, after{});
        f32x4_t part_sum[TN][BT] = {};
        const unsigned char* stage = smem + (step & 1) * 3 * kPlane;
#pragma unroll
        for (int part = 2; part >= 0; --part)                      // (the smallest parts first)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                split_u32x4_t f[BT];
#pragma unroll
                for (int b = 0; b < BT; ++b) f[b] = *reinterpret_cast<const split_u32x4_t*>(stage + part * kPlane + b * 2048 + x_from[kb]);
#pragma unroll
                for (int a = 0; a < TN; ++a)
#pragma unroll
                    for (int b = 0; b < BT; ++b)
                        part_sum[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[S][kb][a]), __builtin_bit_cast(bf16x8_t, f[b]),
                                                                                 part_sum[a][b], 0, 0, 0);
            }
        if (step + 1 < steps) store_x((step + 1) & 1, next{});
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < BT; ++b) sum[a][b] += part_sum[a][b];
    };
    using zero = std::integral_constant<int, 0>;
    using one = std::integral_constant<int, 1>;
    using two = std::integral_constant<int, 2>;
    request_x(0, zero{});
    request_w(0, zero{});
    request_x(1, one{});
    request_w(1, one{});
    store_x(0, zero{});
    int step = 0;
    for (; step + 3 <= steps; step += 3) {
        one_step(step, zero{});
        one_step(step + 1, one{});
        one_step(step + 2, two{});
    }
    if (step < steps) one_step(step++, zero{});
    if (step < steps) one_step(step, one{});

    if constexpr (KS > 1) {                                        // the shares of the reduction, added in order
        f32x4_t* const others = reinterpret_cast<f32x4_t*>(all_smem);
        __syncthreads();
        if (share > 0) {
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < BT; ++b) others[(((share - 1) * TN + a) * BT + b) * kDecThreads + tid] = sum[a][b];
        }
        __syncthreads();
        if (share > 0) return;
#pragma unroll
        for (int other = 0; other < KS - 1; ++other)
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < BT; ++b) sum[a][b] += others[((other * TN + a) * BT + b) * kDecThreads + tid];
    }
    // a lane holds columns 4 g .. 4 g + 3 of a tile's sixteen for token row l16
    bool good = true;
#pragma unroll
    for (int b = 0; b < BT; ++b) {
        const int row = row0 + 16 * b + l16;
        if (row >= rows) continue;
        if (pair) {
            if constexpr (TN == 2) {
                float4 v;
                float* to = static_cast<float*>(group.out) + static_cast<int64_t>(row) * group.ldo + channel0 + 4 * g;
                v.x = silu_f32(sum[0][b][0]) * sum[1][b][0];
                v.y = silu_f32(sum[0][b][1]) * sum[1][b][1];
                v.z = silu_f32(sum[0][b][2]) * sum[1][b][2];
                v.w = silu_f32(sum[0][b][3]) * sum[1][b][3];
                *reinterpret_cast<float4*>(to) = v;
                good = good && v.x == v.x && v.y == v.y && v.z == v.z && v.w == v.w;
            }
        } else {
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                const int channel = channel0 + 16 * a;
                if (channel >= group.n) continue;
                *reinterpret_cast<float4*>(group.out32 + static_cast<int64_t>(row) * group.ldo + channel + 4 * g) =
                    make_float4(sum[a][b][0], sum[a][b][1], sum[a][b][2], sum[a][b][3]);
#pragma unroll
                for (int r = 0; r < 4; ++r) good = good && (fabsf(sum[a][b][r]) >= kF32Small || sum[a][b][r] == 0.0f);
            }
        }
    }
    // The zeros among an input's lower parts make a NaN of an infinite weight, where the input itself makes an infinity of it.  Outputs
    // that are no number, or small (a pair's product of such would be zero), are therefore formed again from the inputs as they are.
    if (good) return;
    const float* const inputs = static_cast<const float*>(group.x);
    float* const outputs = pair ? static_cast<float*>(group.out) : group.out32;
#pragma unroll 1
    for (int i = 0; i < 4 * BT * (pair ? 1 : TN); ++i) {
        const int row = row0 + 16 * (i / 4 % BT) + l16, channel = channel0 + 16 * (i / (4 * BT)) + 4 * g + i % 4;
        if (row >= rows || channel >= group.n) continue;
        float* const at = outputs + static_cast<int64_t>(row) * group.ldo + channel;
        if (pair ? *at == *at : fabsf(*at) >= kF32Small) continue;
        const float* const x_row = inputs + static_cast<int64_t>(row) * group.ldx;
        const int64_t w_row = static_cast<int64_t>(channel) * k;
        const float first = plain_dot(x_row, group.w + w_row, k);
        *at = pair ? silu_f32(first) * plain_dot(x_row, group.w_up + w_row, k) : first;
    }
}

template <int BT, int TN, int KS>
static int32_t launch_split_as(const DecLinearParams& linears, hipStream_t stream) {
    SplitLinearParams prm = {};
    prm.linears = linears;
    for (int g = 0; g < linears.groups; ++g) {
        const int channels = TN == 2 && linears.group[g].w_up ? 64 : 64 * TN;
        prm.first_tile[g + 1] = prm.first_tile[g] + (linears.group[g].n + channels - 1) / channels;
    }
    const dim3 grid(prm.first_tile[linears.groups], (linears.rows + 16 * BT - 1) / (16 * BT));
    if (grid.y > 65535u) return QM_ERR_ARGUMENT;
    constexpr int smem = KS * 2 * 3 * 16 * BT * kF32Step * 2;
    static_assert(smem >= (KS - 1) * TN * BT * kDecThreads * 16, "the shares' sums");
    static std::atomic<bool> raised[kMaxDevices];
    const int32_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(split_linear_kernel<BT, TN, KS>), smem, raised);
    if (rc != QM_OK) return rc;
    hipLaunchKernelGGL((split_linear_kernel<BT, TN, KS>), grid, dim3(kDecThreads * KS), smem, stream, prm);
    return launch_status();
}

int32_t launch_split_linears(const DecLinearParams& given, hipStream_t stream) {
    DecLinearParams linears = given;
    // long reductions first, so that none of them starts late
    std::stable_sort(linears.group, linears.group + linears.groups, [](const DecLinearGroup& a, const DecLinearGroup& b) { return a.k > b.k; });
    bool pair = false, quarters = true;
    int64_t tiles64 = 0, tiles128 = 0;                             // of 64 and of 128 weight rows
    for (int g = 0; g < linears.groups; ++g) {
        const DecLinearGroup& d = linears.group[g];
        pair = pair || d.w_up;
        quarters = quarters && d.k % 256 == 0;
        tiles64 += (d.n + 63) / 64;
        tiles128 += d.w_up ? d.n / 64 : (d.n + 127) / 128;
    }
    const int64_t rows32 = (linears.rows + 31) / 32, rows64 = (linears.rows + 63) / 64;
    // A block's time is its chain of steps (0.5 to 1.2 us each, the longer the more rows it splits), so few blocks take small
    // tiles and share the reduction among up to four groups of waves; many blocks take large tiles, which read less.
    // Measured, 1024 inputs to 5120 outputs and 3072 pairs at 16 / 40 / 100 / 300 / 512 rows: <1,2,2> 12 / 21, <2,2,2> 14 / 14 / 26 / 50,
    // <4,2,2> 18 / 19 / 20 / 38 / 56, <4,2,1> 24 / 24 / 25 / 36 / 55 us; 1024, 1024 and 3072 inputs to 1024 outputs each: <1,1,4> 19 / 19 / 27 / 52,
    // <2,1,4> 20 / 21 / 21 / 38 / 52, <2,1,2> 23 / 23 / 23 / 30 / 51, <2,1,1> 36 / 36 / 36 / 40 / 46, <4,2,1> 65 / 66 / 66 / 67 / 68 us.
    if (pair) {
        if (linears.rows <= 16) return launch_split_as<1, 2, 2>(linears, stream);
        if (tiles128 * rows32 <= 256) return launch_split_as<2, 2, 2>(linears, stream);
        return tiles128 * rows64 <= 256 ? launch_split_as<4, 2, 2>(linears, stream) : launch_split_as<4, 2, 1>(linears, stream);
    }
    if (linears.rows <= 16) return quarters ? launch_split_as<1, 1, 4>(linears, stream) : launch_split_as<1, 1, 2>(linears, stream);
    if (quarters && tiles64 * rows32 <= 256) return launch_split_as<2, 1, 4>(linears, stream);
    if (tiles64 * rows32 <= 512) return launch_split_as<2, 1, 2>(linears, stream);
    return tiles64 * rows32 <= 1024 ? launch_split_as<2, 1, 1>(linears, stream) : launch_split_as<4, 2, 1>(linears, stream);
}

}  // namespace qm
