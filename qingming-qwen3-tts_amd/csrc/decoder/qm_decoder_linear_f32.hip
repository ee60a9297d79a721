// qm_decoder_linear_f32.hip — linears of the 32-bit mode over several token rows on the bf16 matrix cores (gfx950).
//
// An fp32 input of at least 2^-110 is the exact sum of three bf16 numbers (its upper eight significant bits, the next eight, the
// last eight: splitting a number over several narrow products is the common way to a wide product on narrow matrix cores) and the
// weights are bf16 as they are, so three bf16 products with fp32 accumulation form what fp32 products form: every product is exact.
// Of a smaller input what lies under 2^-133 is lost, so outputs so small that it could tell are formed again in fp32.  The sums are
// taken in two levels — 64 terms, the smallest parts first, then those sums one after the other — which keeps the chains of
// roundings as short as a wave's lanes keep them in the dot-product kernel.
//
// Two kernels: few blocks or short reductions split the inputs in the blocks (as follows), a long prompt's are split once beforehand (the second part).
//
// A block of four waves takes 16 BT token rows and 64 TN weight rows (a gate/up pair: 32 TN channels, gate and up rows in the
// same lanes), 64 k a step.  Weights are a wave's own and go straight to its registers, requested two steps ahead, a row's
// 64 bytes per instruction; inputs are read once per block, split by the threads that fetched them and shared through two
// LDS stages (a row's 16-byte pieces swizzled over the banks).  Bound: three times the bf16 matrix-core flops of the shape.
#include <algorithm>
#include <utility>

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

// What launch_split_linears takes: 16 ROWS token rows and 64 WEIGHTS weight rows a block, the reduction shared among SHARES groups of waves.
struct SplitShape {
    int rows, weights, shares;
};
static SplitShape split_shape(const DecLinearParams& linears) {
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
        if (linears.rows <= 16) return {1, 2, 2};
        if (tiles128 * rows32 <= 256) return {2, 2, 2};
        return {4, 2, tiles128 * rows64 <= 256 ? 2 : 1};
    }
    if (linears.rows <= 16) return {1, 1, quarters ? 4 : 2};
    if (quarters && tiles64 * rows32 <= 256) return {2, 1, 4};
    if (tiles64 * rows32 <= 512) return {2, 1, 2};
    return tiles64 * rows32 <= 1024 ? SplitShape{2, 1, 1} : SplitShape{4, 2, 1};
}

int32_t launch_split_linears(const DecLinearParams& given, hipStream_t stream) {
    DecLinearParams linears = given;
    // long reductions first, so that none of them starts late
    std::stable_sort(linears.group, linears.group + linears.groups, [](const DecLinearGroup& a, const DecLinearGroup& b) { return a.k > b.k; });
    const SplitShape shape = split_shape(linears);
    if (shape.weights == 2) {
        if (shape.rows == 1) return launch_split_as<1, 2, 2>(linears, stream);
        if (shape.rows == 2) return launch_split_as<2, 2, 2>(linears, stream);
        return shape.shares == 2 ? launch_split_as<4, 2, 2>(linears, stream) : launch_split_as<4, 2, 1>(linears, stream);
    }
    if (shape.rows == 1) return shape.shares == 4 ? launch_split_as<1, 1, 4>(linears, stream) : launch_split_as<1, 1, 2>(linears, stream);
    if (shape.shares == 4) return launch_split_as<2, 1, 4>(linears, stream);
    return shape.shares == 2 ? launch_split_as<2, 1, 2>(linears, stream) : launch_split_as<2, 1, 1>(linears, stream);
}

// ---- inputs split beforehand ---------------------------------------------------------------------------------------------
// With memory for them the inputs' three parts are made once, as planes of bf16, and the linears become three bf16 products of the same
// weights: above, every block of a row's 64 or 88 column tiles splits the row anew (its threads' 20 vector instructions an element are as long as
// its products), and weights go to registers in a matrix operand's order, which the address path takes one lane a cycle.
//
// A block of four waves takes 64 token rows and BN weight rows (a pair: BN / 2 channels, a wave's gate and up rows side by side), 64 k a step, both
// operands by buffer_load ... lds into rings of stages (planes two or three, weights one more, since they come from further away).  Of 256 weight rows
// a wave takes 64 for all token rows, of 128 for 32 of them; a step's 56 KiB (40) are as long in the address path (46 bytes a cycle) as its matrix
// instructions (1536 cycles, 768).  The parts below the first gather in sums of their own, whose roundings lie 2^-8 lower, and the first's in two
// levels of 128 terms, added while the last of the lower parts are multiplied.  A step's one barrier stands in front of its last k block.
constexpr int kPlaneLinears = kDecGroups + kMorePlanes;

struct PlaneLinear {
    const uint16_t* x;             // [3][x_plane]: this linear's columns of the planes' rows
    const float* x32;              // the same as they were
    const uint16_t* w;
    const uint16_t* w_up;
    float* out;
    int x_plane, ldx32, ldo, n, k, pitch;    // k: of this piece; pitch: of planes and weights
};
struct PlaneLinearsParams {
    PlaneLinear linear[kPlaneLinears];
    int first_tile[kPlaneLinears + 1];       // column tiles in front of each
    int linears, rows;
};

struct PlaneInput {
    const float* x;
    uint16_t* planes;              // [3][rows][k]
    int64_t ldx;
    int k;
};
struct SplitRowsParams {
    PlaneInput input[kDecGroups];
    int first_block[kDecGroups];             // along a row, kSplitColumns each
    int inputs, rows;
};
constexpr int kSplitThreads = 64, kSplitColumns = 8 * kSplitThreads;
__global__ __launch_bounds__(kSplitThreads) void split_rows_kernel(SplitRowsParams prm) {
    request_arguments(prm);
    const int row = static_cast<int>(blockIdx.x);                  // (a grid is higher than 65535 in its first dimension only)
    int which = 0;
    while (which + 1 < prm.inputs && static_cast<int>(blockIdx.y) >= prm.first_block[which + 1]) ++which;
    const PlaneInput& in = prm.input[which];
    const int c = (static_cast<int>(blockIdx.y) - prm.first_block[which]) * kSplitColumns + 8 * threadIdx.x;
    if (c >= in.k) return;
    const float* from = in.x + row * in.ldx + c;
    const float4 a = *reinterpret_cast<const float4*>(from), b = *reinterpret_cast<const float4*>(from + 4);
    float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int part = 0; part < 3; ++part) {
        uint32_t upper[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) upper[e] = part < 2 ? take_upper(v[e]) : __float_as_uint(v[e]);
        split_u32x4_t packed;
#pragma unroll
        for (int e = 0; e < 4; ++e) packed[e] = __builtin_amdgcn_perm(upper[2 * e + 1], upper[2 * e], 0x07060302U);
        *reinterpret_cast<split_u32x4_t*>(in.planes + (static_cast<int64_t>(part) * prm.rows + row) * in.k + c) = packed;
    }
}

typedef float plane_f32x16_t __attribute__((ext_vector_type(16)));

template <int BN>
struct PlaneShape {
    static constexpr int kAcross = BN == 256 ? 4 : 2, kTm = kAcross / 2;       // waves along the weight rows; a wave's 32-row tiles (and two of 32 weight rows)
    static constexpr int kXStages = BN == 256 ? 2 : 3, kWStages = kXStages + 1;
    static constexpr int kPlane = kPlaneRows * 128, kXBytes = 3 * kPlane, kWBytes = BN * 128;
    static constexpr int kLds = kXStages * kXBytes + kWStages * kWBytes;
    static constexpr int kXEach = kXBytes / 4096, kWEach = kWBytes / 4096;     // requests of a wave per stage
};
template <int TM>
struct PlaneFrags {
    split_u32x4_t w[2], x[3][TM];
};
template <int OFFSET>
__device__ __forceinline__ void plane_read(split_u32x4_t& to, uint32_t at) { asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(at), "n"(OFFSET)); }
// fragment N of a k block, in the order of use
template <int N, int TM>
__device__ __forceinline__ void plane_read_nth(PlaneFrags<TM>& f, uint32_t x_at, uint32_t w_at) {
    if constexpr (N == 0) plane_read<0>(f.w[0], w_at);
    else if constexpr (N <= TM) plane_read<4096 * (N - 1)>(f.x[0][N - 1], x_at);
    else if constexpr (N == TM + 1) plane_read<4096>(f.w[1], w_at);
    else if constexpr (N < 2 + 3 * TM) plane_read<kPlaneRows * 128 * ((N - 2) / TM) + 4096 * ((N - 2) % TM)>(f.x[(N - 2) / TM][(N - 2) % TM], x_at);
}
__device__ __forceinline__ void plane_arrived(PlaneFrags<1>& f) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.w[0]), "+v"(f.w[1]), "+v"(f.x[0][0]), "+v"(f.x[1][0]), "+v"(f.x[2][0])::"memory");
}
__device__ __forceinline__ void plane_arrived(PlaneFrags<2>& f) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.w[0]), "+v"(f.w[1]), "+v"(f.x[0][0]), "+v"(f.x[1][0]), "+v"(f.x[2][0]), "+v"(f.x[0][1]), "+v"(f.x[1][1]),
                 "+v"(f.x[2][1])::"memory");
}
template <int LATER>
__device__ __forceinline__ void plane_landed() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LATER) : "memory"); }
template <class F, int... I>
__device__ __forceinline__ void plane_each_of(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void plane_each(F&& f) { plane_each_of(f, std::make_integer_sequence<int, N>{}); }

template <int BN>
__global__ __launch_bounds__(kDecThreads, 1) void plane_linear_kernel(PlaneLinearsParams prm) {
    using Shape = PlaneShape<BN>;
    request_large_argument(prm);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];      // x [kXStages][3][64][128 bytes], w [kWStages][BN][128 bytes]
    constexpr int kTm = Shape::kTm;
    const int lane = threadIdx.x & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave_n = wave % Shape::kAcross, wave_m = wave / Shape::kAcross;
    // linear by linear, the long reductions first
    const int row_tiles = static_cast<int>(gridDim.y);
    int at = static_cast<int>(blockIdx.y * gridDim.x + blockIdx.x), which = 0;
    while (which + 1 < prm.linears && at >= prm.first_tile[which + 1] * row_tiles) ++which;
    at -= prm.first_tile[which] * row_tiles;
    const int across = prm.first_tile[which + 1] - prm.first_tile[which];
    const PlaneLinear& linear = prm.linear[which];
    const int row0 = at / across * kPlaneRows, tile = at % across;
    const int k = linear.k, pitch = linear.pitch, rows = prm.rows;
    const bool pair = linear.w_up != nullptr;
    const int first = tile * (pair ? BN / 2 : BN);                 // weight row or channel

    // ---- requests: 8 rows of 128 bytes an instruction, lane l slot l % 8 of row l / 8, where piece (l % 8) ^ (row / 2 % 8) stands; a wave's rows are 8 wave + 32 i ----
    const uint32_t lane_off = static_cast<uint32_t>((8 * wave + (lane >> 3)) * pitch * 2 + 16 * ((lane & 7) ^ ((4 * wave + (lane >> 4)) & 7)));
    const uint32_t rows32 = static_cast<uint32_t>(32 * pitch * 2);
    auto rows_from = [&](const uint16_t* from, int count) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(from), 0, ((count - 1) * pitch + k) * 2, 0x00020000);
    };
    const int x_rows = min(rows - row0, kPlaneRows), w_rows = min(linear.n - first, pair ? BN / 2 : BN);
    const uint16_t* const x_first = linear.x + static_cast<int64_t>(row0) * pitch;
    const __amdgpu_buffer_rsrc_t x_rsrc[3] = {rows_from(x_first, x_rows), rows_from(x_first + linear.x_plane, x_rows), rows_from(x_first + 2 * static_cast<int64_t>(linear.x_plane), x_rows)};
    const __amdgpu_buffer_rsrc_t w_rsrc = rows_from(linear.w + static_cast<int64_t>(first) * pitch, w_rows);
    const __amdgpu_buffer_rsrc_t u_rsrc = rows_from((pair ? linear.w_up : linear.w) + static_cast<int64_t>(first) * pitch, w_rows);
    const int steps = k / kF32Step;                                // (even)
    unsigned char* const x_lds = smem + 1024 * wave;
    unsigned char* const w_lds = x_lds + Shape::kXStages * Shape::kXBytes;
    // (requests past the last step repeat it, into stages that nobody reads again: the waits count them)
    auto request_x = [&](int step, int i) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x_rsrc[i / 2], (__attribute__((address_space(3))) void*)(x_lds + step % Shape::kXStages * Shape::kXBytes + 4096 * i), 16,
                                                 static_cast<int>(lane_off + i % 2 * rows32), min(step, steps - 1) * 128, 0, 0);
    };
    auto request_w = [&](int step, int i) __attribute__((always_inline)) {
        const uint32_t off = lane_off + static_cast<uint32_t>(pair ? i / 2 : i) * rows32;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(pair && i % 2 ? u_rsrc : w_rsrc, (__attribute__((address_space(3))) void*)(w_lds + step % Shape::kWStages * Shape::kWBytes + 4096 * i), 16,
                                                 static_cast<int>(off), min(step, steps - 1) * 128, 0, 0);
    };
    // request N of those that follow a step's barrier: planes, then weights
    auto request = [&](int step, auto n) __attribute__((always_inline)) {
        constexpr int N = decltype(n)::value;
        if constexpr (N < Shape::kXEach) request_x(step + Shape::kXStages, N);
        else if constexpr (N < Shape::kXEach + Shape::kWEach) request_w(step + Shape::kWStages, N - Shape::kXEach);
    };

    // ---- fragments: lane's row lane % 32 of a tile, piece 2 kb + half ----
    const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)smem));
    uint32_t x_kb[4], w_kb[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        const uint32_t in_tile = static_cast<uint32_t>((lane & 31) * 128 + 16 * ((2 * kb + half) ^ ((lane >> 1) & 7)));
        x_kb[kb] = lds_base + in_tile + static_cast<uint32_t>(wave_m * 4096);
        w_kb[kb] = lds_base + in_tile + static_cast<uint32_t>(Shape::kXStages * Shape::kXBytes + wave_n * 8192);
    }

    plane_f32x16_t sum[2][kTm], part[2][kTm], low[2][kTm];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < kTm; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[a][b][r] = low[a][b][r] = 0.0f;

    constexpr int kTiles = 2 * kTm, kMfmas = 3 * kTiles, kReads = 2 + 3 * kTm, kRequests = Shape::kXEach + Shape::kWEach;
    // The products of one k block from f, between them the reads of the next one's fragments into g (at x_at, w_at), requests [R0, R0 + RN) of `step`, and with FLUSH the
    // first part's sums (which stand first) onto the whole ones.
    auto k_block = [&](PlaneFrags<kTm>& f, PlaneFrags<kTm>& g, uint32_t x_at, uint32_t w_at, int step, auto fresh, auto flush, auto r0, auto rn) __attribute__((always_inline)) {
        constexpr int R0 = decltype(r0)::value, RN = decltype(rn)::value;
        plane_each<kMfmas>([&](auto number) __attribute__((always_inline)) {
            constexpr int S = decltype(number)::value, p = S / kTiles, a = S % kTiles / kTm, b = S % kTm;
            const bf16x8_t w = __builtin_bit_cast(bf16x8_t, f.w[a]), x = __builtin_bit_cast(bf16x8_t, f.x[p][b]);
            if constexpr (p == 0) {
                if constexpr (decltype(fresh)::value) {
                    plane_f32x16_t zero;
#pragma unroll
                    for (int r = 0; r < 16; ++r) zero[r] = 0.0f;
                    part[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, zero, 0, 0, 0);
                } else {
                    part[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, part[a][b], 0, 0, 0);
                }
            } else {
                low[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, x, low[a][b], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (S < kReads) plane_read_nth<S>(g, x_at, w_at);
            // (the requests stand in the later places)
            constexpr int kFrom = RN * S / kMfmas, kTo = RN * (S + 1) / kMfmas;
            if constexpr (kFrom < kTo) request(step, std::integral_constant<int, R0 + kFrom>{});
            if constexpr (kFrom + 1 < kTo) request(step, std::integral_constant<int, R0 + kFrom + 1>{});
            if constexpr (kFrom + 2 < kTo) request(step, std::integral_constant<int, R0 + kFrom + 2>{});
            static_assert(kTo - kFrom <= 3, "listed above");
            if constexpr (decltype(flush)::value && p > 0) {       // eight sums behind each of the other products
                constexpr int kTile = (S - kTiles) / 2, kHalf = (S - kTiles) % 2;
#pragma unroll
                for (int r = 8 * kHalf; r < 8 * kHalf + 8; ++r) sum[kTile / kTm][kTile % kTm][r] += part[kTile / kTm][kTile % kTm][r];
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using std::integral_constant;
    // how many of a step's requests stand in its last k block and in the next step's first three
    constexpr int kIn3 = kRequests * 4 / 14, kIn0 = kRequests * 4 / 14, kIn1 = (kRequests - kIn3 - kIn0 + 1) / 2, kIn2 = kRequests - kIn3 - kIn0 - kIn1;

#pragma unroll
    for (int step = 0; step < Shape::kWStages; ++step) {           // planes 0, weights 0, planes 1, ..
        if (step < Shape::kXStages)
            for (int i = 0; i < Shape::kXEach; ++i) request_x(step, i);
        for (int i = 0; i < Shape::kWEach; ++i) request_w(step, i);
    }
    plane_landed<(Shape::kXStages - 1) * Shape::kXEach + (Shape::kWStages - 1) * Shape::kWEach>();
    asm volatile("s_barrier" ::: "memory");
    PlaneFrags<kTm> f0, f1;
    plane_each<kReads>([&](auto n) { plane_read_nth<decltype(n)::value>(f0, x_kb[0], w_kb[0]); });
    auto one_step = [&](int step, auto odd) __attribute__((always_inline)) {
        constexpr bool ODD = decltype(odd)::value;
        const uint32_t x_at = static_cast<uint32_t>(step % Shape::kXStages * Shape::kXBytes), x_next = static_cast<uint32_t>((step + 1) % Shape::kXStages * Shape::kXBytes);
        const uint32_t w_at = static_cast<uint32_t>(step % Shape::kWStages * Shape::kWBytes), w_next = static_cast<uint32_t>((step + 1) % Shape::kWStages * Shape::kWBytes);
        using no = std::false_type;
        plane_arrived(f0);
        k_block(f0, f1, x_kb[1] + x_at, w_kb[1] + w_at, step - 1, std::integral_constant<bool, !ODD>{}, no{}, integral_constant<int, kIn3>{}, integral_constant<int, kIn0>{});
        plane_arrived(f1);
        k_block(f1, f0, x_kb[2] + x_at, w_kb[2] + w_at, step - 1, no{}, no{}, integral_constant<int, kIn3 + kIn0>{}, integral_constant<int, kIn1>{});
        plane_arrived(f0);
        k_block(f0, f1, x_kb[3] + x_at, w_kb[3] + w_at, step - 1, no{}, no{}, integral_constant<int, kIn3 + kIn0 + kIn1>{}, integral_constant<int, kIn2>{});
        plane_arrived(f1);
        plane_landed<(Shape::kXStages - 2) * Shape::kXEach + (Shape::kWStages - 2) * Shape::kWEach>();   // this wave's pieces of the next step have landed
        asm volatile("s_barrier" ::: "memory");                    // everybody's have; and everybody has read this step's
        k_block(f1, f0, x_kb[0] + x_next, w_kb[0] + w_next, step, no{}, std::integral_constant<bool, ODD>{}, integral_constant<int, 0>{}, integral_constant<int, kIn3>{});
    };
    plane_f32x16_t early[2][kTm];                                  // the first half's sums
    const int middle = steps / 4 * 2;
#pragma unroll 1
    for (int step = 0; step < steps;) {
        const int end = step < middle ? middle : steps;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < kTm; ++b) {
                early[a][b] = sum[a][b];
#pragma unroll
                for (int r = 0; r < 16; ++r) sum[a][b][r] = 0.0f;
            }
        for (; step < end; step += 2) {
            one_step(step, std::false_type{});
            one_step(step + 1, std::true_type{});
        }
    }
    plane_arrived(f0);               // (what was read and asked for past the last step)
    plane_landed<0>();

    // ---- outputs: a lane holds columns 8 (r / 4) + 4 half + r % 4 of a tile's 32 for token row lane % 32; through LDS they leave as whole rows ----
    bool good = true;
#pragma unroll
    for (int b = 0; b < kTm; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            sum[0][b][r] = early[0][b][r] + (sum[0][b][r] + low[0][b][r]);
            sum[1][b][r] = early[1][b][r] + (sum[1][b][r] + low[1][b][r]);
            if (pair) {
                sum[0][b][r] = silu_f32(sum[0][b][r]) * sum[1][b][r];
                good = good && sum[0][b][r] == sum[0][b][r];
            } else {
                good = good && (fabsf(sum[0][b][r]) >= kF32Small || sum[0][b][r] == 0.0f) && (fabsf(sum[1][b][r]) >= kF32Small || sum[1][b][r] == 0.0f);
            }
        }
    asm volatile("s_barrier" ::: "memory");
    auto leave = [&](auto columns_, int from) __attribute__((always_inline)) {
        constexpr int kColumns = decltype(columns_)::value, kPitch = kColumns * 4 + 16, kChunks = kColumns / 4;
        static_assert(kPlaneRows * kPitch <= Shape::kLds, "the tile's outputs");
#pragma unroll
        for (int a = 0; a < kColumns * 2 / BN; ++a)
#pragma unroll
            for (int b = 0; b < kTm; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    *reinterpret_cast<float4*>(smem + (32 * (kTm * wave_m + b) + (lane & 31)) * kPitch + 4 * (kColumns / Shape::kAcross * wave_n + 32 * a + 8 * g + 4 * half)) =
                        make_float4(sum[a][b][4 * g], sum[a][b][4 * g + 1], sum[a][b][4 * g + 2], sum[a][b][4 * g + 3]);
        __syncthreads();
#pragma unroll 4
        for (int i = threadIdx.x; i < kPlaneRows * kChunks; i += kDecThreads) {
            const int row = i / kChunks, column = 4 * (i % kChunks);
            if (row < x_rows && column < w_rows)
                *reinterpret_cast<float4*>(linear.out + static_cast<int64_t>(row0 + row) * linear.ldo + from + column) = *reinterpret_cast<const float4*>(smem + row * kPitch + 4 * column);
        }
    };
    if (pair) leave(integral_constant<int, BN / 2>{}, first);
    else leave(integral_constant<int, BN>{}, first);
    // Outputs that are no number, or small (see above), are formed again from the inputs as they are, once the block's stores are out.
    if (!__syncthreads_or(!good)) return;
    if (good) return;
#pragma unroll 1
    for (int i = 0; i < 16 * kTm * (pair ? 1 : 2); ++i) {
        const int row = row0 + 32 * (kTm * wave_m + i / 16 % kTm) + (lane & 31);
        const int channel = first + (pair ? 32 : 64) * wave_n + 32 * (i / (16 * kTm)) + 8 * (i % 16 / 4) + 4 * half + i % 4;
        if (row >= rows || channel >= linear.n) continue;
        float* const at_output = linear.out + static_cast<int64_t>(row) * linear.ldo + channel;
        if (pair ? *at_output == *at_output : fabsf(*at_output) >= kF32Small) continue;
        const float* const x_row = linear.x32 + static_cast<int64_t>(row) * linear.ldx32;
        const int64_t w_row = static_cast<int64_t>(channel) * pitch;
        const float gate = plain_dot(x_row, linear.w + w_row, k);
        *at_output = pair ? silu_f32(gate) * plain_dot(x_row, linear.w_up + w_row, k) : gate;
    }
}

template <int BN>
static int32_t launch_planes_as(PlaneLinearsParams& prm, hipStream_t stream) {
    for (int i = 0; i < prm.linears; ++i) {
        const int columns = prm.linear[i].w_up ? BN / 2 : BN;
        prm.first_tile[i + 1] = prm.first_tile[i] + (prm.linear[i].n + columns - 1) / columns;
    }
    const dim3 grid(prm.first_tile[prm.linears], (prm.rows + kPlaneRows - 1) / kPlaneRows);
    if (grid.y > 65535u) return QM_ERR_ARGUMENT;
    static std::atomic<bool> raised[kMaxDevices];
    const int32_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(plane_linear_kernel<BN>), PlaneShape<BN>::kLds, raised);
    if (rc != QM_OK) return rc;
    hipLaunchKernelGGL(plane_linear_kernel<BN>, grid, dim3(kDecThreads), PlaneShape<BN>::kLds, stream, prm);
    return launch_status();
}

// A linear's blocks of BN weight rows and 64 token rows.
static int64_t plane_blocks(const DecLinearGroup& d, int rows, int bn) {
    return (static_cast<int64_t>(d.n) * (d.w_up ? 2 : 1) + bn - 1) / bn * ((rows + kPlaneRows - 1) / kPlaneRows);
}
// The busiest CU's steps with blocks of bn weight rows; what a block takes beside its steps is as long as four of them.
static int64_t plane_steps(const DecLinearParams& prm, int pieces, int bn) {
    int64_t count[kDecGroups], steps[kDecGroups];
    for (int g = 0; g < prm.groups; ++g) {
        const int cut = g == prm.groups - 1 ? pieces : 1;
        count[g] = plane_blocks(prm.group[g], prm.rows, bn) * cut;
        steps[g] = prm.group[g].k / kF32Step / cut + 4;
    }
    return steps_of_busiest_cu(prm.groups, count, steps);
}

int64_t plane_elements(const DecLinearParams& prm) {
    int64_t k = 0;
    for (int g = 0; g < prm.groups; ++g) {
        bool known = false;
        for (int before = 0; before < g; ++before) known = known || (prm.group[before].x == prm.group[g].x && prm.group[before].k == prm.group[g].k && prm.group[before].ldx == prm.group[g].ldx);
        if (!known) k += prm.group[g].k;
    }
    return 3 * k * prm.rows;
}

// (us, 1024 outputs each of 1024, 1024 and 3072 inputs, in one, two and three pieces: 100 rows 34 / 23 / 20, 300 rows 37 / 27 / 25, 400 rows 39 / 30 / 37, 512 rows
// 40 / 33 / 39, 1024 rows 52 / 56 / 60.)  A piece more is a plane of sums written and read: a step's time (0.45 us) for each 2 MB.
int plane_pieces(const DecLinearParams& prm) {
    const DecLinearGroup& last = prm.group[prm.groups - 1];
    if (prm.groups < 2 || last.w_up || last.ldo != last.n) return 1;
    int best = 1;
    int64_t least = plane_steps(prm, 1, 128);
    for (int parts = 2; parts <= 1 + kMorePlanes; ++parts) {
        if (last.k % (128 * parts)) continue;
        const int64_t steps = plane_steps(prm, parts, 128) + (parts - 1) * (static_cast<int64_t>(prm.rows) * last.n * 8 / 2000000 + 1);
        if (steps < least) {
            least = steps;
            best = parts;
        }
    }
    return best;
}

// What the kernel's 32-bit offsets and its vectors of four take.
bool planes_fit(const DecLinearParams& prm) {
    for (int g = 0; g < prm.groups; ++g) {
        const DecLinearGroup& d = prm.group[g];
        const uintptr_t at = reinterpret_cast<uintptr_t>(d.x) | reinterpret_cast<uintptr_t>(d.w) | reinterpret_cast<uintptr_t>(d.w_up) |
                             reinterpret_cast<uintptr_t>(d.w_up ? d.out : d.out32);
        if ((at & 15) || d.k > (1 << 20) || static_cast<int64_t>(prm.rows) * d.k > (int64_t{1} << 28) || d.ldx > INT32_MAX || d.ldo > INT32_MAX) return false;
    }
    return true;
}

// Whether planes end first, and no linear of the launch comes out further from 64 bits.  A plane's sums are the same whatever the grid; those of
// launch_split_linears are the closer the more groups of waves share a reduction, so that the shortest one decides.  (Relative error x 1e8, split in the blocks /
// beforehand.  One walks it all: 1024 inputs 9.15 / 7.92, 512 7.34 / 7.33, 384 6.79 / 7.23; two groups: 1024 7.94 / 7.92, 896 7.69 / 7.83, pairs of them 13.0 / 12.9
// and 12.7 / 12.8; four: 3072 9.63 / 9.57, 2560 9.15 / 9.21, 1024 7.54 / 7.92.)  The launch that splits is 4 to 7 us, so that planes end first where no groups share,
// or where they do and the reduction is long and can be cut or has many blocks (us, split in the blocks / beforehand: 5120 outputs of 1024 inputs beside 3072 pairs,
// 100, 200, 300, 512 and 1024 rows 20.8 / 17.9, 34.6 / 27.8, 38.5 / 30.8, 59 / 50, 108 / 83; the three linears above, the last one cut, 300 rows 30.1 / 25.0, 512
// 46 / 40; 4096 of 4096, 300 rows 79.7 / 49.2; those that stay: 1024 of 1024, 300 rows 9.7 / 17.7, 2048 of 2048, 300 rows 25.9 / 27.5, 2048 of 512, 1024 rows 16.4 /
// 18.1, and, for their shorter reductions, the three at 100 rows 21.5 / 20.5).
bool planes_pay(const DecLinearParams& prm, int pieces) {
    if (prm.rows <= 16 || !planes_fit(prm)) return false;
    int longest = 0, shortest = prm.group[0].k;
    int64_t tiles64 = 0;
    bool pair = false;
    for (int g = 0; g < prm.groups; ++g) {
        const DecLinearGroup& d = prm.group[g];
        longest = std::max(longest, d.k);
        shortest = std::min(shortest, d.k);
        tiles64 += (d.n + 63) / 64;
        pair = pair || d.w_up;
    }
    const SplitShape shape = split_shape(prm);
    if (longest < 768 || shortest < (shape.shares == 4 ? 3072 : shape.shares == 2 ? 1024 : 512)) return false;
    if (pair) return shape.rows == 4;
    return shape.shares == 1 || (longest >= 3072 && (pieces > 1 || tiles64 * ((prm.rows + 31) / 32) > 256));
}

int32_t launch_plane_linears(const DecLinearParams& given, const PlaneMemory& memory, hipStream_t stream, ReductionCut* cut) {
    uint16_t* planes = memory.at;
    SplitRowsParams split = {};
    split.rows = given.rows;
    PlaneLinear all[kPlaneLinears] = {};
    int count = given.groups;
    for (int g = 0; g < given.groups; ++g) {
        const DecLinearGroup& d = given.group[g];
        int input = 0;
        while (input < split.inputs && (split.input[input].x != d.x || split.input[input].ldx != d.ldx || split.input[input].k != d.k)) ++input;
        if (input == split.inputs) {
            split.input[split.inputs++] = {static_cast<const float*>(d.x), planes, d.ldx, d.k};
            planes += 3 * static_cast<int64_t>(given.rows) * d.k;
        }
        all[g] = {split.input[input].planes, static_cast<const float*>(d.x), d.w, d.w_up, d.w_up ? static_cast<float*>(d.out) : d.out32,
                  given.rows * d.k, static_cast<int>(d.ldx), static_cast<int>(d.ldo), d.n, d.k, d.k};
    }
    if (cut) {
        PlaneLinear& last = all[count - 1];
        cut->plane = static_cast<int64_t>(given.rows) * last.n;
        int pieces = plane_pieces(given);
        if ((pieces - 1) * cut->plane > cut->room) pieces = 1;
        last.k /= pieces;
        for (; cut->planes < pieces - 1; ++cut->planes, ++count) {
            const int64_t at = (cut->planes + 1) * static_cast<int64_t>(last.k);
            all[count] = last;
            all[count].x += at;
            all[count].x32 += at;
            all[count].w += at;
            all[count].out = cut->sums + cut->planes * cut->plane;
            all[count].ldo = last.n;
        }
    }
    PlaneLinearsParams prm = {};
    prm.linears = count;
    prm.rows = given.rows;
    std::copy(all, all + count, prm.linear);
    std::stable_sort(prm.linear, prm.linear + count, [](const PlaneLinear& a, const PlaneLinear& b) { return a.k > b.k; });    // (long reductions first)
    int blocks = 0;
    for (int i = 0; i < split.inputs; ++i) {
        split.first_block[i] = blocks;
        blocks += (split.input[i].k + kSplitColumns - 1) / kSplitColumns;
    }
    if (!memory.split || split.inputs != 1) {
        hipLaunchKernelGGL(split_rows_kernel, dim3(given.rows, blocks), dim3(kSplitThreads), 0, stream, split);
        const int32_t rc = launch_status();
        if (rc != QM_OK) return rc;
    }
    // Wide blocks read less for their products; a step of theirs is as long as 1.75 of the others'.
    const int pieces = cut ? cut->planes + 1 : 1;
    return 7 * plane_steps(given, pieces, 256) < 4 * plane_steps(given, pieces, 128) ? launch_planes_as<256>(prm, stream) : launch_planes_as<128>(prm, stream);
}

}  // namespace qm
