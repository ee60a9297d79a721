// qm_decoder_linear.hip — linears of the decoder language models for few token rows (a decode step, a short portion of a
// prompt): weight-streaming dot products; many rows are handed to the matrix-core kernels (bf16, and the 32-bit mode's).
//
// Bound by HBM: every weight is read once per group of R rows.  A wave owns NR weight rows and streams them 16 bytes a
// lane, `kDotAhead` pieces of each row requested before the first is used; the input rows live in LDS as T.  Sums are fp32
// (packed bf16 dot products, or fmaf in the 32-bit mode), combined over the wave's lanes at the end.
#include <algorithm>
#include <map>
#include <numeric>
#include <vector>

#include "qm_decoder_device.h"
#include "../qm_host.h"
#include "../qm_linear_rows_params.h"
#include "qm_decoder_dot.h"

namespace qm {

constexpr int kLinearRows = 4;                 // weight rows a wave streams at once

template <class T, int R>
__global__ __launch_bounds__(kDecThreads) void decoder_linear_kernel(DecLinearParams prm) {
    request_arguments(prm);
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    T* xs = reinterpret_cast<T*>(smem);
    int tile = static_cast<int>(blockIdx.x);
    const DecLinearGroup& group = prm.group[dot_group<kLinearRows>(prm, tile)];
    const int row0 = static_cast<int>(blockIdx.y) * R;
    const int rows = min(R, prm.rows - row0);
    const int k = group.k;
    const auto d = dot_rows<kLinearRows>(group, tile);
    uint4 piece[kDotAhead][kLinearRows];
    dot_request(d, k, piece);
    constexpr int kVec = 16 / sizeof(T);
    for (int r = 0; r < R; ++r) {
        const int src = row0 + min(r, rows - 1);               // (a row past the end repeats the last one, never stored)
        const T* x = static_cast<const T*>(group.x) + src * group.ldx;
        for (int c = threadIdx.x * kVec; c < k; c += kDecThreads * kVec)
            *reinterpret_cast<uint4*>(xs + r * k + c) = *reinterpret_cast<const uint4*>(x + c);
    }
    __syncthreads();
    dot_finish<T, R>(group, d, piece, xs, row0, rows);
}

template <class T, int R>
static int32_t launch_streaming(const DecLinearParams& prm, hipStream_t stream) {
    int k = 0;
    for (int g = 0; g < prm.groups; ++g) k = prm.group[g].k > k ? prm.group[g].k : k;
    const int tiles = dot_tiles_of<kLinearRows>(prm);
    static std::atomic<bool> raised[kMaxDevices];
    const int32_t rc = ensure_dynamic_lds(reinterpret_cast<const void*>(decoder_linear_kernel<T, R>), kDotLdsMost, raised);
    if (rc != QM_OK) return rc;
    hipLaunchKernelGGL((decoder_linear_kernel<T, R>), dim3(tiles, (prm.rows + R - 1) / R), dim3(kDecThreads), sizeof(T) * R * k, stream, prm);
    return launch_status();
}

template <class T>
static int64_t longest_row_bytes(const DecLinearParams& prm) {
    int k = 0;
    for (int g = 0; g < prm.groups; ++g) k = prm.group[g].k > k ? prm.group[g].k : k;
    return static_cast<int64_t>(k) * sizeof(T);
}
// Token rows that a block of the dot products takes (0: a row does not fit its LDS).
static int streaming_rows(int rows, int64_t row_bytes) {
    if (row_bytes > kDotLds) return 0;
    if (rows > 4 && 8 * row_bytes <= kDotLds) return 8;
    if (rows > 2 && 4 * row_bytes <= kDotLds) return 4;
    return rows > 1 && 2 * row_bytes <= kDotLds ? 2 : 1;
}
template <class T>
static int32_t streaming(const DecLinearParams& prm, hipStream_t stream) {
    switch (streaming_rows(prm.rows, longest_row_bytes<T>(prm))) {
        case 8: return launch_streaming<T, 8>(prm, stream);
        case 4: return launch_streaming<T, 4>(prm, stream);
        case 2: return launch_streaming<T, 2>(prm, stream);
        case 1: return launch_streaming<T, 1>(prm, stream);
        default: return QM_ERR_GEOMETRY;
    }
}

// A linear of few columns (a router) over many bf16 rows: the large tiles of the matrix-core kernel would leave most CUs
// without a block and walk the whole reduction one step after the other.  Here a block takes 16 rows, its four waves every
// fourth 128 terms of the reduction (v_mfma_f32_16x16x32_bf16, operands straight from memory; the weights are few and stay in
// L2), and the four sums meet in LDS.  Bound by the latency of a wave's loads.
constexpr int kNarrowRows = 16;                        // token rows of a block
constexpr int kNarrowColumns = 64;                     // most columns
template <int TILES>
__global__ __launch_bounds__(kDecThreads) void narrow_linear_kernel(DecLinearGroup group, int rows) {
    __shared__ float sums[4][TILES * 16 * (kNarrowRows + 1)];
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, l16 = lane & 15;
    const int row0 = static_cast<int>(blockIdx.x) * kNarrowRows;
    const uint16_t* x = static_cast<const uint16_t*>(group.x) + min(row0 + l16, rows - 1) * group.ldx + 8 * g;
    const uint16_t* w[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) w[t] = group.w + static_cast<int64_t>(min(16 * t, group.n - 16) + l16) * group.k + 8 * g;
    f32x4_t acc[TILES] = {};
    for (int k = wave * 128; k < group.k; k += 512) {  // (all of 128 terms is asked for before the first is used)
        u32x4 b[4], a[4][TILES];
#pragma unroll
        for (int u = 0; u < 4; ++u) b[u] = *reinterpret_cast<const u32x4*>(x + k + 32 * u);
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u][t] = *reinterpret_cast<const u32x4*>(w[t] + k + 32 * u);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int t = 0; t < TILES; ++t)
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[u][t]), __builtin_bit_cast(bf16x8_t, b[u]), acc[t], 0, 0, 0);
    }
    // acc[t][r] is column 16 t + 4 g + r of row l16
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) sums[wave][(16 * t + 4 * g + r) * (kNarrowRows + 1) + l16] = acc[t][r];
    __syncthreads();
    for (int i = threadIdx.x; i < kNarrowRows * TILES * 16; i += kDecThreads) {
        const int row = i / (TILES * 16), c = i % (TILES * 16), at = c * (kNarrowRows + 1) + row;
        if (row0 + row < rows && c < group.n)
            group.out32[static_cast<int64_t>(row0 + row) * group.ldo + c] = (sums[0][at] + sums[1][at]) + (sums[2][at] + sums[3][at]);
    }
}
template <int TILES>
static int32_t launch_narrow(const DecLinearParams& prm, hipStream_t stream) {
    hipLaunchKernelGGL(narrow_linear_kernel<TILES>, dim3((prm.rows + kNarrowRows - 1) / kNarrowRows), dim3(kDecThreads), 0, stream, prm.group[0], prm.rows);
    return launch_status();
}

// Rows from which bf16 goes to the matrix cores.  Below, one tile is mostly empty, and a pair's gate and up would be rounded to bf16
// before their product, where the dot products keep them in fp32 and round once: up to 15 rows the results are the dot products',
// whatever rows go together.  (The matrix cores would end earlier from nine rows on, and from five where a reduction is long: us, dot
// products / matrix cores, inputs 10240 + 2 x 6144 by 2048 of 9 / 15 rows 43 / 44 against 28 to 29.)
constexpr int kDecMatrixRows = 16;

// Whether fp32 rows go to the matrix cores: up to eight rows every weight is streamed once either way, and below about 2^26 products
// the dot-product kernel's many short chains end first (us, dot products / matrix cores; products in millions: router 32 x 1024 of 1000
// rows 33: 7.9 / 8.8; 320 x 1024 of 100 rows 33: 7.2 / 8.9; 1024 x 1024 of 64 rows 67: 7.9 / 9.0, of 100 rows 105: 13.4 / 9.2, of 300
// rows 315: 28.7 / 9.6; 5120 + 2 x 3072 by 1024 of 8 rows 92: 12.3 / 11.5, of 300 rows 3460: 224 / 36).  Beyond, the matrix cores' time
// is one block's chain while the dot products' grows with their rounds of blocks, so that long reductions to few columns stay with
// those as long as they fit a round or two (1024 x 3072 of 32 / 33 rows 15.1 / 20.7 and 23.5 / 20.8; 2048 x 6144 of 16 / 17 rows 31.6 /
// 33.4 and 42.3 / 36.3; 2048 x 2048 of 32 / 33 rows 13.2 / 14.4 and 18.5 / 14.3).  Both in tenths of a microsecond, as measured.
static bool split_pays(const DecLinearParams& prm) {
    const int64_t row_bytes = longest_row_bytes<float>(prm), k = row_bytes / 4;
    const int64_t together = streaming_rows(prm.rows, row_bytes);
    if (prm.rows <= 8 || together == 0) return false;
    int64_t products = 0;
    bool pair = false;
    for (int g = 0; g < prm.groups; ++g) {     // (four columns a store there, single ones here)
        const DecLinearGroup& d = prm.group[g];
        if (reinterpret_cast<uintptr_t>(d.w_up ? d.out : d.out32) & 15) return false;
        products += static_cast<int64_t>(d.n) * d.k * (d.w_up ? 2 : 1);
        pair = pair || d.w_up;
    }
    if (products * prm.rows <= (int64_t{1} << 26)) return false;
    const int64_t blocks = dot_tiles_of<kLinearRows>(prm) * ((prm.rows + together - 1) / together), pass = k * together / 8;
    // (two blocks of the dot products to a CU, where a CU that ends early takes the next; or one)
    const int64_t dots = 2 * together * row_bytes <= 160 * 1024 ? std::max<int64_t>(blocks, 512) * (20 + pass * 53 / 1024) / 512
                                                                 : (blocks + 255) / 256 * (20 + pass * 42 / 1024);
    return dots > 33 + k * (pair ? 85 : prm.rows <= 16 ? 46 : 56) / 1024;
}

int64_t steps_of_busiest_cu(int kinds, const int64_t* count, const int64_t* steps) {
    std::vector<int> order(static_cast<size_t>(kinds));
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return steps[a] > steps[b]; });
    std::map<int64_t, int64_t> cus = {{0, 256}};                               // steps dealt so far -> how many CUs have as many
    for (int kind : order)
        for (int64_t left = count[kind]; left > 0;) {
            const auto [at, many] = *cus.begin();
            const int64_t taken = std::min(left, many);
            cus.erase(cus.begin());
            if (many > taken) cus[at] = many - taken;
            cus[at + steps[kind]] += taken;
            left -= taken;
        }
    return cus.rbegin()->first;
}
// Steps of 64 k that the busiest CU walks when blocks of 128 x 128 outputs are dealt out long reductions first, the last one in `parts` pieces; a
// block's first stages and its outputs are about three steps more.
static int64_t steps_of_busiest(const DecLinearParams& prm, int parts) {
    int64_t count[kDecGroups], steps[kDecGroups];
    for (int g = 0; g < prm.groups; ++g) {
        const int pieces = g == prm.groups - 1 ? parts : 1;
        count[g] = static_cast<int64_t>(prm.group[g].n / 128) * ((prm.rows + 127) / 128) * pieces;
        steps[g] = prm.group[g].k / 64 / pieces + 3;
    }
    return steps_of_busiest_cu(prm.groups, count, steps);
}
// Into how many pieces the last linear's reduction is cut: where the linears' blocks leave CUs idle behind the longest reduction, its pieces
// fill them.  (us, 1024 rows, 2048 outputs of 6144: beside 2048 of 2048, three pieces, 66 -> 55; beside twice that, two pieces, 70 -> 65; the norm
// behind, which adds the pieces, 11.5 -> 14.)  A piece more is a plane of sums written and read, rows x outputs x 8 bytes: a step's time (0.73 us)
// for each 3 MB.
int reduction_pieces(const DecLinearParams& prm) {
    const DecLinearGroup& last = prm.group[prm.groups - 1];
    int64_t blocks = 0;
    for (int g = 0; g < prm.groups; ++g) blocks += static_cast<int64_t>(prm.group[g].n / 128) * ((prm.rows + 127) / 128);
    if (prm.groups < 2 || blocks < 200) return 1;                              // (fewer take smaller tiles)
    int best = 1;
    int64_t least = steps_of_busiest(prm, 1);
    for (int parts = 2; parts <= 1 + kMorePlanes; ++parts) {
        if (last.k % (128 * parts)) continue;
        const int64_t steps = steps_of_busiest(prm, parts) + (parts - 1) * (static_cast<int64_t>(prm.rows) * last.n * 8 / 3000000 + 1);
        if (steps < least) {
            least = steps;
            best = parts;
        }
    }
    return best;
}

int64_t reduction_cut_floats(const DecLinearParams& prm, int max_rows) {
    int64_t most = 0;
    DecLinearParams tile = prm;
    for (int row = 0; row < max_rows; row += 128) {                            // (of a row tile's rows the first has the most pieces, the last the most rows)
        tile.rows = row + 1;
        most = std::max(most, static_cast<int64_t>(reduction_pieces(tile) - 1) * std::min(row + 128, max_rows) * prm.group[prm.groups - 1].n);
    }
    return most;
}

static bool has_sizes(const DecLinearGroup& d) {
    return d.n > 0 && d.k > 0 && d.n % (d.w_up ? 128 : 16) == 0 && d.k % 128 == 0 && d.ldx >= d.k && d.ldo >= d.n && d.ldx % 8 == 0 && d.ldo % 4 == 0;
}
bool linears_have_sizes(const DecLinearParams& prm) { return std::all_of(prm.group, prm.group + prm.groups, has_sizes); }
int32_t check_linears(const DecLinearParams& prm) {
    if (prm.rows < 0 || prm.groups < 1 || prm.groups > kDecGroups) return QM_ERR_ARGUMENT;
    for (int g = 0; g < prm.groups; ++g) {
        const DecLinearGroup& d = prm.group[g];
        if (!d.x || !d.w || (d.w_up ? !d.out : !d.out32)) return QM_ERR_NULL;
        if (!has_sizes(d)) return QM_ERR_GEOMETRY;
    }
    return QM_OK;
}

static bool planes_end_first(const DecLinearParams& prm, bool cut) {
    return split_pays(prm) && (planes_pay(prm, 1) || (cut && planes_pay(prm, 2) && plane_pieces(prm) > 1));
}
bool goes_through_planes(const DecLinearParams& prm, int f32, const ReductionCut* cut, const PlaneMemory& planes) {
    return f32 && check_linears(prm) == QM_OK && prm.rows > 0 && plane_elements(prm) <= planes.elements && planes_end_first(prm, cut != nullptr);
}
int64_t plane_elements_up_to(const DecLinearParams& prm, int max_rows, bool cut) {
    DecLinearParams some = prm;
    for (some.rows = max_rows; some.rows > 0; --some.rows)                     // (more rows take more)
        if (planes_end_first(some, cut)) return plane_elements(some);
    return 0;
}
int64_t plane_cut_floats(const DecLinearParams& prm, int max_rows) {
    int64_t most = 0;
    DecLinearParams tile = prm;
    for (int row = 0; row < max_rows; row += kPlaneRows) {                     // (of a row tile's rows the first has the most pieces, the last the most rows)
        const int last = std::min(row + kPlaneRows, max_rows);
        tile.rows = row + 1;
        const int more = plane_pieces(tile) - 1;
        const int64_t floats = static_cast<int64_t>(more) * last * prm.group[prm.groups - 1].n;
        for (; floats > most && tile.rows <= last; ++tile.rows)
            if (planes_end_first(tile, true)) most = floats;
    }
    return most;
}

int32_t launch_decoder_linears(const DecLinearParams& prm, int f32, hipStream_t stream, ReductionCut* cut, const PlaneMemory& planes) {
    if (cut) cut->planes = 0;
    const int32_t checked = check_linears(prm);
    if (checked != QM_OK || prm.rows == 0) return checked;
    if (f32) {
        if (!split_pays(prm)) return streaming<float>(prm, stream);
        return goes_through_planes(prm, f32, cut, planes) ? launch_plane_linears(prm, planes, stream, cut) : launch_split_linears(prm, stream);
    }
    bool matrix = prm.rows >= kDecMatrixRows;
    if (matrix && prm.groups == 1 && prm.group[0].n <= kNarrowColumns && !prm.group[0].w_up)
        return prm.group[0].n <= 32 ? launch_narrow<2>(prm, stream) : launch_narrow<4>(prm, stream);
    for (int g = 0; g < prm.groups; ++g) matrix = matrix && prm.group[g].n % 128 == 0 && prm.group[g].ldx == prm.group[g].k && prm.group[g].ldo == prm.group[g].n;
    if (!matrix) return streaming<uint16_t>(prm, stream);
    LinearRowsParams plain = {};
    static_assert(kDecGroups + kMorePlanes <= kRowsGroups, "the pieces of a reduction are linears of their own");
    DecLinearGroup all[kDecGroups + kMorePlanes];
    int pitch[kDecGroups + kMorePlanes], order[kDecGroups + kMorePlanes], count = prm.groups;
    for (int g = 0; g < count; ++g) {
        all[g] = prm.group[g];
        pitch[g] = prm.group[g].k;
        if (prm.group[g].w_up) cut = nullptr;
    }
    if (cut) {
        DecLinearGroup& last = all[count - 1];
        cut->plane = static_cast<int64_t>(prm.rows) * last.n;
        int pieces = reduction_pieces(prm);
        if ((pieces - 1) * cut->plane > cut->room) pieces = 1;
        last.k /= pieces;
        for (; cut->planes < pieces - 1; ++cut->planes, ++count) {
            all[count] = last;
            all[count].x = static_cast<const uint16_t*>(last.x) + (cut->planes + 1) * last.k;
            all[count].w += (cut->planes + 1) * last.k;
            all[count].out32 = cut->sums + cut->planes * cut->plane;
            pitch[count] = pitch[prm.groups - 1];
        }
    }
    std::iota(order, order + count, 0);        // long reductions first
    std::stable_sort(order, order + count, [&](int a, int b) { return all[a].k > all[b].k; });
    for (int i = 0; i < count; ++i) {
        const DecLinearGroup& d = all[order[i]];
        if (d.w_up) {
            LinearRowsParams pair = {};
            pair.input = static_cast<const uint16_t*>(d.x);
            pair.weight[0] = d.w; pair.weight[1] = d.w_up;
            pair.output = static_cast<uint16_t*>(d.out);
            pair.rows = prm.rows; pair.columns = d.n; pair.reduction = d.k;
            pair.reduction_parts = 1; pair.groups = 1;
            const int32_t rc = launch_rows_mfma(pair, true, stream);
            if (rc != QM_OK) return rc;
            continue;
        }
        if (plain.groups == 0) {
            plain.input = static_cast<const uint16_t*>(d.x);
            plain.weight[0] = plain.weight[1] = d.w;
            plain.sums = d.out32;
            plain.rows = prm.rows; plain.columns = d.n; plain.reduction = d.k;
            plain.pitch = pitch[order[i]];
            plain.reduction_parts = 1;
        } else {
            const int at = plain.groups - 1;
            const int before = at == 0 ? 0 : plain.group_first_tile[at - 1];
            plain.group_first_tile[at] = before + (at == 0 ? plain.columns : plain.group_columns[at - 1]) / 128;
            plain.group_input[at] = static_cast<const uint16_t*>(d.x);
            plain.group_weight[at] = d.w;
            plain.group_sums[at] = d.out32;
            plain.group_columns[at] = d.n;
            plain.group_reduction[at] = d.k;
            plain.group_pitch[at] = pitch[order[i]];
        }
        ++plain.groups;
    }
    plain.linear_by_linear = plain.groups > 1;
    return plain.groups ? launch_rows_mfma(plain, false, stream) : QM_OK;
}

}  // namespace qm
