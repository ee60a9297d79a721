// qm_decoder_norm.hip — row operators around the decoder language models' mixers: the residual sum with the norm that
// reads it, and the gated norm behind a recurrent mixer.  One block of 256 threads per row; a row is a few tens of KB, so
// both are bound by memory latency for few rows and by bandwidth for a prompt.
#include "qm_decoder_device.h"
#include "../qm_host.h"

namespace qm {

template <class T, int NV, bool MORE>
__global__ __launch_bounds__(kDecThreads) void residual_norm_kernel(ResidualParams prm, MoreOfTerm more) {
    __shared__ float sh_red[16];
    const int row = static_cast<int>(blockIdx.x);
    residual_norm_row<T, NV, false, MORE>(prm, row, sh_red, static_cast<T*>(prm.h) + row * prm.ld_h, true, NothingBehind(), more);
}

// The row of h also split into three parts, for linears that want their inputs so.  A launch of its own reads h again: 4.9 us for 300 rows of 1024,
// where this kernel takes 6.9 us with the parts and 6.2 without (a prompt of four layers 443 -> 435 us).
template <int NV, bool MORE>
__global__ __launch_bounds__(kDecThreads) void residual_norm_split_kernel(ResidualParams prm, MoreOfTerm more, uint16_t* parts, int64_t plane) {
    __shared__ float sh_red[16];
    const int row = static_cast<int>(blockIdx.x);
    const SplitRow to = {static_cast<float*>(prm.h) + row * prm.ld_h, parts + row * prm.ld_h, plane};
    residual_norm_row<float, NV, false, MORE>(prm, row, sh_red, to, true, NothingBehind(), more);
}

template <class T, int AT_ONCE>
__global__ __launch_bounds__(kDecThreads) void gated_norm_kernel(GatedNormParams prm) {
    __shared__ float sh_red[4];
    const int64_t row = blockIdx.x;
    gated_norm_row<T, AT_ONCE>(prm, row, sh_red, static_cast<T*>(prm.out) + row * prm.ld_out);
}

int32_t check_residual(const ResidualParams& prm) {
    if (prm.width <= 0 || prm.ld_h < prm.width || prm.terms < 0 || prm.terms > 3) return QM_ERR_ARGUMENT;
    if (!prm.norm_w || (!prm.x_in && (!prm.embed || !prm.tokens))) return QM_ERR_NULL;
    if (prm.ld_h % 4 || prm.ld_h > kDecMaxWidth) return QM_ERR_GEOMETRY;
    if (!prm.x_in && prm.buckets > 0 && !prm.bigram) return QM_ERR_NULL;
    if (prm.buckets < 0 || (prm.buckets > 0 && (prm.mul_prev < 0 || prm.mul_cur < 0))) return QM_ERR_ARGUMENT;
    for (int i = 0; i < prm.terms; ++i) {
        if (!prm.term[i].y) return QM_ERR_NULL;
        if (prm.term[i].ld < prm.ld_h || prm.term[i].ld % 4) return QM_ERR_GEOMETRY;
    }
    return QM_OK;
}

template <class T, bool MORE>
static int32_t residual_as(const ResidualParams& prm, int rows, const MoreOfTerm& more, hipStream_t stream) {
    switch (row_vectors(prm.ld_h)) {
        case 1: hipLaunchKernelGGL((residual_norm_kernel<T, 1, MORE>), dim3(rows), dim3(kDecThreads), 0, stream, prm, more); break;
        case 2: hipLaunchKernelGGL((residual_norm_kernel<T, 2, MORE>), dim3(rows), dim3(kDecThreads), 0, stream, prm, more); break;
        case 4: hipLaunchKernelGGL((residual_norm_kernel<T, 4, MORE>), dim3(rows), dim3(kDecThreads), 0, stream, prm, more); break;
        default: hipLaunchKernelGGL((residual_norm_kernel<T, 12, MORE>), dim3(rows), dim3(kDecThreads), 0, stream, prm, more); break;
    }
    return launch_status();
}

template <bool MORE>
static int32_t residual_split(const ResidualParams& prm, int rows, const MoreOfTerm& more, uint16_t* parts, hipStream_t stream) {
    const int64_t plane = static_cast<int64_t>(rows) * prm.ld_h;
    switch (row_vectors(prm.ld_h)) {
        case 1: hipLaunchKernelGGL((residual_norm_split_kernel<1, MORE>), dim3(rows), dim3(kDecThreads), 0, stream, prm, more, parts, plane); break;
        case 2: hipLaunchKernelGGL((residual_norm_split_kernel<2, MORE>), dim3(rows), dim3(kDecThreads), 0, stream, prm, more, parts, plane); break;
        case 4: hipLaunchKernelGGL((residual_norm_split_kernel<4, MORE>), dim3(rows), dim3(kDecThreads), 0, stream, prm, more, parts, plane); break;
        default: hipLaunchKernelGGL((residual_norm_split_kernel<12, MORE>), dim3(rows), dim3(kDecThreads), 0, stream, prm, more, parts, plane); break;
    }
    return launch_status();
}

int32_t launch_residual_norm(const ResidualParams& prm, int rows, int f32, hipStream_t stream, const MoreOfTerm& more, uint16_t* parts) {
    const int32_t rc = check_residual(prm);
    if (rc != QM_OK) return rc;
    if (rows < 0) return QM_ERR_ARGUMENT;
    if (!prm.h) return QM_ERR_NULL;
    if (rows == 0) return QM_OK;
    if (parts && !f32) return QM_ERR_ARGUMENT;
    if (more.planes > 0) {                     // (the matrix cores leave a term in pieces)
        if (!more.sums) return QM_ERR_NULL;
        if (more.planes > kMorePlanes || prm.terms == 0) return QM_ERR_ARGUMENT;
        if (parts) return residual_split<true>(prm, rows, more, parts, stream);
        return f32 ? residual_as<float, true>(prm, rows, more, stream) : residual_as<uint16_t, true>(prm, rows, more, stream);
    }
    if (parts) return residual_split<false>(prm, rows, more, parts, stream);
    return f32 ? residual_as<float, false>(prm, rows, more, stream) : residual_as<uint16_t, false>(prm, rows, more, stream);
}

int32_t launch_gated_norm(const GatedNormParams& prm, int rows, int f32, hipStream_t stream) {
    if (rows < 0 || prm.groups <= 0 || prm.size <= 0 || prm.ld_out < static_cast<int64_t>(prm.groups) * prm.size) return QM_ERR_ARGUMENT;
    if (!prm.o || !prm.gate || !prm.out) return QM_ERR_NULL;
    if (rows == 0) return QM_OK;
    const bool many = prm.groups > 1 && gated_norm_many(prm, rows);
    const auto kernel = f32 ? (many ? gated_norm_kernel<float, 4> : gated_norm_kernel<float, 1>)
                            : (many ? gated_norm_kernel<uint16_t, 4> : gated_norm_kernel<uint16_t, 1>);
    hipLaunchKernelGGL(kernel, dim3(rows), dim3(kDecThreads), 0, stream, prm);
    return launch_status();
}

}  // namespace qm
