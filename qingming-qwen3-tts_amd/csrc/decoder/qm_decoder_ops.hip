// qm_decoder_ops.hip — C ABI of the decoder language models' operators.
#include "../qm_host.h"
#include "qm_decoder_ops.h"

extern "C" int32_t qm_residual_norm_rows(const qm_residual_norm* op, int32_t rows, int32_t f32, void* hip_stream) {
    return op ? qm::launch_residual_norm(*op, rows, f32, static_cast<hipStream_t>(hip_stream)) : QM_ERR_NULL;
}
extern "C" int32_t qm_gated_norm_rows(const qm_gated_norm* op, int32_t rows, int32_t f32, void* hip_stream) {
    return op ? qm::launch_gated_norm(*op, rows, f32, static_cast<hipStream_t>(hip_stream)) : QM_ERR_NULL;
}
static bool linears_of(const qm_decoder_linear* linears, int32_t count, int32_t rows, qm::DecLinearParams& prm) {
    if (!linears || count < 1 || count > qm::kDecGroups) return false;
    for (int i = 0; i < count; ++i) prm.group[i] = linears[i];
    prm.groups = count;
    prm.rows = rows;
    return true;
}
extern "C" int32_t qm_decoder_linear_rows(const qm_decoder_linear* linears, int32_t count, int32_t rows, int32_t f32, void* hip_stream) {
    qm::DecLinearParams prm = {};
    if (!linears) return QM_ERR_NULL;
    if (!linears_of(linears, count, rows, prm)) return QM_ERR_ARGUMENT;
    return qm::launch_decoder_linears(prm, f32, static_cast<hipStream_t>(hip_stream));
}
extern "C" int64_t qm_decoder_linear_planes_bytes(const qm_decoder_linear* linears, int32_t count, int32_t rows) {
    qm::DecLinearParams prm = {};
    return linears_of(linears, count, rows, prm) && rows > 0 && qm::linears_have_sizes(prm) && qm::planes_fit(prm) ? 2 * qm::plane_elements(prm) : 0;
}
extern "C" int32_t qm_decoder_linear_rows_planes(const qm_decoder_linear* linears, int32_t count, int32_t rows, void* planes, int64_t planes_bytes, void* hip_stream) {
    qm::DecLinearParams prm = {};
    if (!linears || !planes) return QM_ERR_NULL;
    if (!linears_of(linears, count, rows, prm)) return QM_ERR_ARGUMENT;
    const int32_t rc = qm::check_linears(prm);
    if (rc != QM_OK || rows == 0) return rc;
    if (!qm::planes_fit(prm) || (reinterpret_cast<uintptr_t>(planes) & 15)) return QM_ERR_GEOMETRY;
    if (planes_bytes < 2 * qm::plane_elements(prm)) return QM_ERR_WORKSPACE;
    return qm::launch_plane_linears(prm, {static_cast<uint16_t*>(planes), planes_bytes / 2}, static_cast<hipStream_t>(hip_stream), nullptr);
}
extern "C" int32_t qm_chunk_attention_rows(const qm_chunk_attention* op, int32_t f32, void* hip_stream) {
    return op ? qm::launch_chunk_attention(*op, f32, static_cast<hipStream_t>(hip_stream)) : QM_ERR_NULL;
}
extern "C" int32_t qm_decay_attention_rows(const qm_decay_attention* op, void* hip_stream) {
    return op ? qm::launch_decay_attention(*op, static_cast<hipStream_t>(hip_stream)) : QM_ERR_NULL;
}
extern "C" int32_t qm_general_delta_rows(const qm_general_delta* op, void* hip_stream) {
    return op ? qm::launch_general_delta(*op, static_cast<hipStream_t>(hip_stream)) : QM_ERR_NULL;
}
extern "C" int64_t qm_decay_attention_scratch_floats(int32_t rows, int32_t heads, int32_t dim, int32_t vdim) {
    return qm::decay_scratch_floats(rows, heads, dim, vdim);
}
extern "C" int64_t qm_general_delta_scratch_floats(int32_t rows, int32_t heads, int32_t dim) {
    return qm::delta_scratch_floats(rows, heads, dim);
}
