// qm_decoder_ops.h — launch parameters and launchers of the decoder language models' kernels, as the engine calls them.
// Every launcher checks its arguments on the host, enqueues on `stream` and returns a QM_* code.  `f32` chooses the
// activation type: 0 bf16, 1 fp32.
#pragma once

#include <hip/hip_runtime.h>

#include "../../../include/qm_attn.h"
#include "../../../include/qm_decoder.h"

namespace qm {

constexpr int kDecMaxWidth = 12288;       // columns of the residual stream (a block's threads hold a row)
constexpr int kDecMaxSplits = 64;         // key splits of one attention (a wave's lanes combine them)
constexpr int kDecMaxMerge = 4096;        // heads * key splits of one attention (their factors lie in LDS)
constexpr int kDecMaxHead = 256;          // channels of a head
constexpr int kAttentionMatrixRows = 16;  // rows from which bf16 attention goes to the matrix cores
constexpr int kChunkedRows = 16;          // rows from which a recurrence is computed in chunks (given scratch)
constexpr int kDecGroups = 3;             // linears in one launch
constexpr int kDotLdsMost = 159 * 1024;   // dynamic LDS of one block

// Linears of one launch.
struct DecLinearParams {
    qm_decoder_linear group[kDecGroups];
    int groups, rows;
    int streaming;                   // a one-token step's weights with the non-temporal hint (qm_decoder_dot.h)
};
using ResidualParams = qm_residual_norm;
using GatedNormParams = qm_gated_norm;
using AttentionPartials = qm_attention_partials;
using DecLinearGroup = qm_decoder_linear;
using ChunkAttentionParams = qm_chunk_attention;
using DecayAttentionParams = qm_decay_attention;
using DeltaParams = qm_general_delta;
using LatentRowsParams = qm_latent_rows;
using LatentAttentionParams = qm_latent_attention;
using ExpertParams = qm_experts;
constexpr int kLatentKeys = 64;           // keys per pass of the attention over latents; its splits are whole passes
constexpr int kLatentMaxRank = 1024;      // channels of a latent
constexpr int kLatentMaxRotary = 256;     // channels of the key part that heads share
constexpr int kExpertsMost = 1024;
constexpr int kDecayChunk = QM_DECAY_CHUNK;
constexpr int kDecayPowers = QM_DECAY_POWERS;

// float4s of a row that each of a block's 256 threads holds: the kernels' choices for a row of ld columns.
inline int row_vectors(int64_t ld) { return ld <= 1024 ? 1 : ld <= 2048 ? 2 : ld <= 4096 ? 4 : 12; }

// Whether the kernels take these arguments.
int32_t check_residual(const ResidualParams& prm);
int32_t check_linears(const DecLinearParams& prm);
bool linears_have_sizes(const DecLinearParams& prm);            // (of that, what no pointer is needed for)
int32_t check_attention(const ChunkAttentionParams& prm);
int32_t check_decay_attention(const DecayAttentionParams& prm);
// The last term in pieces: `planes` more of them, `plane` floats apart, laid out as the term's own and added to it in order.
constexpr int kMorePlanes = 2;
struct MoreOfTerm {
    const float* sums = nullptr;
    int64_t plane = 0;
    int planes = 0;
};
// parts: h also goes there, split as PlaneMemory below has it (fp32 only).
int32_t launch_residual_norm(const ResidualParams& prm, int rows, int f32, hipStream_t stream, const MoreOfTerm& more = MoreOfTerm(),
                             uint16_t* parts = nullptr);
int32_t launch_gated_norm(const GatedNormParams& prm, int rows, int f32, hipStream_t stream);
// Many rows of bf16 go to the matrix cores (linears of one launch in one grid, a gate/up pair in its own), few rows and
// fp32 to the streaming kernel.
// cut: the last linear's reduction may be taken in pieces, whose sums behind the first's go to cut->sums in planes of [rows][n], as many as `room`
// floats hold; how many do is left in cut->planes.
struct ReductionCut {
    float* sums;
    int64_t room;
    int64_t plane;
    int planes;
};
// Into how many pieces that is, and the most floats that they take with any number of rows up to max_rows.
int reduction_pieces(const DecLinearParams& prm);
int64_t reduction_cut_floats(const DecLinearParams& prm, int max_rows);
constexpr int kPlaneRows = 64;            // token rows of a block whose inputs are split beforehand
// Memory in which fp32 inputs are split into their three parts beforehand: three times rows x k elements for each of the linears' different inputs.
struct PlaneMemory {
    uint16_t* at = nullptr;
    int64_t elements = 0;
    bool split = false;              // the linears' one input is there, split
};
int32_t launch_decoder_linears(const DecLinearParams& prm, int f32, hipStream_t stream, ReductionCut* cut = nullptr, const PlaneMemory& planes = PlaneMemory());
int32_t launch_split_linears(const DecLinearParams& prm, hipStream_t stream);    // fp32 rows on the matrix cores
// The same with inputs split beforehand: whether they can be, and whether that ends first (given that the matrix cores do), with the last reduction in so
// many pieces; into how many it is cut; the launch, which cuts if `cut` has room.
bool planes_fit(const DecLinearParams& prm);
bool goes_through_planes(const DecLinearParams& prm, int f32, const ReductionCut* cut, const PlaneMemory& planes);    // (what launch_decoder_linears does)
bool planes_pay(const DecLinearParams& prm, int pieces);
int plane_pieces(const DecLinearParams& prm);
int64_t plane_elements(const DecLinearParams& prm);
// What they take at most with any number of rows up to max_rows: elements of split inputs, and floats of pieces (given that memory).
int64_t plane_elements_up_to(const DecLinearParams& prm, int max_rows, bool cut);
int64_t plane_cut_floats(const DecLinearParams& prm, int max_rows);
int32_t launch_plane_linears(const DecLinearParams& prm, const PlaneMemory& planes, hipStream_t stream, ReductionCut* cut);
// Steps that the busiest of 256 CUs walks when `kinds` kinds of blocks, `count` of `steps` steps each, are dealt out one to a CU, long ones first.
int64_t steps_of_busiest_cu(int kinds, const int64_t* count, const int64_t* steps);
// Rotation and cache write, then the attention.
int32_t launch_chunk_attention(const ChunkAttentionParams& prm, int f32, hipStream_t stream);
int32_t check_chunk_attention_mfma(const ChunkAttentionParams& prm);              // what it asks for beside check_attention
int32_t launch_chunk_attention_mfma(const ChunkAttentionParams& prm, hipStream_t stream);
bool attention_f32_pays(const ChunkAttentionParams& prm);                         // whether many fp32 rows go to the matrix cores
int32_t launch_chunk_attention_f32(const ChunkAttentionParams& prm, hipStream_t stream);
int32_t launch_decay_attention(const DecayAttentionParams& prm, hipStream_t stream);
// Floats of scratch with which a pass of `rows` tokens is computed in chunks (0: it is not).
int64_t decay_scratch_floats(int rows, int heads, int dim, int vdim);
int64_t delta_scratch_floats(int rows, int heads, int dim);
bool delta_chunks_fit(const DeltaParams& prm);
int32_t launch_decay_chunks(const DecayAttentionParams& prm, hipStream_t stream);
int32_t launch_delta_chunks(const DeltaParams& prm, hipStream_t stream);
int32_t check_general_delta(const DeltaParams& prm);
int32_t launch_general_delta(const DeltaParams& prm, hipStream_t stream);
int32_t launch_latent_rows(const LatentRowsParams& prm, int f32, hipStream_t stream);
// keep: what the step's token leaves in the cache, written by the launch that prepares the queries (NULL: it is there).
int32_t launch_latent_attention(const LatentAttentionParams& prm, const LatentRowsParams* keep, int f32, hipStream_t stream);
int32_t launch_latent_partials_mfma(const LatentAttentionParams& prm, hipStream_t stream);
bool latent_partials_fit_mfma(const LatentAttentionParams& prm);
int latent_q_stride(int kv_rank, int rot_dim);
int64_t expert_scratch_bytes(int rows, int experts, int top, int width_p, int ff_p, int f32);
int32_t launch_experts(const ExpertParams& prm, int f32, hipStream_t stream);

// ---- one token: a layer run in three launches -----------------------------------------------------------------------
// Residual sum and norm by every block for itself, then the linears that read it (row 0 of everything); the norm's output
// also goes to residual.h if that is given.
struct LayerInParams {
    ResidualParams residual;
    DecLinearParams linears;
};
// The output linears, each block preparing the input of its own: 0 as it is in memory, 1 the attention's key splits
// combined, 2 the gated norm, 3 a slice of fp32 values divided by its root mean square and weighted.
struct SliceNorm {
    const float* x;
    const float* weight;
    int n;
    float eps;
};
struct LayerOutParams {
    DecLinearParams linears;
    int input[kDecGroups];
    int chunk;                       // of the attention (input 1)
    AttentionPartials part;
    const int32_t* position_dev;
    GatedNormParams gated;           // (input 2)
    SliceNorm slice;                 // (input 3)
};
int32_t launch_layer_in(const LayerInParams& prm, int f32, hipStream_t stream);
// The attention (rotation and cache write included) beside the decayed linear attention, and the delta rule, one token each; and
// beside either one linear whose input is in memory as it is (or none).
int32_t launch_mixer_step(const ChunkAttentionParams& attention, const DecayAttentionParams& decay, const DecLinearParams& beside, int f32,
                          hipStream_t stream);
int32_t launch_delta_step(const DeltaParams& delta, const DecLinearParams& beside, int f32, hipStream_t stream);
int32_t launch_layer_out(const LayerOutParams& prm, int f32, hipStream_t stream);
// the id of the highest of `vocab` scores (lowest among equals)
int32_t launch_argmax(const float* scores, int vocab, int32_t* token, hipStream_t stream);
// step = the words below: the chosen token is put out and becomes the one to feed, the token that was fed the one before it,
// and the position moves on by `advance`
enum StepWord { kStepPosition, kStepBefore, kStepToken, kStepEmitted, kStepChosen, kStepTicket, kStepWords };
int32_t launch_emit(int32_t* step, int32_t* out, int advance, hipStream_t stream);
// The words from pinned host memory; and `vocab` scores into pinned host memory, each of mail_blocks(vocab) blocks raising its flag
// (kMailFlagStride words apart) to the ticket behind what it wrote: a host that sees every flag has every score.
constexpr int kMailBlocks = 16, kMailFlagStride = 16;
inline int mail_blocks(int vocab) { return vocab < 1024 ? 1 : vocab / 1024 < kMailBlocks ? vocab / 1024 : kMailBlocks; }
int32_t launch_take_words(const int32_t* host, int32_t* step, hipStream_t stream);
int32_t launch_mail_scores(const float* scores, int vocab, float* host, uint32_t* flags, const int32_t* ticket, hipStream_t stream);

}  // namespace qm
