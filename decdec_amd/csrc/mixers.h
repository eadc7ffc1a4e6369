// Launch interface between the mixer kernels and their C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include "../../include/decdec_mixers.h"
#include "common.h"
#include "tile_attention.h"

namespace decdec {

constexpr uint32_t kChunkRows = 64;        // tokens per chunk of a recurrence
constexpr uint32_t kMaxRank = 1024;        // of the low-rank maps of a recurrence

hipError_t launch_mix_gemv(int dt, const void* w, const void* x, void* out, const void* act, uint32_t act_rows, int act_kind,
                           float scale, uint32_t N, uint32_t K, hipStream_t s);
hipError_t launch_mix_gemv_residual_tanh(int dt, const void* w, const void* in, float* x, const decdec_tanh_norm& norm, void* out, uint32_t N,
                                         uint32_t K, hipStream_t s);
// 32-bit products on the fp16 units (k_splitgemm.hip): tiles of 16 tokens a workgroup, ranges of K, the time that they should take.
struct SplitPlan { uint32_t tm, ks; float us; };
SplitPlan split_plan(uint32_t M, uint32_t N, uint32_t K);
size_t split_workspace(const SplitPlan& plan, uint32_t M, uint32_t N, uint32_t K);
float* split_sums(const SplitPlan& plan, void* ws, uint32_t M, uint32_t K);
hipError_t launch_split_gemm(const SplitPlan& plan, const float* x, uint32_t ldx, const float* w, uint32_t ldw, float* out, uint32_t ldo, void* ws,
                             uint32_t M, uint32_t N, uint32_t K, bool wide, hipStream_t s);
size_t row_gemm_workspace(int dt, uint32_t M, uint32_t N, uint32_t K);
int row_gemm_pieces(int dt, uint32_t M, uint32_t N, uint32_t K, uint32_t ldw);       // ranges of K of a product on fp16 pieces, 0: it is not one
hipError_t launch_row_gemm(int dt, const void* x, uint32_t ldx, const void* w, uint32_t ldw, void* out, uint32_t ldo, void* ws, uint32_t M,
                           uint32_t N, uint32_t K, hipStream_t s);
hipError_t launch_mix_embed(int dt, const void* table, const long long* tokens, float* x, void* xe, const decdec_tanh_norm* norm,
                            uint32_t rows, uint32_t vocab, uint32_t dim, hipStream_t s);
hipError_t launch_mix_residual_tanh(int dt, float* x, const void* y, const decdec_tanh_norm& norm, void* out, uint32_t rows,
                                    uint32_t dim, hipStream_t s);
hipError_t launch_mix_gated_residual(int dt, float* x, const void* y, const void* gate, uint32_t gate_ld, const void* bias,
                                     const void* weight, void* xe, const void* fw, void* fo, uint32_t rows, uint32_t dim,
                                     float eps, hipStream_t s);
hipError_t launch_mix_rmsnorm(int dt, const float* x, const void* weight, void* out, uint32_t rows, uint32_t dim, float eps,
                              hipStream_t s);
hipError_t launch_mix_activation(int dt, const void* in, uint32_t ld, const void* act, int kind, void* out, uint32_t rows,
                                 uint32_t n, hipStream_t s);
hipError_t launch_mix_group_norm_gate(int dt, const float* o, const void* gate, uint32_t ld, const void* weight, void* out,
                                      uint32_t out_ld, uint32_t rows, uint32_t groups, uint32_t n, float eps, int kind,
                                      float scale, hipStream_t s);
// Shares of a token's grouped attention on their way to its heads' results.
struct GroupedMerge {
    const float* parts;                // [share][heads][vdim + 2]: sums, maximum, sum of weights
    void* out;                         // [heads * vdim]
    const int64_t* pos;
    const void* gates;                 // the projections where there are gates
    uint32_t off_g, heads, vdim, max_seq, max_splits;
    float sink, out_scale;
};
bool recurrence_step_fuses(uint32_t dim, uint32_t vdim);
bool recurrence_step_merges(const decdec_recurrence& p);
// `merge`: shares that are merged beside the step, by workgroups behind its own (null: none; otherwise `out` is set and recurrence_step_merges holds).
hipError_t launch_recurrence_step(int dt, const decdec_recurrence& p, float* o, void* out, const void* nw, float eps, int kind,
                                  const GroupedMerge* merge, hipStream_t s);
size_t recurrence_workspace(const decdec_recurrence& p, uint32_t rows);
hipError_t launch_recurrence_rows(int dt, const decdec_recurrence& p, float* o, void* ws, uint32_t rows, hipStream_t s);
hipError_t launch_tile_attention(int dt, const TileAttention& p, uint32_t start, uint32_t rows, hipStream_t s);
hipError_t launch_grouped_append(int dt, const decdec_grouped& p, void* q_out, uint32_t rows, hipStream_t s);
hipError_t launch_grouped_attention(int dt, const decdec_grouped& p, const void* q, void* out, uint32_t start, uint32_t rows,
                                    hipStream_t s);
size_t grouped_step_workspace(const decdec_grouped& p);
hipError_t launch_grouped_step(int dt, const decdec_grouped& p, void* out, void* ws, hipStream_t s);
hipError_t launch_grouped_shares(int dt, const decdec_grouped& p, void* ws, hipStream_t s);       // without the merge
GroupedMerge grouped_merge_of(const decdec_grouped& p, void* out, void* ws);
hipError_t launch_latent_append(int dt, const decdec_latent& p, void* q_out, uint32_t rows, hipStream_t s);
hipError_t launch_latent_attention(int dt, const decdec_latent& p, const void* q, const void* k, const void* vt, uint32_t vt_ld,
                                   void* out, uint32_t start, uint32_t rows, hipStream_t s);
size_t latent_step_workspace(const decdec_latent& p);
hipError_t launch_latent_step(int dt, const decdec_latent& p, void* out, void* ws, hipStream_t s);

}  // namespace decdec
