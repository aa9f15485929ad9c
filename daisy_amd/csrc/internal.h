// Kernels of this library that the package's native glue (native.cpp) launches directly, beside the C ABI.
// Host code only: the glue is compiled by the host compiler.
#pragma once

#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include "../../include/daisy_hip.h"

namespace daisy {

// The value-embedding gate of a layer: sigmoid(logit) rounded to bf16, the dtype in which the mix is evaluated.
// Either the value itself (fp32, as the C ABI takes it) or the layer's logit, which a kernel turns into the value
// where it is needed instead of three launches of a tensor library in front of it.
struct GateSource {
  enum Kind { kValue = 0, kLogitF32 = 1, kLogitBf16 = 2 };
  const void* p;
  int kind;
};

// Everything between the QKV projection and the attention: RMS norm of q, k, v, RoPE of q, k at rows pos0 + t of the
// tables, gate * v + (1 - gate) * ve; outputs [B, T, H, D] with {batch, token, head} strides in elements.
struct QkvEpilogue {
  uint16_t* q; int64_t q_sb, q_st, q_sh;
  uint16_t* k; int64_t k_sb, k_st, k_sh;
  uint16_t* v; int64_t v_sb, v_st, v_sh;
  const uint16_t* ve; int64_t ve_sb, ve_st, ve_sh;
  GateSource gate;
  const float* cos; const float* sin;
  int pos0, H, T;
  float eps;
};

// Whether prefill attention of so many (batch, head) pairs takes the kernel with 32 queries per workgroup.
bool prefill_split_wanted(int pairs, int T, int D, int window, bool docs);
// y [M, N] = x [M, K] w [N, K]^T (+ bias), fp32 accumulation, one rounding.  tile: 0 = by the sizes.
int proj_linear(const uint16_t* x, int64_t x_sm, const uint16_t* w, int64_t w_sn, const uint16_t* bias,
                uint16_t* y, int64_t y_sm, int M, int N, int K, hipStream_t s, int tile = 0);
// The decay gate of the KDA layer as a product's epilogue: y = -exp(A_log[h]) * softplus(y + dt_bias) on the bf16 product, heads of Dk
// channels (a multiple of 8), and beside it beta [M, H] = bf16(sigmoid(logits)) as fp32, logits rows `logits_row` elements apart.
struct KdaGates {
  const float *A_log, *dt_bias;      // [H], [H * Dk]
  int H, Dk;
  const uint16_t* logits; int64_t logits_row;
  float* beta;
};
// One of several products over the same number of rows M and the same K that share a launch: y = x w^T (+ bias).  N need not be a
// multiple of 8 where y's rows have room for it (y_sm >= N rounded up to 8; the columns from N on are then scribbled over).
struct ProjSegment {
  const uint16_t* x; int64_t x_sm;
  const uint16_t* w; int64_t w_sn;
  const uint16_t* bias;
  uint16_t* y; int64_t y_sm;
  int N, tile_end;      // tile_end: filled in by the launch
};
constexpr int kMaxSegments = 6;
// gates: what becomes of the first product on its way out (its N is H Dk).
int proj_segments(const ProjSegment* seg, int n, int M, int K, hipStream_t s, int tile = 0, const KdaGates* gates = nullptr);
// The same through the weight-streaming kernel of linear.hip, M <= 8 (no bias); every row as daisy_linear_rows_fwd computes it.
int linear_segments(const ProjSegment* seg, int n, int M, int K, hipStream_t s);
// Whether the tiled kernel is the better choice for these sizes than the library GEMM (and, for the QKV projection, than
// the library GEMM with qkv_prep_kernel behind it).
bool proj_wanted(int M, int N, int K);              // one product
bool proj_segments_wanted(int M, int N, int K);     // several, N columns in all
bool proj_layer_wanted(int M, int N, int K);        // the KDA layer's six, N columns in all
bool proj_qkv_wanted(int M, int N, int K);
// The QKV projection of x [B * T, K] with its epilogue.
int proj_qkv(const uint16_t* x, int64_t x_sm, const uint16_t* w, int64_t w_sn, const QkvEpilogue& e,
             int B, int K, int D, hipStream_t s, int tile = 0);

// What a one-launch attention step adds to a decode launch: the kernel prepares the rows of the projection itself.
// k_rows / v_rows: NULL, or bf16 [B, H, D] contiguous copies of the new rows as the ring holds them (an fp16 ring's
// rows in the model's dtype, without another pass over them).
// out: a product y [N] = o [H * D] w [N, H * D]^T that takes the attention's place in memory (o is then not written), for the calls that
// step_projects says it serves: one sequence whose ring is split.
struct StepProjection { const uint16_t* w; int64_t w_sn; uint16_t* y; int N; };
bool step_projects(int B, int H, int D, int n_rows);
struct StepPrep {
  int pos_host; const float* cos; const float* sin; int table_rows; float eps;
  const void* ve; const int64_t* ve_strides; GateSource gate;
  int cache_f16; int32_t* status;
  uint16_t* k_rows; uint16_t* v_rows;
  StepProjection out = {nullptr, 0, nullptr, 0};
};
int decode_launch(const void* q, const int64_t* q_strides,
                  const void* k_new, const int64_t* k_new_strides,
                  const void* v_new, const int64_t* v_new_strides,
                  void* k_cache, const int64_t* k_cache_strides,
                  void* v_cache, const int64_t* v_cache_strides,
                  const float* cos_row, const float* sin_row,
                  void* o, const int64_t* o_strides,
                  int B, int H, int D,
                  int n_rows, int new_idx, const int32_t* pos_dev, int write_back,
                  float scale, int nsplit,
                  void* workspace, size_t workspace_bytes, void* stream, const StepPrep* prep = nullptr,
                  bool f32_io = false);
int attn_step_launch(const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides,
                     const void* v, const int64_t* v_strides, void* k_cache, const int64_t* k_cache_strides,
                     void* v_cache, const int64_t* v_cache_strides, void* o, const int64_t* o_strides,
                     int B, int H, int D, int ring_rows, const int32_t* pos_dev, float scale, int nsplit,
                     void* workspace, size_t workspace_bytes, void* stream, const StepPrep& prep);

// y [rows, C] = x rsqrt(mean(x^2) + eps), bf16, contiguous; the sizes that it takes.
bool rms_rows_serves(int64_t rows, int64_t C);
int rms_rows(const uint16_t* x, uint16_t* y, int rows, int C, float eps, hipStream_t s);

// qkv_prep_kernel with the gate as the layer holds it.
int prep_launch(const void* q, const int64_t* q_strides, const void* k, const int64_t* k_strides,
                const void* v, const int64_t* v_strides, const void* ve, const int64_t* ve_strides, GateSource gate,
                const float* cos, const float* sin, int pos0, const int32_t* pos0_dev, int table_rows, int32_t* status,
                void* q_out, const int64_t* q_out_strides, void* k_out, const int64_t* k_out_strides,
                void* v_out, const int64_t* v_out_strides, int B, int T, int H, int D, float eps, void* stream);

// A decode step of the KDA layer (attention_kimi.py) between its first and its last projection, one token per sequence: short
// convolutions with SiLU (windows shifted in place), the second halves of the two low-rank projections, decay gate,
// beta, delta-rule update of the state (in place), gated RMS norm.  Rows of q, k, v, f, g, b: one per sequence, `row`
// elements apart.
struct KdaLayerStep {
  const uint16_t *q, *k, *v, *f, *g, *b; int64_t q_row, k_row, v_row, f_row, g_row, b_row;
  const uint16_t* conv_w[3]; const uint16_t* conv_bias[3]; uint16_t* window[3]; int taps;     // [C, taps], [C] or NULL, [B, C, taps]
  const uint16_t *wf, *wg, *g_bias;       // [H * Dk, Dv], [H * Dv, Dv], [H * Dv] or NULL
  const float *A_log, *dt_bias;           // [H], [H * Dk]
  const uint16_t* norm_w;                 // [Dv]
  float* state;                           // [B, H, Dk, Dv]
  uint16_t* o; int64_t o_row;             // [B, H * Dv]
  int H, Dk; float scale, l2_eps, norm_eps;
};
// daisy_short_conv_fwd for one to three inputs of the same B, T and number of taps in one launch.
struct ConvPart {
  const uint16_t* x; int64_t x_sb, x_st;       // [B, T, C], channel stride 1
  const uint16_t* w;                           // [C, K]
  const uint16_t* bias;                        // [C] or null
  const uint16_t* cache_in;                    // [B, C, K] or null: the last K inputs before t = 0 (the first is unused)
  uint16_t* y; int64_t y_sb, y_st;             // [B, T, C]
  uint16_t* cache_out;                         // [B, C, K] or null: the last K inputs of the extended sequence
  int C;
};
// The KDA layer's low-rank products, x [M, K] w [N, K]^T with K = 64 or 128, a value head's width: through the decay gate into y [M, N],
// with beta; or as the gate of the gated RMS norm over the N / K heads of o [M, N], in place (bias [N] or NULL, norm_weight [K]).
int low_rank_walkers(int M, int groups);       // their workgroups per group of columns
bool low_rank_wanted(int M, int N, int K);     // whether they are the better choice than proj_segments and gated_rmsnorm_kernel
int low_rank_gate(const uint16_t* x, int64_t x_sm, const uint16_t* w, const KdaGates& gates, uint16_t* y, int M, int N, int K, hipStream_t s);
int low_rank_norm(const uint16_t* x, int64_t x_sm, const uint16_t* w, const uint16_t* bias, const uint16_t* norm_weight, uint16_t* o, float eps,
                  int M, int N, int K, hipStream_t s);
int short_conv_group(const ConvPart* parts, int n, int B, int T, int K, int silu, hipStream_t s);
bool kda_layer_step_serves(int Dk, int Dv, int taps);
bool gated_rmsnorm_serves(int D);      // the widths that daisy_gated_rmsnorm_fwd takes
int kda_layer_step(const KdaLayerStep& p, int B, int Dv, hipStream_t s);

}  // namespace daisy
