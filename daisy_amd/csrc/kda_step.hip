// Token-by-token Kimi Delta Attention for decode (and short prompts) on gfx950.
//
// The recurrence of the chunked kernel, one token at a time with the fp32 state held in
// registers for the whole call:
//     S <- diag(exp(g_t)) S;   S <- S + beta_t k_t (v_t - S^T k_t)^T;   o_t = scale * S^T q_t
// This is the "fused_recurrent" mode that models/daisy/attention_kimi.py:70,144 names but does
// not support; a generation loop calls it with T = 1 per step.  At T = 1 the call is bound by
// HBM: it reads and writes the [Dk, Dv] fp32 state of every (batch, head) once (128 KiB each).
//
// Workgroup = one (batch, head) and one slab of 128 value columns (value columns are independent of each
// other; key channels beyond Dk read as zeros, whose state rows stay zero), 4 wavefronts; wavefront w
// owns value columns [32w, 32w+32) of the slab.
// Lane (dq = lane/8, jc = lane%8) holds S[16dq .. 16dq+15][32w+4jc .. +3] as 16 float4: state
// loads and stores are 128-byte row segments, the per-token vectors k, q, exp(g) are 16
// consecutive floats per lane read from LDS, and the two matrix-vector products reduce over the
// 8 dq lanes of a column group with cross-lane moves.
#include "common.h"

#include <type_traits>

namespace daisy {

constexpr int RD = 128;   // key channels and value columns a workgroup works on

struct KdaStepParams {
  const uint16_t* q; const uint16_t* k; const uint16_t* v;
  const void* g; int g_bf16;
  const float* beta;
  const float* s_in; float* s_out;
  uint16_t* o;
  int B, T, H;
  int Dk, Dv;   // the tensors' own widths (Dk <= 128)
  float scale; int l2norm; float l2eps;
  // Packed sequences (B == 1, T = all tokens): workgroup (s, h) walks rows cu[s] .. cu[s+1]-1.
  const int32_t* cu; int n_seq;
};

// Sum over the 8 lanes that share jc (lane bits 3, 4, 5).
__device__ __forceinline__ float sum_over_dq(float x) {
  x = dpp_add<0x128>(x);                 // row_ror 8: lane ^ 8 inside a row of 16
  x += __shfl_xor(x, 16);
  x += __shfl_xor(x, 32);
  return x;
}

__global__ __launch_bounds__(256) void kda_recurrent_kernel(KdaStepParams p) {
  __shared__ __attribute__((aligned(16))) float kf[RD];
  __shared__ __attribute__((aligned(16))) float qf[RD];
  __shared__ __attribute__((aligned(16))) float eg[RD];
  __shared__ float red[2][4];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int dq = lane >> 3, jc = lane & 7;
  const int h = blockIdx.x % p.H, b = blockIdx.x / p.H;
  const int col = RD * blockIdx.y + 32 * wave + 4 * jc;     // first of this lane's four value columns
  const bool col_live = col < p.Dv;                         // (Dv is a multiple of 8: four columns are live or dead together)
  const int64_t sbase = ((int64_t)(b * p.H + h) * p.Dk + 16 * dq) * p.Dv + col;

  f32x4 S[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p.s_in != nullptr && col_live && 16 * dq + i < p.Dk)
      S[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p.s_in + sbase + (int64_t)i * p.Dv));
  }

  // Token rows of this recurrence on the flattened token axis; bounds read from the device are
  // forced into 0 <= first <= end <= T so that no input can lead outside the tensors.
  int tok0 = b * p.T, tok_end = tok0 + p.T;
  if (p.cu != nullptr) {
    tok0 = min(max(p.cu[b], 0), p.T);
    tok_end = min(max(p.cu[b + 1], tok0), p.T);
  }
  for (int tok = tok0; tok < tok_end; ++tok) {
    const int64_t row = (int64_t)tok * p.H + h;
    // ---- stage k, q (L2-normalised) and exp(g) of this token in LDS ---------
    float kx = 0.f, qx = 0.f;
    if (tid < RD) {
      float gx = 0.f;
      if (tid < p.Dk) {
        kx = bf16lo_to_f32(p.k[row * p.Dk + tid]);
        qx = bf16lo_to_f32(p.q[row * p.Dk + tid]);
        gx = p.g_bf16 ? bf16lo_to_f32(reinterpret_cast<const uint16_t*>(p.g)[row * p.Dk + tid])
                      : reinterpret_cast<const float*>(p.g)[row * p.Dk + tid];
      }
      eg[tid] = __expf(gx);
    }
    if (p.l2norm) {
      float ks = kx * kx, qs = qx * qx;      // zero in wavefronts 2 and 3
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) { ks += __shfl_xor(ks, m); qs += __shfl_xor(qs, m); }
      if (lane == 0) { red[0][wave] = ks; red[1][wave] = qs; }
      __syncthreads();
      const float kn = rsqrtf(red[0][0] + red[0][1] + p.l2eps);
      const float qn = rsqrtf(red[1][0] + red[1][1] + p.l2eps);
      kx *= kn;
      qx *= qn;
    }
    if (tid < RD) { kf[tid] = kx; qf[tid] = qx; }
    u32x2 vraw = {0u, 0u};
    if (col_live) vraw = *reinterpret_cast<const u32x2*>(p.v + row * p.Dv + col);
    const f32x4 v4 = {bf16lo_to_f32(vraw.x), bf16hi_to_f32(vraw.x), bf16lo_to_f32(vraw.y), bf16hi_to_f32(vraw.y)};
    const float beta = p.beta[row];
    __syncthreads();

    // ---- decay, prediction S^T k ------------------------------------------------
    f32x4 pred = {0.f, 0.f, 0.f, 0.f};
    float kk[16];
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4 e4 = *reinterpret_cast<const f32x4*>(&eg[16 * dq + 4 * i4]);
      const f32x4 k4 = *reinterpret_cast<const f32x4*>(&kf[16 * dq + 4 * i4]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * i4 + e;
        kk[i] = k4[e];
        S[i] *= e4[e];
        pred += S[i] * k4[e];
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) pred[c] = sum_over_dq(pred[c]);
    const f32x4 delta = (v4 - pred) * beta;

    // ---- rank-one update, read-out S^T q -----------------------------------------
    f32x4 out = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4) {
      const f32x4 q4 = *reinterpret_cast<const f32x4*>(&qf[16 * dq + 4 * i4]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = 4 * i4 + e;
        S[i] += delta * kk[i];
        out += S[i] * q4[e];
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) out[c] = sum_over_dq(out[c]) * p.scale;
    if (dq == 0 && col_live) {
      u32x2 w = {pack_bf16x2(out[0], out[1]), pack_bf16x2(out[2], out[3])};
      *reinterpret_cast<u32x2*>(p.o + row * p.Dv + col) = w;
    }
    __syncthreads();   // kf / qf / eg are rewritten by the next token
  }

  if (p.s_out != nullptr && col_live) {
#pragma unroll
    for (int i = 0; i < 16; ++i)
      if (16 * dq + i < p.Dk) __builtin_nontemporal_store(S[i], reinterpret_cast<f32x4*>(p.s_out + sbase + (int64_t)i * p.Dv));
  }
}

// The same step with everything of the KDA layer that lies between its projections.
//
// What bounds it: HBM, the state in and out (134 MB for 64 sequences of 16 heads of 128 x 128: 27.6 us at what a copy
// reaches, 28.6 us measured).  As separate launches the token passed through eleven kernels (three convolutions, two
// projections from the low rank, gate, two for beta, recurrence, copy, norm), 70 us of GPU time and as much again between them.  Here one
// workgroup per (sequence, head) requests its inputs, then its state, and does the small work while the state arrives:
// the two products from the low rank are 32 KB of weights per head and matrix, read through the L2 by all sequences.
// The state's requests have to leave early: nothing ahead of them converts or branches on what was loaded, which would wait
// for it, and the weights come in whole rows.  32.8 us at the size above -> 30.0 without the waits, 28.6 with the weights
// through the LDS.
// VD / 16 wavefronts; wavefront w owns value columns [32 (w / 2), .. + 32) of half w % 2 of the key channels, lane (dq, jc)
// channels KD / 16 dq .. of that half and columns 4 jc ..: rows of 128 bytes as in kda_recurrent_kernel (with 64-byte
// rows the step of 64 sequences took 3 us more), and half as much state per lane, so that two workgroups fit a CU
// (128 registers).  The products run on the matrix cores, weights as left operand and all sixteen columns of the right
// operand the same row: fifteen of them are waste, but nothing is unpacked and nothing summed across lanes.
__device__ __forceinline__ float sum_over_rows(float x) {          // lane bits 3, 4, 5
  const LanePair r = row_pair(dpp_add<0x128>(x));                   // row_ror 8
  const LanePair t = half_pair(r.x + r.y);
  return t.x + t.y;
}
template <int KD, int VD>
__global__ __launch_bounds__(4 * VD, 4) void kda_layer_step_kernel(KdaLayerStep p) {
  constexpr int NW = VD / 16, NT = 64 * NW, ROWS = KD / 16;
  // Outputs of the low-rank products: tiles of 16 decay channels, then of 16 gate channels; wavefront w makes tiles w + NW t.
  constexpr int SLOTS = KD + VD, TILES = SLOTS / 16, TPW = (TILES + NW - 1) / NW, KS = VD / 32;
  constexpr int CH = 2 * KD + VD, CROUNDS = (CH + NT - 1) / NT;   // convolution channels: q, k, v
  __shared__ __attribute__((aligned(16))) float qkv[CH];
  __shared__ __attribute__((aligned(16))) float eg_gate[SLOTS];   // exp(g), then sigmoid(gate)
  __shared__ __attribute__((aligned(16))) f32x4 part[2][2][VD / 4];   // [half][prediction, read-out][columns]
  __shared__ float red[VD / 32];
  constexpr int RB = 2 * VD, PPR = RB / 16;                       // bytes and 16-byte pieces of a weight row
  __shared__ __attribute__((aligned(1024))) char weights[NW * TPW][16 * RB];

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = wave & 1, dq = lane >> 3, jc = lane & 7, d0 = KD / 2 * half + ROWS * dq;     // d0: this lane's first key channel
  const int ln = lane & 15, q4 = lane >> 4;                       // matrix operands: row or column ln, contraction group q4
  const int h = blockIdx.x % p.H, b = blockIdx.x / p.H;
  const int Dk = p.Dk;

  // ---- requests: the low-rank rows and weights, the convolutions' inputs, the state --------------------------------
  // Weights: the 16 rows of a tile through the LDS (a wavefront's own), swizzled, in whole rows.  Straight into operand layout,
  // 16 rows by 64 bytes per load, they kept the address unit busy for 4 us and the state's requests behind them.
#pragma unroll
  for (int t = 0; t < TPW; ++t) {
    const int s0 = 16 * min(wave + NW * t, TILES - 1);            // (surplus tiles redo the last one)
    const uint16_t* const w = s0 < KD ? p.wf + (int64_t)h * Dk * VD : p.wg + ((int64_t)h * VD + s0 - KD) * VD;
    const int rows_left = s0 < KD ? Dk - s0 : 16, row0 = s0 < KD ? s0 : 0;    // (channels beyond Dk re-read the last row)
#pragma unroll
    for (int j = 0; j < 16 * RB / 1024; ++j) {
      const int r = 1024 / RB * j + lane / PPR, piece = (lane % PPR) ^ piece_swizzle<RB>(r);
      copy16_to_lds_async(w, (row0 + min(r, rows_left - 1)) * RB + 16 * piece, lds_address(&weights[wave + NW * t][0]) + 1024 * j);
    }
  }
  u32x4 low_f[KS], low_g[KS];
#pragma unroll
  for (int m = 0; m < KS; ++m) {
    low_f[m] = *reinterpret_cast<const u32x4*>(p.f + b * p.f_row + 32 * m + 8 * q4);
    low_g[m] = *reinterpret_cast<const u32x4*>(p.g + b * p.g_row + 32 * m + 8 * q4);
  }
  // Taps and window of a channel as four bf16 aligned at the newest end: tap 3 meets the new input, window entry j tap j - 1.
  // (Nothing is converted here: that would wait for the load, and the state's requests with it.  Which convolution a channel belongs
  // to is the same for a whole wavefront, so that its pointers are scalar loads.)
  static_assert(KD % 64 == 0, "a wavefront's channels belong to one convolution");
  uint32_t xraw[CROUNDS], braw[CROUNDS];
  u32x2 cw[CROUNDS], win[CROUNDS];
#pragma unroll
  for (int r = 0; r < CROUNDS; ++r) {
    const int c0 = 64 * wave + NT * r, kind = c0 < KD ? 0 : c0 < 2 * KD ? 1 : 2, D = kind == 2 ? VD : Dk;
    const int ch = h * D + min(c0 + lane - KD * kind, D - 1);     // (channels beyond the last re-read it)
    const uint16_t* const x = kind == 0 ? p.q + b * p.q_row : kind == 1 ? p.k + b * p.k_row : p.v + b * p.v_row;
    const uint16_t* const bias = p.conv_bias[kind];
    const uint16_t *wp = p.conv_w[kind] + (int64_t)ch * p.taps, *cp = p.window[kind] + ((int64_t)b * p.H * D + ch) * p.taps;
    xraw[r] = x[ch];
    braw[r] = (bias != nullptr ? bias : x)[ch];                   // (no branch around a load either; dropped below)
    if (p.taps == 4) {
      cw[r] = *reinterpret_cast<const u32x2*>(wp);
      win[r] = *reinterpret_cast<const u32x2*>(cp);
    } else {
      const uint32_t w0 = p.taps == 3 ? wp[0] : 0, c0 = p.taps == 3 ? cp[0] : 0;
      cw[r] = u32x2{w0 << 16, (uint32_t)wp[p.taps - 2] | (uint32_t)wp[p.taps - 1] << 16};
      win[r] = u32x2{c0 << 16, (uint32_t)cp[p.taps - 2] | (uint32_t)cp[p.taps - 1] << 16};
    }
  }
  const uint32_t b_logit = p.b[b * p.b_row + h];
  const int col = 32 * (wave >> 1) + 4 * jc;
  float* const state = p.state + ((int64_t)blockIdx.x * Dk + d0) * VD + col;
  // What the products' results meet: lane (ln, q4) has row 4 q4 + ln % 4 of tile ln / 4 of every four.
  constexpr int ROUNDS = (TPW + 3) / 4;
  auto slot_of = [&](int r) { return 16 * (wave + NW * (4 * r + (ln >> 2))) + 4 * q4 + (ln & 3); };
  float dt[ROUNDS];
  uint32_t gb[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int slot = slot_of(r);
    dt[r] = p.dt_bias[h * Dk + min(slot, Dk - 1)];
    gb[r] = (p.g_bias != nullptr ? p.g_bias + (int64_t)h * VD : p.norm_w)[min(max(slot - KD, 0), VD - 1)];
  }
  const float a_log = p.A_log[h];
  const u32x2 nw = *reinterpret_cast<const u32x2*>(p.norm_w + col);
  __builtin_amdgcn_sched_barrier(0);
  f32x4 S[ROWS];                                  // (rows beyond Dk: read as copies of others, then zeroed)
  const char* const state_in = (const char*)(p.state + (int64_t)blockIdx.x * Dk * VD);
  const uint32_t at = 4u * (uint32_t)(min(d0, Dk - ROWS) * VD + col);
#pragma unroll
  for (int i = 0; i < ROWS; ++i) S[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(state_in + at + 4 * VD * i));
  __builtin_amdgcn_sched_barrier(0);

  __builtin_amdgcn_s_waitcnt(0x0F70 | ROWS);      // everything older than the state has arrived, the weights among it
  asm volatile("" ::: "memory");

  // ---- convolutions ----------------------------------------------------------------------------------------------
#pragma unroll
  for (int r = 0; r < CROUNDS; ++r) {
    const int c0 = 64 * wave + NT * r, kind = c0 < KD ? 0 : c0 < 2 * KD ? 1 : 2, D = kind == 2 ? VD : Dk;
    const int c = c0 + lane, d = c - KD * kind;
    if (c >= CH) continue;
    float a = 0.f;
    if (d < D) {
      const float x = bf16lo_to_f32(xraw[r]);
      a = p.conv_bias[kind] != nullptr ? bf16lo_to_f32(braw[r]) : 0.f;
      a = fmaf(bf16lo_to_f32(cw[r].x), bf16hi_to_f32(win[r].x), a);
      a = fmaf(bf16hi_to_f32(cw[r].x), bf16lo_to_f32(win[r].y), a);
      a = fmaf(bf16lo_to_f32(cw[r].y), bf16hi_to_f32(win[r].y), a);
      a = round_bf16(fmaf(bf16hi_to_f32(cw[r].y), x, a));
      a = round_bf16(a * __builtin_amdgcn_rcpf(1.f + __expf(-a)));
      uint16_t* cp = p.window[kind] + ((int64_t)b * p.H * D + h * D + d) * p.taps;
      const u32x2 next = {win[r].x >> 16 | win[r].y << 16, win[r].y >> 16 | xraw[r] << 16};
      if (p.taps == 4) *reinterpret_cast<u32x2*>(cp) = next;
      else {
        if (p.taps == 3) cp[0] = (uint16_t)(next.x >> 16);
        cp[p.taps - 2] = (uint16_t)next.y;
        cp[p.taps - 1] = (uint16_t)(next.y >> 16);
      }
    }
    qkv[c] = a;
  }
  // ---- g = f wf^T and gate = g wg^T + bias: every column of a tile is the same
#pragma unroll
  for (int t0 = 0; t0 < TPW; t0 += 4) {
    f32x4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (t0 + t >= TPW) continue;
      const bool decay = 16 * (wave + NW * (t0 + t)) < KD;
#pragma unroll
      for (int m = 0; m < KS; ++m)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(&weights[wave + NW * (t0 + t)][ln * RB + 16 * ((4 * m + q4) ^ piece_swizzle<RB>(ln))]),
                                                         __builtin_bit_cast(bf16x8, decay ? low_f[m] : low_g[m]), acc[t], 0, 0, 0);
    }
    f32x4 mine = acc[0];
#pragma unroll
    for (int t = 1; t < 4; ++t) mine = (ln >> 2) == t ? acc[t] : mine;
    float x = mine[0];
#pragma unroll
    for (int r = 1; r < 4; ++r) x = (ln & 3) == r ? mine[r] : x;
    const int t = t0 + (ln >> 2), slot = slot_of(t0 / 4);
    if (t < TPW && slot < SLOTS) {
      float y;
      if (slot < KD) {
        // every intermediate rounded as the tensor that holds it in the layer
        const float gl = -expf(a_log) * softplus(round_bf16(x) + dt[t0 / 4], 1.f, 20.f, 1.f);
        y = slot < Dk ? __expf(round_bf16(gl)) : 1.f;
      } else {
        if (p.g_bias != nullptr) x += bf16lo_to_f32(gb[t0 / 4]);
        y = __builtin_amdgcn_rcpf(1.f + __expf(-round_bf16(x)));
      }
      eg_gate[slot] = y;
    }
  }
  const float beta = round_bf16(1.f / (1.f + expf(-bf16lo_to_f32(b_logit))));
  __syncthreads();

  // ---- the delta rule; q and k L2-normalised (every wavefront sums for itself) ---------------------------------------
  float qs = 0.f, ks = 0.f, kq = 0.f;
#pragma unroll
  for (int e = 0; e < KD / 64; ++e) {
    const float q1 = qkv[lane + 64 * e], k1 = qkv[KD + lane + 64 * e];
    qs = fmaf(q1, q1, qs);
    ks = fmaf(k1, k1, ks);
    kq = fmaf(k1, q1, kq);
  }
  qs = sum_over_rows(group_sum<8>(qs));
  ks = sum_over_rows(group_sum<8>(ks));
  kq = sum_over_rows(group_sum<8>(kq));
  const float qn = rsqrtf(qs + p.l2_eps), kn = rsqrtf(ks + p.l2_eps);
  kq *= kn * qn;
  // With S the decayed state: pred = S^T k, delta = beta (v - pred), the new state S + k delta^T and its read-out
  // S^T q + (k . q) delta: both products over the old state in one pass and one round of cross-lane sums.
  f32x4 pred = {0.f, 0.f, 0.f, 0.f}, out = {0.f, 0.f, 0.f, 0.f};
  float kk[ROWS];
  if (d0 >= Dk) {
#pragma unroll
    for (int i = 0; i < ROWS; ++i) S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int i4 = 0; i4 < ROWS / 4; ++i4) {
    const f32x4 e4 = *reinterpret_cast<const f32x4*>(&eg_gate[d0 + 4 * i4]);
    const f32x4 k4 = *reinterpret_cast<const f32x4*>(&qkv[KD + d0 + 4 * i4]);
    const f32x4 q4v = *reinterpret_cast<const f32x4*>(&qkv[d0 + 4 * i4]);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int i = 4 * i4 + e;
      const float qq = q4v[e] * qn;
      kk[i] = k4[e] * kn;
      S[i] *= e4[e];
      pred += S[i] * kk[i];
      out += S[i] * qq;
    }
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    pred[c] = sum_over_rows(pred[c]);
    out[c] = sum_over_rows(out[c]);
  }
  if (dq == 0) {
    part[half][0][col >> 2] = pred;
    part[half][1][col >> 2] = out;
  }
  __syncthreads();
  pred = part[0][0][col >> 2] + part[1][0][col >> 2];
  out = part[0][1][col >> 2] + part[1][1][col >> 2];
  const f32x4 v4 = *reinterpret_cast<const f32x4*>(&qkv[2 * KD + col]);
  const f32x4 delta = (v4 - pred) * beta;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    S[i] += delta * kk[i];
    if (d0 + i < Dk) __builtin_nontemporal_store(S[i], reinterpret_cast<f32x4*>(state + i * VD));
  }
  // ---- gated RMS norm over the head's columns ------------------------------------
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    out[c] = round_bf16(fmaf(kq, delta[c], out[c]) * p.scale);
    ss = fmaf(out[c], out[c], ss);
  }
  ss = group_sum<8>(ss);
  if (lane == 0 && half == 0) red[wave >> 1] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int w = 0; w < VD / 32; ++w) ss += red[w];
  const float rstd = rsqrtf(ss / (float)VD + p.norm_eps);
  if (dq == 0 && half == 0) {
    const f32x4 gt = *reinterpret_cast<const f32x4*>(&eg_gate[KD + col]);
    const float w4[4] = {bf16lo_to_f32(nw.x), bf16hi_to_f32(nw.x), bf16lo_to_f32(nw.y), bf16hi_to_f32(nw.y)};
#pragma unroll
    for (int c = 0; c < 4; ++c) out[c] *= rstd * w4[c] * gt[c];
    *reinterpret_cast<u32x2*>(p.o + b * p.o_row + h * VD + col) = u32x2{pack_bf16x2(out[0], out[1]), pack_bf16x2(out[2], out[3])};
  }
}

bool kda_layer_step_serves(int Dk, int Dv, int taps) {
  return Dk >= 8 && Dk <= 128 && Dk % 8 == 0 && (Dv == 32 || Dv == 64 || Dv == 128) && taps >= 2 && taps <= 4;
}

int kda_layer_step(const KdaLayerStep& p, int B, int Dv, hipStream_t s) {
  DAISY_CHECK_SUPPORTED(kda_layer_step_serves(p.Dk, Dv, p.taps), "kda_layer_step: Dk=%d, Dv=%d, %d taps not supported", p.Dk, Dv, p.taps);
  DAISY_CHECK_ARG(B > 0 && p.H > 0 && (int64_t)B * p.H <= 0x7fffffff, "kda_layer_step: B=%d, H=%d", B, p.H);
  for (const void* t : {(const void*)p.f, (const void*)p.g, (const void*)p.wf, (const void*)p.wg, (const void*)p.state, (const void*)p.norm_w,
                        (const void*)p.o, (const void*)p.window[0], (const void*)p.window[1], (const void*)p.window[2],
                        (const void*)p.conv_w[0], (const void*)p.conv_w[1], (const void*)p.conv_w[2]})
    DAISY_CHECK_ARG(t != nullptr && (reinterpret_cast<uintptr_t>(t) & 15) == 0, "kda_layer_step: NULL or unaligned tensor");
  DAISY_CHECK_ARG(p.q && p.k && p.v && p.b && p.A_log && p.dt_bias && p.f_row % 8 == 0 && p.g_row % 8 == 0 && p.o_row % 8 == 0,
                  "kda_layer_step: NULL tensor or row stride");
  const dim3 grid((unsigned)(B * p.H));
  auto launch = [&](auto kd) {
    constexpr int KD = decltype(kd)::value;
    if (Dv == 128) hipLaunchKernelGGL((kda_layer_step_kernel<KD, 128>), grid, dim3(512), 0, s, p);
    else if (Dv == 64) hipLaunchKernelGGL((kda_layer_step_kernel<KD, 64>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((kda_layer_step_kernel<KD, 32>), grid, dim3(128), 0, s, p);
  };
  if (p.Dk <= 64) launch(std::integral_constant<int, 64>()); else launch(std::integral_constant<int, 128>());
  DAISY_CHECK_LAUNCH("kda_layer_step_kernel");
  return DAISY_OK;
}

}  // namespace daisy

using namespace daisy;

// Shared by the two entry points.  cu_seqlens == NULL: B sequences of T tokens each; otherwise
// B sequences packed into T tokens in all.
static int recurrent_launch(const void* q, const void* k, const void* v,
                            const void* g, int g_is_bf16, const float* beta, const int32_t* cu_seqlens,
                            const float* initial_state, void* o, float* final_state,
                            int B, int T, int H, int Dk, int Dv,
                            float scale, int l2norm_qk, float l2_eps, void* stream) {
  DAISY_CHECK_SUPPORTED(Dk >= 8 && Dk <= RD && Dk % 8 == 0 && Dv >= 8 && Dv % 8 == 0,
                        "kda_recurrent: Dk=%d, Dv=%d not supported (Dk: a multiple of 8 up to %d; Dv: a multiple of 8)", Dk, Dv, RD);
  DAISY_CHECK_ARG(q && k && v && g && beta && o, "kda_recurrent: q, k, v, g, beta and o must be non-NULL");
  DAISY_CHECK_ARG(B > 0 && T > 0 && H > 0, "kda_recurrent: B=%d, T=%d, H=%d must be positive", B, T, H);
  DAISY_CHECK_ARG((int64_t)B * H <= 0x7fffffff && (int64_t)B * T <= 0x7fffffff, "kda_recurrent: B*H or B*T too large");
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  DAISY_CHECK_ARG(al16(o) && al16(v) && al16(initial_state) && al16(final_state), "kda_recurrent: v, o and the states must be 16-byte aligned");
  KdaStepParams p;
  p.q = (const uint16_t*)q; p.k = (const uint16_t*)k; p.v = (const uint16_t*)v;
  p.g = g; p.g_bf16 = g_is_bf16; p.beta = beta;
  p.s_in = initial_state; p.s_out = final_state; p.o = (uint16_t*)o;
  p.B = B; p.T = T; p.H = H; p.Dk = Dk; p.Dv = Dv;
  p.scale = scale; p.l2norm = l2norm_qk; p.l2eps = l2_eps;
  p.cu = cu_seqlens; p.n_seq = cu_seqlens ? B : 0;
  DAISY_CHECK_ARG((Dv + RD - 1) / RD <= 65535, "kda_recurrent: Dv=%d too wide", Dv);
  hipLaunchKernelGGL(kda_recurrent_kernel, dim3((unsigned)(B * H), (unsigned)((Dv + RD - 1) / RD)), dim3(256), 0, (hipStream_t)stream, p);
  DAISY_CHECK_LAUNCH("kda_recurrent_kernel");
  return DAISY_OK;
}

extern "C" int daisy_kda_recurrent_fwd(const void* q, const void* k, const void* v,
                                       const void* g, int g_is_bf16, const float* beta,
                                       const float* initial_state, void* o, float* final_state,
                                       int B, int T, int H, int Dk, int Dv,
                                       float scale, int l2norm_qk, float l2_eps, void* stream) {
  return recurrent_launch(q, k, v, g, g_is_bf16, beta, nullptr, initial_state, o, final_state, B, T, H, Dk, Dv,
                          scale, l2norm_qk, l2_eps, stream);
}

extern "C" int daisy_kda_recurrent_varlen_fwd(const void* q, const void* k, const void* v,
                                              const void* g, int g_is_bf16, const float* beta,
                                              const int32_t* cu_seqlens, int n_seq,
                                              const float* initial_state, void* o, float* final_state,
                                              int T, int H, int Dk, int Dv,
                                              float scale, int l2norm_qk, float l2_eps, void* stream) {
  DAISY_CHECK_ARG(cu_seqlens != nullptr && n_seq >= 1, "kda_recurrent_varlen: cu_seqlens and n_seq >= 1 are required");
  return recurrent_launch(q, k, v, g, g_is_bf16, beta, cu_seqlens, initial_state, o, final_state, n_seq, T, H, Dk, Dv,
                          scale, l2norm_qk, l2_eps, stream);
}
