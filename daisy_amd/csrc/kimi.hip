// Streaming kernels of the KDA layer around the delta-rule core (gfx950).
//
// models/daisy/attention_kimi.py:155-158,136-137 puts three depthwise short convolutions
// (q, k, v: 4 taps, causal, SiLU) in front of chunk_kda and a gated RMS norm behind it; both
// come from a package that is absent from the reference checkout, so what is restated here is
// their documented arithmetic:
//   conv :  y[t, c] = silu( bias[c] + sum_j w[c, j] * x[t - (K-1) + j, c] ),  x[<0] from the
//           carried window (the last K-1 inputs of the previous call) or zero
//   norm :  out = x * rsqrt(mean(x^2) + eps) * weight * sigmoid(gate)      over the last dim
// Both are one pass over their tensors: 16-byte loads and stores, no LDS.
#include "common.h"

namespace daisy {

// The varlen kernel's arguments.
struct ConvParams {
  const uint16_t* x; int64_t x_sb, x_st;       // [B, T, C], channel stride 1
  const uint16_t* w;                           // [C, K]
  const uint16_t* bias;                        // [C] or null
  const uint16_t* cache_in;                    // [B, C, K] or null: the last K inputs before t = 0 (the first is unused)
  uint16_t* y; int64_t y_sb, y_st;             // [B, T, C]
  uint16_t* cache_out;                         // [B, C, K] or null: the last K inputs of the extended sequence
  int B, T, C, silu;
};
// Up to three convolutions over the same positions in one launch, told apart by the column of workgroups.
struct ConvGroup {
  ConvPart part[3];
  int block_end[3];      // first column of workgroups behind each part
  int T, silu, seg;      // seg: time steps per thread
};

constexpr int kConvSeg = 32;        // time steps per thread
constexpr int kConvSegShort = 8;    // ... of a short input

// A thread owns 8 consecutive channels and `seg` consecutive time steps; the K-1 inputs
// before its first step come from the sequence itself or from the carried window.  The sum is
// taken in fp32 and rounded to bf16 before the activation, which is again evaluated in fp32 and
// rounded (the two roundings of a bf16 convolution followed by a bf16 SiLU).
template <int K>
__global__ __launch_bounds__(256) void short_conv_kernel(ConvGroup group) {
  int part = 0;
  while (part < 2 && (int)blockIdx.x >= group.block_end[part]) ++part;
  const ConvPart p = group.part[part];
  const int T = group.T;
  const int cg = (blockIdx.x - (part > 0 ? group.block_end[part - 1] : 0)) * 256 + threadIdx.x;        // group of 8 channels
  const int c0 = 8 * cg;
  if (c0 >= p.C) return;
  const int b = blockIdx.z;
  const int t0 = blockIdx.y * group.seg;
  const int t1 = min(t0 + group.seg, T);

  // The rows ahead of the first step are asked for beside the weights, without a branch around any (ahead of the sequence: its first row, put
  // right below): behind a branch each was waited for by itself, 6.6 -> 5.6 us for 3 x 235 rows of 3 x 512 channels.  (The first steps' rows
  // with them: the same there, 32768 rows of 3 x 2048 channels 130.3 -> 132.3.)
  constexpr int U = 8;   // steps whose inputs are in flight together
  auto load_row = [&](int t) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.x + b * p.x_sb + (int64_t)t * p.x_st + c0)); };
  u32x4 before[K - 1], raw[U];
#pragma unroll
  for (int j = 0; j < K - 1; ++j) before[j] = load_row(max(t0 - (K - 1) + j, 0));
  __builtin_amdgcn_sched_barrier(0);
  float w[K][8], acc0[8];
  {
    // channel c's taps are K consecutive values; 8 channels = 8K consecutive bf16
    const uint16_t* wp = p.w + (int64_t)c0 * K;
    if (K == 4) {   // 64 contiguous bytes: four 16-byte loads, two channels each
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float f[8];
        unpack8(*reinterpret_cast<const u32x4*>(wp + 8 * v), f);
#pragma unroll
        for (int j = 0; j < K; ++j) { w[j][2 * v] = f[j % 8]; w[j][2 * v + 1] = f[(4 + j) % 8]; }
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int j = 0; j < K; ++j) w[j][e] = bf16lo_to_f32(wp[e * K + j]);
    }
    if (p.bias != nullptr) unpack8(*reinterpret_cast<const u32x4*>(p.bias + c0), acc0);
    else {
#pragma unroll
      for (int e = 0; e < 8; ++e) acc0[e] = 0.f;
    }
  }
  // The carried window of 8 channels is 8K contiguous values; for K = 4 it is read and written
  // as four 16-byte pieces (two channels each).
  float carried[K][8];
  if (K == 4 && p.cache_in != nullptr && t0 < K - 1) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      float f[8];
      unpack8(*reinterpret_cast<const u32x4*>(p.cache_in + ((int64_t)b * p.C + c0) * K + 8 * v), f);
#pragma unroll
      for (int j = 0; j < K; ++j) { carried[j][2 * v] = f[j % 8]; carried[j][2 * v + 1] = f[(4 + j) % 8]; }
    }
  }
  // Input at time ti < 0: carried window or zero.
  auto input_ahead = [&](int ti, float* f) {
    if (p.cache_in != nullptr) {
      if (K == 4) {
#pragma unroll
        for (int j = 1; j < K; ++j)
          if (K + ti == j) {
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = carried[j][e];
          }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = bf16lo_to_f32(p.cache_in[((int64_t)b * p.C + c0 + e) * K + K + ti]);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = 0.f;
    }
  };

  float win[K - 1][8];   // win[j] = input at t - (K-1) + j for the step t about to be computed
#pragma unroll
  for (int j = 0; j < K - 1; ++j) {
    unpack8(before[j], win[j]);
    if (t0 - (K - 1) + j < 0) input_ahead(t0 - (K - 1) + j, win[j]);
  }
  for (int tb = t0; tb < t1; tb += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) raw[u] = load_row(min(tb + u, T - 1));
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float xin[8], out[8];
      unpack8(raw[u], xin);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float a = acc0[e];
#pragma unroll
        for (int j = 0; j < K - 1; ++j) a = fmaf(w[j][e], win[j][e], a);
        a = round_bf16(fmaf(w[K - 1][e], xin[e], a));
        if (group.silu) a = a * __builtin_amdgcn_rcpf(1.f + __expf(-a));
        out[e] = a;
      }
      if (tb + u < t1) *reinterpret_cast<u32x4*>(p.y + b * p.y_sb + (int64_t)(tb + u) * p.y_st + c0) = pack8(out);
#pragma unroll
      for (int j = 0; j + 1 < K - 1; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) win[j][e] = win[j + 1][e];
#pragma unroll
      for (int e = 0; e < 8; ++e) win[K - 2][e] = xin[e];
    }
  }
  // The thread that reaches the end of the sequence leaves the window for the next call.
  if (p.cache_out != nullptr && t1 == T) {
    float last[K][8];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (T - K + j >= 0) unpack8(load_row(T - K + j), last[j]);
      else input_ahead(T - K + j, last[j]);
    }
    if (K == 4) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float f[8];
#pragma unroll
        for (int j = 0; j < K; ++j) { f[j % 8] = last[j][2 * v]; f[(4 + j) % 8] = last[j][2 * v + 1]; }
        *reinterpret_cast<u32x4*>(p.cache_out + ((int64_t)b * p.C + c0) * K + 8 * v) = pack8(f);
      }
    } else {
#pragma unroll
      for (int j = 0; j < K; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          p.cache_out[((int64_t)b * p.C + c0 + e) * K + j] = (uint16_t)(pack_bf16x2(last[j][e], 0.f) & 0xffffu);
    }
  }
}

// Sequences packed along T of a batch of one: the taps of a step must not reach across the start of
// the step's sequence (they read the sequence's carried window [n_seq, C, K] or zero instead), and
// every sequence leaves its own window.  The bounds cu [n_seq + 1] are read on the device and forced
// into 0..T; a thread finds the sequence of its first step by bisection and walks on from there.
// Taps are re-read from global memory (they hit the cache) instead of kept in registers, which keeps
// the boundary handling in one place.
template <int K>
__global__ __launch_bounds__(256) void short_conv_varlen_kernel(ConvParams p, const int32_t* cu, int n_seq) {
  const int cg = blockIdx.x * 256 + threadIdx.x;
  const int c0 = 8 * cg;
  if (c0 >= p.C) return;
  const int t0 = blockIdx.y * kConvSeg;
  const int t1 = min(t0 + kConvSeg, p.T);
  auto bound = [&](int i) { return min(max(cu[i], 0), p.T); };

  float w[K][8], acc0[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
#pragma unroll
    for (int j = 0; j < K; ++j) w[j][e] = bf16lo_to_f32(p.w[(int64_t)(c0 + e) * K + j]);
    acc0[e] = p.bias ? bf16lo_to_f32(p.bias[c0 + e]) : 0.f;
  }
  // Input of sequence `seq` (first row `start`) at row ti; rows before the start come from the window.
  auto input_at = [&](int seq, int start, int ti, float* f) {
    if (ti >= start) {
      unpack8(*reinterpret_cast<const u32x4*>(p.x + (int64_t)ti * p.x_st + c0), f);
    } else {
      const int slot = K + (ti - start);     // window slot: K-1 is the input just before the sequence
#pragma unroll
      for (int e = 0; e < 8; ++e)
        f[e] = (p.cache_in != nullptr && seq < n_seq && slot >= 0) ? bf16lo_to_f32(p.cache_in[((int64_t)seq * p.C + c0 + e) * K + slot]) : 0.f;
    }
  };
  auto leave_window = [&](int seq, int start, int end) {
#pragma unroll
    for (int j = 0; j < K; ++j) {
      float f[8];
      input_at(seq, start, end - K + j, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) p.cache_out[((int64_t)seq * p.C + c0 + e) * K + j] = (uint16_t)(pack_bf16x2(f[e], 0.f) & 0xffffu);
    }
  };

  // smallest seq in [0, n_seq] whose end lies beyond t0 (n_seq: rows behind the last bound, a sequence
  // of their own without a window)
  int lo = 0, hi = n_seq;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (bound(mid + 1) > t0) hi = mid; else lo = mid + 1;
  }
  int seq = lo;
  int start = bound(min(seq, n_seq)), end = seq < n_seq ? bound(seq + 1) : p.T;
  for (int t = t0; t < t1; ++t) {
    while (t >= end && seq < n_seq) {
      ++seq;
      start = bound(min(seq, n_seq));
      end = seq < n_seq ? bound(seq + 1) : p.T;
    }
    float a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = acc0[e];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      float f[8];
      input_at(seq, start, t - (K - 1) + j, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) a[e] = fmaf(w[j][e], f[e], a[e]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      a[e] = round_bf16(a[e]);
      if (p.silu) a[e] = a[e] * __builtin_amdgcn_rcpf(1.f + __expf(-a[e]));
    }
    *reinterpret_cast<u32x4*>(p.y + (int64_t)t * p.y_st + c0) = pack8(a);
    if (p.cache_out != nullptr && seq < n_seq && t == end - 1) leave_window(seq, start, end);
  }
  // Empty sequences keep their window; the threads of the first time segment see to it.
  if (p.cache_out != nullptr && blockIdx.y == 0) {
    for (int i = 0; i < n_seq; ++i) {
      const int b0 = bound(i), b1 = bound(i + 1);
      if (b1 <= b0) leave_window(i, b0, b0);
    }
  }
}

struct GatedNormParams {
  const uint16_t* x; const uint16_t* gate; const uint16_t* weight; uint16_t* out;
  int64_t rows; float eps;
};

// D/8 lanes share a row; statistics in fp32 over the row, one rounding at the end.
template <int D>
__global__ __launch_bounds__(256) void gated_rmsnorm_kernel(GatedNormParams p) {
  constexpr int LPR = D / 8;
  const int64_t row = ((int64_t)blockIdx.x * 256 + threadIdx.x) / LPR;
  const int c = threadIdx.x % LPR;
  const int64_t r = row < p.rows ? row : p.rows - 1;   // surplus lanes redo the last row (the sums need full groups)
  float x[8], g[8], w[8], o[8];
  unpack8(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.x + r * D + 8 * c)), x);
  unpack8(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.gate + r * D + 8 * c)), g);
  unpack8(*reinterpret_cast<const u32x4*>(p.weight + 8 * c), w);
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
  ss = group_sum<LPR>(ss);
  const float rstd = rsqrtf(ss / (float)D + p.eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = x[e] * rstd * w[e] * __builtin_amdgcn_rcpf(1.f + __expf(-g[e]));
  if (row < p.rows) *reinterpret_cast<u32x4*>(p.out + r * D + 8 * c) = pack8(o);
}

bool gated_rmsnorm_serves(int D) { return D == 32 || D == 64 || D == 128 || D == 256; }

// ---- the low-rank products of the KDA layer with what follows them ---------------------------------------------
// y [M, N] = x [M, K] w [N, K]^T with K = 64 or 128, the width of a value head: two or four products deep, so that it is all operands and
// results.  A workgroup keeps its columns of w (a head's, or 128) in the LDS as operands, and each of its wavefronts takes block after block
// of 16 rows of x, straight from memory, the next block's while the present one is worked on.  The rows of w are dealt to the accumulators
// such that a lane ends with 8 consecutive columns of a row; rounded to bf16 they pass through a corner of the LDS, 4 KB, and what follows
// works on whole rows, 4 of them per access (straight from the accumulators' layout, 64 bytes of 16 rows per access, 134 MB were stored in
// 75 us).
// EPI 0: the decay gate, and beta.  EPI 1: the output gate, and with it the gated RMS norm of the rows of o, in place; the gate itself is
// not written.
// 32768 rows of 16 heads of 128: the two products as tiles of 128 x 128 with the gate in their epilogue and gated_rmsnorm_kernel behind them took
// 115 + 62 us; these take 61 (134 MB written, 36 us of vector instructions) and 61 us (276 MB).  Beta is shared out among the groups of columns: as
// the first group's it came last in the launch, a chain of loads of 25 us.
// Nothing in the loop is conditional: rows and columns past the end are the last ones over again, stored as such.  (Behind a branch around
// a store the next block's operands are waited for together with the stores.)
struct LowRankParams {
  const uint16_t* x; int64_t x_sm;
  const uint16_t* w;
  int M, N, groups;                    // groups of columns
  KdaGates gates; uint16_t* y;         // EPI 0
  const uint16_t* bias; const uint16_t* weight; uint16_t* o; float eps;      // EPI 1: bias [N] or NULL, norm weight [K], o [M, N]
};
constexpr int kLowRankWaves = 4;
template <int K, int EPI>
__global__ __launch_bounds__(64 * kLowRankWaves, 3) void low_rank_kernel(LowRankParams p) {
  constexpr int COLS = EPI == 0 ? 128 : K, NG = COLS / 32, KS = K / 32;        // columns of a wavefront, groups of 32 of them, products per sum
  constexpr int LPR = COLS / 8, RPA = 64 / LPR, NR = 16 / RPA;                 // lanes per row, rows per access, accesses per block
  __shared__ __attribute__((aligned(16))) u32x4 ws[2 * NG][KS][64];
  __shared__ __attribute__((aligned(16))) u32x4 turn[kLowRankWaves][16][LPR];
  __shared__ __attribute__((aligned(16))) float bs[COLS];                      // EPI 1: the gate's bias
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int piece = lane % LPR, row_in = lane / LPR;                           // the lane's place in whole rows
  // The columns of a walker's rows in consecutive workgroups of one XCD, whose L2 then holds these rows of x.
  const int in_xcd = blockIdx.x >> 3, n0 = in_xcd % p.groups * COLS;
  const int walker = (in_xcd / p.groups * 8 + (blockIdx.x & 7)) * kLowRankWaves + wave, walkers = gridDim.x / p.groups * kLowRankWaves;
  const int blocks = (p.M + 15) / 16;
  const int col8 = min(n0 + 8 * piece, p.N - 8);

  auto load_x = [&](int block, u32x4* xv) {
    const uint16_t* row = p.x + (int64_t)min(16 * block + li, p.M - 1) * p.x_sm + 8 * q4;
#pragma unroll
    for (int s = 0; s < KS; ++s) xv[s] = *reinterpret_cast<const u32x4*>(row + 32 * s);
  };
  auto row_at = [&](int block, int j) { return (int64_t)min(16 * block + RPA * j + row_in, p.M - 1) * p.N + col8; };
  auto load_o = [&](int block, u32x4* ov) {
#pragma unroll
    for (int j = 0; j < NR; ++j) ov[j] = *reinterpret_cast<const u32x4*>(p.o + row_at(block, j));
  };
  u32x4 xv[KS], ov[EPI == 1 ? NR : 1];
  load_x(min(walker, blocks - 1), xv);
  if constexpr (EPI == 1) load_o(min(walker, blocks - 1), ov);
  // Row a of tile 2 m + u is column 32 m + 8 (a / 4) + 4 u + a % 4: a lane's rows of the two tiles are columns 32 m + 8 q4 ..
#pragma unroll
  for (int t = wave; t < 2 * NG; t += kLowRankWaves) {
    const int col = min(n0 + 32 * (t >> 1) + 8 * (li >> 2), p.N - 8) + 4 * (t & 1) + (li & 3);
    const uint16_t* row = p.w + (int64_t)col * K + 8 * q4;
#pragma unroll
    for (int s = 0; s < KS; ++s) ws[t][s][lane] = *reinterpret_cast<const u32x4*>(row + 32 * s);
  }
  if (EPI == 1 && tid < COLS) bs[tid] = p.bias != nullptr ? bf16lo_to_f32(p.bias[n0 + tid]) : 0.f;
  // What goes with the lane's columns: the decay gate's bias and scale, or the norm's weight.
  float c8[8], scale = 1.f;
  if constexpr (EPI == 0) {
    scale = -expf(p.gates.A_log[col8 / p.gates.Dk]);
#pragma unroll
    for (int e = 0; e < 8; ++e) c8[e] = p.gates.dt_bias[col8 + e];
  } else {
    unpack8(*reinterpret_cast<const u32x4*>(p.weight + 8 * piece), c8);
  }
  __syncthreads();

  for (int block = walker; block < blocks; block += walkers) {
    f32x4 acc[2 * NG];
#pragma unroll
    for (int t = 0; t < 2 * NG; ++t)
      acc[t] = EPI == 1 ? *reinterpret_cast<const f32x4*>(&bs[32 * (t >> 1) + 8 * q4 + 4 * (t & 1)]) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const bf16x8 xs = __builtin_bit_cast(bf16x8, xv[s]);
#pragma unroll
      for (int t = 0; t < 2 * NG; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ws[t][s][lane]), xs, acc[t], 0, 0, 0);
    }
    const int next = min(block + walkers, blocks - 1);
    load_x(next, xv);
#pragma unroll
    for (int m = 0; m < NG; ++m)
      turn[wave][li][(4 * m + q4) ^ (li & (LPR - 1))] =
          u32x4{pack_bf16x2(acc[2 * m][0], acc[2 * m][1]), pack_bf16x2(acc[2 * m][2], acc[2 * m][3]),
                pack_bf16x2(acc[2 * m + 1][0], acc[2 * m + 1][1]), pack_bf16x2(acc[2 * m + 1][2], acc[2 * m + 1][3])};
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    u32x4 of[EPI == 1 ? NR : 1];
    if constexpr (EPI == 1) {
#pragma unroll
      for (int j = 0; j < NR; ++j) of[j] = ov[j];
      load_o(next, ov);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < NR; ++j) {
      const int r = RPA * j + row_in;
      float y[8], f[8];
      unpack8(turn[wave][r][piece ^ (r & (LPR - 1))], y);
      if constexpr (EPI == 0) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = scale * softplus(y[e] + c8[e]);
        *reinterpret_cast<u32x4*>(p.y + row_at(block, j)) = pack8(f);
      } else {
        float x[8], ss = 0.f;
        unpack8(of[j], x);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fmaf(x[e], x[e], ss);
        ss = group_sum<LPR>(ss);
        const float rstd = rsqrtf(ss / (float)K + p.eps);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = x[e] * rstd * c8[e] * __builtin_amdgcn_rcpf(1.f + __expf(-y[e]));
        *reinterpret_cast<u32x4*>(p.o + row_at(block, j)) = pack8(f);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  if (EPI == 0) {                      // beta of the walker's rows, a block in turn by every group of columns
    for (int block = walker + walkers * (in_xcd % p.groups); block < blocks; block += walkers * p.groups) {
      const int count = min(16, p.M - 16 * block) * p.gates.H;
      for (int i = lane; i < count; i += 64) {
        const float logit = bf16lo_to_f32(p.gates.logits[(int64_t)(16 * block + i / p.gates.H) * p.gates.logits_row + i % p.gates.H]);
        p.gates.beta[(int64_t)16 * block * p.gates.H + i] = round_bf16(1.f / (1.f + expf(-logit)));
      }
    }
  }
}

// Workgroups per group of columns.  Three workgroups fit a compute unit; every wavefront walks the rows as often as that takes.  Whole
// eights, one per XCD, and never none: a layer of more than 768 heads has more groups than fit.  More than fit at once walk a whole share
// alone at the end, so the eights are rounded down, unless that leaves a sixth of the chip empty (gate / gated norm, heads of 128, rounded up ->
// down, us: 10 heads x 52343 rows 57.5 / 77.3 -> 53.6 / 67.6, 14 x 37388 56.7 / 78.2 -> 54.6 / 71.6, 22 x 23792 54.5 / 75.4 -> 53.1 / 69.5, 22 x 5681
// 19.8 / 21.3 -> 21.2 / 19.8; but 40 x 13085 53.7 / 71.8 -> 58.0 / 74.9).
int low_rank_walkers(int M, int groups) {
  const int wanted = (M + 16 * kLowRankWaves - 1) / (16 * kLowRankWaves), fit = 768 / groups, down = fit / 8 * 8;
  const int most = down * groups > 640 ? down : (fit / 8 + 1) * 8;
  return wanted < most ? (wanted + 7) / 8 * 8 : most;
}
template <int K, int EPI>
static int launch_low_rank(LowRankParams& p, hipStream_t s) {
  p.groups = EPI == 0 ? (p.N + 127) / 128 : p.N / K;
  hipLaunchKernelGGL((low_rank_kernel<K, EPI>), dim3((unsigned)(low_rank_walkers(p.M, p.groups) * p.groups)), dim3(64 * kLowRankWaves), 0, s, p);
  DAISY_CHECK_LAUNCH("low_rank_kernel");
  return DAISY_OK;
}
// From about four million outputs on.  Below, a workgroup's own latencies (its columns into the LDS, a block or two, beta) are what the call waits
// for, and tiles have fewer of them: a layer's call, tiles and the gated norm / these kernels, 64 rows of 8 heads of 128 41.5 / 47.8 us, 200 of 16
// 62 / 67, 777 of 12 89.5 / 91.5, 2048 of 16 175 / 175, 8000 of 8 222 / 218, 32768 of 8 of 64 420 / 404, 40000 of 16 of 128 2190 / 2120.
// Asked of the gate's outputs for both kernels, also where values are wider or narrower than keys: from four million on the pair is ahead of tiles and norm
// at every ratio (in a recorded chain, 16 heads, keys by values: 128 by 64, 2001 rows 16.8 / 13.9, 64 by 128, 4003 rows 27.1 / 23.6, 256 by 64, 1000 rows
// 14.3 / 12.0), and one of them with tiles for the other is a launch more than either (17.8, 31.2, 15.6 with the gate's own kernel).
bool low_rank_wanted(int M, int N, int K) { return (K == 64 || K == 128) && (int64_t)M * N >= 4000000; }
static int low_rank_check(const LowRankParams& p, int K) {
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  DAISY_CHECK_SUPPORTED(K == 64 || K == 128, "low_rank: K=%d (64 or 128)", K);
  DAISY_CHECK_ARG(p.x && p.w && p.M > 0 && p.N >= 8 && p.N % 8 == 0 && al16(p.x) && al16(p.w) && p.x_sm % 8 == 0 && p.x_sm >= K,
                  "low_rank: M=%d, N=%d, rows %lld elements apart on 16-byte boundaries", p.M, p.N, (long long)p.x_sm);
  return DAISY_OK;
}
int low_rank_gate(const uint16_t* x, int64_t x_sm, const uint16_t* w, const KdaGates& gates, uint16_t* y, int M, int N, int K, hipStream_t s) {
  LowRankParams p{};
  p.x = x; p.x_sm = x_sm; p.w = w; p.M = M; p.N = N; p.gates = gates; p.y = y;
  if (const int rc = low_rank_check(p, K); rc != DAISY_OK) return rc;
  DAISY_CHECK_ARG(y && gates.A_log && gates.dt_bias && gates.logits && gates.beta && gates.H > 0 && gates.Dk % 8 == 0 && N == gates.H * gates.Dk &&
                      (reinterpret_cast<uintptr_t>(y) & 15) == 0, "low_rank_gate: %d heads of %d channels on a product of %d", gates.H, gates.Dk, N);
  return K == 64 ? launch_low_rank<64, 0>(p, s) : launch_low_rank<128, 0>(p, s);
}
int low_rank_norm(const uint16_t* x, int64_t x_sm, const uint16_t* w, const uint16_t* bias, const uint16_t* norm_weight, uint16_t* o, float eps,
                  int M, int N, int K, hipStream_t s) {
  LowRankParams p{};
  p.x = x; p.x_sm = x_sm; p.w = w; p.M = M; p.N = N; p.bias = bias; p.weight = norm_weight; p.o = o; p.eps = eps;
  if (const int rc = low_rank_check(p, K); rc != DAISY_OK) return rc;
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  DAISY_CHECK_ARG(o && norm_weight && N % K == 0 && al16(o) && al16(bias) && al16(norm_weight), "low_rank_norm: N=%d in heads of %d, tensors on 16-byte boundaries", N, K);
  return K == 64 ? launch_low_rank<64, 1>(p, s) : launch_low_rank<128, 1>(p, s);
}

}  // namespace daisy

using namespace daisy;

// A thread walks its steps eight inputs at a time, so a short input, whose threads do not fill the chip, lasts as long as one
// thread's chain of loads: threads of eight steps there (three more rows read per eight, all cached).  The KDA layer over 64 rows
// of 8 heads of 128: 50.5 -> 46.3 us, 300 rows of 12: 65 -> 59.5, 2048 rows of 16: 210.5 -> 208.3; level from a workgroup per compute unit on.
int daisy::short_conv_group(const ConvPart* parts, int n, int B, int T, int K, int silu, hipStream_t s) {
  DAISY_CHECK_ARG(parts && n >= 1 && n <= 3 && B > 0 && T > 0, "short_conv: %d parts, B=%d, T=%d", n, B, T);
  DAISY_CHECK_SUPPORTED(K >= 2 && K <= 4, "short_conv: kernel size %d not supported (2..4)", K);
  DAISY_CHECK_ARG(B <= 65535, "short_conv: B must be <= 65535");
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  ConvGroup g{};
  int columns = 0;
  bool in_place = false;
  for (int i = 0; i < 3; ++i) {
    if (i < n) {
      const ConvPart& p = parts[i];
      DAISY_CHECK_ARG(p.x && p.w && p.y && p.C > 0, "short_conv: x, weight and y must be non-NULL, C=%d positive", p.C);
      DAISY_CHECK_SUPPORTED(p.C % 8 == 0, "short_conv: channels (%d) must be a multiple of 8", p.C);
      DAISY_CHECK_ARG(al16(p.x) && al16(p.y) && al16(p.bias) && al16(p.w) && al16(p.cache_in) && al16(p.cache_out),
                      "short_conv: x, y, weight, bias and the windows must be 16-byte aligned");
      DAISY_CHECK_ARG(p.x_sb % 8 == 0 && p.x_st % 8 == 0 && p.y_sb % 8 == 0 && p.y_st % 8 == 0, "short_conv: strides must be multiples of 8 elements");
      // Updating the window in place is safe only while the thread that writes it is the one that read it.
      const bool same = p.cache_out != nullptr && p.cache_out == p.cache_in;
      DAISY_CHECK_ARG(!same || T <= kConvSeg, "short_conv: the window can be updated in place for T <= %d only (T=%d)", kConvSeg, T);
      in_place |= same;
      g.part[i] = p;
      columns += (p.C / 8 + 255) / 256;
    }
    g.block_end[i] = columns;
  }
  g.T = T; g.silu = silu;
  const int64_t workgroups = (int64_t)columns * B * ((T + kConvSeg - 1) / kConvSeg);
  g.seg = workgroups < 256 && !in_place ? kConvSegShort : kConvSeg;
  const dim3 grid((unsigned)columns, (unsigned)((T + g.seg - 1) / g.seg), (unsigned)B);
  DAISY_CHECK_ARG(grid.y <= 65535, "short_conv: T=%d too long for one launch", T);
  if (K == 4) hipLaunchKernelGGL(short_conv_kernel<4>, grid, dim3(256), 0, s, g);
  else if (K == 3) hipLaunchKernelGGL(short_conv_kernel<3>, grid, dim3(256), 0, s, g);
  else hipLaunchKernelGGL(short_conv_kernel<2>, grid, dim3(256), 0, s, g);
  DAISY_CHECK_LAUNCH("short_conv_kernel");
  return DAISY_OK;
}

extern "C" int daisy_short_conv_fwd(const void* x, const int64_t* x_strides, const void* weight, const void* bias,
                                    const void* cache_in, void* y, const int64_t* y_strides, void* cache_out,
                                    int B, int T, int C, int K, int apply_silu, void* stream) {
  DAISY_CHECK_ARG(x && weight && y && x_strides && y_strides, "short_conv: x, weight, y and the stride arrays must be non-NULL");
  DAISY_CHECK_ARG(B > 0 && T > 0 && C > 0, "short_conv: B=%d, T=%d, C=%d must be positive", B, T, C);
  const ConvPart p{(const uint16_t*)x, x_strides[0], x_strides[1], (const uint16_t*)weight, (const uint16_t*)bias, (const uint16_t*)cache_in,
                   (uint16_t*)y, y_strides[0], y_strides[1], (uint16_t*)cache_out, C};
  return daisy::short_conv_group(&p, 1, B, T, K, apply_silu, (hipStream_t)stream);
}

extern "C" int daisy_short_conv_varlen_fwd(const void* x, int64_t x_row_stride, const void* weight, const void* bias,
                                           const int32_t* cu_seqlens, int n_seq, const void* cache_in,
                                           void* y, int64_t y_row_stride, void* cache_out,
                                           int T, int C, int K, int apply_silu, void* stream) {
  DAISY_CHECK_ARG(x && weight && y, "short_conv_varlen: x, weight and y must be non-NULL");
  DAISY_CHECK_ARG(cu_seqlens != nullptr && n_seq >= 1, "short_conv_varlen: cu_seqlens and n_seq >= 1 are required");
  DAISY_CHECK_ARG(T > 0 && C > 0, "short_conv_varlen: T=%d, C=%d must be positive", T, C);
  DAISY_CHECK_SUPPORTED(K >= 2 && K <= 4, "short_conv_varlen: kernel size %d not supported (2..4)", K);
  DAISY_CHECK_SUPPORTED(C % 8 == 0, "short_conv_varlen: channels (%d) must be a multiple of 8", C);
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  DAISY_CHECK_ARG(al16(x) && al16(y) && x_row_stride % 8 == 0 && y_row_stride % 8 == 0,
                  "short_conv_varlen: x and y must be 16-byte aligned with row strides that are multiples of 8 elements");
  DAISY_CHECK_ARG(cache_out == nullptr || cache_out != cache_in, "short_conv_varlen: the windows cannot be updated in place");
  ConvParams p;
  p.x = (const uint16_t*)x; p.x_sb = 0; p.x_st = x_row_stride;
  p.w = (const uint16_t*)weight; p.bias = (const uint16_t*)bias; p.cache_in = (const uint16_t*)cache_in;
  p.y = (uint16_t*)y; p.y_sb = 0; p.y_st = y_row_stride;
  p.cache_out = (uint16_t*)cache_out;
  p.B = 1; p.T = T; p.C = C; p.silu = apply_silu;
  const dim3 grid((unsigned)((C / 8 + 255) / 256), (unsigned)((T + kConvSeg - 1) / kConvSeg), 1);
  DAISY_CHECK_ARG(grid.y <= 65535, "short_conv_varlen: T=%d too long for one launch", T);
  hipStream_t s = (hipStream_t)stream;
  if (K == 4) hipLaunchKernelGGL(short_conv_varlen_kernel<4>, grid, dim3(256), 0, s, p, cu_seqlens, n_seq);
  else if (K == 3) hipLaunchKernelGGL(short_conv_varlen_kernel<3>, grid, dim3(256), 0, s, p, cu_seqlens, n_seq);
  else hipLaunchKernelGGL(short_conv_varlen_kernel<2>, grid, dim3(256), 0, s, p, cu_seqlens, n_seq);
  DAISY_CHECK_LAUNCH("short_conv_varlen_kernel");
  return DAISY_OK;
}

extern "C" int daisy_gated_rmsnorm_fwd(const void* x, const void* gate, const void* weight, void* out,
                                       int64_t rows, int D, float eps, void* stream) {
  DAISY_CHECK_ARG(x && gate && weight && out, "gated_rmsnorm: x, gate, weight and out must be non-NULL");
  DAISY_CHECK_ARG(rows > 0, "gated_rmsnorm: rows=%lld must be positive", (long long)rows);
  DAISY_CHECK_SUPPORTED(gated_rmsnorm_serves(D), "gated_rmsnorm: last dim %d not supported (32, 64, 128 or 256)", D);
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  DAISY_CHECK_ARG(al16(x) && al16(gate) && al16(weight) && al16(out), "gated_rmsnorm: tensors must be 16-byte aligned");
  GatedNormParams p;
  p.x = (const uint16_t*)x; p.gate = (const uint16_t*)gate; p.weight = (const uint16_t*)weight; p.out = (uint16_t*)out;
  p.rows = rows; p.eps = eps;
  const int64_t nwg = (rows * (D / 8) + 255) / 256;
  DAISY_CHECK_ARG(nwg <= 0x7fffffff, "gated_rmsnorm: too many rows (%lld)", (long long)rows);
  hipStream_t s = (hipStream_t)stream;
  if (D == 128) hipLaunchKernelGGL(gated_rmsnorm_kernel<128>, dim3((unsigned)nwg), dim3(256), 0, s, p);
  else if (D == 256) hipLaunchKernelGGL(gated_rmsnorm_kernel<256>, dim3((unsigned)nwg), dim3(256), 0, s, p);
  else if (D == 32) hipLaunchKernelGGL(gated_rmsnorm_kernel<32>, dim3((unsigned)nwg), dim3(256), 0, s, p);
  else hipLaunchKernelGGL(gated_rmsnorm_kernel<64>, dim3((unsigned)nwg), dim3(256), 0, s, p);
  DAISY_CHECK_LAUNCH("gated_rmsnorm_kernel");
  return DAISY_OK;
}
