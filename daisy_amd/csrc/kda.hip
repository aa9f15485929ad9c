// Kernel 3: chunked Kimi Delta Attention forward and its log-decay gate (gfx950).
#include "common.h"
#include <type_traits>

namespace daisy {

// out = -exp(A_log[h]) * softplus(g + bias[h, d]).  VEC = 8: a thread takes 8 consecutive channels
// (Dk a multiple of 8), 16-byte accesses; VEC = 1: one element per thread, any Dk.
template <bool BF16, int VEC>
__global__ __launch_bounds__(256) void kda_gate_kernel(const void* g, const float* A_log, const float* bias, void* out,
                                                       int64_t total, int H, int Dk, float sp_beta, float threshold) {
  const uint32_t vi = blockIdx.x * blockDim.x + threadIdx.x;   // 32-bit index arithmetic (64-bit division is slow)
  const int64_t i = (int64_t)vi * VEC;
  if (i >= total) return;
  const uint32_t per_row = (uint32_t)(H * Dk) / VEC, in_row = vi % per_row;
  const int h = (int)(in_row / (uint32_t)(Dk / VEC));
  const int d = (int)(in_row % (uint32_t)(Dk / VEC)) * VEC;
  const float scale = -expf(A_log[h]);
  float x[VEC], y[VEC];
  if (VEC == 8) {
    if (BF16) unpack8(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>((const uint16_t*)g + i)), x);
    else {
      const f32x4 a = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>((const float*)g + i));
      const f32x4 b = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>((const float*)g + i + 4));
#pragma unroll
      for (int e = 0; e < 4; ++e) { x[e] = a[e]; x[4 + e] = b[e]; }
    }
  } else {
    x[0] = BF16 ? bf16lo_to_f32(((const uint16_t*)g)[i]) : ((const float*)g)[i];
  }
  float bv[VEC];
  if (bias == nullptr) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) bv[e] = 0.f;
  } else if (VEC == 8) {
    const f32x4 b0 = *reinterpret_cast<const f32x4*>(bias + h * Dk + d), b1 = *reinterpret_cast<const f32x4*>(bias + h * Dk + d + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { bv[e] = b0[e]; bv[(4 + e) % VEC] = b1[e]; }
  } else {
    bv[0] = bias[h * Dk + d];
  }
  const float inv_beta = 1.f / sp_beta;
#pragma unroll
  for (int e = 0; e < VEC; ++e) y[e] = scale * softplus(x[e] + bv[e], sp_beta, threshold, inv_beta);
  if (VEC == 8) {
    if (BF16) *reinterpret_cast<u32x4*>((uint16_t*)out + i) = pack8(y);
    else {
      *reinterpret_cast<f32x4*>((float*)out + i) = f32x4{y[0], y[1], y[2], y[3]};
      *reinterpret_cast<f32x4*>((float*)out + i + 4) = f32x4{y[4], y[5], y[6], y[7]};
    }
  } else {
    if (BF16) ((uint16_t*)out)[i] = (uint16_t)(pack_bf16x2(y[0], 0.f) & 0xffffu);
    else ((float*)out)[i] = y[0];
  }
}


// ===========================================================================
// Chunked forward.  Per (batch, head), chunk of C = 32 positions.  The kernels work on KD = 64 or 128 key
// channels; a smaller Dk (a multiple of 8) is served by reading the missing channels as zeros (zero channels of q, k
// and g change nothing: they add nothing to any dot product or norm, and their state rows stay zero), and value
// columns are independent of each other, so any Dv (a multiple of 8) is served in groups of 32.
//
// With G_i the inclusive running sum of the log-decay g inside the chunk (per channel), S0 the state at the chunk
// start, and (per channel products written with (.)):
//   A_ij = beta_i sum_d k_id k_jd exp(G_id - G_jd)     (j <  i)
//   P_ij =        sum_d q_id k_jd exp(G_id - G_jd)     (j <= i)
//   T  = (I + A)^-1 diag(beta)
//   X  = V - (exp(G) (.) K) S0
//   O  = scale ((exp(G) (.) Q) S0 + (P T) X)
//   S' = diag(exp(G_last)) S0 + ((exp(G_last - G) (.) K)^T T) X
//
// kda_prep_kernel (all chunks in parallel) produces everything that depends on neither S0 nor V, one block of
// KdaBlob<KD>::kBytes per chunk, laid out as the other kernel wants it in LDS:
//   Kg  = -exp(G) (.) K             bf16 [32][KD]   contraction index (channel) permuted
//   Qg  = scale exp(G) (.) Q        bf16 [32][KD]   channel permuted
//   Mh + Ml = (exp(G_last - G) (.) K)^T T split into two bf16 terms, [KD][32], column (position) permuted
//   Ph + Pl = scale tril(P) T       the same, [32][32]
//   dec = exp(G_last)               fp32 [KD]
// kda_state_kernel (one workgroup per (batch, head, 32 value columns)) then walks the chunks in order with the fp32
// state in registers; every product in it is a v_mfma_f32_16x16x32_bf16 whose B operand is an accumulator (S0 or X)
// converted to bf16 in place: in the 16x16 accumulator layout lane l holds column l%16 and rows 4*(l/16)+r of each
// tile, so two stacked tiles give the lane 8 contraction indices 16*t + 4*(l/16) + r (t = 0,1; r = 0..3).  The A
// operands are stored with their contraction index permuted inside every aligned group of 32 (perm32) so that those 8
// indices are 8 consecutive elements, one 16-byte load.
//
// What bounds it.  The first kernel moves bytes, with the conversions in between: 1.29 GB (673 MB of inputs, 612 MB of blocks)
// in 217 us at B4 T8192 H16 (5.9 TB/s);
// with chunks of 64 and W = T K, U0 = T V in the workspace (107 KB per 64 positions, from a solve with 256 right-hand
// sides) it took 355 us.  The second kernel is a serial chain of chunks, bound by the latency of a link: folding T into
// the two matrices above takes a product and a conversion out of it, and chunks of 32 let three stages of everything the
// chain needs fit the LDS, so that no computing wavefront waits for global memory (those loads alone were 90 us of 284).
// It takes 230 us at that size, 0.9 us per chunk; 165 us of them remain without the copies into the LDS.
//
// Numerics: the 16x16 blocks of A and P run on MFMA with both operands referenced to the row before the block (every
// exponent <= 0 off the diagonal); a diagonal block whose total decay exceeds exp(-80) is referenced to its middle row
// instead (exponents up to the decay of 8 rows either way), when those go beyond exp(-80) to four rows in four passes, and
// when four rows do, it is accumulated in fp32 pair by pair with exp(G_i - G_j), j < i (no exponent is ever positive, so
// strong decays cannot overflow).
// T is computed in fp32; the products with T, the state update and the output's second term use two-term bf16 splits of
// both operands (three MFMAs each, relative error ~2^-17), which keeps the state error near fp32.
// ===========================================================================
constexpr int KC = 32;    // chunk length
constexpr int KDMAX = 128;
constexpr int KVS = 16;   // value columns per state wavefront

// One chunk's block in the workspace: byte offsets of its parts; rows of 16-byte pieces XOR-swizzled (below).
template <int KD> struct KdaBlob {
  static constexpr int kKg = 0, kQg = KC * KD * 2, kMh = 2 * KC * KD * 2, kMl = 3 * KC * KD * 2;
  static constexpr int kPh = 4 * KC * KD * 2, kPl = kPh + KC * KC * 2, kDec = kPl + KC * KC * 2;
  static constexpr int kBytes = (kDec + KD * 4 + 1023) & ~1023;     // whole 1 KiB copies
};
static_assert(KdaBlob<128>::kBytes == 37 * 1024 && KdaBlob<64>::kBytes == 21 * 1024, "");
// Swizzle of a row's 16-byte pieces: the 16 lanes that a 16-byte LDS read serves together must fall into 16 different slots
// of the 256-byte bank window.  Those are not 16 consecutive lanes but lanes 0-3, 12-15 and 20-27 (and so on): rows 0-3
// and 12-15 of one k-group with rows 4-11 of the next.  For rows of 64 bytes (row >> 2) & 3 itself puts two of them into every
// slot (256 of 930 LDS cycles per chunk); the permutation 0 2 3 1 of it puts one.  Rows of 256, 128 and 64 bytes:
template <int ROWBYTES> __host__ __device__ constexpr int piece_swizzle(int row) {
  return ROWBYTES == 256 ? (row & 15) : ROWBYTES == 128 ? ((row >> 1) & 7) : ((row >> 3) & 1) | (((row >> 2) ^ (row >> 3)) & 1) << 1;
}

struct KdaParams {
  const uint16_t* q; const uint16_t* k; const uint16_t* v;
  const void* g; int g_bf16; const float* beta;
  const float* s0; uint16_t* o; float* s_out;
  int B, T, H, NC; float scale; int l2norm; float l2eps;
  int Dk, Dv;     // the tensors' own widths: Dk <= KD key channels, Dv value columns
  char* blobs;    // [H][nc_total][KdaBlob<KD>::kBytes]
  // Sequences packed along the token axis of a batch of one (B == 1, T = all tokens): n_seq > 0, cu [n_seq + 1] = the
  // caller's running lengths; NC is the host's upper bound T / 32 + n_seq on the chunk slots.  Up to kScanSeqs sequences a
  // wavefront finds its way by itself (packed_span); beyond, kda_chunk_table_kernel writes bounds [n_seq + 1] = sanitised
  // running lengths, seq_chunk0 [n_seq + 1] = first chunk slot of every sequence, chunk_seq [NC] = sequence of every slot.
  int n_seq; const int32_t* cu; const int32_t* bounds; const int32_t* seq_chunk0; const int32_t* chunk_seq;
  int nc_total;   // chunk slots per head in the workspace: B * NC, or NC for a packed batch
};

// Where a sequence lives: token rows [tok0, tok_end) of the flattened [B * T] token axis and
// chunk slots [c0, c0 + nc) of the workspace.  A batch element is a sequence of its own.
struct SeqSpan { int tok0, tok_end, c0, nc; };

// Sequence `key` of a packed batch, or (by_slot) the one that owns chunk slot `key`: nc == 0 when there is none.  `rows_end`
// gets the end of the last sequence.  Bounds = the caller's, forced to start at 0, to stay within 0..T and not to decrease
// (whatever was passed, no kernel then leaves the tensors); chunk slots = running sum of ceil(len / 32).  A lane per
// sequence, two scans: about 0.5 us in every workgroup of both kernels instead of a launch of one workgroup in front of
// them (6 us).
constexpr int kScanSeqs = 64;
__device__ __forceinline__ SeqSpan packed_span(const KdaParams& p, int key, bool by_slot, int& rows_end) {
  SeqSpan s{0, 0, 0, 0};
  if (p.bounds != nullptr) {
    rows_end = p.bounds[p.n_seq];
    if (by_slot) {
      if (key >= p.seq_chunk0[p.n_seq]) return s;
      key = p.chunk_seq[key];
    }
    s.tok0 = p.bounds[key]; s.tok_end = p.bounds[key + 1];
    s.c0 = p.seq_chunk0[key]; s.nc = p.seq_chunk0[key + 1] - s.c0;
    return s;
  }
  const int lane = threadIdx.x & 63;
  int end = min(max(p.cu[min(lane + 1, p.n_seq)], p.cu[0]), p.T);
  end = max(end, 0);
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int left = __shfl_up(end, off);
    if (lane >= off) end = max(end, left);
  }
  int begin = __shfl_up(end, 1);
  begin = lane == 0 ? 0 : begin;
  const int nc = lane < p.n_seq ? (end - begin + KC - 1) / KC : 0;
  int upto = nc;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int left = __shfl_up(upto, off);
    if (lane >= off) upto += left;
  }
  rows_end = __builtin_amdgcn_readlane(end, 63);     // (lanes past the last sequence repeat its end)
  if (by_slot) {
    const uint64_t owner = __ballot(key >= upto - nc && key < upto);
    if (owner == 0) return s;
    key = __builtin_ctzll(owner);
  }
  s.tok0 = __builtin_amdgcn_readlane(begin, key); s.tok_end = __builtin_amdgcn_readlane(end, key);
  s.nc = __builtin_amdgcn_readlane(nc, key); s.c0 = __builtin_amdgcn_readlane(upto, key) - s.nc;
  return s;
}
__device__ __forceinline__ SeqSpan seq_span(const KdaParams& p, int seq, int& rows_end) {
  if (p.n_seq > 0) return packed_span(p, seq, false, rows_end);
  rows_end = p.B * p.T;
  return SeqSpan{seq * p.T, (seq + 1) * p.T, seq * p.NC, p.NC};
}

// Chunk slots of more than kScanSeqs packed sequences, built on the device so that the host never reads the bounds.
// bounds = cu_seqlens forced to start at 0, to stay within 0..T and not to decrease (whatever the
// caller passed, no kernel then leaves the tensors); seq_chunk0 = running sum of ceil(len / 32);
// chunk_seq = the sequence of every slot.  One workgroup; thread i takes a run of sequences.
__global__ __launch_bounds__(256) void kda_chunk_table_kernel(const int32_t* cu, int n_seq, int T, int nc_max,
                                                              int32_t* bounds, int32_t* seq_chunk0, int32_t* chunk_seq) {
  __shared__ int part[256];
  const int tid = threadIdx.x;
  const int per = (n_seq + 1 + 255) / 256;
  const int a = min(tid * per, n_seq + 1), b = min(a + per, n_seq + 1);
  int hi = 0;
  for (int i = a; i < b; ++i) hi = max(hi, min(max(cu[i], 0), T));
  part[tid] = hi;
  __syncthreads();
  hi = 0;
  for (int w = 0; w < tid; ++w) hi = max(hi, part[w]);
  for (int i = a; i < b; ++i) {
    hi = max(hi, min(max(cu[i], 0), T));
    bounds[i] = (i == 0) ? 0 : hi;
  }
  __threadfence_block();
  __syncthreads();
  const int per_s = (n_seq + 255) / 256;
  const int sa = min(tid * per_s, n_seq), sb = min(sa + per_s, n_seq);
  int mine = 0;
  for (int i = sa; i < sb; ++i) mine += (bounds[i + 1] - bounds[i] + KC - 1) / KC;
  __syncthreads();
  part[tid] = mine;
  __syncthreads();
  int run = 0;
  for (int w = 0; w < tid; ++w) run += part[w];
  for (int i = sa; i < sb; ++i) {
    const int nc = (bounds[i + 1] - bounds[i] + KC - 1) / KC;
    seq_chunk0[i] = min(run, nc_max);
    for (int c = 0; c < nc; ++c)
      if (run + c < nc_max) chunk_seq[run + c] = i;
    run += nc;
  }
  if (tid == 255) seq_chunk0[n_seq] = min(run, nc_max);   // the last thread's run ends at the total
}

// Stored position of contraction index x inside its aligned group of 32: bits (4,3,2) -> (3,2,4).
__host__ __device__ constexpr int perm32(int x) { return (x & ~0x1c) | ((x & 0x0c) << 1) | ((x & 0x10) >> 2); }
__host__ __device__ constexpr int perm32_inv(int p) { return (p & ~0x1c) | ((p & 0x18) >> 1) | ((p & 0x04) << 2); }

__device__ __forceinline__ f32x4 lds_f4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// A float as two bf16 terms (value = hi + lo up to 2^-17 relative).
__device__ __forceinline__ void split_bf16(float x, float& hi, float& lo) { hi = round_bf16(x); lo = x - hi; }
// Eight floats as two 16-byte pieces of bf16 terms.
__device__ __forceinline__ void split_pack8(const float* x, u32x4& hi, u32x4& lo) {
  float h[8], l[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) split_bf16(x[e], h[e], l[e]);
  hi = pack8(h);
  lo = pack8(l);
}
// LDS writes of a wavefront before this point are seen by all of its lanes after it.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ uint32_t dpp_xor2(uint32_t x) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xf, 0xf, false); }

// A workgroup makes two neighbouring chunk slots (64 rows; they may belong to different sequences).
template <int KD>
__global__ __launch_bounds__(256, KD == 128 ? 2 : 3) void kda_prep_kernel(KdaParams p) {
  using Blob = KdaBlob<KD>;
  constexpr int CPR = KD / 8, RPP = 256 / CPR, NP = 64 / RPP;         // 16-byte pieces per row, rows per pass, passes
  constexpr int NM = KD / 32;                                         // contraction groups of 32 channels
  __shared__ __attribute__((aligned(16))) float G[64][KD + 4];        // inclusive running log-decay (rows 4 banks apart: 16 rows read side by side do not collide)
  __shared__ __attribute__((aligned(16))) uint16_t Kr[64][KD + 8];    // k as given (bf16)
  __shared__ __attribute__((aligned(16))) uint16_t Qr[64][KD + 8];    // q as given
  __shared__ __attribute__((aligned(16))) float Ad[4][16][16];        // diagonal blocks of A, [block][column j][row i]
  __shared__ __attribute__((aligned(16))) float Ao[2][16][20];        // the block A_10 of either chunk, [row][column]
  __shared__ __attribute__((aligned(16))) float Td[4][16][20];        // (I + A_II)^-1, [block][row][column]
  __shared__ __attribute__((aligned(16))) float rk[64], rq[64], bt[64];   // 1/|k|, 1/|q|, beta (0 for padded rows)
  __shared__ int steep[4];      // per 16-row block: decay beyond exp(-80) over all of it (1), over 8 of its rows (2), over 4 (3)

  const int h = blockIdx.y;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  // First token row and live rows of the two chunks.  A slot without a chunk has no live rows and is not stored; its
  // loads go to the first chunk's first row.
  int t0[2], n_live[2];
  int64_t ci[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int slot = 2 * blockIdx.x + c;
    t0[c] = 0;
    n_live[c] = 0;
    int gc = slot;
    if (p.n_seq > 0) {
      int rows_end;
      const SeqSpan sp = packed_span(p, slot, true, rows_end);
      if (sp.nc > 0) {
        t0[c] = sp.tok0 + (slot - sp.c0) * KC;
        n_live[c] = min(sp.tok_end - t0[c], KC);
      }
    } else {
      gc = blockIdx.z * p.NC + slot;
      if (slot < p.NC) {
        t0[c] = blockIdx.z * p.T + slot * KC;
        n_live[c] = min((int)(blockIdx.z + 1) * p.T - t0[c], KC);
      }
    }
    if (c == 0 && n_live[0] <= 0) return;      // surplus slots (the grid covers the upper bound)
    if (n_live[c] <= 0) { t0[c] = t0[0]; n_live[c] = 0; }
    ci[c] = (int64_t)h * p.nc_total + gc;
  }
  // Addresses: a wavefront-uniform 64-bit base per array and chunk plus a 32-bit offset per lane.
  const uint32_t row_stride = (uint32_t)p.H * (uint32_t)p.Dk;     // elements between token rows of one head (q, k, g)
  const int64_t tok_base[2] = {((int64_t)t0[0] * p.H + h) * p.Dk, ((int64_t)t0[1] * p.H + h) * p.Dk};
  char* const blob[2] = {p.blobs + ci[0] * Blob::kBytes, p.blobs + ci[1] * Blob::kBytes};

  // ---- phase 0a: G = cumsum(g) -----------------------------------------------
  // Every global load of the chunks (g here, then q, k and beta of phase 0b) goes out before the first result is used,
  // so that the memory latency is paid once.  Inputs are read once and the workspace is written once: both as streaming
  // (non-temporal) accesses.
  if (tid < 4) steep[tid] = 0;
  __syncthreads();
  const int cc = tid % CPR, r4 = tid / CPR;
  u32x4 qraw[NP], kraw[NP];
  float btv[NP];
  constexpr int GR = 64 * KD / 256;               // rows of one channel per thread: a whole chunk (128) or half of one (64)
  {
    const int d = tid % KD, part = __builtin_amdgcn_readfirstlane(tid / KD);   // the row of a g load is wavefront-uniform
    const int c = part * GR / KC, row0 = part * GR % KC;
    const bool d_live = d < p.Dk;                 // channels beyond Dk read as zero (their loads re-read the last channel)
    const int dl = min(d, p.Dk - 1);
    // Rows past the end re-read the last row (always valid) and are zeroed afterwards, so that the loads carry no
    // branches and all go out together; the dtype is decided once, outside the loops, for the same reason.  bf16 g: the
    // two channels of a pair read the same dword (no sub-dword loads) and take their half.
    const int last = max((c ? n_live[1] : n_live[0]) - 1, 0), live = c ? n_live[1] : n_live[0];
    const int64_t base = c ? tok_base[1] : tok_base[0];
    uint32_t graw[GR];
    if (p.g_bf16) {
#pragma unroll
      for (int i = 0; i < GR; ++i) {
        const uint32_t* row = reinterpret_cast<const uint32_t*>(p.g) + ((base + (uint32_t)min(row0 + i, last) * row_stride) >> 1);
        graw[i] = __builtin_nontemporal_load(row + (uint32_t)(dl >> 1));
      }
    } else {
#pragma unroll
      for (int i = 0; i < GR; ++i) {
        const uint32_t* row = reinterpret_cast<const uint32_t*>(p.g) + (base + (uint32_t)min(row0 + i, last) * row_stride);
        graw[i] = __builtin_nontemporal_load(row + (uint32_t)dl);
      }
    }
    const int ccl = min(cc, p.Dk / 8 - 1);
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int r = r4 + RPP * i, rc = r >> 5;    // (a pass of 16 or 32 rows lies inside one chunk)
      const uint32_t row = (uint32_t)min(r & 31, max((rc ? n_live[1] : n_live[0]) - 1, 0));
      const int64_t at = (rc ? tok_base[1] : tok_base[0]) + row * row_stride + 8u * ccl;
      kraw[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.k + at));
      qraw[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.q + at));
      btv[i] = p.beta[(int64_t)((rc ? t0[1] : t0[0]) + row) * p.H + h];
    }
    __builtin_amdgcn_sched_barrier(0);
    float gv[GR];
    const bool g16 = p.g_bf16 != 0, odd = (d & 1) != 0;
#pragma unroll
    for (int i = 0; i < GR; ++i) {
      const float x = g16 ? (odd ? bf16hi_to_f32(graw[i]) : bf16lo_to_f32(graw[i])) : __uint_as_float(graw[i]);
      gv[i] = (row0 + i < live && d_live) ? x : 0.f;
    }
    // G holds the running sum in units of log 2 (g * log2(e)): every exponential below is a bare v_exp_f32.
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < GR; ++i) {
      acc += gv[i] * kLog2e;
      G[part * GR + i][d] = acc;
    }
#pragma unroll
    for (int blk = 0; blk < GR / 16; ++blk) {
      float t4[4];
#pragma unroll
      for (int f = 0; f < 4; ++f) t4[f] = gv[16 * blk + 4 * f] + gv[16 * blk + 4 * f + 1] + gv[16 * blk + 4 * f + 2] + gv[16 * blk + 4 * f + 3];
      const float lo = t4[0] + t4[1], hi = t4[2] + t4[3];
      if (__any(lo + hi < -80.f)) {
        const bool four = __any(fminf(fminf(t4[0], t4[1]), fminf(t4[2], t4[3])) < -80.f), eight = __any(fminf(lo, hi) < -80.f);
        if ((tid & 63) == 0) atomicMax(&steep[part * GR / 16 + blk], four ? 3 : eight ? 2 : 1);
      }
    }
    if constexpr (GR < KC) {                      // the second half of a chunk continues from the first
      __syncthreads();
      if (row0 != 0) {
        const float add = G[part * GR - 1][d];
#pragma unroll
        for (int i = 0; i < GR; ++i) G[part * GR + i][d] += add;
      }
    }
  }

  // ---- phase 0b: raw q, k to LDS, row norms, beta ---------------------------
  float rkv[NP], rqv[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int r = r4 + RPP * i;
    const bool live = (r & 31) < ((r >> 5) ? n_live[1] : n_live[0]);
    const u32x4 zero4 = {0, 0, 0, 0};
    if (!live || 8 * cc >= p.Dk) { kraw[i] = zero4; qraw[i] = zero4; }
    float kf[8], qf[8];
    unpack8(kraw[i], kf);
    unpack8(qraw[i], qf);
    float sk = 0.f, sq = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) { sk = fmaf(kf[e], kf[e], sk); sq = fmaf(qf[e], qf[e], sq); }
    sk = group_sum<CPR>(sk);
    sq = group_sum<CPR>(sq);
    rkv[i] = p.l2norm ? rsqrtf(sk + p.l2eps) : 1.f;
    rqv[i] = p.l2norm ? rsqrtf(sq + p.l2eps) : 1.f;
    if (cc == 0) {
      rk[r] = rkv[i];
      rq[r] = rqv[i];
      bt[r] = live ? btv[i] : 0.f;
    }
    *reinterpret_cast<u32x4*>(&Kr[r][8 * cc]) = kraw[i];
    *reinterpret_cast<u32x4*>(&Qr[r][8 * cc]) = qraw[i];
  }
  __syncthreads();

  // ---- phase 1: Kg = -exp(G) k/|k|, Qg = scale exp(G) q/|q| (channel permuted), dec = exp(G_last) ----
  {
    // The stored 16-byte piece a of a group of 32 channels holds channels 4a..+3 and 16 + 4a..+3: lanes cc and cc ^ 2 each
    // own half of two pieces and swap one half.
    const int b2 = cc & 3;
    const bool low = b2 < 2;
    const int piece = (cc & ~3) + 2 * (b2 & 1) + (low ? 0 : 1);
    auto join = [&](const u32x4& pk) -> u32x4 {
      const uint32_t s0 = low ? pk.z : pk.x, s1 = low ? pk.w : pk.y;
      const uint32_t x0 = dpp_xor2(s0), x1 = dpp_xor2(s1);
      return low ? u32x4{pk.x, pk.y, x0, x1} : u32x4{x0, x1, pk.z, pk.w};
    };
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int r = r4 + RPP * i, rc = r >> 5, row = r & 31;
      float qf[8], kf[8], o8[8], k8[8];
      unpack8(qraw[i], qf);
      unpack8(kraw[i], kf);
      const f32x4 g0 = lds_f4(&G[r][8 * cc]), g1 = lds_f4(&G[r][8 * cc + 4]);
      const float sq = p.scale * rqv[i], sk = -rkv[i];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = __builtin_amdgcn_exp2f(e < 4 ? g0[e & 3] : g1[e & 3]);
        o8[e] = sq * f * qf[e];
        k8[e] = sk * f * kf[e];
      }
      const uint32_t at = (uint32_t)(row * 2 * KD + 16 * (piece ^ piece_swizzle<2 * KD>(row)));
      const u32x4 kp = join(pack8(k8)), qp = join(pack8(o8));
      if (rc == 0 || n_live[1] > 0) {
        char* dst = (rc ? blob[1] : blob[0]) + at;
        __builtin_nontemporal_store(kp, reinterpret_cast<u32x4*>(dst + Blob::kKg));
        __builtin_nontemporal_store(qp, reinterpret_cast<u32x4*>(dst + Blob::kQg));
      }
    }
    if (tid < 2 * KD / 4) {
      const int c = tid / (KD / 4), d4 = 4 * (tid % (KD / 4));
      const f32x4 gl = lds_f4(&G[KC * c + KC - 1][d4]);
      f32x4 dv;
#pragma unroll
      for (int e = 0; e < 4; ++e) dv[e] = __builtin_amdgcn_exp2f(gl[e]);
      if (c == 0 || n_live[1] > 0) *reinterpret_cast<f32x4*>((c ? blob[1] : blob[0]) + Blob::kDec + 4 * d4) = dv;
    }
  }

  // ---- phase 2: 16x16 blocks of A and P on MFMA --------------------------------
  // Block rows bi = 0..3 of the 64 rows (chunk bi / 2, I = bi % 2).  Block (I, J), J <= I: both operands are referenced to
  // the row before block I (the chunk's start for I = 0: G_ref = 0), so the row factor exp(G_i - G_ref) is <= 1 and, for J < I,
  // so is the column factor exp(G_ref - G_j).  For a diagonal block (J == I) the column factor grows to exp(total decay
  // of the block); beyond exp(80) the block's middle row is the reference, each factor then growing to the decay of 8 rows
  // (four passes took 60 us more per 32768 rows of 16 heads with the decays of a freshly initialised layer).
  // Wavefront w takes block row w: its diagonal block and, in the second block row of a chunk, block (1, 0).
  const int li = lane & 15, q4 = lane >> 4;
  const int chunk = wave >> 1, I = wave & 1;
  const int ri = 16 * wave + li;
  char* const my_blob = chunk ? blob[1] : blob[0];
  const bool stored = chunk == 0 || n_live[1] > 0;
  bf16x8 va[NM], vq[NM];
  // Row operands k_i f_i, q_i f_i with f_i = exp(G_i - G_ref(i)); `ref` is the lane's reference row (-1: G_ref = 0).
  auto row_operands = [&](int ref) {
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int d0 = 32 * m + 8 * q4;
      float ki[8], qi[8], ak[8], aq[8];
      unpack8(*reinterpret_cast<const u32x4*>(&Kr[ri][d0]), ki);
      unpack8(*reinterpret_cast<const u32x4*>(&Qr[ri][d0]), qi);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        const f32x4 gi = lds_f4(&G[ri][d0 + 4 * hf]);
        const f32x4 gr = (ref >= 0) ? lds_f4(&G[max(ref, 0)][d0 + 4 * hf]) : zero;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float fi = __builtin_amdgcn_exp2f(gi[e] - gr[e]);
          ak[4 * hf + e] = ki[4 * hf + e] * fi;
          aq[4 * hf + e] = qi[4 * hf + e] * fi;
        }
      }
      va[m] = __builtin_bit_cast(bf16x8, pack8(ak));
      vq[m] = __builtin_bit_cast(bf16x8, pack8(aq));
    }
  };
  // This wavefront's rows of scale tril(P), as a product's operand wants them: row 16 I + li, columns 4 q4 + r of either
  // column block.
  f32x4 P[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  auto mfma_block = [&](int J, int ref) {
    const int rj = 32 * chunk + 16 * J + li;
    f32x4 accA = {0.f, 0.f, 0.f, 0.f}, accP = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int d0 = 32 * m + 8 * q4;
      float kj[8], bk[8];
      unpack8(*reinterpret_cast<const u32x4*>(&Kr[rj][d0]), kj);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        const f32x4 gj = lds_f4(&G[rj][d0 + 4 * hf]);
        const f32x4 gr = (ref >= 0) ? lds_f4(&G[max(ref, 0)][d0 + 4 * hf]) : zero;
#pragma unroll
        for (int e = 0; e < 4; ++e) bk[4 * hf + e] = kj[4 * hf + e] * __builtin_amdgcn_exp2f(gr[e] - gj[e]);
      }
      const bf16x8 vb = __builtin_bit_cast(bf16x8, pack8(bk));
      accA = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[m], vb, accA, 0, 0, 0);
      // P comes out transposed (operands swapped: both operand layouts hold 8 contraction indices of
      // one row / column per lane): a lane then owns four consecutive columns of one row of P.
      accP = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, vq[m], accP, 0, 0, 0);
    }
    // accA: lane holds column j = 16J + li, rows i = 16I + 4*q4 + r
    const float rkj = rk[rj];
    f32x4 av;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * wave + 4 * q4 + r;
      av[r] = bt[i] * rk[i] * rkj * accA[r];
    }
    {
      // accP: lane holds row i = 16I + li, columns j = 16J + 4*q4 + r
      const int ip = 16 * I + li, jp = 16 * J + 4 * q4;
      const f32x4 rk4 = lds_f4(&rk[32 * chunk + jp]);
      const float qs = p.scale * rq[ri];
      f32x4 pv;
#pragma unroll
      for (int r = 0; r < 4; ++r) pv[r] = (jp + r <= ip) ? qs * rk4[r] * accP[r] : 0.f;
      if (J == 0) P[0] = pv; else P[1] = pv;
    }
    if (I == J) {
      *reinterpret_cast<f32x4*>(&Ad[wave][li][4 * q4]) = av;   // entries with i <= j are never read
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) Ao[chunk][4 * q4 + r][li] = av[r];
    }
  };
  // A diagonal block whose decay is too steep for the MFMA path even with a reference row per four rows is accumulated
  // in fp32 pair by pair with exp(G_i - G_j), j < i, where no exponent is ever positive.
  auto steep_diagonal = [&]() {
    const int il = lane >> 2, dq = lane & 3;
    const int rr = 16 * wave + il;
    float a[16], pp[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) { a[j] = 0.f; pp[j] = 0.f; }
#pragma unroll 1
    for (int dc = 0; dc < KD / 32; ++dc) {
      const int d0 = (KD / 4) * dq + 8 * dc;
      float ki[8], qi[8];
      unpack8(*reinterpret_cast<const u32x4*>(&Kr[rr][d0]), ki);
      unpack8(*reinterpret_cast<const u32x4*>(&Qr[rr][d0]), qi);
      const f32x4 gi0 = lds_f4(&G[rr][d0]), gi1 = lds_f4(&G[rr][d0 + 4]);
#pragma unroll
      for (int j = 15; j >= 0; --j) {
        const int rj = 16 * wave + j;
        float kj[8];
        unpack8(*reinterpret_cast<const u32x4*>(&Kr[rj][d0]), kj);
        // exp(G_i - G_j) for j < i: the exponent is a sum of log-decays, never positive; rows at or
        // above the diagonal take the factor 1 (only j == i is used, by P).
        const f32x4 gj0 = lds_f4(&G[rj][d0]), gj1 = lds_f4(&G[rj][d0 + 4]);
        const bool below = j < il;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float diff = (e < 4) ? gi0[e & 3] - gj0[e & 3] : gi1[e & 3] - gj1[e & 3];
          const float t = kj[e] * (below ? __builtin_amdgcn_exp2f(diff) : 1.f);
          a[j] = fmaf(ki[e], t, a[j]);
          pp[j] = fmaf(qi[e], t, pp[j]);
        }
      }
    }
    const float bi = bt[rr] * rk[rr], qs = p.scale * rq[rr];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      float av = dpp_add<0x4E>(dpp_add<0xB1>(a[j]));         // sum over the 4 channel quarters
      float pv = dpp_add<0x4E>(dpp_add<0xB1>(pp[j]));
      const float rkj = rk[16 * wave + j];
      if ((j & 3) == dq && j < il) Ad[wave][j][il] = bi * rkj * av;
      if ((j & 3) == dq) Td[wave][il][j] = (j <= il) ? qs * rkj * pv : 0.f;   // (on the way to the operand layout)
    }
    wave_lds_fence();
    if (I == 0) P[0] = lds_f4(&Td[wave][li][4 * q4]); else P[1] = lds_f4(&Td[wave][li][4 * q4]);
    wave_lds_fence();
  };
  // A steep diagonal block on the matrix cores after all: with one reference row per group of four
  // rows (the row before the group) every row factor exp(G_i - G_ref(i)) is <= 1, and the column
  // factors exp(G_ref - G_j) are <= 1 for columns of earlier groups and at most the decay of four
  // rows inside the group.  Pass r multiplies all rows by the columns scaled for the reference of
  // group r; the accumulator layout gives rows 4r..4r+3 (A) resp. the lanes of those rows (P, transposed) that pass's result.
  auto steep_diagonal_mfma = [&]() {
    row_operands((I == 0 && li < 4) ? -1 : 16 * wave + (li & ~3) - 1);
    f32x4 accA = {0.f, 0.f, 0.f, 0.f}, accP = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int r = 0; r < 4; ++r) {
      const int ref = (I == 0 && r == 0) ? -1 : 16 * wave + 4 * r - 1;
      const bool live = (li >> 2) <= r;     // later columns are above the diagonal for every row of the group
      f32x4 pa = {0.f, 0.f, 0.f, 0.f}, pp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const int d0 = 32 * m + 8 * q4;
        float kj[8], bk[8];
        unpack8(*reinterpret_cast<const u32x4*>(&Kr[ri][d0]), kj);
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          const f32x4 gj = lds_f4(&G[ri][d0 + 4 * hf]);
          const f32x4 gr = (ref >= 0) ? lds_f4(&G[max(ref, 0)][d0 + 4 * hf]) : zero;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            bk[4 * hf + e] = live ? kj[4 * hf + e] * __builtin_amdgcn_exp2f(fminf(gr[e] - gj[e], 120.f)) : 0.f;
        }
        const bf16x8 vb = __builtin_bit_cast(bf16x8, pack8(bk));
        pa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(va[m], vb, pa, 0, 0, 0);
        pp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vb, vq[m], pp, 0, 0, 0);
      }
      if (q4 == r) accA = pa;               // rows 4 q4 .. of A
      if ((li >> 2) == r) accP = pp;        // row li of P
    }
    const float rkj = rk[ri];
    f32x4 av;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = 16 * wave + 4 * q4 + r;
      av[r] = bt[i] * rk[i] * rkj * accA[r];
    }
    *reinterpret_cast<f32x4*>(&Ad[wave][li][4 * q4]) = av;   // entries with i <= j are never read
    const f32x4 rk4 = lds_f4(&rk[16 * wave + 4 * q4]);
    const float qs = p.scale * rq[ri];
    f32x4 pv;
#pragma unroll
    for (int r = 0; r < 4; ++r) pv[r] = (4 * q4 + r <= li) ? qs * rk4[r] * accP[r] : 0.f;
    if (I == 0) P[0] = pv; else P[1] = pv;
  };
  {
    const int sp = __builtin_amdgcn_readfirstlane(steep[wave]), before = I ? 16 * wave - 1 : -1, middle = 16 * wave + 7;
    if (I == 1 || sp == 0) row_operands(before);
    if (I == 1) mfma_block(0, before);
    if (sp == 3) steep_diagonal();
    else if (sp == 2) steep_diagonal_mfma();
    else {
      // With the middle row as reference the entries above the diagonal may overflow; nothing reads them.
      if (sp == 1) row_operands(middle);
      mfma_block(I, sp == 1 ? middle : before);
    }
  }

  // ---- phase 3: T = (I + A)^-1 diag(beta).  The inverse of diagonal block `wave` in fp32, one column per lane (lanes
  // 16.. repeat the work of lane & 15).
  wave_lds_fence();
  {
    float tc[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) tc[i] = (i == li) ? 1.f : 0.f;
#pragma unroll
    for (int j = 0; j < 15; ++j) {
      f32x4 ar[4];
#pragma unroll
      for (int i4 = (j + 1) / 4; i4 < 4; ++i4) ar[i4] = lds_f4(&Ad[wave][j][4 * i4]);
      const float xj = tc[j];
#pragma unroll
      for (int i = j + 1; i < 16; ++i) tc[i] = fmaf(-ar[i >> 2][i & 3], xj, tc[i]);
    }
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < 16; ++i) Td[wave][i][li] = tc[i];
    }
  }
  __syncthreads();   // both inverses and A_10 of either chunk are in place
  // T_10 = -T_11 (A_10 T_00) in two fp32 matrix products, both wavefronts of a chunk all of it.  As right operand (lane
  // (column li, rows 4 q4 + e)) and as result the layout is the same, and it is also the one T^T is wanted in below.  (As
  // multiply-adds from LDS this took 3400 of the workgroup's 27000 cycles.)
  f32x4 t00, t10, t11;
  {
    const f32x4 a10 = lds_f4(&Ao[chunk][li][4 * q4]), r11 = lds_f4(&Td[2 * chunk + 1][li][4 * q4]);
    f32x4 m1 = {0.f, 0.f, 0.f, 0.f};
    t10 = m1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      t00[e] = Td[2 * chunk][4 * q4 + e][li];
      t11[e] = Td[2 * chunk + 1][4 * q4 + e][li];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) m1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a10[e], t00[e], m1, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e) t10 = __builtin_amdgcn_mfma_f32_16x16x4f32(-r11[e], m1[e], t10, 0, 0, 0);
  }
  // T^T as left operand: row (column of T) 16 J + li, contraction slots (q4, e): positions 4 q4 + e for e < 4,
  // 16 + 4 q4 + (e - 4) for e >= 4; two bf16 terms.
  bf16x8 th[2], tl[2];
  {
    const float b0 = bt[32 * chunk + li], b1 = bt[32 * chunk + 16 + li];
    float v0[8], v1[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v0[e] = b0 * t00[e];
      v0[4 + e] = b0 * t10[e];
      v1[e] = 0.f;
      v1[4 + e] = b1 * t11[e];
    }
    u32x4 hi, lo;
    split_pack8(v0, hi, lo);
    th[0] = __builtin_bit_cast(bf16x8, hi);
    tl[0] = __builtin_bit_cast(bf16x8, lo);
    split_pack8(v1, hi, lo);
    th[1] = __builtin_bit_cast(bf16x8, hi);
    tl[1] = __builtin_bit_cast(bf16x8, lo);
  }
  // Row `row` of (right operand)^T T: the products come out with four consecutive columns of T per lane and column block,
  // which is the stored piece q4 of that row; both terms of it leave from here, 16 whole rows per instruction.
  auto times_t = [&](const float* r8, char* dst_hi, char* dst_lo, int row) {
    u32x4 hi, lo;
    split_pack8(r8, hi, lo);
    const bf16x8 rh = __builtin_bit_cast(bf16x8, hi), rl = __builtin_bit_cast(bf16x8, lo);
    float out[8];
#pragma unroll
    for (int J = 0; J < 2; ++J) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tl[J], rh, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(th[J], rl, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(th[J], rh, acc, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) out[4 * J + r] = acc[r];
    }
    split_pack8(out, hi, lo);
    const int at = row * 64 + 16 * (q4 ^ piece_swizzle<64>(row));
    if (stored) {
      __builtin_nontemporal_store(hi, reinterpret_cast<u32x4*>(dst_hi + at));
      __builtin_nontemporal_store(lo, reinterpret_cast<u32x4*>(dst_lo + at));
    }
  };
  {
    float pv[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) { pv[e] = P[0][e]; pv[4 + e] = P[1][e]; }
    times_t(pv, my_blob + Blob::kPh, my_blob + Blob::kPl, 16 * I + li);
  }
  // ---- phase 4: M = (exp(G_last - G) k/|k|)^T T, half of the chunk's channels per wavefront
  {
    const f32x4 r0 = lds_f4(&rk[32 * chunk + 4 * q4]), r1 = lds_f4(&rk[32 * chunk + 16 + 4 * q4]);
#pragma unroll
    for (int i = 0; i < KD / 32; ++i) {
      const int d = 16 * (KD / 32 * I + i) + li;
      const float glast = G[32 * chunk + 31][d];
      float kv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int r = 32 * chunk + (e < 4 ? 4 * q4 + e : 12 + 4 * q4 + e);
        kv[e] = __builtin_amdgcn_exp2f(glast - G[r][d]) * bf16lo_to_f32(Kr[r][d]) * (e < 4 ? r0[e & 3] : r1[e & 3]);
      }
      times_t(kv, my_blob + Blob::kMh, my_blob + Blob::kMl, d);
    }
  }
}

__device__ __forceinline__ bf16x8 pack_acc2(const f32x4& t0, const f32x4& t1) {
  u32x4 r;
  r.x = pack_bf16x2(t0[0], t0[1]); r.y = pack_bf16x2(t0[2], t0[3]);
  r.z = pack_bf16x2(t1[0], t1[1]); r.w = pack_bf16x2(t1[2], t1[3]);
  return __builtin_bit_cast(bf16x8, r);
}
// ... and what the rounding left over, as a second operand.
__device__ __forceinline__ bf16x8 pack_rest2(const f32x4& t0, const f32x4& t1, bf16x8 high) {
  const u32x4 hb = __builtin_bit_cast(u32x4, high);
  f32x4 l0, l1;
  l0[0] = t0[0] - bf16lo_to_f32(hb.x); l0[1] = t0[1] - bf16hi_to_f32(hb.x);
  l0[2] = t0[2] - bf16lo_to_f32(hb.y); l0[3] = t0[3] - bf16hi_to_f32(hb.y);
  l1[0] = t1[0] - bf16lo_to_f32(hb.z); l1[1] = t1[1] - bf16hi_to_f32(hb.z);
  l1[2] = t1[2] - bf16lo_to_f32(hb.w); l1[3] = t1[3] - bf16hi_to_f32(hb.w);
  return pack_acc2(l0, l1);
}

typedef __attribute__((address_space(3))) const char* lds_cptr;
__device__ __forceinline__ bf16x8 lds_bf16x8(lds_cptr p) {
  return __builtin_bit_cast(bf16x8, *(const u32x4 __attribute__((address_space(3)))*)p);
}
__device__ __forceinline__ f32x4 lds_f32x4(lds_cptr p) { return *(const f32x4 __attribute__((address_space(3)))*)p; }
// LDS transpose read: inside a block of 16 lanes that address, lane i, row i / 4 and columns 4 (i % 4) .. + 3 of a bf16
// tile, lane i receives column i of the four rows.
typedef short s16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x2 lds_column4(lds_cptr p) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)p));
}

constexpr int KCT = 2;                        // tiles of 16 value columns per workgroup
constexpr int KPW = 4;                        // data-moving wavefronts per workgroup
constexpr int KSTAGES = 3;                    // LDS stages of chunk data
constexpr int kStateThreads = 64 * (2 * KCT + KPW);

// The chunk-to-chunk chain sets the time of this kernel once its data are there, and next to it what the CU's LDS can
// deliver (about 110 KB of operands and copies per chunk).  So:
//  * one wavefront owns one tile of 16 value columns with all of its state rows: the state never leaves its registers
//    (as right operand it is the accumulators converted in place), nothing of the chain waits for another wavefront,
//    and every operand of the chain is read once per column tile.  Two wavefronts per tile with half of the state each,
//    both computing X and handing state halves over through LDS, took 250 us instead of 230 (B4 T8192 H16, 128 x 128);
//  * the outputs are not part of the chain: a second wavefront per tile makes Qg S0 of the chunk from the bf16 state
//    the first one left in LDS, adds (P T) X when X has arrived, and stores the rows one chunk later;
//  * neither waits for global memory: four further wavefronts issue the asynchronous copies of the chunk two ahead (the
//    chunk's block is one linear copy of 37 or 21 KiB, V 32 rows of 64 bytes).
template <int KD>
__global__ __launch_bounds__(kStateThreads, 1) void kda_state_kernel(KdaParams p) {
  using Blob = KdaBlob<KD>;
  constexpr int NM = KD / 32, NS = KD / 16;                    // channel groups of 32, state tiles of 16 rows
  constexpr int kV = Blob::kBytes, kStage = Blob::kBytes + KC * KVS * KCT * 2;
  constexpr int NCP = Blob::kBytes / 1024;
  __shared__ __attribute__((aligned(1024))) char stage[KSTAGES][kStage];
  __shared__ __attribute__((aligned(16))) u32x4 xs[2][KCT][NM][64];           // [chunk parity][column tile][channel group][lane]: S0 as right operand
  __shared__ __attribute__((aligned(16))) u32x4 xx[2][KCT][2][64];            // X as right operand, two terms
  __shared__ __attribute__((aligned(16))) uint16_t ost[KCT][KC][KVS];         // output rows on their way out

  // Keep the column groups of one (batch, head) on one XCD: they read the same chunk data.
  int vid = blockIdx.x;
  if ((gridDim.x & 7) == 0) vid = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int NGRP = (p.Dv + KVS * KCT - 1) / (KVS * KCT);       // groups of 32 value columns
  const int grp = vid % NGRP, bh = vid / NGRP;
  const int h = bh % p.H, b = bh / p.H;     // b: batch element, or sequence of a packed batch
  int rows_end;
  const SeqSpan sp = seq_span(p, b, rows_end);
  const int nc = sp.nc;                      // chunks of this sequence (0 for an empty one)
  const int64_t ci0 = (int64_t)h * p.nc_total + sp.c0;
  const int lane = threadIdx.x & 63, ln = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  if (wave >= 2 * KCT) {
    // ================= data-moving wavefront =================
    const int pw = wave - 2 * KCT;
    const uint32_t stage_lds = lds_address(&stage[0][0]);
    // V: a copy moves 16 rows of 64 bytes; lane i lands at row i / 4, piece i % 4.  Pieces past the last column re-read
    // the last one (columns are independent and dead ones are not stored).
    const int v_row = lane >> 2, v_piece = min(KVS * KCT * grp / 8 + (lane & 3), p.Dv / 8 - 1);
    const char* const my_blobs = p.blobs + ci0 * Blob::kBytes;
    auto issue_copies = [&](int n, int st) {
      const uint16_t* src = reinterpret_cast<const uint16_t*>(my_blobs + (int64_t)n * Blob::kBytes);
      const uint32_t dst = stage_lds + st * kStage;
#pragma unroll
      for (int j = pw; j < NCP; j += KPW) copy16_to_lds_async(src + 512 * j, 16 * lane, dst + 1024 * j);
      if (pw >= 2) {
        const int tok = sp.tok0 + n * KC;
        const int row = min(16 * (pw - 2) + v_row, sp.tok_end - 1 - tok);
        copy16_to_lds_async(p.v + ((int64_t)tok * p.H + h) * p.Dv, 2 * (row * p.H * p.Dv + 8 * v_piece), dst + kV + 1024 * (pw - 2));
      }
    };
    // The workgroups of a (batch, head) copy the same blocks at about the same time; each asks for its share of the block
    // two chunks beyond the copies (one dword per 128-byte line, by wavefronts 0 and 1) so that the copies find it in
    // the L2.  The target register is tied up for the whole loop.
    constexpr int kAhead = 4;                 // (6 and 8 gave the same time)
    uint32_t touched = 0;
    const int t_line = (64 * pw + lane) * NGRP + grp;
    const int t_off = 128 * min(t_line, Blob::kBytes / 128 - 1);
    auto touch_ahead = [&](int n) {
      asm volatile("global_load_dword %0, %1, %2" : "+v"(touched) : "v"(t_off), "s"(my_blobs + (int64_t)n * Blob::kBytes) : "memory");
    };
    // Copies of one chunk that this wavefront has in flight: they are its youngest when it waits for the chunk before.
    static_assert(NCP % KPW == 1 && NCP / KPW + 2 < 16, "copies per wavefront: base + 1 (0), base (1), base + 1 (2, 3: V)");
    auto older_landed = [&](bool more, bool touching) {
      constexpr int base = NCP / KPW;
      if (!more) __builtin_amdgcn_s_waitcnt(0x0F70);
      else if (pw == 0 && touching) __builtin_amdgcn_s_waitcnt(0x0F70 | (base + 2));
      else if (pw != 1 || touching) __builtin_amdgcn_s_waitcnt(0x0F70 | (base + 1));
      else __builtin_amdgcn_s_waitcnt(0x0F70 | base);
      asm volatile("" ::: "memory");
    };
    if (nc > 0) issue_copies(0, 0);
    if (nc > 1) issue_copies(1, 1);
    older_landed(nc > 1, false);
    __syncthreads();
    int st = 2;                               // stage of chunk n + 2
    for (int n = 0; n < nc; ++n) {
      const bool touching = n + kAhead < nc;
      if (n + 2 < nc) issue_copies(n + 2, st);
      if (touching && pw < 2) touch_ahead(n + kAhead);
      older_landed(n + 2 < nc, touching);
      st = st == KSTAGES - 1 ? 0 : st + 1;
      __syncthreads();
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);
    asm volatile("" :: "v"(touched));
    return;
  }

  // ---- per-lane LDS read offsets (bytes, inside a stage) ------------------------------------
  // A operand of a 16x16x32 MFMA: lane (row ln, k-group q4) reads piece 4m + q4 of its row; rows 16 apart share a swizzle.
  const int ct = wave % KCT;
  int rdk[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) rdk[m] = ln * 2 * KD + 16 * ((4 * m + q4) ^ piece_swizzle<2 * KD>(ln));
  const int rd64 = ln * 64 + 16 * (q4 ^ piece_swizzle<64>(ln));
  lds_cptr stage0 = (lds_cptr)&stage[0][0];
  int so = 0;                                 // stage of the chunk at hand

  if (wave >= KCT) {
    // ================= output wavefront =================
    const int piece = lane & 1, col = KVS * (KCT * grp + ct) + 8 * piece;
    f32x4 O[2];
    bf16x8 ph[2], pl[2];
    // O(n) += (P T) X, then the 32 rows of 32 bytes leave: two lanes per row
    auto finish = [&](int n) {
      const bf16x8 Xh = __builtin_bit_cast(bf16x8, xx[n & 1][ct][0][lane]), Xl = __builtin_bit_cast(bf16x8, xx[n & 1][ct][1][lane]);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        O[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pl[mt], Xh, O[mt], 0, 0, 0);
        O[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph[mt], Xl, O[mt], 0, 0, 0);
        O[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ph[mt], Xh, O[mt], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) ost[ct][16 * mt + 4 * q4 + r][ln] = (uint16_t)(pack_bf16x2(O[mt][r], 0.f) & 0xffffu);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const u32x4 v = *reinterpret_cast<const u32x4*>(&ost[ct][lane >> 1][8 * piece]);
      const int tok = sp.tok0 + n * KC + (lane >> 1);
      if (tok < sp.tok_end && col < p.Dv) *reinterpret_cast<u32x4*>(p.o + ((int64_t)tok * p.H + h) * p.Dv + col) = v;
    };
    __syncthreads();
    for (int n = 0; n < nc; ++n) {
      lds_cptr sb = stage0 + so;
      so = so == (KSTAGES - 1) * kStage ? 0 : so + kStage;
      if (n > 0) finish(n - 1);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        ph[mt] = lds_bf16x8(sb + Blob::kPh + 16 * mt * 64 + rd64);
        pl[mt] = lds_bf16x8(sb + Blob::kPl + 16 * mt * 64 + rd64);
        O[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const bf16x8 Sb = __builtin_bit_cast(bf16x8, xs[n & 1][ct][m][lane]);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          O[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_bf16x8(sb + Blob::kQg + 16 * mt * 2 * KD + rdk[m]), Sb, O[mt], 0, 0, 0);
      }
      __syncthreads();
    }
    if (nc > 0) finish(nc - 1);
    // rows behind the last sequence of a packed batch belong to none: zeros
    if (p.n_seq > 0 && b == p.n_seq - 1 && col < p.Dv)
      for (int tok = rows_end + (lane >> 1); tok < p.T; tok += 32) *reinterpret_cast<u32x4*>(p.o + ((int64_t)tok * p.H + h) * p.Dv + col) = u32x4{0u, 0u, 0u, 0u};
    return;
  }

  // ================= chain wavefront =================
  const int vcol = KVS * (KCT * grp + ct) + ln;
  const int rdv = kV + (4 * q4 + (ln >> 2)) * 64 + 2 * (KVS * ct + 4 * (ln & 3));
  // State tile i: rows (key channels) 16*i + 4*q4 + r, column vcol; rows beyond Dk and columns beyond Dv do not
  // exist in the caller's [Dk, Dv] state: they are zero and stay zero.
  const bool col_live = vcol < p.Dv;
  f32x4 S[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * i + 4 * q4 + r;
      S[i][r] = (p.s0 && col_live && row < p.Dk) ? p.s0[((int64_t)bh * p.Dk + row) * p.Dv + vcol] : 0.f;
    }
  }
  bf16x8 Sb[NM];   // the state as right operand, by channel group
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    Sb[m] = pack_acc2(S[2 * m], S[2 * m + 1]);
    xs[0][ct][m][lane] = __builtin_bit_cast(u32x4, Sb[m]);
  }
  __syncthreads();

  for (int n = 0; n < nc; ++n) {
    const int par = n & 1;
    lds_cptr sb = stage0 + so;
    so = so == (KSTAGES - 1) * kStage ? 0 : so + kStage;

    // A 16-byte LDS read keeps a wavefront's port for 16 cycles and this wavefront needs forty of them per chunk: what
    // X needs is read first, everything else between the products and the conversions that do not need it.
    bf16x8 ka[2][NM], mh[NS], ml[NS];
    u32x2 vr[2];
    f32x4 dcc[NS];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) vr[mt] = lds_column4(sb + rdv + 16 * mt * 64);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) ka[mt][m] = lds_bf16x8(sb + Blob::kKg + 16 * mt * 2 * KD + rdk[m]);
    }
    __builtin_amdgcn_sched_barrier(0);

    // X = V + (-exp(G) K) S0, row tile mt: positions 16*mt + 4*q4 + r, column vcol
    f32x4 X[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) X[mt] = f32x4{bf16lo_to_f32(vr[mt].x), bf16hi_to_f32(vr[mt].x), bf16lo_to_f32(vr[mt].y), bf16hi_to_f32(vr[mt].y)};
#pragma unroll
    for (int m = 0; m < NM; ++m) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) X[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[mt][m], Sb[m], X[mt], 0, 0, 0);
#pragma unroll
      for (int i = m * NS / NM; i < (m + 1) * NS / NM; ++i) dcc[i] = lds_f32x4(sb + Blob::kDec + 4 * (16 * i + 4 * q4));
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      ml[i] = lds_bf16x8(sb + Blob::kMl + 16 * i * 64 + rd64);
      mh[i] = lds_bf16x8(sb + Blob::kMh + 16 * i * 64 + rd64);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] *= dcc[i][r];
      __builtin_amdgcn_sched_barrier(0);
    }
    // S = exp(G_last) (.) S + M X, both operands split into two bf16 terms
    const bf16x8 Xh = pack_acc2(X[0], X[1]);
#pragma unroll
    for (int i = 0; i < NS; ++i) S[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ml[i], Xh, S[i], 0, 0, 0);
    const bf16x8 Xl = pack_rest2(X[0], X[1], Xh);
    {
      xx[par][ct][0][lane] = __builtin_bit_cast(u32x4, Xh);
      xx[par][ct][1][lane] = __builtin_bit_cast(u32x4, Xl);
    }
#pragma unroll
    for (int i = 0; i < NS; ++i) S[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mh[i], Xh, S[i], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < NS; ++i) S[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mh[i], Xl, S[i], 0, 0, 0);
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      Sb[m] = pack_acc2(S[2 * m], S[2 * m + 1]);
      xs[par ^ 1][ct][m][lane] = __builtin_bit_cast(u32x4, Sb[m]);
    }
    __syncthreads();
  }
  if (p.s_out != nullptr && col_live) {
#pragma unroll
    for (int i = 0; i < NS; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * i + 4 * q4 + r;
        if (row < p.Dk) p.s_out[((int64_t)bh * p.Dk + row) * p.Dv + vcol] = S[i][r];
      }
  }
}

}  // namespace daisy

using namespace daisy;

extern "C" int daisy_kda_gate_fwd(const void* g, const float* A_log, const float* bias, void* out,
                                  int64_t rows, int H, int Dk, int io_is_bf16,
                                  float softplus_beta, float threshold, void* stream) {
  DAISY_CHECK_ARG(g && A_log && out, "kda_gate: g, A_log and out must be non-NULL");
  DAISY_CHECK_ARG(rows >= 0 && H > 0 && Dk > 0, "kda_gate: rows=%lld, H=%d, Dk=%d invalid", (long long)rows, H, Dk);
  DAISY_CHECK_ARG(softplus_beta > 0.f, "kda_gate: softplus beta must be positive");
  const int64_t total = rows * H * Dk;
  if (total == 0) return DAISY_OK;
  hipStream_t s = (hipStream_t)stream;
  const bool vec = Dk % 8 == 0 && (reinterpret_cast<uintptr_t>(g) & 15) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  const int64_t nblk = ((vec ? total / 8 : total) + 255) / 256;
  DAISY_CHECK_ARG(nblk <= 0x7fffffff, "kda_gate: too many elements");
  const dim3 grid((unsigned)nblk), block(256);
  if (vec && io_is_bf16) hipLaunchKernelGGL((kda_gate_kernel<true, 8>), grid, block, 0, s, g, A_log, bias, out, total, H, Dk, softplus_beta, threshold);
  else if (vec) hipLaunchKernelGGL((kda_gate_kernel<false, 8>), grid, block, 0, s, g, A_log, bias, out, total, H, Dk, softplus_beta, threshold);
  else if (io_is_bf16) hipLaunchKernelGGL((kda_gate_kernel<true, 1>), grid, block, 0, s, g, A_log, bias, out, total, H, Dk, softplus_beta, threshold);
  else hipLaunchKernelGGL((kda_gate_kernel<false, 1>), grid, block, 0, s, g, A_log, bias, out, total, H, Dk, softplus_beta, threshold);
  DAISY_CHECK_LAUNCH("kda_gate_kernel");
  return DAISY_OK;
}


// Chunk slots of the workspace: B * ceil(T / 32), or for n_seq packed sequences of T tokens in all
// the upper bound T / 32 + n_seq on sum(ceil(len / 32)).
static size_t kda_chunk_slots(int B, int T, int n_seq) {
  return n_seq > 0 ? (size_t)T / KC + (size_t)n_seq : (size_t)B * ((size_t)(T + KC - 1) / KC);
}
static size_t kda_table_bytes(int T, int n_seq) {
  if (n_seq <= 0) return 0;
  const size_t ints = 2 * ((size_t)n_seq + 1) + kda_chunk_slots(1, T, n_seq);
  return (ints * sizeof(int32_t) + 255) & ~(size_t)255;
}
// The workspace is sized for the widest heads whatever the width (part of the contract); narrower ones leave its end untouched.
constexpr size_t kBlobBytes = KdaBlob<128>::kBytes;

// Head widths the kernels serve: Dk a multiple of 8 up to 128, Dv any multiple of 8.  `chunk` is the caller's idea of the
// algorithm's chunk (64); the result does not depend on where the chunks lie, and the kernels use 32.
constexpr int kApiChunk = 64;
static bool kda_dims_ok(int Dk, int Dv) { return Dk >= 8 && Dk <= KDMAX && Dk % 8 == 0 && Dv >= 8 && Dv % 8 == 0; }

extern "C" size_t daisy_kda_workspace_bytes(int B, int T, int H, int Dk, int Dv, int chunk) {
  if (B <= 0 || T <= 0 || H <= 0 || !kda_dims_ok(Dk, Dv) || chunk != kApiChunk) return 0;
  return kda_chunk_slots(B, T, 0) * H * kBlobBytes;
}

extern "C" size_t daisy_kda_varlen_workspace_bytes(int T, int n_seq, int H, int Dk, int Dv, int chunk) {
  if (T <= 0 || n_seq <= 0 || H <= 0 || !kda_dims_ok(Dk, Dv) || chunk != kApiChunk) return 0;
  return kda_chunk_slots(1, T, n_seq) * H * kBlobBytes + kda_table_bytes(T, n_seq);
}

template <int KD>
static int kda_launch_width(const KdaParams& p, int n_streams, hipStream_t s) {
  const int groups = (p.Dv + KVS * KCT - 1) / (KVS * KCT);
  hipLaunchKernelGGL(kda_prep_kernel<KD>, dim3((p.NC + 1) / 2, p.H, p.n_seq > 0 ? 1 : p.B), dim3(256), 0, s, p);
  DAISY_CHECK_LAUNCH("kda_prep_kernel");
  hipLaunchKernelGGL(kda_state_kernel<KD>, dim3((unsigned)(n_streams * p.H * groups)), dim3(kStateThreads), 0, s, p);
  DAISY_CHECK_LAUNCH("kda_state_kernel");
  return DAISY_OK;
}

// Shared by the batched and the packed entry point (n_seq == 0: batched).
static int kda_chunk_launch(const void* q, const void* k, const void* v,
                            const void* g, int g_is_bf16, const float* beta,
                            const int32_t* cu_seqlens, int n_seq,
                            const float* initial_state, void* o, float* final_state,
                            int B, int T, int H, int Dk, int Dv, int chunk,
                            float scale, int l2norm_qk, float l2_eps,
                            void* workspace, size_t workspace_bytes, void* stream) {
  DAISY_CHECK_SUPPORTED(kda_dims_ok(Dk, Dv), "kda: Dk=%d, Dv=%d not supported (Dk: a multiple of 8 up to %d; Dv: a multiple of 8)", Dk, Dv, KDMAX);
  DAISY_CHECK_SUPPORTED(chunk == kApiChunk, "kda: chunk=%d not supported (must be %d)", chunk, kApiChunk);
  DAISY_CHECK_ARG(q && k && v && g && beta && o, "kda: q, k, v, g, beta and o must be non-NULL");
  DAISY_CHECK_ARG(B > 0 && T > 0 && H > 0, "kda: B=%d, T=%d, H=%d must be positive", B, T, H);
  DAISY_CHECK_ARG(B <= 65535 && H <= 65535, "kda: B and H must each be <= 65535");
  DAISY_CHECK_ARG((int64_t)B * T <= 0x7fffffff, "kda: B*T too large");
  DAISY_CHECK_ARG((int64_t)H * Dk * KC < 0x7fffffff && (int64_t)H * Dv * KC * 2 < 0x7fffffff, "kda: token rows too long");
  auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  DAISY_CHECK_ARG(al16(q) && al16(k) && al16(v) && al16(g) && al16(o) && al16(workspace),
                  "kda: tensors and workspace must be 16-byte aligned");
  const size_t slots = kda_chunk_slots(B, T, n_seq);
  const size_t need = slots * H * kBlobBytes + kda_table_bytes(T, n_seq);
  if (!workspace || workspace_bytes < need) {
    set_error("kda: workspace of %zu bytes needed, got %zu", need, workspace_bytes);
    return DAISY_ERR_WORKSPACE;
  }
  DAISY_CHECK_ARG(slots <= 0x7fffffff && (int64_t)(n_seq > 0 ? n_seq : B) * H * ((Dv + KVS * KCT - 1) / (KVS * KCT)) <= 0x7fffffff,
                  "kda: too many chunks or sequences");
  KdaParams p;
  p.q = (const uint16_t*)q; p.k = (const uint16_t*)k; p.v = (const uint16_t*)v;
  p.g = g; p.g_bf16 = g_is_bf16; p.beta = beta;
  p.s0 = initial_state; p.o = (uint16_t*)o; p.s_out = final_state;
  p.B = B; p.T = T; p.H = H;
  p.NC = n_seq > 0 ? (int)slots : (T + KC - 1) / KC;
  p.nc_total = (int)slots;
  p.scale = scale; p.l2norm = l2norm_qk; p.l2eps = l2_eps;
  char* w = (char*)workspace;
  p.blobs = w;
  w += slots * H * kBlobBytes;
  p.n_seq = n_seq; p.cu = cu_seqlens; p.bounds = p.seq_chunk0 = p.chunk_seq = nullptr;
  hipStream_t s = (hipStream_t)stream;
  if (n_seq > kScanSeqs) {
    int32_t* tab = (int32_t*)w;
    int32_t* bounds = tab; int32_t* seq_chunk0 = tab + n_seq + 1; int32_t* chunk_seq = tab + 2 * (n_seq + 1);
    hipLaunchKernelGGL(kda_chunk_table_kernel, dim3(1), dim3(256), 0, s, cu_seqlens, n_seq, T, (int)slots, bounds, seq_chunk0, chunk_seq);
    DAISY_CHECK_LAUNCH("kda_chunk_table_kernel");
    p.bounds = bounds; p.seq_chunk0 = seq_chunk0; p.chunk_seq = chunk_seq;
  }
  const int n_streams = n_seq > 0 ? n_seq : B;    // independent recurrences per head
  p.Dk = Dk; p.Dv = Dv;
  return Dk <= 64 ? kda_launch_width<64>(p, n_streams, s) : kda_launch_width<128>(p, n_streams, s);
}

extern "C" int daisy_kda_chunk_fwd(const void* q, const void* k, const void* v,
                                   const void* g, int g_is_bf16, const float* beta,
                                   const float* initial_state, void* o, float* final_state,
                                   int B, int T, int H, int Dk, int Dv, int chunk,
                                   float scale, int l2norm_qk, float l2_eps,
                                   void* workspace, size_t workspace_bytes, void* stream) {
  return kda_chunk_launch(q, k, v, g, g_is_bf16, beta, nullptr, 0, initial_state, o, final_state, B, T, H, Dk, Dv, chunk,
                          scale, l2norm_qk, l2_eps, workspace, workspace_bytes, stream);
}

extern "C" int daisy_kda_chunk_varlen_fwd(const void* q, const void* k, const void* v,
                                          const void* g, int g_is_bf16, const float* beta,
                                          const int32_t* cu_seqlens, int n_seq,
                                          const float* initial_state, void* o, float* final_state,
                                          int T, int H, int Dk, int Dv, int chunk,
                                          float scale, int l2norm_qk, float l2_eps,
                                          void* workspace, size_t workspace_bytes, void* stream) {
  DAISY_CHECK_ARG(cu_seqlens != nullptr && n_seq >= 1, "kda_varlen: cu_seqlens and n_seq >= 1 are required");
  return kda_chunk_launch(q, k, v, g, g_is_bf16, beta, cu_seqlens, n_seq, initial_state, o, final_state, 1, T, H, Dk, Dv,
                          chunk, scale, l2norm_qk, l2_eps, workspace, workspace_bytes, stream);
}
