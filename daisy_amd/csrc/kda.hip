// Kernel 3: chunked Kimi Delta Attention forward and its log-decay gate (gfx950).
#include "common.h"
#include <type_traits>
#include <utility>

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
// columns are independent of each other, so any Dv (a multiple of 8) is served in groups of 32 or 64.
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
// KdaBlob<KD>::kBytes per chunk, whose KiB are operands as the lanes of the other kernel hold them (piece i of 16 bytes is lane i's):
//   Kg  = -exp(G) (.) K             bf16 [32][KD]
//   Qg  = scale exp(G) (.) Q        bf16 [32][KD]
//   Mh + Ml = (exp(G_last - G) (.) K)^T T split into two bf16 terms, [KD][32]: rows in the order of the state's tiles, columns
//                                   (positions) permuted
//   Ph + Pl = scale tril(P) T       the same, [32][32], columns permuted
//   dec = exp(G_last)               fp32 [KD]
// kda_state_kernel (one workgroup per (batch, head, 32 or 64 value columns)) then walks the chunks in order with the fp32
// state in registers; every product in it is a v_mfma_f32_16x16x32_bf16 whose B operand is an accumulator (S0 or X)
// converted to bf16 in place: in the 16x16 accumulator layout lane l holds column l%16 and rows 4*(l/16)+r of each
// tile, so two stacked tiles give the lane 8 contraction indices, (t, r) with t = 0,1; r = 0..3.  The state's tiles 2 m and 2 m + 1
// hold channels 32 m + 8 (row/4) + 4 t + row%4, so that a lane's eight are neighbours and one 16-byte piece of Kg or Qg as they
// are; X's tiles hold positions 16 t + 4 (row/4) + row%4, and M and P are stored with their columns permuted to match.
//
// What bounds it.  Of the first kernel, at B4 T8192 H16 with fp32 log-decays, mostly memory: 1.15 GB (539 MB of inputs, 612 MB of blocks) in
// 203 us, 5.7 TB/s where the streaming kernels reach 6.3; otherwise its vector instructions and their latency.  The second is a serial chain of chunks; what sets the time of a
// link is not the chain itself (without it the kernel is as fast) but its 39 KB of operands: a compute unit has about 64 KB
// of requests in flight, 62 GB/s from memory (160 GB/s if they are in the L2).  0.57 us a link at T = 8192 with 4 heads of
// 128 (0.63 before operands lay in the lanes' order and the outputs' came past the LDS), 0.39 us with 4 heads of 64, 0.67 us with 16 of 128,
// whose blocks come from memory and not from the last-level cache (0.70), 0.88 us with 64 of 128 (0.93), where all compute units ask at once.
//
// Numerics: the 16x16 blocks of A and P run on MFMA with both operands referenced to the row before the block (every
// exponent <= 0 off the diagonal); a diagonal block whose total decay exceeds exp(-80) is referenced to its middle row
// instead (exponents up to the decay of 8 rows either way); when those go beyond exp(-80) it is taken by halves, of 8, 4, 2 and
// 1 rows: no exponent is ever positive, so strong decays cannot overflow.  These products are in two-term bf16 splits (2^-18 of
// either operand) and, where four rows alone decay beyond exp(-80), in fp32.
// T is computed in fp32; the products with T, the state update and the output's second term use two-term bf16 splits of
// both operands (three MFMAs each, relative error ~2^-17), which keeps the state error near fp32.
// ===========================================================================
constexpr int KC = 32;    // chunk length
constexpr int KDMAX = 128;
constexpr int KVS = 16;   // value columns per state wavefront

// One chunk's block in the workspace: byte offsets of its parts (first what the chain reads, then what the outputs read).
template <int KD> struct KdaBlob {
  static constexpr int kKg = 0, kMh = KC * KD * 2, kMl = 2 * KC * KD * 2, kDec = 3 * KC * KD * 2;
  static constexpr int kChain = (kDec + KD * 4 + 1023) & ~1023;      // whole 1 KiB copies
  static constexpr int kQg = kChain, kPh = kQg + KC * KD * 2, kPl = kPh + KC * KC * 2;
  static constexpr int kBytes = kPl + KC * KC * 2;
};
static_assert(KdaBlob<128>::kBytes == 37 * 1024 && KdaBlob<64>::kBytes == 21 * 1024, "");
struct KdaParams {
  const uint16_t* q; const uint16_t* k; const uint16_t* v;
  const void* g; int g_bf16; const float* beta;
  const float* s0; uint16_t* o; float* s_out;
  int B, T, H, NC; float scale; int l2norm; float l2eps;
  int Dk, Dv;     // the tensors' own widths: Dk <= KD key channels, Dv value columns
  char* blobs;    // [nc_total][H][KdaBlob<KD>::kBytes]
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
// them (6 us).  BY_LENGTH: `key` counts from the longest one on, equal ones in their order (a lane per sequence only); it becomes
// the sequence's number.
constexpr int kScanSeqs = 64;
struct SeqScan { int begin, end, nc, upto; };      // a sequence per lane: token rows, chunks, chunks up to its end
__device__ __forceinline__ SeqScan packed_scan(const KdaParams& p) {
  const int lane = threadIdx.x & 63;
  SeqScan c;
  c.end = min(max(p.cu[min(lane + 1, p.n_seq)], p.cu[0]), p.T);
  c.end = max(c.end, 0);
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int left = __shfl_up(c.end, off);
    if (lane >= off) c.end = max(c.end, left);
  }
  c.begin = __shfl_up(c.end, 1);
  c.begin = lane == 0 ? 0 : c.begin;
  c.nc = lane < p.n_seq ? (c.end - c.begin + KC - 1) / KC : 0;
  c.upto = c.nc;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int left = __shfl_up(c.upto, off);
    if (lane >= off) c.upto += left;
  }
  return c;
}
// A lane's sequence's rank by length, the longest has 0, equal ones in their order; the sequence of a rank.
__device__ __forceinline__ int length_rank(const KdaParams& p, const SeqScan& c) {
  const uint32_t mine = ((uint32_t)c.nc << 6) + 63 - (threadIdx.x & 63);          // (no two the same)
  int ahead = 0;
#pragma unroll 4
  for (int j = 0; j < p.n_seq; ++j) ahead += (uint32_t)__builtin_amdgcn_readlane((int)mine, j) > mine ? 1 : 0;
  return ahead;
}
__device__ __forceinline__ int sequence_ranked(const KdaParams& p, int rank, int which) {
  return __builtin_ctzll(__ballot((int)(threadIdx.x & 63) < p.n_seq && rank == which));
}
template <bool BY_LENGTH> __device__ __forceinline__ SeqSpan scanned_span(const KdaParams& p, const SeqScan& c, int& key, bool by_slot, int& rows_end) {
  SeqSpan s{0, 0, 0, 0};
  const int lane = threadIdx.x & 63;
  rows_end = __builtin_amdgcn_readlane(c.end, 63);     // (lanes past the last sequence repeat its end)
  if (by_slot) {
    const uint64_t owner = __ballot(key >= c.upto - c.nc && key < c.upto);
    if (owner == 0) return s;
    key = __builtin_ctzll(owner);
  }
  if constexpr (BY_LENGTH) {
    const int before = __shfl_up(c.nc, 1);
    if (__ballot(c.nc > before && lane > 0) != 0) key = sequence_ranked(p, length_rank(p, c), key);      // (not in that order already)
  }
  s.tok0 = __builtin_amdgcn_readlane(c.begin, key); s.tok_end = __builtin_amdgcn_readlane(c.end, key);
  s.nc = __builtin_amdgcn_readlane(c.nc, key); s.c0 = __builtin_amdgcn_readlane(c.upto, key) - s.nc;
  return s;
}
template <bool BY_LENGTH = false> __device__ __forceinline__ SeqSpan packed_span(const KdaParams& p, int& key, bool by_slot, int& rows_end) {
  if (p.bounds != nullptr) {
    SeqSpan s{0, 0, 0, 0};
    rows_end = p.bounds[p.n_seq];
    if (by_slot) {
      if (key >= p.seq_chunk0[p.n_seq]) return s;
      key = p.chunk_seq[key];
    }
    s.tok0 = p.bounds[key]; s.tok_end = p.bounds[key + 1];
    s.c0 = p.seq_chunk0[key]; s.nc = p.seq_chunk0[key + 1] - s.c0;
    return s;
  }
  return scanned_span<BY_LENGTH>(p, packed_scan(p), key, by_slot, rows_end);
}
template <bool BY_LENGTH> __device__ __forceinline__ SeqSpan seq_span(const KdaParams& p, int& seq, int& rows_end) {
  if (p.n_seq > 0) return packed_span<BY_LENGTH>(p, seq, false, rows_end);
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

__device__ __forceinline__ f32x4 lds_f4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

// Eight floats as two 16-byte pieces of bf16 terms (value = hi + lo up to 2^-18 relative).
__device__ __forceinline__ void split_pack8(const float* x, u32x4& hi, u32x4& lo) {
  float h[8], l[8];
  hi = pack8(x);
  unpack8(hi, h);
#pragma unroll
  for (int e = 0; e < 8; ++e) l[e] = x[e] - h[e];
  lo = pack8(l);
}
// LDS writes of a wavefront before this point are seen by all of its lanes after it.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
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
// The value that lane N of the same 16 holds.
template <int N> __device__ __forceinline__ float from_row(float x) { return dpp_move<0x150 + N>(x); }
__device__ __forceinline__ float sum_over_q4(float x) {       // over the four lanes that share a row of an operand
  const LanePair r = row_pair(x);
  const LanePair t = half_pair(r.x + r.y);
  return t.x + t.y;
}

// A chunk's block in the workspace, stored in pieces of 16 bytes past the caches or through them: there the cache policy sc1 writes
// through the L2 at once.  Left dirty there, all blocks of a launch of a few rounds are written back at its end (512 chunks x heads of
// 128: 16.7 us, 13.3 written through).  As buffer stores, which take the policy as an argument.  The whole offset is the lane's: the
// instruction behind a store of 16 bytes must not write its data registers yet, and with an offset in a scalar register the compiler
// does not keep it from that (the first word of a piece was then, in some 20 of 928 blocks, what the next instruction had put there).
constexpr int kWriteThrough = 16;             // sc1
constexpr int kBufferWord3 = 0x00020000;      // an untyped buffer of bytes
template <bool STREAMED> struct BlockOut {
  char* base;
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ BlockOut(char* b, int bytes) : base(b), rsrc(__builtin_amdgcn_make_buffer_rsrc(b, 0, bytes, kBufferWord3)) {}
  __device__ __forceinline__ void store(const u32x4& v, int at, int part) const {        // byte `at` (the lane's) of the part at byte `part`
    if (STREAMED) __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(base + part + at));
    else __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, at + part, 0, kWriteThrough);
  }
};

// A workgroup makes one chunk, a wavefront one block of 16 rows.  Everything a wavefront does before the triangle's inverse
// it does in the layout of a matrix operand: lane (row li, q4) holds channels 32 m + 8 q4 + e of its row, of k, of q and of
// the running log-decay.  The running sum comes in that layout from a product with a triangle of ones on the fp32 matrix
// instructions (left operand: channels, straight from memory, two of them per load), so g passes through neither LDS nor
// vector instructions; it is the sum inside the wavefront's own 16 rows, which is the reference the block's products want.
// Each factor is then one exponential per element for everything it is needed for, and rows 3, 7, 11, 15 that serve as
// references are lane moves.  Two chunks per workgroup with sums, norms, block rows and operands each in a layout of their own and
// exponentials taken anew for each were bound by their vector instructions, 27000 cycles per 64 rows: with the layer's log-decays
// (bf16, half of the diagonal blocks steep) B4 T8192 H16 took 292 us and takes 203, T = 777 of 8 heads 24.5 and 12.
// *Tried:* both kernels in one launch, two of these wavefronts beside the chain's and blocks shared by flags through the L2: a
// wavefront alone needs 15000 cycles per block, 2 us a link.  *Tried:* the running sum by adds across lanes (fewer instructions, one
// more round through the LDS for g): the same time.
template <int KD, bool STREAMED>
__global__ __launch_bounds__(128, 3) void kda_prep_kernel(KdaParams p) {
  using Blob = KdaBlob<KD>;
  constexpr int NM = KD / 32, ROW = 2 * KD;                           // contraction groups of 32 channels, bytes of a bf16 row
  // rows[0] / rows[1]: k / q as given; then the two terms of exp(G_last - G) k.  A
  // wavefront's 16 rows are its own until the last use.
  __shared__ __attribute__((aligned(1024))) char rows[2][KC * ROW];
  __shared__ __attribute__((aligned(16))) char kcol[16 * ROW];        // the first block's columns for block (1, 0)
  __shared__ __attribute__((aligned(16))) float Et[2][KD];            // decay of either block of 16 rows
  __shared__ __attribute__((aligned(16))) float Td[2][16][20];        // first A_II as [column j][row i] of 16 x 16, then (I + A_II)^-1 as [row][column]
  __shared__ __attribute__((aligned(16))) float Ao[16][20];           // A_10, [row][column]
  __shared__ __attribute__((aligned(16))) float bt[KC], rks[KC];      // beta (0 for padded rows), 1 / |k|

  // 32 chunks of a head in neighbouring workgroups, then as many of the next head: what runs at a time reads and writes neighbouring memory, token
  // rows as much as blocks, whose order in the workspace is the tokens'; and workgroups of one head, which differ in how steep their decays
  // are, run side by side.  T = 8192, 16 heads, all chunks of a head (and of its blocks) in a row / 32 / 1: mild fp32 log-decays B = 1 62 / 57 / 57 us, 2
  // 115 / 105 / 104, 3 168 / 151 / 152, 4 213 / 204 / 203; a layer's first gates (bf16) B = 2 121 / 116 / 132, 4 251 / 248 / 273.
  int h, slot;
  {
    constexpr uint32_t kRun = 32;
    const uint32_t run = blockIdx.x / (kRun * p.H), at = blockIdx.x % (kRun * p.H), n = min(kRun, p.NC - kRun * run);
    h = (int)(at / n);
    slot = (int)(kRun * run + at % n);
  }
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, q4 = lane >> 4;
  const int I = __builtin_amdgcn_readfirstlane(tid >> 6);
  int t0, n_live;
  int64_t ci;
  {
    if (p.n_seq > 0) {
      int seq = slot, rows_end;
      const SeqSpan sp = packed_span(p, seq, true, rows_end);
      if (sp.nc == 0) return;                    // surplus slots (the grid covers the upper bound)
      t0 = sp.tok0 + (slot - sp.c0) * KC;
      n_live = min(sp.tok_end - t0, KC);
      ci = (int64_t)slot * p.H + h;
    } else {
      t0 = blockIdx.z * p.T + slot * KC;
      n_live = min((int)(blockIdx.z + 1) * p.T - t0, KC);
      ci = ((int64_t)blockIdx.z * p.NC + slot) * p.H + h;
    }
  }
  const bool edge = n_live < KC || p.Dk < KD;     // rows or channels that do not exist: read as copies of others, then zeroed
  const uint32_t row_stride = (uint32_t)p.H * (uint32_t)p.Dk;         // elements between token rows of one head (q, k, g)
  const int64_t tok_base = ((int64_t)t0 * p.H + h) * p.Dk;
  const BlockOut<STREAMED> block(p.blobs + ci * Blob::kBytes, Blob::kBytes);

  // ---- every global load goes out at once: g as left operand, k and q rows into the LDS (swizzled), beta ----
  // g: tile t of group m holds channels 32 m + 8 (row / 4) + 2 (row % 4) + t, so that a lane's two tiles are neighbours and the
  // product's rows 4 q4 + r are channels 8 q4 + 2 r + t; contraction step s: position 4 s + q4 of the block.
  const int last = n_live - 1;
  u32x2 graw[NM][4];
  {
    const int ch = 8 * (li >> 2) + 2 * (li & 3);
    auto at = [&](int s, int m) { return (uint32_t)min(16 * I + 4 * s + q4, last) * row_stride + (uint32_t)min(32 * m + ch, p.Dk - 2); };
    if (p.g_bf16) {
#pragma unroll
      for (int i = 0; i < 4 * NM; ++i)
        graw[i % NM][i / NM].x = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>((const uint16_t*)p.g + tok_base + at(i / NM, i % NM)));
    } else {
#pragma unroll
      for (int i = 0; i < 4 * NM; ++i)
        graw[i % NM][i / NM] = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>((const float*)p.g + tok_base + at(i / NM, i % NM)));
    }
  }
  const float beta = p.beta[(int64_t)(t0 + min(16 * I + li, last)) * p.H + h];
  __builtin_amdgcn_sched_barrier(0);
  lds_cptr const my_rows[2] = {(lds_cptr)&rows[0][16 * I * ROW], (lds_cptr)&rows[1][16 * I * ROW]};
  {
    constexpr int RPI = 1024 / ROW, PPR = ROW / 16;                   // rows per copy, pieces per row
#pragma unroll
    for (int j = 0; j < 16 / RPI; ++j) {
      const int r = RPI * j + lane / PPR, piece = (lane % PPR) ^ piece_swizzle<ROW>(r);
      const int off = 2 * (int)((uint32_t)min(16 * I + r, last) * row_stride + 8u * (uint32_t)min(piece, p.Dk / 8 - 1));
      copy16_to_lds_async<true>(p.k + tok_base, off, (uint32_t)(size_t)my_rows[0] + 1024 * j);
      copy16_to_lds_async<true>(p.q + tok_base, off, (uint32_t)(size_t)my_rows[1] + 1024 * j);
    }
  }

  // ---- G: running log-decay inside the block, in units of log 2; element e of group m is G[m][e % 2][e / 2] ----
  // The product multiplies rows behind a position by 0, which an infinite log-decay must not meet: one below kForgets counts as that,
  // whose exponential is 0 in fp32 already (and sums over many such rows keep the bits of the mild ones).  NaN stays NaN.
  constexpr float kForgets = -104.f;
  f32x4 G[NM][2];
#pragma unroll
  for (int m = 0; m < NM; ++m) G[m][0] = G[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const float ones = (4 * s + q4 <= li) ? kLog2e : 0.f;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      float g0 = p.g_bf16 ? bf16lo_to_f32(graw[m][s].x) : __uint_as_float(graw[m][s].x);
      float g1 = p.g_bf16 ? bf16hi_to_f32(graw[m][s].x) : __uint_as_float(graw[m][s].y);
      g0 = __builtin_elementwise_maximum(g0, kForgets);
      g1 = __builtin_elementwise_maximum(g1, kForgets);
      if (edge && (16 * I + 4 * s + q4 >= n_live || 32 * m + 8 * (li >> 2) >= p.Dk)) g0 = g1 = 0.f;
      G[m][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(g0, ones, G[m][0], 0, 0, 0);
      G[m][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(g1, ones, G[m][1], 0, 0, 0);
    }
  }

  // ---- k and q of the lane's row, and 1 over their norms ----
  const int swz = piece_swizzle<ROW>(li);
  int at[NM];                                     // the lane's piece of group m inside its wavefront's rows
#pragma unroll
  for (int m = 0; m < NM; ++m) at[m] = li * ROW + 16 * ((4 * m + q4) ^ swz);
  __builtin_amdgcn_s_waitcnt(0x0F70);             // vmcnt(0): the wavefront's own copies have landed
  asm volatile("" ::: "memory");
  float kn[NM][8], qn[NM][8], sk = 0.f, sq = 0.f;
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    u32x4 kr = __builtin_bit_cast(u32x4, lds_bf16x8(my_rows[0] + at[m])), qr = __builtin_bit_cast(u32x4, lds_bf16x8(my_rows[1] + at[m]));
    if (edge && (16 * I + li >= n_live || 32 * m + 8 * q4 >= p.Dk)) kr = qr = u32x4{0u, 0u, 0u, 0u};
    unpack8(kr, kn[m]);
    unpack8(qr, qn[m]);
#pragma unroll
    for (int e = 0; e < 8; ++e) { sk = fmaf(kn[m][e], kn[m][e], sk); sq = fmaf(qn[m][e], qn[m][e], sq); }
  }
  // The norms (and scale) come in behind the products of k and q with their factors: where those are 1, no rounding is added.
  const float rk = p.l2norm ? rsqrtf(sum_over_q4(sk) + p.l2eps) : 1.f;
  const float rq = p.scale * (p.l2norm ? rsqrtf(sum_over_q4(sq) + p.l2eps) : 1.f);

  // ---- factors.  How steep the block is (wavefront-uniform): `gentle` while exp(-G) of every element is safe (exponents up to
  // 80); else with the block's middle row as reference while that is; else, or where a group of four rows is `steepest`, by halves. ----
  constexpr float kSafe = 80.f * kLog2e;
  float far0 = 0.f;
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int e = 0; e < 8; ++e) far0 = fmaxf(far0, fabsf(G[m][e & 1][e >> 1]));
  const bool gentle = !__any(far0 > kSafe);
  // Diagonal block of A and P on MFMA.  accA: lane holds column j = li, rows i = 4 q4 + r of the block.  P comes out
  // transposed (operands swapped: both operand layouts hold 8 contraction indices of one row / column per lane): row i = li,
  // columns j = 4 q4 + r.
  f32x4 accA = {0.f, 0.f, 0.f, 0.f}, accP = {0.f, 0.f, 0.f, 0.f};
  if (!gentle) {
    float far7 = 0.f, far4 = 0.f;
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float g = G[m][e & 1][e >> 1];
        far7 = fmaxf(far7, fabsf(g - from_row<7>(g)));
        far4 = fmaxf(far4, fabsf(g - dpp_move<0x114>(g)));      // row_shr 4, zero for the first four: in row 4 n + 3 the sum of rows 4 n ..
      }
    const bool steepest = __any((li & 3) == 3 && far4 > kSafe);
    if (!steepest && !__any(far7 > kSafe)) {
      // With the middle row as reference the entries above the diagonal may overflow; nothing reads them.
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        float ak[8], aq[8], bk[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float g = G[m][e & 1][e >> 1], d = g - from_row<7>(g), f = __builtin_amdgcn_exp2f(d);
          ak[e] = kn[m][e] * f;
          aq[e] = qn[m][e] * f;
          bk[e] = kn[m][e] * __builtin_amdgcn_exp2f(-d);
        }
        const bf16x8 col = __builtin_bit_cast(bf16x8, pack8(bk));
        accA = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pack8(ak)), col, accA, 0, 0, 0);
        accP = __builtin_amdgcn_mfma_f32_16x16x32_bf16(col, __builtin_bit_cast(bf16x8, pack8(aq)), accP, 0, 0, 0);
      }
    } else {
      // Any decay: rows and columns that differ first in bit `lev` of their number meet at the last row of the lower half of
      // their group of 2 lev rows.  The lane's row is on the row's side of that product or on the column's, never on both,
      // so a level takes one exponential per element, of a sum of log-decays; entries of other levels are dropped.  Both
      // operands in two bf16 terms, 2^-18 of either; in a block with a steepest group of four as they are, on the fp32 instructions
      // (27 % of the blocks of 6001 rows, 12 heads of 64, with a layer's first gates: both kernels 45.3 us in two terms, 47.5 with
      // products of 16 x 16 at every level, 46.2 with those of 4 x 4 below; 20 rows of 4 heads of 128, all of them steepest: 17.1 and 18.3).
      float pd = 0.f;
#pragma unroll
      for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int e = 0; e < 8; ++e) pd = fmaf(kn[m][e], qn[m][e], pd);
      pd = sum_over_q4(pd);
#pragma unroll
      for (int r = 0; r < 4; ++r) accP[r] = (4 * q4 + r == li) ? pd : 0.f;
      auto level = [&](auto lev_, auto exact_, auto ref_of) {
        constexpr int lev = decltype(lev_)::value;
        constexpr bool exact = decltype(exact_)::value;
        const bool low = (li & lev) == 0;
        f32x4 pa = {0.f, 0.f, 0.f, 0.f}, pp = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          float wk[8], wq[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float g = G[m][e & 1][e >> 1], d = g - ref_of(g), f = __builtin_amdgcn_exp2f(low ? -d : d);
            wk[e] = kn[m][e] * f;
            wq[e] = qn[m][e] * f;
          }
          if constexpr (exact && lev <= 4) {
            // Inside four rows, and of four rows with the four before them (row_shr 4): a product per group of four and q4, in a
            // quarter of the 16 x 16 one's time.
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float col = lev == 4 ? dpp_move<0x114>(wk[e]) : wk[e];
              pa = __builtin_amdgcn_mfma_f32_4x4x1f32(wk[e], col, pa, 0, 0, 0);
              pp = __builtin_amdgcn_mfma_f32_4x4x1f32(col, wq[e], pp, 0, 0, 0);
            }
          } else if constexpr (exact) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              pa = __builtin_amdgcn_mfma_f32_16x16x4f32(wk[e], wk[e], pa, 0, 0, 0);
              pp = __builtin_amdgcn_mfma_f32_16x16x4f32(wk[e], wq[e], pp, 0, 0, 0);
            }
          } else {
            u32x4 kh, kl, qh, ql;
            split_pack8(wk, kh, kl);
            split_pack8(wq, qh, ql);
            auto add = [&](const u32x4& col, const u32x4& row_k, const u32x4& row_q) {
              pa = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, row_k), __builtin_bit_cast(bf16x8, col), pa, 0, 0, 0);
              pp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, col), __builtin_bit_cast(bf16x8, row_q), pp, 0, 0, 0);
            };
            add(kl, kh, qh);
            add(kh, kl, ql);
            add(kh, kh, qh);
          }
        }
        if constexpr (exact && lev <= 4) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            pa[r] = sum_over_q4(lev == 4 ? dpp_move<0x104>(pa[r]) : pa[r]);        // (row_shl 4: back to the column's lane)
            pp[r] = sum_over_q4(pp[r]);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int x = (4 * q4 + r) ^ li;
          if (x >= lev && x < 2 * lev) { accA[r] = pa[r]; accP[r] = pp[r]; }
        }
      };
      auto levels = [&](auto exact) {
        level(std::integral_constant<int, 8>{}, exact, [&](float g) { return from_row<7>(g); });
        level(std::integral_constant<int, 4>{}, exact, [&](float g) { const float lower = from_row<3>(g), upper = from_row<11>(g); return (li & 8) ? upper : lower; });
        level(std::integral_constant<int, 2>{}, exact, [&](float g) { return dpp_move<0x55>(g); });        // row 1 of every quad
        level(std::integral_constant<int, 1>{}, exact, [&](float g) { return dpp_move<0xA0>(g); });        // the even row of every pair
      };
      if (steepest) levels(std::true_type{}); else levels(std::false_type{});
    }
  }
  // k f and q f with f = exp(G) take the place of k and q, kd = exp(G_15 - G) k that of G.
  float kd[NM][8];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    float f[8], bk[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float g = G[m][e & 1][e >> 1];
      f[e] = __builtin_amdgcn_exp2f(g);
      // gentle: bk = k exp(-G), kd = bk exp(G_15); else kd = bk = k exp(G_15 - G).  Selections: as a branch per element this and the
      // loads of g above took 0.3 of 45 us (6001 rows of 12 heads of 64), 8 to 10 of 1600 (a layer of 32768 rows, 16 heads of 128).
      const float g15 = from_row<15>(g), f15 = from_row<15>(f[e]);
      bk[e] = kn[m][e] * __builtin_amdgcn_exp2f((gentle ? 0.f : g15) - g);
      kd[m][e] = bk[e] * (gentle ? f15 : 1.f);
      kn[m][e] *= f[e];
      qn[m][e] *= f[e];
    }
    if (gentle) {
      const bf16x8 col = __builtin_bit_cast(bf16x8, pack8(bk));
      accA = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pack8(kn[m])), col, accA, 0, 0, 0);
      accP = __builtin_amdgcn_mfma_f32_16x16x32_bf16(col, __builtin_bit_cast(bf16x8, pack8(qn[m])), accP, 0, 0, 0);
    }
    if (li == 15) {
      *reinterpret_cast<f32x4*>(&Et[I][32 * m + 8 * q4]) = f32x4{f[0], f[1], f[2], f[3]};
      *reinterpret_cast<f32x4*>(&Et[I][32 * m + 8 * q4 + 4]) = f32x4{f[4], f[5], f[6], f[7]};
    }
    if (I == 0) *reinterpret_cast<u32x4*>(&kcol[at[m]]) = pack8(kd[m]);
  }
  if (q4 == 0) {
    bt[16 * I + li] = (16 * I + li < n_live) ? beta : 0.f;
    rks[16 * I + li] = rk;
  }
  __syncthreads();   // decays, beta and the first block's columns are in place

  f32x4 P[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};          // this wavefront's rows of scale tril(P), either column block
  {
    const f32x4 bt4 = lds_f4(&bt[16 * I + 4 * q4]), rk4 = lds_f4(&rks[16 * I + 4 * q4]);
    f32x4 av, pv;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      av[r] = bt4[r] * rk4[r] * rk * accA[r];     // entries with i <= j are never read
      pv[r] = (4 * q4 + r <= li) ? rq * rk4[r] * accP[r] : 0.f;
    }
    *reinterpret_cast<f32x4*>(&Td[I][0][0] + 16 * li + 4 * q4) = av;
    if (I == 0) P[0] = pv;
    else {
      P[1] = pv;
      f32x4 a10 = {0.f, 0.f, 0.f, 0.f};           // block (1, 0)
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const bf16x8 col = lds_bf16x8((lds_cptr)&kcol[0] + at[m]);
        a10 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pack8(kn[m])), col, a10, 0, 0, 0);
        P[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(col, __builtin_bit_cast(bf16x8, pack8(qn[m])), P[0], 0, 0, 0);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) Ao[4 * q4 + r][li] = bt4[r] * rk4[r] * rks[li] * a10[r];
      P[0] *= rq * lds_f4(&rks[4 * q4]);
    }
  }
  // ---- Kg = -exp(G) k, Qg = scale exp(G) q with G from the chunk's start: as the lanes hold them, whole KiB out ----
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    if (I == 1) {
      const f32x4 e0 = lds_f4(&Et[0][32 * m + 8 * q4]), e1 = lds_f4(&Et[0][32 * m + 8 * q4 + 4]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float f = e < 4 ? e0[e & 3] : e1[e & 3];
        kn[m][e] *= -rk * f;
        qn[m][e] *= rq * f;
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) { kn[m][e] *= -rk; qn[m][e] *= rq; }
    }
    block.store(pack8(kn[m]), 16 * lane, Blob::kKg + 1024 * (NM * I + m));
    block.store(pack8(qn[m]), 16 * lane, Blob::kQg + 1024 * (NM * I + m));
  }
  if (tid < KD / 4) *reinterpret_cast<f32x4*>(block.base + Blob::kDec + 16 * tid) = lds_f4(&Et[0][4 * tid]) * lds_f4(&Et[1][4 * tid]);
  // ---- exp(G_last - G) k in two bf16 terms, for the transposing reads below ----
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    if (I == 0) {
      const f32x4 e0 = lds_f4(&Et[1][32 * m + 8 * q4]), e1 = lds_f4(&Et[1][32 * m + 8 * q4 + 4]);
#pragma unroll
      for (int e = 0; e < 8; ++e) kd[m][e] *= rk * (e < 4 ? e0[e & 3] : e1[e & 3]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) kd[m][e] *= rk;
    }
    u32x4 hi, lo;
    split_pack8(kd[m], hi, lo);
    *reinterpret_cast<u32x4*>(&rows[0][16 * I * ROW + at[m]]) = hi;
    *reinterpret_cast<u32x4*>(&rows[1][16 * I * ROW + at[m]]) = lo;
  }

  // ---- T = (I + A)^-1 diag(beta).  The inverse of the wavefront's diagonal block in fp32, one column per lane (lanes
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
      for (int i4 = (j + 1) / 4; i4 < 4; ++i4) ar[i4] = lds_f4(&Td[I][0][0] + 16 * j + 4 * i4);
      const float xj = tc[j];
#pragma unroll
      for (int i = j + 1; i < 16; ++i) tc[i] = fmaf(-ar[i >> 2][i & 3], xj, tc[i]);
    }
    wave_lds_fence();
#pragma unroll
    for (int i = 0; i < 16; ++i) Td[I][i][li] = tc[i];      // all lanes, four the same: into a branch around this the compiler moves the sums, behind
                                                            // all of their operands (heads of 64: 164 registers instead of 126, three wavefronts a SIMD)
  }
  __syncthreads();   // both inverses, A_10 and the rows are in place
  // T_10 = -T_11 (A_10 T_00) in two fp32 matrix products, both wavefronts all of it.  As right operand (lane
  // (column li, rows 4 q4 + e)) and as result the layout is the same, and it is also the one T^T is wanted in below.
  f32x4 t00, t10, t11;
  {
    const f32x4 a10 = lds_f4(&Ao[li][4 * q4]), r11 = lds_f4(&Td[1][li][4 * q4]);
    f32x4 m1 = {0.f, 0.f, 0.f, 0.f};
    t10 = m1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      t00[e] = Td[0][4 * q4 + e][li];
      t11[e] = Td[1][4 * q4 + e][li];
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
    const float b0 = bt[li], b1 = bt[16 + li];
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
  // Row 16 tile + li of (right operand)^T T: the products come out with four consecutive columns of T per lane and column block,
  // which is the piece the lane's place in an operand wants; both terms of it leave from here, a KiB per instruction.
  auto times_t = [&](const bf16x8& rh, const bf16x8& rl, int part_hi, int part_lo, int tile) {
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
    u32x4 hi, lo;
    split_pack8(out, hi, lo);
    block.store(hi, 16 * lane, part_hi + 1024 * tile);
    block.store(lo, 16 * lane, part_lo + 1024 * tile);
  };
  {
    float pv[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) { pv[e] = P[0][e]; pv[4 + e] = P[1][e]; }
    u32x4 hi, lo;
    split_pack8(pv, hi, lo);
    times_t(__builtin_bit_cast(bf16x8, hi), __builtin_bit_cast(bf16x8, lo), Blob::kPh, Blob::kPl, I);
  }
  // ---- M = (exp(G_last - G) k)^T T, half of the chunk's channels per wavefront: row 16 i + li of the block is channel
  // 32 (i / 2) + 8 (li / 4) + 4 (i % 2) + li % 4, the one that row of the state's tile i stands for
  const int r0 = 4 * q4 + (li >> 2);
#pragma unroll
  for (int n = 0; n < KD / 32; ++n) {
    const int i = KD / 32 * I + n, piece = 4 * (i >> 1) + (li & 3), half = 8 * (i & 1);
    const int a0 = r0 * ROW + 16 * (piece ^ piece_swizzle<ROW>(r0)) + half;     // rows 16 apart share a swizzle
    u32x4 hi, lo;
    const u32x2 h0 = lds_column4((lds_cptr)&rows[0][0] + a0), h1 = lds_column4((lds_cptr)&rows[0][0] + a0 + 16 * ROW);
    const u32x2 l0 = lds_column4((lds_cptr)&rows[1][0] + a0), l1 = lds_column4((lds_cptr)&rows[1][0] + a0 + 16 * ROW);
    hi = u32x4{h0.x, h0.y, h1.x, h1.y};
    lo = u32x4{l0.x, l0.y, l1.x, l1.y};
    times_t(__builtin_bit_cast(bf16x8, hi), __builtin_bit_cast(bf16x8, lo), Blob::kMh, Blob::kMl, i);
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

// Tiles I .. N - 1 of a state times the decays of their rows: dec[i] those of tile i, or one register set of which lane i of 16 holds
// tile i's (a lane move in the product's operand).  `behind(i)`: what follows tile i.
template <int I, int N, int SETS, typename F> __device__ __forceinline__ void decay_tiles(f32x4* S, const f32x4 (&dec)[SETS], F behind) {
  if constexpr (I < N) {
#pragma unroll
    for (int r = 0; r < 4; ++r) S[I][r] *= SETS == 1 ? from_row<I>(dec[0][r]) : dec[I % SETS][r];
    behind(I);
    decay_tiles<I + 1, N>(S, dec, behind);
  }
}

constexpr int KPW = 2;                        // data-moving wavefronts per workgroup, and as many for the outputs
template <typename F, int... I> __device__ __forceinline__ void each_constant(F f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
constexpr int KSTAGES = 3;                    // LDS stages of chunk data
constexpr int KSETS = 4;                      // register sets of an output wavefront
template <int KCT> constexpr int kStateThreads = 64 * (KCT + 2 * KPW);

// The chunk-to-chunk chain sets the time of this kernel once its data are there, and next to it what the CU's LDS can
// deliver, 128 bytes a clock (heads of 128: some 116 KB of operands and copies per chunk with two column tiles, KCT = 2, 206 KB with four,
// which sets their link).  So:
//  * one wavefront owns one tile of 16 value columns with all of its state rows: the state never leaves its registers
//    (as right operand it is the accumulators converted in place), nothing of the chain waits for another wavefront,
//    and every operand of the chain is read once per column tile.  Two wavefronts per tile with half of the state each,
//    both computing X and handing state halves over through LDS, took 250 us instead of 230 (B4 T8192 H16, 128 x 128);
//  * the outputs are not part of the chain: two more wavefronts, with 16 of the chunk's positions each, make Qg S0 from the bf16 state
//    that the chain left in LDS, add (P T) X when X has arrived, and store the rows one chunk later.  Their operands come from memory
//    into registers, KSETS - 1 chunks ahead, once for all column tiles; a wavefront per tile, with operands through the LDS: T = 8192,
//    up to 8 heads of 128 162 -> 145 us, 16 heads 180 -> 172, 64 heads 237 -> 226 (two sets fewer or more: level);
//  * the chain does not wait for global memory: two further wavefronts issue the asynchronous copies of the chunks ahead.

// What a chain keeps in the LDS, in arrays of their own so that the compiler can tell their accesses apart.
template <int KD, int KCT> constexpr int kStageBytes = KdaBlob<KD>::kChain + KC * KVS * KCT * 2;
template <int KD, int KCT> using StageLds = char[KSTAGES][kStageBytes<KD, KCT>];
template <int KD, int KCT> using StateLds = u32x4[2][KCT][KD / 32][64];       // [chunk parity][column tile][channel group][lane]: S0 as operand
template <int KCT> using XLds = u32x4[2][KCT][2][64];                         // X as operand, two terms
// The chain of this workgroup.  span_of(b, rows_end): where sequence b lives; BY_LENGTH: b counts from the longest one on and becomes the sequence's number.
template <int KD, int KCT, bool BY_LENGTH, typename SPAN>
__device__ __forceinline__ void kda_chain(const KdaParams& p, StageLds<KD, KCT>& stage, StateLds<KD, KCT>& xs, XLds<KCT>& xx, SPAN span_of) {
  using Blob = KdaBlob<KD>;
  constexpr int NM = KD / 32, NS = KD / 16;                    // channel groups of 32, state tiles of 16 rows
  constexpr int kV = Blob::kChain, kStage = kStageBytes<KD, KCT>;
  // Links are cut by workgroup barriers.  Interval n between two of them copies the chain's part of chunk n; the chain reads it in
  // interval n + 2 and computes link n, beside its outputs, in interval n + 3.

  // The column groups of one (batch, head) on one XCD, in consecutive workgroups of it: they read the same blocks.
  const int NGRP = (p.Dv + KVS * KCT - 1) / (KVS * KCT);
  const int slot = blockIdx.x >> 3, grp = slot % NGRP;
  int bh = 8 * (slot / NGRP) + (blockIdx.x & 7);
  if (bh >= (p.n_seq > 0 ? p.n_seq : p.B) * p.H) return;
  const int h = bh % p.H;
  int b = bh / p.H, rows_end;               // b: batch element, or sequence of a packed batch
  const SeqSpan sp = span_of(b, rows_end);
  if constexpr (BY_LENGTH) bh = b * p.H + h;
  const int nc = sp.nc;                      // chunks of this sequence (0 for an empty one)
  const int64_t ci0 = (int64_t)sp.c0 * p.H + h, step = (int64_t)p.H * Blob::kBytes;
  const int lane = threadIdx.x & 63, ln = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const char* const my_blobs = p.blobs + ci0 * Blob::kBytes;
  const int col0 = KVS * KCT * grp;          // the workgroup's first value column

  if (wave >= KCT + KPW) {
    // ================= data-moving wavefront =================
    // Their instructions count: with an address, a branch and an m0 of its own for every KiB (some 250 scalar instructions
    // per chunk) these wavefronts set the time of a link.  So each takes a run of the chain's part, KiB after KiB by the instruction's own offset, the KiB with the decays (both of them, the same bytes) and 16 rows of V:
    // lane i lands at row i / 4, piece i % 4.  Pieces past the last column re-read the last one (columns are independent and dead
    // ones are not stored).
    // The column groups of a (batch, head) ask for the same bytes at the same time.  Each begins its run at another place, so that
    // first requests differ and later ones find the L2 filled (T = 8192: 64 heads of 128 469 -> 455 us, both kernels), and
    // in turns with a pause between: all at once they delay the other wavefronts' LDS and store traffic.  The pause in units of 64
    // clocks: 0 / 1 / 2 / 4 with few chains of T = 8192, heads of 128, 147 / 145 / 147 / 169 us, with 256 workgroups 231 / 229.5 / 233 (3) / 231.
    // The first chunks, which nothing computes beside, are asked for without (64 sequences of 64 rows, 16 heads of 64: 52.1 -> 50.4
    // us; 4 of 100 rows, 24 heads of 128: 32.5 -> 31.0).  *Tried:* a fourth stage: level.  *Tried:* one dword of every line fetched further
    // ahead, by these or by a wavefront of its own, and from the scalar side: slower, answers come back in order and hits wait behind misses.
    const int pw = wave - KCT - KPW;
    constexpr int NM1 = 3 * KC * KD * 2 / 1024 / KPW;
    static_assert(NM1 * KPW * 1024 == Blob::kDec && Blob::kChain - Blob::kDec == 1024, "runs of whole KiB");
    constexpr int kTurns = NM1 / 3;
    const uint32_t stage_lds = lds_address(&stage[0][0]);
    const int n_rows = sp.tok_end - sp.tok0, v_pitch = 2 * p.H * p.Dv;
    const char* const my_v = (const char*)(p.v + ((int64_t)sp.tok0 * p.H + h) * p.Dv);
    const int v_row = 16 * pw + (lane >> 2);
    int v_off[KCT / 2];
#pragma unroll
    for (int u = 0; u < KCT / 2; ++u) v_off[u] = 16 * min(col0 / 8 + 4 * u + (lane & 3), p.Dv / 8 - 1);
    auto copy_chain = [&](int n, int st) {
      const char* const block = my_blobs + n * step;
      const uint32_t to = stage_lds + st * kStage;
#pragma unroll
      for (int i = 0; i < kTurns; ++i) {
        const int first = (pw * kTurns + (i + grp) % kTurns) * (NM1 / kTurns) * 1024;
        copy_kib_to_lds_async<NM1 / kTurns>(block + first, 16 * lane, to + first);
        if (n < KSTAGES) continue;
        __builtin_amdgcn_s_sleep(1);
      }
      copy_kib_to_lds_async<1>(block + Blob::kDec, 16 * lane, to + Blob::kDec);
#pragma unroll
      for (int u = 0; u < KCT / 2; ++u)
        copy_kib_to_lds_async<1>(my_v + (int64_t)n * KC * v_pitch, min(v_row, n_rows - n * KC - 1) * v_pitch + v_off[u], to + kV + 2048 * u + 1024 * pw);
    };
    auto landed = [&](auto still) {           // all copies but the youngest `still` of this wavefront are in the LDS
      constexpr int N = decltype(still)::value;
      static_assert(N < 64, "");
      __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | (N >> 4) << 14);
      asm volatile("" ::: "memory");
    };
    int st = 0;                               // stage of chunk n
    for (int n = 0; n < nc + KSTAGES; ++n) {
      if (n < nc) {
        copy_chain(n, st);
        landed(std::integral_constant<int, (KSTAGES - 2) * (NM1 + 1 + KCT / 2)>{});
      } else {
        landed(std::integral_constant<int, 0>{});
      }
      st = st == KSTAGES - 1 ? 0 : st + 1;
      __syncthreads();
    }
    return;
  }

  if (wave >= KCT) {
    // ================= output wavefront: 16 positions of every chunk, all columns =================
    // Its rows of Qg and P come straight into registers, as operands, KSETS - 1 links ahead; the products are O^T, so that a lane has
    // four neighbouring columns of one position per tile and, of the tiles 2 u and 2 u + 1, eight.
    const int mt = wave - KCT;
    const char* const my_q = my_blobs + Blob::kQg + 1024 * NM * mt + 16 * lane;
    const char* const my_p = my_blobs + Blob::kPh + 1024 * mt + 16 * lane;
    bf16x8 qg[KSETS][NM], pt[KSETS][2];
    auto fetch = [&](auto set, int n) {
      constexpr int s = decltype(set)::value;
      const int64_t at = n * step;
#pragma unroll
      for (int m = 0; m < NM; ++m) qg[s][m] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(my_q + at + 1024 * m));
#pragma unroll
      for (int t = 0; t < 2; ++t) pt[s][t] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(my_p + at + (Blob::kPl - Blob::kPh) * t));
    };
    f32x4 O[KCT];
    uint16_t* const my_o = p.o + ((int64_t)(sp.tok0 + 16 * mt + ln) * p.H + h) * p.Dv + col0 + 8 * q4;
    // O(n) += (P T) X, then the rows leave
    auto finish = [&](auto set, int n) {
      constexpr int s = decltype(set)::value;
#pragma unroll
      for (int ct = 0; ct < KCT; ++ct) {
        const bf16x8 Xh = __builtin_bit_cast(bf16x8, xx[n & 1][ct][0][lane]), Xl = __builtin_bit_cast(bf16x8, xx[n & 1][ct][1][lane]);
        O[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Xh, pt[s][1], O[ct], 0, 0, 0);
        O[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Xl, pt[s][0], O[ct], 0, 0, 0);
        O[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Xh, pt[s][0], O[ct], 0, 0, 0);
      }
      const bool live = sp.tok0 + n * KC + 16 * mt + ln < sp.tok_end;
#pragma unroll
      for (int u = 0; u < KCT / 2; ++u) {
        const u32x4 v = {pack_bf16x2(O[2 * u][0], O[2 * u][1]), pack_bf16x2(O[2 * u][2], O[2 * u][3]),
                         pack_bf16x2(O[2 * u + 1][0], O[2 * u + 1][1]), pack_bf16x2(O[2 * u + 1][2], O[2 * u + 1][3])};
        if (live && col0 + 32 * u + 8 * q4 < p.Dv) *reinterpret_cast<u32x4*>(my_o + (int64_t)n * KC * p.H * p.Dv + 32 * u) = v;
      }
    };
    auto link = [&](auto set, int n) {
      constexpr int s = decltype(set)::value, before = (s + KSETS - 1) % KSETS;
      if (n > 0) finish(std::integral_constant<int, before>{}, n - 1);
      fetch(std::integral_constant<int, before>{}, min(n + KSETS - 1, nc - 1));
#pragma unroll
      for (int ct = 0; ct < KCT; ++ct) {
        O[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < NM; ++m)
          O[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xs[n & 1][ct][m][lane]), qg[s][m], O[ct], 0, 0, 0);
      }
      __syncthreads();
    };
    auto each_set = [](auto f) { each_constant(f, std::make_integer_sequence<int, KSETS>{}); };
    if (nc > 0) each_set([&](auto set) { if constexpr (decltype(set)::value < KSETS - 1) fetch(set, min((int)decltype(set)::value, nc - 1)); });
    for (int i = 0; i < KSTAGES; ++i) __syncthreads();
    for (int n = 0; n < nc; n += KSETS)
      each_set([&](auto set) {
        constexpr int s = decltype(set)::value;
        if (n + s < nc) link(set, n + s);
        if (n + s == nc - 1) finish(set, n + s);
      });
    // rows behind the last sequence of a packed batch belong to none: zeros
    if (p.n_seq > 0 && b == p.n_seq - 1)
      for (int u = 0; u < KCT / 2; ++u)
        for (int tok = rows_end + 16 * mt + ln; tok < p.T; tok += 32)
          if (col0 + 32 * u + 8 * q4 < p.Dv) *reinterpret_cast<u32x4*>(p.o + ((int64_t)tok * p.H + h) * p.Dv + col0 + 32 * u + 8 * q4) = u32x4{0u, 0u, 0u, 0u};
    return;
  }

  // ================= chain wavefront =================
  // Column ln of tile ct: the tiles 2 u and 2 u + 1 take turns in the fours of 32 columns, for the outputs' sake.
  const int ct = wave, vcol = col0 + 32 * (ct >> 1) + 8 * (ln >> 2) + 4 * (ct & 1) + (ln & 3);
  const int rdv = kV + 2048 * (ct >> 1) + (4 * q4 + (ln >> 2)) * 64 + 2 * (8 * (ln & 3) + 4 * (ct & 1));
  const int rd = 16 * lane;                   // a lane's piece of a KiB of operands
  lds_cptr const stage0 = (lds_cptr)&stage[0][0];
  int so = 0;                                 // stage of the chunk at hand
  // State tile i: rows (key channels) 32*(i/2) + 8*q4 + 4*(i%2) + r, column vcol; rows beyond Dk and columns beyond Dv do not
  // exist in the caller's [Dk, Dv] state: they are zero and stay zero.
  const bool col_live = vcol < p.Dv;
  f32x4 S[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 32 * (i >> 1) + 8 * q4 + 4 * (i & 1) + r;
      S[i][r] = (p.s0 && col_live && row < p.Dk) ? p.s0[((int64_t)bh * p.Dk + row) * p.Dv + vcol] : 0.f;
    }
  }
  bf16x8 Sb[NM];   // the state as right operand, by channel group
  auto next_operand = [&](int from, int to, int par) {
#pragma unroll
    for (int m = from; m < to; ++m) {
      Sb[m] = pack_acc2(S[2 * m], S[2 * m + 1]);
      xs[par][ct][m][lane] = __builtin_bit_cast(u32x4, Sb[m]);
    }
  };
  next_operand(0, NM, 0);
  for (int i = 0; i < KSTAGES - 1; ++i) __syncthreads();

  // A link's operands are read during the link before it, each register as soon as its last product has been issued: a 16-byte
  // LDS read keeps a wavefront's port for 16 cycles and a chunk needs 25 of them (heads of 64: 16), which in front of their use, 34 with the
  // decays of all tiles read by every lane, was half of the link.
  bf16x8 ka[2][NM], mh[NS], ml[NS];
  u32x2 vr[2];
  // The decays of a lane's rows of all tiles are the same for 16 lanes.  With 8 tiles each lane reads those of one of them (8 heads of 128 of
  // 2 x 1000 rows 37.9 -> 37.4 us, 4 of 8192 181.5 -> 175.3), with 4 all of them (4 heads of 64 of 8192 rows 112.8 us, 114.4 with one).
  constexpr int DECS = KD == 128 ? 1 : NS;
  f32x4 dec[DECS];
  auto read_v = [&](lds_cptr sb) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) vr[mt] = lds_column4(sb + rdv + 16 * mt * 64);
  };
  auto read_ka = [&](lds_cptr sb, int m) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) ka[mt][m] = lds_bf16x8(sb + Blob::kKg + 1024 * (NM * mt + m) + rd);
  };
  auto read_dec = [&](lds_cptr sb, int set) {
    const int i = DECS == 1 ? ln & (NS - 1) : set;
    dec[set] = lds_f32x4(sb + Blob::kDec + 4 * (32 * (i >> 1) + 8 * q4 + 4 * (i & 1)));
  };
  auto read_ml = [&](lds_cptr sb, int i) { ml[i] = lds_bf16x8(sb + Blob::kMl + 1024 * i + rd); };
  auto read_mh = [&](lds_cptr sb, int i) { mh[i] = lds_bf16x8(sb + Blob::kMh + 1024 * i + rd); };
  read_v(stage0);
#pragma unroll
  for (int m = 0; m < NM; ++m) read_ka(stage0, m);
#pragma unroll
  for (int i = 0; i < DECS; ++i) read_dec(stage0, i);
#pragma unroll
  for (int i = 0; i < NS; ++i) { read_ml(stage0, i); read_mh(stage0, i); }
  __syncthreads();

  for (int n = 0; n < nc; ++n) {
    const int par = n & 1;
    so = so == (KSTAGES - 1) * kStage ? 0 : so + kStage;
    lds_cptr sb = stage0 + so;                // chunk n + 1 (behind the last one: what the stage holds, never used)

    // X = V + (-exp(G) K) S0, row tile mt: positions 16*mt + 4*q4 + r, column vcol
    f32x4 X[2];
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) X[mt] = f32x4{bf16lo_to_f32(vr[mt].x), bf16hi_to_f32(vr[mt].x), bf16lo_to_f32(vr[mt].y), bf16hi_to_f32(vr[mt].y)};
    read_v(sb);
    auto group = [&](auto which) {
      constexpr int m = decltype(which)::value;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) X[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ka[mt][m], Sb[m], X[mt], 0, 0, 0);
      read_ka(sb, m);
      decay_tiles<m * NS / NM, (m + 1) * NS / NM>(S, dec, [&](int i) {
        if (DECS > 1 || i == NS - 1) read_dec(sb, DECS > 1 ? i : 0);
      });
      __builtin_amdgcn_sched_barrier(0);
    };
    group(std::integral_constant<int, 0>{});
    group(std::integral_constant<int, 1>{});
    if constexpr (NM > 2) {
      group(std::integral_constant<int, 2>{});
      group(std::integral_constant<int, NM - 1>{});
    }
    // S = exp(G_last) (.) S + M X, both operands split into two bf16 terms; the tiles in two halves, so that the first
    // one's conversions run beside the second one's products
    const bf16x8 Xh = pack_acc2(X[0], X[1]);
    bf16x8 Xl;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      constexpr int HT = NS / 2;
#pragma unroll
      for (int i = half * HT; i < (half + 1) * HT; ++i) {
        S[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ml[i], Xh, S[i], 0, 0, 0);
        read_ml(sb, i);
      }
      if (half == 0) {
        Xl = pack_rest2(X[0], X[1], Xh);
        xx[par][ct][0][lane] = __builtin_bit_cast(u32x4, Xh);
        xx[par][ct][1][lane] = __builtin_bit_cast(u32x4, Xl);
      }
#pragma unroll
      for (int i = half * HT; i < (half + 1) * HT; ++i) S[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mh[i], Xh, S[i], 0, 0, 0);
#pragma unroll
      for (int i = half * HT; i < (half + 1) * HT; ++i) {
        S[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(mh[i], Xl, S[i], 0, 0, 0);
        read_mh(sb, i);
      }
      if (half == 1) next_operand(0, NM / 2, par ^ 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    next_operand(NM / 2, NM, par ^ 1);
    __syncthreads();
  }
  if (p.s_out != nullptr && col_live) {
    int row0 = 8 * q4;
    asm volatile("" : "+v"(row0));            // (the addresses are worked out here and not kept, spilled, across the loop)
#pragma unroll
    for (int i = 0; i < NS; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 32 * (i >> 1) + row0 + 4 * (i & 1) + r;
        if (row < p.Dk) p.s_out[((int64_t)bh * p.Dk + row) * p.Dv + vcol] = S[i][r];
      }
  }
}

// BY_LENGTH: packed sequences from the longest one on (a kernel of its own: with that code ahead of their loop other calls' chains are 1 to 2 % slower).
template <int KD, int KCT, bool BY_LENGTH>
__global__ __launch_bounds__(kStateThreads<KCT>, 1) void kda_state_kernel(KdaParams p) {
  __shared__ __attribute__((aligned(1024))) StageLds<KD, KCT> stage;
  __shared__ __attribute__((aligned(16))) StateLds<KD, KCT> xs;
  __shared__ __attribute__((aligned(16))) XLds<KCT> xx;
  kda_chain<KD, KCT, BY_LENGTH>(p, stage, xs, xx, [&](int& b, int& rows_end) { return seq_span<BY_LENGTH>(p, b, rows_end); });
}

// Up to kScanSeqs packed sequences in groups of 64 columns or of 32, as their lengths, which only the device knows, want it: 64 where the
// longest chain, whose links they lengthen, is no more than three quarters of the links of 32 that fall to a compute unit, each chain counted for four more that it
// takes to start, or three quarters of the 256th and 257th longest together, one of which has to wait for the other and then start (with up to one and a half rounds of chains, where that
// is more than the share, and where ranking them, 1 us, is worth it: 9 sequences, 16 heads of 64 x 64, T = 16000, equal, 288 chains of 32, 139 -> 117, T = 9000 67.2 -> 58.9, 12 of
// 14000, 8 heads of 128 114 -> 105; with it at 512 chains 16 of 3000, 16 heads of 64 x 64, at random 31.9 -> 34.1).  Columns come in whole groups of 64; the grid is that of 32.  us, 32 / 64 columns (that ratio), heads of 128: 16 sequences, 16 heads, T = 6000,
// equal (0.18) 91.9 / 82.5, the longest a fifth (0.57) 93.1 / 88.7, cut at random (0.78) 97.4 / 99.5, the longest two fifths (1.1) 95.6 / 120, nearly all (2.8) 149 / 204;
// T = 16000, cut at random (0.68) 238 / 228, 8 heads (1.4) 142 / 159; 33 sequences, T = 6000, at random (0.53) 114 / 95, the longest two fifths (0.89) 118 / 123, 8 heads,
// at random (1.0) 62 / 72, T = 16000 (0.64) 151 / 149.  Key heads of 64, of whose groups of 32 two workgroups fit a compute unit, of this kernel one (32 by their own
// kernel / 64 / this kernel): 16 sequences, 16 heads of 64 x 128, T = 16000, equal 147 / 126 / 127, the longest two fifths 177 / 199 / 177, nearly all 298 / 343 / 299; 12 heads, T = 9000, cut
// at random 65.8 / 72.5 / 66.7, a fourth 65.8 / 76.9 / 68.2; T = 3000, equal 30.3 / 29.3 / 29.9, a fourth 31.8 / 32.6 / 34.2.
template <int KD, bool BY_LENGTH>
__global__ __launch_bounds__(kStateThreads<4>, 1) void kda_packed_state_kernel(KdaParams p) {
  __shared__ __attribute__((aligned(1024))) StageLds<KD, 4> stage;
  __shared__ __attribute__((aligned(16))) StateLds<KD, 4> xs;
  __shared__ __attribute__((aligned(16))) XLds<4> xx;
  const SeqScan scan = packed_scan(p);
  int longest = scan.nc;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) longest = max(longest, __shfl_xor(longest, off));
  longest = __builtin_amdgcn_readfirstlane(longest);
  const int groups = p.H * (p.Dv / (2 * KVS));       // a sequence's chains of 32 columns
  int64_t share = (int64_t)(__builtin_amdgcn_readlane(scan.upto, 63) + 4 * p.n_seq) * groups;       // 256 times
  if (BY_LENGTH && p.n_seq * groups <= 384) {
    const int rank = length_rank(p, scan);
    share = max(share, (int64_t)256 * (4 + __builtin_amdgcn_readlane(scan.nc, sequence_ranked(p, rank, 255 / groups)) +
                                       __builtin_amdgcn_readlane(scan.nc, sequence_ranked(p, rank, 256 / groups))));
  }
  auto chain = [&](auto columns) {
    constexpr int KCT = decltype(columns)::value;
    if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= kStateThreads<KCT>) return;
    kda_chain<KD, KCT, BY_LENGTH>(p, reinterpret_cast<StageLds<KD, KCT>&>(stage), reinterpret_cast<StateLds<KD, KCT>&>(xs), reinterpret_cast<XLds<KCT>&>(xx),
                                  [&](int& b, int& rows_end) { return scanned_span<BY_LENGTH>(p, scan, b, false, rows_end); });
  };
  if (longest * (int64_t)(256 * 4) <= 3 * share) chain(std::integral_constant<int, 4>{});
  else chain(std::integral_constant<int, 2>{});
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

// Blocks of up to this many bytes are stored through the caches (the last level holds 256 MB), where the second kernel finds them.  Both
// kernels, past / through them: 21 MB (T = 8192, 4 heads of 64) 155 / 114 us, 81 MB (T = 6016, 12 heads of 128) 168 / 158, 126 MB (T = 8192,
// 24 heads of 64) 198 / 143; 296 MB (T = 8192, 32 heads of 128) 310 / 333.
// *Tried:* 170 MB, and up to 240 MB the first 128 of every sequence's: with the same inputs in every call 3 to 30 % faster, with others in every call,
// which pass through the same caches, 4 x 2048 rows, 16 heads of 128 124.6 -> 127.7, 10104 in 4 sequences, 12 heads 134.7 -> 138.5, 15500 in 6, 16 of 64 by 128
// 168 -> 176, against 2 x 7500, 8 heads of 128 260 -> 252.
constexpr int64_t kCachedBytes = (int64_t)128 << 20;

template <int KD>
static int kda_launch_width(const KdaParams& p, int n_streams, hipStream_t s) {
  const dim3 chunks((unsigned)p.NC * (unsigned)p.H, 1, p.n_seq > 0 ? 1 : p.B);
  const int64_t bytes = (int64_t)p.H * p.nc_total * KdaBlob<KD>::kBytes;
  if (bytes > kCachedBytes) {
    hipLaunchKernelGGL((kda_prep_kernel<KD, true>), chunks, dim3(128), 0, s, p);
  } else {
    hipLaunchKernelGGL((kda_prep_kernel<KD, false>), chunks, dim3(128), 0, s, p);
  }
  DAISY_CHECK_LAUNCH("kda_prep_kernel");
  // A chain fills a compute unit.  Groups of 64 value columns where they take fewer rounds of 256 than groups of 32: a link of 64 columns takes longer (0.8 us
  // against 0.57 with few chains, by its LDS reads), but one round of them less than two.  Chains of T = 4096, 32 / 64 columns, us: heads of 128, 256 groups of 32 167 /
  // 183, 320 206 / 140, 384 210 / 155, 512 228 / 187, T = 2048 1024 229 / 187; key heads of 64 256 114 / 125, 320 156 / 106, 512 172 / 128, 64 sequences of 64 rows 22 / 20.
  // Both kernels, T = 2048, where a dead half makes the rounds as many: 9 x 16 heads of 128 x 96 (432 / 288 groups) 242 / 270, 10 x 16 of 64 x 96 160 / 176; T = 1024, 6 x 16
  // of 128 x 160 (480 / 288) 93 / 107; as many or fewer: 11 x 16 of 128 x 96 (528 / 352) 314 / 299, 20 x 16 (960 / 640) level, 17 x 16 of 128 x 40 (544 / 272) 219 / 220.
  const int64_t streams = (int64_t)n_streams * p.H;
  const int narrow = (p.Dv + 2 * KVS - 1) / (2 * KVS), wide = (p.Dv + 4 * KVS - 1) / (4 * KVS);
  const unsigned chains = (unsigned)((streams + 7) / 8 * 8 * narrow);
  if (p.n_seq == 0) {
    if ((streams * wide + 255) / 256 < (streams * narrow + 255) / 256) {
      hipLaunchKernelGGL((kda_state_kernel<KD, 4, false>), dim3((unsigned)((streams + 7) / 8 * 8 * wide)), dim3(kStateThreads<4>), 0, s, p);
    } else {
      hipLaunchKernelGGL((kda_state_kernel<KD, 2, false>), dim3(chains), dim3(kStateThreads<2>), 0, s, p);
    }
  } else {
    // Where there are more than 256, a long sequence that starts late ends alone.  Longest first, cut at random places, both
    // kernels: 10 sequences of T = 4689, 16 heads of 128 102 -> 87 us, 7 of 3000, 12 heads 53 -> 44.4, 7 of 6164, 16 of 64 67.3 -> 56; 40 such batches 4 % on
    // average.  Where the longest one comes early anyway ranking costs (12 of 12000, 16 of 64 95.5 -> 97.3): 0.03 us a sequence in every workgroup, so
    // only up to a tenth of a mean chain (else 16 of T = 2088, 8 heads of 128 34.5 -> 35.5, 13 of 148, 12 heads 18.2 -> 19.8); not where they are in that order.
    const bool by_length = chains > 256 && p.n_seq > 1 && p.n_seq <= kScanSeqs && p.NC >= p.n_seq * p.n_seq;
    const bool either = p.n_seq <= kScanSeqs && streams * narrow > 256 && p.Dv % (4 * KVS) == 0;
    if (either && by_length) hipLaunchKernelGGL((kda_packed_state_kernel<KD, true>), dim3(chains), dim3(kStateThreads<4>), 0, s, p);
    else if (either) hipLaunchKernelGGL((kda_packed_state_kernel<KD, false>), dim3(chains), dim3(kStateThreads<4>), 0, s, p);
    else if (by_length) hipLaunchKernelGGL((kda_state_kernel<KD, 2, true>), dim3(chains), dim3(kStateThreads<2>), 0, s, p);
    else hipLaunchKernelGGL((kda_state_kernel<KD, 2, false>), dim3(chains), dim3(kStateThreads<2>), 0, s, p);
  }
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
  DAISY_CHECK_ARG((int64_t)slots * H <= 0x1ffffff && ((int64_t)(n_seq > 0 ? n_seq : B) * H + 7) * ((Dv + 2 * KVS - 1) / (2 * KVS)) <= 0x7fffffff,
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
