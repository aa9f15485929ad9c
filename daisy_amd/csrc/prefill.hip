// Kernel 1: sliding-window causal flash-attention prefill with fused RoPE (gfx950).
//
// Work decomposition
//   workgroup = 4 wavefronts = 128 consecutive query rows of one (batch, head);
//   wavefront = 32 query rows.  Key/value rows are visited in tiles of 32 rows, and
//   only tiles that intersect [lo(q_first), q_last] are loaded at all, where
//   lo(q) = max(q - window + 1, doc_start[q], 0) is non-decreasing in q.
//
// MFMA formulation (v_mfma_f32_32x32x16_bf16, wave64)
//   The kernel computes the TRANSPOSED products  S^T = K Q^T  and
//   O^T = V^T P^T.  In the 32x32 accumulator layout a lane owns one column, so
//   every lane owns one QUERY: lane l holds query (l % 32) and, per accumulator
//   register r, key row 8*(r/4) + 4*(l/32) + (r%4).  Row max / row sum are
//   therefore per-lane loops plus one exchange between lanes l and l^32, the
//   rescale of O^T is a per-lane scalar, and the accumulator registers of S^T,
//   converted to bf16, already ARE the B operand of the second product: the
//   contraction index of an MFMA may be enumerated in any order as long as the
//   A and B operands agree, so the V^T operand simply fetches, per lane, the key
//   rows 16m + 8g + 4*(l/32) + 0..3 that the lane's P registers hold.
//
// LDS (double buffered): K and V tiles [rows][D] bf16, row major, filled by direct
// global->LDS copies (global_load_lds_dwordx4: no staging registers, no LDS
// store instructions); the 16-byte chunks of each row are XOR-swizzled so that
// operand reads are bank-conflict free.  V^T operands come out of the row-major
// V tile through LDS transpose reads (ds_read_b64_tr_b16): inside a block of 16
// lanes, lane L receives element L%4 of the four 8-byte chunks addressed by
// lanes L/4, L/4+4, L/4+8, L/4+12; with lane i of a block addressing key i/4,
// channels 4*(i%4)..+3, lane i receives channel i of four consecutive keys.
//
// Keys reach the tile kernels rotated: by the caller, or by rope_k_kernel, a
// pre-pass that writes the rotated keys the reference's prefill returns anyway.
//
// Algorithmic work: 4*D flops per visible (query, key) pair.
#include "common.h"

#include <algorithm>
#include <cfloat>
#include <type_traits>

namespace daisy {

struct PrefillParams {
  const uint16_t* q; int64_t q_sb, q_st, q_sh;
  const uint16_t* k; int64_t k_sb, k_st, k_sh;
  const uint16_t* v; int64_t v_sb, v_st, v_sh;
  const float* cos; const float* sin;
  const int32_t* doc_start;
  uint16_t* o; int64_t o_sb, o_st, o_sh;
  uint16_t* k_out; int64_t ko_sb, ko_st, ko_sh;
  int B, T, H, D, window, nqb;
  int keys;      // key rows per tile
  int period;    // tiles in a full window's range (0 = no window): the rotation period of the tile order
  int n_light;   // leading query blocks that see fewer keys than a full window (0 = order by block only)
  int order_shift;   // documents: query blocks in the order of their lengths, in units of 2^order_shift tiles; -1: by block
  int order_bit;     // the highest bit of such a length
  int runs;          // prefill_split_kernel: neighbouring blocks to one XCD, else (batch, head) pairs in turn
  float scale_log2e;
};

constexpr int kBM = 128;  // query rows per workgroup
constexpr int kPrefillThreads = 256;

__device__ __forceinline__ int row_lo(const PrefillParams& p, int q) {
  int lo = (p.window > 0) ? max(q - p.window + 1, 0) : 0;
  if (p.doc_start != nullptr) lo = max(lo, p.doc_start[q]);
  return lo;
}

// With documents the length of a block depends on where its document starts, which only the device knows: item `idx` of a group of
// gsize (batch, head) pairs in the order of decreasing length, pair by pair from the last block down within a length.  Block by
// block from the end, the last workgroups of the grid were those of the first two documents, of any length (T = 20001, 16 heads
// of 64, window 4096, seven documents: 183 -> 161 us; T = 65536, 4 heads of 64, five documents: 520 -> 453 us).  One wavefront works it out: it holds the lengths of up to 512 blocks, and counts
// with ballots; any lengths give every block once.
constexpr int kOrderChunks = 8;
__device__ __forceinline__ void block_by_length(const PrefillParams& p, int gsize, int idx, int& local, int& qb, int& lo) {
  const int lane = threadIdx.x & 63;
  int len[kOrderChunks];     // 0..2 order_bit - 1, -1 past the last block
  int first[kOrderChunks];   // the first key of a block
#pragma unroll
  for (int c = 0; c < kOrderChunks; ++c) {
    len[c] = -1;
    if (64 * c < p.nqb) {
      const int i = 64 * c + lane, q0 = min(i, p.nqb - 1) * kBM;
      first[c] = row_lo(p, q0);
      const int n = min(q0 + kBM - 1, p.T - 1) / 32 - first[c] / 32 + 1;
      if (i < p.nqb) len[c] = min(max(n, 0) >> p.order_shift, 2 * p.order_bit - 1);
    }
  }
  auto at_least = [&](int v) {
    int n = 0;
#pragma unroll
    for (int c = 0; c < kOrderChunks; ++c)
      if (64 * c < p.nqb) n += __popcll(__ballot(len[c] >= v));
    return n;
  };
  int v = 0;                 // the largest length with more than idx items at least as long
  for (int bit = p.order_bit; bit > 0; bit >>= 1)
    if (gsize * at_least(v + bit) > idx) v += bit;
  const int above = at_least(v + 1), here = at_least(v) - above, k = idx - gsize * above;
  local = k / here;
  int j = here - 1 - k % here;      // which of the blocks of this length, counted from the first
  qb = lo = 0;
#pragma unroll
  for (int c = 0; c < kOrderChunks; ++c) {
    if (64 * c >= p.nqb) break;
    const uint64_t same = __ballot(len[c] == v);
    const int n = __popcll(same);
    if (j >= 0 && j < n) {
      const bool mine = (same >> lane & 1) != 0 && __popcll(same & ((1ull << lane) - 1)) == j;
      const int at = __ffsll((unsigned long long)__ballot(mine)) - 1;
      qb = 64 * c + at;
      lo = __builtin_amdgcn_readlane(first[c], at);
    }
    j -= n;
  }
  local = __builtin_amdgcn_readfirstlane(local);
  qb = __builtin_amdgcn_readfirstlane(qb);
  lo = __builtin_amdgcn_readfirstlane(lo);
}

// Workgroup -> (batch*head, query block).  Workgroups are dealt round-robin to the 8 XCDs, each
// with its own L2: an XCD is given a contiguous group of (batch, head) pairs, or of blocks, so that the query
// blocks sharing K/V rows share an L2.  Inside a group the blocks with a full window of keys
// come first, pair by pair from the last block down; the n_light shorter blocks at the start of
// every sequence come last, longest first across the whole group, and fill the tail of the grid.
__device__ __forceinline__ void workgroup_to_block(const PrefillParams& p, int* found, int& bh, int& qb, int& lo) {
  const int nbh = p.B * p.H;
  int group = 0, gsize = nbh, idx = blockIdx.x;
  if ((nbh & 7) == 0) { group = blockIdx.x & 7; gsize = nbh >> 3; idx = blockIdx.x >> 3; }
  const int n_full = p.nqb - p.n_light;
  int local;
  // Pairs that are no multiple of eight: an XCD takes a run of neighbouring blocks with a full window (the shorter ones fill the tail as they come).  Dealt to
  // the XCDs one by one, every L2 fetched every key: 3 x 5000 rows, 12 heads of 128, window 800 98.9 -> 80.7 us; 16384 rows, 12 heads, 1024 127.8 -> 118.8,
  // 4096 335 -> 332; 60000 rows, 4 heads, 1427 196.7 -> 185.9; heads of 64, 30000 rows, 12 heads, 1000 126.4 -> 115.1, but 20000 rows, 4 heads, 4096 95.1 / 96.6.
  // Of documents under a short window each XCD takes an eighth of every pair's full-window blocks, of each pair another one, because documents make parts of a
  // row cheap: 16384 rows, 12 heads, window 1024, six documents / one 121.9 / 125.9 -> 106.1 / 108.0 us, half the row in documents of 200 96.1 -> 82.6; 20000 rows, 10
  // heads, 2000 186.7 / 196.4 -> 178.1 / 192.1; 30000 rows, 4 heads, 1000 98.6 / 99.0 -> 79.7 / 75.5; heads of 64, 60000 rows, 4 heads, 1024 89.5 / 94.1 -> 77.8 / 81.9.
  // (Runs of an eighth of all blocks: 30000 rows, 4 heads, 2000, half in short ones 84.9 -> 111.9.)  Fewer pairs cannot make up for a cheap part (4 heads, 3072
  // 169.9 -> 193.1; two, 1000 61.9 -> 73.6), nor can blocks that all run at once (7 heads, 14200 rows, 1500 63.5 -> 70.7; 5, 9000, 1000 42.7 -> 45.2;
  // three fit a compute unit, four of heads of 64).
  if ((nbh & 7) != 0 && p.period > 0 && p.doc_start == nullptr && p.window < 64 * p.D) {
    const int runs = (nbh * n_full) & ~7;
    if (idx < runs) idx = (idx & 7) * (runs >> 3) + (idx >> 3);
  } else if ((nbh & 7) != 0 && nbh >= 4 && p.period > 0 && p.doc_start != nullptr && p.order_shift < 0 && p.window <= (nbh >= 8 ? 2048 : 1024) && nbh * p.nqb > (p.D == 64 ? 1024 : 768)) {
    const int m = n_full >> 3, rest = n_full & 7, runs = nbh * m * 8;
    if (idx < runs) {
      const int pair = (idx >> 3) / m, turn = (pair & 1) * 4 + (pair & 2) + (pair >> 2 & 1);
      idx = pair * n_full + ((idx + turn) & 7) * m + (idx >> 3) % m;
    } else if (idx < nbh * n_full) {
      idx -= runs;
      idx = idx / rest * n_full + 8 * m + idx % rest;
    }
  }
  // (a lone document, which the last row's bound shows, leaves a window's blocks equally long: T = 16384, window 2048, 8 heads of
  // 128: 145.2 us by length, 142.6 us without, as without documents; one scalar load, which several documents do not feel)
  const bool by_length = p.order_shift >= 0 && (p.n_light == 0 || p.doc_start[p.T - 1] > 0);
  if (by_length) {
    if (threadIdx.x < 64) {      // (a load per block touches a cache line each: one wavefront's are enough)
      block_by_length(p, gsize, idx, local, qb, lo);
      if (threadIdx.x == 0) { found[0] = local; found[1] = qb; found[2] = lo; }
    }
    __syncthreads();
    local = __builtin_amdgcn_readfirstlane(found[0]);
    qb = __builtin_amdgcn_readfirstlane(found[1]);
    lo = __builtin_amdgcn_readfirstlane(found[2]);
  } else if (idx < gsize * n_full) {
    local = idx / n_full;
    qb = p.nqb - 1 - idx % n_full;
  } else {
    const int j = idx - gsize * n_full;
    qb = p.n_light - 1 - j / gsize;
    local = j % gsize;
  }
  if (!by_length) lo = row_lo(p, qb * kBM);
  bh = group * gsize + local;
}

// Exchange with the lane that holds the other half of this query's keys.
__device__ __forceinline__ float pair_max(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
  return fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
  return __int_as_float(r[0]) + __int_as_float(r[1]);
}

// Online softmax of a tile (log2 domain): its probabilities as operands, against the wavefront's reference maxima, which move only
// when some query's share of the tile's sum exceeds kMost.  Until then no probability does, which bf16 and the fp32 sums hold
// without loss, and neither the tile's maxima are looked for nor is O touched: the scores' exponentials come straight behind their
// products.  A query that has seen no key has -FLT_MAX for a reference: what it does not see stays 0, its first key overflows the sum and sets it.  (Behind
// a document's start the queries of a wavefront wait through every tile of the document ahead.  While any of them did, each tile took the long way: 20000
// rows in seven documents, 4 heads of 128 172 us, 24545 in twenty, 8 heads 211, 5900 in three, 16 of 64 52.4; now 149, 186 and 49.8, with the maxima of every tile
// 147, 185 and 49.2.)
// kFirst: a wavefront's first tile takes the long way at once, so that short rows do not work out its exponentials twice; the branch costs the tile
// kernel for heads of 128 more where it is bound by latency, two or three blocks to a compute unit, so there it is kSums: 9000 rows, 8 heads 202.5 us with the
// maxima of every tile, 208.7 with the branch, 203.8 without; 20000 in documents that start with a block, 4 heads 113.5, 115.8, 114.6.  (Heads of 64 need it: 128
// registers do not hold both ends of the block that the products and the exponentials then share.)
// kMaxima: the maxima of every tile ahead of its exponentials, a reference moves at 2^8.  For windows of a few tiles, most of which are some query's first or last:
// sums / maxima, us, heads of 128: 8 x 4096 rows, window 100 / 256 / 383 / 450 15.0 / 14.2, 17.1 / 16.2, 19.2 / 18.4, 20.7 / 20.1, 16 x 30000 102 / 100, 121 / 119, 146.8 / 146.6, 163.6 /
// 165.3; heads of 64: 12 x 2 x 8192, 100 / 200 / 300 26.5 / 24.8, 29.1 / 28.1, 31.8 / 31.9, 16 x 30000 57.3 / 56.6, 63.8 / 64.0, 71.5 / 73.5.
// The tile kernels are bound by their vector instructions (head dim 64: 855 cycles of them per 64 keys against 512 of the matrix pipe) and by power, which fewer of
// them spare: with the maxima of every tile worked out and compared (a reference moved at 2^8) 65536 rows, 16 heads of 128, full causal took 15.00 ms, now
// 14.56; 20001 rows in seven documents, 16 heads of 64, 178.6 us, now 171.4; a layer of 8 x 4096 rows, 8 heads of 128, window 1024, 406.2 and 403.8.
struct SoftmaxRef {
  float minus = FLT_MAX;   // less the reference (scaled), the same in both lanes of a query: what is added to the scaled scores
  float l = 0.f;           // this lane's share of the running sum
  bool first = true;       // the wavefront has seen no tile
};
constexpr float kMost = 4096.f;
enum SoftmaxMode { kSums, kFirst, kMaxima };
template <SoftmaxMode MODE, int SUB, int NDT>
__device__ __forceinline__ void softmax_tile(const f32x16 (&sacc)[SUB], float scale_log2e, SoftmaxRef& ref, f32x16 (&oacc)[NDT],
                                             bf16x8 (&pfrag)[2 * SUB]) {
  float lsum;
  auto exponentials = [&]() {
    lsum = 0.f;
#pragma unroll
    for (int m = 0; m < 2 * SUB; ++m) {
      float pv[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        pv[e] = fast_exp2(fmaf(sacc[m >> 1][8 * (m & 1) + e], scale_log2e, ref.minus));
        lsum += pv[e];
      }
      pfrag[m] = __builtin_bit_cast(bf16x8, pack8(pv));
    }
  };
  bool moves = MODE == kMaxima || (MODE == kFirst && ref.first);
  if (!moves) {
    exponentials();
    moves = __builtin_amdgcn_ballot_w64(lsum > kMost) != 0;
  }
  if (moves) {
    ref.first = false;
    float mt = -INFINITY;
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) mt = fmaxf(mt, sacc[u][r]);
    mt = pair_max(mt) * scale_log2e;
    if (MODE != kMaxima || __builtin_amdgcn_ballot_w64(mt > 8.f - ref.minus) != 0) {
      const float minus = fminf(ref.minus, -mt), alpha = fast_exp2(minus - ref.minus);
      ref.minus = minus;
      ref.l *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[dt][r] *= alpha;
    }
    exponentials();
  }
  ref.l += lsum;
}

// LDS transpose read (ds_read_b64_tr_b16); semantics in the header comment.
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) const uint16_t* lds_u16_ptr;
__device__ __forceinline__ u32x2 lds_read_tr16_as3(lds_u16_ptr p) {
  s16x4 v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)p);
  return __builtin_bit_cast(u32x2, v);
}

// Main kernel (keys already rotated, or no RoPE on keys).  32-key tiles, and nothing of a step is
// overlapped inside a wavefront: scores, softmax and the product of one tile follow each other.  The
// kernel is small instead -- 167 VGPRs and 48 KiB of LDS at D = 128 -- so that THREE workgroups fit a
// CU, three wavefronts a SIMD, and the latencies of one wavefront's step (the issue of its tile
// copies, the LDS operand reads, the softmax chain, the barrier) are covered by the other two: matrix
// instructions of one wavefront and vector instructions of another do run side by side on a SIMD.
//   step n:  copies K(n+1), V(n+1) -> the other buffer;  S = K(n) Q^T;  P = softmax(S);  O += V(n)^T P;
//            wait for the copies, barrier.
// A wavefront computes only the tiles its 32 queries can see; a tile at the window / document edge or
// on the diagonal is masked per element.  The Q block at the start and the O block at the end pass
// through an LDS area of the wavefront's own, so that every global access of the kernel covers whole
// rows (a CU's memory path, shared by its three workgroups, is busy per cache line touched).
//
// KEYS = 64 (prefill_wide_tile_kernel, head dim 64): a tile is two products side by side, with one maximum, one check of the reference and
// one barrier for both (128 registers and 32 KiB, still four workgroups per CU: the Q and O blocks fit Ks[1] and Vs[1]).
constexpr int kTBN = 32;   // key rows of a product
template <int D, int KEYS, SoftmaxMode MODE>
__device__ __forceinline__ void prefill_tiles(const PrefillParams& p) {
  constexpr int NS = D / 16, NDT = D / 32, HALF = D / 2, CPR = D / 8;
  constexpr int SUB = KEYS / kTBN;               // products of a tile
  static_assert(SUB == 1 || (SUB == 2 && D == 64), "");
  constexpr int RPL = 64 / CPR, NLD = KEYS / RPL / 4, TILE = KEYS * D;
  static_assert(NLD >= 1, "a tile is at least one copy per wavefront");
  auto swz_k = [](int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); };
  auto swz_v = [](int r) { return D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1); };

  __shared__ __attribute__((aligned(1024))) uint16_t Ks[2][TILE];
  __shared__ __attribute__((aligned(1024))) uint16_t Vs[2][TILE];
  // Two more tile-sized areas: with Ks[1] and Vs[1] they give every wavefront 32 rows x D of its own for
  // turning the row-major Q block into operand fragments at the start (while the first K/V tile lands in
  // Ks[0] / Vs[0]) and the accumulators into row-major O at the end.
  __shared__ __attribute__((aligned(1024))) uint16_t Xs[SUB == 1 ? 2 : 1][SUB == 1 ? TILE : 1];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, lh = lane >> 5;

  int bh, qb, lo_first;
  __shared__ int found[3];
  workgroup_to_block(p, found, bh, qb, lo_first);
  const int h = bh % p.H, b = bh / p.H;

  const int q0 = qb * kBM;
  const int qw0 = q0 + wave * 32;
  const int qrow = min(qw0 + lq, p.T - 1);
  const int lo_q = row_lo(p, qrow);
  const int lo_w_min = __builtin_amdgcn_readlane(lo_q, 0);
  const int lo_w_max = __builtin_amdgcn_readlane(lo_q, 31);
  const int q_w_min = min(qw0, p.T - 1), q_w_max = min(qw0 + 31, p.T - 1);
  const bool wave_live = qw0 < p.T;

  // Tiles are visited in rotated order: start at the tile whose index is a multiple of the
  // window's tile count (one exists in every full range), run up to t_hi, wrap to t_lo.  The
  // online softmax does not care about the order, and the query blocks of one (batch, head)
  // that run side by side then read the same K/V tile at the same step, so one fetch into the
  // L2 serves all of them.  With no window every range starts at tile 0 and nothing is rotated.
  const int t_lo = lo_first / KEYS;
  const int t_hi = min(q0 + kBM - 1, p.T - 1) / KEYS;
  const int n_tiles = t_hi - t_lo + 1;
  int t_first = t_lo;
  if (p.period > 0) {
    const int c = (t_lo + p.period - 1) / p.period * p.period;
    if (c <= t_hi) t_first = c;
  }

  const uint16_t* kbase = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t* vbase = p.v + b * p.v_sb + h * p.v_sh;

  // ---- global -> LDS copies ------------------------------------------------------------------
  // Wavefront copy j of a tile moves rows RPL*j .. RPL*j+RPL-1 (1 KiB); lane i lands at chunk
  // position i % CPR of row i / CPR, so it fetches the chunk that belongs there (the swizzle is
  // applied on the global side).  This wavefront issues the copies wave, wave + 4, ...: their rows
  // are 16 apart, the swizzles of such rows coincide, so one per-lane offset serves all of them and
  // the row step goes into the wavefront-uniform base.
  const int ld_row = lane / CPR, ld_pos = lane % CPR;
  const int r0 = RPL * wave + ld_row;
  const int k_off = 2 * (r0 * (int)p.k_st + 8 * (ld_pos ^ swz_k(r0)));   // bytes
  const int v_off = 2 * (r0 * (int)p.v_st + 8 * (ld_pos ^ swz_v(r0)));
  const uint32_t ks_lds = lds_address(&Ks[0][0]) + 1024 * wave, vs_lds = lds_address(&Vs[0][0]) + 1024 * wave;
  // The copies walk the tiles in visiting order; the source pointers move by one tile per step and go
  // back to the first tile of the range once (kept incrementally: the scalar unit would otherwise
  // rebuild two 64-bit products per step).
  const int64_t k_step = (int64_t)KEYS * p.k_st, v_step = (int64_t)KEYS * p.v_st;
  const uint16_t* const k_lo = kbase + t_lo * k_step;
  const uint16_t* const v_lo = vbase + t_lo * v_step;
  int t_cp = t_first;                                   // tile the next copy_tiles() call fetches
  const uint16_t* kt = kbase + t_first * k_step;
  const uint16_t* vt = vbase + t_first * v_step;
  auto copy_tiles = [&](int buf) {
    const int kv0 = t_cp * KEYS;
    if (kv0 + KEYS <= p.T) {
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        copy16_to_lds_async(kt + (int64_t)(4 * RPL * i) * p.k_st, k_off, ks_lds + 2 * (buf * TILE) + 4096 * i);
        copy16_to_lds_async(vt + (int64_t)(4 * RPL * i) * p.v_st, v_off, vs_lds + 2 * (buf * TILE) + 4096 * i);
      }
    } else {
      // The tile reaches past the last row: clamp (the surplus rows are masked by causality).
#pragma unroll
      for (int i = 0; i < NLD; ++i) {
        const int r = r0 + 4 * RPL * i;
        const int row = min(r, p.T - 1 - kv0);
        copy16_to_lds_async(kt, 2 * (row * (int)p.k_st + 8 * (ld_pos ^ swz_k(r))), ks_lds + 2 * (buf * TILE) + 4096 * i);
        copy16_to_lds_async(vt, 2 * (row * (int)p.v_st + 8 * (ld_pos ^ swz_v(r))), vs_lds + 2 * (buf * TILE) + 4096 * i);
      }
    }
    if (++t_cp > t_hi) { t_cp = t_lo; kt = k_lo; vt = v_lo; }
    else { kt += k_step; vt += v_step; }
  };
  auto copies_landed = [&]() {
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0), visible to the compiler's wait-count model
    asm volatile("" ::: "memory");
  };
  // The first tile goes out before anything else so that its latency overlaps the Q loads.
  copy_tiles(0);
  int t_cur = t_first;                                  // tile the next iteration works on

  // ---- Q fragments (B operand), RoPE fused -------------------------------------------------------
  // Global loads with whole rows per group of lanes (lane -> row lane / CH, pair chunk lane % CH: the
  // 16 bytes at channel 8 ch and the 16 bytes at HALF + 8 ch, with the matching 32 bytes of the cos and
  // sin rows), rotated in that layout, written to this wavefront's own LDS area in the K tile layout
  // and read back as fragments.  Fetching the fragments straight from global memory would touch 32
  // rows with every instruction (32 bytes of each), and the CU's memory path, which the other
  // workgroups' tile copies share, would be busy four times as long.
  constexpr int CH = HALF / 8;          // pair chunks per row
  constexpr int QRI = 64 / CH;          // rows per load instruction
  constexpr int QT = 32 / QRI;          // loads of each kind per lane
  const uint32_t x_lds = SUB > 1 ? lds_address(wave < 2 ? &Ks[1][0] : &Vs[1][0]) + 2 * kTBN * D * (wave & 1)
                         : wave == 0 ? lds_address(&Ks[1][0]) : wave == 1 ? lds_address(&Vs[1][0]) : lds_address(&Xs[SUB > 1 ? 0 : wave - 2][0]);
  bf16x8 qreg[NS];
  {
    const int qr = lane / CH, qc = lane % CH;
    u32x4 x1[QT], x2[QT];
#pragma unroll
    for (int j = 0; j < QT; ++j) {
      const int row = min(qw0 + QRI * j + qr, p.T - 1);
      const uint16_t* qptr = p.q + b * p.q_sb + (int64_t)row * p.q_st + h * p.q_sh + 8 * qc;
      x1[j] = *reinterpret_cast<const u32x4*>(qptr);
      x2[j] = *reinterpret_cast<const u32x4*>(qptr + HALF);
    }
    if (p.cos != nullptr) {
#pragma unroll
      for (int j = 0; j < QT; ++j) {
        const int row = min(qw0 + QRI * j + qr, p.T - 1);
        const float* cr = p.cos + (int64_t)row * HALF + 8 * qc;
        const float* sr = p.sin + (int64_t)row * HALF + 8 * qc;
        float a1[8], a2[8], y1[8], y2[8];
        unpack8(x1[j], a1);
        unpack8(x2[j], a2);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float c = cr[e], sn = sr[e];
          y1[e] = rope_lo(a1[e], a2[e], c, sn);
          y2[e] = rope_hi(a1[e], a2[e], c, sn);
        }
        x1[j] = pack8(y1);
        x2[j] = pack8(y2);
      }
    }
#pragma unroll
    for (int j = 0; j < QT; ++j) {
      const int r = QRI * j + qr;
      *(u32x4 __attribute__((address_space(3)))*)(size_t)(x_lds + 2 * (r * D + 8 * (qc ^ swz_k(r)))) = x1[j];
      *(u32x4 __attribute__((address_space(3)))*)(size_t)(x_lds + 2 * (r * D + 8 * ((CH + qc) ^ swz_k(r)))) = x2[j];
    }
    const uint32_t q_a0 = x_lds + 2 * (lq * D + 8 * (lh ^ swz_k(lq)));
#pragma unroll
    for (int s = 0; s < NS; ++s)
      qreg[s] = __builtin_bit_cast(bf16x8, *(const u32x4 __attribute__((address_space(3)))*)(size_t)(q_a0 ^ (32u * s)));
  }

  // Operand addresses inside a tile (LDS byte addresses of buffer 0).  The swizzles are XORs on the
  // chunk index, so the K fragment of contraction slice s sits at k_a0 ^ (32 s) and the V fragment of
  // output tile dt at v_a0 ^ (64 dt): one register each instead of one per fragment.
  //   K (A operand of S^T): row = key lq, slice s wants chunk (2s + lh) ^ swz_k(lq).
  //   V (A operand of O^T, LDS transpose read): the lane's block of 16 covers output channels
  //   32dt + 16*(block & 1) + 0..15 and keys 4*lh + 0..3 (+8, +16 as immediates); lane i of the
  //   block addresses key i/4, channels 4*(i%4)..+3 and receives channel i, four keys.
  const uint32_t k_a0 = lds_address(&Ks[0][0]) + 2 * (lq * D + 8 * (lh ^ swz_k(lq)));
  uint32_t v_a0;
  {
    const int i16 = lane & 15, vrow = 4 * lh + (i16 >> 2);
    const int chunk = 2 * ((lane >> 4) & 1) + ((i16 & 3) >> 1);
    v_a0 = lds_address(&Vs[0][0]) + 2 * (vrow * D + 8 * (chunk ^ swz_v(vrow)) + 4 * (i16 & 1));
  }

  f32x16 oacc[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
  SoftmaxRef ref;

  // One tile of 32 keys.  There is ONE code path for clean and masked tiles (the mask is a small
  // conditional region): two instantiations of the products would make the compiler keep a second
  // copy of the accumulators across the join.
  auto process_tile = [&](auto buf_tag, int kv0, bool masked) {
    constexpr int buf = decltype(buf_tag)::value;
    f32x16 sacc[SUB];
#pragma unroll
    for (int u = 0; u < SUB; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) sacc[u][r] = 0.f;
    // K fragments: four reads ahead of the products (an LDS read takes about as long as four MFMAs;
    // left alone the compiler keeps one fragment register set and waits for every read in turn).
    {
      constexpr int N = NS * SUB;
      bf16x8 kf[N];
#pragma unroll
      for (int s = 0; s < N; ++s)
        kf[s] = __builtin_bit_cast(bf16x8, *(const u32x4 __attribute__((address_space(3)))*)(size_t)((k_a0 ^ (32u * (s / SUB))) + 2 * (buf * TILE + s % SUB * kTBN * D)));
#pragma unroll
      for (int s = 0; s < N; ++s) sacc[s % SUB] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qreg[s / SUB], sacc[s % SUB], 0, 0, 0);
      constexpr int AHEAD = N < 4 ? N : 4;
      __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);          // DS reads
#pragma unroll
      for (int s = 0; s < N - AHEAD; ++s) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);            // MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
    }
    if (masked) {
      // element r of this lane is key kv0 + 4lh + c_r with c_r = 8*(r/4) + r%4; visible iff lo <= c_r <= hi
      const int hi = qrow - (kv0 + 4 * lh);
      const int lo = lo_q - (kv0 + 4 * lh);
#pragma unroll
      for (int u = 0; u < SUB; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int c = kTBN * u + 8 * (r >> 2) + (r & 3);
          if (c > hi || c < lo) sacc[u][r] = -INFINITY;
        }
    }
    bf16x8 pfrag[2 * SUB];
    auto v_frag = [&](int m, int dt) {
      lds_u16_ptr vp = (lds_u16_ptr)(size_t)((v_a0 ^ (64u * dt)) + 2 * (buf * TILE + 16 * m * D));
      const u32x2 a0 = lds_read_tr16_as3(vp);            // keys 16m + 4lh + 0..3
      const u32x2 a1 = lds_read_tr16_as3(vp + 8 * D);    // keys 16m + 8 + 4lh + 0..3
      return u32x4{a0.x, a0.y, a1.x, a1.y};
    };
    // The first V fragments are asked for ahead of the exponentials: behind the branch at their end, where the reads of all but those stand, each tile
    // waits for the first one, which shows where a SIMD has one or two wavefronts.  As many as the registers hold (167 and 128).  us, none / these: 9000 rows, 8
    // heads of 128, no window 205.9 / 201.8, 5900 x 12 in documents that start with a block 99.3 / 97.2, x 16 of 64 in three 50.4 / 49.8.
    constexpr int EARLY = MODE == kMaxima ? 0 : D == 128 ? 2 : 1;
    u32x4 early[EARLY + 1];
#pragma unroll
    for (int i = 0; i < EARLY; ++i) early[i] = v_frag(0, i);
    softmax_tile<MODE, SUB, NDT>(sacc, p.scale_log2e, ref, oacc, pfrag);
    // O^T += V^T P^T
#pragma unroll
    for (int m = 0; m < 2 * SUB; ++m) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        const u32x4 av = m == 0 && dt < EARLY ? early[dt] : v_frag(m, dt);
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av), pfrag[m], oacc[dt], 0, 0, 0);
      }
    }
  };

  using Buf0 = std::integral_constant<int, 0>;
  using Buf1 = std::integral_constant<int, 1>;
  copies_landed();
  __syncthreads();
  auto iteration = [&](int n, auto buf_tag) {
    constexpr int buf = decltype(buf_tag)::value;
    if (n + 1 < n_tiles) copy_tiles(buf ^ 1);
    const int kv0 = t_cur * KEYS;
    t_cur = t_cur < t_hi ? t_cur + 1 : t_lo;
    if (wave_live && kv0 <= q_w_max && kv0 + KEYS - 1 >= lo_w_min) {
      const bool clean = kv0 + KEYS - 1 <= q_w_min && kv0 >= lo_w_max;
      process_tile(buf_tag, kv0, !clean);
    }
    copies_landed();
    __syncthreads();
  };
  for (int n = 0; n < n_tiles; n += 2) {
    iteration(n, Buf0{});
    if (n + 1 < n_tiles) iteration(n + 1, Buf1{});
  }

  // Epilogue: normalise, turn the accumulators (a lane holds four channels of one query per register
  // group) into row-major bf16 through this wavefront's LDS area, and store 16 bytes per lane with whole
  // rows per group of lanes.  The tile buffers are free: the loop ends with a barrier.
  const float l_tot = pair_sum(ref.l);
  const float inv = 1.f / l_tot;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      u32x2 w;
      w.x = pack_bf16x2(oacc[dt][4 * g + 0] * inv, oacc[dt][4 * g + 1] * inv);
      w.y = pack_bf16x2(oacc[dt][4 * g + 2] * inv, oacc[dt][4 * g + 3] * inv);
      // channels 32 dt + 8 g + 4 lh + 0..3 of query lq: chunk 4 dt + g, half lh
      *(u32x2 __attribute__((address_space(3)))*)(size_t)(x_lds + 2 * (lq * D + 8 * ((4 * dt + g) ^ swz_k(lq)) + 4 * lh)) = w;
    }
  }
  uint16_t* obase = p.o + b * p.o_sb + h * p.o_sh + 8 * ld_pos;
#pragma unroll
  for (int i = 0; i < 32 / RPL; ++i) {
    const int r = RPL * i + ld_row;
    const u32x4 w = *(const u32x4 __attribute__((address_space(3)))*)(size_t)(x_lds + 2 * (r * D + 8 * (ld_pos ^ swz_k(r))));
    // whole rows, written once and not read again by this kernel: streaming stores leave the last-level
    // cache to q, k and v (the same store from the accumulator layout, 16 bytes per row, must not be
    // streaming: such partial lines are then no longer merged on their way out)
    if (qw0 + r < p.T) __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(obase + (int64_t)(qw0 + r) * p.o_st));
  }
}

template <int D>
__global__ __launch_bounds__(kPrefillThreads, 3) void prefill_tile_kernel(PrefillParams p) { prefill_tiles<D, kTBN, D == 64 ? kFirst : kSums>(p); }
template <int D>
__global__ __launch_bounds__(kPrefillThreads, 3) void prefill_short_window_kernel(PrefillParams p) { prefill_tiles<D, kTBN, kMaxima>(p); }
__global__ __launch_bounds__(kPrefillThreads, 4) void prefill_wide_tile_kernel(PrefillParams p) { prefill_tiles<64, 2 * kTBN, kFirst>(p); }

// Few workgroups (a prompt of one or two thousand tokens of one sequence): blocks of 128 queries leave most compute
// units idle and the last block walks all of its keys with one step in flight.  Here a workgroup is 32 queries, its
// W wavefronts (four, or eight: eight_wavefronts) take every W-th key tile each -- tiles of their own, copied into LDS areas of their own, no
// barrier in the loop -- and the partial results (maximum, sum, O^T) meet in LDS at the end.  K(n+1) is copied
// while the softmax and the second product of tile n run, V(n+1) while the scores of tile n+1 do (in-order vmcnt:
// at most one tensor's copies stay outstanding).  A tile is fetched once per 32 queries instead of once per 128, so
// long grids are better off with prefill_tile_kernel (the rule stands at launch_mfma).
template <int D, int W>
__global__ __launch_bounds__(64 * W, W == 4 ? 2 : W / 4) void prefill_split_kernel(PrefillParams p) {
  constexpr int NS = D / 16, NDT = D / 32, HALF = D / 2, CPR = D / 8;
  constexpr int RPL = 64 / CPR, NCP = kTBN / RPL, TILE = kTBN * D;    // NCP copies of 1 KiB per tile
  auto swz_k = [](int r) { return D == 128 ? (r & 15) : ((r >> 1) & 7); };
  auto swz_v = [](int r) { return D == 128 ? 4 * (r & 3) : 4 * ((r >> 1) & 1); };
  __shared__ __attribute__((aligned(1024))) uint16_t tiles[W][2][TILE];   // [wavefront][K, V]; the fp32 partial O at the end
  __shared__ float part_m[W][32], part_l[W][32];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lq = lane & 31, lh = lane >> 5;

  // (batch, head) pairs in contiguous groups per XCD; inside a pair the block with the most keys first
  const int nbh = p.B * p.H, nqb = (p.T + 31) >> 5;
  int bh, qb;
  if ((nbh & 7) == 0) {
    const int g = nbh >> 3, idx = blockIdx.x >> 3;
    bh = (blockIdx.x & 7) * g + idx % g;
    qb = nqb - 1 - idx / g;
  } else if (p.runs) {               // an XCD takes a run of neighbouring blocks
    const int runs = (nbh * nqb) & ~7, i = blockIdx.x, at = i < runs ? (i & 7) * (runs >> 3) + (i >> 3) : i;
    bh = at / nqb;
    qb = nqb - 1 - at % nqb;
  } else {
    bh = blockIdx.x % nbh;
    qb = nqb - 1 - blockIdx.x / nbh;
  }
  const int h = bh % p.H, b = bh / p.H;
  const int q0 = qb * 32;
  const int qrow = min(q0 + lq, p.T - 1);
  const int lo_q = row_lo(p, qrow);
  const int lo_min = __builtin_amdgcn_readlane(lo_q, 0), lo_max = __builtin_amdgcn_readlane(lo_q, 31);
  const int q_max = min(q0 + 31, p.T - 1);
  const int t_lo = lo_min / kTBN, t_hi = q_max / kTBN;

  const uint16_t* kbase = p.k + b * p.k_sb + h * p.k_sh;
  const uint16_t* vbase = p.v + b * p.v_sb + h * p.v_sh;
  const int ld_row = lane / CPR, ld_pos = lane % CPR;
  const uint32_t k_lds = lds_address(&tiles[wave][0][0]), v_lds = lds_address(&tiles[wave][1][0]);
  // copy j moves rows RPL * j .. of a tile; rows past the sequence re-read its last row (masked by causality)
  auto copy_k = [&](int t) {
    const int kv0 = t * kTBN;
    const uint16_t* src = kbase + (int64_t)kv0 * p.k_st;
#pragma unroll
    for (int j = 0; j < NCP; ++j) {
      const int r = RPL * j + ld_row;
      copy16_to_lds_async(src, 2 * (min(r, p.T - 1 - kv0) * (int)p.k_st + 8 * (ld_pos ^ swz_k(r))), k_lds + 1024 * j);
    }
  };
  auto copy_v = [&](int t) {
    const int kv0 = t * kTBN;
    const uint16_t* src = vbase + (int64_t)kv0 * p.v_st;
#pragma unroll
    for (int j = 0; j < NCP; ++j) {
      const int r = RPL * j + ld_row;
      copy16_to_lds_async(src, 2 * (min(r, p.T - 1 - kv0) * (int)p.v_st + 8 * (ld_pos ^ swz_v(r))), v_lds + 1024 * j);
    }
  };
  int t = t_lo + wave;
  const bool any = t <= t_hi;

  // ---- Q fragments: whole rows from global memory, rotated, through this wavefront's V area -----------------
  constexpr int CH = HALF / 8, QRI = 64 / CH, QT = 32 / QRI;
  bf16x8 qreg[NS];
  {
    const int qr = lane / CH, qc = lane % CH;
    u32x4 x1[QT], x2[QT];
#pragma unroll
    for (int j = 0; j < QT; ++j) {
      const int row = min(q0 + QRI * j + qr, p.T - 1);
      const uint16_t* qptr = p.q + b * p.q_sb + (int64_t)row * p.q_st + h * p.q_sh + 8 * qc;
      x1[j] = *reinterpret_cast<const u32x4*>(qptr);
      x2[j] = *reinterpret_cast<const u32x4*>(qptr + HALF);
    }
    if (p.cos != nullptr) {
#pragma unroll
      for (int j = 0; j < QT; ++j) {
        const int row = min(q0 + QRI * j + qr, p.T - 1);
        const float* cr = p.cos + (int64_t)row * HALF + 8 * qc;
        const float* sr = p.sin + (int64_t)row * HALF + 8 * qc;
        float a1[8], a2[8], y1[8], y2[8];
        unpack8(x1[j], a1);
        unpack8(x2[j], a2);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          y1[e] = rope_lo(a1[e], a2[e], cr[e], sr[e]);
          y2[e] = rope_hi(a1[e], a2[e], cr[e], sr[e]);
        }
        x1[j] = pack8(y1);
        x2[j] = pack8(y2);
      }
    }
#pragma unroll
    for (int j = 0; j < QT; ++j) {
      const int r = QRI * j + qr;
      *(u32x4 __attribute__((address_space(3)))*)(size_t)(v_lds + 2 * (r * D + 8 * (qc ^ swz_k(r)))) = x1[j];
      *(u32x4 __attribute__((address_space(3)))*)(size_t)(v_lds + 2 * (r * D + 8 * ((CH + qc) ^ swz_k(r)))) = x2[j];
    }
    const uint32_t q_a0 = v_lds + 2 * (lq * D + 8 * (lh ^ swz_k(lq)));
#pragma unroll
    for (int s = 0; s < NS; ++s)
      qreg[s] = __builtin_bit_cast(bf16x8, *(const u32x4 __attribute__((address_space(3)))*)(size_t)(q_a0 ^ (32u * s)));
    // the fragments are in registers (and the global loads behind them done) before the first copies go out
    __builtin_amdgcn_s_waitcnt(0x0070);
    asm volatile("" ::: "memory");
  }
  if (any) { copy_k(t); copy_v(t); }

  const uint32_t k_a0 = k_lds + 2 * (lq * D + 8 * (lh ^ swz_k(lq)));
  uint32_t v_a0;
  {
    const int i16 = lane & 15, vrow = 4 * lh + (i16 >> 2);
    const int chunk = 2 * ((lane >> 4) & 1) + ((i16 & 3) >> 1);
    v_a0 = v_lds + 2 * (vrow * D + 8 * (chunk ^ swz_v(vrow)) + 4 * (i16 & 1));
  }
  f32x16 oacc[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[dt][r] = 0.f;
  SoftmaxRef ref;

  for (; t <= t_hi; t += W) {
    const int kv0 = t * kTBN;
    const bool more = t + W <= t_hi;
    // K(n) has landed when only V(n)'s copies are outstanding
    __builtin_amdgcn_s_waitcnt(0x0F70 | NCP);
    asm volatile("" ::: "memory");
    f32x16 sacc[1];
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[0][r] = 0.f;
    bf16x8 kf[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s)
      kf[s] = __builtin_bit_cast(bf16x8, *(const u32x4 __attribute__((address_space(3)))*)(size_t)(k_a0 ^ (32u * s)));
    __builtin_amdgcn_s_waitcnt(0xC07F);    // lgkmcnt(0): the fragments are out of LDS, the area takes the next tile
    asm volatile("" ::: "memory");
    if (more) copy_k(t + W);
#pragma unroll
    for (int s = 0; s < NS; ++s) sacc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], qreg[s], sacc[0], 0, 0, 0);
    if (!(kv0 + kTBN - 1 <= min(q0, p.T - 1) && kv0 >= lo_max)) {
      const int hi = qrow - (kv0 + 4 * lh), lo = lo_q - (kv0 + 4 * lh);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int c = 8 * (r >> 2) + (r & 3);
        if (c > hi || c < lo) sacc[0][r] = -INFINITY;
      }
    }
    bf16x8 pfrag[2];
    softmax_tile<kFirst, 1, NDT>(sacc, p.scale_log2e, ref, oacc, pfrag);
    // V(n) has landed when only K(n + 1)'s copies are outstanding
    if (more) __builtin_amdgcn_s_waitcnt(0x0F70 | NCP);
    else __builtin_amdgcn_s_waitcnt(0x0F70);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) {
        lds_u16_ptr vp = (lds_u16_ptr)(size_t)((v_a0 ^ (64u * dt)) + 2 * (16 * m * D));
        const u32x2 a0 = lds_read_tr16_as3(vp), a1 = lds_read_tr16_as3(vp + 8 * D);
        const u32x4 av = {a0.x, a0.y, a1.x, a1.y};
        oacc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av), pfrag[m], oacc[dt], 0, 0, 0);
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);    // the V fragments are out of LDS
    asm volatile("" ::: "memory");
    if (more) copy_v(t + W);
  }

  // Partial results: each lane of a pair holds its share of the row sum; O^T as [query][channel] fp32 in the
  // wavefront's own tile area, 16-byte pieces swizzled by the query.
  const float l_tot = pair_sum(ref.l);
  if (lh == 0) { part_m[wave][lq] = -ref.minus; part_l[wave][lq] = l_tot; }
  float* const po = reinterpret_cast<float*>(&tiles[wave][0][0]);
  constexpr int PC = D / 4;
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int piece = 8 * dt + 2 * g + lh;      // channels 32 dt + 8 g + 4 lh + 0..3
      *reinterpret_cast<f32x4*>(po + lq * D + 4 * (piece ^ (lq & (PC - 1)))) =
          f32x4{oacc[dt][4 * g], oacc[dt][4 * g + 1], oacc[dt][4 * g + 2], oacc[dt][4 * g + 3]};
    }
  __syncthreads();
  // 8 channels per thread and pass
#pragma unroll
  for (int it = 0; it < (32 * CPR + 64 * W - 1) / (64 * W); ++it) {
    const int idx = tid + 64 * W * it, row = idx / CPR, c = idx % CPR;
    if (32 * CPR < 64 * W && idx >= 32 * CPR) break;
    float m = part_m[0][row];
#pragma unroll
    for (int w = 1; w < W; ++w) m = fmaxf(m, part_m[w][row]);
    float l = 0.f, acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float a = fast_exp2(part_m[w][row] - m);
      l = fmaf(part_l[w][row], a, l);
      const float* src = reinterpret_cast<const float*>(&tiles[w][0][0]) + row * D;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const f32x4 o4 = *reinterpret_cast<const f32x4*>(src + 4 * ((2 * c + v) ^ (row & (PC - 1))));
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[4 * v + i] = fmaf(o4[i], a, acc[4 * v + i]);
      }
    }
    const float inv = 1.f / l;
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] *= inv;
    if (q0 + row < p.T)
      store_through(p.o + b * p.o_sb + (int64_t)(q0 + row) * p.o_st + h * p.o_sh + 8 * c, pack8(acc));
  }
}

// Rotates keys once and stores them with the caller's output strides: a copy, bound by memory.  A lane takes 16 bytes of a row, so that every
// access covers whole rows (of 64 channels in particular, half of which are half a line), of HPT heads of one position, for which the
// cos and sin values are fetched once; the channels they are rotated with come from the lane half a row away.  Before, a lane took both
// halves' 16 bytes.  20001 rows, 16 heads of 64 17.2 -> 15.1 us (82 MB: 5.4 TB/s), 8000 rows, 6 heads 17.6 -> 17.1 with the attention behind it; heads of
// 128 level (8 x 4096 rows, 8 heads 78.5 / 78.1 with it).
template <int D, int HPT>
__global__ __launch_bounds__(256) void rope_k_kernel(PrefillParams p) {
  constexpr int HALF = D / 2, CPR = D / 8;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int HG = p.H / HPT;
  // Surplus lanes read the last row as well, since whole rows exchange, and store nothing: k_out may be k, and another wavefront's lanes
  // own that row.
  const int64_t rows = (int64_t)p.B * p.T * HG, row = min(idx / CPR, rows - 1);
  const bool live = idx / CPR < rows;
  const int ch = (int)(idx % CPR), hg = (int)(row % HG), t = (int)(row / HG % p.T), b = (int)(row / HG / p.T);
  u32x4 own[HPT];
  // The unrotated keys are not needed again: read them past the caches, so that q, v and the
  // rotated keys this pass writes are what the attention kernel finds there.
#pragma unroll
  for (int j = 0; j < HPT; ++j)
    own[j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p.k + b * p.k_sb + (int64_t)t * p.k_st + (hg + j * HG) * p.k_sh + 8 * ch));
  const bool lower = ch < CPR / 2;
  const int tl = 8 * (lower ? ch : ch - CPR / 2);
  const float* cr = p.cos + (int64_t)t * HALF + tl;
  const float* sr = p.sin + (int64_t)t * HALF + tl;
  float c[8], sn[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) { c[e] = cr[e]; sn[e] = sr[e]; }
  auto across = [](uint32_t x) {
    const float f = __uint_as_float(x);
    return __float_as_uint(D == 128 ? dpp_move<0x128>(f)                     // row_ror 8: lane i ^ 8 of 16
                                    : dpp_move<0x1B>(dpp_move<0x141>(f)));   // row_half_mirror, then every quad reversed: lane i ^ 4 of 8
  };
#pragma unroll
  for (int j = 0; j < HPT; ++j) {
    const u32x4 other = {across(own[j].x), across(own[j].y), across(own[j].z), across(own[j].w)};
    float x[8], o[8], y[8];
    unpack8(own[j], x);
    unpack8(other, o);
#pragma unroll
    for (int e = 0; e < 8; ++e) y[e] = lower ? rope_lo(x[e], o[e], c[e], sn[e]) : rope_hi(o[e], x[e], c[e], sn[e]);
    if (live) *reinterpret_cast<u32x4*>(p.k_out + b * p.ko_sb + (int64_t)t * p.ko_st + (hg + j * HG) * p.ko_sh + 8 * ch) = pack8(y);
  }
}

// Scalar kernel for head dims the MFMA kernel does not cover (any even D <= 256) and for fp32
// tensors.  One wavefront per (batch, head, query); lanes split the head dim.  Slow by
// design: it serves tiny shapes and the full-precision mode only.  E = uint16_t (bf16 bits;
// rotated values are rounded to bf16 as the bf16 tensors of the reference are) or float
// (nothing is rounded: fp32 in, fp32 arithmetic, fp32 out).
template <typename E>
__global__ __launch_bounds__(64) void prefill_scalar_kernel(PrefillParams p) {
  const int t = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int lane = threadIdx.x;
  const int D = p.D, HALF = D / 2;
  constexpr int MAXPL = 4;  // channels per lane (D <= 256)
  float qv[MAXPL], acc[MAXPL];
  const E* qbase = reinterpret_cast<const E*>(p.q);
  const E* kbase = reinterpret_cast<const E*>(p.k);
  const E* vbase = reinterpret_cast<const E*>(p.v);
  const E* qp = qbase + b * p.q_sb + (int64_t)t * p.q_st + h * p.q_sh;
  auto rot_load = [&](const E* vec, int pos, int d) -> float {
    float x = load_elem<E>(vec, d);
    if (p.cos != nullptr) {
      const bool lower = d < HALF;
      const float xp = load_elem<E>(vec, lower ? d + HALF : d - HALF);
      const float c = p.cos[(int64_t)pos * HALF + (lower ? d : d - HALF)];
      const float s = p.sin[(int64_t)pos * HALF + (lower ? d : d - HALF)];
      x = round_elem<E>(lower ? rope_lo(x, xp, c, s) : rope_hi(xp, x, c, s));
    }
    return x;
  };
#pragma unroll
  for (int i = 0; i < MAXPL; ++i) {
    const int d = lane + 64 * i;
    qv[i] = (d < D) ? rot_load(qp, t, d) * p.scale_log2e : 0.f;
    acc[i] = 0.f;
  }
  if (p.k_out != nullptr && p.cos != nullptr) {
    const E* kp = kbase + b * p.k_sb + (int64_t)t * p.k_st + h * p.k_sh;
    E* op = reinterpret_cast<E*>(p.k_out) + b * p.ko_sb + (int64_t)t * p.ko_st + h * p.ko_sh;
    for (int d = lane; d < D; d += 64) store_elem<E>(op, d, rot_load(kp, t, d));
  }
  float m = -INFINITY, l = 0.f;
  const int lo = row_lo(p, t);
  for (int kv = lo; kv <= t; ++kv) {
    const E* kp = kbase + b * p.k_sb + (int64_t)kv * p.k_st + h * p.k_sh;
    const E* vp = vbase + b * p.v_sb + (int64_t)kv * p.v_st + h * p.v_sh;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < MAXPL; ++i) {
      const int d = lane + 64 * i;
      if (d < D) s = fmaf(qv[i], rot_load(kp, kv, d), s);
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
    const float mn = fmaxf(m, s);
    const float alpha = fast_exp2(m - mn);
    const float pw = fast_exp2(s - mn);
    l = l * alpha + pw;
#pragma unroll
    for (int i = 0; i < MAXPL; ++i) {
      const int d = lane + 64 * i;
      if (d < D) acc[i] = acc[i] * alpha + pw * load_elem<E>(vp, d);
    }
    m = mn;
  }
  E* op = reinterpret_cast<E*>(p.o) + b * p.o_sb + (int64_t)t * p.o_st + h * p.o_sh;
#pragma unroll
  for (int i = 0; i < MAXPL; ++i) {
    const int d = lane + 64 * i;
    if (d < D) store_elem<E>(op, d, acc[i] / l);
  }
}

// Bytes of keys and values that an XCD meets in the kernel with 32 queries per workgroup, whose (batch, head) pairs go round the XCDs in turn:
// those of pairs / gcd(pairs, 8) of them, which find their blocks' neighbours in its L2 (4 MB) or not.
static int64_t met_bytes(int pairs, int T, int D) { return (int64_t)pairs / std::min(pairs & -pairs, 8) * T * D * 4; }
constexpr int64_t kMetBytes = 5 << 20;
// Whether the kernel with four wavefronts per 32 queries is the faster one: up to so many blocks of 128 queries.  It is 1.4 to 2.4 times as fast
// while the blocks leave compute units idle (12 heads of 128, T = 777: 19.4 -> 11.0 us; 8 heads of 64, T = 2048:
// 32.7 -> 14.4 us) and slower beyond (it fetches every key tile four times as often).  From sweeps over 3 to 24 (batch, head) pairs, 145 to 780
// blocks, windows of 120 to 8192 and none, one to hundreds of documents.  us, 128 queries / 32 (heads x rows, blocks of 128):
// Documents, whose lengths the host does not know.  Heads of 128: 12 x 3000 (288) in documents of 20 to 200 tokens 17.7 / 18.0, 200 to 900 32.3 / 23.0, one 68.9 /
// 51.2; 8 x 5100 (320) likewise 18.2 / 20.0, 30.3 / 27.4, 109 / 80; 8 x 8100 (512) 18.5 / 27.4, 34.0 / 40.2, 184 / 181: to 288, from where short ones lose, though long ones
// gain for longer.  With a window under 1024, 8 x 3100 (200), 400 keys 22.4 / 17.8, 8 x 4096 (256) 20.9 / 22.1.  Heads of 64: 12 x 5000 (480) 14.4 / 13.1,
// 21.6 / 18.9; 8 x 8100 (512), 1500 keys 23.9 / 21.9, but one document, a window's mask, 35.7 / 39.6; 24 x 3670 (696) two 39.6 / 43.9.
// Keys past an XCD's L2 and no runs of blocks (below) to help, that is documents, or a window of more than a fourth of the row: heads of 128: 7 x 4000 (224), 1500
// keys, one document 41.0 / 59.7, no window 84.5 / 52.1; 5 x 6000 (235), 1500 keys 41.3 / 67.9, no window, documents of 20 to 200 17.2 / 18.0; 7 x 8000 (441), 4096 keys 102 / 227.
// Heads of 64: 5 x 9000 (355), 4096 keys 57.5 / 68.6; 9 x 4816 (342), 2017 32.8 / 37.9; no window, 9 x 6884 (486) one document 92.2 / 95.2, 7 x 8000 (441) documents of 200 to
// 900 25.9 / 23.2.
// Windows, heads of 128: 8 x 3100 (200), 150 / 400 keys 14.7 / 13.9, 19.7 / 17.8, but 4 x 6472 (204), 236 16.9 / 19.1, 12 x 2491 (240), 438 20.4 / 21.7; 2000 x 16 (256), 800 25.2 /
// 24.1; half of the row or more: 3000 x 12 (288), 1500 42.0 / 41.5, 2 x 5000 x 4 (320), 4096 88 / 78.  Heads of 64: 12000 x 4 (376), 200 / 1500 14.6 / 11.8, 35.8 / 33.5; 10 x 700 x 8
// (480), 400 14.8 / 14.9; 5000 x 12 (480), 1500 37 / 42.
bool prefill_split_wanted(int pairs, int T, int D, int window, bool docs) {
  const bool windowed = window > 0 && window < T, far = !windowed || window >= 1024;
  const bool near = met_bytes(pairs, T, D) <= kMetBytes || (!docs && 4 * (int64_t)window <= T);
  int64_t limit;
  if (!windowed && !docs) limit = D == 64 ? 768 : T >= 1024 ? 384 : 288;
  else if (D == 64) limit = near ? (docs && far ? 500 : 448) : windowed ? 320 : 440;
  else if (windowed && window < 600) limit = pairs % 8 == 0 ? 208 : 144;
  else if (!near) limit = windowed ? 192 : 224;
  else if (docs) limit = far ? 288 : 208;
  else limit = 2 * (int64_t)window >= T ? 320 : 256;
  return (int64_t)pairs * ((T + kBM - 1) / kBM) <= limit;
}
// When the keys and values that an XCD meets leave its L2 and a window makes blocks equally long, it takes a run of neighbouring blocks instead: 4000 rows, 5
// heads of 128 (10 MB), window 200 / 800 / 1500 18.1 / 34.7 / 42.5 -> 13.0 / 22.8 / 33.9 us; 4283 rows, 6 heads (6.6 MB), 200 / 1500 19.2 / 37.9 -> 14.9 / 37.5; but 3000
// rows, 12 heads (4.6 MB), 1500 41.5 -> 45.7.
static bool runs_of_blocks(const PrefillParams& p) {
  const int pairs = p.B * p.H;
  if (p.doc_start != nullptr || p.window <= 0 || 2 * (int64_t)p.window > p.T || pairs % 8 == 0) return false;
  return met_bytes(pairs, p.T, p.D) > kMetBytes;
}

// When those are eight wavefronts: while a compute unit has no second workgroup to run and the longest block has more key tiles than four of them
// take in two turns, in one where a window makes most blocks as long as the longest (us, four / eight; heads of 128, no window: 12 heads x 384 rows 7.0 / 6.6, 8 x 1024 11.3 / 10.1, 4 x 2048 18.3 / 14.9, 2 x 4096 31 / 23;
// window 1024, 4 x 2048 12.7 / 10.3; 256, 8 x 1024 7.5 / 7.0; 128, 32 x 256 6.6 / 6.1; heads of 64, 4 x 2048 13.3 / 10.1; 128 rows 5.0 / 5.2, 256 5.9 / 6.0;
// window 1024, 6 x 2048 14.0 / 16.7).  Causal blocks differ in length, so that long ones gain with twice the workgroups too (heads of 64, 16 x 1024 8.9 /
// 8.8, 8 x 2048 13.8 / 12.2; of 128, 12 x 1024 12.4 / 12.9, 8 x 1536 15.8 / 13.9, 4 x 4096 35 / 30).  Documents' lengths are not known here.
template <int D>
static bool eight_wavefronts(const PrefillParams& p, int64_t workgroups) {
  if (p.doc_start != nullptr) return false;
  const bool full = p.window <= 0 || p.window >= p.T;
  const int tiles = full ? (p.T + kTBN - 1) / kTBN : (p.window - 2 + kTBN) / kTBN + 1;      // of the longest block
  if (workgroups <= 256) return tiles >= (full ? 9 : 5);
  return full && workgroups <= 512 && tiles >= (D == 64 ? 32 : 48);
}

template <int D>
static int launch_mfma(PrefillParams p, hipStream_t s) {
  const int64_t nwg = (int64_t)p.nqb * p.H * p.B;
  if (nwg > 0x7fffffff) {
    set_error("prefill: too many workgroups (%lld)", (long long)nwg);
    return DAISY_ERR_INVALID_ARGUMENT;
  }
  if (p.cos != nullptr) {
    // Pre-pass: rotate K once into k_out, then attend over k_out.
    // (four heads a thread, four 16-byte accesses under way: heads of 128 are better off with two, whose rotation is twice as long: 77.9 and 78.8 us
    // for 8 x 4096 rows, 8 heads, with the attention)
    constexpr int kHeads = D == 64 ? 4 : 2;
    const int hpt = p.H % kHeads == 0 ? kHeads : p.H % 2 == 0 ? 2 : 1;
    const int64_t total = (int64_t)p.B * p.T * (p.H / hpt) * (D / 8);
    const dim3 grid((unsigned)((total + 255) / 256));
    if (hpt == kHeads) hipLaunchKernelGGL((rope_k_kernel<D, kHeads>), grid, dim3(256), 0, s, p);
    else if (hpt == 2) hipLaunchKernelGGL((rope_k_kernel<D, 2>), grid, dim3(256), 0, s, p);
    else hipLaunchKernelGGL((rope_k_kernel<D, 1>), grid, dim3(256), 0, s, p);
    DAISY_CHECK_LAUNCH("rope_k_kernel");
    p.k = p.k_out; p.k_sb = p.ko_sb; p.k_st = p.ko_st; p.k_sh = p.ko_sh;
  }
  if (prefill_split_wanted(p.B * p.H, p.T, D, p.window, p.doc_start != nullptr)) {
    const int64_t nsw = (int64_t)((p.T + 31) / 32) * p.H * p.B;
    p.runs = runs_of_blocks(p);
    if (eight_wavefronts<D>(p, nsw)) hipLaunchKernelGGL((prefill_split_kernel<D, 8>), dim3((unsigned)nsw), dim3(512), 0, s, p);
    else hipLaunchKernelGGL((prefill_split_kernel<D, 4>), dim3((unsigned)nsw), dim3(kPrefillThreads), 0, s, p);
    DAISY_CHECK_LAUNCH("prefill_split_kernel");
    return DAISY_OK;
  }
  if (D == 64 && p.keys > kTBN) hipLaunchKernelGGL(prefill_wide_tile_kernel, dim3((unsigned)nwg), dim3(kPrefillThreads), 0, s, p);
  else if (p.period > 0 && p.window < (D == 64 ? 256 : 384)) hipLaunchKernelGGL((prefill_short_window_kernel<D>), dim3((unsigned)nwg), dim3(kPrefillThreads), 0, s, p);
  else hipLaunchKernelGGL((prefill_tile_kernel<D>), dim3((unsigned)nwg), dim3(kPrefillThreads), 0, s, p);
  DAISY_CHECK_LAUNCH("prefill_tile_kernel");
  return DAISY_OK;
}

// Argument checks and parameter block shared by the bf16 and the fp32 entry point.
static int fill_prefill_params(PrefillParams& p, const void* q, const int64_t* q_strides,
                               const void* k, const int64_t* k_strides,
                               const void* v, const int64_t* v_strides,
                               const float* cos, const float* sin, const int32_t* doc_start,
                               void* o, const int64_t* o_strides,
                               void* k_out, const int64_t* k_out_strides,
                               int B, int T, int H, int D, int window, float scale) {
  DAISY_CHECK_ARG(q && k && v && o, "prefill: q, k, v and o must be non-NULL");
  DAISY_CHECK_ARG(q_strides && k_strides && v_strides && o_strides, "prefill: stride arrays must be non-NULL");
  DAISY_CHECK_ARG(B > 0 && T > 0 && H > 0, "prefill: B=%d, T=%d, H=%d must be positive", B, T, H);
  DAISY_CHECK_ARG((cos == nullptr) == (sin == nullptr), "prefill: cos and sin must both be given or both NULL");
  DAISY_CHECK_ARG(k_out == nullptr || k_out_strides != nullptr, "prefill: k_out needs k_out_strides");
  DAISY_CHECK_SUPPORTED(D >= 2 && D <= 256 && D % 2 == 0, "prefill: head_dim %d not supported (even, 2..256)", D);
  p.q = (const uint16_t*)q; p.q_sb = q_strides[0]; p.q_st = q_strides[1]; p.q_sh = q_strides[2];
  p.k = (const uint16_t*)k; p.k_sb = k_strides[0]; p.k_st = k_strides[1]; p.k_sh = k_strides[2];
  p.v = (const uint16_t*)v; p.v_sb = v_strides[0]; p.v_st = v_strides[1]; p.v_sh = v_strides[2];
  p.cos = cos; p.sin = sin; p.doc_start = doc_start;
  p.o = (uint16_t*)o; p.o_sb = o_strides[0]; p.o_st = o_strides[1]; p.o_sh = o_strides[2];
  p.k_out = (uint16_t*)k_out;
  p.ko_sb = k_out ? k_out_strides[0] : 0; p.ko_st = k_out ? k_out_strides[1] : 0; p.ko_sh = k_out ? k_out_strides[2] : 0;
  p.B = B; p.T = T; p.H = H; p.D = D; p.window = window;
  p.nqb = (T + kBM - 1) / kBM;
  // Head dim 64: tiles of 64 keys, but for short windows, of which the tiles at their edges are a larger part.  32 / 64 keys a tile, us:
  // T = 16384, 12 heads, no window 605 / 558; T = 32768, 32 heads 4440 / 4344; window 8192, five documents of T = 65536, 4 heads 425 / 412; window
  // 4096, seven of T = 20001, 16 heads 154.5 / 154.2; 2048, T = 32768, 16 heads 300 / 293; 1024, 8 x 4096, 16 heads 147 / 145.5; 384, T = 32768, 8 heads
  // 48.2 / 45.5; 256, 4 x 8192, 16 heads 66.6 / 67; 128, 16 x 2048, 8 heads 26.6 / 27.
  const bool windowed = window > 0 && window < T;
  const int keys = p.keys = D == 64 && !(windowed && window < 384) ? 2 * kTBN : kTBN;
  p.period = (window > 0 && window < T) ? (kBM - 1) / keys + 1 + (window - 1 + keys - 1) / keys : 0;
  p.n_light = (window > 0 && window < T) ? min((window - 1 + kBM - 1) / kBM, p.nqb) : 0;
  p.order_shift = -1; p.order_bit = 0;
  // Finding the order costs a workgroup about 1 us; the lengths differ enough to pay for it where a window is an eighth of the
  // row or more (three documents of T = 16384, window 2048: 197 -> 182 us; at a sixteenth nine documents take 258 against 270 us).
  // Without a window they differ also within a lone document (T = 8192, 16 heads of 64: 207 -> 171 us); bounds of rows that all
  // reach equally far back only pay (8 key blocks of T = 32768: 144 -> 151 us), so a caller who knows how far gives that as the window.
  if (doc_start != nullptr && p.nqb <= 64 * kOrderChunks && (window <= 0 || (int64_t)window * 8 >= T)) {
    int longest = (window > 0 && window < T ? window : T) / 32 + 6;     // tiles of a block
    for (p.order_shift = 0; longest > 255; longest >>= 1) ++p.order_shift;
    for (p.order_bit = 1; 2 * p.order_bit <= longest; p.order_bit *= 2) {}
  }
  p.scale_log2e = scale * kLog2e;
  return DAISY_OK;
}

}  // namespace daisy

using namespace daisy;

extern "C" int daisy_prefill_fwd(const void* q, const int64_t* q_strides,
                                 const void* k, const int64_t* k_strides,
                                 const void* v, const int64_t* v_strides,
                                 const float* cos, const float* sin,
                                 const int32_t* doc_start,
                                 void* o, const int64_t* o_strides,
                                 void* k_out, const int64_t* k_out_strides,
                                 int B, int T, int H, int D,
                                 int window, float scale, int flags, void* stream) {
  PrefillParams p;
  const int rc = fill_prefill_params(p, q, q_strides, k, k_strides, v, v_strides, cos, sin, doc_start, o, o_strides,
                                     k_out, k_out_strides, B, T, H, D, window, scale);
  if (rc != DAISY_OK) return rc;
  hipStream_t s = (hipStream_t)stream;
  DAISY_CHECK_ARG(flags == 0, "prefill: flags must be 0 (got %d)", flags);

  if (D == 64 || D == 128) {
    auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
    DAISY_CHECK_ARG(al16(q) && al16(k) && al16(v) && al16(o) && al16(k_out) && al16(cos) && al16(sin),
                    "prefill: tensors must be 16-byte aligned");
    for (int i = 0; i < 3; ++i) {
      DAISY_CHECK_ARG(q_strides[i] % 8 == 0 && k_strides[i] % 8 == 0 && v_strides[i] % 8 == 0 && o_strides[i] % 8 == 0 &&
                          (!k_out || k_out_strides[i] % 8 == 0),
                      "prefill: strides must be multiples of 8 elements");
    }
    // The keys are rotated once, into k_out, and attended from there: without that buffer every query
    // block would have to rotate every key tile again (measured 3.7 times slower), so it is required.
    DAISY_CHECK_ARG(cos == nullptr || k_out != nullptr,
                    "prefill: cos/sin with head_dim %d need k_out (the rotated keys are written there and attended from there)", D);
    return D == 128 ? launch_mfma<128>(p, s) : launch_mfma<64>(p, s);
  }

  DAISY_CHECK_ARG(B <= 65535 && H <= 65535, "prefill: B and H must each be <= 65535 for the scalar kernel");
  hipLaunchKernelGGL(prefill_scalar_kernel<uint16_t>, dim3(T, H, B), dim3(64), 0, s, p);
  DAISY_CHECK_LAUNCH("prefill_scalar_kernel");
  return DAISY_OK;
}

extern "C" int daisy_prefill_fwd_f32(const float* q, const int64_t* q_strides,
                                     const float* k, const int64_t* k_strides,
                                     const float* v, const int64_t* v_strides,
                                     const float* cos, const float* sin,
                                     const int32_t* doc_start,
                                     float* o, const int64_t* o_strides,
                                     float* k_out, const int64_t* k_out_strides,
                                     int B, int T, int H, int D,
                                     int window, float scale, void* stream) {
  PrefillParams p;
  const int rc = fill_prefill_params(p, q, q_strides, k, k_strides, v, v_strides, cos, sin, doc_start, o, o_strides,
                                     k_out, k_out_strides, B, T, H, D, window, scale);
  if (rc != DAISY_OK) return rc;
  DAISY_CHECK_ARG(B <= 65535 && H <= 65535, "prefill: B and H must each be <= 65535 for the fp32 kernel");
  hipLaunchKernelGGL(prefill_scalar_kernel<float>, dim3(T, H, B), dim3(64), 0, (hipStream_t)stream, p);
  DAISY_CHECK_LAUNCH("prefill_scalar_kernel<float>");
  return DAISY_OK;
}
