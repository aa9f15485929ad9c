// Projections of a few hundred activation rows for gfx950: y = x W^T on the matrix cores, and the QKV projection
// with everything that follows it up to the attention (models/daisy/attention.py:116-135) in its epilogue.
//
// What bounds it.  A prompt of a few hundred tokens (or a decode step of a few dozen sequences) has too few output
// tiles to give every compute unit several workgroups, so nothing hides a workgroup's own latencies: with one K step in
// flight, a step lasts a memory round trip (about 0.7 us) where its matrix instructions take 0.2 us.  The kernel
// keeps up to three K steps in flight (asynchronous global -> LDS copies; a wavefront waits with vmcnt for the oldest
// step only), reads the operands of the next products beside the ones at hand, and the tile shape follows the number of
// tiles (kProjTiles).  Large products are bound by the matrix cores and by what the compute units can pull through the
// L2, hence the order of the tiles (below).
//
// Operands: both x [M, K] and W [N, K] have K contiguous, so both tiles are rows of 64 or 128 bf16 in LDS, their
// 16-byte chunks XOR-swizzled so that 16 rows read side by side fall into 16 different slots of the 256-byte bank
// window.  v_mfma_f32_16x16x32_bf16 with W as left operand: a lane's accumulator holds four
// consecutive output columns of one row, which go through LDS once and leave as whole rows.
#include "common.h"

#include <type_traits>

namespace daisy {

struct ProjParams {
  ProjSegment one;                     // the product (bias and y: plain epilogue only)
  int M, K, MT, NT;
  QkvEpilogue e;                       // QKV epilogue
};
// Several products, told apart by the column of tiles.
struct ProjSegmentsParams {
  ProjSegment seg[kMaxSegments];
  int n, M, K, MT, NT;
  KdaGates gates;                      // EPI 3
};

// At most N vector-memory operations outstanding (bits 3:0 and 15:14 of the immediate) and every LDS read back.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | ((N >> 4) << 14));
}

// EPI 0: y = x W^T (+ bias), bf16, of one or (SEGMENTS) several products.  EPI 1 / 2: the QKV epilogue for heads of 64 / 128 channels.
// EPI 3: as 0, the first product through the KDA layer's decay gate.
// WVM x WVN wavefronts; BK elements of K per step.
template <int BM, int BN, int WVM, int WVN, int BK, int STAGES, int EPI, bool SEGMENTS = false>
__global__ __launch_bounds__(64 * WVM * WVN) void proj_kernel(std::conditional_t<SEGMENTS, ProjSegmentsParams, ProjParams> p) {
  constexpr int NW = WVM * WVN, NTHR = 64 * NW;
  constexpr int WM = BM / WVM, WN = BN / WVN, MI = WM / 16, NI = WN / 16, KK = BK / 32;
  constexpr int RB = 2 * BK, CPRW = BK / 8, RPC = 64 / CPRW;   // bytes and 16-byte chunks per tile row, rows per copy
  constexpr int CA = BM / RPC / NW, CB = BN / RPC / NW;        // copies per wavefront and step
  constexpr int CPW = CA + CB;
  constexpr int ABYTES = BM * RB, STAGE = (BM + BN) * RB;
  static_assert(CA >= 1 && CB >= 1 && MI >= 1 && NI >= 1, "every wavefront copies and multiplies");
  static_assert(STAGES <= 4 && CPW * (STAGES - 2) < 64, "vmcnt counts to 63");
  static_assert(STAGES * STAGE >= BM * BN * 2, "the output tile passes through the stages");
  __shared__ __attribute__((aligned(1024))) char smem[STAGES * STAGE];
  // swizzle of a row's chunks: 16 rows read side by side must fall into 16 slots of the 256-byte bank window
  auto swz = [](int r) { return BK == 128 ? (r & 15) : ((r >> 1) & 7); };

  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WVM, wn = wave / WVM;

  // Workgroups are dealt round-robin to the 8 XCDs: an XCD takes a contiguous run of tiles, in panels of eight rows of
  // tiles walked column by column, so that the tiles in flight on an XCD share rows of x and of W in its L2 (32 of them
  // at a time: 8 x 4 tiles read 12 strips, a column of 32 would read 33 and be bound by the bandwidth behind the L2).
  const int total = p.MT * p.NT, per = total >> 3, rest = total & 7;
  const int xcd = blockIdx.x & 7, vid = xcd * per + min(xcd, rest) + (blockIdx.x >> 3);
  const int panel = vid / (8 * p.NT), in_panel = vid - panel * 8 * p.NT, rows = min(8, p.MT - 8 * panel);
  const int mt = 8 * panel + in_panel % rows;
  int nt = in_panel / rows;
  const ProjSegment* gp;
  [[maybe_unused]] bool gated = false;
  if constexpr (SEGMENTS) {
    // gated and plain columns of tiles in turn: the gate's arithmetic runs beside the other workgroups' stores (32768 rows of 16
    // heads of 128, which low_rank_kernel takes by now: 146 -> 134 us)
    if (EPI == 3 && p.NT == 2 * p.seg[0].tile_end) nt = (nt >> 1) + (nt & 1) * p.seg[0].tile_end;
    int i = 0;
    while (i + 1 < p.n && nt >= p.seg[i].tile_end) ++i;
    if (i > 0) nt -= p.seg[i - 1].tile_end;
    gp = &p.seg[i];
    gated = EPI == 3 && i == 0;
  } else {
    gp = &p.one;
  }
  const ProjSegment g = *gp;
  const int m0 = mt * BM, n0 = nt * BN;

  // Copy j of this wavefront covers tile rows RPC (wave + NW j) ..: lane i lands at row i / CPRW, chunk position i % CPRW and
  // fetches the chunk that belongs there.  Rows past the end re-read the last row (their results are not stored).
  const int cr = lane / CPRW, cp = lane % CPRW;
  int offa[CA], offb[CB];
#pragma unroll
  for (int j = 0; j < CA; ++j) {
    const int r = RPC * (wave + NW * j) + cr;
    offa[j] = 2 * (int)((min(m0 + r, p.M - 1) - m0) * g.x_sm) + 16 * (cp ^ swz(r));
  }
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int r = RPC * (wave + NW * j) + cr;
    offb[j] = 2 * (int)((min(n0 + r, g.N - 1) - n0) * g.w_sn) + 16 * (cp ^ swz(r));
  }
  const uint16_t* xa = g.x + (int64_t)m0 * g.x_sm;
  const uint16_t* wb = g.w + (int64_t)n0 * g.w_sn;
  const uint32_t lds0 = lds_address(smem) + 1024 * wave;
  auto issue = [&](int st) {
    const uint32_t dst = lds0 + st * STAGE;
#pragma unroll
    for (int j = 0; j < CB; ++j) copy16_to_lds_async(wb, offb[j], dst + ABYTES + 1024 * NW * j);
#pragma unroll
    for (int j = 0; j < CA; ++j) copy16_to_lds_async(xa, offa[j], dst + 1024 * NW * j);
    xa += BK;
    wb += BK;
  };

  f32x4 acc[NI][MI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nk = p.K / BK;
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nk) issue(s);

  // Fragment addresses inside a stage: chunk (4 kk + q4) ^ swizzle of its row; rows 16 apart share a swizzle.
  const uint32_t fa = lds_address(smem) + (WM * wm + ln) * RB + 16 * (q4 ^ swz(ln));
  const uint32_t fb = lds_address(smem) + ABYTES + (WN * wn + ln) * RB + 16 * (q4 ^ swz(ln));
  auto frag = [&](uint32_t a) { return __builtin_bit_cast(bf16x8, *(const u32x4 __attribute__((address_space(3)))*)(size_t)a); };

  // The copies of a step have landed when at most those of the `behind` steps after it are outstanding.
  auto landed = [&](int behind) {
    if (STAGES == 2 || behind <= 0) wait_vmcnt<0>();
    else if (behind >= STAGES - 2) wait_vmcnt<CPW * (STAGES - 2)>();
    else wait_vmcnt<CPW>();                  // STAGES <= 4: one step behind
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  bf16x8 a[2][NI], b[2][MI];                 // operands of 32 elements of K, and the next ones
  auto read = [&](int kk, uint32_t so) {
#pragma unroll
    for (int i = 0; i < NI; ++i) a[kk & 1][i] = frag((fb ^ (64u * kk)) + so + 16 * RB * i);
#pragma unroll
    for (int j = 0; j < MI; ++j) b[kk & 1][j] = frag((fa ^ (64u * kk)) + so + 16 * RB * j);
  };
  auto multiply = [&](int kk) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < MI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk & 1][i], b[kk & 1][j], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  static_assert(KK % 2 == 0, "a step ends on the second set");
  int st = 0;
  if constexpr (STAGES == 2) {
    for (int k = 0; k < nk; ++k) {
      landed(0);
      const uint32_t so = st * STAGE;
      read(0, so);
      __builtin_amdgcn_sched_barrier(0);
      // every wavefront is done with step k - 1: its stage takes step k + 1
      if (k + 1 < nk) issue(st ^ 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        if (kk + 1 < KK) read(kk + 1, so);
        multiply(kk);
      }
      st ^= 1;
    }
  } else {
    // The operands of a step's first products are read beside the last ones of the step before, so that only the barrier lies between
    // two steps' products, not the reads (0.2 of 0.41 us a step of 128 x 128 x 64 on eight wavefronts; its matrix instructions take 0.32 at the
    // clock that they are granted).  us, before / now: 16 x 4608 x 1536 (tile 9) 5.21 / 4.89, 64 x 2048 x 2048 6.03 / 5.44; 128 x 2048 x 2048 (10) 6.38 /
    // 5.78; 128 x 6144 x 2048 (2) 9.25 / 8.80; 777 x 4608 x 1536 (5) 15.4 / 14.9; tiles 1, 3 and 4 level; with two stages it loses (6: 1500 x 4608 x 1536 23.4 /
    // 27.6; 7: a layer of 8 x 4096 rows 403 / 411).
    // `inside`: there are STAGES more steps; else `behind` of them after the next one, -1: no next one.
    uint32_t so = 0;
    auto step = [&](auto inside, int behind) {
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        if (kk + 1 < KK) {
          read(kk + 1, so);
        } else if (inside || behind >= 0) {
          // the step's last operands are in registers, of all wavefronts behind the barrier: its stage takes the step STAGES ahead
          landed(inside ? STAGES - 2 : behind);
          so = st + 1 == STAGES ? 0 : so + STAGE;
          read(0, so);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (inside) issue(st);
          st = st + 1 == STAGES ? 0 : st + 1;
        }
        multiply(kk);
      }
    };
    landed(min(STAGES - 1, nk) - 1);
    if (STAGES - 1 < nk) issue(STAGES - 1);
    read(0, 0);
    // (with a scalar load pending here the compiler, which cannot tell their order, would wait for every LDS read ahead of the products)
    __builtin_amdgcn_s_waitcnt(0xC07F);       // lgkmcnt(0)
    int k = 0;
    for (; k + STAGES < nk; ++k) step(std::true_type{}, 0);
    for (; k < nk; ++k) step(std::false_type{}, nk - 2 - k);
  }
  __syncthreads();

  // Output tile [BM][BN] bf16 in LDS, 16-byte chunks swizzled by the row.
  constexpr int CHN = BN / 8;                      // chunks per row
  auto tile_at = [&](int m, int c) { return smem + m * (2 * BN) + 16 * (c ^ (m & (CHN - 1))); };
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int n = WN * wn + 16 * i + 4 * q4;       // four consecutive columns
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if ((EPI == 0 || EPI == 3) && g.bias != nullptr) {
#pragma unroll
      for (int r = 0; r < 4; ++r) bv[r] = bf16lo_to_f32(g.bias[min(n0 + n + r, g.N - 1)]);
    }
#pragma unroll
    for (int j = 0; j < MI; ++j) {
      const int m = WM * wm + 16 * j + ln;
      const u32x2 v = {pack_bf16x2(acc[i][j][0] + bv[0], acc[i][j][1] + bv[1]), pack_bf16x2(acc[i][j][2] + bv[2], acc[i][j][3] + bv[3])};
      *reinterpret_cast<u32x2*>(tile_at(m, n >> 3) + 2 * (n & 7)) = v;
    }
  }
  __syncthreads();

  if constexpr (EPI == 3) {
    // The gate was a kernel of its own behind the product: 134 MB read and written once more for 32768 rows of 16 heads of 128.
    if (gated) {
      const KdaGates& kg = p.gates;
      static_assert(NTHR % CHN == 0, "a thread keeps its channels");
      const int c = tid % CHN, col = n0 + 8 * c;
      if (col < g.N) {
        const float scale = -expf(kg.A_log[col / kg.Dk]);
        float bv[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) bv[e] = kg.dt_bias[col + e];
        for (int m = tid / CHN; m < min(BM, p.M - m0); m += NTHR / CHN) {
          float f[8];
          unpack8(*reinterpret_cast<const u32x4*>(tile_at(m, c)), f);
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] = scale * softplus(f[e] + bv[e], 1.f, 20.f, 1.f);
          *reinterpret_cast<u32x4*>(g.y + (int64_t)(m0 + m) * g.y_sm + col) = pack8(f);
        }
      }
      if (n0 == 0) {                         // beta of these rows
        const int count = min(BM, p.M - m0) * kg.H;
        for (int i = tid; i < count; i += NTHR) {
          const float logit = bf16lo_to_f32(kg.logits[(int64_t)(m0 + i / kg.H) * kg.logits_row + i % kg.H]);
          kg.beta[(int64_t)m0 * kg.H + i] = round_bf16(1.f / (1.f + expf(-logit)));
        }
      }
      return;
    }
  }
  if constexpr (EPI == 0 || EPI == 3) {
#pragma unroll
    for (int it = 0; it < (BM * CHN + NTHR - 1) / NTHR; ++it) {
      const int idx = tid + NTHR * it, m = idx / CHN, c = idx % CHN;
      if (BM * CHN % NTHR != 0 && m >= BM) break;
      const u32x4 v = *reinterpret_cast<const u32x4*>(tile_at(m, c));
      if (m0 + m < p.M && n0 + 8 * c < g.N) store_through(g.y + (int64_t)(m0 + m) * g.y_sm + n0 + 8 * c, v);
    }
  } else {
    constexpr int D = EPI == 1 ? 64 : 128, HALF = D / 2, LPR = D / 16, HPT = BN / D;
    static_assert(BN % D == 0, "a tile holds whole heads");
    const QkvEpilogue& e = p.e;
    // A thread takes the same channels of all heads of its row where that still gives every thread a row: it then fetches the
    // rotation (four times the bytes of the channels it turns) once.
    constexpr int HS = BM * LPR % NTHR == 0 ? HPT : 1;
    static_assert(BM * BN / 16 / HS % 64 == 0, "whole wavefronts");
    constexpr int PASSES = (BM * BN / 16 / HS + NTHR - 1) / NTHR, UNROLL = 4 / HS > 0 ? 4 / HS : 1;
#pragma unroll(PASSES < UNROLL ? PASSES : UNROLL)
    for (int it = 0; it < PASSES; ++it) {
      // LPR lanes share one (row, head): lane c holds channels [8c, 8c + 8) and their rotation partners
      const int idx = tid + NTHR * it, c = idx % LPR, h0 = idx / LPR % (HPT / HS) * HS, m = idx / (LPR * (HPT / HS));
      if (BM * BN / 16 / HS % NTHR != 0 && m >= BM) break;
      const int row = min(m0 + m, p.M - 1);
      const int t = row % e.T, b = row / e.T;
      f32x4 cs[2], sn[2];
      if (n0 + h0 * D < 2 * e.H * D) {
        const int64_t off = (int64_t)(e.pos0 + t) * HALF + 8 * c;
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          cs[v] = *reinterpret_cast<const f32x4*>(e.cos + off + 4 * v);
          sn[v] = *reinterpret_cast<const f32x4*>(e.sin + off + 4 * v);
        }
      }
#pragma unroll
      for (int j = 0; j < HS; ++j) {
        const int hh = h0 + j;
        const int n = n0 + hh * D;
        const bool live = m0 + m < p.M && n < g.N;
        const int third = min(n / (e.H * D), 2), h = min(n / D - third * e.H, e.H - 1);
        float lo[8], hi[8];
        unpack8(*reinterpret_cast<const u32x4*>(tile_at(m, hh * (D / 8) + c)), lo);
        unpack8(*reinterpret_cast<const u32x4*>(tile_at(m, hh * (D / 8) + LPR + c)), hi);
        // x * rsqrt(mean(x^2) + eps), rounded to bf16 like the norm's output tensor
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += lo[i] * lo[i];
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += hi[i] * hi[i];
        ss = group_sum<LPR>(ss);
        const float rstd = rsqrtf(ss / (float)D + e.eps);
#pragma unroll
        for (int i = 0; i < 8; ++i) { lo[i] = round_bf16(lo[i] * rstd); hi[i] = round_bf16(hi[i] * rstd); }
        uint16_t* dst;
        if (third < 2) {
#pragma unroll
          for (int i = 0; i < 8; ++i) {
            const float x1 = lo[i], x2 = hi[i];
            lo[i] = rope_lo(x1, x2, cs[i / 4][i % 4], sn[i / 4][i % 4]);
            hi[i] = rope_hi(x1, x2, cs[i / 4][i % 4], sn[i / 4][i % 4]);
          }
          dst = third == 0 ? e.q + b * e.q_sb + t * e.q_st + h * e.q_sh : e.k + b * e.k_sb + t * e.k_st + h * e.k_sh;
        } else {
          if (e.ve != nullptr) {
            // g*v + (1-g)*ve with every product, the difference and the sum rounded to bf16
            const float gv = gate_value(e.gate), og = round_bf16(1.0f - gv);
            const uint16_t* vp = e.ve + b * e.ve_sb + t * e.ve_st + h * e.ve_sh + 8 * c;
            float el[8], eh[8];
            unpack8(*reinterpret_cast<const u32x4*>(vp), el);
            unpack8(*reinterpret_cast<const u32x4*>(vp + HALF), eh);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              lo[i] = round_bf16(gv * lo[i]) + round_bf16(og * el[i]);
              hi[i] = round_bf16(gv * hi[i]) + round_bf16(og * eh[i]);
            }
          }
          dst = e.v + b * e.v_sb + t * e.v_st + h * e.v_sh;
        }
        if (live) {
          store_through(dst + 8 * c, pack8(lo));
          store_through(dst + 8 * c + HALF, pack8(hi));
        }
      }
    }
  }
}

// Several narrow products of the same rows of x in one tile of 128 rows and up to 288 columns, so that x is read once: with a column of
// tiles of its own per product, two or three of 128, every one of them pulls x again.  M = 32768, K = 2048, N = 128 + 128 + 16: 52.9 us with
// 128 x 128 -> 39.0 (3.7 TB/s of x and results).  A step of 64 elements of K takes 1.0 us even of a single workgroup: reads of the LDS, products
// and waits in a row.  Eight wavefronts of 32 rows x 144 columns.  *Tried:* 64 x 80 (fewer LDS reads): 40.9; only the copies that narrower products
// need: 39.4, and 35.5 instead of 32.4 for a single workgroup.
constexpr int kJoinedRows = 128, kJoinedColumns = 288;
__global__ __launch_bounds__(512) void proj_joined_kernel(ProjSegmentsParams p) {
  constexpr int BM = kJoinedRows, BN = kJoinedColumns, BK = 64, STAGES = 3, NW = 8;
  constexpr int WM = 32, WN = 144, MI = WM / 16, NI = WN / 16, KK = BK / 32;
  constexpr int RB = 2 * BK, ABYTES = BM * RB, STAGE = (BM + BN) * RB;
  constexpr int CA = BM / 8 / NW, CB = (BN / 8 + NW - 1) / NW, CPW = CA + CB;       // copies of 8 rows per wavefront and step
  __shared__ __attribute__((aligned(1024))) char smem[STAGES * STAGE];
  auto swz = [](int r) { return (r >> 1) & 7; };

  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 15, q4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 3, wn = wave >> 2;
  const int m0 = blockIdx.x * BM;

  // Eight rows of W per copy, of one product: each begins at a multiple of eight columns (tile_end: of the last one behind it).  Copies past
  // the last column, and the ones that the last wavefronts do not have, repeat the last one that there is, into the same place.
  const int cr = lane / 8, cp = lane % 8;
  int offa[CA], offb[CB], to[CB];
  const uint16_t* wb[CB];
  const uint16_t* xa = p.seg[0].x + (int64_t)m0 * p.seg[0].x_sm;
#pragma unroll
  for (int j = 0; j < CA; ++j) {
    const int r = 8 * (wave + NW * j) + cr;
    offa[j] = 2 * (int)((min(m0 + r, p.M - 1) - m0) * p.seg[0].x_sm) + 16 * (cp ^ swz(r));
  }
#pragma unroll
  for (int j = 0; j < CB; ++j) {
    const int c8 = 8 * min(wave + NW * j, p.NT - 1);
    int i = 0;
    while (i + 1 < p.n && c8 >= p.seg[i].tile_end) ++i;
    const int row0 = c8 - (i > 0 ? p.seg[i - 1].tile_end : 0);
    wb[j] = p.seg[i].w + (int64_t)row0 * p.seg[i].w_sn;
    offb[j] = 2 * (int)((min(row0 + cr, p.seg[i].N - 1) - row0) * p.seg[i].w_sn) + 16 * (cp ^ swz(c8 + cr));
    to[j] = ABYTES + c8 * RB;
  }
  const uint32_t lds0 = lds_address(smem);
  auto issue = [&](int st) {
    const uint32_t dst = lds0 + st * STAGE;
#pragma unroll
    for (int j = 0; j < CB; ++j) { copy16_to_lds_async(wb[j], offb[j], dst + to[j]); wb[j] += BK; }
#pragma unroll
    for (int j = 0; j < CA; ++j) copy16_to_lds_async(xa, offa[j], dst + 1024 * (wave + NW * j));
    xa += BK;
  };

  f32x4 acc[NI][MI];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MI; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int nk = p.K / BK;
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < nk) issue(s);
  // (columns that no product has are multiplied from what the LDS holds and not stored)
  const uint32_t fa = lds0 + (WM * wm + ln) * RB + 16 * (q4 ^ swz(ln));
  const uint32_t fb = lds0 + ABYTES + (WN * wn + ln) * RB + 16 * (q4 ^ swz(ln));
  auto frag = [&](uint32_t a) { return __builtin_bit_cast(bf16x8, *(const u32x4 __attribute__((address_space(3)))*)(size_t)a); };

  int st = 0;
  for (int k = 0; k < nk; ++k) {
    if (k + 1 == nk) wait_vmcnt<0>(); else wait_vmcnt<CPW>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint32_t so = st * STAGE;
    bf16x8 a[KK][NI], b[KK][MI];
#pragma unroll
    for (int j = 0; j < MI; ++j) b[0][j] = frag(fa + so + 16 * RB * j);
#pragma unroll
    for (int i = 0; i < NI; ++i) a[0][i] = frag(fb + so + 16 * RB * i);
    __builtin_amdgcn_sched_barrier(0);
    // every wavefront is done with step k - 1: its stage takes step k + 2
    if (k + STAGES - 1 < nk) issue(st == 0 ? STAGES - 1 : st - 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      if (kk + 1 < KK) {
#pragma unroll
        for (int j = 0; j < MI; ++j) b[kk + 1][j] = frag((fa ^ (64u * (kk + 1))) + so + 16 * RB * j);
#pragma unroll
        for (int i = 0; i < NI; ++i) a[kk + 1][i] = frag((fb ^ (64u * (kk + 1))) + so + 16 * RB * i);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < MI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[kk][i], b[kk][j], acc[i][j], 0, 0, 0);
    }
    st = st + 1 == STAGES ? 0 : st + 1;
  }
  __syncthreads();

  // Output tile [BM][BN] bf16 in LDS, its pieces in fours swizzled by the row, then whole rows of every product.
  constexpr int CHN = BN / 8;
  auto tile_at = [&](int m, int c) { return smem + m * (2 * BN) + 16 * (c ^ (m & 3)); };
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int n = WN * wn + 16 * i + 4 * q4;
#pragma unroll
    for (int j = 0; j < MI; ++j)
      *reinterpret_cast<u32x2*>(tile_at(WM * wm + 16 * j + ln, n >> 3) + 2 * (n & 7)) =
          u32x2{pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3])};
  }
  __syncthreads();
  for (int idx = tid; idx < BM * CHN; idx += 64 * NW) {
    const int m = idx / CHN, c = idx % CHN;
    if (m0 + m >= p.M || c >= p.NT) continue;
    const u32x4 v = *reinterpret_cast<const u32x4*>(tile_at(m, c));
    uint16_t* y = p.seg[0].y + (int64_t)(m0 + m) * p.seg[0].y_sm + 8 * c;
#pragma unroll
    for (int i = 1; i < kMaxSegments; ++i)
      if (i < p.n && 8 * c >= p.seg[i - 1].tile_end) y = p.seg[i].y + (int64_t)(m0 + m) * p.seg[i].y_sm + 8 * c - p.seg[i - 1].tile_end;
    *reinterpret_cast<u32x4*>(y) = v;
  }
}

// The tile shapes, and what choosing one costs.  `per_cu` workgroups of a shape fit a compute unit; one round of a
// workgroup on every compute unit takes `one` us at K = 2048 (measured with the operands behind the L2; the time is
// proportional to K), a round with all of them `full`.  A product of n tiles then costs about 1.5 us plus its rounds, and
// the shape with the least cost is taken: the small ones while their tiles fit one round, the large ones from there on.
// (M = 777, N = 4608, K = 1536: 16.6 us with 128 x 128 and 8 wavefronts, 18.6 us with 64 x 128, 24.4 us with 64 x 64,
// 17.9 us in the library; M = 64, N = 6144, K = 2048: 7.3 us with 32 x 64, 9.7 us in the library (a KDA decode step's six input projections in
// one launch: 8.3 us, one by one 42 us); M = 8192,
// N = 6144, K = 2048: 155 us with 256 x 256, 178 us with 128 x 128, 141 us in the library.)
// The two smallest are for products whose 32 x 64 tiles leave most compute units idle: what a workgroup then waits for is its own
// K * (bm + bn) operands, at the 60 to 150 GB/s that one compute unit pulls, and smaller tiles on more of them have less of it
// each (weights from memory: M = 64, N = K = 2048: 9.6 us with 32 x 64, 7.1 with 32 x 32, 6.7 with 16 x 32; M = 128: 9.4, 7.1, 9.0;
// M = 16, N = 4608, K = 1536: 8.2, 6.35, 6.2; M = N = K = 256: 2.65, 2.5, 2.4).  16 rows only while all rows of tiles are one panel:
// beyond, the weights are read twice (M = 200, N = K = 512: 3.2, 3.0, 3.3).  32 x 128 does the same for the QKV projection, whose
// narrower tiles would not hold a head of 128 (a layer of 12 heads, 100 tokens: 21.2 us with 64 x 128, 19.5; 160 tokens: 22.6, 21.1; in
// two rounds it loses: 256 tokens 23.7, 28.1); with heads of 64, 32 x 64 stays ahead of it (16 heads, 100 tokens: 14.7, 15.4).
struct ProjTile { int code, bm, bn, bk, per_cu; float one, full; };
constexpr ProjTile kProjTiles[] = {
    {9, 16, 32, 128, 3, 3.6f, 6.6f},      // 2 wavefronts, 4 stages
    {10, 32, 32, 128, 2, 4.0f, 6.6f},     // 4 wavefronts, 4 stages
    {1, 32, 64, 128, 2, 5.8f, 8.0f},      // 4 wavefronts, 3 stages
    {2, 64, 64, 128, 1, 7.2f, 7.2f},      // 8 wavefronts, 4 stages
    {11, 32, 128, 128, 1, 8.3f, 8.3f},    // 8 wavefronts, 3 stages; QKV projection with heads of 128 only
    {3, 64, 128, 128, 1, 10.3f, 10.3f},   // 8 wavefronts, 3 stages
    {4, 64, 128, 64, 2, 12.3f, 19.0f},    // 4 wavefronts, 3 stages
    {5, 128, 128, 64, 1, 15.8f, 15.8f},   // 8 wavefronts, 4 stages
    {6, 128, 128, 64, 2, 20.2f, 25.3f},   // 4 wavefronts, 2 stages
    {7, 256, 256, 64, 1, 42.0f, 42.0f},   // 8 wavefronts, 2 stages
};
constexpr float kJoinedRound = 30.0f;         // the joined tile, 128 x 288, in the same units
template <typename COLUMNS>      // columns(bn): columns of tiles of that width
static int proj_tile(int M, int K, int head, COLUMNS columns, float* its_cost = nullptr) {
  int best = 0;
  float least = 0.f;
  for (const ProjTile& t : kProjTiles) {
    if (K % t.bk != 0 || t.bn % head != 0) continue;    // (head: a tile of the QKV projection holds whole heads)
    if ((t.bm == 16 && M > 8 * t.bm) || (t.code == 11 && head != 128)) continue;
    const int64_t n = (int64_t)((M + t.bm - 1) / t.bm) * columns(t.bn), round = 256 * t.per_cu;
    const int64_t tail = n % round;
    const float cost = (float)(n / round) * t.full + (tail > 256 ? t.full : tail > 0 ? t.one : 0.f);
    if (best == 0 || cost < least) { best = t.code; least = cost; }
  }
  if (its_cost) *its_cost = least;
  return best;
}

// Against the library GEMM: level or ahead (1.0 to 1.7 times as fast) up to about four million outputs, and for short
// rows at any size; 0.9 beyond that.  With the QKV epilogue it replaces the library GEMM and qkv_prep_kernel behind it
// (another read and write of every row, 62 us of 228 us at M = 32768, N = 3072, K = 1024).  That pass is a fixed price per
// output and the library's lead grows with K: ahead at every M up to K = 1536 (whole layer, M = 32768: 640 against 655 us),
// behind from K = 2048 on where the product is large (M = 32768: 1014 against 981 us; M = 8192: 251 against 257 us).
bool proj_segments_wanted(int M, int N, int K) { return K % 64 == 0 && N % 8 == 0 && (K <= 512 || (int64_t)M * N <= 4300000); }
// One product also where its tiles of 128 x 128, of which two fit a compute unit, nearly fill one round: 384 to 512 of them, from 440 for rows of more
// than 1024, none of more than 1536, of which the library's tiles make better use.  Library / this, us (200 sizes, M from 1000, K from 576): 8192 x 1024 x 576 15.0 / 12.1, 8192 x
// 1024 x 1024 19.6 / 16.8, 7000 x 1024 x 1024 18.9 / 17.0, 2176 x 3072 x 1024 (408) 18.8 / 17.9, 29212 x 256 x 1024 20.3 / 19.0, 5760 x 1280 x 1536 (450) 26.3 / 25.4, but 4096
// x 1536 x 1536 (384) 21.9 / 21.8, 1472 x 4096 x 1536 (384) 22.4 / 24.1, 3072 x 2048 x 1280 (384) 20.0 / 21.4; 4096 x 2048 x 2048 32.3 / 30.8, but 6144 x 1024 x 2048 (384) 26.7 /
// 29.1, 25756 x 256 x 1792 30.5 / 38.2; one column of tiles 49152 x 128 x 1024 26.5 / 28.9, 60159 x 128 x 1536 44.9 / 45.9.  With fewer tiles either may be ahead (288: 16.7 /
// 12.7 and 13.3 / 13.7, 352: 25.4 / 28.5), with more the library is (516: 27.8 / 36.3, 17.8 / 21.3).
bool proj_wanted(int M, int N, int K) {
  const int64_t tiles = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
  return proj_segments_wanted(M, N, K) ||
         (K % 64 == 0 && N % 8 == 0 && K <= 1536 && N >= 256 && M >= 1000 && tiles >= (K <= 1024 ? 384 : 440) && tiles <= 512);
}
// A KDA layer's six products of the same rows, N columns in all, in one launch rather than the three large ones by themselves (this kernel's or
// the library's) and the rest in another: one launch for four, and whole rounds of tiles for four that end in part of one.  Layers of 12 heads
// of 64, 8, 12 and 16 of 128, us apart / in one: 3000 rows 128.4 / 114.0; 2300 137.1 / 119.9, 4100 206.6 / 185.1, 7000 (19 million) 282.3 / 276.7;
// 900 104.9 / 93.2, 2800 210.6 / 182.4, 4900 (23 million) 277.9 / 271.5; 1280 148.8 / 126.0, 2300 220.9 / 190.1, 3700 (24 million) 281.9 / 276.0.  Beyond, either
// may be ahead: 8 heads 8100 (26 million) 307 / 310, 9000 385 / 354; 16 heads 4090 (26 million) 296 / 301, 4400 353 / 325, 6000 409 / 422.
bool proj_layer_wanted(int M, int N, int K) { return proj_segments_wanted(M, N, K) || (K % 64 == 0 && N % 8 == 0 && K <= 2048 && (int64_t)M * N <= 25000000); }
bool proj_qkv_wanted(int M, int N, int K) { return K % 64 == 0 && (K <= 1536 || (int64_t)M * N <= 80000000); }

template <int BM, int BN, int WVM, int WVN, int BK, int STAGES, int EPI>
static int launch_proj(ProjParams& p, hipStream_t s) {
  p.MT = (p.M + BM - 1) / BM;
  p.NT = (p.one.N + BN - 1) / BN;
  hipLaunchKernelGGL((proj_kernel<BM, BN, WVM, WVN, BK, STAGES, EPI>), dim3((unsigned)(p.MT * p.NT)), dim3(64 * WVM * WVN), 0, s, p);
  DAISY_CHECK_LAUNCH("proj_kernel");
  return DAISY_OK;
}
template <int BM, int BN, int WVM, int WVN, int BK, int STAGES, int EPI>
static int launch_proj(ProjSegmentsParams& p, hipStream_t s) {
  p.MT = (p.M + BM - 1) / BM;
  p.NT = 0;
  for (int i = 0; i < p.n; ++i) p.seg[i].tile_end = p.NT += (p.seg[i].N + BN - 1) / BN;
  hipLaunchKernelGGL((proj_kernel<BM, BN, WVM, WVN, BK, STAGES, EPI, true>), dim3((unsigned)(p.MT * p.NT)), dim3(64 * WVM * WVN), 0, s, p);
  DAISY_CHECK_LAUNCH("proj_kernel");
  return DAISY_OK;
}

template <int EPI, typename PARAMS>
static int dispatch_proj(int tile, PARAMS& p, hipStream_t s) {
  for (const ProjTile& t : kProjTiles)
    DAISY_CHECK_SUPPORTED(t.code != tile || (p.K % t.bk == 0 && !(EPI == 2 && t.bn % 128 != 0) && !(EPI == 1 && t.bn % 64 != 0) && !(EPI != 2 && t.code == 11) && !(EPI == 3 && t.code == 7)),
                          "proj: tile %d does not serve K=%d with epilogue %d", tile, p.K, EPI);
  if constexpr (EPI != 2) {
    if (tile == 1) return launch_proj<32, 64, 2, 2, 128, 3, EPI>(p, s);
    if constexpr (EPI != 1) {
      if (tile == 10) return launch_proj<32, 32, 2, 2, 128, 4, EPI>(p, s);
      if (tile == 9) return launch_proj<16, 32, 1, 2, 128, 4, EPI>(p, s);
    }
    if (tile == 2) return launch_proj<64, 64, 2, 4, 128, 4, EPI>(p, s);
  }
  if constexpr (EPI == 2) {
    if (tile == 11) return launch_proj<32, 128, 2, 4, 128, 3, EPI>(p, s);
  }
  if constexpr (EPI != 3) {
    if (tile == 7) return launch_proj<256, 256, 2, 4, 64, 2, EPI>(p, s);
  }
  switch (tile) {
    case 3: return launch_proj<64, 128, 2, 4, 128, 3, EPI>(p, s);
    case 4: return launch_proj<64, 128, 2, 2, 64, 3, EPI>(p, s);
    case 5: return launch_proj<128, 128, 4, 2, 64, 4, EPI>(p, s);
    case 6: return launch_proj<128, 128, 2, 2, 64, 2, EPI>(p, s);
    default: DAISY_CHECK_SUPPORTED(false, "proj: no tile %d", tile);
  }
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int proj_linear(const uint16_t* x, int64_t x_sm, const uint16_t* w, int64_t w_sn, const uint16_t* bias,
                uint16_t* y, int64_t y_sm, int M, int N, int K, hipStream_t s, int tile) {
  DAISY_CHECK_ARG(x && w && y && M > 0 && N > 0 && K > 0, "proj_linear: NULL tensor or M=%d, N=%d, K=%d", M, N, K);
  DAISY_CHECK_SUPPORTED(K % 64 == 0 && N % 8 == 0, "proj_linear: K=%d must be a multiple of 64 and N=%d of 8", K, N);
  DAISY_CHECK_ARG(aligned16(x) && aligned16(w) && aligned16(y) && x_sm % 8 == 0 && w_sn % 8 == 0 && y_sm % 8 == 0,
                  "proj_linear: rows must start on 16-byte boundaries");
  DAISY_CHECK_ARG(x_sm < (1 << 22) && w_sn < (1 << 22), "proj_linear: row strides too long");
  ProjParams p{};
  p.one = ProjSegment{x, x_sm, w, w_sn, bias, y, y_sm, N, 0}; p.M = M; p.K = K;
  return dispatch_proj<0>(tile ? tile : proj_tile(M, K, 8, [&](int bn) { return (N + bn - 1) / bn; }), p, s);
}

int proj_segments(const ProjSegment* seg, int n, int M, int K, hipStream_t s, int tile, const KdaGates* gates) {
  DAISY_CHECK_ARG(seg && n >= 1 && n <= kMaxSegments && M > 0 && K > 0, "proj_segments: %d products, M=%d, K=%d", n, M, K);
  DAISY_CHECK_SUPPORTED(K % 64 == 0, "proj_segments: K=%d must be a multiple of 64", K);
  ProjSegmentsParams p{};
  for (int i = 0; i < n; ++i) {
    const ProjSegment& g = seg[i];
    DAISY_CHECK_ARG(g.x && g.w && g.y && g.N > 0, "proj_segments: NULL tensor or N=%d", g.N);
    DAISY_CHECK_ARG(aligned16(g.x) && aligned16(g.w) && aligned16(g.y) && g.x_sm % 8 == 0 && g.w_sn % 8 == 0 && g.y_sm % 8 == 0 &&
                        g.y_sm >= ((g.N + 7) & ~7) && g.x_sm < (1 << 22) && g.w_sn < (1 << 22),
                    "proj_segments: rows must start on 16-byte boundaries, with room for whole 16-byte pieces");
    p.seg[i] = g;
  }
  p.n = n; p.M = M; p.K = K;
  auto columns = [&](int bn) {
    int c = 0;
    for (int i = 0; i < n; ++i) c += (seg[i].N + bn - 1) / bn;
    return c;
  };
  // All products in one tile across (code 12): the same rows of x, no bias, together at most a tile wide.  By cost, which is a round of its
  // workgroups (30 at K = 2048, as proj_tile counts); 128 + 128 + 16 columns, the best other tile / this one: K = 2048 and 20000 rows 31.5 / 34.8,
  // 22000 48.5 / 35.5, 40000 59.3 / 68.1, 45000 75.5 / 69.1, 131072 224 / 183 us; K = 1024, 24000 rows 26.2 / 22.6, 65536 50.8 / 46.7: ahead where
  // the others need another round, from some 21000 rows to 32768 and again from some 45000, level between, where they are taken.  Narrower ones alike (K = 2048,
  // 24000 rows, 64 + 64 + 16 columns 41.8 / 34.9, a lone product of 280 46.1 / 34.9; of 128 or 256 the others are never dearer and are taken).  Of
  // short rows the fixed part of a round is too much: K = 512, 32768 rows 19.6 / 17.1, but 45000 26.3 / 28.2; K = 256, 131072 37.5 / 44.9.
  int across = 0;
  bool joined = !gates && ((!tile && K >= 1024) || tile == 12);
  for (int i = 0; i < n; ++i) {
    across += (seg[i].N + 7) & ~7;
    joined = joined && seg[i].x == seg[0].x && seg[i].x_sm == seg[0].x_sm && !seg[i].bias;
  }
  joined = joined && across <= kJoinedColumns;
  DAISY_CHECK_SUPPORTED(joined || tile != 12, "proj_segments: tile 12 does not serve these products");
  float cost = 0.f;
  const int by_size = tile ? tile : proj_tile(M, K, 8, columns, &cost);
  const int row_tiles = (M + kJoinedRows - 1) / kJoinedRows;
  if (joined && (tile || kJoinedRound * ((row_tiles + 255) / 256) < cost)) {
    int at = 0;
    for (int i = 0; i < n; ++i) p.seg[i].tile_end = at += (seg[i].N + 7) & ~7;
    p.NT = across / 8;
    hipLaunchKernelGGL(proj_joined_kernel, dim3((unsigned)row_tiles), dim3(512), 0, s, p);
    DAISY_CHECK_LAUNCH("proj_joined_kernel");
    return DAISY_OK;
  }
  if (!gates) return dispatch_proj<0>(by_size, p, s);
  DAISY_CHECK_ARG(gates->A_log && gates->dt_bias && gates->logits && gates->beta && gates->H > 0 && gates->Dk % 8 == 0 && seg[0].N == gates->H * gates->Dk,
                  "proj_segments: gate of %d heads of %d channels on a product of %d", gates->H, gates->Dk, seg[0].N);
  p.gates = *gates;
  // (no gate with tile 7: of tile 6 two workgroups fit a compute unit, and the gate of one runs beside the copies of the other;
  // 32768 rows, whole layer: 1674 against 1680 us)
  return dispatch_proj<3>(!tile && by_size == 7 ? 6 : by_size, p, s);
}

int proj_qkv(const uint16_t* x, int64_t x_sm, const uint16_t* w, int64_t w_sn, const QkvEpilogue& e,
             int B, int K, int D, hipStream_t s, int tile) {
  const int M = B * e.T, N = 3 * e.H * D;
  DAISY_CHECK_ARG(x && w && e.q && e.k && e.v && e.cos && e.sin && M > 0 && K > 0, "proj_qkv: NULL tensor or empty shape");
  DAISY_CHECK_SUPPORTED(K % 64 == 0 && (D == 64 || D == 128), "proj_qkv: K=%d must be a multiple of 64 and D=%d 64 or 128", K, D);
  DAISY_CHECK_ARG(aligned16(x) && aligned16(w) && aligned16(e.q) && aligned16(e.k) && aligned16(e.v) && aligned16(e.ve) &&
                      aligned16(e.cos) && aligned16(e.sin) && x_sm % 8 == 0 && w_sn % 8 == 0,
                  "proj_qkv: tensors must be 16-byte aligned");
  const int64_t st[] = {e.q_sb, e.q_st, e.q_sh, e.k_sb, e.k_st, e.k_sh, e.v_sb, e.v_st, e.v_sh, e.ve_sb, e.ve_st, e.ve_sh};
  for (int64_t v : st) DAISY_CHECK_ARG(v % 8 == 0, "proj_qkv: strides must be multiples of 8 elements");
  DAISY_CHECK_ARG(x_sm < (1 << 22) && w_sn < (1 << 22), "proj_qkv: row strides too long");
  ProjParams p{};
  p.one = ProjSegment{x, x_sm, w, w_sn, nullptr, nullptr, 0, N, 0}; p.M = M; p.K = K; p.e = e;
  if (!tile) tile = proj_tile(M, K, D, [&](int bn) { return (N + bn - 1) / bn; });
  return D == 128 ? dispatch_proj<2>(tile, p, s) : dispatch_proj<1>(tile, p, s);
}

}  // namespace daisy
