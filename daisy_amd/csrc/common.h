// Shared device/host helpers for the gfx950 attention kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "internal.h"

namespace daisy {

// ---- vector types ---------------------------------------------------------
typedef __bf16 bf16_t;
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.4426950408889634f;

// ---- bf16 <-> fp32 ----------------------------------------------------------
// A bf16 is the high half of an fp32, so widening is a shift.
__device__ __forceinline__ float bf16lo_to_f32(uint32_t packed) { return __uint_as_float(packed << 16); }
__device__ __forceinline__ float bf16hi_to_f32(uint32_t packed) { return __uint_as_float(packed & 0xffff0000u); }

// Round-to-nearest-even pack of two fp32 into one dword of bf16 (lo = a, hi = b).
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  f32x2 x = {a, b};
  bf16x2 y = __builtin_convertvector(x, bf16x2);
  return __builtin_bit_cast(uint32_t, y);
}
__device__ __forceinline__ float round_bf16(float a) {
  return bf16lo_to_f32(pack_bf16x2(a, 0.f));
}

// The value of a gate on the device.
__device__ __forceinline__ float gate_value(const GateSource& g) {
  if (g.kind == GateSource::kValue) return *(const float*)g.p;
  const float x = g.kind == GateSource::kLogitBf16 ? bf16lo_to_f32(*(const uint16_t*)g.p) : *(const float*)g.p;
  return round_bf16(1.f / (1.f + expf(-x)));
}

// Unpack 8 bf16 held in a 16-byte register quad into 8 floats.
__device__ __forceinline__ void unpack8(const u32x4& r, float* f) {
  f[0] = bf16lo_to_f32(r.x); f[1] = bf16hi_to_f32(r.x);
  f[2] = bf16lo_to_f32(r.y); f[3] = bf16hi_to_f32(r.y);
  f[4] = bf16lo_to_f32(r.z); f[5] = bf16hi_to_f32(r.z);
  f[6] = bf16lo_to_f32(r.w); f[7] = bf16hi_to_f32(r.w);
}
__device__ __forceinline__ u32x4 pack8(const float* f) {
  u32x4 r;
  r.x = pack_bf16x2(f[0], f[1]); r.y = pack_bf16x2(f[2], f[3]);
  r.z = pack_bf16x2(f[4], f[5]); r.w = pack_bf16x2(f[6], f[7]);
  return r;
}

// RoPE on one pair (x1 at channel i, x2 at channel i + D/2):
//   y1 = x1*cos + x2*sin,  y2 = -x1*sin + x2*cos.
// Products and sum are rounded separately (no fused multiply-add), the way an
// elementwise tensor library evaluates the expression, so that the bf16 result
// is bit-identical to it.
__device__ __forceinline__ float rope_lo(float x1, float x2, float c, float s) {
#pragma clang fp contract(off)
  const float a = x1 * c;
  const float b = x2 * s;
  return a + b;
}
__device__ __forceinline__ float rope_hi(float x1, float x2, float c, float s) {
#pragma clang fp contract(off)
  const float a = x1 * -s;
  const float b = x2 * c;
  return a + b;
}

// Element access for kernels templated on the tensor element: uint16_t = bf16 bits, float = fp32.
// round_elem rounds a computed value the way a tensor of that element type would hold it.
template <typename E> __device__ __forceinline__ float load_elem(const E* p, int64_t i);
template <> __device__ __forceinline__ float load_elem<uint16_t>(const uint16_t* p, int64_t i) { return bf16lo_to_f32(p[i]); }
template <> __device__ __forceinline__ float load_elem<float>(const float* p, int64_t i) { return p[i]; }
template <typename E> __device__ __forceinline__ void store_elem(E* p, int64_t i, float x);
template <> __device__ __forceinline__ void store_elem<uint16_t>(uint16_t* p, int64_t i, float x) {
  p[i] = (uint16_t)(pack_bf16x2(x, 0.f) & 0xffffu);
}
template <> __device__ __forceinline__ void store_elem<float>(float* p, int64_t i, float x) { p[i] = x; }
template <typename E> __device__ __forceinline__ float round_elem(float x);
template <> __device__ __forceinline__ float round_elem<uint16_t>(float x) { return round_bf16(x); }
template <> __device__ __forceinline__ float round_elem<float>(float x) { return x; }

// log(1 + e^v) = max(v, 0) + log1p(t) with t = exp(-|v|); above 17 it is v in fp32.
// log1p(t) = 2 artanh(s), s = t / (2 + t) <= 1/3; 2 artanh(s) / s = 2 + 2 s^2 / 3 + ... as a polynomial of degree 4 in s^2, found by
// exchange of the extrema of its error over 0 .. 1/9; with the coefficients rounded to fp32, the last one to 2, the error is -7.8e-9 to 1.2e-9 of the value
// (the series as far as s^12 has 1.5e-8 and two terms more): no branch, one reciprocal.  The library's logarithm of 1 + t, with a series below t = 1/64, is some forty instructions under two execution masks
// and has an error up to 3.8e-6 of the value where 1 + t is rounded (here 2.3e-7; the whole softplus over -30 .. 30 against 64
// bits: 4.0e-6 -> 1.8e-6, the exponential's).
__device__ __forceinline__ float softplus(float v) {
  const float t = __builtin_amdgcn_exp2f(-fabsf(v) * kLog2e);
  const float s = t * __builtin_amdgcn_rcpf(2.f + t), z = s * s;
  float l = fmaf(z, 0.28178334f, 0.279606f);
  l = fmaf(z, l, 0.4002491f);
  l = fmaf(z, l, 0.66666317f);
  l = fmaf(z, l, 2.f);
  return fmaf(l, s, fmaxf(v, 0.f));
}
// With slope `beta`, linear above the threshold.
__device__ __forceinline__ float softplus(float v, float beta, float threshold, float inv_beta) {
  const float bx = v * beta;
  return (bx > threshold) ? v : softplus(bx) * inv_beta;
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// ---- cross-lane sums with DPP (no LDS traffic) -------------------------------
template <int CTRL>
__device__ __forceinline__ float dpp_move(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) { return x + dpp_move<CTRL>(x); }

// x and its value in the neighbouring row of 16 lanes (rows 0 and 1, 2 and 3) or in the other half of the wavefront.
struct LanePair { float x, y; };
__device__ __forceinline__ LanePair row_pair(float x) {
  const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false));
  return {__uint_as_float(t.x), __uint_as_float(t.y)};
}
__device__ __forceinline__ LanePair half_pair(float x) {
  const u32x2 t = __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false));
  return {__uint_as_float(t.x), __uint_as_float(t.y)};
}

// Sum over the LPR consecutive lanes that share a cache row; every lane of the
// group ends with the total.
template <int LPR>
__device__ __forceinline__ float group_sum(float x) {
  x = dpp_add<0xB1>(x);                     // quad_perm [1,0,3,2]   (xor 1)
  x = dpp_add<0x4E>(x);                     // quad_perm [2,3,0,1]   (xor 2)
  if (LPR >= 8) x = dpp_add<0x141>(x);      // row_half_mirror       (joins the two quads of 8 lanes)
  if (LPR >= 16) x = dpp_add<0x128>(x);     // row_ror 8             (joins the two halves of 16 lanes)
  if (LPR >= 32) { const LanePair t = row_pair(x); x = t.x + t.y; }
  return x;
}
__device__ __forceinline__ float wave_sum(float x) {
  const LanePair t = half_pair(group_sum<32>(x));
  return t.x + t.y;
}

// ---- asynchronous global -> LDS copies ------------------------------------------
// Asynchronous 16-byte global -> LDS copy that bypasses the vector registers
// (global_load_lds_dwordx4): lane i of the wavefront deposits the 16 bytes at
// gbase + byte_off at LDS address lds_addr + 16*i.  gbase and lds_addr are wavefront-uniform.
// Issued as inline assembly so that the compiler does not serialise later LDS reads of the
// OTHER buffer behind it; the caller waits with s_waitcnt vmcnt(0) before publishing the tile.
template <bool STREAMED = false>
__device__ __forceinline__ void copy16_to_lds_async(const uint16_t* gbase, int byte_off, uint32_t lds_addr) {
  if (STREAMED)
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" :: "v"(byte_off), "s"(gbase), "s"(lds_addr) : "memory");
  else
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(byte_off), "s"(gbase), "s"(lds_addr) : "memory");
}
// N KiB in a row: the instruction's offset moves the global and the LDS address alike, four copies per address.
template <int N>
__device__ __forceinline__ void copy_kib_to_lds_async(const char* gbase, int byte_off, uint32_t lds_addr) {
  if constexpr (N >= 4) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:2048\n\tglobal_load_lds_dwordx4 %0, %1 offset:3072"
                 :: "v"(byte_off), "s"(gbase), "s"(lds_addr) : "memory");
    if constexpr (N > 4) copy_kib_to_lds_async<N - 4>(gbase + 4096, byte_off, lds_addr + 4096);
  } else if constexpr (N == 3) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:2048"
                 :: "v"(byte_off), "s"(gbase), "s"(lds_addr) : "memory");
  } else if constexpr (N == 2) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024"
                 :: "v"(byte_off), "s"(gbase), "s"(lds_addr) : "memory");
  } else {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" :: "v"(byte_off), "s"(gbase), "s"(lds_addr) : "memory");
  }
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return (uint32_t)(size_t)(__attribute__((address_space(3))) const void*)p;
}

// Stores 16 bytes through the L2 at once (policy sc1).  What a kernel leaves dirty in the L2 is written back at its end, behind its last
// workgroup: its last round's results, all of them for a launch of one round.  The store's data registers are free one wait state
// behind it, which the block holds.  us, a plain store / this: a layer's prefill of 777 rows, 12 heads of 128, QKV projection 37.5 / 37.0,
// attention output and output projection 36.8 / 36.5; of 8 x 4096 rows, 8 heads, 400 / 396; 4096 x 2048 x 512 17.2 / 16.0; products of a decode
// batch, 9 to 512 rows, level (0.99 to 1.02) up to 2048 columns, 128 to 512 rows of 8192 x 1536 3 % ahead.
__device__ __forceinline__ void store_through(void* at, const u32x4& v) {
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(at), "v"(v) : "memory");
}

// ---- LDS layout ---------------------------------------------------------------
// Swizzle of a row's 16-byte pieces: the 16 lanes that a 16-byte LDS read serves together must fall into 16 different slots
// of the 256-byte bank window.  Those are not 16 consecutive lanes but lanes 0-3, 12-15 and 20-27 (and so on): rows 0-3
// and 12-15 of one k-group with rows 4-11 of the next.  For rows of 64 bytes (row >> 2) & 3 itself puts two of them into every
// slot (256 of 930 LDS cycles per chunk of the KDA chain); the permutation 0 2 3 1 of it puts one.  Rows of 256, 128 and 64 bytes:
template <int ROWBYTES> __host__ __device__ constexpr int piece_swizzle(int row) {
  return ROWBYTES == 256 ? (row & 15) : ROWBYTES == 128 ? ((row >> 1) & 7) : ((row >> 3) & 1) | (((row >> 2) ^ (row >> 3)) & 1) << 1;
}

// ---- host-side error plumbing --------------------------------------------
void set_error(const char* fmt, ...);

#define DAISY_CHECK_ARG(cond, ...)            \
  do {                                        \
    if (!(cond)) {                            \
      daisy::set_error(__VA_ARGS__);          \
      return DAISY_ERR_INVALID_ARGUMENT;      \
    }                                         \
  } while (0)

#define DAISY_CHECK_SUPPORTED(cond, ...)      \
  do {                                        \
    if (!(cond)) {                            \
      daisy::set_error(__VA_ARGS__);          \
      return DAISY_ERR_UNSUPPORTED;           \
    }                                         \
  } while (0)

// Checks the launch error state after a kernel launch.
#define DAISY_CHECK_LAUNCH(what)                                                   \
  do {                                                                             \
    hipError_t e_ = hipGetLastError();                                             \
    if (e_ != hipSuccess) {                                                        \
      daisy::set_error("%s: launch failed: %s", what, hipGetErrorString(e_));      \
      return DAISY_ERR_LAUNCH;                                                     \
    }                                                                              \
  } while (0)

}  // namespace daisy
