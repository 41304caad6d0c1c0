// Shared device/host helpers for the gfx950 ring-attention step kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "../../include/mercury_hip.h"

namespace mhip {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2;

constexpr int kMaxGroup = MHIP_MAX_GROUP;     // blocks of a step in one launch,
constexpr int kGroupWorkgroups = 2048;        // and their workgroups: eight rounds on 256 CUs

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

// Two fp32 -> one dword of two bf16 (round to nearest even), low half = a.
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  f32x2 v = {a, b};
  bf16x2 r = __builtin_convertvector(v, bf16x2);
  return __builtin_bit_cast(uint32_t, r);
}

__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// max / sum of x over the lane pair (l, l ^ 32).  v_permlane32_swap exchanges the upper half of
// its first operand with the lower half of its second, so with both operands = x every lane ends
// up holding {own value, partner's value} in the two results (in an order that depends on the
// half) -- a symmetric combine needs no lane test.  The two results are taken out as ints first:
// __builtin_bit_cast applied directly to r[1] reads r[0] with this compiler.
__device__ __forceinline__ void pair_exchange(float x, float& a, float& b) {
  const int xi = __float_as_int(x);
  auto r = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
  const int r0 = r[0], r1 = r[1];
  a = __int_as_float(r0);
  b = __int_as_float(r1);
}
__device__ __forceinline__ float pair_max(float x) {
  float a, b;
  pair_exchange(x, a, b);
  return fmaxf(a, b);
}
__device__ __forceinline__ float pair_sum(float x) {
  float a, b;
  pair_exchange(x, a, b);
  return a + b;
}

// the same over the lanes l, l ^ 16, l ^ 32 and l ^ 48
__device__ __forceinline__ float quad_max(float x) {
  x = pair_max(x);
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x), false, false);
  const unsigned a = r[0], b = r[1];
  return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}
__device__ __forceinline__ float quad_sum(float x) {
  x = pair_sum(x);
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x), __builtin_bit_cast(unsigned, x), false, false);
  const unsigned a = r[0], b = r[1];
  return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}

// sum of x over the lane's group of 16, in all of its lanes
__device__ __forceinline__ float row16_sum(float x) {
  auto rotated = [](float v, auto n) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + decltype(n)::value, 0xf, 0xf, false));
  };
  x += rotated(x, std::integral_constant<int, 8>{});
  x += rotated(x, std::integral_constant<int, 4>{});
  x += rotated(x, std::integral_constant<int, 2>{});
  x += rotated(x, std::integral_constant<int, 1>{});
  return x;
}

// and over its group of 8
__device__ __forceinline__ float row8_sum(float x) {
  auto permuted = [](float v, auto ctrl) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), decltype(ctrl)::value, 0xf, 0xf, false));
  };
  x += permuted(x, std::integral_constant<int, 0xb1>{});     // the other of a pair
  x += permuted(x, std::integral_constant<int, 0x4e>{});     // the other pair of four
  x += permuted(x, std::integral_constant<int, 0x141>{});    // the other four of eight, mirrored
  return x;
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float fast_log2(float x) { return __builtin_amdgcn_logf(x); }

// Buffer descriptor over `bytes` bytes at `base`, as four scalar words: loads whose offset (vector +
// scalar part) falls past the end return zero.
__device__ __forceinline__ u32x4 rsrc_words(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)base;
  u32x4 r;
  // wavefront-uniform by construction; readfirstlane makes that visible to the register allocator
  r[0] = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r[1] = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
  r[2] = __builtin_amdgcn_readfirstlane(bytes);
  r[3] = 0x00020000u;
  return r;
}

// Global -> LDS copy of 16 (or 4) bytes per lane without passing through registers: lane l's bytes land
// at LDS address `lds_addr` + 16 l (+ 4 l); the base is wavefront-uniform and travels in M0.  Lanes whose
// offset is out of the descriptor's range write zeros.  Completion is counted by vmcnt.  Written as
// inline assembly so that the compiler's own wait-count insertion does not see the copies: it would
// otherwise wait for all of them before every transposing LDS read.  The kernels place the waits by hand.
// M0 is written here and is not on the clobber list: the compiler treats it as a reserved register, warns
// that a clobber of it "may not be preserved" and ignores it.  That is safe as long as nothing else in a
// kernel that copies this way needs M0 (no register-indexed moves, no s_sendmsg, no GWS, no other LDS-direct
// load): every copy sets M0 itself immediately before its load, so it never relies on an earlier value.
__device__ __forceinline__ void copy16_to_lds(u32x4 rsrc, uint32_t lds_addr, int voffset, int soffset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voffset), "s"(rsrc),
                  "s"(__builtin_amdgcn_readfirstlane(soffset)) : "memory");
}
__device__ __forceinline__ void copy4_to_lds(u32x4 rsrc, uint32_t lds_addr, int voffset, int soffset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
               :: "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voffset), "s"(rsrc),
                  "s"(__builtin_amdgcn_readfirstlane(soffset)) : "memory");
}

// The same with a 64-bit address per lane and no range check: every address has to be readable.
__device__ __forceinline__ void copy16_to_lds(const void* src, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(src) : "memory");
}

// The same for 4 bytes per lane.
__device__ __forceinline__ void copy4_to_lds(const void* src, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off"
               :: "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(src) : "memory");
}

// Tiles copied that way are rows of 256 bytes (128 bf16) without padding; chunk c (16 bytes) of row r is
// kept at chunk position c ^ lds_row_swizzle(r).  With this map both access patterns of the MFMA operand
// reads are free of bank conflicts: 32 consecutive rows x one chunk (ds_read_b128 of a row-major operand)
// and 8 rows x 4 consecutive chunks (ds_read_b64_tr_b16 of a transposed operand).
__device__ __forceinline__ constexpr int lds_row_swizzle(int row) { return ((row & 3) << 2) | ((row >> 2) & 3); }

// The same for 16 x 16 MFMA tiles, which read 16 rows x 4 chunks of a row-major operand and 16 rows x 2 consecutive chunks of a
// transposed one.  ds_read_b128 serves lanes 0-3, 12-15 and 20-27 of a half-wave together, which are rows 0-3 and 12-15 of one chunk
// and rows 4-11 of the next; ds_read_b64_tr_b16 half a wave, 8 consecutive rows.  With the map above both meet in the same banks.
// (The dQ pass of 4096 x 4096 H32 loses 51 M LDS cycles of 103 M to conflicts with that one, 0.4 M with this.  The forward kernel is
// no faster for it, 1572 us / 1570 a step of 8 such blocks, and keeps the map above.)
__device__ __forceinline__ constexpr int lds_row_swizzle_16(int row) {
  return ((row & 3) << 2) | (((row >> 1) ^ (row >> 2)) & 2) | ((row >> 3) & 1);
}

// Division of a number below 2^31 by a divisor the host knows: a multiplication and a shift on the scalar unit instead of
// some twenty dependent instructions through the vector unit's reciprocal.  With s = ceil(log2 d) and
// mul = floor(2^32 (2^s - d) / d) + 1 the quotient is (mulhi(n, mul) + n) >> s (Granlund and Montgomery, 1994).
struct Divisor {
  uint32_t mul, shift, d;
  Divisor() = default;
  explicit Divisor(int divisor) : d((uint32_t)(divisor > 0 ? divisor : 1)) {
    shift = d > 1 ? 32 - __builtin_clz(d - 1) : 0;
    mul = (uint32_t)(((uint64_t(1) << 32) * ((uint64_t(1) << shift) - d)) / d + 1);
  }
  __device__ __forceinline__ int quotient(int n, int& rest) const {
    const uint32_t q = (__umulhi((uint32_t)n, mul) + (uint32_t)n) >> shift;
    rest = n - (int)(q * d);
    return (int)q;
  }
  __device__ __forceinline__ int quotient(int n) const { return (int)((__umulhi((uint32_t)n, mul) + (uint32_t)n) >> shift); }
};

// The arguments a workgroup of a forward kernel needs before its first copy are in registers where this stands: the
// compiler otherwise reads each one shortly before its first use, five or six rounds of scalar loads, every one of which
// misses the cache in a fresh workgroup.  With this and without divisions a block takes 0.25 - 0.5 us less (512 x 512 B4 H5
// 9.6 -> 9.3, 1024 x 1024 H32 20.7 -> 20.4, 2048 x 2048 H32 62.5 -> 61.9).  (One statement: separate ones are waited for
// one by one.)
template <bool CAUSAL, class P>
__device__ __forceinline__ void load_now(const P& p, const float& scale) {
  const Divisor& by = CAUSAL ? p.by_order : p.by_q_tiles;
  asm volatile("" ::"s"(p.per_xcd), "s"(p.total), "s"(p.blocks), "s"(p.nq_tiles), "s"(p.heads_per_xcd), "s"(p.Sq), "s"(p.Sc),
               "s"(p.D), "s"(by.mul), "s"(by.shift), "s"(by.d), "s"(p.by_hq.mul), "s"(p.by_hq.shift), "s"(p.by_hq.d),
               "s"(p.by_group.mul), "s"(p.by_group.shift), "s"(p.q), "s"(p.k0), "s"(p.v0), "s"(p.q_sb), "s"(p.q_ss),
               "s"(p.q_sh), "s"(p.k_sb), "s"(p.k_ss), "s"(p.k_sh), "s"(p.v_sb), "s"(p.v_ss), "s"(p.v_sh), "s"(scale));
}

// Estimated time (us) of a launch of n workgroups of t tile steps each, one workgroup per CU at a time: `fixed` per workgroup
// and `step` per tile, plus `busy` times the share of the CUs at work (clock and L2).
struct LaunchCost { float fixed, step, busy; };
inline float rounds_time(float n, float t, const LaunchCost& c) {
  const float full = (float)(int64_t)(n / 256.f), part = n / 256.f - full;
  return full * (c.fixed + t * (c.step + c.busy)) + (part > 0.f ? c.fixed + t * (c.step + part * c.busy) : 0.f);
}
// and of the fold of a step's results, which is not needed for one
inline float fold_time(int results, int B, int Sq, int Hq, int D) {
  return results > 1 ? 4.f + (results + 1) * (2.f * B * Sq * Hq * D) / 5.3e6f : 0.f;
}

// lds_row_swizzle for rows of 128 bytes (64 bf16), of which two share the 256 bytes that cover all banks: 16 consecutive rows x one
// chunk take each of the 16 places once, and so do 4 rows x 4 consecutive chunks.
__device__ __forceinline__ constexpr int lds_half_row_swizzle(int row) { return (((row >> 1) & 1) << 2) | ((row >> 2) & 3); }

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline int launch_status() {
  return hipGetLastError() == hipSuccess ? MHIP_OK : MHIP_ELAUNCH;
}

}  // namespace mhip
