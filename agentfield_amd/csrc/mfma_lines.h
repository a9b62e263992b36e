// Lines of row-major bf16 matrices (128 bytes = 64 elements of a row) in LDS, and MFMA
// operands from them: shared by the GEMMs that stream weights.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8r;
typedef __attribute__((address_space(3))) char lds_b;
typedef __attribute__((address_space(3))) s16x8 lds_v8;

__device__ __forceinline__ bf16x8r as_bf16x8r(s16x8 v) {
  union { s16x8 s; bf16x8r b; } u;
  u.s = v;
  return u.b;
}

// 8 rows x 128 bytes of a row-major matrix into linear LDS: lane l brings chunk
// (l & 7) ^ (row & 7) of row l >> 3, so that chunk c of row r sits at slot
// c ^ (r & 7).
template <int AUX>
__device__ __forceinline__ void load_line8(const u16* src, lds_b* dst) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) uint32_t*)src,
      (__attribute__((address_space(3))) uint32_t*)dst, 16, 0, AUX);
}
constexpr int STREAM = 2, KEEP = 0;   // AUX: nontemporal, cached

// s_waitcnt operand: all but n of a wave's vector loads have landed
constexpr int vmcnt_only(int n) { return (n & 15) | (n >> 4) << 14 | 0x0f70; }

// operand fragment: lane (r = lane & 15, q = lane >> 4) gets k = 32 h + 8 q .. +8
// of row r of a 16-row piece
__device__ __forceinline__ bf16x8r frag(const lds_b* piece, int h) {
  const int lane = threadIdx.x & 63, r = lane & 15;
  const int c = (h * 4 + (lane >> 4)) ^ (r & 7);
  return as_bf16x8r(*reinterpret_cast<const lds_v8*>(piece + r * 128 + c * 16));
}

// All but n groups of PER of a wave's loads have landed (n <= 4), its LDS reads are
// done, and so it is for every wave of the block.  By builtins: the compiler has to
// know that the operands are there, or it waits for the next ones as well.
template <int PER>
__device__ __forceinline__ void meet(int n) {
  asm volatile("" ::: "memory");
  if (n >= 4) __builtin_amdgcn_s_waitcnt(vmcnt_only(4 * PER) & ~0x0f00);
  else if (n == 3) __builtin_amdgcn_s_waitcnt(vmcnt_only(3 * PER) & ~0x0f00);
  else if (n == 2) __builtin_amdgcn_s_waitcnt(vmcnt_only(2 * PER) & ~0x0f00);
  else if (n == 1) __builtin_amdgcn_s_waitcnt(vmcnt_only(PER) & ~0x0f00);
  else __builtin_amdgcn_s_waitcnt(vmcnt_only(0) & ~0x0f00);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
