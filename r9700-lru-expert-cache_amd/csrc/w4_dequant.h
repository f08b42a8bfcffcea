// The W4 format's operand types, MFMA and dequantization, shared by the W4 lm_head kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gemm_common.h"
#include "wave.h"

namespace rlu {
namespace w4 {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

constexpr int MAXGQ = 8;       // groups per wave: K / 128 / split <= 8, so K <= 4096
constexpr int MAXK = 4096;     // x in LDS: 16 rows x K bf16 = 2 K * 16 bytes
constexpr int BUF_WORD3 = 0x00020000;   // raw buffer descriptor word 3 on gfx9 (no format)
constexpr int SLC = 2;                  // buffer cache policy: streaming (the codes are read once)

__device__ __forceinline__ v4f mfma_bf16(v4u a, v4u b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a),
                                                 __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
}

// (v & mask) | magic in one VALU op; the mask rides in an SGPR and the magic in a VGPR (a VOP3
// op on gfx9 takes no literal and one scalar operand), which the compiler would not pick itself
__device__ __forceinline__ unsigned and_or(unsigned v, unsigned mask, unsigned magic) {
  unsigned r;
  asm volatile("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(mask), "v"(magic));
  return r;
}

// 64-bit right shift by a constant, as one instruction (the compiler splits a 64-bit shift
// into two 32-bit ones, alignbit + shift)
template <int S>
__device__ __forceinline__ unsigned long long shr64(unsigned long long v) {
  unsigned long long r;
  asm volatile("v_lshrrev_b64 %0, %1, %2" : "=v"(r) : "i"(S), "v"(v));
  return r;
}

// the 16 bf16 pairs (128 + q_2t, 128 + q_2t+1) of one tile lane: b[i] feeds MFMA i. One 64-bit
// shift serves two dwords: the bits that cross into the low dword land at bit 20 and above,
// which the mask drops.
__device__ __forceinline__ void dequant(v4u w, unsigned mask, unsigned magic, v4u* b) {
  const unsigned long long p0 = ((unsigned long long)w.y << 32) | w.x;
  const unsigned long long p1 = ((unsigned long long)w.w << 32) | w.z;
  const unsigned long long a4 = shr64<4>(p0), a8 = shr64<8>(p0), a12 = shr64<12>(p0);
  const unsigned long long c4 = shr64<4>(p1), c8 = shr64<8>(p1), c12 = shr64<12>(p1);
  b[0] = v4u{and_or(w.x, mask, magic), and_or((unsigned)a4, mask, magic),
             and_or((unsigned)a8, mask, magic), and_or((unsigned)a12, mask, magic)};
  b[1] = v4u{and_or(w.y, mask, magic), and_or((unsigned)(a4 >> 32), mask, magic),
             and_or((unsigned)(a8 >> 32), mask, magic), and_or((unsigned)(a12 >> 32), mask, magic)};
  b[2] = v4u{and_or(w.z, mask, magic), and_or((unsigned)c4, mask, magic),
             and_or((unsigned)c8, mask, magic), and_or((unsigned)c12, mask, magic)};
  b[3] = v4u{and_or(w.w, mask, magic), and_or((unsigned)(c4 >> 32), mask, magic),
             and_or((unsigned)(c8 >> 32), mask, magic), and_or((unsigned)(c12 >> 32), mask, magic)};
}

}  // namespace w4
}  // namespace rlu
