// gemm_common.hpp - what the dequant-GEMM's kernels share (gemm.hip, gemm_n128.hip): the call's parameters, the exact
// dequant of a code word to fp16, and the activations' activation function.
#pragma once
#include "common.hpp"

namespace p0 {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(4)));   // a 16-byte load at 4-byte alignment
typedef uint32_t u32x4n __attribute__((ext_vector_type(4)));               // 16-byte aligned (LDS, registers)
typedef float float16v __attribute__((ext_vector_type(16)));

struct GemmP {
  const uint8_t* w; int64_t wG; int64_t Nw;
  const _Float16* x; int64_t ldx;   // fp16 X' rows (the caller's, or the staging workspace), k offset folded in
  int M, N, K;
  int64_t wr0, wr1, wk0;
  int epi;
  uint8_t* y; int64_t ldy, ny0;
  const float* ev; int64_t evOff;
  const float* bv; int64_t bvOff, bvUp;
  int act, store, res;
  // heads epilogue: head-major rows of Ltot, query / key head counts, eps, RoPE mode and table
  int64_t hLtot, hRow0;
  int hq, hkv, hrope;
  float heps;
  const float* rope;
};

__device__ __forceinline__ _Float16 to_h(float v) { return (_Float16)v; }   // RNE
__device__ __forceinline__ uint32_t pack_h2(float lo, float hi) {
  return (uint32_t)__builtin_bit_cast(uint16_t, to_h(lo)) | ((uint32_t)__builtin_bit_cast(uint16_t, to_h(hi)) << 16);
}

__device__ __forceinline__ float act_f(const GemmP& p, float g) {
  if (p.act == P0_ACT_GELU) {
    float t = 0.7978845608f * (g + 0.044715f * g * g * g);
    t = fminf(15.0f, fmaxf(-15.0f, t));
    return g * 0.5f * (1.0f + tanhf(t));
  }
  return g / (1.0f + __expf(-g));
}

// q s + m is exact in fp32 for every q in [0, 15] when the fp16 exponent fields a = max(e_s, 1), b = max(e_m, 1)
// satisfy -12 <= a - b <= 8 (the sum then spans at most 24 bits), or when s or m is zero
__device__ __forceinline__ bool pk_exact(uint32_t sm) {
  const int es = (sm >> 10) & 31, em = (sm >> 26) & 31;
  const int a = es > 1 ? es : 1, b = em > 1 ? em : 1;
  const bool zero = (sm & 0x7FFFu) == 0 || (sm & 0x7FFF0000u) == 0;
  return zero || (a - b <= 8 && a - b >= -12);
}

// One q4 code word (k = 8 w .. 8 w + 7 of one row) -> 8 fp16 weights in k order, each fl16(fl32(q s + m)).
// Fast path: the byte j of the word holds k 2j (low nibble) and 2j + 1 (high nibble); a byte permute spreads the
// nibbles of byte j into the two halves of pair j, OR-ing 0x6400 makes them fp16 1024 + q, v_pk_add_f16 takes 1024 off
// exactly and v_pk_fma_f16 rounds q s + m once to fp16. That single rounding equals fl16(fl32(q s + m)) whenever q s + m
// is exact in fp32 (pk_exact); otherwise the fp32 path rounds twice, exactly as the reference does.
__device__ __forceinline__ u32x4n deq_word(uint32_t v, uint32_t sm, bool fast) {
  u32x4n o;
  if (fast) {
    const h2 s2 = {__builtin_bit_cast(h2, sm).x, __builtin_bit_cast(h2, sm).x};
    const h2 m2 = {__builtin_bit_cast(h2, sm).y, __builtin_bit_cast(h2, sm).y};
    const h2 k1024 = {(_Float16)1024.0f, (_Float16)1024.0f};
    const uint32_t lo = v & 0x0F0F0F0Fu, hi = (v >> 4) & 0x0F0F0F0Fu;   // byte j: k 2j | k 2j + 1
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // bytes [lo.j, 0, hi.j, 0] (selector 0x0C gives zero); then the fp16 exponent of 1024
      const uint32_t sel = (uint32_t)j | (0x0Cu << 8) | ((uint32_t)(4 + j) << 16) | (0x0Cu << 24);
      const uint32_t b = __builtin_amdgcn_perm(hi, lo, sel) | 0x64006400u;
      const h2 q = __builtin_bit_cast(h2, b) - k1024;
      o[j] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(q, s2, m2));
    }
  } else {
    const float s = (float)__builtin_bit_cast(h2, sm).x, m = (float)__builtin_bit_cast(h2, sm).y;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float q0 = (float)((v >> (8 * j)) & 15u), q1 = (float)((v >> (8 * j + 4)) & 15u);
      // two roundings: left to itself, the compiler folds the fma and the conversion into one v_fma_mixlo_f16, which rounds once
      float f0 = __builtin_fmaf(q0, s, m), f1 = __builtin_fmaf(q1, s, m);
      asm("" : "+v"(f0), "+v"(f1));
      o[j] = pack_h2(f0, f1);
    }
  }
  return o;
}

// the GEMM for calls whose 256 x 256 tiles would leave CUs idle (gemm_n128.hip): can it take the call, and its launch
bool n128_takes(const GemmP& p);
void launch_n128(const GemmP& p, hipStream_t s);
int n128_init();

}  // namespace p0
