// Device functions of lowp_mode INT8 that several kernels share: dynamic quantization of activations (IEEE fp32, expression by
// expression as the reference has it) and the decoding of 4-bit weight codes to int8.
#pragma once
#include "woq_common.h"

namespace woq {

// lane's eight values of one chunk
__device__ __forceinline__ void aq_unpack(u4 raw, bool bf16, float (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint16_t lo = (uint16_t)(raw[i] & 0xFFFFu), hi = (uint16_t)(raw[i] >> 16);
    v[2 * i] = bf16 ? bf16_bits_to_f32(lo) : f16_bits_to_f32(lo);
    v[2 * i + 1] = bf16 ? bf16_bits_to_f32(hi) : f16_bits_to_f32(hi);
  }
}

struct AqParams {
  float s, zp;
};

__device__ __forceinline__ AqParams aq_params(float mn, float mx, bool sym, int32_t* zp_out) {
  AqParams p;
  if (sym) {
    p.s = __fdiv_rn(fmaxf(fabsf(mx), fabsf(mn)), 127.0f);
    p.zp = 0.0f;
  } else {
    p.s = __fdiv_rn(__fsub_rn(mx, mn), 255.0f);
    const int32_t z = (int32_t)(-rintf(__fdiv_rn(mn, p.s)));
    p.zp = (float)z;
    if (zp_out) *zp_out = z;
  }
  return p;
}

__device__ __forceinline__ uint8_t aq_quant(float v, AqParams p, bool sym, bool offset128) {
  float t = __fadd_rn(__fdiv_rn(v, p.s), p.zp);
  t = rintf(t);
  const float lo = sym ? -128.0f : 0.0f, hi = sym ? 127.0f : 255.0f;
  t = fminf(fmaxf(t, lo), hi);
  if (p.s == 0.0f || t != t) t = sym ? 0.0f : p.zp;  // all-zero group: the reference divides 0 by 0
  return sym ? (uint8_t)(int8_t)(int)t : (uint8_t)((int)t ^ (offset128 ? 0x80 : 0));
}

// Four bytes at once: ((b | 0x80808080) - z4) ^ 0x80808080 never borrows across bytes for
// |q - z| < 128 and leaves q - z in two's complement.
__device__ __forceinline__ uint32_t w8_sub_bytes(uint32_t b, uint32_t z4) {
  return ((b | 0x80808080u) - z4) ^ 0x80808080u;
}
// sixteen K values of one lane from two packed dwords, in the order [e0 e4 e1 e5][e2 e6 e3 e7] per dword
__device__ __forceinline__ i4 w8_decode16(uint32_t d0, uint32_t d1, uint32_t z4) {
  i4 r;
  r[0] = (int)w8_sub_bytes(d0 & 0x0F0F0F0Fu, z4);
  r[1] = (int)w8_sub_bytes((d0 >> 4) & 0x0F0F0F0Fu, z4);
  r[2] = (int)w8_sub_bytes(d1 & 0x0F0F0F0Fu, z4);
  r[3] = (int)w8_sub_bytes((d1 >> 4) & 0x0F0F0F0Fu, z4);
  return r;
}

// One K block's int32 sum into the fp32 accumulator.  The reference computes
// C += (float(sum) * s_a) * s_w per block (csrc/cpu/aten/utils/woq.h:2172-2186; its compiler is free to
// contract the last multiply and the addition).  PER_K: exactly that, with the contraction: convert,
// multiply, fused multiply-add.  Otherwise s_a is the same for every block of a row and is applied
// once after the K loop, C = (sum over blocks of float(sum) * s_w) * s_a: convert and one fused
// multiply-add per block, a third fewer VALU instructions in a loop that they bound; the results
// differ from the per-block order by fp32 rounding only (~1e-7 relative).
template <bool PER_K>
__device__ __forceinline__ float w8_accumulate(int sum, float s_a, float s_w, float acc) {
  if constexpr (PER_K)
    return __builtin_fmaf((float)sum * s_a, s_w, acc);
  else
    return __builtin_fmaf((float)sum, s_w, acc);
}

}  // namespace woq
