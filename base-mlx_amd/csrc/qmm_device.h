// Shared by the dequantizing GEMM kernels (qmm.hip, qmm_slab.hip): their
// parameters and the dequantization of a weight word.
#pragma once

#include "bmx_device.h"

namespace bmx {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;

struct QmmParams {
  const uint16_t* x;   // [M, K]
  const uint32_t* w;   // [N, K/8] (SwiGLU: gate)
  const uint16_t* s;   // [N, K/64]
  const uint16_t* b;   // [N, K/64]
  const uint32_t* w2;  // SwiGLU: up weight, scales and biases
  const uint16_t* s2;
  const uint16_t* b2;
  const uint16_t* res;  // residual: [M, N] (may alias y)
  uint16_t* y;          // [M, N] bf16 (one split)
  float* part;          // [splits, M, N] fp32 partials (several splits)
  int M, N, K;
  int gps;     // groups per split
  int mtiles;  // row tiles of x (the grid's x dimension enumerates mtiles x column tiles)
  int xcd;     // tile order: 0 row-major; XCD-grouped 1 column-major, 2 row-major
  // Store epilogue over up to 3 column segments (q | k | v of one layer in
  // one launch): segment i covers output columns [seg_n0[i], seg_n0[i+1])
  // of the launch (multiples of the tile width) with its own W, s, b and y
  // (y row stride = the segment's width).  nseg = 0: the plain product.
  int nseg;
  int seg_n0[4];
  const uint32_t* seg_w[3];
  const uint16_t* seg_s[3];
  const uint16_t* seg_b[3];
  uint16_t* seg_y[3];
  // Group-major weights (the model's prefill copy): w, w2 and seg_w hold
  // [K/64][N][8] words (each row's 64 nibbles of one group, rows of a group
  // consecutive), and sb, sb2 and seg_sb [K/64][N] words s | b << 16, so a
  // tile's W and s|b of one group are contiguous
  const uint32_t* sb;
  const uint32_t* sb2;
  const uint32_t* seg_sb[3];
  // QMM_QKV_ROPE: where the normed / rotated rows go
  QkvRopeOut rope;
};

// The GEMM for up to a few hundred rows (qmm_slab.hip, MLX-layout weights).
// How it takes a product of M x N x K with K split over at most max_splits
// workgroups (partials to QmmParams::part): 16-row tiles of x and W rows per
// workgroup, splits of gps groups.  fits is false where qmm_kernel is taken.
struct SlabPlan {
  bool fits;
  int mt, bn, splits, gps;
};
SlabPlan slab_plan(QmmEpilogue epi, int M, int N, int K, int max_splits);
int launch_qmm_slab(QmmEpilogue epi, const QmmParams& p, const SlabPlan& plan, hipStream_t stream);

// two floats -> packed bf16 pair, round to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint32_t pk_bf16(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t{lo, hi}), bf16x2_t));
}

// The 8 nibbles of a word as bf16(s q + b), in order (the value
// mlx_rs::ops::dequantize produces, one rounding)
__device__ __forceinline__ uint4 qmm_dequant_word(uint32_t word, float sv, float bv) {
  // nibble k of the word is value k: even k in the low nibble of byte k/2,
  // odd k in the high nibble
  uint32_t lo = word & 0x0f0f0f0fu, hi = (word >> 4) & 0x0f0f0f0fu;
  // opaque, so each byte converts with one v_cvt_f32_ubyte<n> instead of a
  // bit-field extract and a convert
  asm volatile("" : "+v"(lo), "+v"(hi));
  uint4 o;
  o.x = pk_bf16(fmaf(sv, static_cast<float>(lo & 0xffu), bv), fmaf(sv, static_cast<float>(hi & 0xffu), bv));
  o.y = pk_bf16(fmaf(sv, static_cast<float>((lo >> 8) & 0xffu), bv),
                fmaf(sv, static_cast<float>((hi >> 8) & 0xffu), bv));
  o.z = pk_bf16(fmaf(sv, static_cast<float>((lo >> 16) & 0xffu), bv),
                fmaf(sv, static_cast<float>((hi >> 16) & 0xffu), bv));
  o.w = pk_bf16(fmaf(sv, static_cast<float>(lo >> 24), bv), fmaf(sv, static_cast<float>(hi >> 24), bv));
  return o;
}

}  // namespace bmx
