// Dequantization epilogue of the INT8 GEMM kernels, per output element: the
// scale / bias / activation orders of include/qgemm.h (qg_epilogue), the
// optional residual term and the one rounding to the output type.
#pragma once
#include "qg_common.h"
#include "qg_internal.h"

namespace qg {

namespace {

enum EpiMode { EPI_INT = 0, EPI_F = 1, EPI_FMA = 2, EPI_EAGER = 3, EPI_GELU = 4 };

__device__ __forceinline__ float gelu_tanh(float x) {
#pragma clang fp contract(off)
  // 0.5 * x * (1 + tanh(u)), u = sqrt(2/pi) * (x + 0.044715 * x^3): the
  // tanh approximation of ATen's CPU GeluKernel, evaluated as the identical
  // x * sigmoid(2u) = x / (1 + 2^(-2u log2 e)) with 2u log2 e = x (c0 + c1 x^2),
  // the hardware exp2 and reciprocal. Absolute error a few 1e-7, far below
  // one fp16/bf16 ulp of the result; large +x gives x, large -x gives -0 and
  // -inf gives NaN, as the reference formula does.
  const float c0 = 2.3022082f;   // 2 sqrt(2/pi) log2(e)
  const float c1 = 0.10294324f;  // c0 * 0.044715
  const float p = __builtin_fmaf(c1, x * x, c0);
  const float e = __builtin_amdgcn_exp2f(-(x * p));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ float silu(float g) {
#pragma clang fp contract(off)
  // g / (1 + e^-g) with the hardware exp2 and reciprocal (a few ulps)
  return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f));
}

// Raw storage bits of bias[col] (fp32, fp16 or bf16) and their fp32 value.
__device__ __forceinline__ uint32_t load_bias_bits(const void* bias, int dtype, int col) {
  if (dtype == QG_F32) return static_cast<const uint32_t*>(bias)[col];
  return static_cast<const uint16_t*>(bias)[col];
}
__device__ __forceinline__ float bias_value(uint32_t bits, int dtype) {
  if (dtype == QG_F32) return __uint_as_float(bits);
  return dtype == QG_F16 ? f16_to_f32(static_cast<uint16_t>(bits)) : bf16_to_f32(static_cast<uint16_t>(bits));
}

template <int OUT>
__device__ __forceinline__ float round_to(float v) {
  if constexpr (OUT == QG_F16) return f16_to_f32(f32_to_f16(v));
  else if constexpr (OUT == QG_BF16) return bf16_to_f32(f32_to_bf16(v));
  else return v;
}

template <int OUT>
constexpr int out_size() { return (OUT == QG_F16 || OUT == QG_BF16) ? 2 : 4; }

// Row stride (elements) of a dense kernel's output: out_sm, or N when 0.
__device__ __forceinline__ int64_t out_ld(const I8GemmArgs& p) { return p.out_sm > 0 ? p.out_sm : p.N; }

// Storage bits of one output element.
//   EPI_F:     v = f32(acc) * (sa * sb); v = v + bias           (int8_gemm.py:53-63)
//   EPI_FMA:   v = fma(f32(acc), sa * sb, bias)                 (rounding="fused", :191)
//   EPI_EAGER: t = out(f32(acc) * (sa * sb)); t = out(t + out(bias))  (comfy_int8.py:128-143)
//   EPI_GELU:  EPI_F followed by GELU-tanh in fp32
template <int OUT, int MODE, typename ACC>
__device__ __forceinline__ float epi_value(ACC acc, float sa, float sb, float bv, bool has_bias) {
#pragma clang fp contract(off)
  const float scale = sa * sb;
  const float accf = static_cast<float>(acc);  // exact for int32 |acc| < 2^24, identity for fp32
  float v;
  if constexpr (MODE == EPI_EAGER) {
    v = accf * scale;
    // the fp32 product, rounded: folded into the conversion (v_fma_mixlo_f16) it
    // would round once, to fp16 (6 of 100,000 results differed)
    asm("" : "+v"(v));
    v = round_to<OUT>(v);
    if (has_bias) v = v + round_to<OUT>(bv);
  } else if constexpr (MODE == EPI_FMA) {
    v = has_bias ? __builtin_fmaf(accf, scale, bv) : accf * scale;
  } else {
    v = accf * scale;
    if (has_bias) v = v + bv;
    if constexpr (MODE == EPI_GELU) v = gelu_tanh(v);
  }
  return v;
}
template <int OUT, int MODE>
__device__ __forceinline__ uint32_t epi_bits(int32_t acc, float sa, float sb, float bv, bool has_bias) {
  if constexpr (MODE == EPI_INT) {
    return static_cast<uint32_t>(acc);
  } else {
    const float v = epi_value<OUT, MODE>(acc, sa, sb, bv, has_bias);
    if constexpr (OUT == QG_F32) return __float_as_uint(v);
    else if constexpr (OUT == QG_F16) return f32_to_f16(v);
    else return f32_to_bf16(v);
  }
}

// The residual term of output element (row, col) (p.residual non-null).
__device__ __forceinline__ float residual_term(const I8GemmArgs& p, int row, int col) {
#pragma clang fp contract(off)
  const int64_t idx = static_cast<int64_t>(row) * p.residual_sm + col;
  float r;
  if (p.residual_dtype == QG_F32) r = static_cast<const float*>(p.residual)[idx];
  else if (p.residual_dtype == QG_F16) r = f16_to_f32(static_cast<const uint16_t*>(p.residual)[idx]);
  else r = bf16_to_f32(static_cast<const uint16_t*>(p.residual)[idx]);
  if (p.residual_scale) r = r * p.residual_scale[p.residual_scalar ? 0 : col];
  return r;
}

// Output bits of one element with the residual term (MODE != EPI_INT / EPI_EAGER).
template <int OUT, int MODE>
__device__ __forceinline__ uint32_t epi_bits_res(const I8GemmArgs& p, int32_t acc, float sa, float sb, float bv,
                                                 bool has_bias, int row, int col) {
#pragma clang fp contract(off)
  float v = epi_value<OUT, MODE>(acc, sa, sb, bv, has_bias);
  v = v + residual_term(p, row, col);
  if constexpr (OUT == QG_F32) return __float_as_uint(v);
  else if constexpr (OUT == QG_F16) return f32_to_f16(v);
  else return f32_to_bf16(v);
}

template <int OUT>
__device__ __forceinline__ void store_elem(void* out, int64_t idx, uint32_t bits) {
  if constexpr (out_size<OUT>() == 4) static_cast<uint32_t*>(out)[idx] = bits;
  else static_cast<uint16_t*>(out)[idx] = static_cast<uint16_t>(bits);
}

// One output element of p from its int32 sum, the epilogue chosen at run time
// (kernels whose time is not in the epilogue).
template <int OUT>
__device__ __forceinline__ void i8_store_as(const I8GemmArgs& p, int row, int col, int acc) {
  const float sa = p.a_scale[row], sb = p.b_scale[p.b_scalar ? 0 : col];
  const bool has_bias = p.bias != nullptr;
  const float bv = has_bias ? bias_value(load_bias_bits(p.bias, p.bias_dtype, col), p.bias_dtype) : 0.0f;
  const int64_t idx = static_cast<int64_t>(row) * out_ld(p) + col;
  uint32_t bits;
  if (p.residual) {
    if (p.epi & QG_EPI_GELU_TANH) bits = epi_bits_res<OUT, EPI_GELU>(p, acc, sa, sb, bv, has_bias, row, col);
    else if (p.epi & QG_EPI_ORDER_FUSED_FMA) bits = epi_bits_res<OUT, EPI_FMA>(p, acc, sa, sb, bv, has_bias, row, col);
    else bits = epi_bits_res<OUT, EPI_F>(p, acc, sa, sb, bv, has_bias, row, col);
  } else if (p.epi & QG_EPI_GELU_TANH) {
    bits = epi_bits<OUT, EPI_GELU>(acc, sa, sb, bv, has_bias);
  } else if (p.epi & QG_EPI_ORDER_FUSED_FMA) {
    bits = epi_bits<OUT, EPI_FMA>(acc, sa, sb, bv, has_bias);
  } else if (OUT != QG_F32 && (p.epi & QG_EPI_ORDER_EAGER)) {  // orders F and E coincide for fp32
    bits = epi_bits<OUT, EPI_EAGER>(acc, sa, sb, bv, has_bias);
  } else {
    bits = epi_bits<OUT, EPI_F>(acc, sa, sb, bv, has_bias);
  }
  store_elem<OUT>(p.out, idx, bits);
}
__device__ __forceinline__ void i8_store_out(const I8GemmArgs& p, int row, int col, int acc) {
  if (p.a_scale == nullptr)
    store_elem<QG_I32>(p.out, static_cast<int64_t>(row) * out_ld(p) + col, static_cast<uint32_t>(acc));
  else if (p.out_dtype == QG_F16) i8_store_as<QG_F16>(p, row, col, acc);
  else if (p.out_dtype == QG_BF16) i8_store_as<QG_BF16>(p, row, col, acc);
  else i8_store_as<QG_F32>(p, row, col, acc);
}

}  // namespace

}  // namespace qg
