// Common device-side definitions for the gfx950 (CDNA4, MI355X) kernels.
//
// Everything here is written for wave64 + MFMA: vector types that match the
// MFMA operand registers, wave reductions over 64 lanes, and small helpers
// for 16-byte vectorised bf16 access (hipcc does not auto-vectorise bf16).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gai {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kWave = 64;

#define GAI_LDS(p) ((__attribute__((address_space(3))) void*)(p))

// Sum and maximum over a wave, in every lane; the whole wave has to be active. The butterfly over 32, 16, 8, 4, 2, 1 lanes
// on VALU operands: half and row swaps, then DPP. After the step over 8 lanes a row of 16 holds equal values 8 apart, so a
// rotation by 4 brings the partner of the step over 4. The pairs, and so every bit, are those of the same butterfly through
// ds_bpermute, whose six LDS round trips (~100 clocks each, and four address instructions) these replace.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

template <typename F>
__device__ __forceinline__ float wave_butterfly(float v, F f) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(h[0]), __uint_as_float(h[1]));
  const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(q[0]), __uint_as_float(q[1]));
  v = f(v, dpp_f32<0x128>(v));   // row_ror:8
  v = f(v, dpp_f32<0x124>(v));   // row_ror:4
  v = f(v, dpp_f32<0x4E>(v));    // quad_perm [2, 3, 0, 1]
  return f(v, dpp_f32<0xB1>(v));  // quad_perm [1, 0, 3, 2]
}

__device__ __forceinline__ float wave_sum(float v) {
  return wave_butterfly(v, [](float a, float b) { return a + b; });
}

__device__ __forceinline__ float wave_max(float v) {
  return wave_butterfly(v, [](float a, float b) { return fmaxf(a, b); });
}

// Reduce within aligned groups of `W` lanes (W power of two <= 64).
template <int W>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int o = W / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <int W>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
  for (int o = W / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  return v;
}

__device__ __forceinline__ bf16x8 load8(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }
__device__ __forceinline__ void store8(bf16* p, bf16x8 v) { *reinterpret_cast<bf16x8*>(p) = v; }

// ---- fp8 KV cache (OCP e4m3fn, gfx950 native conversions) ----
typedef uint8_t fp8;
// 8 fp8 values (one 8-byte load) -> 8 bf16, each multiplied by `s` (v_cvt_scalef32_pk_bf16_fp8)
__device__ __forceinline__ bf16x8 fp8x8_to_bf16(uint2 v, float s) {
  const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v.x, s, false);
  const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v.x, s, true);
  const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v.y, s, false);
  const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v.y, s, true);
  return bf16x8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]};
}
// 4 floats * inv_s -> 4 packed e4m3fn bytes, saturated to +-448
__device__ __forceinline__ uint32_t f32x4_to_fp8(float a, float b, float c, float d, float inv_s) {
  auto sat = [&](float x) { return fminf(fmaxf(x * inv_s, -448.f), 448.f); };
  int w = __builtin_amdgcn_cvt_pk_fp8_f32(sat(a), sat(b), 0, false);
  w = __builtin_amdgcn_cvt_pk_fp8_f32(sat(c), sat(d), w, true);
  return (uint32_t)w;
}
// 8 cache elements -> bf16x8: a plain 16-byte load for bf16, an 8-byte load + conversion for fp8
__device__ __forceinline__ bf16x8 load_kv8(const bf16* p, float) { return load8(p); }
__device__ __forceinline__ bf16x8 load_kv8(const fp8* p, float s) {
  return fp8x8_to_bf16(*reinterpret_cast<const uint2*>(p), s);
}

__device__ __forceinline__ float silu(float x) { return x / (1.0f + __expf(-x)); }
// GELU with erfc by Abramowitz & Stegun 7.1.26 (|error| <= 1.5e-7), branch-free: one v_rcp_f32, one v_exp_f32 and ~10
// full-rate operations per element. The device libm erff is piecewise with data-dependent branches: in the 256x256 GEMM
// epilogue of an encoder FFN-up projection (K = 1024, so the epilogue is not hidden behind a long main loop) it made the
// bias + GELU GEMM 2x slower than the bias-only one (e5-large ingest at M = 65536: 990 vs ~450 us per layer, profiles/r6).
// As max(x, 0) - |x| / 2 erfc(|x| / sqrt 2): four operations less than 0.5 x (1 + erf), and for a negative x the error
// falls with erfc (relative 1.6e-3 at -5, where 1 + erf cancels to 5e-2). (The last product takes a finite |x|: inf stays inf.)
__device__ __forceinline__ float gelu_erf(float x) {
  const float z = fabsf(x);
  const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f * 0.70710678118654752f, z, 1.0f));
  float p = fmaf(0.5f * 1.061405429f, t, 0.5f * -1.453152027f);
  p = fmaf(p, t, 0.5f * 1.421413741f);
  p = fmaf(p, t, 0.5f * -0.284496736f);
  p = fmaf(p, t, 0.5f * 0.254829592f);
  const float e = __builtin_amdgcn_exp2f(x * (x * (-0.5f * 1.4426950408889634f)));
  return fmaf(-fminf(z, 3e38f), p * t * e, fmaxf(x, 0.f));
}
// tanh-GELU as x * sigmoid(2u): 0.5 x (1 + tanh(u)) == x / (1 + e^{-2u}), no libm tanhf
__device__ __forceinline__ float gelu_tanh(float x) {
  const float k0 = 0.7978845608028654f, k1 = 0.044715f;
  const float u = k0 * fmaf(k1 * x, x * x, x);
  return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-2.0f * 1.4426950408889634f * u));
}

// Block-level reduction for up to 1024 threads (16 waves). `scratch` holds >= 16 floats.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float r = 0.f;
  for (int i = 0; i < nw; ++i) r += scratch[i];
  return r;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wid] = v;
  __syncthreads();
  float r = -INFINITY;
  for (int i = 0; i < nw; ++i) r = fmaxf(r, scratch[i]);
  return r;
}

// XCD-aware, bijective remap of a linear workgroup id (cdna_hip_programming §5 T1):
// consecutive logical ids land on the same XCD (blocks b and b+8 share one).
__device__ __forceinline__ int xcd_remap(int bid, int nwg) {
  const int xcd = bid & 7, q = nwg >> 3, r = nwg & 7;
  const int base = xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q;
  return base + (bid >> 3);
}

}  // namespace gai

#define GAI_LAUNCH_CHECK()                                                        \
  do {                                                                            \
    hipError_t e_ = hipGetLastError();                                            \
    if (e_ != hipSuccess) gai_launch_error(__FILE__, __LINE__, hipGetErrorString(e_)); \
  } while (0)

void gai_launch_error(const char* file, int line, const char* msg);
