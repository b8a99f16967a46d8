// Rotation of the heads in the rotate-half layout with the write of the cached rows (attention_window.hip), for the launches that it
// shares with others.
#pragma once
#include "gai_common.h"

namespace gai {

template <typename TA>
struct RotaryHalf {
  const TA* q;
  int ldq;
  const TA* k;
  int ldk;
  const TA* v;
  int ldv;
  const int *positions, *slots;
  TA *q_out, *k_cache, *v_cache;
  int T, H, G, DK, DV;
  const double* inv_freq;
  int half;
  float unit_eps;
  int lph;
};
constexpr int kHalfRegs = 8;

// Workgroups 0 .. T - 1: q and k heads of one token, `lph` lanes (a power of two) per head with NJ groups of VEC channels
// each, so a wave holds 64 / lph heads; the others: v of VT tokens, a thread per channel, so that tokens filling a whole page
// store its V^T row at once. 256 threads; cs: 2 half floats of LDS.
template <typename TA, int VEC, int NJ, int VT>
__device__ __forceinline__ void rotary_half_body(const RotaryHalf<TA>& a, int wg, float* cs) {
  const TA *__restrict__ q = a.q, *__restrict__ k = a.k, *__restrict__ v = a.v;
  const int *__restrict__ positions = a.positions, *__restrict__ slots = a.slots;
  TA *__restrict__ q_out = a.q_out, *__restrict__ k_cache = a.k_cache, *__restrict__ v_cache = a.v_cache;
  const double* __restrict__ inv_freq = a.inv_freq;
  const int ldq = a.ldq, ldk = a.ldk, ldv = a.ldv, T = a.T, H = a.H, G = a.G, DK = a.DK, DV = a.DV, half = a.half, lph = a.lph;
  const float unit_eps = a.unit_eps;
  const int tid = threadIdx.x;
  if (wg >= T) {
    const int t0 = (wg - T) * VT, n = min(VT, T - t0), NV = G * DV, s0 = slots[t0];
    const bool page = VT == 16 && n == 16 && (s0 & 15) == 0 && __all(slots[t0 + (tid & 15)] == s0 + (tid & 15));
    for (int i = tid; i < NV; i += 256) {
      const int g = i / DV, c = i - g * DV;
      const TA* src = v + (size_t)t0 * ldv + i;
      if (page) {
        TA* dst = v_cache + (((size_t)(s0 >> 4) * G + g) * DV + c) * 16;
        __attribute__((aligned(16))) TA x[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) x[j] = src[(size_t)j * ldv];
#pragma unroll
        for (int j = 0; j < (int)sizeof(TA); ++j)
          reinterpret_cast<uint4*>(dst)[j] = reinterpret_cast<const uint4*>(x)[j];
      } else {
        for (int j = 0; j < n; ++j) {
          const int s = slots[t0 + j];
          v_cache[(((size_t)(s >> 4) * G + g) * DV + c) * 16 + (s & 15)] = src[(size_t)j * ldv];
        }
      }
    }
    return;
  }
  // cs: cos[half] | sin[half]
  const int t = wg, lane = tid & (lph - 1);
  const double pos = (double)positions[t];
  for (int i = tid; i < half; i += 256) {
    const double a = pos * inv_freq[i];
    const double r = a - 6.283185307179586476925 * rint(a * 0.15915494309189533577);
    float sn, c;
    sincosf((float)r, &sn, &c);
    cs[i] = c;
    cs[half + i] = sn;
  }
  __syncthreads();
  const int slot = slots[t], off = slot & 15;
  const size_t page = slot >> 4;
  typedef TA vec __attribute__((ext_vector_type(VEC)));
  for (int hh = tid / lph; hh < H + G; hh += 256 / lph) {  // q heads, then k heads: uniform over the head's lanes
    const bool isq = hh < H;
    const int g = isq ? hh : hh - H;
    const TA* src = isq ? q + (size_t)t * ldq + (size_t)g * DK : k + (size_t)t * ldk + (size_t)g * DK;
    TA* dst = isq ? q_out + ((size_t)t * H + g) * DK : k_cache + ((page * G + g) * 16 + off) * DK;
    float y[NJ][VEC];
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < NJ; ++r) {
      const int i = (lane + lph * r) * VEC;
      if (i < DK) {
        const vec x = *reinterpret_cast<const vec*>(src + i);
        if (i < 2 * half) {   // VEC divides half: the group has one partner group
          const bool up = i >= half;
          const vec p = *reinterpret_cast<const vec*>(src + (up ? i - half : i + half));
          const int f = up ? i - half : i;
#pragma unroll
          for (int e = 0; e < VEC; ++e) {
            const float c = cs[f + e], sn = cs[half + f + e];
            y[r][e] = up ? (float)x[e] * c + (float)p[e] * sn : (float)x[e] * c - (float)p[e] * sn;
          }
        } else {
#pragma unroll
          for (int e = 0; e < VEC; ++e) y[r][e] = (float)x[e];
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) ss += y[r][e] * y[r][e];
      }
    }
    float inv = 1.0f;
    if (unit_eps >= 0.f) {
      for (int o = lph >> 1; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
      inv = 1.0f / sqrtf(ss / DK + unit_eps);
    }
#pragma unroll
    for (int r = 0; r < NJ; ++r) {
      const int i = (lane + lph * r) * VEC;
      if (i < DK) {
        vec o;
#pragma unroll
        for (int e = 0; e < VEC; ++e) o[e] = (TA)(y[r][e] * inv);
        *reinterpret_cast<vec*>(dst + i) = o;
      }
    }
  }
}

}  // namespace gai

// gemm_slim.hip: the slices of gai_gemm_slim_few_ks (A . W^T, W in fragment order) beside the rotation of up to 64 rows (heads by 8s)
void gai_gemm_slim_partials_rotary(const void* A, const void* W, int M, int N, int K, float* ws, const gai::RotaryHalf<gai::bf16>& r,
                                   hipStream_t st);
