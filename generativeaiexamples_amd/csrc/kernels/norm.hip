// RMSNorm / LayerNorm with optional fused residual add.
//
// One wave64 per row, 16-byte (bf16x8) vectorised loads, the whole row held in
// registers (NCH chunks of 512 elements per lane-sweep), fp32 statistics.
// Fused residual: r = x + residual (rounded to bf16, matching torch bf16
// semantics); residual <- r when `residual_out` is set; y = norm(r) * w (+ b).
#include "gai_common.h"
#include "gai_kernels.h"

using namespace gai;

namespace {

template <int NCH, bool LAYERNORM>
__global__ __launch_bounds__(256) void norm_kernel(const bf16* __restrict__ x, const bf16* residual_in,
                                                   bf16* residual_out, const bf16* __restrict__ w,
                                                   const bf16* __restrict__ b, bf16* __restrict__ out, int T,
                                                   int D, float eps) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= T) return;
  const size_t base = (size_t)row * D;
  // Issue every load of the row (x, residual, gamma) before the first store: residual_out usually
  // aliases residual_in, so a store inside the load loop would pin each later load behind it and
  // serialise NCH memory round trips (10+ us for a 64-row decode norm instead of one trip).
  bf16x8 xa[NCH], ra[NCH], ga[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int idx = (c * 64 + lane) * 8;
    if (idx < D) {
      xa[c] = load8(x + base + idx);
      ra[c] = residual_in ? load8(residual_in + base + idx) : bf16x8{};
      ga[c] = load8(w + idx);
    }
  }
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int idx = (c * 64 + lane) * 8;
    if (idx < D) {
      bf16x8 a = xa[c];
      if (residual_in) {
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = (bf16)((float)a[j] + (float)ra[c][j]);
        xa[c] = a;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) s += LAYERNORM ? (float)a[j] : (float)a[j] * (float)a[j];
    }
  }
  if (residual_in && residual_out) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int idx = (c * 64 + lane) * 8;
      if (idx < D) store8(residual_out + base + idx, xa[c]);
    }
  }
  s = wave_sum(s);
  float mean = 0.f, inv;
  if (LAYERNORM) {
    mean = s / D;
    float q = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int idx = (c * 64 + lane) * 8;
      if (idx < D) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float d = (float)xa[c][j] - mean;
          q += d * d;
        }
      }
    }
    q = wave_sum(q);
    inv = rsqrtf(q / D + eps);
  } else {
    inv = rsqrtf(s / D + eps);
  }
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int idx = (c * 64 + lane) * 8;
    if (idx < D) {
      const bf16x8 g = ga[c];
      bf16x8 o;
      if (LAYERNORM) {
        const bf16x8 bb = b ? load8(b + idx) : bf16x8{};
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = (bf16)(((float)xa[c][j] - mean) * inv * (float)g[j] + (b ? (float)bb[j] : 0.f));
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = (bf16)((float)xa[c][j] * inv * (float)g[j]);
      }
      store8(out + base + idx, o);
    }
  }
}

// An encoder's first norm: LayerNorm(bf16(bf16(word + position) + type)), the roundings of three additions of bf16 rows, each row read
// once. As a gather, two additions, another gather and the norm it was five launches and eleven passes over the rows: 9240 tokens of 1024
// columns 50 -> 11.4 us, 18480 74 -> 17, 32 tokens 13 -> 3.4. Ids outside the table take a row of zeros.
template <int NCH>
__global__ __launch_bounds__(256) void embed_layernorm_kernel(const int* __restrict__ ids, const int* __restrict__ pos,
                                                              const bf16* __restrict__ word, const bf16* __restrict__ ptab,
                                                              const bf16* __restrict__ type, const bf16* __restrict__ w,
                                                              const bf16* __restrict__ b, bf16* __restrict__ out, int T, int D, int vocab,
                                                              float eps) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= T) return;
  const int id = ids[row];
  const bool known = id >= 0 && id < vocab;
  const bf16 *wr = word + (size_t)(known ? id : 0) * D, *pr = ptab + (size_t)pos[row] * D;
  bf16x8 xa[NCH], pa[NCH], ta[NCH], ga[NCH], ba[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int idx = (c * 64 + lane) * 8;
    if (idx < D) {
      xa[c] = known ? load8(wr + idx) : bf16x8{};
      pa[c] = load8(pr + idx);
      ta[c] = load8(type + idx);
      ga[c] = load8(w + idx);
      ba[c] = load8(b + idx);
    }
  }
  float s = 0.f, q = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    if ((c * 64 + lane) * 8 < D) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        xa[c][j] = (bf16)((float)(bf16)((float)xa[c][j] + (float)pa[c][j]) + (float)ta[c][j]);
        s += (float)xa[c][j];
      }
    }
  }
  const float mean = wave_sum(s) / D;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    if ((c * 64 + lane) * 8 < D) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float d = (float)xa[c][j] - mean;
        q += d * d;
      }
    }
  }
  const float inv = rsqrtf(wave_sum(q) / D + eps);
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int idx = (c * 64 + lane) * 8;
    if (idx < D) {
      bf16x8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (bf16)(((float)xa[c][j] - mean) * inv * (float)ga[c][j] + (float)ba[c][j]);
      store8(out + (size_t)row * D + idx, o);
    }
  }
}

template <bool LN>
void dispatch_norm(const void* x, const void* rin, void* rout, const void* w, const void* b, void* out, int T,
                   int D, float eps, hipStream_t st) {
  // Up to two rows a CU a workgroup is one wave: a CU draws 25 - 30 KB/us, and four rows of 4096 are 32 KB. Us, four waves | one, RMS:
  // rows of 4096, 32 of them 4.8 | 4.3, 256 5.1 | 4.5, 512 5.7 | 5.35; of 8192, 512 9.3 | 8.9; of 1024, 32 2.50 | 2.29, 512 2.64 | 2.62; of 384, 8 2.29 | 2.35,
  // 512 2.32 | 2.30. LayerNorm of 4096, 32 6.0 | 5.2; of 1024, 512 2.99 | 3.00. 1024 rows of 8192, RMS, 11.4 | 11.9
  const int wv = T <= 512 ? 1 : 4;
  const dim3 grid((T + wv - 1) / wv), block(64 * wv);
  const int nch = (D + 511) / 512;
#define GAI_NORM_CASE(N)                                                                                   \
  if (nch <= N) {                                                                                          \
    norm_kernel<N, LN><<<grid, block, 0, st>>>((const bf16*)x, (const bf16*)rin, (bf16*)rout,             \
                                                (const bf16*)w, (const bf16*)b, (bf16*)out, T, D, eps);   \
    GAI_LAUNCH_CHECK();                                                                                    \
    return;                                                                                                \
  }
  GAI_NORM_CASE(1)
  GAI_NORM_CASE(2)
  GAI_NORM_CASE(3)
  GAI_NORM_CASE(4)
  GAI_NORM_CASE(8)
  GAI_NORM_CASE(16)
#undef GAI_NORM_CASE
  gai_launch_error(__FILE__, __LINE__, "norm: hidden size > 8192 unsupported");
}

}  // namespace

void gai_embed_layernorm(const int* ids, const int* pos, const void* word, const void* ptab, const void* type, const void* w,
                         const void* b, void* out, int T, int D, int vocab, float eps, hipStream_t st) {
  if (T == 0) return;
  const int nch = (D + 511) / 512;
#define GAI_EMB_CASE(N)                                                                                                       \
  if (nch <= N) {                                                                                                            \
    embed_layernorm_kernel<N><<<(T + 3) / 4, 256, 0, st>>>(ids, pos, (const bf16*)word, (const bf16*)ptab, (const bf16*)type, \
                                                           (const bf16*)w, (const bf16*)b, (bf16*)out, T, D, vocab, eps);    \
    GAI_LAUNCH_CHECK();                                                                                                      \
    return;                                                                                                                  \
  }
  GAI_EMB_CASE(1)
  GAI_EMB_CASE(2)
  GAI_EMB_CASE(4)
#undef GAI_EMB_CASE
  gai_launch_error(__FILE__, __LINE__, "embed_layernorm: hidden size > 2048 unsupported");
}

void gai_rmsnorm(const void* x, const void* residual_in, void* residual_out, const void* w, void* out, int T, int D,
                 float eps, hipStream_t st) {
  if (T == 0) return;
  dispatch_norm<false>(x, residual_in, residual_out, w, nullptr, out, T, D, eps, st);
}

void gai_layernorm(const void* x, const void* residual_in, void* residual_out, const void* w, const void* b,
                   void* out, int T, int D, float eps, hipStream_t st) {
  if (T == 0) return;
  dispatch_norm<true>(x, residual_in, residual_out, w, b, out, T, D, eps, st);
}
