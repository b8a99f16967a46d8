// Small memory-bound kernels: embedding gather (vocab-parallel aware), sequence
// pooling + L2 normalisation, standalone activations.
// All loads/stores are 16-byte bf16x8 vectors (cdna_hip_programming Guideline 13).
#include "gai_common.h"
#include "gai_kernels.h"

using namespace gai;

namespace {

// out[t] = table[ids[t] - vstart] if vstart <= ids[t] < vend else 0 (vocab-parallel shard)
__global__ __launch_bounds__(256) void embedding_kernel(const int* __restrict__ ids, const bf16* __restrict__ table,
                                                        bf16* __restrict__ out, int T, int D, int vstart, int vend) {
  const int units = D / 8;
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long)T * units) return;
  const int t = (int)(e / units), u = (int)(e % units);
  const int id = ids[t];
  bf16x8 v = bf16x8{};
  if (id >= vstart && id < vend) v = load8(table + (size_t)(id - vstart) * D + u * 8);
  store8(out + (size_t)t * D + u * 8, v);
}

// Pool each sequence of hidden [T, D] (varlen via cu_seqlens) into out [B, D] fp32.
// mode 0 = masked mean, 1 = first token (CLS), 2 = last token. normalize -> v / ||v||. With lens, sequence b is the first lens[b] of its
// rows (padded batches; the first and last token of an empty one is its first row).
// One workgroup a sequence, bound by what its CU fetches: 16-byte column units times as many row groups as the threads
// hold, eight rows of each in flight, the groups' sums added in LDS. 61 sequences of ~300 rows of 1024: one row group of 128
// threads, a row at a time, took 142 us; with 1024 threads 20.
template <int kPoolThreads>
__global__ __launch_bounds__(kPoolThreads) void pool_kernel(const bf16* __restrict__ h, const int* __restrict__ cu,
                                                            const int* __restrict__ lens, float* __restrict__ out, int D, int mode, int normalize) {
  extern __shared__ float sh[];  // [groups][D] sums + 16 scratch
  const int units = D / 8, cols = max(min(units, kPoolThreads), 1);
  const int b = blockIdx.x;
  const int s0 = cu[b], s1 = lens ? min(s0 + max(lens[b], mode == 0 ? 0 : 1), cu[b + 1]) : cu[b + 1], n = s1 - s0;
  int r0 = s0, r1 = s1;
  if (mode == 1) r1 = min(s0 + 1, s1);
  if (mode == 2) r0 = max(s1 - 1, s0);
  const int rows = max(r1 - r0, 1), groups = min(kPoolThreads / cols, rows);
  float* scratch = sh + groups * D;
  constexpr int U = 8;
  if (rows == 1) {
    for (int u = threadIdx.x; u < units; u += kPoolThreads) {
      const bf16x8 v = r1 > r0 ? load8(h + (size_t)r0 * D + u * 8) : bf16x8{};
#pragma unroll
      for (int j = 0; j < 8; ++j) sh[u * 8 + j] = (float)v[j];
    }
  } else if (const int g = threadIdx.x / cols; g < groups) {
    for (int u = threadIdx.x % cols; u < units; u += cols) {
      float a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      for (int r = r0 + g; r < r1; r += U * groups) {
        bf16x8 v[U];
#pragma unroll
        for (int i = 0; i < U; ++i) v[i] = load8(h + (size_t)min(r + i * groups, r1 - 1) * D + u * 8);
#pragma unroll
        for (int i = 0; i < U; ++i)
          if (r + i * groups < r1) {
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] += (float)v[i][j];
          }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) sh[g * D + u * 8 + j] = a[j];
    }
  }
  __syncthreads();
  const float div = (mode == 0 && n > 0) ? 1.f / n : 1.f;
  float ss = 0.f;
  for (int d = threadIdx.x; d < D; d += kPoolThreads) {
    float v = 0.f;
    if (d < units * 8) {
      v = sh[d];
      for (int k = 1; k < groups; ++k) v += sh[k * D + d];
      v *= div;
    }
    sh[d] = v;  // column d is this thread's alone
    ss += v * v;
  }
  float scale = 1.f;
  if (normalize) {
    ss = block_sum(ss, scratch);
    scale = 1.f / fmaxf(sqrtf(ss), 1e-12f);
  }
  for (int d = threadIdx.x; d < D; d += kPoolThreads) out[(size_t)b * D + d] = sh[d] * scale;
}

// MODE 0: y[t, i] = silu(x[t, i]) * x[t, I + i] (non-interleaved gate|up); 1: gelu_erf(x);
// 2: SwiGLU on the interleaved-per-16 [gate16|up16] layout; 3: gelu_tanh(x); 4: GeGLU (gelu_tanh(gate) * up,
// interleaved layout: Gemma).
template <int MODE>
__global__ __launch_bounds__(256) void act_kernel(const bf16* __restrict__ x, bf16* __restrict__ y, int T, int I) {
  const int units = I / 8;
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long)T * units) return;
  const int t = (int)(e / units), u = (int)(e % units);
  bf16x8 o;
  if (MODE == 2 || MODE == 4) {  // gate/up interleaved per 16 columns (the fused-GLU weight layout)
    const int c = u * 8, p = c >> 4, c0 = c & 15;
    const bf16x8 g = load8(x + (size_t)t * 2 * I + 32 * p + c0);
    const bf16x8 up = load8(x + (size_t)t * 2 * I + 32 * p + 16 + c0);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      o[j] = (bf16)((MODE == 2 ? silu((float)g[j]) : gelu_tanh((float)g[j])) * (float)up[j]);
  } else if (MODE == 3) {
    const bf16x8 a = load8(x + (size_t)t * I + u * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (bf16)gelu_tanh((float)a[j]);
  } else if (MODE == 0) {
    const bf16x8 g = load8(x + (size_t)t * 2 * I + u * 8);
    const bf16x8 up = load8(x + (size_t)t * 2 * I + I + u * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (bf16)(silu((float)g[j]) * (float)up[j]);
  } else {
    const bf16x8 a = load8(x + (size_t)t * I + u * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (bf16)gelu_erf((float)a[j]);
  }
  store8(y + (size_t)t * I + u * 8, o);
}

// Multi-step decode: feed the token sampled at step j back as step j+1's input, inside one HIP
// graph. Row r < *n_valid: ids <- toks, pos += 1, ctx = pos + 1, slot from the block table
// (pages for the whole run are reserved by Scheduler.reserve_decode). Padded rows stay frozen
// on the scratch page.
__global__ __launch_bounds__(256) void decode_advance_kernel(const int* __restrict__ toks, int* __restrict__ ids,
                                                             int* __restrict__ pos, int* __restrict__ ctx,
                                                             int* __restrict__ slots, const int* __restrict__ bt,
                                                             int max_blocks, const int* __restrict__ n_valid, int B,
                                                             int block) {
  const int r = blockIdx.x * 256 + threadIdx.x;
  if (r >= B || r >= *n_valid) return;
  const int p = pos[r] + 1;
  ids[r] = toks[r];
  pos[r] = p;
  ctx[r] = p + 1;
  slots[r] = bt[(size_t)r * max_blocks + p / block] * block + p % block;
}

}  // namespace

void gai_decode_advance(const int* toks, int* ids, int* pos, int* ctx, int* slots, const int* bt, int max_blocks,
                        const int* n_valid, int B, int block, hipStream_t st) {
  if (B == 0) return;
  decode_advance_kernel<<<(B + 255) / 256, 256, 0, st>>>(toks, ids, pos, ctx, slots, bt, max_blocks, n_valid, B,
                                                         block);
  GAI_LAUNCH_CHECK();
}

void gai_embedding(const int* ids, const void* table, void* out, int T, int D, int vstart, int vend, hipStream_t st) {
  if (T == 0) return;
  const long n = (long)T * (D / 8);
  embedding_kernel<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(ids, (const bf16*)table, (bf16*)out, T, D, vstart,
                                                                 vend);
  GAI_LAUNCH_CHECK();
}

template <int NT>
static void launch_pool(const void* h, const int* cu, const int* lens, float* out, int B, int D, int mode, int normalize, hipStream_t st) {
  const int groups = D < 16 ? NT : D < 8 * NT ? NT / (D / 8) : 1;
  pool_kernel<NT><<<B, NT, (groups * D + 16) * sizeof(float), st>>>((const bf16*)h, cu, lens, out, D, mode, normalize);
  GAI_LAUNCH_CHECK();
}

// T rows in B sequences. 256 threads where 1024 wait for each other over little: one row a sequence (1024 columns, 64 sequences 3.9 -> 3.2 us,
// 1024 sequences 9.3 -> 4.1) or short ones (1024 x 8 rows of 1024 columns 10.5 -> 5.6). Wide rows fill 1024 threads by themselves (4096
// columns, 64 x 20 rows 8.7 -> 6.1) unless there are more sequences than the chip holds such workgroups (1024 x 1 row 12.3 -> 8.9).
void gai_pool(const void* h, const int* cu, const int* lens, float* out, int T, int B, int D, int mode, int normalize, hipStream_t st) {
  if (B == 0) return;
  const bool narrow = D <= 2048;
  if ((narrow || B > 512) && (mode != 0 || T / (narrow ? 32 : 16) < B)) launch_pool<256>(h, cu, lens, out, B, D, mode, normalize, st);
  else launch_pool<1024>(h, cu, lens, out, B, D, mode, normalize, st);
}

void gai_silu_mul(const void* x, void* y, int T, int I, hipStream_t st) {
  if (T == 0) return;
  const long n = (long)T * (I / 8);
  act_kernel<0><<<(unsigned)((n + 255) / 256), 256, 0, st>>>((const bf16*)x, (bf16*)y, T, I);
  GAI_LAUNCH_CHECK();
}

void gai_silu_mul_interleaved(const void* x, void* y, int T, int I, hipStream_t st) {
  if (T == 0) return;
  const long n = (long)T * (I / 8);
  act_kernel<2><<<(unsigned)((n + 255) / 256), 256, 0, st>>>((const bf16*)x, (bf16*)y, T, I);
  GAI_LAUNCH_CHECK();
}

void gai_gelu_tanh(const void* x, void* y, int T, int I, hipStream_t st) {
  if (T == 0) return;
  const long n = (long)T * (I / 8);
  act_kernel<3><<<(unsigned)((n + 255) / 256), 256, 0, st>>>((const bf16*)x, (bf16*)y, T, I);
  GAI_LAUNCH_CHECK();
}

void gai_geglu_interleaved(const void* x, void* y, int T, int I, hipStream_t st) {
  if (T == 0) return;
  const long n = (long)T * (I / 8);
  act_kernel<4><<<(unsigned)((n + 255) / 256), 256, 0, st>>>((const bf16*)x, (bf16*)y, T, I);
  GAI_LAUNCH_CHECK();
}

void gai_gelu(const void* x, void* y, int T, int I, hipStream_t st) {
  if (T == 0) return;
  const long n = (long)T * (I / 8);
  act_kernel<1><<<(unsigned)((n + 255) / 256), 256, 0, st>>>((const bf16*)x, (bf16*)y, T, I);
  GAI_LAUNCH_CHECK();
}
