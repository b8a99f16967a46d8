// Gated DeltaNet (Qwen3-Next linear-attention layers): the recurrent decode step, then the prompt kernels.
//
// Per (sequence b, value head h) the layer keeps a fp32 state S [DK][DV] in a slot pool; one decode
// token applies
//     S <- exp(g) S;  m = S^T k;  d = beta (v - m);  S <- S + k d^T;  o = S^T q
// (q, k l2-normalised, q pre-scaled by DK^-1/2). The step is a pure state stream: read + write
// DK*DV*4 bytes per head, ~4 flops per byte, so it is HBM-bound. One workgroup per (h, b); thread (r, j)
// owns rows [32r, 32r+32) of state column j: it walks the DK rows with coalesced 4-B loads (a row of DV floats is
// contiguous across the workgroup), keeps its slice of the column in VGPRs between the read and the
// write-back, and q / k live in LDS. The update is in place through `slots` (no gather / scatter copies), so the
// launch is graph-capturable with the slot vector as a static input.
#include <type_traits>

#include "gai_common.h"
#include "gai_kernels.h"

using namespace gai;

namespace {

// DK / 32 row groups x 128 columns: thread (r, j) keeps rows [32r, 32r + 32) of column j in VGPRs;
// the two column reductions (m = S^T k, o = S^T q) combine the row groups through LDS.
template <int DK>
__global__ __launch_bounds__(DK * 4) void gdn_decode_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                            const float* __restrict__ v, const float* __restrict__ g,
                                                            const float* __restrict__ beta, float* __restrict__ state,
                                                            const int* __restrict__ slots, float* __restrict__ out,
                                                            int Hk, int Hv, int DV) {
  constexpr int RG = DK / 32;
  __shared__ float qs[DK], ks[DK], red[RG][128];
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x;
  const int j0 = tid & 127, r = tid >> 7;  // r is wave-uniform (128 = 2 waves)
  const size_t bh = (size_t)b * Hv + h, bk = (size_t)b * Hk + h / (Hv / Hk);
  if (tid < DK) {
    qs[tid] = q[bk * DK + tid];
    ks[tid] = k[bk * DK + tid];
  }
  __syncthreads();
  const float eg = __expf(g[bh]), bt = beta[bh];
  float* S = state + ((size_t)slots[b] * Hv + h) * DK * DV + (size_t)(32 * r) * DV;
  for (int jb = 0; jb < DV; jb += 128) {
    const int j = jb + j0;
    const bool on = j < DV;
    float col[32];
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      col[i] = on ? S[(size_t)i * DV + j] * eg : 0.f;
      m += col[i] * ks[32 * r + i];
    }
    red[r][j0] = m;
    __syncthreads();
    m = 0.f;
#pragma unroll
    for (int t = 0; t < RG; ++t) m += red[t][j0];
    const float d = on ? (v[bh * DV + j] - m) * bt : 0.f;
    float o = 0.f;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      col[i] += ks[32 * r + i] * d;
      o += col[i] * qs[32 * r + i];
      if (on) S[(size_t)i * DV + j] = col[i];
    }
    __syncthreads();  // every thread has read red[][] for m
    red[r][j0] = o;
    __syncthreads();
    if (r == 0 && on) {
      float acc = 0.f;
#pragma unroll
      for (int t = 0; t < RG; ++t) acc += red[t][j0];
      out[bh * DV + j] = acc;
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------------------
// Prompt portions. Inputs of the rule first (gdn_prep): causal depthwise convolution over four tokens + SiLU of the
// projected q | k | v channels, unit q (x DK^-1/2) and k per key head, log decay and write strength per value head. A wave
// owns one head's channels for RUN tokens, so the taps stay in registers; all rows of the run are loaded before the first is
// used, and a run inside one sequence takes a path without its branches. 10095 tokens x 4096 channels: 248 MB, 115 -> 78 us
// (a load and a wait per row before), bound now by ~60 VALU instructions a channel (exponential and division at full
// precision); as separate torch kernels 4.6 ms.
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ float softplusf(float x) { return x > 20.f ? x : log1pf(expf(x)); }

template <typename TA, int DK, int RUN>
__global__ __launch_bounds__(256) void gdn_prep_kernel(const TA* __restrict__ proj, int ld, const float* __restrict__ cw,
                                                       const float* __restrict__ cstate, const int* __restrict__ cu,
                                                       const int* __restrict__ slots, int S, int T, int Hk, int Hv, int DV,
                                                       const float* __restrict__ A_log, const float* __restrict__ dt_bias,
                                                       float* __restrict__ q, float* __restrict__ k, float* __restrict__ v,
                                                       float* __restrict__ g, float* __restrict__ beta) {
  constexpr int CPL = DK / 64;  // channels per lane
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t0 = blockIdx.x * RUN, kd = Hk * DK, vd = Hv * DV, cd = 2 * kd + vd;
  if (blockIdx.y == gridDim.y - 1) {  // gates
    for (int e = threadIdx.x; e < RUN * Hv; e += 256) {
      const int t = t0 + e / Hv, h = e % Hv;
      if (t >= T) break;
      const TA* row = proj + (size_t)t * ld + cd + vd;
      beta[(size_t)t * Hv + h] = 1.f / (1.f + expf(-(float)row[h]));
      g[(size_t)t * Hv + h] = -expf(A_log[h]) * softplusf((float)row[Hv + h] + dt_bias[h]);
    }
    return;
  }
  const int vec = blockIdx.y * 4 + wid, c0 = vec * DK + lane * CPL;
  if (c0 >= cd) return;
  const bool on_v = vec >= 2 * Hk;
  const bool full = (vec + 1) * DK <= cd;  // every lane's channels exist
  int ci[CPL];                             // loads past the channels or the tokens read the last one: no branch parts them
#pragma unroll
  for (int i = 0; i < CPL; ++i) ci[i] = min(c0 + i, cd - 1);
  float w[CPL][4];
  TA x[RUN + 3][CPL];  // the taps' reach before the run, then the run
#pragma unroll
  for (int r = 0; r < RUN; ++r)
#pragma unroll
    for (int i = 0; i < CPL; ++i) x[r + 3][i] = proj[(size_t)min(t0 + r, T - 1) * ld + ci[i]];
#pragma unroll
  for (int i = 0; i < CPL; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) w[i][j] = cw[(size_t)ci[i] * 4 + j];
  int s = 0, hi = S;
  while (hi - s > 1) {
    const int mid = (s + hi) >> 1;
    if (cu[mid] <= t0) s = mid; else hi = mid;
  }
  int first = cu[s], next = cu[s + 1];
  auto back = [&](int t, int i) -> float {  // channel i of row t, which may lie before its sequence's first
    return t >= first ? (float)proj[(size_t)t * ld + ci[i]] : cstate[((size_t)slots[s] * 3 + 3 + t - first) * cd + ci[i]];
  };
  const float scale = vec < Hk ? 1.f / sqrtf((float)DK) : 1.f;
  const int ldo = on_v ? vd : kd, oc = on_v ? c0 - 2 * kd : vec < Hk ? c0 : c0 - kd;
  float* o = (on_v ? v : vec < Hk ? q : k) + oc;
  auto row = [&](const float(&y0)[CPL], const float(&y1)[CPL], const float(&y2)[CPL], const float(&y3)[CPL], int t) {
    float y[CPL], ss = 0.f;
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      const float a = fmaf(y3[i], w[i][3], fmaf(y2[i], w[i][2], fmaf(y1[i], w[i][1], y0[i] * w[i][0])));
      y[i] = a / (1.f + expf(-a));
      ss += y[i] * y[i];
    }
    if (!on_v) {
      const float inv = rsqrtf(wave_sum(ss) + 1e-6f) * scale;
#pragma unroll
      for (int i = 0; i < CPL; ++i) y[i] *= inv;
    }
#pragma unroll
    for (int i = 0; i < CPL; ++i)
      if (full || c0 + i < cd) o[(size_t)t * ldo + i] = y[i];
  };
  if (t0 - 3 >= first && t0 + RUN <= T && t0 + RUN <= next) {  // all of one sequence's rows
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < CPL; ++i) x[j][i] = proj[(size_t)(t0 - 3 + j) * ld + ci[i]];
    float f[4][CPL];
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
      for (int i = 0; i < CPL; ++i) f[j][i] = (float)x[j][i];
#pragma unroll
    for (int r = 0; r < RUN; ++r) {
#pragma unroll
      for (int i = 0; i < CPL; ++i) f[(r + 3) & 3][i] = (float)x[r + 3][i];
      row(f[r & 3], f[(r + 1) & 3], f[(r + 2) & 3], f[(r + 3) & 3], t0 + r);
    }
    return;
  }
  float hist[3][CPL];
#pragma unroll
  for (int j = 0; j < 3; ++j)
#pragma unroll
    for (int i = 0; i < CPL; ++i) hist[j][i] = back(t0 - 3 + j, i);
#pragma unroll
  for (int r = 0; r < RUN; ++r) {
    const int t = t0 + r;
    if (t >= T) return;
    if (t == next) {  // the next (non-empty) sequence
      do { ++s; } while (cu[s + 1] == t);
      first = t;
      next = cu[s + 1];
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < CPL; ++i) hist[j][i] = back(t - 3 + j, i);
    }
    float now[CPL];
#pragma unroll
    for (int i = 0; i < CPL; ++i) now[i] = (float)x[r + 3][i];
    row(hist[0], hist[1], hist[2], now, t);
#pragma unroll
    for (int i = 0; i < CPL; ++i) {
      hist[0][i] = hist[1][i];
      hist[1][i] = hist[2][i];
      hist[2][i] = now[i];
    }
  }
}

// ------------------------------------------------------------------------------------------------
// The rule over chunks of 64 tokens, in fp32 on the matrix cores. With G the running sum of the log decay inside a chunk,
// the writes u of the chunk solve (I + L) u = beta (v - e^G k S), L[t, s] = beta_t e^(G_t - G_s) k_t . k_s below the
// diagonal, S the state at the chunk's start. What does not depend on S is done for all chunks at once:
//   gdn_chunk  (one workgroup per chunk and head): Ti = (I + L)^-1 by 16 x 16 blocks,
//              M[t, s] = e^(G_t - G_s) q_t . k_s on and below the diagonal, and the row factors;
//   gdn_carry  (one workgroup per sequence, head and 16 value channels, chunk after chunk): u = Ti beta (v - e^G k S),
//              o = e^G q S + M u, S <- e^(G_end) S + k^T (e^(G_end - G) u).
// MFMA 16x16x4: the contraction runs over 16 indices in four steps, step i taking index 4 * (lane >> 4) + i - the rows a
// lane holds of an accumulator, so S and u feed the next product as B operands straight from the accumulator layout, and
// A operands are 16-byte loads. A wave owns 16 rows of the chunk and its share of S; S, the right side and u reach the
// other waves through LDS, three barriers a chunk. G is summed in double: a chunk's sum reaches -100, and the rounding of a
// difference of such sums would be the largest error of the whole rule. Bound by the chain of chunks; the figures are at
// gai_gdn_chunks.
// ------------------------------------------------------------------------------------------------
constexpr int kC = 64;
constexpr int kFac = 3 * kC;  // per chunk and head: e^G, e^(G_end - G), beta (0 past the chunk's length)

__device__ __forceinline__ f32x4 mfma4(f32x4 a, f32x4 b, f32x4 c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
  return c;
}
__device__ __forceinline__ f32x4 load4f(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
// barrier for LDS contents only: loads from memory that are on their way stay on their way
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int DK>
__global__ __launch_bounds__(256) void gdn_chunk_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                        const float* __restrict__ g, const float* __restrict__ beta,
                                                        const int* __restrict__ chunks, int Hk, int Hv,
                                                        float* __restrict__ To, float* __restrict__ Mo,
                                                        float* __restrict__ Fo) {
  constexpr int LK = DK + 4, LC = kC + 4;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float* Ks = sm;            // [64][LK]
  float* Ti = Ks;            // [64][LC] once k is used up; blocks above the diagonal are not kept
  float* Ls = Ks + kC * (LK > LC ? LK : LC);  // [64][LC]
  __shared__ double Gs[kC];
  __shared__ float Bs[kC];
  const int c = blockIdx.x, h = blockIdx.y, hk = h / (Hv / Hk);
  const int t0 = chunks[2 * c], len = chunks[2 * c + 1];
  const int tid = threadIdx.x, lane = tid & 63, lc = lane & 15, lr = 4 * (lane >> 4);
  const int w = ((tid >> 6) + c + h) & 3;  // this wave's block of 16 rows: block 3 has four tiles, block 0 one
  for (int e = tid; e < kC * DK / 4; e += 256) {
    const int r = e / (DK / 4), col = e % (DK / 4) * 4;
    *reinterpret_cast<f32x4*>(Ks + r * LK + col) =
        r < len ? load4f(k + ((size_t)(t0 + r) * Hk + hk) * DK + col) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (tid < 64) {  // running sum of the log decay
    double x = lane < len ? (double)g[(size_t)(t0 + lane) * Hv + h] : 0.;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const double y = __shfl_up(x, d, 64);
      if (lane >= d) x += y;
    }
    const float bt = lane < len ? beta[(size_t)(t0 + lane) * Hv + h] : 0.f;
    Gs[lane] = x;
    Bs[lane] = bt;
    float* F = Fo + ((size_t)c * Hv + h) * kFac;
    F[lane] = expf((float)x);
    F[kC + lane] = expf((float)(__shfl(x, 63, 64) - x));
    F[2 * kC + lane] = bt;
  }
  f32x4 qf[DK / 16];
  {
    const float* qp = q + ((size_t)(t0 + min(16 * w + lc, len - 1)) * Hk + hk) * DK + lr;
#pragma unroll
    for (int j = 0; j < DK / 16; ++j) qf[j] = load4f(qp + 16 * j);
  }
  __syncthreads();
  float* Mc = Mo + ((size_t)c * Hv + h) * kC * kC;
  for (int m = 0; m <= w; ++m) {  // 16 x 16 tiles on and below the diagonal
    f32x4 kk = {0.f, 0.f, 0.f, 0.f}, qk = kk;
#pragma unroll
    for (int j = 0; j < DK / 16; ++j) {
      const f32x4 b = load4f(Ks + (16 * m + lc) * LK + 16 * j + lr);
      kk = mfma4(load4f(Ks + (16 * w + lc) * LK + 16 * j + lr), b, kk);
      qk = mfma4(qf[j], b, qk);
    }
    const int s = 16 * m + lc;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * w + lr + i;
      const float e = s <= t ? expf((float)(Gs[t] - Gs[s])) : 0.f;
      Ls[t * LC + s] = s < t ? Bs[t] * e * kk[i] : 0.f;
      Mc[t * kC + s] = e * qk[i];
    }
  }
  __syncthreads();
  {  // inverse of the diagonal blocks, one per wave, a column per lane (the four lane groups alike)
    float x[16];
    const float* Lb = Ls + 16 * w * LC + 16 * w;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float a = i == lc ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) a -= Lb[i * LC + j] * x[j];
      x[i] = a;
    }
    if (lane < 16) {
#pragma unroll
      for (int i = 0; i < 16; ++i) Ti[(16 * w + i) * LC + 16 * w + lc] = x[i];
    }
  }
  __syncthreads();
  for (int d = 1; d < 4; ++d) {  // blocks d below the diagonal: Ti[w][j] = -Ti[w][w] sum_m L[w][m] Ti[m][j]
    if (w >= d) {
      const int j = w - d;
      f32x4 a = {0.f, 0.f, 0.f, 0.f};
      for (int m = j; m < w; ++m) {
        f32x4 b;
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = Ti[(16 * m + lr + i) * LC + 16 * j + lc];
        a = mfma4(load4f(Ls + (16 * w + lc) * LC + 16 * m + lr), b, a);
      }
      a = mfma4(load4f(Ti + (16 * w + lc) * LC + 16 * w + lr), a, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
      for (int i = 0; i < 4; ++i) Ti[(16 * w + lr + i) * LC + 16 * j + lc] = -a[i];
    }
    __syncthreads();
  }
  float* Tc = To + ((size_t)c * Hv + h) * kC * kC;
  for (int e = tid; e < kC * kC / 4; e += 256) {
    const int r = e / (kC / 4), col = e % (kC / 4) * 4;
    *reinterpret_cast<f32x4*>(Tc + r * kC + col) = col / 16 <= r / 16 ? load4f(Ti + r * LC + col) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// Of a chunk's products only k S, Ti x and k^T u are between one S and the next. Waves 0 - 3 make those, at the higher priority;
// waves 4 - 7 make o of the chunk before meanwhile, q S and M u, and bring k into LDS (it is read both by rows and by columns). A SIMD's
// matrix unit has 1.75 us of work a chunk (128 x 128, 16 value channels), its chain 1.1 us and the latencies of three barriers: four
// waves that did one after the other took 4.5 us a chunk, these 3.0 (the chain by itself about 2.1). (Loaded by columns from memory, k made 64 loads a chunk,
// more than the counter of outstanding loads holds: 5.9 us.)
template <int DK>
__global__ __launch_bounds__(512, 1) void gdn_carry_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ To,
    const float* __restrict__ Mo, const float* __restrict__ Fo, const int* __restrict__ chunks,
    const int* __restrict__ chunk0, const int* __restrict__ slots, int Hk, int Hv, int DV, float* __restrict__ state,
    float* __restrict__ out) {
  constexpr int NT = DK / 16, ST = NT / 4;  // row tiles of S, of which each of four waves owns ST
  constexpr int LK = DK + 4, KR = kC * DK / 1024;  // 16-byte pieces of a k chunk per thread of four waves
  extern __shared__ __attribute__((aligned(16))) float sm[];
  f32x4* Ss = reinterpret_cast<f32x4*>(sm);  // [3][NT * 64]: chunk i's at i % 3
  f32x4* Rs = Ss + 3 * NT * 64;              // [4 * 64]
  f32x4* Us = Rs + 4 * 64;                   // [2][4 * 64]
  f32x4* Ud = Us + 8 * 64;                   // [4 * 64]
  float* Ks = reinterpret_cast<float*>(Ud + 4 * 64);  // [2][64][LK]
  const int tid = threadIdx.x & 255, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), lc = lane & 15,
            lr = 4 * (lane >> 4);
  const bool chain = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) == 0;
  const int id = xcd_remap(blockIdx.x, gridDim.x), ns = DV / 16;  // the slices of a head share its rows in one XCD's L2
  const int n = id % ns, h = id / ns % Hv, s = id / ns / Hv, hk = h / (Hv / Hk);
  const int c0 = chunk0[s], nc = chunk0[s + 1] - c0;
  if (nc <= 0) return;
  // A chunk's rows through buffers that begin at its first row and end at its last one (past it: zeros; stores are dropped), so
  // that a lane's offsets are the same for every chunk. The chunk's entry is read a chunk ahead of them: a scalar load
  // and the address arithmetic of every load cost the chain 0.4 us a chunk.
  struct Entry {
    int t0, len;
  };
  auto entry = [&](int i) { return Entry{chunks[2 * (c0 + min(i, nc - 1))], chunks[2 * (c0 + min(i, nc - 1)) + 1]}; };
  auto buffer = [&](const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, bytes, 0x00020000);
  };
  auto get4 = [&](const __amdgpu_buffer_rsrc_t& r, int off) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  };
  if (chain) {
    __builtin_amdgcn_s_setprio(3);
    float* Sg = state + ((size_t)slots[s] * Hv + h) * DK * DV + 16 * n + lc;
    f32x4 S[ST], kp[NT];
#pragma unroll
    for (int j = 0; j < ST; ++j) {
#pragma unroll
      for (int i = 0; i < 4; ++i) S[j][i] = Sg[(size_t)(16 * (ST * w + j) + lr + i) * DV];
      Ss[(ST * w + j) * 64 + lane] = S[j];
    }
    struct Rows {  // this wave's 16 rows of Ti, v and the factors
      f32x4 T[4], v, e0, ed, bt;
      float eg;
    };
    int ov[4], oT[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ov[i] = ((16 * w + lr + i) * Hv * DV + lc) * 4;
      oT[i] = ((16 * w + lc) * kC + 16 * min(i, w) + lr) * 4;
    }
    const int oF = (16 * w + lr) * 4;
    auto fetch = [&](int c, const Entry& e, Rows& r) {  // past the chunk's end: beta is 0, so the row's write is
      const size_t ch = (size_t)(c0 + c) * Hv + h;
      const auto bv = buffer(v + ((size_t)e.t0 * Hv + h) * DV + 16 * n, (e.len - 1) * Hv * DV * 4 + 64);
      const auto bT = buffer(To + ch * kC * kC, kC * kC * 4), bF = buffer(Fo + ch * kFac, kFac * 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        r.v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(bv, ov[i], 0, 0));
        r.T[i] = get4(bT, oT[i]);
      }
      r.e0 = get4(bF, oF);
      r.ed = get4(bF, oF + kC * 4);
      r.bt = get4(bF, oF + 2 * kC * 4);
      r.eg = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(bF, (kC - 1) * 4, 0, 0));
    };
    auto read_k = [&](int c) {
#pragma unroll
      for (int j = 0; j < NT; ++j) kp[j] = load4f(Ks + ((c & 1) * kC + 16 * w + lc) * LK + 16 * j + lr);
    };
    Entry ahead = entry(1);  // of the chunk after the one at work
    auto step = [&](int c, const Rows& r, Rows& next) {
      const float* Kb = Ks + (c & 1) * kC * LK;
      const f32x4* Sb = Ss + c % 3 * NT * 64;
      f32x4 p[2] = {}, u = {0.f, 0.f, 0.f, 0.f}, x, ud, kc[4][ST];
      lds_barrier();  // S of this chunk is in LDS
      if (c + 1 < nc) fetch(c + 1, ahead, next);
      ahead = entry(c + 2);
#pragma unroll
      for (int j = 0; j < NT; ++j) p[j & 1] = mfma4(kp[j], Sb[j * 64 + lane], p[j & 1]);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = r.bt[i] * (r.v[i] - r.e0[i] * (p[0][i] + p[1][i]));
      Rs[w * 64 + lane] = x;
      lds_barrier();
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (m <= w) u = mfma4(r.T[m], Rs[m * 64 + lane], u);
#pragma unroll
      for (int i = 0; i < 4; ++i) ud[i] = u[i] * r.ed[i];
      Us[(c & 1) * 256 + w * 64 + lane] = u;
      Ud[w * 64 + lane] = ud;
#pragma unroll
      for (int j = 0; j < ST; ++j) {
#pragma unroll
        for (int i = 0; i < 4; ++i) S[j][i] *= r.eg;
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) kc[m][j][i] = Kb[(16 * m + lr + i) * LK + 16 * (ST * w + j) + lc];
      }
      lds_barrier();  // u, and k of the next chunk
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const f32x4 um = Ud[m * 64 + lane];
#pragma unroll
        for (int j = 0; j < ST; ++j) S[j] = mfma4(kc[m][j], um, S[j]);
      }
#pragma unroll
      for (int j = 0; j < ST; ++j) Ss[((c + 1) % 3 * NT + ST * w + j) * 64 + lane] = S[j];
      if (c + 1 < nc) read_k(c + 1);
    };
    Rows ra, rb;
    fetch(0, entry(0), ra);
    lds_barrier();  // k of the first chunk
    read_k(0);
    for (int c = 0; c < nc; c += 2) {
      step(c, ra, rb);
      if (c + 1 < nc) step(c + 1, rb, ra);
    }
    lds_barrier();
#pragma unroll
    for (int j = 0; j < ST; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) Sg[(size_t)(16 * (ST * w + j) + lr + i) * DV] = S[j][i];
  } else {
    struct Rows {  // this wave's 16 rows of q, M and e^G
      f32x4 Q[NT], M[4], e0;
      Entry e;
    };
    f32x4 K[KR];
    int ok[KR], oM[4], oo[4];
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      const int e = tid + 256 * j;
      ok[j] = (e / (DK / 4) * Hk * DK + e % (DK / 4) * 4) * 4;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      oM[i] = ((16 * w + lc) * kC + 16 * min(i, w) + lr) * 4;
      oo[i] = ((16 * w + lr + i) * Hv * DV + lc) * 4;
    }
    const int oq = ((16 * w + lc) * Hk * DK + lr) * 4, oF = (16 * w + lr) * 4;
    auto fetch_k = [&](const Entry& e) {
      const auto bk = buffer(k + ((size_t)e.t0 * Hk + hk) * DK, ((e.len - 1) * Hk + 1) * DK * 4);
#pragma unroll
      for (int j = 0; j < KR; ++j) K[j] = get4(bk, ok[j]);
    };
    auto stage_k = [&](int c) {
#pragma unroll
      for (int j = 0; j < KR; ++j) {
        const int e = tid + 256 * j;
        *reinterpret_cast<f32x4*>(Ks + ((c & 1) * kC + e / (DK / 4)) * LK + e % (DK / 4) * 4) = K[j];
      }
    };
    auto fetch = [&](int c, const Entry& e, Rows& r) {
      const size_t ch = (size_t)(c0 + c) * Hv + h;
      const auto bq = buffer(q + ((size_t)e.t0 * Hk + hk) * DK, ((e.len - 1) * Hk + 1) * DK * 4);
      const auto bM = buffer(Mo + ch * kC * kC, kC * kC * 4);
      r.e = e;
#pragma unroll
      for (int j = 0; j < NT; ++j) r.Q[j] = get4(bq, oq + 64 * j);
#pragma unroll
      for (int i = 0; i < 4; ++i) r.M[i] = get4(bM, oM[i]);
      r.e0 = get4(buffer(Fo + ch * kFac, kFac * 4), oF);
    };
    // operands are read ahead of the barrier that their products follow: those then run while the chain waits for its own
    constexpr int HT = NT / 2;
    f32x4 o[2], a[HT > 4 ? HT : 4];
    auto read_s = [&](int c, int half) {
#pragma unroll
      for (int j = 0; j < HT; ++j) a[j] = Ss[(c % 3 * NT + half * HT + j) * 64 + lane];
    };
    auto q_s = [&](const Rows& r, auto half) {
      constexpr int H = decltype(half)::value * HT;
#pragma unroll
      for (int j = 0; j < HT; ++j) o[(H + j) & 1] = mfma4(r.Q[H + j], a[j], o[(H + j) & 1]);
    };
    auto read_u = [&](int c) {
#pragma unroll
      for (int m = 0; m < 4; ++m) a[m] = Us[(c & 1) * 256 + m * 64 + lane];
    };
    auto rest = [&](const Rows& r) {
#pragma unroll
      for (int i = 0; i < 4; ++i) o[0][i] = r.e0[i] * (o[0][i] + o[1][i]);
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (m <= w) o[0] = mfma4(r.M[m], a[m], o[0]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[0][i]),
                                              buffer(out + ((size_t)r.e.t0 * Hv + h) * DV + 16 * n, (r.e.len - 1) * Hv * DV * 4 + 64),
                                              oo[i], 0, 0);
    };
    using First = std::integral_constant<int, 0>;
    using Second = std::integral_constant<int, 1>;
    // while the others are at chunk c: o of chunk c - 1 (r), k of c + 1 into LDS, k of c + 2 and the rows of c on their way
    Entry e0 = entry(0), e1 = entry(1), e2 = entry(2);  // of chunks c, c + 1, c + 2
    auto step = [&](int c, const Rows& r, Rows& next) {
      o[0] = o[1] = f32x4{0.f, 0.f, 0.f, 0.f};
      lds_barrier();
      if (c > 0) {
        q_s(r, First{});
        read_s(c - 1, 1);
      }
      fetch(c, e0, next);
      e0 = e1;
      e1 = e2;
      e2 = entry(c + 3);
      lds_barrier();
      if (c > 0) {
        q_s(r, Second{});
        read_u(c - 1);
      }
      if (c + 1 < nc) {
        stage_k(c + 1);
        if (c + 2 < nc) fetch_k(e1);
      }
      lds_barrier();
      if (c > 0) rest(r);
      read_s(c, 0);
    };
    Rows ra, rb;
    fetch_k(e0);
    stage_k(0);
    if (nc > 1) fetch_k(e1);
    lds_barrier();
    for (int c = 0; c < nc; c += 2) {
      step(c, rb, ra);
      if (c + 1 < nc) step(c + 1, ra, rb);
    }
    lds_barrier();
    const Rows& r = nc & 1 ? ra : rb;
    o[0] = o[1] = f32x4{0.f, 0.f, 0.f, 0.f};
    q_s(r, First{});
    read_s(nc - 1, 1);
    q_s(r, Second{});
    read_u(nc - 1);
    rest(r);
  }
}

// Four waves do everything, a chunk's rows are fetched when it begins: key heads of 256, for two chunks of which there are neither
// registers nor LDS, and many short portions (the rule at the launch), where the next workgroup hides what the next chunk does not.
template <int DK>
__global__ __launch_bounds__(256, 1) void gdn_carry_plain_kernel(
    const float* __restrict__ q, const float* __restrict__ k, const float* __restrict__ v, const float* __restrict__ To,
    const float* __restrict__ Mo, const float* __restrict__ Fo, const int* __restrict__ chunks,
    const int* __restrict__ chunk0, const int* __restrict__ slots, int Hk, int Hv, int DV, float* __restrict__ state,
    float* __restrict__ out) {
  constexpr int NT = DK / 16, ST = NT / 4;  // row tiles of S, of which each wave owns ST
  constexpr int LK = DK + 4, KR = kC * DK / 1024;  // 16-byte pieces of a k chunk per thread
  extern __shared__ __attribute__((aligned(16))) float sm[];
  f32x4* Ss = reinterpret_cast<f32x4*>(sm);  // [2][NT * 64]
  f32x4* Rs = Ss + 2 * NT * 64;              // [4 * 64] each
  f32x4* Us = Rs + 4 * 64;
  f32x4* Ud = Us + 4 * 64;
  float* Ks = reinterpret_cast<float*>(Ud + 4 * 64);  // [64][LK]
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, lc = lane & 15, lr = 4 * (lane >> 4);
  const int id = xcd_remap(blockIdx.x, gridDim.x), ns = DV / 16;  // the slices of a head share its rows in one XCD's L2
  const int n = id % ns, h = id / ns % Hv, s = id / ns / Hv, hk = h / (Hv / Hk);
  const int c0 = chunk0[s], c1 = chunk0[s + 1];
  if (c1 <= c0) return;
  float* Sg = state + ((size_t)slots[s] * Hv + h) * DK * DV + 16 * n + lc;
  f32x4 S[ST];
#pragma unroll
  for (int j = 0; j < ST; ++j) {
#pragma unroll
    for (int i = 0; i < 4; ++i) S[j][i] = Sg[(size_t)(16 * (ST * w + j) + lr + i) * DV];
    Ss[(ST * w + j) * 64 + lane] = S[j];
  }
  struct Rows {  // what a chunk needs besides S: its k (shared), this wave's 16 rows of q, Ti, M and v
    f32x4 K[KR], Q[NT], T[4], M[4], v, e0, ed, bt;
    float eg;
    int t0, len;
  };
  auto fetch = [&](int c, Rows& r) {
    const size_t ch = (size_t)c * Hv + h;
    r.t0 = chunks[2 * c];
    r.len = chunks[2 * c + 1];
    const int last = r.len - 1;
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      const int e = tid + 256 * j;
      r.K[j] = load4f(k + ((size_t)(r.t0 + min(e / (DK / 4), last)) * Hk + hk) * DK + e % (DK / 4) * 4);
    }
    const float* qp = q + ((size_t)(r.t0 + min(16 * w + lc, last)) * Hk + hk) * DK + lr;
#pragma unroll
    for (int j = 0; j < NT; ++j) r.Q[j] = load4f(qp + 16 * j);
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // past the chunk's end: beta is 0, so the row's write is
      r.v[i] = v[((size_t)(r.t0 + min(16 * w + lr + i, last)) * Hv + h) * DV + 16 * n + lc];
      r.T[i] = load4f(To + (ch * kC + 16 * w + lc) * kC + 16 * min(i, w) + lr);
      r.M[i] = load4f(Mo + (ch * kC + 16 * w + lc) * kC + 16 * min(i, w) + lr);
    }
    const float* F = Fo + ch * kFac;
    r.e0 = load4f(F + 16 * w + lr);
    r.ed = load4f(F + kC + 16 * w + lr);
    r.bt = load4f(F + 2 * kC + 16 * w + lr);
    r.eg = F[kC - 1];
  };
  auto stage = [&](const Rows& r) {
#pragma unroll
    for (int j = 0; j < KR; ++j) {
      const int e = tid + 256 * j;
      *reinterpret_cast<f32x4*>(Ks + e / (DK / 4) * LK + e % (DK / 4) * 4) = r.K[j];
    }
  };
  auto step = [&](int b, const Rows& r) {
    lds_barrier();  // S and k of this chunk are in LDS
    const f32x4* Sb = Ss + b * NT * 64;
    const float* Kb = Ks;
    f32x4 p[2] = {}, o[2] = {}, u = {0.f, 0.f, 0.f, 0.f}, x, ud;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const f32x4 sj = Sb[j * 64 + lane];
      p[j & 1] = mfma4(load4f(Kb + (16 * w + lc) * LK + 16 * j + lr), sj, p[j & 1]);
      o[j & 1] = mfma4(r.Q[j], sj, o[j & 1]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i] = r.bt[i] * (r.v[i] - r.e0[i] * (p[0][i] + p[1][i]));
      o[0][i] = r.e0[i] * (o[0][i] + o[1][i]);
    }
    Rs[w * 64 + lane] = x;
    lds_barrier();
#pragma unroll
    for (int m = 0; m < 4; ++m)
      if (m <= w) u = mfma4(r.T[m], Rs[m * 64 + lane], u);
#pragma unroll
    for (int i = 0; i < 4; ++i) ud[i] = u[i] * r.ed[i];
    Us[w * 64 + lane] = u;
    Ud[w * 64 + lane] = ud;
#pragma unroll
    for (int j = 0; j < ST; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) S[j][i] *= r.eg;
    lds_barrier();
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const f32x4 um = Ud[m * 64 + lane];
#pragma unroll
      for (int j = 0; j < ST; ++j) {
        f32x4 kc;
#pragma unroll
        for (int i = 0; i < 4; ++i) kc[i] = Kb[(16 * m + lr + i) * LK + 16 * (ST * w + j) + lc];
        S[j] = mfma4(kc, um, S[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < ST; ++j) Ss[(b ^ 1) * NT * 64 + (ST * w + j) * 64 + lane] = S[j];
#pragma unroll
    for (int m = 0; m < 4; ++m)
      if (m <= w) o[0] = mfma4(r.M[m], Us[m * 64 + lane], o[0]);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = 16 * w + lr + i;
      if (t < r.len) out[((size_t)(r.t0 + t) * Hv + h) * DV + 16 * n + lc] = o[0][i];
    }
  };
  for (int c = c0; c < c1; ++c) {
    Rows r;
    fetch(c, r);
    lds_barrier();  // the last chunk's k has been read
    stage(r);
    step((c - c0) & 1, r);
  }
#pragma unroll
  for (int j = 0; j < ST; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) Sg[(size_t)(16 * (ST * w + j) + lr + i) * DV] = S[j][i];
}

// y = silu(z) * (w * norm(o)), with the roundings to the model's type of the published formulation (after the norm, after
// the weight, at the end). A wave takes R heads in a row, all of whose loads are in flight at once (10095 tokens x 16 heads
// of 128: 165 MB, 67 -> 41 us; one head a wave waited for the row, the sum, the row again); NJ 0 reads heads of any width
// twice.
template <typename TA, int NJ, int R>
__global__ __launch_bounds__(256) void gdn_out_kernel(const float* __restrict__ o, const TA* __restrict__ z, int ldz,
                                                      const TA* __restrict__ w, TA* __restrict__ y, int TH, int Hv, int DV,
                                                      float eps) {
  const int lane = threadIdx.x & 63;
  const int th0 = (blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * R;
  if constexpr (NJ == 0) {
    if (th0 >= TH) return;
    const float* orow = o + (size_t)th0 * DV;
    float s = 0.f;
    for (int i = lane; i < DV; i += 64) s += orow[i] * orow[i];
    const float inv = rsqrtf(wave_sum(s) / DV + eps);
    const TA* zr = z + (size_t)(th0 / Hv) * ldz + (size_t)(th0 % Hv) * DV;
    for (int i = lane; i < DV; i += 64) {
      const float zf = (float)zr[i];
      const TA a = (TA)(orow[i] * inv), b = (TA)((float)w[i] * (float)a);
      y[(size_t)th0 * DV + i] = (TA)((float)b * (zf / (1.f + expf(-zf))));
    }
    return;
  }
  constexpr int N = NJ ? NJ : 1;
  float x[R][N], g[N];
  TA zv[R][N];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int th = min(th0 + r, TH - 1);  // past the end: the last head's values, not written
    const float* orow = o + (size_t)th * DV;
    const TA* zr = z + (size_t)(th / Hv) * ldz + (size_t)(th % Hv) * DV;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {  // no branch parts the loads
      const int i = min(lane + 64 * j, DV - 1);
      x[r][j] = orow[i];
      zv[r][j] = zr[i];
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) g[j] = (float)w[min(lane + 64 * j, DV - 1)];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) s = lane + 64 * j < DV ? fmaf(x[r][j], x[r][j], s) : s;
    const float inv = rsqrtf(wave_sum(s) / DV + eps);
    if (th0 + r >= TH) return;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const float zf = (float)zv[r][j];
      const TA a = (TA)(x[r][j] * inv), b = (TA)(g[j] * (float)a);
      if (lane + 64 * j < DV) y[(size_t)(th0 + r) * DV + lane + 64 * j] = (TA)((float)b * (zf / (1.f + expf(-zf))));
    }
  }
}

}  // namespace

void gai_gdn_prep(const void* proj, int ld, const float* cw, const float* cstate, const int* cu, const int* slots, int S,
                  int T, int Hk, int Hv, int DK, int DV, const float* A_log, const float* dt_bias, float* q, float* k,
                  float* v, float* g, float* beta, int dt, hipStream_t st) {
  if (T == 0) return;
  const int vecs = 2 * Hk + (Hv * DV + DK - 1) / DK;
  // few tokens (decode steps): one token per wave, or the chip stays empty
#define GAI_PREP(TA, D, RUN)                                                                                            \
  gdn_prep_kernel<TA, D, RUN><<<dim3((T + RUN - 1) / RUN, (vecs + 3) / 4 + 1), 256, 0, st>>>(                           \
      (const TA*)proj, ld, cw, cstate, cu, slots, S, T, Hk, Hv, DV, A_log, dt_bias, q, k, v, g, beta)
#define GAI_PREP_D(D)                                                                                                   \
  if (DK == D) {                                                                                                        \
    if (dt) { if (T > 512) GAI_PREP(float, D, 8); else GAI_PREP(float, D, 1); }                                         \
    else { if (T > 512) GAI_PREP(bf16, D, 8); else GAI_PREP(bf16, D, 1); }                                              \
    GAI_LAUNCH_CHECK();                                                                                                 \
    return;                                                                                                             \
  }
  GAI_PREP_D(64)
  GAI_PREP_D(128)
  GAI_PREP_D(256)
#undef GAI_PREP_D
#undef GAI_PREP
  gai_launch_error(__FILE__, __LINE__, "gdn_prep: key head dim must be 64, 128 or 256");
}

// 6000 + 4095 tokens, 8 key / 16 value heads of 128 x 128: gdn_chunk 90 us (two workgroups a CU, the inverse beside k in LDS, and the
// block of four tiles always on one SIMD: 101; its bytes alone 45), gdn_carry 290 us (94 chunks in a row at 3.0 us,
// 256 workgroups), against 47 ms for the same rule as batched fp32 products and triangular solves chunk by chunk in torch;
// error of o against float64 2.2e-7 - 3.4e-7 (torch 3.2e-7 - 1.1e-6).
// Key heads of 64 and many workgroups: two plain ones share a CU, which hides more than one of split roles does by itself. us with
// gdn_chunk, split / plain, 16 heads of 64 x 128: 64 portions of 16 tokens 136 / 94, of 300 522 / 452, of 1000 1525 / 1379; 8
// portions of one token (1024 workgroups) 25 / 21, 16 of 190 82 / 73. 8 heads of 64 x 64, 32 portions of 250 (1024 workgroups, four chunks
// each) 70.0 / 71.3, 2 of 5000 217 / 314.
void gai_gdn_chunks(const float* q, const float* k, const float* v, const float* g, const float* beta, const int* chunks,
                    const int* chunk0, const int* slots, int nc, int S, int Hk, int Hv, int DK, int DV, float* Ti, float* M,
                    float* F, float* state, float* out, hipStream_t st) {
  if (nc == 0) return;
#define GAI_GDN(D)                                                                                                      \
  if (DK == D) {                                                                                                        \
    const int lds = (kC * (D + 4) + kC * (kC + 4)) * 4;                                                                 \
    const int wgs = S * Hv * (DV / 16);                                                                                 \
    constexpr int lds_plain = (2 * D / 16 + 12) * 64 * 16 + kC * (D + 4) * 4;                                           \
    constexpr int lds_split = (3 * D / 16 + 16) * 64 * 16 + 2 * kC * (D + 4) * 4;                                       \
    constexpr int DP = D == 128 ? 64 : D, DS = D > 128 ? 128 : D; /* the widths that either kernel is reached with */   \
    const bool plain = D > 128 || (D == 64 && (wgs >= 2048 || (wgs > 256 && nc < 4 * S)));                             \
    static bool once = false;                                                                                           \
    if (!once) {                                                                                                        \
      auto allow = [](const void* f, int bytes) {                                                                       \
        (void)hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);                                \
      };                                                                                                                \
      allow(reinterpret_cast<const void*>(gdn_chunk_kernel<D>), lds);                                                   \
      allow(reinterpret_cast<const void*>(gdn_carry_plain_kernel<DP>), lds_plain);                                       \
      if (D <= 128) allow(reinterpret_cast<const void*>(gdn_carry_kernel<DS>), lds_split);                              \
      once = true;                                                                                                      \
    }                                                                                                                   \
    gdn_chunk_kernel<D><<<dim3(nc, Hv), 256, lds, st>>>(q, k, g, beta, chunks, Hk, Hv, Ti, M, F);                       \
    GAI_LAUNCH_CHECK();                                                                                                 \
    if (plain)                                                                                                          \
      gdn_carry_plain_kernel<DP><<<wgs, 256, lds_plain, st>>>(q, k, v, Ti, M, F, chunks, chunk0, slots, Hk, Hv, DV,      \
                                                             state, out);                                               \
    else                                                                                                                \
      gdn_carry_kernel<DS><<<wgs, 512, lds_split, st>>>(q, k, v, Ti, M, F, chunks, chunk0, slots, Hk, Hv, DV, state,    \
                                                        out);                                                           \
    GAI_LAUNCH_CHECK();                                                                                                 \
    return;                                                                                                             \
  }
  GAI_GDN(64)
  GAI_GDN(128)
  GAI_GDN(256)
#undef GAI_GDN
  gai_launch_error(__FILE__, __LINE__, "gdn_chunks: key head dim must be 64, 128 or 256");
}

void gai_gdn_out(const float* o, const void* z, int ldz, const void* w, void* y, int T, int Hv, int DV, float eps, int dt,
                 hipStream_t st) {
  const int TH = T * Hv;
  if (TH == 0) return;
  // One head a wave where few heads leave the chip empty, four where their loads in flight pay. us a launch, one | four a wave, heads
  // of 128: 2048 heads 2.6 | 3.9, 10240 4.5 | 5.1, 16384 6.0 | 6.1, 32768 9.6 | 9.5, 65536 18.7 | 17.7, 192000 49.5 | 42.4; of 64:
  // 8192 3.4 | 3.7, 16384 4.9 | 5.0, 32768 7.9 | 7.3.
#define GAI_OUT(TA, NJ, R)                                                                                              \
  gdn_out_kernel<TA, NJ, R><<<(TH + 4 * R - 1) / (4 * R), 256, 0, st>>>(o, (const TA*)z, ldz, (const TA*)w, (TA*)y, TH, Hv, \
                                                                        DV, eps)
#define GAI_OUT_N(TA)                                                                                                   \
  if (DV <= 128) { if (TH > 16384) GAI_OUT(TA, 2, 4); else GAI_OUT(TA, 2, 1); }                                            \
  else if (DV <= 256) GAI_OUT(TA, 4, 1);                                                                                \
  else GAI_OUT(TA, 0, 1)
  if (dt) { GAI_OUT_N(float); } else { GAI_OUT_N(bf16); }
#undef GAI_OUT_N
#undef GAI_OUT
  GAI_LAUNCH_CHECK();
}

void gai_gdn_decode(const float* q, const float* k, const float* v, const float* g, const float* beta, float* state,
                    const int* slots, float* out, int B, int Hk, int Hv, int DK, int DV, hipStream_t st) {
  if (B == 0) return;
  const dim3 grid(Hv, B);
#define GAI_GDN(D)                                                                                    \
  if (DK == D) {                                                                                      \
    gdn_decode_kernel<D><<<grid, D * 4, 0, st>>>(q, k, v, g, beta, state, slots, out, Hk, Hv, DV);    \
    GAI_LAUNCH_CHECK();                                                                               \
    return;                                                                                           \
  }
  GAI_GDN(64)
  GAI_GDN(128)
  GAI_GDN(256)
#undef GAI_GDN
  gai_launch_error(__FILE__, __LINE__, "gdn_decode: key head dim must be 64, 128 or 256");
}
