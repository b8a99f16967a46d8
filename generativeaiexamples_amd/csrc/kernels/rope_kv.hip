// Fused RoPE + paged KV-cache write.
//
// Input is the packed output of the fused QKV projection, [T, (Hq + 2*Hkv) * D].
// Per token it (1) rotates q and k (neox rotate-half pairs (i, i + D/2) with a
// host-precomputed fp32 cos/sin table [max_pos, D] = [cos(D/2) | sin(D/2)]),
// (2) writes q to q_out [T, Hq, D], (3) writes k into the paged K cache laid out
// [num_blocks, Hkv, 16, D] and v into the *transposed* paged V cache
// [num_blocks, Hkv, D, 16] -- the V^T layout lets both attention kernels feed
// P.V MFMAs with 8-byte contiguous loads (no LDS transpose).
// slot_mapping[t] = block * 16 + offset, or < 0 to skip the cache write.
// rope == 0 skips the rotation (encoder / BERT path).
// KV = fp8: the cache holds OCP e4m3fn values x / scale (per-layer k / v scales, saturated) -- the fp8 KV
// cache option, half the bytes per token for decode attention.
#include "gai_common.h"
#include "gai_kernels.h"
#include "gai_rope.h"

using namespace gai;

namespace {

template <int D, typename KV>
__global__ __launch_bounds__(256) void rope_kv_kernel(const bf16* __restrict__ qkv, const int* __restrict__ pos,
                                                      const float* __restrict__ cos_sin,
                                                      const int* __restrict__ slots, bf16* __restrict__ q_out,
                                                      KV* __restrict__ k_cache, KV* __restrict__ v_cache,
                                                      int T, int Hq, int Hkv, int rope, float inv_ks, float inv_vs) {
  constexpr int LPH = D / 8;  // lanes per head: each lane owns 4 rotation pairs
  constexpr int HPB = 256 / LPH;
  if (threadIdx.x >= HPB * LPH) return;  // D = 96: 12 lanes per head, 21 heads per block, 4 idle lanes
  const int H = Hq + 2 * Hkv;
  const long item = (long)blockIdx.x * HPB + threadIdx.x / LPH;  // (token, head)
  if (item >= (long)T * H) return;
  const int t = (int)(item / H), h = (int)(item % H);
  const int i0 = (threadIdx.x % LPH) * 4;  // pair indices i0..i0+3 and i0+D/2..
  const bf16* src = qkv + ((size_t)t * H + h) * D;
  const bf16x4 x1 = *reinterpret_cast<const bf16x4*>(src + i0);
  const bf16x4 x2 = *reinterpret_cast<const bf16x4*>(src + i0 + D / 2);
  rope_kv_store<D>(x1, x2, t, h, i0, pos, cos_sin, slots, q_out, k_cache, v_cache, Hq, Hkv, rope, inv_ks, inv_vs);
}

// The same for a prompt's tokens and bf16 pages, with an optional RMS norm of every q and k head (weights wq / wk, rounded to bf16 before
// the rotation). Bound by one read and one write of the rows; what kept it from that was V^T, whose elements went out two bytes at a time,
// 32 bytes apart (a page row is one channel of 16 tokens). Here a workgroup takes four heads of q and k of TOK tokens - 16-byte loads and stores,
// all four heads' rows in flight, the token's angles read once for them - or one head of v of half as many, 16 bytes a thread, turned in LDS:
// eight tokens that fill half a page row go out as 16 bytes, others (a prompt that begins anywhere in the packed rows, tokens in pages of
// their own) a token's neighbours side by side, all at once: one after the other they took 400 tokens in pages of their own to 7.2 us for 6.3.
// Us, rope_kv_kernel | here | here, prompts that begin off a half page: 10095 tokens of 16 + 4 + 4 heads of 128 39.4 | 24.2 | 25.5, 3389 of 32 + 8 + 8
// 28.9 | 14.5 | 15.5, 999 12.1 | 5.2 | 5.8, 187 4.1 | 3.2 | 3.2; 3000 of 3 x 16 of 64 22.8 | 7.3 | 8.9. With the norm, which was copies of the heads, two
// norm launches and copies back, 10095 tokens 119 | 23.9.
template <int D>
constexpr int value_tokens() { return 256 / (D / 8) / 8 * 8; }  // 16 bytes a thread
template <int D>
constexpr int rows_tokens() { return 2 * value_tokens<D>(); }
constexpr int kHeadsAWg = 4;

template <int D, bool NORM>
__global__ __launch_bounds__(256) void rope_kv_rows_kernel(const bf16* __restrict__ qkv, const int* __restrict__ pos,
                                                           const float* __restrict__ cos_sin, const int* __restrict__ slots,
                                                           bf16* __restrict__ q_out, bf16* __restrict__ k_cache,
                                                           bf16* __restrict__ v_cache, int T, int Hq, int Hkv, int rope,
                                                           const bf16* __restrict__ wq, const bf16* __restrict__ wk, float eps) {
  constexpr int LP = D / 16, TOK = rows_tokens<D>(), LV = D / 8, TV = value_tokens<D>();
  __shared__ __attribute__((aligned(16))) bf16 vs[TV][D + 8];
  const int tid = threadIdx.x, H = Hq + 2 * Hkv, qk = (Hq + Hkv + kHeadsAWg - 1) / kHeadsAWg;
  if ((int)blockIdx.y < qk) {
    const int t = blockIdx.x * TOK + tid / LP, i0 = tid % LP * 8;
    if (tid >= TOK * LP || t >= T) return;
    const int h0 = blockIdx.y * kHeadsAWg, hn = min(kHeadsAWg, Hq + Hkv - h0), slot = slots[t];
    const bf16* src = qkv + ((size_t)t * H + h0) * D + i0;
    bf16x8 x[kHeadsAWg][2];
#pragma unroll
    for (int j = 0; j < kHeadsAWg; ++j)
      if (j < hn) {
        x[j][0] = load8(src + j * D);
        x[j][1] = load8(src + j * D + D / 2);
      }
    float c[8], s[8];
    if (rope) {
      const float* cs = cos_sin + (size_t)pos[t] * D + i0;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        c[e] = cs[e];
        s[e] = cs[e + D / 2];
      }
    }
#pragma unroll
    for (int j = 0; j < kHeadsAWg; ++j) {
      if (j >= hn) break;
      const int h = h0 + j;
      if constexpr (NORM) {
        float ss = 0.f;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int e = 0; e < 8; ++e) ss += (float)x[j][u][e] * (float)x[j][u][e];
#pragma unroll
        for (int d = 1; d < LP; d <<= 1) ss += __shfl_xor(ss, d, 64);
        const float inv = rsqrtf(ss / D + eps);
        const bf16* w = (h < Hq ? wq : wk) + i0;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const bf16x8 g = load8(w + u * (D / 2));
#pragma unroll
          for (int e = 0; e < 8; ++e) x[j][u][e] = (bf16)((float)x[j][u][e] * inv * (float)g[e]);
        }
      }
      if (rope) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float a = (float)x[j][0][e], b = (float)x[j][1][e];
          x[j][0][e] = (bf16)(a * c[e] - b * s[e]);
          x[j][1][e] = (bf16)(b * c[e] + a * s[e]);
        }
      }
      bf16* dst;
      if (h < Hq) dst = q_out + ((size_t)t * Hq + h) * D + i0;
      else if (slot >= 0) dst = k_cache + (((size_t)(slot / kKvBlock) * Hkv + h - Hq) * kKvBlock + slot % kKvBlock) * D + i0;
      else continue;
      store8(dst, x[j][0]);
      store8(dst + D / 2, x[j][1]);
    }
    return;
  }
  // an eight of tokens: rows r & ~7 on, D threads, j the one of them
  const int y = blockIdx.y - qk, g = y >> 1, r = tid / LV, col = tid % LV * 8, t = (2 * blockIdx.x + (y & 1)) * TV + r;
  const int r8 = r & ~7, tg = t - (r & 7), j = tid - r8 * LV, tj = tg + (j & 7);
  const bf16x8 x = load8(qkv + ((size_t)min(t, T - 1) * H + Hq + Hkv + g) * D + col);
  const int slot = slots[min(tj, T - 1)];
  int s[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) s[i] = slots[min(tg + i, T - 1)];
  if (r < TV) *reinterpret_cast<bf16x8*>(&vs[r][col]) = x;
  __syncthreads();
  if (r >= TV) return;
  bool whole = tg + 7 < T && s[0] >= 0 && s[0] % 8 == 0;  // side by side in one half of a page
#pragma unroll
  for (int i = 1; i < 8; ++i) whole &= s[i] == s[0] + i;
  if (whole) {  // a channel a thread
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = vs[r8 + i][j];
    store8(v_cache + (((size_t)(s[0] / kKvBlock) * Hkv + g) * D + j) * kKvBlock + s[0] % kKvBlock, o);
  } else if (tj < T && slot >= 0) {  // eight channels of a token, its neighbours' beside them
    bf16* dst = v_cache + ((size_t)(slot / kKvBlock) * Hkv + g) * D * kKvBlock + slot % kKvBlock;
#pragma unroll
    for (int i = 0; i < 8; ++i) dst[(j / 8 + i * LV) * kKvBlock] = vs[r8 + (j & 7)][j / 8 + i * LV];
  }
}

// Encoder self-attention (no RoPE, K / V straight from the packed QKV rows): one workgroup per (transient page, kv
// head) writes the page's K image [16][D] and V^T image [D][16] whole, with 16-B stores; V is transposed through LDS.
// Replaces rope_kv_kernel's per-(token, head) scatter for encoders, whose V^T half is 2-B stores 32 B apart and which
// also copied q (the attention reads q from the QKV rows, q_ld): e5-large ingest at 65536 tokens spent 379 us per
// layer there (profiles/r6).
template <int D>
__global__ __launch_bounds__(64) void kv_pack_kernel(const bf16* __restrict__ qkv, int ld, int koff, int voff,
                                                     const int* __restrict__ blk_tok, const int* __restrict__ blk_n,
                                                     bf16* __restrict__ k_cache, bf16* __restrict__ v_cache, int Hkv) {
  constexpr int CPR = D / 8;       // 16-B chunks per row
  constexpr int PIECES = 16 * CPR;
  __shared__ __attribute__((aligned(16))) bf16 vs[16][D + 8];  // V rows, padded against bank conflicts
  const int b = blockIdx.x, g = blockIdx.y, lane = threadIdx.x;
  const int t0 = blk_tok[b], n = blk_n[b];
  bf16* kp = k_cache + ((size_t)b * Hkv + g) * 16 * D;
  bf16* vp = v_cache + ((size_t)b * Hkv + g) * D * 16;
#pragma unroll
  for (int p = lane; p < PIECES; p += 64) {
    const int r = p / CPR, c = (p % CPR) * 8;
    bf16x8 kv = {}, vv = {};
    if (r < n) {
      const bf16* src = qkv + (size_t)(t0 + r) * ld + (size_t)g * D + c;
      kv = load8(src + koff);
      vv = load8(src + voff);
    }
    store8(kp + r * D + c, kv);
    *reinterpret_cast<bf16x8*>(&vs[r][c]) = vv;
  }
  __syncthreads();
#pragma unroll
  for (int p = lane; p < PIECES; p += 64) {  // V^T row d = 16 tokens = two 16-B pieces
    const int d = p >> 1, h8 = (p & 1) * 8;
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = vs[h8 + e][d];
    store8(vp + d * 16 + h8, o);
  }
}

}  // namespace

void gai_kv_pack(const void* qkv, int ld, int koff, int voff, const int* blk_tok, const int* blk_n, int nblk,
                 void* k_cache, void* v_cache, int Hkv, int D, hipStream_t st) {
  if (nblk == 0) return;
  const dim3 grid(nblk, Hkv);
#define GAI_KVP(DD)                                                                                          \
  if (D == DD) {                                                                                             \
    kv_pack_kernel<DD><<<grid, 64, 0, st>>>((const bf16*)qkv, ld, koff, voff, blk_tok, blk_n, (bf16*)k_cache, \
                                            (bf16*)v_cache, Hkv);                                            \
    GAI_LAUNCH_CHECK();                                                                                      \
    return;                                                                                                  \
  }
  GAI_KVP(64)
  GAI_KVP(96)
  GAI_KVP(128)
  GAI_KVP(256)
#undef GAI_KVP
  gai_launch_error(__FILE__, __LINE__, "kv_pack: head_dim must be 64, 96, 128 or 256");
}

// Steps that take rope_kv_rows_kernel. Decode-sized and small ones are a launch and one chain of loads, and rope_kv_kernel has four times the
// workgroups for that; what it pays for is values (two bytes a store), about four times a query's elements. Us, that kernel | this one, tokens
// in order / each in a page of its own: 65 x (32 + 8 + 8) x 128 3.25 | 3.01 / 3.31 | 3.51, 100 of those 3.47 | 3.02 / 3.64 | 3.71; 65 x (16 + 16 + 16) x 128
// 3.81 | 2.95 / 4.11 | 3.75; (16 + 4 + 4) x 128, 100 2.90 | 2.97 / 2.94 | 3.26, 187 3.41 | 3.05 / 3.55 | 3.54; (8 + 1 + 1) x 256, 187 3.01 | 3.08 / 2.93 | 3.32,
// 400 3.35 | 3.26 / 3.54 | 3.78; (14 + 2 + 2) x 64, 400 3.01 | 3.02 / 3.04 | 3.27, 1000 3.73 | 3.17.
static bool rope_rows(int T, int Hq, int Hkv, int D) { return T > 64 && (long)T * (Hq + 4 * Hkv) * D >= 9 << 16; }

int gai_rope_kv_norm_ok(int D) { return D == 64 || D == 128 || D == 256; }

// wq / wk: weights of the norms of q and k heads (both or none; bf16 pages, gai_rope_kv_norm_ok)
void gai_rope_kv_rows(const void* qkv, const int* pos, const float* cos_sin, const int* slots, void* q_out, void* k_cache, void* v_cache,
                      int T, int Hq, int Hkv, int D, int rope, const void* wq, const void* wk, float eps, hipStream_t st) {
  if (T == 0) return;
  if ((wq == nullptr) != (wk == nullptr) || (wq && !gai_rope_kv_norm_ok(D)))
    gai_launch_error(__FILE__, __LINE__, "rope_kv: head norms need both weights and head_dim 64, 128 or 256");
#define GAI_ROWS(DD, N)                                                                                                              \
  rope_kv_rows_kernel<DD, N><<<dim3((T + rows_tokens<DD>() - 1) / rows_tokens<DD>(), (Hq + Hkv + kHeadsAWg - 1) / kHeadsAWg + 2 * Hkv), \
                               256, 0, st>>>((const bf16*)qkv, pos, cos_sin, slots, (bf16*)q_out, (bf16*)k_cache, (bf16*)v_cache, T, \
                                             Hq, Hkv, rope, (const bf16*)wq, (const bf16*)wk, eps)
  if (D == 64) { if (wq) GAI_ROWS(64, true); else GAI_ROWS(64, false); }
  else if (D == 96) GAI_ROWS(96, false);
  else if (D == 128) { if (wq) GAI_ROWS(128, true); else GAI_ROWS(128, false); }
  else if (D == 256) { if (wq) GAI_ROWS(256, true); else GAI_ROWS(256, false); }
  else gai_launch_error(__FILE__, __LINE__, "rope_kv: head_dim must be 64, 96, 128 or 256");
#undef GAI_ROWS
  GAI_LAUNCH_CHECK();
}

void gai_rope_kv_write(const void* qkv, const int* pos, const float* cos_sin, const int* slots, void* q_out,
                       void* k_cache, void* v_cache, int T, int Hq, int Hkv, int D, int rope, int kv_fp8,
                       float k_scale, float v_scale, hipStream_t st) {
  if (T == 0) return;
  const bool on16 = (((size_t)qkv | (size_t)q_out | (size_t)k_cache | (size_t)v_cache) & 15) == 0;
  if (rope_rows(T, Hq, Hkv, D) && !kv_fp8 && on16 && D % 32 == 0 && D <= 256)
    return gai_rope_kv_rows(qkv, pos, cos_sin, slots, q_out, k_cache, v_cache, T, Hq, Hkv, D, rope, nullptr, nullptr, 0.f, st);
  const long items = (long)T * (Hq + 2 * Hkv);
  const float iks = 1.f / k_scale, ivs = 1.f / v_scale;
#define GAI_ROPE_CASE(DD)                                                                                   \
  if (D == DD) {                                                                                            \
    constexpr int HPB = 256 / (DD / 8);                                                                     \
    const unsigned grid = (unsigned)((items + HPB - 1) / HPB);                                              \
    if (kv_fp8)                                                                                             \
      rope_kv_kernel<DD, fp8><<<grid, 256, 0, st>>>((const bf16*)qkv, pos, cos_sin, slots, (bf16*)q_out,   \
                                                     (fp8*)k_cache, (fp8*)v_cache, T, Hq, Hkv, rope, iks, ivs); \
    else                                                                                                    \
      rope_kv_kernel<DD, bf16><<<grid, 256, 0, st>>>((const bf16*)qkv, pos, cos_sin, slots, (bf16*)q_out,  \
                                                      (bf16*)k_cache, (bf16*)v_cache, T, Hq, Hkv, rope, iks, ivs); \
    GAI_LAUNCH_CHECK();                                                                                     \
    return;                                                                                                 \
  }
  GAI_ROPE_CASE(64)
  GAI_ROPE_CASE(96)
  GAI_ROPE_CASE(128)
  GAI_ROPE_CASE(256)
#undef GAI_ROPE_CASE
  gai_launch_error(__FILE__, __LINE__, "rope_kv: head_dim must be 64, 96, 128 or 256");
}
