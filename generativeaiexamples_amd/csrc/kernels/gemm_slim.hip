// Decode-sized GEMM in one launch: C[M, N] = A[M, K] . W[N, K]^T (+ epilogue), M <= 64, K <= 4096, K % 512 == 0.
//
// Bound by latency, not by bytes: an encoder's 1024-wide projection of a short question is 2-8 MB of weights, 0.4-1.6 us
// at the card's read rate, and the split-K kernel plus its reduce launch took 10-12 us for it (fp32 partials written,
// a launch, read again). Here a workgroup owns 16 NF columns for ALL of K and every load of it is in flight at once:
//  * its 8 waves split K; a wave's weight fragments (<= 16 k32 steps, 64 NF registers) are all loaded before anything
//    is waited for;
//  * the activations go through LDS in two 64 KiB stages (LDS-DMA, 16-B chunks XOR-swizzled: conflict-free b128 reads),
//    since fragments read straight from global memory (16 rows x 64 B a load) cost about 2 us per 64 KiB of them;
//  * the waves' sums meet in LDS, in wave order, and the epilogue runs there: no fp32 partials, no second launch. (A product
//    whose rows a layer norm takes next is the exception: K in slices, fp32 sums of which the norm's launch adds up,
//    gai_gemm_slim_layernorm.)
// MI355X, weights cold, row-major | fragment order, us, against split-K + reduce (two launches; the gap of about 1 us
// between them not counted):
//   M 32, N 3072, K 1024   5.3 | 4.9   was  10.4 |  8.3        M 32, N 2048, K 2048   7.4 | 6.6   was 10.5 |  8.4
//   M 32, N 1024, K 1024   4.9 | 4.7   was   9.9 |  7.9        M 64, N 2048, K 2048   9.1 | 8.1   was 12.4 | 10.0
//   M 32, N 4096, K 1024   5.8 | 5.3   was  10.9 |  8.6        M 32, N 1024, K 4096  10.1 | 8.7   was 10.5 |  8.5
//   M 64, N 4096, K 1024   6.8 | 6.4   was  13.0 | 10.2        M 32, N 4096, K 4096  12.2 | 11.0  was 13.9 | 13.4
#include <type_traits>

#include "gai_common.h"
#include "gai_epilogue.h"
#include "gai_gemm_slim.h"
#include "gai_kernels.h"
#include "gai_rotary.h"

using namespace gai;

namespace {

constexpr int kWaves = 8;
constexpr int kMaxSlabs = 8;
constexpr int kStageBytes = 64 * 1024;     // activation columns of one stage, all rows
constexpr int kPairK = kWaves * 64;        // k columns of one pair step of the workgroup: 2 x 32 per wave
// the largest K of a slice: every weight fragment of a wave's share is in registers at once; beyond 2560 only the forms that the rules
// below take
constexpr int max_k(int mt, int nf) { return mt == 4 || nf == 2 ? 2560 : 4096; }

// a product's slices in 512s of K: `each`, the first `longer` of them one more. (Divided on the host: in the kernel it cost every launch of an
// embedded question 0.06 us.)
struct Slices {
  int each, longer;
  Slices(int K, int slices) : each(K / kPairK / slices), longer(K / kPairK % slices) {}
  __device__ __forceinline__ int begin(int y) const { return each * y + min(y, longer); }
  __device__ __forceinline__ int size(int y) const { return each + (y < longer); }
};
int slice_k(int K, int slices) { return (K + slices * kPairK - 1) / (slices * kPairK) * kPairK; }  // the longest

template <int EPI, bool OUTF32>
__device__ __forceinline__ void slim_store4(void* C, const bf16* bias, const bf16* R, int ldc, int m, int n, int M,
                                            const f32x4& v) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (m + r < M) store_out<EPI, OUTF32>(C, bias, R, ldc, m + r, n, v[r]);
}

template <int EPI>
__device__ __forceinline__ void slim_store(void* C, const bf16* bias, const bf16* R, int ldc, int m, int n, int M,
                                           const f32x4& v, int out_f32) {
  if (out_f32) slim_store4<EPI, true>(C, bias, R, ldc, m, n, M, v);
  else slim_store4<EPI, false>(C, bias, R, ldc, m, n, M, v);
}

// K: all of it; slice y of it into slab y of C
template <int MT, int NF, int STAGE, int MAXK>
__device__ __forceinline__ void slim_body(const bf16* __restrict__ A, const bf16* __restrict__ W, void* C, const bf16* bias,
                                          const bf16* R, int M, int N, int K, int y, Slices slices, int ldc, int epi, int out_f32, int psw,
                                          int bx, char* smem) {
  constexpr int ROWS = 16 * MT;
  constexpr int KC = STAGE / (ROWS * 2);       // columns of a stage
  constexpr int CPR = KC / 8;                        // 16-B chunks of a staged row
  constexpr int P = KC / kPairK;                     // pair steps of a stage
  constexpr int kMaxPairs = MAXK / kPairK;
  constexpr int NST = (kMaxPairs + P - 1) / P;       // stages of the largest K
  constexpr int DMA = STAGE / (64 * kWaves * 16);  // LDS-DMA instructions of a wave and stage
  const int tid = threadIdx.x, lane = tid & 63;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n0 = bx * 16 * NF;
  const int ld = K, k0 = slices.begin(y) * kPairK, np = slices.size(y), nst = (np + P - 1) / P;
  K = np * kPairK;
  A += k0;
  if (y) C = (float*)C + (size_t)y * M * N;
  const int r16 = lane & 15, q = lane >> 4;

  // ---- every weight fragment of this wave: pair p covers k = p * 512 + 64 wid + {0, 32}
  bf16x8 w[kMaxPairs][2][NF];
  const bf16* wp[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int n = min(n0 + 16 * f, N - 16);  // a fragment past N repeats the last one (not stored)
    wp[f] = psw ? W + ((size_t)(n / 16) * (ld / 32) + k0 / 32 + 2 * wid) * 512 + 8 * lane
                : W + (size_t)(n + r16) * ld + k0 + 64 * wid + 8 * q;
  }
#pragma unroll
  for (int p = 0; p < kMaxPairs; ++p) {
    if (p < np) {
      if (psw) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int u = 0; u < 2; ++u)
            w[p][u][f] = __builtin_nontemporal_load(
                reinterpret_cast<const bf16x8*>(wp[f] + (size_t)p * (kPairK / 32) * 512 + u * 512));
      } else {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
          for (int u = 0; u < 2; ++u) w[p][u][f] = load8(wp[f] + p * kPairK + u * 32);
      }
    }
  }

  // ---- activation stage t into slot t & 1: chunk i -> row i / CPR, physical chunk i % CPR = logical ^ (row & 15)
  auto stage = [&](int t) {
    char* dst = smem + (t & 1) * STAGE;
#pragma unroll
    for (int d = 0; d < DMA; ++d) {
      const int base = (d * kWaves + wid) * 64;
      const int i = base + lane, row = i / CPR, c = (i % CPR) ^ (row & 15);
      const bf16* src = A + (size_t)min(row, M - 1) * ld + min(t * KC + c * 8, K - 8);
      __builtin_amdgcn_global_load_lds(src, GAI_LDS(dst + (size_t)base * 16), 16, 0, 0);
    }
  };

  f32x4 acc[MT][NF];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[i][f] = f32x4{0.f, 0.f, 0.f, 0.f};

  stage(0);
  if (nst > 1) stage(1);
#pragma unroll
  for (int t = 0; t < NST; ++t) {
    if (t < nst) {
      // stage t has landed once only the DMAs of stage t + 1 are outstanding (they were issued last)
      if (t + 1 < nst) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(DMA) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      const char* src = smem + (t & 1) * STAGE;
#pragma unroll
      for (int j = 0; j < P; ++j) {
        if (t * P + j < kMaxPairs && t * P + j < np) {
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const int c = (j * kPairK + 64 * wid + 32 * u) / 8 + q;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              const bf16x8 a = *reinterpret_cast<const bf16x8*>(src + (size_t)((16 * i + r16) * CPR + (c ^ r16)) * 16);
#pragma unroll
              for (int f = 0; f < NF; ++f)
                acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[t * P + j][u][f], acc[i][f], 0, 0, 0);
            }
          }
        }
      }
      __syncthreads();  // the slot is free (and, after the last stage, the partial tiles may overwrite it)
      if (t + 2 < nst) stage(t + 2);
    }
  }

  // ---- the waves' K shares are summed through LDS in wave order: [wave][i][f][lane] quads of 4 rows
  f32x4* part = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int f = 0; f < NF; ++f) part[((wid * MT + i) * NF + f) * 64 + lane] = acc[i][f];
  __syncthreads();
  const bool glu = epi == EPI_SWIGLU || epi == EPI_GEGLU;
  for (int e = tid; e < MT * NF * 64; e += 64 * kWaves) {
    const int l = e & 63, f = (e >> 6) % NF, i = (e >> 6) / NF;
    if (glu && (f & 1)) continue;
    auto total = [&](int ff) {
      f32x4 v = part[(i * NF + ff) * 64 + l];
#pragma unroll
      for (int k = 1; k < kWaves; ++k) {
        const f32x4 o = part[((k * MT + i) * NF + ff) * 64 + l];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] += o[r];
      }
      return v;
    };
    const int m = 16 * i + 4 * (l >> 4), n = n0 + 16 * f + (l & 15);
    if (n >= N) continue;
    f32x4 v = total(f);
    if (glu) {
      const f32x4 up = total(f + 1);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        v[r] = epi == EPI_SWIGLU ? glu_act<EPI_SWIGLU>(v[r], up[r]) : glu_act<EPI_GEGLU>(v[r], up[r]);
      slim_store<EPI_NONE>(C, nullptr, nullptr, ldc, m, n0 / 2 + 16 * (f / 2) + (l & 15), M, v, out_f32);
      continue;
    }
    switch (epi) {
      case EPI_NONE: slim_store<EPI_NONE>(C, bias, R, ldc, m, n, M, v, out_f32); break;
      case EPI_BIAS: slim_store<EPI_BIAS>(C, bias, R, ldc, m, n, M, v, out_f32); break;
      case EPI_BIAS_GELU: slim_store<EPI_BIAS_GELU>(C, bias, R, ldc, m, n, M, v, out_f32); break;
      case EPI_RESIDUAL: slim_store<EPI_RESIDUAL>(C, bias, R, ldc, m, n, M, v, out_f32); break;
      case EPI_BIAS_RESIDUAL: slim_store<EPI_BIAS_RESIDUAL>(C, bias, R, ldc, m, n, M, v, out_f32); break;
      case EPI_BIAS_RELU: slim_store<EPI_BIAS_RELU>(C, bias, R, ldc, m, n, M, v, out_f32); break;
      case EPI_BIAS_QUICKGELU: slim_store<EPI_BIAS_QUICKGELU>(C, bias, R, ldc, m, n, M, v, out_f32); break;
    }
  }
}

// smem: 2 stages; reused for the waves' partial tiles
template <int MT, int NF>
__global__ __launch_bounds__(64 * kWaves, 1) void gemm_slim_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W, void* C,
                                                                   const bf16* bias, const bf16* R, int M, int N, int K,
                                                                   Slices slices, int ldc, int epi, int out_f32, int psw) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  slim_body<MT, NF, kStageBytes, max_k(MT, NF)>(A, W, C, bias, R, M, N, K, blockIdx.y, slices, ldc, epi, out_f32, psw, blockIdx.x, smem);
}

// The K slices of a product beside the rotation of a step's heads and its cache write (workgroups below `rot`). Two workgroups share a
// CU, stages of half the size: with one, the last slices waited for the rotations to end (24 rows, 2048 x 5632: 10.9 -> 9.9 us, 11.3 in
// eleven slices of the streaming kernel; a step of the 2k hybrid stack, 24 streams 363 -> 354 us, one 274 -> 264)
constexpr int kBesideStage = kStageBytes / 2, kBesideK = 3072;
template <int MT>
__global__ __launch_bounds__(64 * kWaves, 4) void gemm_slim_rotary_kernel(const bf16* __restrict__ A, const bf16* __restrict__ W,
                                                                          float* __restrict__ part, int M, int N, int K, Slices slices,
                                                                          RotaryHalf<bf16> r, int rot) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int i = (int)blockIdx.x - rot, tiles = N / 16;
  if (i < 0) {
    if (threadIdx.x < 256) rotary_half_body<bf16, 8, 1, 1>(r, blockIdx.x, reinterpret_cast<float*>(smem));
    return;  // (a barrier counts the waves that are left)
  }
  slim_body<MT, 1, kBesideStage, kBesideK>(A, W, part, nullptr, nullptr, M, N, K, i / tiles, slices, N, EPI_NONE, 1, 1, i % tiles, smem);
}

template <int MT, int NF>
void launch_slim(const void* A, const void* W, void* C, const void* bias, const void* R, int M, int N, int K, int ldc,
                 int epi, int out_f32, int psw, hipStream_t st, int ks = 1) {
  static bool once = false;
  if (!once) {
    hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_slim_kernel<MT, NF>),
                        hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    once = true;
  }
  constexpr int stage_k = kStageBytes / (32 * MT);
  const size_t lds = (size_t)(slice_k(K, ks) > stage_k ? 2 : 1) * kStageBytes;  // >= the partial tiles (8 MT NF KiB <= 64 KiB)
  gemm_slim_kernel<MT, NF><<<dim3((N + 16 * NF - 1) / (16 * NF), ks), 64 * kWaves, lds, st>>>(
      (const bf16*)A, (const bf16*)W, C, (const bf16*)bias, (const bf16*)R, M, N, K, Slices(K, ks), ldc, epi, out_f32, psw);
  GAI_LAUNCH_CHECK();
}

// out = LayerNorm(bf16(bf16(sum of the slabs + bias) + R)), the roundings of the product's residual epilogue; a wave a row,
// every load of it in flight at once.
template <int NCH, int KS>  // KS >= ks: slabs loaded, those past ks the last one again, not counted
__global__ __launch_bounds__(64) void slabs_layernorm_kernel(const float* __restrict__ ws, int ks, int M, int N,
                                                             const bf16* __restrict__ bias, const bf16* __restrict__ R,
                                                             const bf16* __restrict__ g, const bf16* __restrict__ b,
                                                             bf16* __restrict__ out, float eps) {
  const int lane = threadIdx.x, row = blockIdx.x;
  const size_t base = (size_t)row * N, slab = (size_t)M * N;
  bf16x8 rv[NCH], bv[NCH], gv[NCH], lb[NCH];
  float v[NCH][8];
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int i = min((c * 64 + lane) * 8, N - 8);  // past the row: the last columns again, not counted
#pragma unroll
    for (int e = 0; e < 8; ++e) v[c][e] = 0.f;
    rv[c] = load8(R + base + i);
    gv[c] = load8(g + i);
    bv[c] = bias ? load8(bias + i) : bf16x8{};
    lb[c] = b ? load8(b + i) : bf16x8{};
  }
#pragma unroll
  for (int k = 0; k < KS; ++k)
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const float* p = ws + min(k, ks - 1) * slab + base + min((c * 64 + lane) * 8, N - 8);
      const f32x4 lo = *reinterpret_cast<const f32x4*>(p), hi = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[c][e] += k < ks ? lo[e] : 0.f;
        v[c][4 + e] += k < ks ? hi[e] : 0.f;
      }
    }
  float s = 0.f, q = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float y = bias ? v[c][e] + (float)bv[c][e] : v[c][e];
      v[c][e] = (float)(bf16)((float)(bf16)y + (float)rv[c][e]);
      s += (c * 64 + lane) * 8 < N ? v[c][e] : 0.f;
    }
  const float mean = wave_sum(s) / N;
#pragma unroll
  for (int c = 0; c < NCH; ++c)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = v[c][e] - mean;
      q += (c * 64 + lane) * 8 < N ? d * d : 0.f;
    }
  const float inv = rsqrtf(wave_sum(q) / N + eps);
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int i = (c * 64 + lane) * 8;
    if (i < N) {
      bf16x8 o;
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (bf16)((v[c][e] - mean) * inv * (float)gv[c][e] + (b ? (float)lb[c][e] : 0.f));
      store8(out + base + i, o);
    }
  }
}

}  // namespace

// Against split-K + reduce (figures above): weights up to 16 MiB, where the reduce launch is a third of the time; above
// that the stream decides and the two are within 15 % of each other (N 4096, K 4096, M 64: 16.7 | 14.3 us against
// 17.0 | 17.2; N 6144: 22.6 | 19.3 against 21.1 | 20.7), and the split partials are what the fused decode tails sum. Two
// fragments a workgroup for the paired epilogues, and where one would need a second round of workgroups (one per CU once
// both stages are in use). At K > 2560 the serial walk over K (4 to 8 stages) costs a workgroup more than the reduce
// does unless there are few rows and one fragment (N 1024, K 4096: M 32 10.1 | 8.7 us, two fragments 14.1 | 11.8,
// M 64 13.3 | 12.0, against 10.5 | 8.5 and 13.2 | 10.1 split).
int gai_gemm_slim_nf(int M, int N, int K, bool glu) {
  if (M < 1 || M > 64 || K < kPairK || K % kPairK || K > 4096 || N < 16 || N % (glu ? 32 : 16) ||
      (long long)N * K > (8 << 20))
    return 0;
  const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int nf = glu || (N / 16 > 256 && K > kStageBytes / (32 * mt)) ? 2 : 1;
  return K <= max_k(mt, nf) ? nf : 0;
}

void gai_gemm_slim(const void* A, const void* W, void* C, const void* bias, const void* R, int M, int N, int K, int ldc,
                   int epi, int out_f32, int nf, int psw, hipStream_t st) {
  const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  if (M < 1 || M > 64 || K < kPairK || K % kPairK || K > max_k(mt, nf) || N < 16 || N % 16 || (nf != 1 && nf != 2) ||
      (epi_glu(epi) && (nf != 2 || N % 32)) || epi < 0 || (epi > EPI_BIAS_QUICKGELU && epi != EPI_GEGLU))
    gai_launch_error(__FILE__, __LINE__, "gemm_slim: needs 1 <= M <= 64, K % 512 == 0, K <= 4096 or 2560, N % 16 == 0");
#define GAI_SLIM(MTV, NFV) \
  if (mt == MTV && nf == NFV) return launch_slim<MTV, NFV>(A, W, C, bias, R, M, N, K, ldc, epi, out_f32, psw, st);
  GAI_SLIM(1, 1)
  GAI_SLIM(1, 2)
  GAI_SLIM(2, 1)
  GAI_SLIM(2, 2)
  GAI_SLIM(4, 1)
  GAI_SLIM(4, 2)
#undef GAI_SLIM
}

// Slices of K for a product whose rows a layer norm takes next (which sums the slabs): the most, up to 8, whose workgroups
// fit the chip at once. One workgroup a 16 columns leaves most of it idle: N 1024, K 4096 has 64, each with 350 KB to fetch
// (27 rows: 10.0 us and 3.9 of norm; in four slices 5.5 and 3.6; K 1024 4.1 + 3.9 and in two slices 4.0 + 3.6).
int gai_gemm_slim_ks(int M, int N, int K) {
  if (M < 1 || M > 64 || N < 16 || N % 16 || N > 2048 || K < 2 * kPairK || K % kPairK || (long long)N * K > (8 << 20)) return 0;
  const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  for (int ks = kMaxSlabs; ks > 1; --ks)
    if (K / kPairK % ks == 0 && N / 16 * ks <= 256 && K / ks <= max_k(mt, 1)) return ks;
  return 0;
}

// Slices of a deeper product of up to 32 rows for a norm that adds them: the fewest that fit a workgroup's registers (two share a CU where
// a rotation is beside them), where all fit the chip at once; the first ones are longer by 512 where K does not divide. Which products
// take them: gemm_splitk.hip
int gai_gemm_slim_few_ks(int M, int N, int K) {
  if (M < 1 || M > 32 || N < 16 || N % 16 || N > 2048 || K < kPairK || K % kPairK || gai_gemm_slim_nf(M, N, K, false)) return 0;
  for (int ks = 2; ks <= kMaxSlabs && N / 16 * ks <= 256; ++ks)
    if (slice_k(K, ks) <= kBesideK) return ks;
  return 0;
}

// those slices, [ks][M][N]
void gai_gemm_slim_partials(const void* A, const void* W, int M, int N, int K, int ks, float* ws, int psw, hipStream_t st) {
  if (ks == 0) gai_launch_error(__FILE__, __LINE__, "gemm_slim_partials: the shape has no slices");
  if (M <= 16) launch_slim<1, 1>(A, W, ws, nullptr, nullptr, M, N, K, N, EPI_NONE, 1, psw, st, ks);
  else if (M <= 32) launch_slim<2, 1>(A, W, ws, nullptr, nullptr, M, N, K, N, EPI_NONE, 1, psw, st, ks);
  else launch_slim<4, 1>(A, W, ws, nullptr, nullptr, M, N, K, N, EPI_NONE, 1, psw, st, ks);
}

// gai_gemm_slim_few_ks of a weight in fragment order beside the rotation r (T rows, a head's channels by 8s)
void gai_gemm_slim_partials_rotary(const void* A, const void* W, int M, int N, int K, float* ws, const RotaryHalf<bf16>& r,
                                   hipStream_t st) {
  const int ks = gai_gemm_slim_few_ks(M, N, K), rot = 2 * r.T;
  if (ks == 0) gai_launch_error(__FILE__, __LINE__, "gemm_slim_partials_rotary: the shape has no slices");
#define GAI_SR(MT)                                                                                                                       \
  {                                                                                                                                      \
    static bool once = false;                                                                                                            \
    if (!once) {                                                                                                                         \
      hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_slim_rotary_kernel<MT>), hipFuncAttributeMaxDynamicSharedMemorySize,        \
                          2 * kBesideStage);                                                                                             \
      once = true;                                                                                                                       \
    }                                                                                                                                    \
    gemm_slim_rotary_kernel<MT><<<rot + N / 16 * ks, 64 * kWaves, 2 * kBesideStage, st>>>((const bf16*)A, (const bf16*)W, ws, M, N, K,     \
                                                                                         Slices(K, ks), r, rot);                         \
  }
  if (M <= 16) GAI_SR(1) else GAI_SR(2)
#undef GAI_SR
  GAI_LAUNCH_CHECK();
}

bool gai_slabs_layernorm_ok(int ks, int N) { return ks >= 1 && ks <= kMaxSlabs && N <= 2048 && N % 8 == 0; }

// the 16-byte pairs of a slab's row that a lane of it asks for: chunks of 512 columns, times the slabs that its kernel is built for
int gai_slabs_layernorm_reads(int ks, int N) { return (N <= 512 ? 1 : N <= 1024 ? 2 : 4) * (ks <= 2 ? 2 : ks <= 4 ? 4 : kMaxSlabs); }

void gai_slabs_layernorm(const float* ws, int ks, const void* bias, const void* R, const void* g, const void* b, void* out, int M, int N,
                         float eps, hipStream_t st) {
  if (!gai_slabs_layernorm_ok(ks, N)) gai_launch_error(__FILE__, __LINE__, "slabs_layernorm: shape");
#define GAI_SLN(NCH, KS)                                                                                                 \
  slabs_layernorm_kernel<NCH, KS><<<M, 64, 0, st>>>(ws, ks, M, N, (const bf16*)bias, (const bf16*)R, (const bf16*)g,     \
                                                    (const bf16*)b, (bf16*)out, eps)
#define GAI_SLN_K(NCH)                   \
  if (ks <= 2) GAI_SLN(NCH, 2);          \
  else if (ks <= 4) GAI_SLN(NCH, 4);     \
  else GAI_SLN(NCH, kMaxSlabs)
  if (N <= 512) { GAI_SLN_K(1); }
  else if (N <= 1024) { GAI_SLN_K(2); }
  else { GAI_SLN_K(4); }
#undef GAI_SLN_K
#undef GAI_SLN
  GAI_LAUNCH_CHECK();
}

void gai_gemm_slim_layernorm(const void* A, const void* W, const void* bias, const void* R, const void* g, const void* b,
                             void* out, int M, int N, int K, float eps, float* ws, int psw, hipStream_t st) {
  const int ks = gai_gemm_slim_ks(M, N, K);
  gai_gemm_slim_partials(A, W, M, N, K, ks, ws, psw, st);
  gai_slabs_layernorm(ws, ks, bias, R, g, b, out, M, N, eps, st);
}
