// bf16 GEMM for a few hundred rows (64 < M <= 2048: short prompts, prompt portions, batches of questions):
// C[M, N] = A[M, K] . B[N, K]^T with the fused epilogues of gemm_impl.h, B row-major or in fragment order.
//
// At these sizes the weights are read once and bound the product (Llama-3-8B down projection, M = 187: 117 MB, 20 us at
// 5.8 TB/s); what keeps a tiled kernel from that rate is latency (a load from HBM takes over 2 us) and the few tiles there
// are. So:
//  * a workgroup takes 16 * MT rows x 64 * NG columns: 128 x 64 (two workgroups share a CU), 128 x 128 or, so that up to
//    192 rows still fetch the weights once, 192 x 128;
//  * weights in fragment order go straight to registers in operand layout (wave = 16 * NG columns x half of a 64-deep K step:
//    nothing is fetched twice); the rows of A, which sit in L2, go to an LDS ring by DMA and are read by all waves. Loads return
//    in order, so A is asked for as far ahead as the weights are (DB steps): with A a step or two ahead, waiting for it
//    waited for weights that were asked for just before (187 rows, 28672 x 4096 SwiGLU 64.3 -> 56.0 us, 4096 x 14336 50.6 ->
//    44.0, 6144 x 4096 30.7 -> 23.7, 4096 x 4096 23.3 -> 20.5; 1024 rows 4096 x 4096 41.4 -> 37.5). What is left: a CU holds
//    about 32 KB of misses (a weight stream of 32 KB in flight per CU is as fast as one of 192 KB: 6.3 TB/s on the chip, 60 KB/us
//    in one CU), and A's 24 KB a step share them, 0.75 us a step without any products. Four waves of 64 columns each (half the
//    LDS reads) gave nothing: 57.5 us for the first of the products above; nor did 192 x 64 tiles, which pad 187 rows less but fetch A twice
//    as often: 4096 x 14336 47.8 | 48.6;
//  * row-major weights go through LDS beside A, by the same DMA in whole lines: in operand layout a load touches 16 lines for 64 bytes
//    of each. Row-major, one way -> the other, us: 187 rows 4096 x 14336 61 -> 47, 28672 x 4096 (SwiGLU) 75 -> 65, 448 rows 97 ->
//    70 and 6144 x 4096 52 -> 36, 512 rows 1024 x 1024 10.5 -> 8.6; the last rows of 18337 x 1024 x 1024 (ORD) 47.5 -> 43.7 in
//    all. Sums are the layout's own in neither: equal bits;
//  * K is cut into S parts, so tile x part items fill the CUs;
//  * measured on one card, weights from HBM, fragment order (row-major: half of 240 products within 7 % of it, nineteen in twenty
//    within 21 %), N x K, against the kernels it replaced: 187 rows 4096 x 14336 200 -> 44 us, 4096 x 4096 67 -> 20, 6144 x 4096
//    58 -> 24, 28672 x 4096 (SwiGLU) 76 -> 56; 512 rows 4096 x 14336 82 -> 74;
//  * MFMA operands swapped (rows = weights), so a lane ends with four consecutive columns of a row: 8-byte stores;
//  * S > 1: every wave stores its fp32 share (write-through) and draws the (tile, wave) ticket; the one that draws the last
//    sums the parts in part order - the same result whichever it is - and runs the epilogue. Nobody waits, and a wave that
//    sees all others done keeps its share in registers;
//  * ORD, for the last rows of a large product (gai_gemm_mid_tail): a wave takes all of K for half the columns, one sum in
//    the order of the 256 x 256 kernels, so equal rows give equal bits wherever they stand. 64 x 128 or 128 x 128 tiles:
//    no weight is fetched twice in a workgroup, A is read from LDS twice as often as with k halves.
#include "gai_common.h"
#include "gai_epilogue.h"
#include "gai_gemm_mid.h"
#include "gai_kernels.h"

#include <algorithm>

using namespace gai;

namespace {

constexpr int kBK = 128;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

constexpr bool epi_bias(int e) {
  return e == EPI_BIAS || e == EPI_BIAS_GELU || e == EPI_BIAS_RESIDUAL || e == EPI_BIAS_RELU || e == EPI_BIAS_QUICKGELU;
}
constexpr bool epi_res(int e) { return e == EPI_RESIDUAL || e == EPI_BIAS_RESIDUAL; }

template <int EPI, bool OUTF32>
__device__ __forceinline__ void store4(void* C, bf16x4 b, bf16x4 x, int ldc, int m, int n, f32x4 v) {
  const size_t o = (size_t)m * ldc + n;
  if constexpr (epi_bias(EPI)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] += (float)b[r];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if constexpr (EPI == EPI_BIAS_GELU) v[r] = gelu_erf(v[r]);
    if constexpr (EPI == EPI_BIAS_RELU) v[r] = fmaxf(v[r], 0.f);
    if constexpr (EPI == EPI_BIAS_QUICKGELU) v[r] = quick_gelu(v[r]);
  }
  if constexpr (epi_res(EPI)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = (OUTF32 ? v[r] : (float)(bf16)v[r]) + (float)x[r];
  }
  if constexpr (OUTF32) {
    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(C) + o) = v;
  } else {
    bf16x4 y;
#pragma unroll
    for (int r = 0; r < 4; ++r) y[r] = (bf16)v[r];
    *reinterpret_cast<bf16x4*>(reinterpret_cast<bf16*>(C) + o) = y;
  }
}

// K steps in LDS: A's, and row-major weights with them (two workgroups of 128 x 64 tiles share a CU)
template <int MT, int NG, bool FRAG>
constexpr int mid_ring() { return FRAG ? (MT == 12 ? 6 : 4) : MT == 12 ? 4 : NG == 1 ? 3 : 5; }
template <int MT, int NG, bool FRAG>
constexpr int mid_step() { return MT * 2048 + (FRAG ? 0 : NG * 8192); }  // bytes of one

template <int MT, int NG, int EPI, bool OUTF32, bool ORD, bool FRAG>
__global__ __launch_bounds__(512, 1) void gemm_mid_kernel(const bf16* __restrict__ A, const bf16* __restrict__ B, void* C,
                                                          const bf16* __restrict__ bias, const bf16* R, int M, int N, int K,
                                                          int ldc, int S, float* ws, int* cnt) {
  constexpr int BM = 16 * MT, BN = 64 * NG, NA = MT / 4, NF = MT / 2 * NG;
  constexpr int FW = ORD ? NG / 2 : NG, KF = ORD ? 2 : 1, RW = ORD ? MT : MT / 2;  // a wave's columns / 16, k32 fragments of a
                                                                                   // step, rows / 16 that it stores
  constexpr int RING = mid_ring<MT, NG, FRAG>(), DB = RING - 1, NB = FW * KF, PART = mid_step<MT, NG, FRAG>();
  constexpr int YOUNGER = FRAG ? DB * NB + (DB - 1) * NA : (DB - 1) * (NA + NG);  // loads after those of a step's LDS
  extern __shared__ __attribute__((aligned(16))) char smem[];  // RING x (BM [+ BN]) x 128 B; at the end the k halves' exchange
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tm_n = (M + BM - 1) / BM, tiles = tm_n * ((N + BN - 1) / BN);
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int part = id / tiles, tile = id - part * tiles;
  const int m0 = tile % tm_n * BM, n0 = tile / tm_n * BN;
  const int nk = K / kBK, k0 = (int)((long long)nk * part / S), n = 2 * ((int)((long long)nk * (part + 1) / S) - k0);
  const int g = ORD ? wid : wid & 3, h = ORD ? 0 : wid >> 2;  // column group, k half

  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(A) + (size_t)m0 * K, (short)0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(B) + (size_t)n0 * K, (short)0, 0x7fffffff, 0x00020000);
  // a DMA load: 8 rows x 128 B, the pieces of a row swizzled
  auto dma_row = [&](int q) { return (q * 8 + wid) * 8 + (lane >> 3); };
  auto dma_col = [&](int row) { return k0 * (2 * kBK) + (((lane & 7) ^ ((row >> 1) & 7)) << 4); };
  int oa[3], ob[2];  // NA, FW (NG) of them
#pragma unroll
  for (int q = 0; q < NA; ++q) oa[q] = (min(m0 + dma_row(q), M - 1) - m0) * K * 2 + dma_col(dma_row(q));
  if constexpr (FRAG) {
#pragma unroll
    for (int f = 0; f < FW; ++f) ob[f] = min((g * FW + f) * 16, N - 16 - n0) * K * 2 + k0 * 4096 + h * 1024 + lane * 16;
  } else {
#pragma unroll
    for (int q = 0; q < NG; ++q) ob[q] = (min(n0 + dma_row(q), N - 1) - n0) * K * 2 + dma_col(dma_row(q));
  }
  bf16x8 br[FRAG ? DB : 1][FW][KF];
  // past the end the last step is read again (from L2): the count of loads stays what the code says
  auto load_lds = [&](int t, int slot) {
    const int so = min(t, n - 1) * 128;
    char* d = smem + slot * PART + wid * 1024;
#pragma unroll
    for (int q = 0; q < NA; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, GAI_LDS(d + q * 8192), 16, oa[q], so, 0, 0);
    if constexpr (!FRAG)
#pragma unroll
      for (int q = 0; q < NG; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, GAI_LDS(d + BM * 128 + q * 8192), 16, ob[q], so, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto load_b = [&](int t, bf16x8(&d)[FW][KF]) {
    const int so = min(t, n - 1) * 2048;
#pragma unroll
    for (int f = 0; f < FW; ++f)
#pragma unroll
      for (int e = 0; e < KF; ++e)
        d[f][e] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rb, ob[f], so + e * 1024, 0));
    __builtin_amdgcn_sched_barrier(0);
  };
  int a_rd[KF];  // + 2048 per 16 rows
#pragma unroll
  for (int e = 0; e < KF; ++e) a_rd[e] = (lane & 15) * 128 + (((4 * (h + e) + (lane >> 4)) ^ ((lane & 15) >> 1)) << 4);
  f32x4 acc[MT][FW];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int f = 0; f < FW; ++f) acc[i][f] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int d = 0; d < DB; ++d) {
    load_lds(d, d);
    if constexpr (FRAG) load_b(d, br[d]);
  }
  int slot = 0, free = DB;
  auto step = [&](int t, bf16x8(&b)[FW][KF]) {
    // this step's rows are in LDS and everybody has left the slot before it
    asm volatile("s_waitcnt vmcnt(%c0)" ::"i"(YOUNGER) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    load_lds(t + DB, free);
    const char* s = smem + slot * PART;
    if constexpr (!FRAG)
#pragma unroll
      for (int f = 0; f < FW; ++f)
#pragma unroll
        for (int e = 0; e < KF; ++e) b[f][e] = *reinterpret_cast<const bf16x8*>(s + BM * 128 + a_rd[e] + (g * FW + f) * 2048);
#pragma unroll
    for (int e = 0; e < KF; ++e) {
      bf16x8 af[MT];
#pragma unroll
      for (int i = 0; i < MT; ++i) af[i] = *reinterpret_cast<const bf16x8*>(s + a_rd[e] + i * 2048);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int f = 0; f < FW; ++f) acc[i][f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[f][e], af[i], acc[i][f], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (FRAG) load_b(t + DB, b);
    free = slot;
    slot = slot + 1 == RING ? 0 : slot + 1;
  };
  int t = 0;
  for (; t + DB <= n; t += DB)
#pragma unroll
    for (int u = 0; u < DB; ++u) step(t + u, br[FRAG ? u : 0]);
  // the rest, outside the loop: an exit from its middle would join its back edge, and every load be waited for there
#pragma unroll
  for (int u = 0; u < DB - 1; ++u)
    if (t + u < n) step(t + u, br[FRAG ? u : 0]);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS is left
  // the epilogue's operands, under way while the sums are exchanged (a wave that another one finishes for has asked in vain):
  // 187 rows with a residual, a graph's launches: 4096 x 14336 46.4 -> 45.6 us, 4096 x 4096 22.1 -> 21.5, 1024 x 4096 16.2 -> 15.3
  bf16x4 rb4[epi_bias(EPI) ? FW : 1], rx[epi_res(EPI) ? RW : 1][epi_res(EPI) ? FW : 1];
  if constexpr (epi_bias(EPI) || epi_res(EPI)) {
#pragma unroll
    for (int f = 0; f < FW; ++f) {
      const int nn = min(n0 + (g * FW + f) * 16, N - 16) + 4 * (lane >> 4);
      if constexpr (epi_bias(EPI)) rb4[f] = *reinterpret_cast<const bf16x4*>(bias + nn);
      if constexpr (epi_res(EPI))
#pragma unroll
        for (int i = 0; i < RW; ++i)
          rx[i][f] = *reinterpret_cast<const bf16x4*>(R + (size_t)min(m0 + 16 * (h * RW + i) + (lane & 15), M - 1) * ldc + nn);
    }
  }
  f32x4 v[NF];  // [RW][FW]
  if constexpr (ORD) {
#pragma unroll
    for (int i = 0; i < RW; ++i)
#pragma unroll
      for (int f = 0; f < FW; ++f) v[i * FW + f] = acc[i][f];
  } else {
    // the k halves: this wave keeps row tiles h * MT / 2 .. of its columns and adds what its partner has of them
    __syncthreads();
    f32x4* x = reinterpret_cast<f32x4*>(smem) + g * 2 * NF * 64 + lane;  // [group][half][NF][64]
#pragma unroll
    for (int i = 0; i < MT / 2; ++i)
#pragma unroll
      for (int f = 0; f < NG; ++f) {
        v[i * NG + f] = h ? acc[MT / 2 + i][f] : acc[i][f];
        x[((h ^ 1) * NF + i * NG + f) * 64] = h ? acc[i][f] : acc[MT / 2 + i][f];
      }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      const f32x4 y = x[(h * NF + e) * 64];
      v[e] = h ? y + v[e] : v[e] + y;  // first half + second half
    }
  }
  if constexpr (!ORD && EPI == EPI_NONE && !OUTF32) {
    if (ws && !cnt) {  // slabs [part][M][N] for the launch that adds them
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        const int m = m0 + 16 * (h * RW + i) + (lane & 15);
        float* d = ws + ((size_t)part * M + m) * N + n0 + g * FW * 16 + 4 * (lane >> 4);
#pragma unroll
        for (int f = 0; f < FW; ++f)
          if (m < M && n0 + (g * FW + f) * 16 < N) *reinterpret_cast<f32x4*>(d + 16 * f) = v[i * FW + f];
      }
      return;
    }
  }
  if (!ORD && S > 1) {
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(ws, (short)0, 0x7fffffff, 0x00020000);
    auto woff = [&](int p, int e) {
      return (unsigned)__builtin_amdgcn_readfirstlane(((p * tiles + tile) * 8 + wid) * (NF * 1024) + e * 1024);
    };
    int* ctr = cnt + tile * 8 + wid;
    bool stored = false;
    if (__builtin_amdgcn_readfirstlane(__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) != S - 1) {
#pragma unroll
      for (int e = 0; e < NF; ++e)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v[e]), rw, lane * 16, woff(part, e), 16);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's share has landed
      int tk = 0;
      if (lane == 0) tk = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__builtin_amdgcn_readfirstlane(tk) != S - 1) return;
      stored = true;
    }
    if (lane == 0) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");  // no instruction: keeps the loads below the ticket
    f32x4 sum[NF], nx[4][NF];  // four parts' loads at a time
#pragma unroll
    for (int e = 0; e < NF; ++e) sum[e] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < S; p += 4) {
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int e = 0; e < NF; ++e)
          nx[d][e] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16, woff(min(p + d, S - 1), e), 16));
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        if (p + d >= S) break;
        const bool own = p + d == part && !stored;
#pragma unroll
        for (int e = 0; e < NF; ++e) sum[e] += own ? v[e] : nx[d][e];
      }
    }
#pragma unroll
    for (int e = 0; e < NF; ++e) v[e] = sum[e];
  }
  // lane: row m of C, columns n .. n + 3 of each 16 x 16 tile
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int m = m0 + 16 * (h * RW + i) + (lane & 15);
    if (m >= M) continue;
    const int nn = n0 + g * FW * 16;
    if constexpr (epi_glu(EPI)) {
      static_assert(FW == 2, "a gated pair of column tiles belongs to one wave");
      if (nn >= N) continue;
      f32x4 y;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = glu_act<EPI>(v[i * NG][r], v[i * NG + NG - 1][r]);
      store4<EPI_NONE, OUTF32>(C, bf16x4{}, bf16x4{}, ldc, m, nn / 2 + 4 * (lane >> 4), y);
    } else {
#pragma unroll
      for (int f = 0; f < FW; ++f)
        if (nn + 16 * f < N) store4<EPI, OUTF32>(C, rb4[epi_bias(EPI) ? f : 0], rx[epi_res(EPI) ? i : 0][epi_res(EPI) ? f : 0], ldc, m,
                               nn + 16 * f + 4 * (lane >> 4), v[i * FW + f]);
    }
  }
}

int mid_cus() {
  static int ncu = 0;
  if (!ncu) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || ncu < 8)
      gai_launch_error(__FILE__, __LINE__, "gemm_mid: cannot query the CU count");
  }
  return ncu;
}

int mid_tiles(int M, int N, int mt, int ng) { return ((M + 16 * mt - 1) / (16 * mt)) * ((N + 64 * ng - 1) / (64 * ng)); }

size_t part_bytes(int M, int N, int mt, int ng, int S) {
  return (size_t)mid_tiles(M, N, mt, ng) * S * 8 * (mt / 2 * ng) * 1024;
}

// 32-bit workspace offsets, and the caller's tickets
bool parts_fit(int M, int N, int mt, int ng, int S) {
  return mid_tiles(M, N, mt, ng) * 8 <= kGaiMidTickets && part_bytes(M, N, mt, ng, S) < (1ull << 31);
}

// Modelled times in us. This kernel: fitted to 2362 timings of 230 products (65 to 2048 rows, N 256 to 28672, K 256 to 14336,
// both weight layouts, weights from HBM) with up to 7 plans each; 19 of 20 within 16 %, the chosen plan on average 0.6 % above the
// best of those (the terms of bias and GELU from an earlier fit over every epilogue). The kernels below: 1376 products, 9 of 10
// within 15 %. Without the bytes of the parts,
// the epilogues and the rounds of short K, the model's first form lost up to 54 % (1535 x 2176 x 384: 9.4 -> 14.4 us; with
// 150 MB of parts 1536 x 11264 x 2048: 90 -> 258).
struct MidFit {
  double base, round, alone, full;  // launch; of a round of workgroups; of a 128-deep K step, few workgroups / full chip
  double weights, few, row_major;   // GB/s / 1000 of the weights, the share of it with few workgroups; the factor of a row-major step whose
                                    // loads were in operand layout
  double part0, part1, parts;       // parts of K: once, each, GB/s / 1000 of the sums written and read
  double out, bias, gelu;           // GB/s / 1000 of residual and result; epilogues
};
constexpr MidFit kFit[3] = {{3.5, 0.7, 0.49, 0.61, 4.45, 0.35, 1.47, 0.7, 0.67, 7.4, 4.5, 0.5, 1.1},   // 128 x 64
                            {3.6, 1.4, 0.79, 0.88, 4.5, 0.7, 1.7, 0.85, 0.8, 6.9, 3.05, 0.95, 2.0},     // 128 x 128
                            {3.9, 2.7, 1.03, 1.16, 4.2, 0.67, 1.47, 1.5, 1.08, 7.2, 3.1, 1.45, 2.7}};   // 192 x 128
constexpr double kTicketFill = 0.8;  // a captured launch clears its tickets (1.6 us): half of it counted always, the plan is the same

// MB written and read by the epilogue; 0 none, 1 bias / residual, 2 GELU and the like
double out_mb(int M, int N, int epi) {
  const bool res = epi == EPI_RESIDUAL || epi == EPI_BIAS_RESIDUAL;
  return (double)M * (epi_glu(epi) ? N / 2 : N) * (res ? 4 : 2) / 1e6;
}
int epi_class(int epi) {
  return epi == EPI_NONE || epi_glu(epi) ? 0 : epi == EPI_BIAS_GELU || epi == EPI_BIAS_QUICKGELU ? 2 : 1;
}

// step: of a layout's K step against one of fragment order
double mid_cost(int M, int N, int K, int epi, int mt, int ng, int S, double step) {
  const MidFit& f = kFit[mt == 12 ? 2 : ng - 1];
  const int items = mid_tiles(M, N, mt, ng) * S, steps = (K / kBK + S - 1) / S, G = mid_cus(), rounds = (items + G - 1) / G;
  const double fill = std::min(1.0, (double)items / G);
  const int ec = epi_class(epi);
  return f.base + std::max(rounds * (f.round + steps * (f.alone + (f.full - f.alone) * fill) * step), (double)N * K * 2 / 1e6 / (f.weights * (f.few + (1 - f.few) * fill))) +
         out_mb(M, N, epi) / f.out + (ec == 1 ? f.bias : ec == 2 ? f.gelu : 0.0) +
         (S > 1 ? f.part0 + f.part1 * S + 2 * part_bytes(M, N, mt, ng, S) / 1e6 / f.parts + kTicketFill : 0.0);
}
// the kernels of gemm_impl.h, by its own rules: skinny, stream-K, 256 x 256 tiles, 128 x 128 tiles
double other_cost(int M, int N, int K, int epi) {
  const int G = mid_cus() & ~7, ec = epi_class(epi), kt = K / 64;
  const int t1 = ((M + 127) / 128) * ((N + 127) / 128), t2 = ((M + 255) / 256) * ((N + 255) / 256), r2 = (t2 + G - 1) / G;
  const double wmb = (double)N * K * 2 / 1e6, out = out_mb(M, N, epi);
  if (M <= 128 && K % 256 == 0) {
    const bool two = epi_glu(epi) || N / 32 >= 512;
    const int r = ((two ? (N + 31) / 32 : (N + 15) / 16) + G - 1) / G;
    return two ? 0.9 + std::max(r * (2.0 + K / 256 * (1.38 + 0.14 * M / 16)), wmb / 3.15) + out / 1.3 + (ec ? 0.7 : 0.0)
               : 3.0 + std::max(r * (0.14 + K / 256 * (0.89 + 0.16 * M / 16)), wmb / 5.0) + out / 4.2;
  }
  if (N >= 256 && K >= 192 && M >= 256) {
    if (K >= 8192 && 2 * t2 < G)  // a tile's sums of G / t2 workgroups are added by one
      return 25.7 + 2.05 * t2 * kt / G + 2.04 * G / t2 + 9.2 * std::max(0.0, 1.0 - t2 * kt / (20.0 * G));
    if (2 * t2 >= G) {
      const double fill = std::min(1.0, (double)t2 / G);
      return N >= 16384 ? 4.9 + r2 * (2.3 + kt * (1.30 + 0.06 * fill)) + out / 9.5 + (ec == 2 ? 10.0 : ec ? 2.5 : 0.0)
                        : 6.7 + r2 * kt * (0.93 + 0.41 * fill) + out / 7.4 + (ec == 2 ? 6.1 : ec ? 0.5 : 0.0);
    }
  }
  const double fill = (double)t1 / G, step = 0.65 + 0.11 * std::min(1.0, fill) + 0.13 * std::min(1.0, std::max(0.0, fill - 1.0)) +
                                             0.25 * std::min(1.0, wmb / 64);
  return 3.6 + (t1 + 2 * G - 1) / (2 * G) * (0.73 + kt * step) + out / 4.0 + (ec == 2 ? 10.1 : ec ? 7.0 : 0.0);
}
// A weight gives the same bits in either layout: which kernel, and into how many parts, is one choice for both; only the tile
// is the layout's own (a sum's order does not depend on it). The parts are those of the smaller row-major + 2 x fragment-order
// time: the large weights, where parts matter most, are stored in fragment order. (The row-major times of that sum are of the
// loads in operand layout: parts, and with them every bit, stay where they were.)
constexpr double kFragShare = 2.0;
constexpr double kRowStep[3] = {1.14, 1.12, 1.1};  // a row-major step by DMA against one of fragment order: 128 x 64, 128, 192 x 128
// A product is taken where the model says so much less time than the kernels it replaces take, in both layouts. Deep K leaves the model
// of the 256 x 256 kernels up to a fifth too slow where the tiles divide the chip evenly. Of 1210 products in one layout (30 weights,
// 22 numbers of rows from 65 to 2048), timed with every plan and on the other kernels, the chosen way is on average 2.6 % above the best;
// with row-major steps at 1.47 - 1.7, and a row-major margin that made up for it at deep K, 3.6 %: 1536 rows 2048 x 2048, fragment
// order, 31.7 us instead of 21.1, 128 rows of a gated 5632 x 2048 22.7 instead of 16.3. The margins up to 128 rows and past 1024
// leave 128 x 1024 x 1024 with bias (11.2 us, 8.6 here) and 1536 rows of a gated 11264 x 2048 (94, 86) on the other kernels.
double margin(int M, int K) { return M >= 256 && K >= 8192 ? 1.2 : 1.05; }
double margin_row_major(int M, int K, bool glu) {
  if (M <= 128) return glu ? 1.05 : 1.28;
  return M >= 256 && K >= 8192 ? 1.27 : M <= 1024 ? 1.1 : 1.21;
}

// the ordered form, fitted to 600 timings of 150 products of up to 3072 rows (17 of 20 within 15 %)
double ordered_cost(int M, int N, int K, int mt, int bfrag) {
  const int items = mid_tiles(M, N, mt, 2), G = mid_cus(), rounds = (items + G - 1) / G;
  const double fill = std::min(1.0, (double)items / G), step = mt == 4 ? 0.61 + 0.04 * fill : 0.81 + 0.12 * fill;
  // row-major weights, as with loads in operand layout: by DMA a step is 1.02 - 1.29 of one in fragment order, but with that the rows of
  // 6000 x 4096 x 4096 were split too (164 -> 178 us)
  const double row = mt == 4 ? 1.68 : 1.42;
  return (mt == 4 ? 2.4 : 2.3) + rounds * ((mt == 4 ? 1.55 : 3.0) + K / kBK * step * (bfrag ? 1.0 : row));
}

// operands of the kernel: whole k steps and column tiles, 4-column loads and stores, 16-byte loads of A and B
bool mid_fits(const void* A, const void* B, const void* C, const void* bias, const void* R, int M, int N, int K, int ldc, int epi,
              int out_f32) {
  if (M < 1 || K % kBK || N % 16 || ldc % 4 || (out_f32 && epi != EPI_NONE)) return false;
  if (!(epi >= EPI_NONE && epi <= EPI_BIAS_QUICKGELU) && !(epi_glu(epi) && N % 32 == 0)) return false;
  auto off = [](const void* p, unsigned a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) != 0; };
  return !(off(A, 16) || off(B, 16) || off(C, out_f32 ? 16 : 8) || off(bias, 8) || off(R, 8));
}

template <int MT, int NG, int EPI, bool OUTF32, bool ORD, bool FRAG>
void launch_mid_order(const void* A, const void* B, void* C, const void* bias, const void* R, int M, int N, int K, int ldc, int S,
                      float* ws, int* cnt, hipStream_t st) {
  constexpr int lds = std::max(mid_step<MT, NG, FRAG>() * mid_ring<MT, NG, FRAG>(), MT * NG * 4096);  // the ring; the exchange
  auto kern = gemm_mid_kernel<MT, NG, EPI, OUTF32, ORD, FRAG>;
  static bool once = false;
  if (!once) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      gai_launch_error(__FILE__, __LINE__, "gemm_mid: LDS size");
    once = true;
  }
  kern<<<mid_tiles(M, N, MT, NG) * S, 512, lds, st>>>((const bf16*)A, (const bf16*)B, C, (const bf16*)bias, (const bf16*)R, M, N, K,
                                                      ldc, S, ws, cnt);
  GAI_LAUNCH_CHECK();
}

template <int MT, int NG, int EPI, bool OUTF32, bool ORD = false>
void launch_mid(const void* A, const void* B, void* C, const void* bias, const void* R, int M, int N, int K, int ldc, int S,
                float* ws, int* cnt, hipStream_t st, int bfrag) {
  if (bfrag) launch_mid_order<MT, NG, EPI, OUTF32, ORD, true>(A, B, C, bias, R, M, N, K, ldc, S, ws, cnt, st);
  else launch_mid_order<MT, NG, EPI, OUTF32, ORD, false>(A, B, C, bias, R, M, N, K, ldc, S, ws, cnt, st);
}

}  // namespace

bool gai_gemm_mid_plan(const void* A, const void* B, const void* C, const void* bias, const void* R, int M, int N, int K,
                       int ldc, int epi, int out_f32, int force, int bfrag, GaiMidPlan* plan) {
  if (!mid_fits(A, B, C, bias, R, M, N, K, ldc, epi, out_f32)) return false;
  if (force == 0 && (M <= 64 || M > 2048 || N < 256)) return false;
  const bool glu = epi_glu(epi);
  GaiMidPlan best{8, 2, 1, 0, 0.0};
  if (force >= 100000) {
    if (glu) return false;
    best = {force == 104201 ? 4 : 8, 2, 1, 0, 0.0, 0, true};
  } else if (force >= 1000) {
    best = {force / 1000, glu ? 2 : force / 100 % 10, std::max(1, std::min(force % 100, K / kBK)), 0, 0.0};
  } else {
    double bc = 1e30, row = 1e30, frag = 1e30;
    for (int S = 1; S <= std::min(16, std::max(1, K / kBK / 4)); ++S) {
      GaiMidPlan at[2] = {{8, 2, S, 0, 1e30}, {8, 2, S, 0, 1e30}};  // row-major, fragment order: the best tile
      double operand = 1e30;
      for (int v = glu ? 1 : 0; v < 3; ++v) {
        const int mt = v == 2 ? 12 : 8, ng = v == 0 ? 1 : 2;
        if (S > 1 && !parts_fit(M, N, mt, ng, S)) continue;
        operand = std::min(operand, mid_cost(M, N, K, epi, mt, ng, S, kFit[v].row_major));
        for (int l = 0; l < 2; ++l) {
          const double c = mid_cost(M, N, K, epi, mt, ng, S, l ? 1.0 : kRowStep[v]);
          if (c < at[l].cost) at[l] = {mt, ng, S, 0, c};
        }
      }
      const double c = operand + kFragShare * at[1].cost;
      if (c < bc) {
        bc = c;
        row = at[0].cost;
        frag = at[1].cost;
        best = at[bfrag ? 1 : 0];
      }
    }
    const double other = other_cost(M, N, K, epi);
    if (force == 0 && (frag * margin(M, K) >= other || row * margin_row_major(M, K, glu) >= other)) return false;
  }
  if (best.parts > 1 && !parts_fit(M, N, best.mt, best.ng, best.parts)) best.parts = 1;
  if (best.parts > 1) {
    best.ws_floats = part_bytes(M, N, best.mt, best.ng, best.parts) / 4;
    best.tickets = 8 * mid_tiles(M, N, best.mt, best.ng);
  }
  *plan = best;
  return true;
}

// The 256 x 256 kernels work in rounds of one tile per CU, 6 us + 1.42 us per 64 of K each (M 16384, N 4096: 28.5, 49, 94 us at
// K 1024, 2048, 4096; 9 more with a residual), however few tiles the last one has. Its rows go to this kernel where the
// model says so with 15 % to spare (its own error) and a launch, and the saving is 5 % of the whole. N 1024 with a residual,
// 18337 rows (288 tiles on 256 CUs): K 1024 57.5 -> 54.4 us, K 4096 167.3 -> 145.0. Over 320 products of 2100 to 60000 rows
// (N 256 to 9000, K 256 to 14336) the rule splits 127, one of them 3 % slower for it; all in all 3.6 % faster, 3.9 % at best.
// At N 3072 and 4096, K 1024 the remainder costs as much as the round it saves; after many rounds (Llama-3-8B gate_up at
// 14500 rows: 25) the tiles have drifted apart and there is no empty round left to save.
int gai_gemm_mid_tail(const void* A, const void* B, const void* C, const void* bias, const void* R, int M, int N, int K, int ldc,
                      int epi, int out_f32, int bfrag, GaiMidPlan* plan) {
  if (M <= 2048 || N < 256 || ldc % 8 || K < 256 || epi_glu(epi) || !mid_fits(A, B, C, bias, R, M, N, K, ldc, epi, out_f32))
    return 0;
  if ((size_t)M * K * 2 >= (1ull << 31) || (size_t)N * K * 2 >= (1ull << 31)) return 0;  // not the 256 x 256 kernels
  const int G = mid_cus() & ~7, tn = (N + 255) / 256, tm = (M + 255) / 256;
  const long long tiles = (long long)tm * tn;
  if (tiles % G == 0) return 0;
  const int m1 = (int)(tiles / G * G / tn) * 256, m2 = M - m1;  // whole rounds, whole row tiles
  if (m1 <= 0 || m2 <= 0 || m2 > 3072) return 0;
  const double c4 = ordered_cost(m2, N, K, 4, bfrag), c8 = ordered_cost(m2, N, K, 8, bfrag);
  *plan = {c4 <= c8 ? 4 : 8, 2, 1, 0, std::min(c4, c8), 0, true};
  const double round = 6.0 + K / 64 * 1.42 + (R ? 9.0 : 0.0);
  const double saved = round - plan->cost * 1.15 - 3.0;
  return saved > 0.05 * round * ((tiles + G - 1) / G) ? m2 : 0;
}

// Where a norm follows, its launch can add the parts: the last workgroup of a tile no longer reads all of them by itself (a CU
// takes in 40 - 60 KB/us: eight parts of 192 x 128 are 15 us), so more parts pay, and K is cut where the rows of A would be fetched for
// few columns. Product and norm, fragment order, us, before | here: 187 rows 4096 x 14336 49.5 | 40.6, 4096 x 4096 25.5 | 21.6, 256 rows 54.2 | 47.0
// and 26.2 | 22.4, 96 rows 38.6 | 31.6 and 21.8 | 17.2, 640 rows 97.0 | 94.2 and 45.6 | 40.7.
// The model: 3336 timings of 200 products (65 to 640 rows, N 2048 to 8192, K 2048 to 14336), nine in ten within 13 %, and for the choice
// product and norm together, here and as they would run without slabs (the plan of the product that adds its own residual, or the kernels
// past this one), fitted to both ways of 2588 products (N 2048 to 8192 before a rms norm, 256 to 2048 before a layer norm, both layouts),
// nine in ten within 10 %. A layer norm's wave reads a row's slabs by itself, so wide rows in many parts cost it most. The rule takes 2265
// of these: before a rms norm 0.84 of the time on average, before a layer norm 0.79; the slowest, us: 160 rows 5120 x 14336 53.5 | 54.3 (row-major
// 55.2 | 56.9), 8192 x 14336 89.8 | 70.7 (72.9 | 74.3); of 700 others that it takes six are more than 1 % slower in fragment order, 417 x 1536 x 1280
// before a layer norm 13.1 | 13.8 the most, and 142 x 7328 x 12288 60.6 | 62.8 (62.5 | 69.0). Without the comparison 385 x 2048 x 1024 took 13.1 instead of 12.3, before a layer norm 385 x 1536 x
// 768 12.5 instead of 11.2, 65 x 2048 x 3072 18.3 instead of 17.1 and 212 x 1088 x 1920 15.8 instead of 14.5; past 512 rows two short parts
// fill the pipeline too often (513 x 4096 x 3072 31.9 instead of 30.3). At 1000 rows the slabs' bytes cost more than the sums did (46.4 |
// 48.2, 126.9 | 131.2).
namespace {
struct SlabFit {
  double base, alone, full, weights, few, slabs, round;  // as MidFit; slabs: GB/s / 1000 written; round: each past the first
};
constexpr SlabFit kSlabFit[3] = {{2.9, 0.54, 0.64, 4.66, 0.31, 2.8, 0.43}, {4.7, 0.77, 1.0, 5.75, 0.39, 4.24, 2.97}, {6.8, 1.0, 1.23, 4.65, 1.0, 4.0, 5.25}};
constexpr double kSlabRead = 0.141, kSlabRows = 0.78e-6;  // the norm: us a MB of slabs, an element of the rows past 256
constexpr double kSlabMargin = 0.95;
// product and norm, us: base + slope x modelled product + read x the norm's reads of slabs one after another + elem x (elements x parts), against
// the same without slabs; least: what has to be saved at least
struct SlabNormFit {
  double base, slope, read, elem, was_base, was_slope, was_elem, least;
};
constexpr SlabNormFit kSlabRms = {4.31, 0.911, 2.05, 0.192e-6, 2.55, 0.974, 1.975e-6, 1.4};
constexpr SlabNormFit kSlabLayer = {2.76, 0.93, 0.194, 0.349e-6, 1.41, 1.021, 2.354e-6, 0.8};
constexpr double kSlabShare = 0.95;

double slabs_cost(int M, int N, int K, int v, int S) {
  const SlabFit& f = kSlabFit[v];
  const int items = mid_tiles(M, N, v == 2 ? 12 : 8, v == 0 ? 1 : 2) * S, G = mid_cus(), rounds = (items + G - 1) / G;
  const int steps = (K / kBK + S - 1) / S;
  const double fill = std::min(1.0, (double)items / G), mb = (double)S * M * N * 4 / 1e6;
  return f.base + std::max(rounds * steps * (f.alone + (f.full - f.alone) * fill), (double)N * K * 2 / 1e6 / (f.weights * (f.few + (1 - f.few) * fill))) +
         mb / f.slabs + f.round * (rounds - 1) + kSlabRead * mb + kSlabRows * std::max(0, M - 256) * N;
}
}  // namespace

bool gai_gemm_mid_slabs_plan(int M, int N, int K, int most, bool layer, GaiMidPlan* plan) {
  if (M <= 64 || M > 640 || N < 256 || N > 8192 || N % 16 || K % kBK || (long long)N * K * 2 >= 1ll << 31) return false;
  double one = 1e30, more = 1e30;
  for (int v = 0; v < 3; ++v)
    for (int S = 1; S <= std::min(most, 16) && K / kBK / S >= 3; ++S) {
      if ((long long)S * M * N * 4 >= 1ll << 31) break;
      const double c = slabs_cost(M, N, K, v, S);
      if (S == 1) {
        one = std::min(one, c);
      } else if (c < more) {
        more = c;
        *plan = {v == 2 ? 12 : 8, v == 0 ? 1 : 2, S, 0, c};
      }
    }
  if (more >= kSlabMargin * one || (!layer && M > 512 && K < 4096)) return false;
  const int epi = layer ? EPI_BIAS_RESIDUAL : EPI_RESIDUAL;
  GaiMidPlan was;
  const double product = gai_gemm_mid_plan(nullptr, nullptr, nullptr, nullptr, nullptr, M, N, K, N, epi, 0, 0, 1, &was) ? was.cost : other_cost(M, N, K, epi);
  const SlabNormFit& f = layer ? kSlabLayer : kSlabRms;
  const int reads = layer ? gai_slabs_layernorm_reads(plan->parts, N) : N > 4096;  // (a rms norm of wider rows has fewer waves a row)
  const double now = f.base + f.slope * more + f.read * reads + f.elem * M * N * plan->parts;
  const double then = f.was_base + f.was_slope * product + f.was_elem * M * N;
  return now < kSlabShare * then && then - now > f.least;
}

// res += product; rms norm: in the product's epilogue, or (apart) by the norm, which then reads the product and the stream and writes the stream
// as well, at the copy's 4.8 TB/s. The kernels of 128 x 128 tiles ask for the residual when their sums are done, 8 - 10 us in all, and a tile of the
// others hides it or has enough rounds to. Both timed at 2286 products of 65 to 14643 rows (N 512 to 8192, K 512 to 14336, both layouts): apart
// at 420 of them, where the epilogue took 1.21 of the time on average and nowhere less than 0.99 (2100 rows 2048 x 4096 63.8 | 70.4 us, 4100 x 1024 x 1024
// 26.1 | 36.5); at the others it takes 0.954, and 10 % more at worst (641 x 1024 x 8192).
bool gai_gemm_residual_apart(int M, int N, int K) {
  auto product = [&](int epi) {
    GaiMidPlan p;
    return gai_gemm_mid_plan(nullptr, nullptr, nullptr, nullptr, nullptr, M, N, K, N, epi, 0, 0, 1, &p) ? p.cost : other_cost(M, N, K, epi);
  };
  return product(EPI_RESIDUAL) > product(EPI_NONE) + (double)M * N * 4 / 4.8e6 + 1.0;
}

void gai_gemm_mid_slabs(const void* A, const void* B, int M, int N, int K, const GaiMidPlan& p, float* ws, hipStream_t st, int bfrag) {
#define GAI_MID_SLABS(MT, NG)   \
  if (p.mt == MT && p.ng == NG) \
    return launch_mid<MT, NG, EPI_NONE, false>(A, B, nullptr, nullptr, nullptr, M, N, K, N, p.parts, ws, nullptr, st, bfrag);
  GAI_MID_SLABS(8, 1)
  GAI_MID_SLABS(8, 2)
  GAI_MID_SLABS(12, 2)
#undef GAI_MID_SLABS
  gai_launch_error(__FILE__, __LINE__, "gemm_mid: no kernel for this plan");
}

void gai_gemm_mid(const void* A, const void* B, void* C, const void* bias, const void* R, int M, int N, int K, int ldc, int epi,
                  int out_f32, const GaiMidPlan& p, float* ws, int* tickets, hipStream_t st, int bfrag) {
  if (p.parts > 1 && !(tickets && ws)) gai_launch_error(__FILE__, __LINE__, "gemm_mid: no workspace for the parts of K");
#define GAI_MID(MT, NG, E, F32)                                                                         \
  if (p.mt == MT && p.ng == NG)                                                                         \
    return launch_mid<MT, NG, E, F32>(A, B, C, bias, R, M, N, K, ldc, p.parts, ws, tickets, st, bfrag);
#define GAI_MID_ORD(MT, E, F32)                                                                           \
  if (p.ordered && p.mt == MT)                                                                            \
    return launch_mid<MT, 2, E, F32, true>(A, B, C, bias, R, M, N, K, ldc, 1, nullptr, nullptr, st, bfrag);
#define GAI_MID_EPI(E, F32)         \
  {                                 \
    GAI_MID_ORD(4, E, F32)          \
    GAI_MID_ORD(8, E, F32)          \
    GAI_MID(8, 1, E, F32)           \
    GAI_MID(8, 2, E, F32)           \
    GAI_MID(12, 2, E, F32)          \
    break;                          \
  }
#define GAI_MID_GLU(E)              \
  {                                 \
    GAI_MID(8, 2, E, false)         \
    GAI_MID(12, 2, E, false)        \
    break;                          \
  }
  switch (epi) {
    case EPI_NONE:
      if (out_f32) GAI_MID_EPI(EPI_NONE, true) else GAI_MID_EPI(EPI_NONE, false)
      break;
    case EPI_BIAS: GAI_MID_EPI(EPI_BIAS, false)
    case EPI_BIAS_GELU: GAI_MID_EPI(EPI_BIAS_GELU, false)
    case EPI_RESIDUAL: GAI_MID_EPI(EPI_RESIDUAL, false)
    case EPI_SWIGLU: GAI_MID_GLU(EPI_SWIGLU)
    case EPI_BIAS_RESIDUAL: GAI_MID_EPI(EPI_BIAS_RESIDUAL, false)
    case EPI_BIAS_RELU: GAI_MID_EPI(EPI_BIAS_RELU, false)
    case EPI_BIAS_QUICKGELU: GAI_MID_EPI(EPI_BIAS_QUICKGELU, false)
    case EPI_GEGLU: GAI_MID_GLU(EPI_GEGLU)
    default: break;
  }
#undef GAI_MID_GLU
#undef GAI_MID_EPI
#undef GAI_MID_ORD
#undef GAI_MID
  gai_launch_error(__FILE__, __LINE__, "gemm_mid: no kernel for this plan");
}
