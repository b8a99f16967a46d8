// Exact brute-force vector search: fused similarity GEMM + top-k.
//
// scores[q, x] = Q[q] . X[x] + bias[x]  with bias = 0 (inner product / cosine on
// normalised vectors), -0.5*|x|^2 (L2 ranking) or -inf (deleted row), so one
// kernel serves IP / cosine / L2 and tombstones. The [nq, N] score matrix is
// never materialised. Both paths stream X once per 64-query tile through
// v_mfma_f32_16x16x32_bf16 (sim_topk_stream):
//   short lists (k <= 8 for one query tile; k <= 4 for more where the form below is slower or does not run): every lane
//   keeps a sorted list of its best rows in registers; the lists of a workgroup are merged in LDS and the workgroups'
//   lists by sim_topk_stage2;
//   else only the largest score of every group of 16 or 4 rows is kept (sim_topk_stream<.., 0 or -4, ..>), and one workgroup per
//   query picks the k best groups - which hold the k best rows - and scores their rows again (sim_topk_select). Which groups:
//   ops._topk_group_rows.
// More than 64 queries in one call (columns a multiple of 64, at least 256) take the groups from a tiled product instead
// (sim_group_max). The caller's slices hold that many up to 8.4M rows.
// us, lists / groups (first form of k > 8: a 64-entry list per lane): 1M x 1024, k = 4, 1 query 353 / 417; k = 8, 64 queries 422 /
// 510; k = 40, 1 query (18263) / 430. Lists / groups of the stream / of the tiled product, 300 queries: 250k x 1024, k = 4 414 / - /
// 238, k = 8 - / 393 / 242, k = 40 (144700) / 470 / 250; 1M x 1024, k = 8 1375 / 1277 / 800; 100k x 384, k = 8 - / 94 / 77; 65
// queries, 250k x 1024, k = 4 193 / 191 / 143. (Where lists stay for k <= 4: ops.sim_topk.)
#include <algorithm>

#include "gai_common.h"
#include "gai_kernels.h"

using namespace gai;

namespace {

// Group maxima of a query: a place per 16 rows, in order, or per 4 rows: of 32 rows, places 2 l + i hold rows 16 i + 4 l .. + 3, as the
// lanes of two accumulator tiles lie.
template <int GR>
__device__ __forceinline__ int place_group(int p) {
  return GR == 16 ? p : (p & ~7) | (p & 1) << 2 | (p >> 1 & 3);
}
template <int GR>
__device__ __forceinline__ int group_place(int g) {
  return GR == 16 ? g : (g & ~7) | (g & 3) << 1 | (g >> 2 & 1);
}
int places(int gr, int N) { return gr == 16 ? (N + 15) / 16 : (N + 31) / 32 * 8; }

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

template <int K>
struct TopK {
  float v[K];
  int i[K];
  __device__ __forceinline__ void init() {
#pragma unroll
    for (int j = 0; j < K; ++j) {
      v[j] = -INFINITY;
      i[j] = -1;
    }
  }
  __device__ __forceinline__ void insert(float s, int id) {
    if (!(s > v[K - 1])) return;
    v[K - 1] = s;
    i[K - 1] = id;
#pragma unroll
    for (int j = K - 1; j > 0; --j) {
      if (v[j] > v[j - 1]) {
        const float tv = v[j];
        v[j] = v[j - 1];
        v[j - 1] = tv;
        const int ti = i[j];
        i[j] = i[j - 1];
        i[j - 1] = ti;
      }
    }
  }
};

// ------------------------------------------------------------------------------------------------
// Streaming stage 1: X at HBM rate, one workgroup per row range (about one per CU) and 16 * MT queries.
//  * MFMA A = 16 X rows, B = 16 queries: lane l ends a 16-row group owning query l&15 (+16i) and rows 4(l>>4)..+3, so
//    the group is finished straight from the accumulator, no LDS transpose;
//  * X fragments flow through a 16-deep register ring (16 KiB in flight per wave) that runs across
//    group boundaries: the two 64-B halves of every 128-B X line are issued back to back;
//  * K > 0: per-lane register top-K lists; the 32 lists of a query (8 waves x 4 row-lanes) are merged in LDS
//    once at the end;
//  * K = 0: the largest score of each group goes to gmax[query][group], 16-byte runs of four groups; K = -4: that of every four rows. Keeping 64 sorted
//    entries per lane instead (the first form of k > 8) made nearly every insertion a divergent 64-step chain: 300
//    queries x 250k rows x 1024, k = 40, took 144 ms; group maxima are 1/16 of the scores at 3 + 2/4 instructions each;
//  * several query tiles read the same X rows: the tiles of one row range run one after the other on one XCD, so all but
//    the first find the rows in its L2 (300 queries x 1M x 1024, k = 4: 1749 -> 1276 us).
// ------------------------------------------------------------------------------------------------
template <int MT, int K, int RING>
__global__ __launch_bounds__(512) void sim_topk_stream(const bf16* __restrict__ Q, const bf16* __restrict__ X,
                                                       const float* __restrict__ bias, int nq, int N, int D,
                                                       int rows_per_wg, int qtiles, float* __restrict__ ws_v,
                                                       int* __restrict__ ws_i, float* __restrict__ gmax, int ngr) {
  constexpr int NQ = 16 * MT;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  char* qimg = smem;
  float* bsm = reinterpret_cast<float*>(smem + (size_t)NQ * D * 2);  // this workgroup's bias rows
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int seq = blockIdx.x >> 3;                              // position in its XCD's order
  const int wgx = seq / qtiles * 8 + (blockIdx.x & 7);          // row range
  const int q0 = seq % qtiles * NQ;                             // query tile
  if (wgx * rows_per_wg >= N) return;                           // the grid is rounded up to whole XCD rounds
  const int ncols = D / 8;
  const int sw = ncols & 15 ? (ncols & 7 ? 3 : 7) : 15;  // the XOR swizzle stays inside a row (D is a multiple of 32)
  const int wg_row0 = wgx * rows_per_wg;
  for (int e = tid; e < NQ * ncols; e += 512) {
    const int r = e / ncols, u = e % ncols;
    bf16x8 v = (q0 + r < nq) ? load8(Q + (size_t)(q0 + r) * D + u * 8) : bf16x8{};
    *reinterpret_cast<bf16x8*>(qimg + (size_t)r * D * 2 + ((u ^ (r & sw)) << 4)) = v;
  }
  // bias through LDS: a global load inside the X stream would make every wait drain the ring
  for (int r = tid; r < rows_per_wg; r += 512) bsm[r] = wg_row0 + r < N ? bias[wg_row0 + r] : -INFINITY;
  __syncthreads();

  TopK<(K > 0 ? K : 1)> tk[MT];
  float best[MT];  // K = 0: this lane's share of the last four groups' maxima
  float last4[K == -4 ? MT : 1][4] = {};
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    tk[i].init();
    best[i] = -INFINITY;
  }
  const int wave_rows = rows_per_wg / 8;  // multiple of 16
  const int r_begin = wg_row0 + wid * wave_rows;
  const int r_end = min(N, r_begin + wave_rows);
  const int ngroups = r_end > r_begin ? (r_end - r_begin + 15) / 16 : 0;
  const int nk = D / 32;             // k-steps per 16-row group; RING divides it
  const int total = ngroups * nk;    // a multiple of RING: no tail guard inside the stream
  // the stream position advances by RING k-steps per chunk; pointers are stepped, and set once per group: rows past the
  // wave's range (the prefetch's last chunk, a partial last group of the index) re-read the index's last row
  int prow = r_begin + (lane & 15);
  auto row_ptr = [&]() { return X + (size_t)(prow < r_end ? prow : N - 1) * D + 8 * (lane >> 4); };
  int pf_t = 0;                  // k-step of the prefetch pointer within its group
  const bf16* pf = row_ptr();    // prefetch pointer (k-step j0 + RING)
  auto advance_pf = [&]() {      // RING k-steps ahead
    pf_t += RING;
    if (pf_t == nk) {
      pf_t = 0;
      prow += 16;
      pf = row_ptr();
    } else {
      pf += 32 * RING;
    }
  };
  bf16x8 ring[RING];
#pragma unroll
  for (int u = 0; u < RING; ++u) ring[u] = load8(pf + 32 * u);
  advance_pf();
  f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  int g = 0, t0 = 0;
  for (int j0 = 0; j0 < total; j0 += RING) {
    // query fragments one k-step ahead (LDS latency hides under the previous step's MFMAs)
    auto rdq = [&](bf16x8* qf, int t) {
      const int uu = 4 * t + (lane >> 4);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int qr = 16 * i + (lane & 15);
        qf[i] = *reinterpret_cast<const bf16x8*>(qimg + (size_t)qr * D * 2 + ((uu ^ (qr & sw)) << 4));
      }
    };
    bf16x8 qa[MT], qb[MT];
    rdq(qa, t0);
#pragma unroll
    for (int u = 0; u < RING; ++u) {
      bf16x8* qc = (u & 1) ? qb : qa;
      bf16x8* qn = (u & 1) ? qa : qb;
      if (u + 1 < RING) rdq(qn, t0 + u + 1);
#pragma unroll
      for (int i = 0; i < MT; ++i)
        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ring[u], qc[i], acc[i], 0, 0, 0);  // D[x row][query]
      ring[u] = load8(pf + 32 * u);  // consumed first, then refilled: the slot keeps its registers
    }
    advance_pf();
    t0 += RING;
    if (t0 == nk) {  // a 16-row group is complete: 4 candidate rows per lane and query tile
      const int rl = r_begin - wg_row0 + 16 * g + 4 * (lane >> 4);
      const f32x4 bv = *reinterpret_cast<const f32x4*>(bsm + rl);
      if constexpr (K > 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = wg_row0 + rl + r;
          if (row < r_end) {
#pragma unroll
            for (int i = 0; i < MT; ++i) tk[i].insert(acc[i][r] + bv[r], row);
          }
        }
      } else if constexpr (K == -4) {
        const int gr = r_begin / 16 + g, u = gr & 3;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          const float m = fmaxf(fmaxf(fmaxf(-INFINITY, acc[i][0] + bv[0]), acc[i][1] + bv[1]),
                                fmaxf(fmaxf(-INFINITY, acc[i][2] + bv[2]), acc[i][3] + bv[3]));
#pragma unroll
          for (int e = 0; e < 4; ++e) last4[i][e] = u == e ? m : last4[i][e];
        }
        if (u == 3 || g + 1 == ngroups) {  // the last four groups at once: a store among the loads waits for those before it
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int lo = (gr & ~3) + 2 * h, at = lo * 4 + (lane >> 4) * 2;
            const bool has_lo = lo >= r_begin / 16 && lo <= gr, has_hi = lo + 1 >= r_begin / 16 && lo + 1 <= gr;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              float* d = gmax + (size_t)(q0 + 16 * i + (lane & 15)) * ngr + at;
              if (q0 + 16 * i + (lane & 15) >= nq) continue;
              if (has_lo && has_hi) *reinterpret_cast<f32x2*>(d) = f32x2{last4[i][2 * h], last4[i][2 * h + 1]};
              else if (has_lo) d[0] = last4[i][2 * h];
              else if (has_hi) d[1] = last4[i][2 * h + 1];
            }
          }
        }
      } else {  // rows past N have bias -inf; fmaxf passes NaN scores over
        const int gr = r_begin / 16 + g;
#pragma unroll
        for (int i = 0; i < MT; ++i) {
          float m = fmaxf(fmaxf(fmaxf(-INFINITY, acc[i][0] + bv[0]), acc[i][1] + bv[1]),
                          fmaxf(fmaxf(-INFINITY, acc[i][2] + bv[2]), acc[i][3] + bv[3]));
          m = fmaxf(m, __shfl_xor(m, 16, 64));
          m = fmaxf(m, __shfl_xor(m, 32, 64));
          if ((lane >> 4) == (gr & 3)) best[i] = m;
        }
        if ((gr & 3) == 3 || g + 1 == ngroups) {  // this lane's group: the one of the last four with its number
          const int mine = (gr & ~3) + (lane >> 4);
          if (mine >= r_begin / 16 && mine <= gr) {
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              const int q = q0 + 16 * i + (lane & 15);
              if (q < nq) gmax[(size_t)q * ngr + mine] = best[i];
            }
          }
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      t0 = 0;
      ++g;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if constexpr (K > 0) {
    // merge the 32 lists of every query (list = 4 * wave + row-lane group) in LDS (aliases the Q image)
    __syncthreads();
    float* mv = reinterpret_cast<float*>(smem);
    int* mi = reinterpret_cast<int*>(smem + (size_t)NQ * 32 * K * 4);
    const int list = wid * 4 + (lane >> 4);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int q = 16 * i + (lane & 15);
#pragma unroll
      for (int jj = 0; jj < K; ++jj) {
        mv[(q * 32 + list) * K + jj] = tk[i].v[jj];
        mi[(q * 32 + list) * K + jj] = tk[i].i[jj];
      }
    }
    __syncthreads();
    if (tid < NQ && q0 + tid < nq) {
      TopK<K> m;
      m.init();
      for (int l = 0; l < 32; ++l)
        for (int jj = 0; jj < K; ++jj) {
          const float v = mv[(tid * 32 + l) * K + jj];
          if (!(v > m.v[K - 1])) break;
          m.insert(v, mi[(tid * 32 + l) * K + jj]);
        }
      const size_t base = ((size_t)wgx * nq + q0 + tid) * K;
#pragma unroll
      for (int jj = 0; jj < K; ++jj) {
        ws_v[base + jj] = m.v[jj];
        ws_i[base + jj] = m.i[jj];
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Group maxima for many queries: a product with both operands staged in LDS. The stream above reads X again for every 64 queries, in
// its operand layout (16 rows x 64 B a load: 37 KB/us in a CU, a quarter of what whole lines get), and a query fragment from LDS
// for every MFMA. Here:
//  * a workgroup takes 32 * RF rows x 16 * QT queries (up to 320, so X is read once), waves half of the rows x half of the queries:
//    RF + QT / 2 fragment reads for RF * QT / 2 MFMAs of a 32-deep K step;
//  * X and Q come by DMA, RING - 2 steps ahead and on into the workgroup's next tile of rows, the loads spread between the MFMAs; the
//    next step's rows are read meanwhile, query fragments three ahead (one wave per SIMD);
//  * every output is one sum over K in order, the same bits as the stream's and the second pass's;
//  * maxima of 4 rows are stored as the lanes hold them; of 16: of the four row tiles of a lane the transposed lane halves leave group
//    4w + (lane >> 4) in place.
// 300 queries x 250007 rows x 1024: 370 -> 189 us with tiles of 128 rows. The matrix work alone is 105 and everything but the loads 119;
// the loads alone take 178: 28 KB a step at 40 KB/us a CU, 8 of X from HBM and 20 of Q from L2 that share 32 KB of outstanding misses
// (whole lines instead of 16 rows x 64 B a load: 200). Taller tiles load less Q for the same rows, see group_max.
// ------------------------------------------------------------------------------------------------
template <int QT, int RF>
constexpr int tile_ring() { return 158 / (2 * RF + QT) < 8 ? 158 / (2 * RF + QT) : 8; }

template <int QT, int RF, int GR>
__global__ __launch_bounds__(256, 1) void sim_group_max(const bf16* __restrict__ Q, const bf16* __restrict__ X,
                                                        const float* __restrict__ bias, int nq, int N, int D, int qblocks,
                                                        float* __restrict__ gmax, int ngr) {
  constexpr int RING = tile_ring<QT, RF>(), TR = 32 * RF, QH = QT / 2, NX = RF / 2, NL = NX + QT / 4, PART = (2 * RF + QT) * 1024;
  constexpr int NM = RF * QH;
  extern __shared__ __attribute__((aligned(16))) char smem[];  // RING steps of 2 RF X and QT query fragments; two tiles' biases
  float* bsm = reinterpret_cast<float*>(smem + RING * PART);
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wid >> 1, wq = wid & 1;
  const int items = (N + TR - 1) / TR * qblocks, G = gridDim.x, nk = D / 32;
  const int n = (items - (int)blockIdx.x + G - 1) / G;  // this workgroup's items: row tile, query block
  if (n <= 0) return;
  const int lrow = lane >> 2, lcol = ((lane & 3) ^ (lrow >> 2 & 3)) * 16;  // a load: 16 rows x 64 B, pieces swizzled by row
  // prefetch position
  __amdgpu_buffer_rsrc_t rx, rq, rb;
  int ox[4], oq[5], ob;
  int pit = 0, pt = 0;
  auto aim = [&]() {
    const int item = blockIdx.x + pit * G, r0 = item / qblocks * TR, q0 = item % qblocks * (16 * QT);
    rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(X) + (size_t)r0 * D, (short)0, 0x7fffffff, 0x00020000);
    rq = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(Q) + (size_t)q0 * D, (short)0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int q = 0; q < NX; ++q) ox[q] = (min(r0 + (q * 4 + wid) * 16 + lrow, N - 1) - r0) * D * 2 + lcol;
#pragma unroll
    for (int q = 0; q < QT / 4; ++q) oq[q] = (min(q0 + (q * 4 + wid) * 16 + lrow, nq - 1) - q0) * D * 2 + lcol;
    rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(bias) + r0, (short)0, 0x7fffffff, 0x00020000);
    ob = (min(r0 + wid % (RF / 2) * 64 + lane, N - 1) - r0) * 4;
  };
  auto load = [&](int q, int slot) {
    char* d = smem + slot * PART + wid * 1024;
    if (q < NX) __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, GAI_LDS(d + q * 4096), 16, ox[q], pt * 64, 0, 0);
    else __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, GAI_LDS(d + q * 4096), 16, oq[q - NX], pt * 64, 0, 0);
  };
  auto load_bias = [&]() {  // with a tile's first step; an extra load only makes a counted wait stricter
    if (pt == 0 && wid < RF / 2) {
      char* d = reinterpret_cast<char*>(bsm + (pit & 1) * TR + wid * 64);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, GAI_LDS(d), 4, ob, 0, 0, 0);
    }
  };
  auto next = [&]() {  // past the last item its last step is read again: the count of loads stays what the code says
    if (pt + 1 < nk) ++pt;
    else if (pit + 1 < n) {
      ++pit;
      pt = 0;
      aim();
    }
  };
  int rd[2];  // this wave's fragments: + 1024 each (16 rows x 64 B)
  rd[0] = wr * RF * 1024 + (lane & 15) * 64 + (((lane >> 4) ^ ((lane & 15) >> 2)) << 4);
  rd[1] = (2 * RF + wq * QH) * 1024 + (rd[0] - wr * RF * 1024);
  bf16x8 xf[2][RF], qf[4];  // rows of this step and the next; queries in use and the three after
  f32x4 acc[RF][QH];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < RF; ++i)
#pragma unroll
      for (int j = 0; j < QH; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto xfrag = [&](const char* s, int i) { return *reinterpret_cast<const bf16x8*>(s + rd[0] + i * 1024); };
  auto qfrag = [&](const char* s, int j) { return *reinterpret_cast<const bf16x8*>(s + rd[1] + j * 1024); };
  aim();
#pragma unroll
  for (int d = 0; d + 1 < RING; ++d) {
    load_bias();
#pragma unroll
    for (int q = 0; q < NL; ++q) load(q, d);
    __builtin_amdgcn_sched_barrier(0);
    next();
  }
  asm volatile("s_waitcnt vmcnt(%c0)" ::"i"((RING - 2) * NL) : "memory");
  __builtin_amdgcn_s_barrier();
#pragma unroll
  for (int i = 0; i < RF; ++i) xf[0][i] = xfrag(smem, i);
  qf[0] = qfrag(smem, 0);
  qf[1] = qfrag(smem, 1);
  qf[2] = qfrag(smem, 2);
  int slot = 0;
  // first: the register of the step's first query fragment
  auto step = [&](const bf16x8(&cur)[RF], bf16x8(&nxt)[RF], int first) __attribute__((always_inline)) {
    const int ns = slot + 1 == RING ? 0 : slot + 1, fs = slot == 0 ? RING - 1 : slot - 1;
    asm volatile("s_waitcnt vmcnt(%c0)" ::"i"((RING - 3) * NL) : "memory");  // the next step's have landed
    __builtin_amdgcn_s_barrier();  // and every wave is through with the step before this one: its slot is free
    __builtin_amdgcn_sched_barrier(0);
    load_bias();
    const char *s = smem + slot * PART, *s1 = smem + ns * PART;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int j = m / RF, i = m % RF;
      if (i == 0) qf[(first + j + 3) % 4] = j + 3 < QH ? qfrag(s, j + 3) : qfrag(s1, j + 3 - QH);
      if (m >= NM / 2 && m < NM / 2 + RF) nxt[m - NM / 2] = xfrag(s1, m - NM / 2);
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur[i], qf[(first + j) % 4], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = m * NL / NM; q < (m + 1) * NL / NM; ++q) load(q, fs);
      __builtin_amdgcn_sched_barrier(0);
    }
    next();
    slot = ns;
  };
  auto finish = [&](int it) {
    const int item = blockIdx.x + it * G, q0 = item % qblocks * (16 * QT) + wq * QH * 16;
#pragma unroll
    for (int h = 0; h < RF; h += 4) {
      constexpr int kLast = RF % 4 ? RF % 4 : 4;  // row tiles of the last round: two stand twice
      const int rt = h + 4 < RF ? 4 : kLast;
      const int gr0 = item / qblocks * (2 * RF) + wr * RF + h;
      f32x4 bv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bv[i] = *reinterpret_cast<const f32x4*>(bsm + (it & 1) * TR + wr * (16 * RF) + (h + i % rt) * 16 + 4 * (lane >> 4));
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if ((gr0 + i % rt) * 16 + 4 * (lane >> 4) + r >= N) bv[i][r] = -INFINITY;
      }
      const int g = gr0 + (lane >> 4);
#pragma unroll
      for (int j = 0; j < QH; ++j) {
        float m[4];  // fmaxf passes NaN scores over
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const f32x4 v = acc[h + i % rt][j];
          m[i] = fmaxf(fmaxf(fmaxf(-INFINITY, v[0] + bv[i][0]), v[1] + bv[i][1]), fmaxf(fmaxf(-INFINITY, v[2] + bv[i][2]), v[3] + bv[i][3]));
        }
        const auto rg = __builtin_amdgcn_make_buffer_rsrc(gmax + (size_t)(q0 + 16 * j) * ngr, (short)0, 64 * ngr, 0x00020000);
        const bool in = q0 + 16 * j + (lane & 15) < nq;
        // a store past the buffer is dropped: no branch, so the sums leave the accumulators a column tile at a time
        if constexpr (GR == 4) {
#pragma unroll
          for (int i = 0; i < rt; i += 2) {
            const int at = (gr0 + i) / 2 * 8 + (lane >> 4) * 2;
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{__float_as_uint(m[i]), __float_as_uint(m[i + 1])}, rg,
                                                  in && at < ngr ? ((lane & 15) * ngr + at) * 4 : -8, 0, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
          continue;
        }
        // lane groups 0 1 2 3 of m[0] m[1] m[2] m[3]: halves of 0 | 2 and 1 | 3, then quarters of all
        const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(m[0]), __float_as_uint(m[2]), false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(m[1]), __float_as_uint(m[3]), false, false);
        const float u = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1])), v = fmaxf(__uint_as_float(y[0]), __uint_as_float(y[1]));
        const auto z = __builtin_amdgcn_permlane16_swap(__float_as_uint(u), __float_as_uint(v), false, false);
        const int at = in && g < ngr && (lane >> 4) < rt ? ((lane & 15) * ngr + g) * 4 : -4;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(fmaxf(__uint_as_float(z[0]), __uint_as_float(z[1]))), rg, at, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  for (int it = 0; it < n; ++it) {
    clear();
    for (int t = 0; t < nk; t += 2) {  // nk is even
      step(xf[0], xf[1], 0);
      step(xf[1], xf[0], QH % 4);
    }
    finish(it);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS is left
}

// ------------------------------------------------------------------------------------------------
// k > 8, second pass: one workgroup per query. A key is (score, lowest row first) as one unsigned number, 0 = none.
// The k groups with the largest maxima hold the k best rows: a row of another group has at least k rows before it, the
// maxima of those groups. The same argument picks the groups: thread t's strided maximum over the group maxima, the k
// best of those 1024 threads, and of their entries the k best. The rows of the k groups (<= 1024) are scored again with
// the stream's own instruction order and sorted. Bound by the fetch of k groups' rows for every query (1.3 MB at k = 40, 1024 columns and
// 16 rows, for 44 of 300 queries on a CU that has another; a CU alone draws 60 KB/us) and by the latency of the maxima and of three
// selections of 45 exchanges. 300 queries of 250007 rows of 1024, k = 40: 119 us with keys exchanged through LDS and maxima loaded
// one after the other, 98 with exchanges on VALU operands and four loads ahead, 56 with groups of 4 rows (a quarter of the fetch, four
// times the maxima). Whole calls, groups of 16 | 4: 30000 rows, 250 queries, k = 50 87 | 49; 5000 rows, 300, k = 40 77 | 57; 60000, 16,
// k = 50 49 | 42; but 1M, 1, k = 40 386 | 392 and 100000 x 384, 300, k = 10 68 | 72. Rows by DMA in whole lines instead of operand by
// operand: k = 40 156 -> 119 us.
// With at most k groups (an index, or a filter's rows, of 16 k rows) all are taken: no stream, one selection. 300 queries, 60
// rows of 1024, k = 16: 20 us, 89 with the stream and with second groups read for nothing (lists 57); 200 rows, k = 8: 48, 61
// (lists 55).
// ------------------------------------------------------------------------------------------------
typedef unsigned long long u64;

__device__ __forceinline__ u64 make_key(float v, int id) {
  if (!(v > -INFINITY)) return 0;  // deleted, absent or NaN
  const uint32_t u = __float_as_uint(v == 0.f ? 0.f : v);
  return ((u64)(u & 0x80000000u ? ~u : u | 0x80000000u) << 32) | (uint32_t)~id;
}
__device__ __forceinline__ int key_id(u64 k) { return (int)~(uint32_t)k; }
__device__ __forceinline__ float key_value(u64 k) {
  const uint32_t u = (uint32_t)(k >> 32);
  return __uint_as_float(u & 0x80000000u ? u & 0x7fffffffu : ~u);
}

// x of lane ^ D: no LDS round trip
template <int D>
__device__ __forceinline__ uint32_t lane_xor(uint32_t x) {
  if constexpr (D == 1) return __builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, true);
  if constexpr (D == 2) return __builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, true);
  if constexpr (D == 4)  // mirrored in eights (^ 7), then in fours (^ 3)
    return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xF, 0xF, true), 0x1B, 0xF, 0xF, true);
  if constexpr (D == 8) return __builtin_amdgcn_mov_dpp((int)x, 0x128, 0xF, 0xF, true);
  if constexpr (D == 16) {
    const auto y = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return threadIdx.x & 16 ? y[0] : y[1];
  }
  const auto y = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return threadIdx.x & 32 ? y[0] : y[1];
}

// one exchange of a bitonic merge of `size` lanes over distance D
template <int D>
__device__ __forceinline__ u64 merge_step(u64 x, int size) {
  const int lane = threadIdx.x & 63;
  const u64 y = (u64)lane_xor<D>((uint32_t)(x >> 32)) << 32 | lane_xor<D>((uint32_t)x);
  const bool high = ((lane & size) == 0) == ((lane & D) == 0);  // this lane keeps the larger key
  return (x > y) == high ? x : y;
}

// lanes' keys -> descending over the lanes (bitonic); merge64: of keys that rise and then fall, or fall and then rise
__device__ __forceinline__ u64 merge64(u64 x) {
  x = merge_step<32>(x, 64);
  x = merge_step<16>(x, 64);
  x = merge_step<8>(x, 64);
  x = merge_step<4>(x, 64);
  x = merge_step<2>(x, 64);
  return merge_step<1>(x, 64);
}
__device__ __forceinline__ u64 wave_sort(u64 x) {
  x = merge_step<1>(x, 2);
  x = merge_step<2>(x, 4);
  x = merge_step<1>(x, 4);
  x = merge_step<4>(x, 8);
  x = merge_step<2>(x, 8);
  x = merge_step<1>(x, 8);
  x = merge_step<8>(x, 16);
  x = merge_step<4>(x, 16);
  x = merge_step<2>(x, 16);
  x = merge_step<1>(x, 16);
  x = merge_step<16>(x, 32);
  x = merge_step<8>(x, 32);
  x = merge_step<4>(x, 32);
  x = merge_step<2>(x, 32);
  x = merge_step<1>(x, 32);
  return merge64(x);
}

// The 64 largest of the first 64 * waves threads' keys (distinct or 0; waves a power of two), descending, in list[0..63]; buf: 1024
// keys. Each wave sorts its own, then pairs of waves merge: the elementwise maximum of one list and the other reversed holds the 64
// largest.
__device__ __forceinline__ void top64(u64 x, u64* buf, u64* list, int waves) {
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (wid < waves) x = wave_sort(x);
  for (int half = waves / 2; half > 0; half >>= 1) {
    __syncthreads();
    if (wid >= half && wid < 2 * half) buf[tid] = x;
    __syncthreads();
    if (wid < half) {
      const u64 y = buf[(wid + half) * 64 + 63 - lane];
      x = merge64(x > y ? x : y);
    }
  }
  if (wid == 0) list[lane] = x;
  __syncthreads();
}
__device__ __forceinline__ int waves_for(int n) { return n <= 64 ? 1 : n <= 128 ? 2 : n <= 256 ? 4 : n <= 512 ? 8 : 16; }

constexpr int kSelectRows = 16 * 4096;

template <int GR>
__global__ __launch_bounds__(1024) void sim_topk_select(const bf16* __restrict__ Q, const bf16* __restrict__ X,
                                                        const float* __restrict__ bias, const float* __restrict__ gmax,
                                                        int ngr, int N, int D, int k, int dma, float* __restrict__ out_v,
                                                        int64_t* __restrict__ out_i) {
  constexpr int V = GR == 4 ? 4 : 1;  // maxima a load: a query's places begin on 32 bytes where a group is 4 rows
  typedef float fV __attribute__((ext_vector_type(V)));
  extern __shared__ __attribute__((aligned(16))) char smem[];  // 4 KB a wave of rows, the first 8 KB also keys; the query
  u64* buf = reinterpret_cast<u64*>(smem);
  bf16* qrow = reinterpret_cast<bf16*>(smem + kSelectRows);
  __shared__ u64 cand[1024], list[64];
  __shared__ float bsm[1024];
  __shared__ int pick[64], cnt;
  const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  if (dma)
    for (int e = tid; e < D / 8; e += 1024) store8(qrow + 8 * e, load8(Q + (size_t)q * D + 8 * e));
  const float* gm = gmax + (size_t)q * ngr;
  const int per = (ngr + 1024 * V - 1) / (1024 * V);  // loads of a thread: c = tid + 1024 i, places V c .. V c + V - 1
  auto key_of = [&](float v, int p) {
    const int g = place_group<GR>(p);
    return g * GR < N ? make_key(v, g) : 0;
  };
  if (ngr > k) {  // else every group is taken, and gmax was not written
    u64 m = 0;
    for (int i = 0; i < per; i += 4) {
      fV v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = *reinterpret_cast<const fV*>(gm + V * min(tid + 1024 * (i + u), ngr / V - 1));
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int c = tid + 1024 * (i + u);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          const u64 x = c < ngr / V ? key_of(v[u][e], V * c + e) : 0;
          m = x > m ? x : m;
        }
      }
    }
    top64(m, buf, list, 16);
  }
  if (V > 1 ? ngr > k : ngr > 1024) {  // a thread has more than one place
    if (tid < k) {
      const int g = key_id(list[tid]);
      pick[tid] = list[tid] ? group_place<GR>(g) / V & 1023 : -1;
    }
    if (tid == 0) cnt = 0;
    u64 bar = list[k - 1];  // the k-th best thread's maximum: nothing below it can be among the k best groups
    __syncthreads();
    const int all = k * per;
    for (int base = 0; base < all; base += 960) {
      const int e = base + tid;
      int c = -1;
      fV v = {};
      if (tid < 960 && e < all) {
        c = pick[e / per];
        if (c >= 0) c += 1024 * (e % per);
        if (c >= ngr / V) c = -1;
        if (c >= 0) v = *reinterpret_cast<const fV*>(gm + V * c);
      }
#pragma unroll
      for (int u = 0; u < V; ++u) {
        if (c >= 0) {
          const u64 x = key_of(v[u], V * c + u);
          if (x && x >= bar) cand[atomicAdd(&cnt, 1)] = x;  // <= 64 held + 960 of this round
        }
        __syncthreads();
        const int n = cnt;
        __syncthreads();  // every thread has read it before the next round adds to it
        if (n > 64 || (u == V - 1 && base + 960 >= all)) {  // keep the k best
          top64(tid < n ? cand[tid] : 0, buf, list, waves_for(n));
          if (tid < k) cand[tid] = list[tid];
          if (tid == 0) cnt = n < k ? n : k;
          if (n >= k) bar = list[k - 1];
          __syncthreads();
        }
      }
    }
  }
  if (tid < k) pick[tid] = ngr <= k ? (tid < ngr ? tid : -1) : list[tid] ? key_id(list[tid]) : -1;
  __syncthreads();
  cand[tid] = 0;
  if (tid < k * GR) {  // before the rows: a load among theirs would wait for them all
    const int row = GR * pick[tid / GR] + tid % GR;
    bsm[tid] = row >= 0 && row < N ? bias[row] : -INFINITY;
  }
  __syncthreads();
  // group j's scores, this wave's, from the accumulator: every column of the product is this query
  auto keep = [&](int j, const f32x4& acc) {
    const int r = lane & 15, at = (GR == 4 ? 0 : 4 * (lane >> 4)) + r, row = GR * pick[j] + at;
    const float v = r == 0 ? acc[0] : r == 1 ? acc[1] : r == 2 ? acc[2] : acc[3];
    if (r < 4 && at < GR && row < N) cand[GR * j + at] = make_key(v + bsm[GR * j + at], row);
  };
  if (!dma) {  // columns no multiple of 64, or rows off 16 bytes
    const bf16* qp = Q + (size_t)q * D + 8 * (lane >> 4);
    for (int j = wid; j < k && pick[j] >= 0; j += 16) {  // (the picked groups come first)
      const bf16* xa = X + (size_t)min(GR * pick[j] + (lane & (GR - 1)), N - 1) * D + 8 * (lane >> 4);
      f32x4 acc = {};
#pragma unroll 8
      for (int t = 0; t < D / 32; ++t)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load8(xa + 32 * t), load8(qp + 32 * t), acc, 0, 0, 0);
      keep(j, acc);
    }
  } else {
    // rows by DMA in whole lines (16 rows x 64 B a load, as operands lie, come at a quarter of the rate), 4 KB in flight per wave, on
    // into its next group: two pieces of 16 rows x 64 columns, or four of 4 rows x 128 columns (a group of 4 rows is the operand's
    // rows four times over)
    constexpr int PC = GR == 4 ? 128 : 64, NL = GR == 4 ? 1 : 2, SLOTS = 4 / NL;  // columns and loads of a piece
    int mine = 0;
    while (wid + 16 * mine < k && pick[wid + 16 * mine] >= 0) ++mine;
    mine = __builtin_amdgcn_readfirstlane(mine);
    const int nc = (D + PC - 1) / PC, pieces = mine * nc;
    char* own = reinterpret_cast<char*>(buf) + wid * 4096;
    int pj = wid, pc = 0;  // next piece to ask for
    int ox[2];
    __amdgpu_buffer_rsrc_t rx;
    auto aim = [&]() {
      const int r0 = __builtin_amdgcn_readfirstlane(GR * pick[pj]);
      rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(X) + (size_t)r0 * D, (short)0, 0x7fffffff, 0x00020000);
#pragma unroll
      for (int h = 0; h < NL; ++h) {
        const int row = GR == 4 ? lane >> 4 : 8 * h + (lane >> 3);
        ox[h] = (min(r0 + row, N - 1) - r0) * D * 2 + (GR == 4 ? ((lane & 15) ^ (4 * row)) << 4 : ((lane & 7) ^ (row >> 1)) << 4);
      }
    };
    auto ask = [&](int slot) {  // past the last piece it is read again: the count of loads stays what the code says
      char* d = own + slot * (1024 * NL);
#pragma unroll
      for (int h = 0; h < NL; ++h) {
        // (a last piece of 64 columns: its second half, not used, is the first one again)
        const int back = GR == 4 && (pc + 1) * PC > D && ((lane & 15) ^ (4 * (lane >> 4))) >= 8 ? 128 : 0;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, GAI_LDS(d + h * 1024), 16, ox[h] - back, pc * (2 * PC), 0, 0);
      }
      if (pc + 1 < nc) ++pc;
      else if (pj + 16 < wid + 16 * mine) {
        pj += 16;
        pc = 0;
        aim();
      }
    };
    if (mine > 0) {
      aim();
#pragma unroll
      for (int u = 0; u < SLOTS; ++u) ask(u);
      const int r = GR == 4 ? lane & 3 : lane & 15, rd = r * (2 * PC), sw = GR == 4 ? 4 * r : r >> 1, g = lane >> 4;
      int j = wid, c = 0;
      f32x4 acc = {};
      for (int p = 0; p < pieces; ++p) {
        const char* s = own + (p % SLOTS) * (1024 * NL);
        asm volatile("s_waitcnt vmcnt(%c0)" ::"i"((SLOTS - 1) * NL) : "memory");  // the loads of the next pieces are younger
        bf16x8 x[PC / 32], y[PC / 32];
#pragma unroll
        for (int e = 0; e < PC / 32; ++e) {
          x[e] = *reinterpret_cast<const bf16x8*>(s + rd + (((4 * e + g) ^ sw) << 4));
          y[e] = *reinterpret_cast<const bf16x8*>(qrow + min(PC * c + 32 * e, D - 32) + 8 * g);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this piece's slot is free
        __builtin_amdgcn_sched_barrier(0);
        ask(p % SLOTS);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < PC / 32; ++e)
          if (GR != 4 || PC * c + 32 * e < D) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[e], y[e], acc, 0, 0, 0);
        if (++c == nc) {
          keep(j, acc);
          acc = f32x4{0.f, 0.f, 0.f, 0.f};
          c = 0;
          j += 16;
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS is left
    }
  }
  __syncthreads();
  top64(cand[tid], buf, list, waves_for(k * GR));
  if (tid < k) {
    const u64 x = list[tid];
    out_v[(size_t)q * k + tid] = x ? key_value(x) : -INFINITY;
    out_i[(size_t)q * k + tid] = x ? key_id(x) : -1;
  }
}

// stage 2: one 256-thread workgroup per query merges nwg lists of K.
template <int K>
__global__ __launch_bounds__(256) void sim_topk_stage2(const float* __restrict__ ws_v, const int* __restrict__ ws_i,
                                                       int nwg, int nq, int k_out, float* __restrict__ out_v,
                                                       int64_t* __restrict__ out_i) {
  __shared__ float mv[128 * K];
  __shared__ int mi[128 * K];
  const int q = blockIdx.x, tid = threadIdx.x;
  TopK<K> tk;
  tk.init();
  for (int w = tid; w < nwg; w += 256) {
    const size_t base = ((size_t)w * nq + q) * K;
    for (int j = 0; j < K; ++j) {
      const float v = ws_v[base + j];
      if (!(v > tk.v[K - 1])) break;
      tk.insert(v, ws_i[base + j]);
    }
  }
  // tree merge: 256 -> 128 -> ... -> 1
#pragma unroll 1
  for (int half = 128; half >= 1; half >>= 1) {
    if (tid >= half && tid < 2 * half) {
#pragma unroll
      for (int j = 0; j < K; ++j) {
        mv[(tid - half) * K + j] = tk.v[j];
        mi[(tid - half) * K + j] = tk.i[j];
      }
    }
    __syncthreads();
    if (tid < half) {
      for (int j = 0; j < K; ++j) {
        const float v = mv[tid * K + j];
        if (!(v > tk.v[K - 1])) break;
        tk.insert(v, mi[tid * K + j]);
      }
    }
    __syncthreads();
  }
  if (tid == 0) {
#pragma unroll
    for (int j = 0; j < K; ++j)
      if (j < k_out) {
        out_v[(size_t)q * k_out + j] = tk.v[j];
        out_i[(size_t)q * k_out + j] = tk.i[j];
      }
  }
}

template <typename F>
void set_max_lds(F* f, int bytes) {
  hipFuncSetAttribute(reinterpret_cast<const void*>(f), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

struct TopkArgs {
  const void *Q, *X;
  const float* bias;
  int nq, N, D, k, nwg, rows_per_wg, gr;  // gr: rows of a group (no lists)
  float* ws_v;
  int* ws_i;
  float* out_v;
  int64_t* out_i;
  hipStream_t st;
};

template <int QT, int RF, int GR>
void run_group_max(const TopkArgs& a, int qblocks) {
  constexpr int lds = tile_ring<QT, RF>() * (2 * RF + QT) * 1024 + 256 * RF;
  static bool once = false;
  if (!once) {
    set_max_lds(sim_group_max<QT, RF, GR>, lds);
    once = true;
  }
  const int items = (a.N + 32 * RF - 1) / (32 * RF) * qblocks;
  sim_group_max<QT, RF, GR><<<std::min(items, 256), 256, lds, a.st>>>((const bf16*)a.Q, (const bf16*)a.X, a.bias, a.nq, a.N, a.D, qblocks,
                                                              a.ws_v, places(GR, a.N));
  GAI_LAUNCH_CHECK();
}

// an image of the queries of a tile fits LDS beside the bias rows
bool tile_fits(const TopkArgs& a, int nq_tile) { return (size_t)nq_tile * a.D * 2 + (size_t)a.rows_per_wg * 4 <= 160 * 1024; }

bool on16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

template <int GR>
void run_select_r(const TopkArgs& a) {
  static bool once = false;
  if (!once) {
    set_max_lds(sim_topk_select<GR>, 146 * 1024);  // (its own 13 KB are beside)
    once = true;
  }
  const int dma = a.D % 64 == 0 && on16(a.X);  // 16-byte loads into LDS
  sim_topk_select<GR><<<a.nq, 1024, kSelectRows + a.D * 2, a.st>>>((const bf16*)a.Q, (const bf16*)a.X, a.bias, a.ws_v,
                                                                   places(GR, a.N), a.N, a.D, a.k, dma, a.out_v, a.out_i);
  GAI_LAUNCH_CHECK();
}
void run_select(const TopkArgs& a) { a.gr == 4 ? run_select_r<4>(a) : run_select_r<16>(a); }

// Rows of a tile: 128, or more where the last round of tiles over the 256 CUs does not cost what that saves. A tile of 192 rows x 320
// queries takes 1.34 times one of 128 (1M x 1024, 300 queries, k = 4: 815 -> 745 us; 170000, k = 40: 185 -> 173; but 200000 in 5 rounds
// for 7: 209 -> 206, 120000 x 768 in 3 for 4: 89 -> 93), one of 256 x 192 or 256 queries 1.77 times (250007 x 1024, 192 queries:
// 165 -> 150, 256: 191 -> 174; 70000, 250 queries, 2 rounds for 3: 66.7 -> 72.1). 256 rows x 320 queries do not fit the registers;
// up to 128 queries X bounds both.
template <int GR>
void group_max(const TopkArgs& a) {
  const int qblocks = (a.nq + 319) / 320, qt = ((a.nq + qblocks - 1) / qblocks + 63) / 64 * 4;
  auto rounds = [&](int rows) { return ((a.N + rows - 1) / rows * qblocks + 255) / 256; };
  const bool by192 = rounds(192) * 136 < rounds(128) * 100, by256 = rounds(256) * 178 < rounds(128) * 100;
  if (qt <= 8) run_group_max<8, 4, GR>(a, qblocks);
  else if (qt <= 12) by256 ? run_group_max<12, 8, GR>(a, qblocks) : run_group_max<12, 4, GR>(a, qblocks);
  else if (qt <= 16) by256 ? run_group_max<16, 8, GR>(a, qblocks) : run_group_max<16, 4, GR>(a, qblocks);
  else by192 ? run_group_max<20, 6, GR>(a, qblocks) : run_group_max<20, 4, GR>(a, qblocks);
}

bool many_queries(const TopkArgs& a) {
  if (a.nq <= 64 || a.D % 64 || a.D < 256 || (a.N + 15) / 16 <= a.k || !on16(a.Q) || !on16(a.X)) return false;
  a.gr == 4 ? group_max<4>(a) : group_max<16>(a);
  run_select(a);
  return true;
}

template <int MT, int K, int RING>
void run_stream_r(const TopkArgs& a) {
  constexpr int NQ = 16 * MT;
  const size_t lds = std::max((size_t)NQ * a.D * 2 + (size_t)a.rows_per_wg * 4, (size_t)(K > 0 ? NQ * 32 * K * 8 : 0));
  auto k1 = sim_topk_stream<MT, K, RING>;
  static bool once = false;
  if (!once) {
    set_max_lds(k1, 160 * 1024);
    once = true;
  }
  const int qtiles = (a.nq + NQ - 1) / NQ, ngr = places(K == -4 ? 4 : 16, a.N);
  if (K > 0 || ngr > a.k) {  // no group to leave out: no maxima
    k1<<<(a.nwg + 7) / 8 * 8 * qtiles, 512, lds, a.st>>>((const bf16*)a.Q, (const bf16*)a.X, a.bias, a.nq, a.N, a.D, a.rows_per_wg,
                                                         qtiles, a.ws_v, a.ws_i, a.ws_v, ngr);
    GAI_LAUNCH_CHECK();
  }
  if constexpr (K > 0)
    sim_topk_stage2<K><<<a.nq, 256, 0, a.st>>>(a.ws_v, a.ws_i, a.nwg, a.nq, a.k, a.out_v, a.out_i);
  else
    return run_select(a);
  GAI_LAUNCH_CHECK();
}

template <int MT, int K>
void run_stream(const TopkArgs& a) {
  const int nk = a.D / 32;
  // several query tiles: X comes from L2 for most of them, half the ring is enough (300 queries x 1M x 1024: 1355 -> 1314 us)
  if constexpr (K <= 0 && MT == 4)
    if (a.nq > 64 && nk % 8 == 0) return run_stream_r<MT, K, 8>(a);
  if (nk % 16 == 0) return run_stream_r<MT, K, 16>(a);
  if (nk % 8 == 0) return run_stream_r<MT, K, 8>(a);
  if (nk % 4 == 0) return run_stream_r<MT, K, 4>(a);
  return run_stream_r<MT, K, 1>(a);
}

template <int K>
void run_topk_k(const TopkArgs& a) {
  // the largest query tile that fits; 16 queries do (gai_sim_topk)
  if (a.nq > 32 && tile_fits(a, 64)) return run_stream<4, K>(a);
  if (a.nq > 16 && tile_fits(a, 32)) return run_stream<2, K>(a);
  run_stream<1, K>(a);
}

// Relevance of euclidean search, 1 - sqrt(max(|q|^2 - 2 s, 0)) / sqrt(2) of the scores s = q . x - |x|^2 / 2: a wave a query, its row in
// one pass. Bound by its launch (300 queries x 1024, k = 40: 1.2 MB): 2.9 us in a graph; as torch operations it was eight launches, 17.4.
__global__ __launch_bounds__(64) void l2_relevance_kernel(const float* __restrict__ q, const float* __restrict__ s, int D, int k,
                                                          float* __restrict__ out) {
  const int lane = threadIdx.x;
  const float* row = q + (size_t)blockIdx.x * D;
  float sum = 0.f;
#pragma unroll 4
  for (int i = lane; i < D; i += 64) sum += row[i] * row[i];
  const float qq = wave_sum(sum);
  for (int j = lane; j < k; j += 64) {
    float d2 = qq - 2.f * s[(size_t)blockIdx.x * k + j];
    d2 = d2 < 0.f ? 0.f : d2;  // (NaN stays)
    out[(size_t)blockIdx.x * k + j] = 1.f - sqrtf(d2) / 1.41421356f;
  }
}

}  // namespace

// Cross-list merge (the sharded index's W shard lists per query): stage 2 alone over ws [nlists][nq][cap].
void gai_topk_merge(const float* vals, const int* idx, int nlists, int nq, int cap, int k, float* out_v, int64_t* out_i,
                    hipStream_t st) {
  if (nq == 0) return;
  switch (cap) {
    case 4: sim_topk_stage2<4><<<nq, 256, 0, st>>>(vals, idx, nlists, nq, k, out_v, out_i); break;
    case 8: sim_topk_stage2<8><<<nq, 256, 0, st>>>(vals, idx, nlists, nq, k, out_v, out_i); break;
    case 16: sim_topk_stage2<16><<<nq, 256, 0, st>>>(vals, idx, nlists, nq, k, out_v, out_i); break;
    case 32: sim_topk_stage2<32><<<nq, 256, 0, st>>>(vals, idx, nlists, nq, k, out_v, out_i); break;
    case 64: sim_topk_stage2<64><<<nq, 256, 0, st>>>(vals, idx, nlists, nq, k, out_v, out_i); break;
    default: gai_launch_error(__FILE__, __LINE__, "topk_merge: cap must be 4, 8, 16, 32 or 64");
  }
  GAI_LAUNCH_CHECK();
}

int gai_topk_places(int group_rows, int N) { return places(group_rows, N); }

int gai_topk_cap(int k) { return k <= 4 ? 4 : k <= 8 ? 8 : k <= 16 ? 16 : k <= 32 ? 32 : 64; }

void gai_l2_relevance(const float* q, const float* s, int nq, int D, int k, float* out, hipStream_t st) {
  if (nq == 0 || k == 0) return;
  l2_relevance_kernel<<<nq, 64, 0, st>>>(q, s, D, k, out);
  GAI_LAUNCH_CHECK();
}

void gai_sim_topk(const void* Q, const void* X, const float* bias, int nq, int N, int D, int k, float* ws_v,
                  int* ws_i, int nwg, int rows_per_wg, int group_rows, float* out_v, int64_t* out_i, hipStream_t st) {
  if (nq == 0) return;
  if (D % 32) gai_launch_error(__FILE__, __LINE__, "sim_topk: D must be a multiple of 32");
  const TopkArgs a{Q, X, bias, nq, N, D, k, nwg, rows_per_wg, group_rows, ws_v, ws_i, out_v, out_i, st};
  // (the tiled product holds no such image, but what it takes must not depend on the number of queries)
  if (!tile_fits(a, 16)) gai_launch_error(__FILE__, __LINE__, "sim_topk: dimension too large for the LDS query tile");
  if (!ws_i) {  // ws_v: the group maxima [nq][gai_topk_places]
    if (group_rows != 4 && group_rows != 16) gai_launch_error(__FILE__, __LINE__, "sim_topk: groups of 4 or 16 rows");
    if (!many_queries(a)) group_rows == 4 ? run_topk_k<-4>(a) : run_topk_k<0>(a);
    return;
  }
  switch (gai_topk_cap(k)) {
    case 4: return run_topk_k<4>(a);
    case 8: return run_topk_k<8>(a);
    default: gai_launch_error(__FILE__, __LINE__, "sim_topk: lists of more than 8 take the group form");
  }
}
