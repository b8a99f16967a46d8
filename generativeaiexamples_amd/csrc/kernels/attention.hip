// Paged flash attention for gfx950.
//
// KV cache layout (written by rope_kv.hip): K [num_blocks, Hkv, 16, D],
// V^T [num_blocks, Hkv, D, 16] (16 tokens per page).
//
// attn_prefill: varlen, causal or bidirectional, GQA. Workgroup = 4 waves; each
// wave owns 32 query rows of one q-head, the workgroup shares 64-key K / V^T tiles
// in LDS (register-staged, issue-early / write-late: K then V^T through one register set,
// one barrier per tile, row-padded images). S^T = K.Q^T on v_mfma_f32_32x32x16_bf16 puts a full query row
// in one lane (swapped QK^T), so the online softmax is in-register; P^T is fed to
// the P.V MFMA straight from the S accumulator (k-order permuted on the V side,
// cdna_hip_programming §3 "accumulator tile as the next MFMA's operand"). exp2
// domain, fp32 statistics. Used for LLM prefill (incl. chunked prefill over a
// cached prefix) and for encoder self-attention (bidirectional, varlen).
//
// attn_decode: one query token per sequence, split-KV flash-decoding. Workgroup =
// (split, kv head, sequence); the GQA group (<= 16 q heads) is the 16-wide MFMA
// column, so K and V^T are read once per kv head with 16-B / 8-B loads straight to
// VGPRs (memory-bound decode row of the glds-vs-register table); the 4 waves
// combine through LDS, splits are merged by attn_decode_reduce.
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <unordered_map>

#include "gai_common.h"
#include "gai_rope.h"
#include "gai_kernels.h"

using namespace gai;

namespace {

constexpr int kBS = 16;
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNeg = -1e30f;
constexpr float kRescaleTh = 8.f;  // deferred running-max update of the prefill softmax (log2 domain)

// Raw v_exp_f32 (2^x). exp2f wraps it in a denormal range fix-up (cmp, 2x cndmask, add, ldexp: 6 VALU
// ops per element); softmax arguments are <= 0, and results below 2^-126 are irrelevant next to the
// row maximum's 1.0, so the bare instruction is exact enough and 6x cheaper on the VALU.
__device__ __forceinline__ float fexp2(float x) { return __builtin_amdgcn_exp2f(x); }

// max / sum of lane l and lane l ^ 32 in every lane: one v_permlane32_swap (lanes 32-63 of the first operand <->
// lanes 0-31 of the second) instead of a ds_bpermute round trip through the LDS unit
__device__ __forceinline__ float max_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_halves(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// ----------------------------------------------------------------------------------------------
// Prefill
// ----------------------------------------------------------------------------------------------
// LDS images are padded by 16 B per row instead of XOR-swizzled: the 16 rows one ds_read_b128 lane group
// reads at the same column then fall on 16 distinct 4-bank slots (row strides of 4 mod 64 or 36 mod 64
// banks), and every fragment address is one per-lane base plus a compile-time offset (no per-read
// address VALU in the loop).
template <int D>
struct PrefillCfg {
  static constexpr int KT = 64;                  // keys per tile
  static constexpr int KRS = D * 2 + 16;         // K image row stride (bytes)
  static constexpr int VRS = KT * 2 + 16;        // V^T image row stride (bytes)
  static constexpr int KBYTES = KT * KRS;        // K tile image
  static constexpr int VBYTES = D * VRS;         // V^T tile image
  static constexpr int BUF = KBYTES + VBYTES;
  static constexpr int CH = D / 32;              // 16-B chunks per thread per operand
  static constexpr int KU = D / 8;               // 16-B units per K row
};

// K image: row = key, 16-B unit u at 16u
template <int D>
__device__ __forceinline__ int k_lds_off(int key, int u) {
  return key * PrefillCfg<D>::KRS + (u << 4);
}
// V^T image: row = d (64 keys) of 8-B units u (4 keys each). Unit u = 4st + 2b1 + b0 is stored at position
// 4st + 2b0 + b1, so the two units one P.V MFMA operand takes (u = 4st + h and 4st + 2 + h) are one
// aligned 16-B pair read by a single ds_read_b128 (no register shuffles).
template <int D>
__device__ __forceinline__ int v_lds_off(int d, int u) {
  const int p = (u & ~3) | ((u & 1) << 1) | ((u >> 1) & 1);
  return d * PrefillCfg<D>::VRS + (p << 3);
}

// 16 (bf16 cache) or 8 (fp8 cache) bytes at base + off through a buffer resource built from the wave-uniform
// page base: the load's only VGPR operand is the loop-invariant lane offset, so no per-tile 64-bit address
// registers exist for the compiler to recycle (and then wait on) while the load is in flight.
template <typename T>
__device__ __forceinline__ T buf_load(const void* base, unsigned off) {
  __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, 0x7fffffff, 0x00020000);
  if constexpr (sizeof(T) == 16) {
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  } else {
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
  }
}

__device__ __forceinline__ bf16x8 kv_to_bf16(bf16x8 v, float) { return v; }
__device__ __forceinline__ bf16x8 kv_to_bf16(uint2 v, float s) { return fp8x8_to_bf16(v, s); }

// KV = bf16 or fp8 (OCP e4m3fn cache, dequantised by the per-layer scale when the tile is written to LDS)
// HL = q heads per wave (1 or 2, same 32 query rows): with 2, every K / V^T fragment a wave reads from LDS feeds two
// MFMAs, halving the LDS read traffic per FLOP (with one head per wave the fragment reads + tile writes, ~2.5K LDS
// cycles per CU per 64-key tile, exceed the ~2K MFMA cycles per SIMD); twice the registers, so one wave per SIMD.
// PIPE (HL == 1): software-pipelined main loop - tile kt+1's QK^T MFMAs are issued interleaved with tile kt's softmax
// exponentials and P.V MFMAs, so the matrix pipe has independent work while the VALU runs the softmax (the one-tile
// loop serialised them: 36.5 % MFMA busy, 7.5 VALU per MFMA, profiles/r5 section 10). K runs one tile ahead of V in
// LDS; the next K and V tiles are staged in two register sets during the iteration.
// NWV = waves per workgroup: 4 (two workgroups per CU) or 8 (one; the row groups of two 4-wave workgroups share each
// staged K / V^T tile, halving the tile loads and LDS writes per FLOP; head_dim 64 / 128, one head per wave)
// ROWS: keys and values straight from the packed rows that q is in (self-attention of an encoder; kc / vc = the first row's key /
// value of head 0, q_ld apart), instead of from pages that a kernel before has packed: 61 passages of e5-large 25 + 66 -> 62 us a
// layer, a question 4.2 + 5.4 -> 5.3. V is turned on its way into LDS: a thread fetches two dims of eight keys, 4 B each
// (whole lines across the wave), and writes two rows of the V^T image. head_dim 64, a kv head per q head. 2: in 128 registers.
// HALF: a workgroup takes one of the two 32-row halves of a tile of the list (few tiles: see prefill_launch)
template <int D, int HPW, typename KV, int HL = 1, bool PIPE = false, int NWV = 4, int ROWS = 0, bool HALF = false>
__global__ __launch_bounds__(64 * NWV, (D > 128 || HL > 1 || NWV == 8) ? 1 : ROWS == 2 ? 4 : 2) void attn_prefill_kernel(
    const bf16* __restrict__ q, const KV* __restrict__ kc, const KV* __restrict__ vc,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ tiles,
    const int* __restrict__ cu_q, const int* __restrict__ ctx_lens, bf16* __restrict__ out, int Hq, int Hkv,
    float scale, int causal, float* __restrict__ lse, float k_scale, float v_scale, int xcd, int q_ld) {
  using Cfg = PrefillCfg<D>;
  static_assert(HL == 1 || HPW % HL == 0, "a wave's heads come from one workgroup head group");
  constexpr int WPR = HPW / HL;  // waves per row group
  constexpr int RPW = NWV / WPR;  // row groups per workgroup
  constexpr int NTH = 64 * NWV;   // threads
  static_assert(NWV == 4 || (NWV == 8 && HL == 1 && !PIPE && (D == 64 || D == 128)), "8-wave workgroups: D 64 / 128");
  constexpr int CH = Cfg::CH * 4 / NWV;  // 16-B staging pieces per thread per tile half
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, h = lane >> 5;
  // xcd: head group = linear workgroup id mod gridDim.y. Workgroups go to the 8 XCDs round-robin by linear id, so
  // with 8 (or a multiple of 8) head groups every XCD serves one kv head (or two): the q tiles running together
  // on it re-read that head's K/V prefixes from the XCD's own L2 instead of all heads' prefixes streaming through
  // every XCD. MI355X (profiles/r3/attn_prefill_xcd): B 4 x S 2048 GQA 32/8 D 128 604 -> 660 TF/s, the headline
  // chunk (7 x 2406) 703 -> 728, Gemma D 256 315 -> 473; 64 x 512 MHA D 64 413 -> 394. GAI_ATTN_XCD=0: off.
  // xcd bits 1-2: wave priority around the MFMA phases (A/B, GAI_ATTN_PRIO): 1 = QK^T at priority 1, 2 = QK^T and P.V
  // xcd bit 3: exact running maximum (GAI_ATTN_RESCALE_TH=0). Otherwise the running maximum only moves when a tile
  // raises it by more than kRescaleTh (log2 units): probabilities then stay <= 2^kRescaleTh (bf16 / fp32 keep their
  // relative precision) and the O / l rescale almost never runs after the first tiles
  const float th = (xcd & 8) ? 0.f : kRescaleTh;
  const int xcd_flags = xcd;
  const int prio = (xcd >> 1) & 3;
  xcd &= 1;
  int bx = blockIdx.x, by = blockIdx.y;
  if (xcd) {
    const int L = blockIdx.y * gridDim.x + blockIdx.x;
    bx = L / gridDim.y;
    by = L % gridDim.y;
  }
  static_assert(!HALF || RPW == 1, "half tiles: one row group a workgroup");
  const int tb = HALF ? bx >> 1 : bx;
  const int seq = tiles[2 * tb], qs = tiles[2 * tb + 1] + (HALF ? 32 * (bx & 1) : 0);
  const int qbeg = cu_q[seq], qlen = cu_q[seq + 1] - qbeg;
  if (HALF && qs >= qlen) return;
  const int ctx = ROWS ? min(ctx_lens[seq], qlen) : ctx_lens[seq];
  static_assert(!ROWS || (D == 64 && HPW == 1 && HL == 1 && !PIPE && NWV == 4 && sizeof(KV) == 2), "rows: encoder heads of 64");
  const int head = by * HPW + HL * (wid % WPR);  // first of this wave's HL heads
  const int g = (by * HPW) / (Hq / Hkv);
  const int r0 = qs + 32 * (wid / WPR);  // first q row (within the sequence) of this wave
  const int qrow = r0 + (lane & 31);
  const int qpos = ctx - qlen + qrow;  // absolute position of this lane's query
  const int klim = (causal ? min(ctx, qpos + 1) : ctx) - 4 * h;  // keys below it (+ 4 h) are seen
  const int* bt = block_tables + (size_t)seq * max_blocks;

  // rows covered by the whole workgroup -> number of key tiles
  const int last_row = min(qs + 32 * RPW, qlen) - 1;
  const int kmax = causal ? (ctx - qlen + last_row + 1) : ctx;
  const int ntiles = (kmax + Cfg::KT - 1) / Cfg::KT;

  // Q fragments (B operand of S^T = K.Q^T): lane (q = lane&31, h) holds Q[q][16t + 8h .. +7]
  // HL == 1: the Q fragments live in registers. HL == 2: in this wave's LDS region (padded rows like the K image),
  // read once per tile per (head, k-step) - two heads' fragments in registers spill.
  constexpr int QL = HL == 1 ? 1 : 0;  // heads whose fragments stay in registers
  bf16x8 qf[QL ? HL : 1][D / 16];
  char* sq = smem + 2 * Cfg::BUF + wid * (HL * 32 * Cfg::KRS);
#pragma unroll
  for (int j = 0; j < HL; ++j) {
    // q rows are q_ld elements apart: Hq * D for a q tensor of its own, the packed QKV row for encoders
    const bf16* qp = q + (size_t)(qbeg + min(qrow, qlen - 1)) * q_ld + (size_t)(head + j) * D + 8 * h;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
      const bf16x8 v = load8(qp + 16 * t);
      if constexpr (QL) qf[j][t] = v;
      else *reinterpret_cast<bf16x8*>(sq + (j * 32 + (lane & 31)) * Cfg::KRS + ((2 * t + h) << 4)) = v;
    }
  }

  // One set of staging registers (raw cache bytes: the fp8 conversion happens at the LDS write), used
  // twice per tile: the next tile's K is loaded at the top and written to the free buffer after QK^T,
  // then its V^T is loaded into the same registers and written before the barrier.
  // Piece c of thread tid (16 B of a tile half) lies in page (c*NTH + tid) / 2D of the tile, which is
  // wave-uniform (a wave's 64 pieces never straddle a page): the page's physical block is looked up with a
  // scalar load one tile ahead (nblk), and each load is a buffer load from that block's scalar base at a
  // loop-invariant 32-bit per-lane offset (no per-lane block-table round trip or 64-bit address math in the loop).
  using Stage = typename std::conditional<sizeof(KV) == 1, uint2, bf16x8>::type;
  Stage stg[CH];
  const int wid_u = __builtin_amdgcn_readfirstlane(wid);
  unsigned voff[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) voff[c] = (unsigned)(((c * NTH + tid) % (2 * D)) * 8 * sizeof(KV));
  int nblk[CH];
  auto lookup_into = [&](int kt, int(&nb)[CH]) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int pidx = kt * 4 + (c * NTH + wid_u * 64) / (2 * D);
      nb[c] = bt[pidx * kBS < ctx ? pidx : 0];
    }
  };
  auto lookup = [&](int kt) { lookup_into(kt, nblk); };
  auto load_half_from = [&](const KV* base, const int(&nb)[CH], Stage(&dst)[CH]) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      // K page is [16][D] contiguous, V^T page [D][16]
      dst[c] = buf_load<Stage>(base + ((size_t)nb[c] * Hkv + g) * (kBS * D), voff[c]);
    }
  };
  auto load_half = [&](const KV* base) { load_half_from(base, nblk, stg); };
  auto write_k_from = [&](int buf, const Stage(&src)[CH]) {
    char* sk = smem + buf * Cfg::BUF;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int id = c * NTH + tid;
      const int page = id / (2 * D), w = id % (2 * D);
      const int key = page * 16 + w / Cfg::KU, u = w % Cfg::KU;
      *reinterpret_cast<bf16x8*>(sk + k_lds_off<D>(key, u)) = kv_to_bf16(src[c], k_scale);
    }
  };
  auto write_v_from = [&](int buf, const Stage(&src)[CH]) {
    char* sv = smem + buf * Cfg::BUF + Cfg::KBYTES;
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int id = c * NTH + tid;
      const int page = id / (2 * D), w = id % (2 * D);
      const int d = w >> 1, half = w & 1;
      const int u8 = 4 * page + 2 * half;
      typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
      const bf16x8 vv = kv_to_bf16(src[c], v_scale);
      const bf16x4_t lo = {vv[0], vv[1], vv[2], vv[3]};
      const bf16x4_t hi = {vv[4], vv[5], vv[6], vv[7]};
      *reinterpret_cast<bf16x4_t*>(sv + v_lds_off<D>(d, u8)) = lo;
      *reinterpret_cast<bf16x4_t*>(sv + v_lds_off<D>(d, u8 + 1)) = hi;
    }
  };
  auto write_k = [&](int buf) { write_k_from(buf, stg); };
  auto write_v = [&](int buf) { write_v_from(buf, stg); };
  // ROWS: tile kt's rows, from a buffer that begins at its first one and ends with the context: beyond it zeros (masked), and a
  // lane's offsets are the same for every tile. Clamped rows took ten multiplications at a quarter of the rate and twenty more
  // instructions of a tile's 240: those 61 passages 68.9 -> 66.2 us, one of 32 tokens 4.13 -> 3.82
  const bf16 *rk = reinterpret_cast<const bf16*>(kc) + (size_t)qbeg * q_ld + g * D,
             *rv = reinterpret_cast<const bf16*>(vc) + (size_t)qbeg * q_ld + g * D;
  auto rows_at = [&](const bf16* p, int kt) {
    const int left = ctx - 64 * kt;  // > 0: tiles that are asked for
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(p) + (size_t)(64 * kt) * q_ld, (short)0, ((left - 1) * q_ld + D) * 2,
                                             0x00020000);
  };
  const int ork = (tid / 8 * q_ld + tid % 8 * 8) * 2, orv = (8 * (tid >> 5) * q_ld + 2 * (tid & 31)) * 2;
  auto rows_k = [&](int kt, bf16x8(&dst)[2]) {
    const __amdgpu_buffer_rsrc_t r = rows_at(rk, kt);
    int o = ork;
    if constexpr (ROWS == 2) asm volatile("" : "+v"(o));  // addresses made anew for each tile, not kept: eight registers
#pragma unroll
    for (int c = 0; c < 2; ++c) dst[c] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, o + c * NTH / 8 * q_ld * 2, 0, 0));
  };
  auto rows_v = [&](int kt, bf16x8(&dst)[2]) {
    const __amdgpu_buffer_rsrc_t r = rows_at(rv, kt);
    int o = orv;
    if constexpr (ROWS == 2) asm volatile("" : "+v"(o));
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const unsigned x = __builtin_amdgcn_raw_buffer_load_b32(r, o + e * q_ld * 2, 0, 0);
      const bf16x2 y = __builtin_bit_cast(bf16x2, x);
      dst[e >> 2][2 * (e & 3)] = y[0];
      dst[e >> 2][2 * (e & 3) + 1] = y[1];
    }
  };
  auto write_rows_k = [&](int buf, const bf16x8(&src)[2]) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int id = c * NTH + tid;
      *reinterpret_cast<bf16x8*>(smem + buf * Cfg::BUF + k_lds_off<D>(id / 8, id % 8)) = src[c];
    }
  };
  auto write_rows_v = [&](int buf, const bf16x8(&src)[2]) {
    char* sv = smem + buf * Cfg::BUF + Cfg::KBYTES;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x4 x = {src[i][p], src[i][2 + p], src[i][4 + p], src[i][6 + p]};
        *reinterpret_cast<bf16x4*>(sv + v_lds_off<D>(2 * (tid & 31) + p, 2 * (tid >> 5) + i)) = x;
      }
  };

  f32x16 acc_o[HL][D / 32];
  float m_run[HL], l_run[HL];
#pragma unroll
  for (int j = 0; j < HL; ++j) {
#pragma unroll
    for (int i = 0; i < D / 32; ++i) acc_o[j][i] = f32x16{};
    m_run[j] = kNeg;
    l_run[j] = 0.f;
  }
  const float sl2 = scale * kLog2e;

  if constexpr (PIPE) {
    static_assert(HL == 1, "the pipelined loop keeps one head per wave");
    // K(kt + 1) and V(kt) are in LDS at iteration kt: K in slot (kt + 1) & 1, V in slot kt & 1 (each slot = K image,
    // V^T image). During the iteration V(kt + 1) and K(kt + 2) stream into two register sets; after the MFMAs they
    // are written to V slot (kt + 1) & 1 (last read by P.V(kt - 1)) and K slot kt & 1 (last read by QK^T(kt), which ran
    // in iteration kt - 1); one barrier per iteration.
    Stage stv[CH];
    int nb_v[CH], nb_k[CH];
    auto qk_part = [&](int kslot, int sub, int t0, int nt, f32x16& acc) {
      const char* skk = smem + kslot * Cfg::BUF;
      const int key = 32 * sub + (lane & 31);
#pragma unroll
      for (int t = t0; t < t0 + nt; ++t) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(skk + k_lds_off<D>(key, 2 * t + h));
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[0][t], acc, 0, 0, 0);
      }
    };
    f32x16 sc[2], sn[2];
    if (ntiles > 0) {
      lookup_into(0, nblk);
      load_half_from(kc, nblk, stg);
      write_k_from(0, stg);
      load_half_from(vc, nblk, stg);
      write_v_from(0, stg);
      if (ntiles > 1) {
        lookup_into(1, nb_v);
        load_half_from(kc, nb_v, stg);
        write_k_from(1, stg);
      }
      lookup_into(2, nb_k);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the Q fragments and the prologue tiles
    __syncthreads();
    sc[0] = f32x16{};
    sc[1] = f32x16{};
    if (ntiles > 0) {
      qk_part(0, 0, 0, D / 16, sc[0]);
      qk_part(0, 1, 0, D / 16, sc[1]);
    }
    __syncthreads();  // every wave has read K(0) before iteration 0 overwrites K slot 0 with K(2)
    for (int kt = 0; kt < ntiles; ++kt) {
      const bool more1 = kt + 1 < ntiles, more2 = kt + 2 < ntiles;
      if (more1) load_half_from(vc, nb_v, stv);  // V(kt + 1)
      if (more2) load_half_from(kc, nb_k, stg);  // K(kt + 2)
      // ---- softmax statistics of tile kt (as the one-tile loop)
      float mt = kNeg;
      const int kend = kt * 64 + 63;
      if (kend < ctx && (!causal || kend <= ctx - qlen + r0)) {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r = 0; r < 16; ++r) mt = fmaxf(mt, sc[sub][r]);
      } else {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const bool ok = 32 * sub + (r & 3) + 8 * (r >> 2) < klim - kt * 64;
            const float x = ok ? sc[sub][r] : kNeg;
            sc[sub][r] = x;
            mt = fmaxf(mt, x);
          }
      }
      mt = max_halves(mt) * sl2;
      const float m_new = mt > m_run[0] + th ? mt : m_run[0];
      const float alpha = fexp2(m_run[0] - m_new);
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int i = 0; i < D / 32; ++i) acc_o[0][i] *= alpha;
      }
      m_run[0] = m_new;
      // ---- tile kt+1's QK^T interleaved with tile kt's exponentials and P.V: per 8-key step, D / 32 QK^T MFMAs
      // (independent of this tile's softmax) beside the step's 8 exps and its D / 32 P.V MFMAs
      sn[0] = f32x16{};
      sn[1] = f32x16{};
      const char* sv = smem + (kt & 1) * Cfg::BUF + Cfg::KBYTES;
      const int kslot = (kt + 1) & 1;
      float rs = 0.f;
      if (prio == 2) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        if (more1) qk_part(kslot, st >> 1, (st & 1) * (D / 32), D / 32, sn[st >> 1]);
        const int sub = st >> 1, sp = st & 1;
        bf16x8 pf;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float pv = fexp2(fmaf(sc[sub][8 * sp + e], sl2, -m_new));
          rs += pv;
          pf[e] = (bf16)pv;
        }
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) {
          const bf16x8 vf = *reinterpret_cast<const bf16x8*>(sv + v_lds_off<D>(32 * dt + (lane & 31), 4 * st + h));
          acc_o[0][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, acc_o[0][dt], 0, 0, 0);
        }
      }
      if (prio == 2) __builtin_amdgcn_s_setprio(0);
      l_run[0] = l_run[0] * alpha + rs;  // this lane half's keys; the halves are summed after the loop
      if (more2) write_k_from(kt & 1, stg);
      if (more1) write_v_from((kt + 1) & 1, stv);
#pragma unroll
      for (int c = 0; c < CH; ++c) nb_v[c] = nb_k[c];
      lookup_into(kt + 3, nb_k);  // pages past the context resolve to entry 0 (never read unmasked)
      __syncthreads();
      sc[0] = sn[0];
      sc[1] = sn[1];
    }
  } else if constexpr (NWV == 8) {
    // Staggered 8-wave loop (MI355X_MICROARCH "Two waves per SIMD", item 9): waves 4-7 (the second row group, each
    // the SIMD partner of wave w - 4) run half an iteration behind - their P.V of tile kt - 1, then their QK^T of tile
    // kt - so on every SIMD one wave's QK^T MFMAs meet the other's softmax VALU and P.V instead of both waves hitting
    // the matrix pipe, then the VALU, together. Tile j lives in LDS slot j % 3 (3 x 35 KiB): in iteration kt the
    // waves read slots kt % 3 and (kt - 1) % 3 while tile kt + 1 is written to the third; ntiles + 1 iterations, one
    // barrier each. The K / V^T of tile kt + 1 are loaded at the top of iteration kt and written at its end.
    const bool late = wid >= 4 && !(xcd_flags & 16);  // GAI_ATTN_STAGGER=0: every wave in step (A/B)
    Stage stv[CH];
    auto slot = [&](int t) { return smem + (t % 3) * Cfg::BUF; };
    auto qk = [&](const char* sk, f32x16(&sc)[2]) {
      constexpr int NT = D / 16;
      bf16x8 ka[NT], kb[NT];
      const int key = lane & 31;
      sc[0] = f32x16{};
      sc[1] = f32x16{};
#pragma unroll
      for (int t = 0; t < NT; ++t) ka[t] = *reinterpret_cast<const bf16x8*>(sk + k_lds_off<D>(key, 2 * t + h));
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        kb[t] = *reinterpret_cast<const bf16x8*>(sk + k_lds_off<D>(32 + key, 2 * t + h));
        sc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[t], qf[0][t], sc[0], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) sc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kb[t], qf[0][t], sc[1], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, NT, 0);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
    };
    // masked row max, deferred running max, O and l rescaled at once (l += the tile's sum after its P.V)
    auto stats = [&](int kt, f32x16(&sc)[2]) {
      float mt = kNeg;
      const int kend = kt * 64 + 63;
      if (kend < ctx && (!causal || kend <= ctx - qlen + r0)) {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r = 0; r < 16; ++r) mt = fmaxf(mt, sc[sub][r]);
      } else {
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const bool ok = 32 * sub + (r & 3) + 8 * (r >> 2) < klim - kt * 64;
            const float x = ok ? sc[sub][r] : kNeg;
            sc[sub][r] = x;
            mt = fmaxf(mt, x);
          }
      }
      mt = max_halves(mt) * sl2;
      const float m_new = mt > m_run[0] + th ? mt : m_run[0];
      const float alpha = fexp2(m_run[0] - m_new);
      if (__any(alpha != 1.f)) {
#pragma unroll
        for (int i = 0; i < D / 32; ++i) acc_o[0][i] *= alpha;
      }
      l_run[0] *= alpha;
      m_run[0] = m_new;
    };
    auto pv = [&](const char* sv, const f32x16(&sc)[2]) {
      float rs = 0.f;
      if (prio == 2) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const int sub = st >> 1, sp = st & 1;
        bf16x8 pf;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p = fexp2(fmaf(sc[sub][8 * sp + e], sl2, -m_run[0]));
          rs += p;
          pf[e] = (bf16)p;
        }
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt) {
          const bf16x8 vf = *reinterpret_cast<const bf16x8*>(sv + v_lds_off<D>(32 * dt + (lane & 31), 4 * st + h));
          acc_o[0][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, acc_o[0][dt], 0, 0, 0);
        }
      }
      if (prio == 2) __builtin_amdgcn_s_setprio(0);
      l_run[0] += rs;  // per lane half (summed after the loop)
    };
    if (ntiles > 0) {
      lookup(0);
      load_half(kc);
      write_k(0);
      load_half(vc);
      write_v(0);
      lookup(1);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the Q fragments and tile 0
    __syncthreads();
    f32x16 sc[2];
    for (int kt = 0; kt <= ntiles; ++kt) {
      const bool more = kt + 1 < ntiles;
      if (more) {
        load_half(kc);
        load_half_from(vc, nblk, stv);
      }
      if (!late) {
        if (kt < ntiles) {
          if (prio) __builtin_amdgcn_s_setprio(1);
          qk(slot(kt), sc);
          if (prio) __builtin_amdgcn_s_setprio(0);
          stats(kt, sc);
          pv(slot(kt) + Cfg::KBYTES, sc);
        }
      } else {
        if (kt > 0) pv(slot(kt - 1) + Cfg::KBYTES, sc);  // tile kt - 1 (its statistics ran last iteration)
        if (kt < ntiles) {
          if (prio) __builtin_amdgcn_s_setprio(1);
          qk(slot(kt), sc);
          if (prio) __builtin_amdgcn_s_setprio(0);
          stats(kt, sc);
        }
      }
      lookup(kt + 2);  // after the LDS reads (an SMEM load in flight forces full lgkmcnt waits)
      if (more) {
        write_k_from((kt + 1) % 3, stg);
        write_v_from((kt + 1) % 3, stv);
      }
      __syncthreads();
    }
  } else {
  // K and V^T of the next tile staged through two register sets, both written at the end of the iteration (D <= 128,
  // one head per wave: +16 VGPRs)
  constexpr bool ESPLIT = HL == 1 && D <= 128;
  if (ntiles > 0) {
    if constexpr (ROWS) {
      Stage first[CH];
      rows_k(0, stg);
      rows_v(0, first);
      write_rows_k(0, stg);
      write_rows_v(0, first);
    } else {
      lookup(0);
      load_half(kc);
      write_k(0);
      load_half(vc);
      write_v(0);
      lookup(1);
    }
  }
  // Q fragments landed: without this wait the ntiles == 0 path reaches the loop header with the Q loads
  // pending, and hipcc's waitcnt pass then keeps vmcnt(7..0) in front of every tile's QK^T MFMAs, which
  // (counters are in order) waits for the next tile's K loads issued just above them.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  for (int kt = 0; kt < ntiles; ++kt) {
    const int cur = kt & 1;
    const bool more = kt + 1 < ntiles;
    // tile kt + 1: K and V^T both loaded here and written at the end of the iteration (a whole iteration of load
    // latency cover; writing K right after QK^T left the K loads only the QK^T MFMAs to land in)
    Stage stv[ESPLIT ? CH : 1];
    if (more) {
      if constexpr (ROWS) {
        rows_k(kt + 1, stg);
        rows_v(kt + 1, stv);
      } else {
        load_half(kc);
        if constexpr (ESPLIT) load_half_from(vc, nblk, stv);
      }
    }
    const char* sk = smem + cur * Cfg::BUF;
    const char* sv = sk + Cfg::KBYTES;

    // S^T[key][q] for two 32-key halves (each K fragment feeds the wave's HL heads)
    if (prio) __builtin_amdgcn_s_setprio(1);
    f32x16 s[HL][2];
#pragma unroll
    for (int sub = 0; sub < 2; ++sub)
#pragma unroll
      for (int j = 0; j < HL; ++j) s[j][sub] = f32x16{};
    if constexpr (QL && D <= 128 && ROWS != 2) {
      // The first 32-key half's D / 16 K fragments are read together, the second half's one per first-half MFMA:
      // no MFMA waits on its own LDS round trip (left to the compiler, one fragment register was re-used and
      // every QK^T MFMA waited lgkmcnt(0) behind its read)
      constexpr int NT = D / 16;
      bf16x8 ka[NT], kb[NT];
      const int key = lane & 31;
#pragma unroll
      for (int t = 0; t < NT; ++t) ka[t] = *reinterpret_cast<const bf16x8*>(sk + k_lds_off<D>(key, 2 * t + h));
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        kb[t] = *reinterpret_cast<const bf16x8*>(sk + k_lds_off<D>(32 + key, 2 * t + h));
        s[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[t], qf[0][t], s[0][0], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) s[0][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kb[t], qf[0][t], s[0][1], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, NT, 0);  // DS reads: first half
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one second-half read
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one first-half MFMA
      }
      __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);  // second-half MFMAs
    } else if constexpr (QL) {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub) {
        const int key = 32 * sub + (lane & 31);
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(sk + k_lds_off<D>(key, 2 * t + h));
#pragma unroll
          for (int j = 0; j < HL; ++j) s[j][sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[j][t], s[j][sub], 0, 0, 0);
        }
      }
    }
    if constexpr (!QL) {  // k-step outer: each K fragment (both halves) and each Q fragment read once per tile
#pragma unroll
      for (int t = 0; t < D / 16; ++t) {
        const bf16x8 kf0 = *reinterpret_cast<const bf16x8*>(sk + k_lds_off<D>(lane & 31, 2 * t + h));
        const bf16x8 kf1 = *reinterpret_cast<const bf16x8*>(sk + k_lds_off<D>(32 + (lane & 31), 2 * t + h));
#pragma unroll
        for (int j = 0; j < HL; ++j) {
          const bf16x8 qv = *reinterpret_cast<const bf16x8*>(sq + (j * 32 + (lane & 31)) * Cfg::KRS + ((2 * t + h) << 4));
          s[j][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf0, qv, s[j][0], 0, 0, 0);
          s[j][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf1, qv, s[j][1], 0, 0, 0);
        }
      }
    }
    if (prio) __builtin_amdgcn_s_setprio(0);
    if (!ESPLIT && more) {  // buffer cur ^ 1 was released by the previous barrier
      write_k(cur ^ 1);
      load_half(vc);
    }
    // online softmax (exp2 domain); lane owns query (lane&31), keys split across lane halves.
    // Interior tiles (every key < ctx and, causal, <= the wave's first query position) skip the
    // per-element mask: wave-uniform test, so only the diagonal / tail tiles pay for it.
    float mt[HL];
#pragma unroll
    for (int j = 0; j < HL; ++j) mt[j] = kNeg;
    const int kend = kt * 64 + 63;
    if (kend < ctx && (!causal || kend <= ctx - qlen + r0)) {
#pragma unroll
      for (int j = 0; j < HL; ++j)
#pragma unroll
        for (int sub = 0; sub < 2; ++sub)
#pragma unroll
          for (int r = 0; r < 16; ++r) mt[j] = fmaxf(mt[j], s[j][sub][r]);
    } else {
#pragma unroll
      for (int sub = 0; sub < 2; ++sub)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool ok = 32 * sub + (r & 3) + 8 * (r >> 2) < klim - kt * 64;
#pragma unroll
          for (int j = 0; j < HL; ++j) {
            const float x = ok ? s[j][sub][r] : kNeg;
            s[j][sub][r] = x;
            mt[j] = fmaxf(mt[j], x);
          }
        }
    }
    // scores stay unscaled; the scale folds into the max (scale > 0) and into one fma per exp
    float m_new[HL], alpha[HL];
#pragma unroll
    for (int j = 0; j < HL; ++j) {
      mt[j] = max_halves(mt[j]) * sl2;
      m_new[j] = mt[j] > m_run[j] + th ? mt[j] : m_run[j];
      alpha[j] = fexp2(m_run[j] - m_new[j]);
      // lazy rescale: once the running maxima settle (most tiles after the first few) alpha == 1 in
      // every lane and the D/32 x 16 accumulator multiplies are skipped (bit-identical result)
      if (__any(alpha[j] != 1.f)) {
#pragma unroll
        for (int i = 0; i < D / 32; ++i) acc_o[j][i] *= alpha[j];
      }
      m_run[j] = m_new[j];
    }

    // O^T[d][q] += V^T[d][key] . P^T[key][q]. The 8 probabilities of each 8-key step are exponentiated
    // right before that step's MFMAs, so step st's MFMAs run in the matrix pipe while step st+1's
    // v_exp / cvt issue (the row sum is only needed after the tile). Each V^T fragment feeds the HL heads.
    float rs[HL];
#pragma unroll
    for (int j = 0; j < HL; ++j) rs[j] = 0.f;
    if (prio == 2) __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      const int sub = st >> 1, sp = st & 1;
      bf16x8 pf[HL];
#pragma unroll
      for (int j = 0; j < HL; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p = fexp2(fmaf(s[j][sub][8 * sp + e], sl2, -m_new[j]));
          rs[j] += p;
          pf[j][e] = (bf16)p;
        }
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) {
        // units 4st + h (lo) and 4st + 2 + h (hi) of row d: one 16-B pair in the image
        const bf16x8 vf = *reinterpret_cast<const bf16x8*>(sv + v_lds_off<D>(32 * dt + (lane & 31), 4 * st + h));
#pragma unroll
        for (int j = 0; j < HL; ++j)
          acc_o[j][dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[j], acc_o[j][dt], 0, 0, 0);
      }
    }
    if (prio == 2) __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int j = 0; j < HL; ++j) l_run[j] = l_run[j] * alpha[j] + rs[j];  // per lane half (summed after the loop)
    // the next-but-one tile's page lookups (scalar loads) after the P.V reads: an SMEM load in flight makes every
    // LDS wait a full lgkmcnt(0) (the two return out of order)
    if constexpr (!ROWS) lookup(kt + 2);  // pages past the context resolve to entry 0 (never read unmasked)
    if (more) {
      if constexpr (ROWS) {
        write_rows_k(cur ^ 1, stg);
        write_rows_v(cur ^ 1, stv);
      } else if constexpr (ESPLIT) {
        write_k(cur ^ 1);
        write_v_from(cur ^ 1, stv);
      } else {
        write_v(cur ^ 1);
      }
    }
    __syncthreads();
  }
  }  // one-tile loop
  // each lane half accumulated the row sum of its own keys (every tile rescaled both by the same alpha)
#pragma unroll
  for (int j = 0; j < HL; ++j) l_run[j] = sum_halves(l_run[j]);

  if (qrow < qlen) {
#pragma unroll
    for (int j = 0; j < HL; ++j) {
      const float inv = l_run[j] > 0.f ? 1.f / l_run[j] : 0.f;
      bf16* op = out + ((size_t)(qbeg + qrow) * Hq + head + j) * D;
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
          bf16x4_t o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = (bf16)(acc_o[j][dt][4 * c + r] * inv);
          *reinterpret_cast<bf16x4_t*>(op + 32 * dt + 8 * c + 4 * h) = o;
        }
      // natural-log softmax normaliser per (row, head): merges partial results (ring attention)
      if (lse != nullptr && h == 0)
        lse[(size_t)(qbeg + qrow) * Hq + head + j] =
            l_run[j] > 0.f ? (m_run[j] + __log2f(l_run[j])) * 0.69314718055994531f : kNeg;
    }
  }
}

// ----------------------------------------------------------------------------------------------
// Decode
// ----------------------------------------------------------------------------------------------
// FUSE (split_cnt != nullptr): the splits of a (sequence, kv head) are merged in the same launch by the split
// that finishes last, instead of a separate attn_decode_reduce launch. Hand-off without any fence
// (cdna_hip_programming Guideline 16, R1 form): the partials are stored write-through (sc1, relaxed agent-scope
// stores, so nothing is left dirty in this XCD's L2) -> every wave vmcnt(0) -> barrier -> lane 0 relaxed agent
// ticket fetch_add; the last arriver reads every split with sc1 loads (they bypass the CU's L1, so no acquire
// is needed). The first version published with a per-workgroup agent release (buffer_wbl2: 192.6 vs 117.4 us
// per layer). cnt[seq * Hkv + g] starts at 0 (zeroed at allocation) and the last arriver resets it for the next
// launch (graph replays).
typedef __attribute__((address_space(1))) unsigned gu32_t;
__device__ __forceinline__ void st_sc1(float* p, float v) {
  __hip_atomic_store((gu32_t*)p, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Merge the flash-decoding partials (O, max, sum) of ns splits for one (sequence, q head, dim): groups of
// kMergeGroup splits, every load of a group issued before its math, running-max rescale between groups. The
// separate reduce launch and the in-launch merge (write-through partials read with sc1 loads) take the same steps,
// so both round identically.
constexpr int kMergeGroup = 8;

// Keys per split. split_keys > 0: fixed. 0: adaptive - each sequence's context is cut into max_splits equal
// 128-key-aligned parts at run time, so a graph captured for the longest context a replay may see (the split count)
// still balances its splits on the contexts it actually runs (a fixed split sized for max_model_len = 3330 left
// a 2500-key context as 1792 + 708 keys: the critical path of the step).
__device__ __forceinline__ int split_len(int split_keys, int ctx, int max_splits) {
  if (split_keys > 0) return split_keys;
  const int per = (ctx + max_splits - 1) / max_splits;
  return max(128, (per + 127) / 128 * 128);
}
template <int N>
struct MergeGroups {  // N groups of splits of neighbouring dims, and their running sums
  float m[N * kMergeGroup], l[N * kMergeGroup];
  float2 o[N * kMergeGroup];
  float M = kNeg, L = 0.f, O0 = 0.f, O1 = 0.f;
  __device__ __forceinline__ void add(int j0, int s0, int ns) {
    float Mn = M;
#pragma unroll
    for (int j = 0; j < kMergeGroup; ++j) Mn = s0 + j < ns ? fmaxf(Mn, m[j0 + j]) : Mn;
    if (s0 > 0) {
      const float a = fexp2(M - Mn);
      L *= a;
      O0 *= a;
      O1 *= a;
    }
#pragma unroll
    for (int j = 0; j < kMergeGroup; ++j) {
      const float f = s0 + j < ns ? fexp2(m[j0 + j] - Mn) : 0.f;
      L = fmaf(l[j0 + j], f, L);
      O0 = fmaf(o[j0 + j].x, f, O0);
      O1 = fmaf(o[j0 + j].y, f, O1);
    }
    M = Mn;
  }
};
// The last workgroup's merge of a (sequence, kv head): a thread takes two neighbouring dims, and up to 8 N splits' partials are on
// their way at once (a round trip past this XCD's L2 is over a microsecond; a dim and a group at a time, 20 splits took six of them: one
// sequence of 2531 keys 12.3 -> 10.1 us, 23 of 1900 - 7900 on 8-bit pages 55.5 -> 53.7).
template <int N>
__device__ __forceinline__ void merge_and_store(const float* ws_o, const float* ws_ml, int B, int Hq, int D, int seq, int h0, int heads,
                                                int ns, bf16* out) {
  const auto ld2 = [](const float* p) {
    const unsigned long long x = __hip_atomic_load((__attribute__((address_space(1))) unsigned long long*)p, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
    return float2{__uint_as_float((unsigned)x), __uint_as_float((unsigned)(x >> 32))};
  };
  for (int e = 2 * threadIdx.x; e < heads * D; e += 512) {
    const int hq = h0 + e / D, d = e % D;
    MergeGroups<N> g;
    auto load = [&](int j0, int s0) {
#pragma unroll
      for (int j = 0; j < kMergeGroup; ++j) {
        const size_t i = ((size_t)min(s0 + j, ns - 1) * B + seq) * Hq + hq;
        const float2 ml = ld2(ws_ml + i * 2);
        g.m[j0 + j] = ml.x;
        g.l[j0 + j] = ml.y;
        g.o[j0 + j] = ld2(ws_o + i * D + d);
      }
    };
    int s0 = 0;
    if constexpr (N > 1) {
      for (; ns - s0 > kMergeGroup; s0 += N * kMergeGroup) {
#pragma unroll
        for (int n = 0; n < N; ++n) load(n * kMergeGroup, s0 + n * kMergeGroup);
#pragma unroll
        for (int n = 0; n < N; ++n)
          if (s0 + n * kMergeGroup < ns) g.add(n * kMergeGroup, s0 + n * kMergeGroup, ns);
      }
    }
    for (; s0 < ns; s0 += kMergeGroup) {
      load(0, s0);
      g.add(0, s0, ns);
    }
    bf16* y = out + ((size_t)seq * Hq + hq) * D + d;
    y[0] = (bf16)(g.L > 0.f ? g.O0 / g.L : 0.f);
    y[1] = (bf16)(g.L > 0.f ? g.O1 / g.L : 0.f);
  }
}
__device__ __forceinline__ void merge_splits(const float* ws_o, const float* ws_ml, int B, int Hq, int D, int seq,
                                             int hq, int d, int ns, float& L, float& O) {
  float M = kNeg;
  L = 0.f;
  O = 0.f;
  for (int s0 = 0; s0 < ns; s0 += kMergeGroup) {
    float m[kMergeGroup], l[kMergeGroup], o[kMergeGroup];
#pragma unroll
    for (int j = 0; j < kMergeGroup; ++j) {
      const size_t i = ((size_t)min(s0 + j, ns - 1) * B + seq) * Hq + hq;
      m[j] = ws_ml[i * 2];
      l[j] = ws_ml[i * 2 + 1];
      o[j] = ws_o[i * D + d];
    }
    float Mn = M;
#pragma unroll
    for (int j = 0; j < kMergeGroup; ++j) Mn = s0 + j < ns ? fmaxf(Mn, m[j]) : Mn;
    if (s0 > 0) {
      const float a = fexp2(M - Mn);
      L *= a;
      O *= a;
    }
#pragma unroll
    for (int j = 0; j < kMergeGroup; ++j) {
      const float f = s0 + j < ns ? fexp2(m[j] - Mn) : 0.f;
      L = fmaf(l[j], f, L);
      O = fmaf(o[j], f, O);
    }
    M = Mn;
  }
}

// A wave step covers H halves of 32 keys (2 pages each). Per half: K rows for the QK^T MFMA (lane:
// key row lane&15, 16 B of dims 32t + 8gq) and V^T columns for the PV MFMA.
//  * V16 = false: S row m of MFMA i is key 16i + m; P^T's k order is then {4gq..4gq+3, 16+4gq..+3}
//    and V^T is read as two 8-B pieces (one per page).
//  * V16 = true: row m of MFMA i is key 8(m>>2) + 4i + (m&3), so lane group gq ends up holding the
//    8 CONSECUTIVE keys 8gq..8gq+7 of P^T, and its V^T operand is one 16-B load (page gq>>1, keys
//    8(gq&1)..+7): half the V load instructions.
// Addresses of a chunk past the split are clamped to its last page (unconditional loads: a
// data-dependent branch around them would force vmcnt(0) waits), and such keys are masked.
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
// physical blocks of a chunk's pages (scalar loads). The non-pipelined loop looks the NEXT chunk's blocks up
// before issuing this chunk's K/V loads, so a K/V load never waits on a block-table round trip of its own.
template <int H>
struct DecBlk {
  int b[H][2];
};
template <int H>
__device__ __forceinline__ void dec_lookup(const int* bt, int kb, int last_page, int ctx, DecBlk<H>& o) {
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const int p0 = min(kb / kBS + 2 * h, last_page);
    o.b[h][0] = bt[p0];
    o.b[h][1] = (p0 + 1) * kBS < ctx ? bt[p0 + 1] : o.b[h][0];
  }
}
// An fp8 K row is read 16 B at a time (8-B reads of 16 rows each end at 4.75 TB/s of a stream, 16-B ones at 6.4): lane group gq
// then holds two 8-B pieces, 2gq and 2gq + 1 of the 64 dims. Two swaps put them where two MFMAs want them: x piece gq, y piece
// 4 + gq. (Rows of 16 lanes, x | y: 0 2 4 6 | 1 3 5 7 -> 0 1 4 5 | 2 3 6 7 -> 0 1 2 3 | 4 5 6 7.)
__device__ __forceinline__ void swap_pieces(unsigned& x, unsigned& y) {
  const auto a = __builtin_amdgcn_permlane16_swap(x, y, false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(a[0], a[1], false, false);
  x = b[0];
  y = b[1];
}
template <int D, int H, bool V16, typename KV, bool NTL>
struct DecChunk {
  // fp8 caches: chunks hold the raw 8-byte pieces, converted to bf16 right before their MFMA
  using Raw = typename std::conditional<sizeof(KV) == 1, uint2, bf16x8>::type;
  Raw k[H][2][D / 32];
  bf16x4_t vlo[H][V16 ? 1 : D / 16], vhi[H][V16 ? 1 : D / 16];
  Raw v8[H][V16 ? D / 16 : 1];

  __device__ __forceinline__ void load(const KV* kc, const KV* vc, int Hkv, int g, const DecBlk<H>& bl) {
    const int lane = threadIdx.x & 63, gq = lane >> 4;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int blk0 = bl.b[h][0], blk1 = bl.b[h][1];
      const size_t pb0 = ((size_t)blk0 * Hkv + g) * kBS * D, pb1 = ((size_t)blk1 * Hkv + g) * kBS * D;
      if (V16) {
        const int m = lane & 15;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int key = 8 * (m >> 2) + 4 * i + (m & 3);  // 0..31 inside the half
          const KV* row = kc + (key < 16 ? pb0 : pb1) + (size_t)(key & 15) * D;
          if constexpr (sizeof(KV) == 1) {
#pragma unroll
            for (int t = 0; t < D / 32; t += 2) {  // (as loaded; add() puts the pieces in their places)
              const uint4 x = *reinterpret_cast<const uint4*>(row + 32 * t + 16 * gq);
              k[h][i][t] = uint2{x.x, x.y};
              k[h][i][t + 1] = uint2{x.z, x.w};
            }
          } else {
            // K is read with the default policy even under NTL: one load instruction covers 16 key rows x 64 B, so
            // each 128-B line is requested in two halves by consecutive instructions, and the second half then hits
            // the line the first one allocated in L2 (B = 64, ctx 2535 graph replay 7.251 / 7.236 -> 7.149 /
            // 7.169 ms per step, profiles/r6/decode/k_policy_ab); V^T loads cover whole lines and stay non-temporal
#pragma unroll
            for (int t = 0; t < D / 32; ++t) k[h][i][t] = *reinterpret_cast<const Raw*>(row + 32 * t + 8 * gq);
          }
        }
        const size_t pbv = gq < 2 ? pb0 : pb1;
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) {
          const Raw* vp = reinterpret_cast<const Raw*>(vc + pbv + (size_t)(16 * dt + (lane & 15)) * kBS + 8 * (gq & 1));
          if constexpr (NTL) v8[h][dt] = __builtin_nontemporal_load(vp);
          else v8[h][dt] = *vp;
        }
      } else if constexpr (sizeof(KV) == 2) {
#pragma unroll
        for (int t = 0; t < D / 32; ++t) {
          k[h][0][t] = load8((const bf16*)kc + pb0 + (size_t)(lane & 15) * D + 32 * t + 8 * gq);
          k[h][1][t] = load8((const bf16*)kc + pb1 + (size_t)(lane & 15) * D + 32 * t + 8 * gq);
        }
#pragma unroll
        for (int dt = 0; dt < D / 16; ++dt) {
          const size_t off = (size_t)(16 * dt + (lane & 15)) * kBS + 4 * gq;
          vlo[h][dt] = *reinterpret_cast<const bf16x4_t*>((const bf16*)vc + pb0 + off);
          vhi[h][dt] = *reinterpret_cast<const bf16x4_t*>((const bf16*)vc + pb1 + off);
        }
      }
    }
  }
};
// a wave's running attention over its chunks: O^T[d = 16dt + 4gq + r][q = lane&15], maximum and sum (log2 domain)
template <int D>
struct DecAcc {
  f32x4 o[D / 16];
  float m, l;
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < D / 16; ++i) o[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    m = kNeg;
    l = 0.f;
  }
  template <int H, bool V16, typename KV, bool NTL>
  __device__ __forceinline__ void add(int kb, int kend, const DecChunk<D, H, V16, KV, NTL>& c, const bf16x8* qf, float sl2,
                                      float k_scale, float v_scale) {
    const int gq = (threadIdx.x & 63) >> 4;
    f32x4 s[H][2];
    float mt = kNeg;
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        s[h][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if constexpr (sizeof(KV) == 1 && V16) {
#pragma unroll
          for (int t = 0; t < D / 32; t += 2) {
            uint2 x = c.k[h][i][t], y = c.k[h][i][t + 1];
            swap_pieces(x.x, y.x);
            swap_pieces(x.y, y.y);
            s[h][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv_to_bf16(x, k_scale), qf[t], s[h][i], 0, 0, 0);
            s[h][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv_to_bf16(y, k_scale), qf[t + 1], s[h][i], 0, 0, 0);
          }
        } else {
#pragma unroll
          for (int t = 0; t < D / 32; ++t)
            s[h][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv_to_bf16(c.k[h][i][t], k_scale), qf[t], s[h][i], 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = kb + 32 * h + (V16 ? 8 * gq + 4 * i + r : 16 * i + 4 * gq + r);
          const float x = key < kend ? s[h][i][r] * sl2 : kNeg;
          s[h][i][r] = x;
          mt = fmaxf(mt, x);
        }
      }
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float m_new = fmaxf(m, mt);
    const float alpha = fexp2(m - m_new);
    float rs = 0.f;
    bf16x8 pf[H];
#pragma unroll
    for (int h = 0; h < H; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float pv = fexp2(s[h][i][r] - m_new);
          rs += pv;
          pf[h][4 * i + r] = (bf16)pv;
        }
    rs += __shfl_xor(rs, 16, 64);
    rs += __shfl_xor(rs, 32, 64);
    l = l * alpha + rs;
    m = m_new;
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) {
      o[dt] *= alpha;
#pragma unroll
      for (int h = 0; h < H; ++h) {
        bf16x8 vf;
        if constexpr (V16) {
          vf = kv_to_bf16(c.v8[h][dt], v_scale);
        } else {
          vf = bf16x8{c.vlo[h][dt][0], c.vlo[h][dt][1], c.vlo[h][dt][2], c.vlo[h][dt][3],
                      c.vhi[h][dt][0], c.vhi[h][dt][1], c.vhi[h][dt][2], c.vhi[h][dt][3]};
        }
        o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf[h], o[dt], 0, 0, 0);
      }
    }
  }
};
// QP prologue: the group's q heads from the split-K slabs (summed, rounded, rotated) into q_lds and on to qf; with `newest`
// also the group's new key and value into the caches. Quarter-row items (4 + 4 rotation partners of one head).
template <int D>
__device__ __forceinline__ void dec_qp_prologue(const GaiQkvFold& fold, bf16 (*q_lds)[D], bf16x8* qf, bf16* kc, bf16* vc, int B,
                                                int Hq, int Hkv, int seq, int g, bool newest) {
  const int tid = threadIdx.x, gq = (tid & 63) >> 4, qi = tid & 15, ratio = Hq / Hkv;
  constexpr int LPH = D / 8;
  const int nh = ratio + (newest ? 2 : 0);
  const size_t slab = (size_t)B * fold.n;
  for (int it = tid; it < nh * LPH; it += 256) {
    const int hh = it / LPH, i0 = (it % LPH) * 4;
    const int habs = hh < ratio ? g * ratio + hh : hh == ratio ? Hq + g : Hq + Hkv + g;
    const float* p1 = fold.part + (size_t)seq * fold.n + habs * D + i0;
    float x[4] = {0.f, 0.f, 0.f, 0.f}, y[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < fold.ks; s0 += 4) {  // 4 slabs in flight; slab order from 0 (the split-K tails' rounding)
      float4 a[4], b[4];
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (s0 + s < fold.ks) {
          a[s] = *reinterpret_cast<const float4*>(p1 + (s0 + s) * slab);
          b[s] = *reinterpret_cast<const float4*>(p1 + (s0 + s) * slab + D / 2);
        }
#pragma unroll
      for (int s = 0; s < 4; ++s)
        if (s0 + s < fold.ks) {
          x[0] += a[s].x; x[1] += a[s].y; x[2] += a[s].z; x[3] += a[s].w;
          y[0] += b[s].x; y[1] += b[s].y; y[2] += b[s].z; y[3] += b[s].w;
        }
    }
    bf16x4 x1, x2;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      x1[j] = (bf16)x[j];
      x2[j] = (bf16)y[j];
    }
    if (hh < ratio) {
      const int pp = fold.pos[seq];
      const float4 c = *reinterpret_cast<const float4*>(fold.cos_sin + (size_t)pp * D + i0);
      const float4 sn = *reinterpret_cast<const float4*>(fold.cos_sin + (size_t)pp * D + D / 2 + i0);
      const float cc[4] = {c.x, c.y, c.z, c.w}, ss[4] = {sn.x, sn.y, sn.z, sn.w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float u = (float)x1[j], w = (float)x2[j];
        x1[j] = (bf16)(u * cc[j] - w * ss[j]);
        x2[j] = (bf16)(w * cc[j] + u * ss[j]);
      }
      *reinterpret_cast<bf16x4*>(&q_lds[hh][i0]) = x1;
      *reinterpret_cast<bf16x4*>(&q_lds[hh][i0 + D / 2]) = x2;
    } else {
      rope_kv_store<D, bf16>(x1, x2, seq, habs, i0, fold.pos, fold.cos_sin, fold.slots, nullptr,
                             kc, vc, Hq, Hkv, 1, 1.f, 1.f);
    }
  }
  if (newest) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the new key / value have landed before any wave reads them
  __syncthreads();
  const bool qv = qi < ratio;
#pragma unroll
  for (int t = 0; t < D / 32; ++t)
    qf[t] = qv ? *reinterpret_cast<const bf16x8*>(&q_lds[qi][32 * t + 8 * gq]) : bf16x8{};
}

// NTL: the V^T cache loads are non-temporal (each decode step streams the cache once; keeps it from evicting the
// L2-resident Q / block tables / split partials)
// Occupancy: unconstrained, the compiler takes 138 VGPRs + 32 AGPRs (2 workgroups per CU, 512 resident), and two
// splits per (sequence, kv head) at B = 64 are exactly two rounds. Held to 3 per CU (no spill) with three splits it
// measured 7.424 vs 7.332 ms per step (profiles/r4/decode/decode_nt_split_ab.txt): kept at 2.
// QP (QkvFold): q is not read from memory - the prologue sums the split-K QKV partial slabs of this workgroup's
// GQA group, rounds to bf16 (the rounding of the unfused GEMM output), applies RoPE (the rounding of rope_kv) and
// stages the group's q rows in LDS; the split that holds the newest key also rotates / stores that key and value
// into the paged caches before its own key loop reads them (the only split that reads that page). This replaces
// the separate split-K RoPE / KV-write tail launch of the decode QKV projection.
template <int D, bool PIPE, int H, bool V16, typename KV, bool FUSE = false, bool NTL = false, bool QP = false>
__global__ __launch_bounds__(256) void attn_decode_kernel(
    const bf16* __restrict__ q, const KV* __restrict__ kc, const KV* __restrict__ vc,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ ctx_lens, bf16* __restrict__ out,
    float* __restrict__ ws_o, float* __restrict__ ws_ml, int B, int Hq, int Hkv, float scale, int split_keys,
    int max_splits, float k_scale, float v_scale, int* __restrict__ cnt, GaiQkvFold fold = GaiQkvFold{}) {
  static_assert(sizeof(KV) == 2 || V16, "fp8 KV decode uses the 16-key V^T loads");
  static_assert(!QP || sizeof(KV) == 2, "the folded QKV tail writes bf16 caches");
  __shared__ __attribute__((aligned(16))) float red_o[4][D][16];
  __shared__ float red_m[4][16], red_l[4][16];
  __shared__ int s_last;
  __shared__ __attribute__((aligned(16))) bf16 q_lds[QP ? 16 : 1][QP ? D : 8];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, gq = lane >> 4;
  const int split = blockIdx.x, g = blockIdx.y, seq = blockIdx.z;
  const int ratio = Hq / Hkv;
  const int ctx = ctx_lens[seq];
  split_keys = split_len(split_keys, ctx, max_splits);
  const int kstart = split * split_keys;
  if (kstart >= ctx) return;
  const int kend = min(ctx, kstart + split_keys);
  const int nsplit = (ctx + split_keys - 1) / split_keys;
  const int* bt = block_tables + (size_t)seq * max_blocks;
  const int qi = lane & 15;  // GQA head index inside the group (MFMA column)

  bf16x8 qf[D / 32];
  // called after this wave's first K / V chunk is in flight, so its latency hides under the stream
  auto qp_prologue = [&]() {
    if constexpr (QP)
      dec_qp_prologue<D>(fold, q_lds, qf, const_cast<bf16*>(reinterpret_cast<const bf16*>(kc)),
                         const_cast<bf16*>(reinterpret_cast<const bf16*>(vc)), B, Hq, Hkv, seq, g, split == nsplit - 1);
  };
  static_assert(!QP || !PIPE, "the folded QKV prologue runs in the non-pipelined loop");
  if constexpr (!QP) {
    const bool qv = qi < ratio;
    const bf16* qp = q + ((size_t)seq * Hq + g * ratio + (qv ? qi : 0)) * D + 8 * gq;
#pragma unroll
    for (int t = 0; t < D / 32; ++t) qf[t] = qv ? load8(qp + 32 * t) : bf16x8{};
  }

  DecAcc<D> acc;
  acc.clear();
  const float sl2 = scale * kLog2e;

  using Chunk = DecChunk<D, H, V16, KV, NTL>;
  using Blk = DecBlk<H>;
  const int last_page = (kend - 1) / kBS;
  auto lookup = [&](int kb, Blk& o) { dec_lookup<H>(bt, kb, last_page, ctx, o); };
  auto load_chunk_blk = [&](int, const Blk& bl, Chunk& c) { c.load(kc, vc, Hkv, g, bl); };
  auto load_chunk = [&](int kb, Chunk& c) {
    Blk bl;
    lookup(kb, bl);
    c.load(kc, vc, Hkv, g, bl);
  };
  auto compute_chunk = [&](int kb, const Chunk& c) { acc.add(kb, kend, c, qf, sl2, k_scale, v_scale); };

  constexpr int kStep = 128 * H;
  int kb = kstart + 32 * H * wid;
  if (PIPE) {
    if (kb < kend) {
      Chunk ca, cb;
      load_chunk(kb, ca);
      for (;;) {
        load_chunk(kb + kStep, cb);
        compute_chunk(kb, ca);
        kb += kStep;
        if (kb >= kend) break;
        load_chunk(kb + kStep, ca);
        compute_chunk(kb, cb);
        kb += kStep;
        if (kb >= kend) break;
      }
    }
  } else if (!QP) {
    if (kb < kend) {
      Blk nb;
      lookup(kb, nb);
      for (; kb < kend; kb += kStep) {
        Chunk c;
        load_chunk_blk(kb, nb, c);  // blocks looked up one chunk earlier
        // the next chunk's blocks, issued after this chunk's K/V loads (SMEM returns out of order, so a wait for the
        // blocks in use would also wait for these) and landing under this chunk's compute; pages past the split
        // clamp to its last page (looked up, never loaded)
        lookup(kb + kStep, nb);
        compute_chunk(kb, c);
      }
    }
  } else {
    // first chunk in flight before the prologue, unless it holds the newest key, whose value the prologue writes
    Blk nb;
    Chunk c0;
    const bool live = kb < kend;
    const bool pre = live && !(split == nsplit - 1 && kb <= ctx - 1 && ctx - 1 < kb + 32 * H);
    if (live) lookup(kb, nb);
    if (pre) load_chunk_blk(kb, nb, c0);
    qp_prologue();  // every wave (barrier inside)
    for (bool first = true; kb < kend; kb += kStep, first = false) {
      Chunk c;
      if (first && pre) c = c0;
      else load_chunk_blk(kb, nb, c);
      lookup(kb + kStep, nb);
      compute_chunk(kb, c);
    }
  }

  // combine the 4 waves: acc_o lane layout O^T[d = 16dt + 4gq + r][q = lane&15]
  if (lane < 16) {
    red_m[wid][lane] = acc.m;
    red_l[wid][lane] = acc.l;
  }
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
    for (int r = 0; r < 4; ++r) red_o[wid][16 * dt + 4 * gq + r][qi] = acc.o[dt][r];
  __syncthreads();
  for (int e = tid; e < ratio * D; e += 256) {
    const int qq = e / D, d = e % D;
    float M = kNeg;
#pragma unroll
    for (int w = 0; w < 4; ++w) M = fmaxf(M, red_m[w][qq]);
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = fexp2(red_m[w][qq] - M);
      L += red_l[w][qq] * f;
      O += red_o[w][d][qq] * f;
    }
    const int hq = g * ratio + qq;
    if (nsplit == 1) {
      out[((size_t)seq * Hq + hq) * D + d] = (bf16)(L > 0.f ? O / L : 0.f);
    } else if constexpr (FUSE) {
      st_sc1(ws_o + (((size_t)split * B + seq) * Hq + hq) * D + d, O);
      if (d == 0) {
        st_sc1(ws_ml + (((size_t)split * B + seq) * Hq + hq) * 2, M);
        st_sc1(ws_ml + (((size_t)split * B + seq) * Hq + hq) * 2 + 1, L);
      }
    } else {
      ws_o[(((size_t)split * B + seq) * Hq + hq) * D + d] = O;
      if (d == 0) {
        ws_ml[(((size_t)split * B + seq) * Hq + hq) * 2] = M;
        ws_ml[(((size_t)split * B + seq) * Hq + hq) * 2 + 1] = L;
      }
    }
  }
  if constexpr (FUSE) {
    if (nsplit == 1) return;  // wave-uniform for the whole workgroup
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's write-through partials have landed
    __syncthreads();
    if (tid == 0) s_last = __hip_atomic_fetch_add(cnt + seq * Hkv + g, 1, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT) == nsplit - 1;
    __syncthreads();
    if (!s_last) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");  // no instruction: keeps the loads below the ticket
    merge_and_store<(D >= 128 ? 3 : 1)>(ws_o, ws_ml, B, Hq, D, seq, g * ratio, ratio, nsplit, out);
    if (tid == 0) __hip_atomic_store(cnt + seq * Hkv + g, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The same parts of every context as attn_decode_kernel's (and the same bits), handed out longest first to the workgroups that are
// resident: each begins with one and draws its next when it is about to finish, from the queue of its XCD (one counter for all,
// drawn from 2048 times, took 2 - 4 us of a launch). There, of ragged contexts' parts the long ones may start last, and every part
// starts anew with nothing in flight; here the next part's first chunk is on its way while the finished one is combined. One
// card, 8 kv heads, graphs captured for 8192, there -> here, us: bf16, 64 sequences of 640 - 2663 keys 102 -> 90, of 40 - 700
// 44.2 -> 31.4, 32 of 500 - 3000 59.3 -> 50.8, 23 of 1900 - 7900 98 -> 92; fp8 66.7 -> 55.2, 33.1 -> 23.9, 43.3 -> 33.5, 67.6 ->
// 56.8. Where every part is resident at once (up to 64 sequences) the launch only spreads them evenly: 24 of 30 - 300 keys 10.8 -> 11.0,
// of 30 - 100 7.4 -> 6.8, 64 of them 20.6 -> 8.8. Ranked and drawn from all the same, 13.2 and 8.9; ranked through LDS by a thread a
// sequence, one after another, 1 us more at 24 sequences and 10 at 256. Equal contexts gain nothing (32 of 2600 - 2700 72.6 -> 74.6).
// Even cuts of the whole batch's keys instead of each sequence's took 83, 30, 49 and 86 us where the parts here took 88, 33, 51 and 86,
// with other sums. Parts dealt beforehand, forth and back, 93, 34, 54, 89. A second chunk in flight per wave changed nothing: what is
// left is the stream of 4-KB (2-KB) pages.
constexpr int kQueueSeqs = 256;  // sequences that the ranking holds
template <int D, typename KV, bool NTL, bool QP>
__global__ __launch_bounds__(256, 3) void attn_decode_queue_kernel(
    const bf16* __restrict__ q, const KV* __restrict__ kc, const KV* __restrict__ vc, const int* __restrict__ block_tables,
    int max_blocks, const int* __restrict__ ctx_lens, bf16* __restrict__ out, float* __restrict__ ws_o,
    float* __restrict__ ws_ml, int B, int Hq, int Hkv, float scale, int max_splits, float k_scale, float v_scale,
    int* __restrict__ cnt, GaiQkvFold fold) {
  static_assert(!QP || sizeof(KV) == 2, "the folded QKV tail writes bf16 caches");
  __shared__ __attribute__((aligned(16))) float red_o[4][D][16];
  __shared__ float red_m[4][16], red_l[4][16];
  __shared__ int s_last, s_next, s_total;
  __shared__ int s_ctx[kQueueSeqs], s_parts[kQueueSeqs], s_seq[kQueueSeqs], s_first[kQueueSeqs];  // the last two by rank
  __shared__ __attribute__((aligned(16))) bf16 q_lds[QP ? 16 : 1][QP ? D : 8];
  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6), gq = lane >> 4, qi = lane & 15;
  const int ratio = Hq / Hkv;
  const float sl2 = scale * kLog2e;
  struct Part {
    int seq, g, split, ctx, kstart, kend, nsplit;
  };
  auto part = [&](int seq, int ctx, int i) {  // part i of a sequence, one kv head after another
    const int len = split_len(0, ctx, max_splits);
    Part p;
    p.seq = seq;
    p.ctx = ctx;
    p.split = i / Hkv;
    p.g = i - p.split * Hkv;
    p.nsplit = (ctx + len - 1) / len;
    p.kstart = p.split * len;
    p.kend = min(ctx, p.kstart + len);
    return p;
  };
  auto parts_of = [&](int ctx) { return (ctx + split_len(0, ctx, max_splits) - 1) / split_len(0, ctx, max_splits); };
  const int x8 = blockIdx.x & 7, G = gridDim.x / 8;
  int item = blockIdx.x >> 3, total = 0;
  Part p;
  bool drawing = true;
  if (B <= 64) {
    // With no more parts than workgroups there is nothing to rank or draw (short contexts in a graph captured for long ones): every
    // wave numbers the parts in the sequences' own order.
    const int ctx = lane < B ? max(ctx_lens[lane], 0) : 0, n = lane < B ? parts_of(ctx) : 0;
    int run = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int up = __shfl_up(run, o, 64);
      if (lane >= o) run += up;
    }
    total = __builtin_amdgcn_readlane(run, 63) * Hkv;
    drawing = total > (int)gridDim.x;
    if (!drawing) {
      const int i = 8 * item + x8;
      if (i >= total) return;
      const int r = __popcll(__ballot(lane < B && (run - n) * Hkv <= i)) - 1;
      p = part(r, __builtin_amdgcn_readlane(ctx, r), i - __builtin_amdgcn_readlane(run - n, r) * Hkv);
    }
  }
  if (drawing) {
    // Sequences by falling length; the parts are numbered in that order. Every wave compares all sequences, one a lane, with a quarter
    // of them, held a lane each and read from there.
    for (int i = tid; i < kQueueSeqs; i += 256) s_seq[i] = 0;
    const int quarter = (B + 3) / 4, j0 = wid * quarter, nj = min(quarter, B - j0);
    int key = 0, val = 0;  // longer first, then as given; one sequence and its parts (B * max_splits < 2^22)
    if (lane < nj) {
      const int j = j0 + lane, ctx = max(ctx_lens[j], 0), n = parts_of(ctx);
      s_ctx[j] = ctx;
      s_parts[j] = n;
      s_first[j] = key = min(ctx, (1 << 23) - 1) << 8 | (255 - j);
      val = n << 9 | 1;
    }
    __syncthreads();
    for (int i0 = 0; i0 < B; i0 += 64) {
      const int i = min(i0 + lane, B - 1), mine = s_first[i];
      int sum = 0;
      for (int j = 0; j < nj; ++j)
        sum += __builtin_amdgcn_readlane(key, j) > mine ? __builtin_amdgcn_readlane(val, j) : 0;
      if (i0 + lane < B && sum) atomicAdd(&s_seq[i], sum);
    }
    __syncthreads();
    const int before = tid < B ? s_seq[tid] : 0;
    __syncthreads();
    if (tid < B) {
      const int rank = before & 511, first = before >> 9;
      s_seq[rank] = tid;
      s_first[rank] = first * Hkv;
      if (rank == B - 1) s_total = (first + s_parts[tid]) * Hkv;
    }
    __syncthreads();
    total = __builtin_amdgcn_readfirstlane(s_total);
  }
  auto find = [&](int item) {
    int r = -1;  // the last rank that begins at or before item
    for (int b0 = 0; b0 < B; b0 += 64) {
      const int n = __popcll(__ballot(b0 + lane < B && s_first[min(b0 + lane, B - 1)] <= item));
      r += n;
      if (n < 64) break;
    }
    r = __builtin_amdgcn_readfirstlane(r);
    const int seq = __builtin_amdgcn_readfirstlane(s_seq[r]);
    return part(seq, __builtin_amdgcn_readfirstlane(s_ctx[seq]), item - __builtin_amdgcn_readfirstlane(s_first[r]));
  };
  // queue x: parts x, x + 8, ..; its workgroups (gridDim.x / 8) begin with the first ones and draw until nothing is left, mine times in
  // all; with no more parts than workgroups nobody draws
  const int mine = (total - x8 + 7) / 8;
  const bool ranked = drawing;
  drawing = mine > G;
  int* queue = cnt + B * Hkv + x8 * 32;  // 0 between launches
  auto draw = [&]() { return __hip_atomic_fetch_add(queue, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  auto drew = [&](int n) {
    if (n == mine - 1) __hip_atomic_store(queue, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if (item >= mine) return;
  if (ranked) p = find(8 * item + x8);

  bf16x8 qf[D / 32];
  DecAcc<D> acc;
  DecBlk<1> nb;
  DecChunk<D, 1, true, KV, NTL> c;
  auto table = [&](const Part& p) { return block_tables + (size_t)p.seq * max_blocks; };
  // The newest key is written by the prologue of the part that holds it: a first chunk with it is not asked for before.
  auto early = [&](const Part& p, int kb) {
    return kb < p.kend && !(QP && p.split == p.nsplit - 1 && kb <= p.ctx - 1 && p.ctx - 1 < kb + 32);
  };
  int kb = p.kstart + 32 * wid;
  dec_lookup<1>(table(p), kb, (p.kend - 1) / kBS, p.ctx, nb);
  bool have = early(p, kb);
  if (have) c.load(kc, vc, Hkv, p.g, nb);
  for (;;) {
    if constexpr (QP) {
      dec_qp_prologue<D>(fold, q_lds, qf, const_cast<bf16*>(reinterpret_cast<const bf16*>(kc)),
                         const_cast<bf16*>(reinterpret_cast<const bf16*>(vc)), B, Hq, Hkv, p.seq, p.g, p.split == p.nsplit - 1);
    } else {
      const bool qv = qi < ratio;
      const bf16* qp = q + ((size_t)p.seq * Hq + p.g * ratio + (qv ? qi : 0)) * D + 8 * gq;
#pragma unroll
      for (int t = 0; t < D / 32; ++t) qf[t] = qv ? load8(qp + 32 * t) : bf16x8{};
    }
    acc.clear();
    const int* bt = table(p);
    const int last_page = (p.kend - 1) / kBS;
    int drawn = 0;
    if (!have && kb < p.kend) c.load(kc, vc, Hkv, p.g, nb);
    while (kb < p.kend) {
      const int next = kb + 128;
      if (next < p.kend) dec_lookup<1>(bt, next, last_page, p.ctx, nb);
      else if (drawing && tid == 0) drawn = draw();  // (wave 0 has keys of every part) under the last chunk's products
      acc.add(kb, p.kend, c, qf, sl2, k_scale, v_scale);
      if (next < p.kend) c.load(kc, vc, Hkv, p.g, nb);
      kb = next;
    }
    // combine the 4 waves
    __syncthreads();  // the previous part's sums have been read
    if (drawing && tid == 0) {
      s_next = G + drawn;
      drew(drawn);
    }
    if (lane < 16) {
      red_m[wid][lane] = acc.m;
      red_l[wid][lane] = acc.l;
    }
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
      for (int r = 0; r < 4; ++r) red_o[wid][16 * dt + 4 * gq + r][qi] = acc.o[dt][r];
    __syncthreads();
    item = drawing ? __builtin_amdgcn_readfirstlane(s_next) : mine;
    const bool more = item < mine;
    Part np = p;
    if (more) {
      np = find(8 * item + x8);
      kb = np.kstart + 32 * wid;
      dec_lookup<1>(table(np), kb, (np.kend - 1) / kBS, np.ctx, nb);
      have = early(np, kb);
      if (have) c.load(kc, vc, Hkv, np.g, nb);
    }
    for (int e = tid; e < ratio * D; e += 256) {
      const int qq = e / D, d = e % D, hq = p.g * ratio + qq;
      float M = kNeg, L = 0.f, O = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) M = fmaxf(M, red_m[w][qq]);
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const float f = fexp2(red_m[w][qq] - M);
        L += red_l[w][qq] * f;
        O += red_o[w][d][qq] * f;
      }
      if (p.nsplit == 1) {
        out[((size_t)p.seq * Hq + hq) * D + d] = (bf16)(L > 0.f ? O / L : 0.f);
      } else {
        const size_t i = ((size_t)p.split * B + p.seq) * Hq + hq;
        st_sc1(ws_o + i * D + d, O);
        if (d == 0) {
          st_sc1(ws_ml + i * 2, M);
          st_sc1(ws_ml + i * 2 + 1, L);
        }
      }
    }
    if (p.nsplit > 1) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's write-through partials have landed
      __syncthreads();
      if (tid == 0) s_last = __hip_atomic_fetch_add(cnt + p.seq * Hkv + p.g, 1, __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT) == p.nsplit - 1;
      __syncthreads();
      if (s_last) {
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");  // no instruction: keeps the loads below the ticket
        merge_and_store<1>(ws_o, ws_ml, B, Hq, D, p.seq, p.g * ratio, ratio, p.nsplit, out);
        if (tid == 0) __hip_atomic_store(cnt + p.seq * Hkv + p.g, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (!more) return;
    p = np;
  }
}

template <int D>
__global__ void attn_decode_reduce_kernel(const float* __restrict__ ws_o, const float* __restrict__ ws_ml,
                                          const int* __restrict__ ctx_lens, bf16* __restrict__ out, int B, int Hq,
                                          int split_keys, int max_splits) {
  const int seq = blockIdx.x, hq = blockIdx.y, d = threadIdx.x;
  const int ctx = ctx_lens[seq];
  split_keys = split_len(split_keys, ctx, max_splits);
  const int ns = (ctx + split_keys - 1) / split_keys;
  if (ns <= 1) return;
  float L, O;
  merge_splits(ws_o, ws_ml, B, Hq, D, seq, hq, d, ns, L, O);
  out[((size_t)seq * Hq + hq) * D + d] = (bf16)(L > 0.f ? O / L : 0.f);
}

// Raise a kernel's dynamic-LDS limit once per KERNEL (a static flag inside a template over the function type would be
// shared by every instantiation with the same signature, e.g. all bf16 prefill kernels).
template <typename F>
void set_max_lds(F* f, int bytes) {
  static std::mutex mu;
  static std::unordered_map<const void*, int> done;
  const void* key = reinterpret_cast<const void*>(f);
  std::lock_guard<std::mutex> lk(mu);
  auto it = done.find(key);
  if (it != done.end() && it->second >= bytes) return;
  hipFuncSetAttribute(key, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  done[key] = bytes;
}

// Heads per wave of the prefill kernel (attn_prefill_kernel HL): 2 for head_dim 128 with >= 4 q heads per kv head when
// enabled (GAI_ATTN_HL=2 or gai_attn_prefill_set_hl), else 1. The tile list's rows per tile follow it
// (gai_attn_prefill_rows_per_tile), so it is read once per process unless set explicitly.
int g_prefill_hl = -1;
int prefill_hl(int D, int ratio) {
  if (g_prefill_hl < 0) g_prefill_hl = getenv("GAI_ATTN_HL") ? atoi(getenv("GAI_ATTN_HL")) : 1;
  return g_prefill_hl == 2 && D == 128 && ratio >= 4 ? 2 : 1;
}

}  // namespace

void gai_attn_prefill_set_hl(int hl) { g_prefill_hl = hl == 2 ? 2 : 1; }

namespace {
// Waves per workgroup of the one-tile prefill kernel: 8 for head_dim 64 / 128 at >= 4 q heads per kv head (one head
// per wave: 2 row groups x 4 heads = 64 rows per tile share each staged K / V^T tile), else 4 (GAI_ATTN_WAVES=4 forces
// it). Same box, interleaved (profiles/r6/attn_prefill/waves_ab_*): headline chunk 7 x 2406 GQA 32/8 782 / 779 ->
// 796 / 828 TF/s, B 4 x 2048 693 / 689 -> 706 / 696. Not for MHA: the 256-row tiles of one head waste up to 3 of
// their causal key tiles on the upper row groups (encoder shape, causal: 415 -> 295). The tile list's rows per tile
// follow it (gai_attn_prefill_rows_per_tile).
int prefill_waves(int D, int ratio) {
  static const int env = getenv("GAI_ATTN_WAVES") ? atoi(getenv("GAI_ATTN_WAVES")) : 8;
  static const int pipe = getenv("GAI_ATTN_PIPE") ? atoi(getenv("GAI_ATTN_PIPE")) : 0;
  return env == 8 && (D == 64 || D == 128) && ratio >= 4 && prefill_hl(D, ratio) == 1 && pipe != 1 ? 8 : 4;
}

int decode_cus() {
  static const int n = [] {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus < 1)
      gai_launch_error(__FILE__, __LINE__, "attention: cannot query the CU count");
    return cus;
  }();
  return n;
}

template <int DD, int HP, typename KV>
void prefill_launch(const void* q, const void* k_cache, const void* v_cache, const int* block_tables, int max_blocks,
                    const int* tiles, int ntiles, const int* cu_q, const int* ctx_lens, void* out, int Hq, int Hkv,
                    float scale, int causal, float* lse, float k_scale, float v_scale, int xcd, int q_ld, int nwv,
                    hipStream_t st) {
  const int lds = 2 * PrefillCfg<DD>::BUF;
  if constexpr (DD == 64 || DD == 128) {
    // Few tiles: 32 of their 64 rows to a workgroup. A tile is a chain of key tiles, and one wave a SIMD goes down it in 1.6 us
    // a key tile, two in 2.0; halves also even out the causal lengths. Up to three halves a CU (two are resident): 32 / 8 heads
    // of 128, a prompt of 17, 66, 187, 600, 1024 tokens 7.1, 10.3, 14.2, 24.9, 38.1 -> 5.9, 6.8, 10.1, 19.7, 30.2 us, 1496 50.6 ->
    // 44.4, 2000 66.4 -> 60.8, 3000 99.6 -> 93.3; 16 / 4 heads 3000 87.7 -> 75.4. Beyond, the key tiles fetched once for 64 rows
    // count too: 4000 145.5 | 149.2, 4095 + 6000 (16 / 4) 238.5 | 241.2, 6 x 2300 306 | 301. Chunks over a prefix, whose keys both halves
    // fetch: 64 rows behind 2000 63.9 -> 49.5, behind 30000 784 -> 634, 1024 behind 8000 248 -> 209. Heads of 64 and fp8 pages alike (0.71 -
    // 0.91 of whole tiles); nothing at the upper end: 32 / 8 heads of 64, 1500 tokens 34.2 | 34.0, 64 / 8 of 128, 1024 behind 8000 300 | 301. Equal
    // bits: a row's key tiles and their order are the same.
    if constexpr (HP == 4) {
      if (nwv == 8 && 2 * ntiles * (Hq / HP) <= 3 * decode_cus()) {
        auto kern = attn_prefill_kernel<DD, HP, KV, 1, false, 4, 0, true>;
        set_max_lds(kern, lds);
        kern<<<dim3(2 * ntiles, Hq / HP), 256, lds, st>>>((const bf16*)q, (const KV*)k_cache, (const KV*)v_cache, block_tables,
                                                          max_blocks, tiles, cu_q, ctx_lens, (bf16*)out, Hq, Hkv, scale, causal,
                                                          lse, k_scale, v_scale, xcd, q_ld);
        GAI_LAUNCH_CHECK();
        return;
      }
    }
    if (nwv == 8) {  // the staggered loop keeps three tile slots
      auto kern = attn_prefill_kernel<DD, HP, KV, 1, false, 8>;
      set_max_lds(kern, 3 * PrefillCfg<DD>::BUF);
      kern<<<dim3(ntiles, Hq / HP), 512, 3 * PrefillCfg<DD>::BUF, st>>>((const bf16*)q, (const KV*)k_cache, (const KV*)v_cache,
                                                    block_tables, max_blocks, tiles, cu_q, ctx_lens, (bf16*)out, Hq,
                                                    Hkv, scale, causal, lse, k_scale, v_scale, xcd, q_ld);
      GAI_LAUNCH_CHECK();
      return;
    }
  }
  auto kern = attn_prefill_kernel<DD, HP, KV>;
  set_max_lds(kern, lds);
  kern<<<dim3(ntiles, Hq / HP), 256, lds, st>>>((const bf16*)q, (const KV*)k_cache, (const KV*)v_cache, block_tables,
                                                max_blocks, tiles, cu_q, ctx_lens, (bf16*)out, Hq, Hkv, scale, causal,
                                                lse, k_scale, v_scale, xcd, q_ld);
  GAI_LAUNCH_CHECK();
}
}  // namespace

void gai_attn_prefill(const void* q, const void* k_cache, const void* v_cache, const int* block_tables,
                      int max_blocks, const int* tiles, int ntiles, const int* cu_q, const int* ctx_lens, void* out,
                      int Hq, int Hkv, int D, float scale, int causal, float* lse, int kv_fp8, float k_scale,
                      float v_scale, hipStream_t st, int q_ld) {
  if (ntiles == 0) return;
  if (q_ld <= 0) q_ld = Hq * D;
  const int ratio = Hq / Hkv;
  const int hpw = ratio >= 4 ? 4 : ratio >= 2 ? 2 : 1;
  // XCD kv-head placement for causal decoder prefill at head_dim >= 128 (long K/V prefixes re-read by many q tiles).
  // Off for the head_dim-64 encoders (413 -> 394 TF/s with it) and for non-causal attention: config 4 (Mllama
  // cross-attention over the vision tokens) ran 6.69 -> 6.52 q/s with it (profiles/r3/attn_prefill_xcd).
  // GAI_ATTN_XCD=0 / 2: off / on everywhere.
  static const int xcd_env = getenv("GAI_ATTN_XCD") ? atoi(getenv("GAI_ATTN_XCD")) : 1;
  // wave priority 1 while a wave issues its QK^T / P.V MFMAs (0 in the softmax): +1-2 % on every head_dim-64/128 shape
  // (headline chunk 707-714 -> 721 TF/s, profiles/r5/attn_prefill/prio_ab.txt); GAI_ATTN_PRIO = 0 / 1 for A/B
  static const int prio_env = getenv("GAI_ATTN_PRIO") ? atoi(getenv("GAI_ATTN_PRIO")) : 2;
  static const bool exact_max = getenv("GAI_ATTN_RESCALE_TH") && atoi(getenv("GAI_ATTN_RESCALE_TH")) == 0;
  static const bool no_stagger = getenv("GAI_ATTN_STAGGER") && atoi(getenv("GAI_ATTN_STAGGER")) == 0;
  const int xcd = (xcd_env == 2 || (xcd_env == 1 && D >= 128 && causal)) | ((prio_env & 3) << 1) | (exact_max ? 8 : 0) |
                  (no_stagger ? 16 : 0);
  const int hl = prefill_hl(D, ratio);
  const int nwv = prefill_waves(D, ratio);
  if (hl == 2) {  // D == 128, hpw == 4: 64 rows per tile; + the 4 waves' Q images (2 heads x 32 rows each)
    const int lds = 2 * PrefillCfg<128>::BUF + 4 * 2 * 32 * PrefillCfg<128>::KRS;
    if (kv_fp8) {
      auto kern = attn_prefill_kernel<128, 4, fp8, 2>;
      set_max_lds(kern, lds);
      kern<<<dim3(ntiles, Hq / 4), 256, lds, st>>>((const bf16*)q, (const fp8*)k_cache, (const fp8*)v_cache,
                                                   block_tables, max_blocks, tiles, cu_q, ctx_lens, (bf16*)out, Hq,
                                                   Hkv, scale, causal, lse, k_scale, v_scale, xcd, q_ld);
    } else {
      auto kern = attn_prefill_kernel<128, 4, bf16, 2>;
      set_max_lds(kern, lds);
      kern<<<dim3(ntiles, Hq / 4), 256, lds, st>>>((const bf16*)q, (const bf16*)k_cache, (const bf16*)v_cache,
                                                   block_tables, max_blocks, tiles, cu_q, ctx_lens, (bf16*)out, Hq,
                                                   Hkv, scale, causal, lse, k_scale, v_scale, xcd, q_ld);
    }
    GAI_LAUNCH_CHECK();
    return;
  }
  // GAI_ATTN_PIPE = 1: the software-pipelined main loop (attn_prefill_kernel PIPE)
  static const int pipe_env = getenv("GAI_ATTN_PIPE") ? atoi(getenv("GAI_ATTN_PIPE")) : 0;
#define GAI_PF(DD, HP)                                                                                         \
  if (D == DD && hpw == HP && pipe_env == 1) {                                                                 \
    const int lds = 2 * PrefillCfg<DD>::BUF;                                                                   \
    if (kv_fp8) {                                                                                              \
      auto kern = attn_prefill_kernel<DD, HP, fp8, 1, true>;                                                   \
      set_max_lds(kern, lds);                                                                                  \
      kern<<<dim3(ntiles, Hq / HP), 256, lds, st>>>((const bf16*)q, (const fp8*)k_cache, (const fp8*)v_cache,  \
                                                    block_tables, max_blocks, tiles, cu_q, ctx_lens, (bf16*)out, \
                                                    Hq, Hkv, scale, causal, lse, k_scale, v_scale, xcd, q_ld); \
    } else {                                                                                                   \
      auto kern = attn_prefill_kernel<DD, HP, bf16, 1, true>;                                                  \
      set_max_lds(kern, lds);                                                                                  \
      kern<<<dim3(ntiles, Hq / HP), 256, lds, st>>>((const bf16*)q, (const bf16*)k_cache, (const bf16*)v_cache, \
                                                    block_tables, max_blocks, tiles, cu_q, ctx_lens, (bf16*)out, \
                                                    Hq, Hkv, scale, causal, lse, k_scale, v_scale, xcd, q_ld); \
    }                                                                                                          \
    GAI_LAUNCH_CHECK();                                                                                        \
    return;                                                                                                    \
  }                                                                                                            \
  if (D == DD && hpw == HP) {                                                                                  \
    if (kv_fp8)                                                                                                \
      prefill_launch<DD, HP, fp8>(q, k_cache, v_cache, block_tables, max_blocks, tiles, ntiles, cu_q, ctx_lens, \
                                  out, Hq, Hkv, scale, causal, lse, k_scale, v_scale, xcd, q_ld, nwv, st);     \
    else                                                                                                       \
      prefill_launch<DD, HP, bf16>(q, k_cache, v_cache, block_tables, max_blocks, tiles, ntiles, cu_q, ctx_lens, \
                                   out, Hq, Hkv, scale, causal, lse, k_scale, v_scale, xcd, q_ld, nwv, st);    \
    return;                                                                                                    \
  }
  GAI_PF(64, 1)
  GAI_PF(64, 2)
  GAI_PF(64, 4)
  GAI_PF(96, 1)  // Mllama vision encoder: head_dim 80 zero-padded to 96 (not 128): 25 % less MFMA work
  GAI_PF(96, 2)
  GAI_PF(96, 4)
  GAI_PF(128, 1)
  GAI_PF(128, 2)
  GAI_PF(128, 4)
  GAI_PF(256, 1)
  GAI_PF(256, 2)
  GAI_PF(256, 4)
#undef GAI_PF
  gai_launch_error(__FILE__, __LINE__, "attn_prefill: unsupported head_dim");
}

// head_dim 64, one kv head per q head: rows [q | k | v] of H heads each, ld apart
void gai_attn_rows(const void* qkv, int ld, const int* tiles, int ntiles, const int* cu_q, const int* ctx_lens, void* out, int H,
                   float scale, int causal, hipStream_t st) {
  if (ntiles == 0) return;
  static const int prio_env = getenv("GAI_ATTN_PRIO") ? atoi(getenv("GAI_ATTN_PRIO")) : 2;
  static const bool exact_max = getenv("GAI_ATTN_RESCALE_TH") && atoi(getenv("GAI_ATTN_RESCALE_TH")) == 0;
  const bf16* q = (const bf16*)qkv;
  const int lds = 2 * PrefillCfg<64>::BUF;
  // Past three workgroups a CU (143 registers) the kernel in 128, of which four are resident: 16 heads, us, three | four: 61
  // passages of 117 - 512 tokens 66.2 | 64.6, 16 of 512 36.9 | 32.3, 64 of 30 8.5 | 7.6; one of 32 3.82 | 3.94, one of 300 8.85 | 9.26
  const bool dense = ntiles * H > 3 * decode_cus();
  auto kern = dense ? attn_prefill_kernel<64, 1, bf16, 1, false, 4, 2> : attn_prefill_kernel<64, 1, bf16, 1, false, 4, 1>;
  set_max_lds(attn_prefill_kernel<64, 1, bf16, 1, false, 4, 1>, lds);
  set_max_lds(attn_prefill_kernel<64, 1, bf16, 1, false, 4, 2>, lds);
  kern<<<dim3(ntiles, H), 256, lds, st>>>(q, q + H * 64, q + 2 * H * 64, nullptr, 0, tiles, cu_q, ctx_lens, (bf16*)out, H, H, scale,
                                          causal, nullptr, 1.f, 1.f, ((prio_env & 3) << 1) | (exact_max ? 8 : 0), ld);
  GAI_LAUNCH_CHECK();
}

namespace {
// Attention of up to 64 rows and its output projection in one launch: a workgroup takes HG heads of a sequence and 64 columns of the
// projection, whose K slices the heads are, and leaves their sums in slab blockIdx.y for the norm that follows. Up to 64 rows both
// launches are latency (the projection's 2 MB are a slice of 16 KB a workgroup, on its way while the heads attend), and every
// workgroup of a head group attends anew, which takes it what one workgroup of attn_prefill_kernel takes. Up to eight sequences
// (attention_layer_norm_ok): with the norm, 1024 x 1024, us, three launches | two: 16 rows 9.6 | 7.6, 32 9.8 | 8.0, 64 10.9 | 10.3,
// four sequences of 16 10.7 | 8.0, eight of 8 10.7 | 8.6, but 64 of one row 12.8 | 21.3 (every sequence reads the slices again).
// A wave takes 32 rows of a head: four heads of up to 32 rows, two of up to 64. The attention's sums are attn_prefill_kernel's.
template <int HG>
__global__ __launch_bounds__(256) void attn_rows_slabs_kernel(const bf16* __restrict__ qkv, int ld, const int* __restrict__ cu_q,
                                                              const int* __restrict__ ctx_lens, const bf16* __restrict__ W,
                                                              float* __restrict__ ws, int M, int N, int H, float scale, int frag) {
  using Cfg = PrefillCfg<64>;
  constexpr int RW = 4 / HG, KS = 2 * HG, OS = HG * 128 + 16;  // waves a head, k32 steps, bytes of a row of the heads' results
  __shared__ __attribute__((aligned(16))) char sv[HG * Cfg::VBYTES], so[32 * RW * OS];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), h = lane >> 5;
  const int hp = blockIdx.y, seq = blockIdx.z, nt = blockIdx.x * 4 + w;  // this wave's 16 columns
  const int qbeg = cu_q[seq], qlen = min(cu_q[seq + 1] - qbeg, 32 * RW);
  if (qlen <= 0) return;
  const int ctx = max(min(ctx_lens[seq], qlen), 0);
  bf16x8 wf[KS];
#pragma unroll
  for (int k = 0; k < KS; ++k)
    wf[k] = load8(frag ? W + ((size_t)nt * (2 * H) + KS * hp + k) * 512 + lane * 8
                       : W + (size_t)(nt * 16 + (lane & 15)) * (H * 64) + (KS * hp + k) * 32 + (lane >> 4) * 8);
  auto rows = [&](int which, int head, int n) {  // n rows of a head, zeros beyond
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(qkv) + (size_t)qbeg * ld + (which * H + head) * 64, (short)0,
                                             n > 0 ? ((n - 1) * ld + 64) * 2 : 0, 0x00020000);
  };
  // values: two dims of eight keys an item, two items a thread
  unsigned vr[2][8];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const auto rv = rows(2, HG * hp + (HG == 2 ? j : 2 * j + (w >> 1)), ctx);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      vr[j][e] = __builtin_amdgcn_raw_buffer_load_b32(rv, ((8 * ((tid >> 5) & (4 * RW - 1)) + e) * ld + 2 * (tid & 31)) * 2, 0, 0);
  }
  const int head = w / RW, r0 = 32 * (w % RW);  // this wave's head of the group and its 32 rows
  bf16x8 qf[4], kf[RW][4];
  {
    const auto rq = rows(0, HG * hp + head, qlen), rk = rows(1, HG * hp + head, ctx);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      qf[t] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rq, ((r0 + (lane & 31)) * ld + 16 * t + 8 * h) * 2, 0, 0));
#pragma unroll
      for (int sub = 0; sub < RW; ++sub)
        kf[sub][t] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(rk, ((32 * sub + (lane & 31)) * ld + 16 * t + 8 * h) * 2, 0, 0));
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load is on its way
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        bf16x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = __builtin_bit_cast(bf16x2, vr[j][4 * i + e])[p];
        *reinterpret_cast<bf16x4*>(sv + (HG == 2 ? j : 2 * j + (w >> 1)) * Cfg::VBYTES +
                                   v_lds_off<64>(2 * (tid & 31) + p, 2 * ((tid >> 5) & (4 * RW - 1)) + i)) = x;
      }
  f32x16 s[2] = {f32x16{}, f32x16{}}, o[2] = {f32x16{}, f32x16{}};
  float l = 0.f;
  bf16x8 pf[2 * RW] = {};
  if (r0 < qlen && ctx > 0) {  // (without a key, the difference of two -1e30 is a rounding of any size)
#pragma unroll
    for (int sub = 0; sub < RW; ++sub)
#pragma unroll
      for (int t = 0; t < 4; ++t) s[sub] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[sub][t], qf[t], s[sub], 0, 0, 0);
    float m = kNeg;
    const float sl2 = scale * kLog2e;
#pragma unroll
    for (int sub = 0; sub < RW; ++sub)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[sub][r] = 32 * sub + (r & 3) + 8 * (r >> 2) < ctx - 4 * h ? s[sub][r] : kNeg;
        m = fmaxf(m, s[sub][r]);
      }
    m = max_halves(m) * sl2;
#pragma unroll
    for (int st = 0; st < 2 * RW; ++st)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float p = fexp2(fmaf(s[st >> 1][8 * (st & 1) + e], sl2, -m));
        l += p;
        pf[st][e] = (bf16)p;
      }
  }
  __syncthreads();
  if (r0 < qlen) {
#pragma unroll
    for (int st = 0; st < 2 * RW; ++st)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) {
        const bf16x8 vf = *reinterpret_cast<const bf16x8*>(sv + head * Cfg::VBYTES + v_lds_off<64>(32 * dt + (lane & 31), 4 * st + h));
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[st], o[dt], 0, 0, 0);
      }
    l = sum_halves(l);
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        bf16x4 x;
#pragma unroll
        for (int r = 0; r < 4; ++r) x[r] = (bf16)(o[dt][4 * c + r] * inv);
        *reinterpret_cast<bf16x4*>(so + (r0 + (lane & 31)) * OS + (head * 64 + 32 * dt + 8 * c + 4 * h) * 2) = x;
      }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2 * RW; ++i) {
    if (16 * i >= qlen) break;
    const int row = 16 * i + (lane & 15);
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < KS; ++k)
      a = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[k], *reinterpret_cast<const bf16x8*>(so + row * OS + k * 64 + (lane >> 4) * 16), a, 0, 0, 0);
    if (row < qlen) *reinterpret_cast<f32x4*>(ws + ((size_t)hp * M + qbeg + row) * N + nt * 16 + 4 * (lane >> 4)) = a;
  }
}
}  // namespace

// Heads a workgroup: slabs of the projection = H / that
int gai_attn_rows_heads(int H, int longest) { return H % 4 == 0 && longest <= 32 ? 4 : H % 2 == 0 && longest <= 64 ? 2 : 0; }

// ws: that many slabs of [M][N]; W row-major or in fragment order (the same bits), N % 64 == 0, no sequence longer than `longest`
void gai_attn_rows_slabs(const void* qkv, int ld, const int* cu_q, const int* ctx_lens, int seqs, int longest, const void* W, float* ws, int M,
                         int N, int H, float scale, int frag, hipStream_t st) {
  if (seqs == 0) return;
  const int hg = gai_attn_rows_heads(H, longest);
  if (!hg) gai_launch_error(__FILE__, __LINE__, "attn_rows_slabs: shape");
  const dim3 grid(N / 64, H / hg, seqs);
  if (hg == 4)
    attn_rows_slabs_kernel<4><<<grid, 256, 0, st>>>((const bf16*)qkv, ld, cu_q, ctx_lens, (const bf16*)W, ws, M, N, H, scale, frag);
  else
    attn_rows_slabs_kernel<2><<<grid, 256, 0, st>>>((const bf16*)qkv, ld, cu_q, ctx_lens, (const bf16*)W, ws, M, N, H, scale, frag);
  GAI_LAUNCH_CHECK();
}

int gai_attn_prefill_rows_per_tile(int Hq, int Hkv, int D) {
  const int ratio = Hq / Hkv;
  const int hpw = ratio >= 4 ? 4 : ratio >= 2 ? 2 : 1;
  return 32 * (prefill_waves(D, ratio) / (hpw / prefill_hl(D, ratio)));
}

void gai_attn_decode(const void* q, const void* k_cache, const void* v_cache, const int* block_tables,
                     int max_blocks, const int* ctx_lens, void* out, float* ws_o, float* ws_ml, int B, int Hq,
                     int Hkv, int D, float scale, int split_keys, int max_splits, int kv_fp8, float k_scale,
                     float v_scale, hipStream_t st, int* split_cnt, const GaiQkvFold* fold, bool queue) {
  if (B == 0) return;
  if (Hq / Hkv > 16) gai_launch_error(__FILE__, __LINE__, "attn_decode: GQA ratio > 16 unsupported");
  if (split_keys < 0 || split_keys % 128)
    gai_launch_error(__FILE__, __LINE__, "attn_decode: split_keys must be 0 (adaptive) or a multiple of 128");
  const dim3 grid(max_splits, Hkv, B);
  // GAI_DECODE_VARIANT: 0 = 8-B V^T pieces, 1 = 16-B V^T loads (default), 2 = 16-B + 64 keys per wave step,
  // 3 = 16-B + register double buffer (software pipelined)
  static const int variant = getenv("GAI_DECODE_VARIANT") ? atoi(getenv("GAI_DECODE_VARIANT")) : 1;
  // in-launch split merge (no attn_decode_reduce launch) when the caller passes the ticket counters
  const bool fuse = split_cnt != nullptr && max_splits > 1 && variant == 1;
  // non-temporal K / V loads in the fused bf16 kernel (GAI_DECODE_NT=0: plain loads). Llama-3-8B B = 64, ctx 2535
  // graph replay 7.84 -> 7.68 ms per step (profiles/r4/decode/decode_nt_split_ab.txt)
  static const bool ntl = !(getenv("GAI_DECODE_NT") && atoi(getenv("GAI_DECODE_NT")) == 0);
  if (fold != nullptr && !(fuse && ntl && !kv_fp8 && D == 128 && fold->ks >= 1 && fold->ks <= 16))
    gai_launch_error(__FILE__, __LINE__, "attn_decode: the folded QKV tail needs the fused non-temporal bf16 kernel");
  if (queue) {
    if (!(fuse && D == 128 && split_keys == 0 && B <= kQueueSeqs && (long long)B * max_splits < 1 << 22 && (kv_fp8 || ntl)))
      gai_launch_error(__FILE__, __LINE__, "attn_decode: the queue is of the fused adaptive form of head_dim 128");
    const GaiQkvFold f = fold ? *fold : GaiQkvFold{};
    const int wgs = (std::min(3 * decode_cus(), B * Hkv * max_splits) + 7) & ~7;  // resident: up to 168 VGPRs, 41 KB of LDS
#define GAI_QUEUE(KV, NT, QPF)                                                                                          \
  attn_decode_queue_kernel<128, KV, NT, QPF><<<wgs, 256, 0, st>>>(                                                       \
      (const bf16*)q, (const KV*)k_cache, (const KV*)v_cache, block_tables, max_blocks, ctx_lens, (bf16*)out, ws_o, ws_ml, B, \
      Hq, Hkv, scale, max_splits, k_scale, v_scale, split_cnt, f)
    if (fold) GAI_QUEUE(bf16, true, true);
    else if (kv_fp8) GAI_QUEUE(fp8, false, false);
    else GAI_QUEUE(bf16, true, false);
#undef GAI_QUEUE
    GAI_LAUNCH_CHECK();
    return;
  }
  if (fold != nullptr) {
    attn_decode_kernel<128, false, 1, true, bf16, true, true, true><<<grid, 256, 0, st>>>(
        (const bf16*)q, (const bf16*)k_cache, (const bf16*)v_cache, block_tables, max_blocks, ctx_lens, (bf16*)out,
        ws_o, ws_ml, B, Hq, Hkv, scale, split_keys, max_splits, k_scale, v_scale, split_cnt, *fold);
    GAI_LAUNCH_CHECK();
    return;
  }
#define GAI_DEC(DD)                                                                                             \
  if (D == DD && fuse && ntl && !kv_fp8) {                                                                      \
    attn_decode_kernel<DD, false, 1, true, bf16, true, true><<<grid, 256, 0, st>>>(                             \
        (const bf16*)q, (const bf16*)k_cache, (const bf16*)v_cache, block_tables, max_blocks, ctx_lens,         \
        (bf16*)out, ws_o, ws_ml, B, Hq, Hkv, scale, split_keys, max_splits, k_scale, v_scale, split_cnt);       \
    GAI_LAUNCH_CHECK();                                                                                         \
    return;                                                                                                     \
  }                                                                                                             \
  if (D == DD && fuse) {                                                                                        \
    if (kv_fp8)                                                                                                 \
      attn_decode_kernel<DD, false, 1, true, fp8, true><<<grid, 256, 0, st>>>(                                  \
          (const bf16*)q, (const fp8*)k_cache, (const fp8*)v_cache, block_tables, max_blocks, ctx_lens,         \
          (bf16*)out, ws_o, ws_ml, B, Hq, Hkv, scale, split_keys, max_splits, k_scale, v_scale, split_cnt);     \
    else                                                                                                        \
      attn_decode_kernel<DD, false, 1, true, bf16, true><<<grid, 256, 0, st>>>(                                 \
          (const bf16*)q, (const bf16*)k_cache, (const bf16*)v_cache, block_tables, max_blocks, ctx_lens,       \
          (bf16*)out, ws_o, ws_ml, B, Hq, Hkv, scale, split_keys, max_splits, k_scale, v_scale, split_cnt);     \
    GAI_LAUNCH_CHECK();                                                                                         \
    return;                                                                                                     \
  }                                                                                                             \
  if (D == DD) {                                                                                                \
    if (kv_fp8) {                                                                                               \
      auto kern = variant == 2   ? attn_decode_kernel<DD, false, 2, true, fp8>                                  \
                  : variant == 3 ? attn_decode_kernel<DD, true, 1, true, fp8>                                   \
                                 : attn_decode_kernel<DD, false, 1, true, fp8>;                                 \
      kern<<<grid, 256, 0, st>>>((const bf16*)q, (const fp8*)k_cache, (const fp8*)v_cache, block_tables,        \
                                 max_blocks, ctx_lens, (bf16*)out, ws_o, ws_ml, B, Hq, Hkv, scale, split_keys,   \
                                 max_splits, k_scale, v_scale, nullptr, GaiQkvFold{});                           \
    } else {                                                                                                    \
      auto kern = variant == 0   ? attn_decode_kernel<DD, false, 1, false, bf16>                                \
                  : variant == 2 ? attn_decode_kernel<DD, false, 2, true, bf16>                                 \
                  : variant == 3 ? attn_decode_kernel<DD, true, 1, true, bf16>                                  \
                                 : attn_decode_kernel<DD, false, 1, true, bf16>;                                \
      kern<<<grid, 256, 0, st>>>((const bf16*)q, (const bf16*)k_cache, (const bf16*)v_cache, block_tables,      \
                                 max_blocks, ctx_lens, (bf16*)out, ws_o, ws_ml, B, Hq, Hkv, scale, split_keys,   \
                                 max_splits, k_scale, v_scale, nullptr, GaiQkvFold{});                           \
    }                                                                                                           \
    GAI_LAUNCH_CHECK();                                                                                         \
    if (max_splits > 1) {                                                                                       \
      attn_decode_reduce_kernel<DD><<<dim3(B, Hq), DD, 0, st>>>(ws_o, ws_ml, ctx_lens, (bf16*)out, B, Hq,       \
                                                                 split_keys, max_splits);                       \
      GAI_LAUNCH_CHECK();                                                                                       \
    }                                                                                                           \
    return;                                                                                                     \
  }
  GAI_DEC(64)
  GAI_DEC(128)
  GAI_DEC(256)
#undef GAI_DEC
  gai_launch_error(__FILE__, __LINE__, "attn_decode: unsupported head_dim");
}
