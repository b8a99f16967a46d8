// bf16 GEMM for a few hundred rows (gemm_mid.hip): plan on the host, then the launch with the caller's workspace.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

constexpr int kGaiMidTickets = 16384;  // the most that a plan asks for
struct GaiMidPlan {
  int mt, ng, parts;  // rows / 16 and columns / 64 of a workgroup's tile, parts of K
  size_t ws_floats;   // fp32 workspace of the parts (0 for one part)
  double cost;        // modelled time, us
  int tickets = 0;    // of the parts: ints, 0 before a launch and 0 again after it
  bool ordered = false;  // every output is one sum over K in order, as in the 256 x 256 kernels (mt 4 or 8, one part)
};
// force 0: false where another kernel is expected to be faster; 14: this kernel, plan chosen; else 1000 mt + 100 ng +
// parts, 104201 / 108201: the ordered form
bool gai_gemm_mid_plan(const void* A, const void* B, const void* C, const void* bias, const void* R, int M, int N, int K,
                       int ldc, int epi, int out_f32, int force, int bfrag, GaiMidPlan* plan);
// ws and tickets of the plan for more than one part; any plan may be run with parts = 1 instead. Launches that may run side by
// side (streams, replays of captured ones) need tickets of their own.
void gai_gemm_mid(const void* A, const void* B, void* C, const void* bias, const void* R, int M, int N, int K, int ldc, int epi,
                  int out_f32, const GaiMidPlan& plan, float* ws, int* tickets, hipStream_t st, int bfrag);
// rows at the end of a large product that this kernel should compute instead of the 256 x 256 kernels' last, partly filled
// round of tiles (0: none), with the same sums; *plan is for those rows
int gai_gemm_mid_tail(const void* A, const void* B, const void* C, const void* bias, const void* R, int M, int N, int K, int ldc,
                      int epi, int out_f32, int bfrag, GaiMidPlan* plan);
// The same kernel's parts as fp32 slabs [parts][M][N] for a launch that adds them with what follows (a layer or rms norm): false where the
// product with its own sums and residual, and the norm, are expected to be faster. The plan is one for both layouts of the weight, rows
// on 16 bytes. most: the parts that launch takes.
bool gai_gemm_mid_slabs_plan(int M, int N, int K, int most, bool layer, GaiMidPlan* plan);
void gai_gemm_mid_slabs(const void* A, const void* B, int M, int N, int K, const GaiMidPlan& plan, float* ws, hipStream_t st,
                        int bfrag);
// a residual in front of a norm is faster added by the norm than by the product's epilogue
bool gai_gemm_residual_apart(int M, int N, int K);
