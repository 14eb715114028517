// MFMA GEMM for the prompt (prefill) path: C = A * B^T with bf16 operands and
// fp32 accumulation on the gfx950 matrix cores.
//
//   A  bf16 [M, K] activations
//   B  Q4 weights in the MLX affine group-64 format, dequantised to
//      bf16(s*q + b) exactly as the reference's prefill QMM rounds them
//      (shaders/linear.metal:862-873), in the kernel or once into a prepared copy
//   C  bf16 [M, N]
//
// Every kernel runs v_mfma_f32_16x16x32_bf16 over k 32 i .. 32 i + 31 in order
// with one accumulator per output, so a row's bits do not depend on the kernel
// or the row tile a launch takes.
#pragma once

#include "common.hpp"

namespace prg {

enum GemmEpi : int {
  kGemmStore = 0,     // C = bf16(acc)
  kGemmResidual = 1,  // C = bf16(float(bf16(acc)) + res)          (linear.metal:932-937)
  kGemmSiluPair = 2,  // C = bf16(silu(bf16(acc_gate)) * bf16(acc_up)), two Q4 matrices
                      //     (qmm + silu_mul_pair_inplace_bf16, elementwise.metal:64-73)
};

constexpr int kGemmMaxSegs = 4;
struct GemmQ4 {
  const uint32_t* w = nullptr;  // u32 [n, K/8]
  const uint16_t* s = nullptr;  // bf16 [n, K/64]
  const uint16_t* b = nullptr;
  uint16_t* c = nullptr;        // bf16 [M, n]
  uint32_t n = 0;
  uint32_t tile0 = 0;           // first output tile of the segment (set by the launcher)
  // Optional prepared copy bf16 [n, K] = dequantised w (launch_dequant_dense).
  // When every segment has one, the kernel stages it instead of
  // dequantising per tile; the results are the same bit for bit.
  const uint16_t* dense = nullptr;
};

struct GemmArgs {
  // A: bf16, row m at a + m * lda
  const uint16_t* a = nullptr;
  uint64_t lda = 0;
  // B: up to 4 weight segments sharing A, each with its own output [M, n] (one
  // launch for projections that read the same activations). The SiLU pair
  // epilogue takes gate in q[0] and up in q[1] (same n, output q[0].c).
  GemmQ4 q[kGemmMaxSegs];
  uint32_t nq = 0;
  const uint16_t* res = nullptr;  // residual input [M, q[0].n]
  uint32_t M = 0, N = 0, K = 0;   // N: the segments' sum (set by the launcher)
};

// Q4 weights in g.q[0..nq). K % 64 == 0; A rows 16-byte aligned (lda % 8 == 0).
// The residual epilogue reads g.res [M, q[0].n].
int launch_gemm_q4(hipStream_t s, GemmArgs g, int epi, const char* name);
// Few activation rows (gemm_small.hip): the form that takes a launch in the
// least time on `cus` CUs and its cost in units of gemm_q4_kernel rows (tn 0 and
// ~0 when the kernel does not take it), and the launch of that form; g as
// launch_gemm_q4 has checked it.
struct GemmSmallPick {
  int tn = 0, mw = 0;  // 16-row weight tiles, 64-row activation tiles per block
  uint64_t cost = ~0ull;
};
GemmSmallPick gemm_small_pick(const GemmArgs& g, int epi, uint32_t cus);
int launch_gemm_small(hipStream_t s, const GemmArgs& g, int epi, const GemmSmallPick& pick, const char* name);
// Prepared bf16 copy out [n, K] of Q4 weights (w, sc, bi): the values the Q4
// GEMM dequantises per tile.
int launch_dequant_dense(hipStream_t s, const uint32_t* w, const uint16_t* sc, const uint16_t* bi, uint16_t* out,
                         uint32_t n, uint32_t K, const char* name);
}  // namespace prg
