// Grouped GEMMs for groups of few rows: bf16 (gmm_thin.hip, called by the dispatch in gmm.hip) and
// blockwise fp8 (gmm_fp8_thin.hip, called by the one in fp8.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include "thin_rows.h"

namespace mtx {

// How a call of few rows per group goes: never to the few-row kernel, always, or by its group sizes
// (few_rows_take).
enum FewRowsMode { FEW_NEVER = 0, FEW_ALWAYS = 1, FEW_BY_SIZES = 2 };

struct ThinArgs {
  const uint16_t* A;     // x [M or gather_rows][Kred], bf16
  const uint16_t* W;     // [E][Kred][N]
  uint16_t* C;           // [M][N], or [M][I] with SwiGLU
  const int32_t* gs;     // [E] rows per group
  const int* take;       // 0 there: another kernel has the call; nullptr: this one has
  const int32_t* gather; // sorted row r reads A row gather[r] / gather_div; nullptr: row r
  int gather_div, gather_rows;
  int M, E, Kred, N;
  int I;                 // SwiGLU: N = 2 I, gate columns first; 0: plain store
  int fast_silu;         // SwiGLU with the hardware exp2 and reciprocal; 0: silu_f32
};

// Whether launch_gmm_thin takes M rows in E groups of Kred x N: widths in 16-byte chunks, 16-byte aligned
// operands (the caller checks), few rows per group on average; and for which group sizes it is to.
FewRowsMode gmm_thin_mode(int64_t M, int64_t E, int64_t Kred, int64_t N, int64_t I);
FewRows gmm_thin_rule(int64_t M, int64_t E, int64_t N, int64_t I);
int launch_gmm_thin(const ThinArgs& a, hipStream_t st);

struct Fp8ThinArgs {
  const uint8_t* xq;  // [M or gather_rows][K] e4m3
  const float* xs;    // [M or gather_rows][K/128]
  const uint8_t* wq;  // [E][N][K] e4m3
  const float* ws;    // [E][N/128][K/128]
  const int32_t* gs;
  const int* take;    // 0 there: another kernel has the call; nullptr: this one has
  uint16_t* out;      // plain: bf16 [M][N]; SwiGLU: bf16 [M][I] or nullptr
  uint8_t* outq;      // SwiGLU: e4m3 [M][I]
  float* outs;        // SwiGLU: [M][I/128]
  const int32_t* gather;
  int gather_div, gather_rows;
  int M, E, K, N;
  int I;              // SwiGLU: N = 2 I, gate rows first; 0: plain store
};

// For which group sizes launch_fp8_thin is the kernel for M rows in E groups of K x N (SwiGLU: N = 2 I).
FewRowsMode fp8_thin_mode(int64_t M, int64_t E, int64_t K, int64_t N, int64_t I);
FewRows fp8_thin_rule(int64_t M, int64_t E, int64_t N, int64_t I);
// p2: power-of-two scales (the MFMA's E8M0 operands); otherwise f32 scales.
int launch_fp8_thin(const Fp8ThinArgs& a, bool p2, hipStream_t st);

}  // namespace mtx
