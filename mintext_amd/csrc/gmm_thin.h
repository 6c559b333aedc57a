// Grouped GEMM for groups of few rows (gmm_thin.hip); called by the dispatch in gmm.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace mtx {

struct ThinArgs {
  const uint16_t* A;     // x [M or gather_rows][Kred], bf16
  const uint16_t* W;     // [E][Kred][N]
  uint16_t* C;           // [M][N], or [M][I] with SwiGLU
  const int32_t* gs;     // [E] rows per group
  const int32_t* gather; // sorted row r reads A row gather[r] / gather_div; nullptr: row r
  int gather_div, gather_rows;
  int M, E, Kred, N;
  int I;                 // SwiGLU: N = 2 I, gate columns first; 0: plain store
};

// Whether launch_gmm_thin takes (and is the faster kernel for) M rows in E groups of Kred x N: widths
// in 16-byte chunks, 16-byte aligned operands (the caller checks), few rows per group on average.
bool gmm_thin_ok(int64_t M, int64_t E, int64_t Kred, int64_t N, int64_t I);
int launch_gmm_thin(const ThinArgs& a, hipStream_t st);

}  // namespace mtx
