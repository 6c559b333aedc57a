// Blockwise-fp8 grouped GEMM (plain bf16 store, or SwiGLU + 1x128 re-quantisation) for groups of few
// rows, where the time is that of streaming the weights once (decoding).
//
// The persistent 256-row kernel (fp8.hip) walks 256-column tiles through an LDS ring with one
// workgroup per CU; with few rows that reached 3.7-4.1 TB/s of weights.  Here a workgroup owns 128
// output columns of one group (SwiGLU: their 128 gate and 128 up rows of W), i.e. contiguous rows of the
// k-contiguous codes.  Its eight waves are four column quarters times two halves of the reduction
// (128-k chunks in turn); W and the tokens go from memory to registers, as the MFMA's operands
// without any rearrangement, two chunks in flight.  The two halves are added through LDS at the end.
// Each 128-k chunk is one v_mfma_scale_f32_16x16x128_f8f6f4 per 16 columns and 16 rows, whose block
// scales are its E8M0 operands in the power-of-two mode; with f32 scales the chunk's product is
// formed with unit scales and added to the accumulator with one FMA per value.
#include "common.h"
#include "gmm_thin.h"
#include "thin_rows.h"

namespace mtx {
namespace f8thin {

typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
typedef __attribute__((ext_vector_type(8))) int i32x8;

constexpr int KC = 128;           // reduction elements per chunk: one scale block
constexpr int KW = 2, CW = 4;     // waves along the reduction, along the columns
constexpr int NT = KW * CW * 64;

__device__ __forceinline__ i32x8 join(const u32x4& lo, const u32x4& hi) {
  return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
}

// TB: 16-row blocks per m-tile.  W by plain loads: each 128-byte line is read by two loads, the second
// of which hits in the L1, where a non-temporal line is not kept (488 rows, 2048 x 1536: 107 us).
template <bool SWIGLU, bool P2, int TB>
__global__ __launch_bounds__(NT) void gmm_fp8_thin_kernel(Fp8ThinArgs p) {
  constexpr int MT = 16 * TB;
  constexpr int NB = SWIGLU ? 4 : 2;   // 16-row blocks of W per wave (SwiGLU: two gate, two up)
  constexpr int NS = SWIGLU ? 2 : 1;   // weight-scale blocks per chunk
  __shared__ __attribute__((aligned(16))) f32x4 part[CW][NB * TB][64];
  __shared__ float s_amax[MT][CW];
  if (p.take && *p.take == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wave / CW, cw = wave % CW;
  const int l16 = lane & 15, kq = lane >> 4;
  const int nn = (SWIGLU ? p.I : p.N) / 128, nkb = p.K / KC;
  const int mt = blockIdx.x / nn, nt = blockIdx.x % nn;
  const ThinRows rows = thin_rows<MT, NT>(p.gs, p.E, p.M, mt);
  const int e = rows.e, r0 = rows.r0, r1 = rows.r1;
  if (e == -2) return;
  if (e < 0) {  // rows of no group: zeros (codes 0 with scale 1, as the quantisers give)
    for (int i = tid; i < MT * 128; i += NT) {
      const int r = r0 + i / 128, c = nt * 128 + i % 128;
      if (r >= r1) continue;
      if (SWIGLU) {
        p.outq[(int64_t)r * p.I + c] = 0;
        if (p.out) p.out[(int64_t)r * p.I + c] = 0;
        if (i % 128 == 0) p.outs[(int64_t)r * nn + nt] = 1.0f;
      } else {
        p.out[(int64_t)r * p.N + c] = 0;
      }
    }
    return;
  }
  const int nb = (r1 - r0 + 15) >> 4;  // 16-row blocks with rows

  // Lane l holds, of row l % 16 of each block, bytes [16 kq, 16 kq + 16) of both halves of a chunk's
  // 128: the same bytes for W and x, so each MFMA lane position is one k of both.
  const uint8_t* we = p.wq + (int64_t)e * p.N * p.K + kq * 16;
  const uint8_t* wr[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int half = SWIGLU ? j / 2 : 0, jj = SWIGLU ? j % 2 : j;
    wr[j] = we + (int64_t)(half * p.I + nt * 128 + cw * 32 + jj * 16 + l16) * p.K;
  }
  const uint8_t* xr[TB];
  const float* xsr[TB];
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    int r = min(r0 + b * 16 + l16, r1 - 1);
    if (p.gather) r = min(max(p.gather[r], 0) / p.gather_div, p.gather_rows - 1);
    xr[b] = p.xq + (int64_t)r * p.K + kq * 16;
    xsr[b] = p.xs + (int64_t)r * nkb;
  }
  const float* wsr[NS];
#pragma unroll
  for (int h = 0; h < NS; ++h) wsr[h] = p.ws + ((int64_t)e * (p.N / 128) + h * (p.I / 128) + nt) * nkb;

  struct Chunk {
    u32x4 w[NB][2], x[TB][2];
    float xs[TB], ws[NS];
  };
  auto load = [&](Chunk& c, int ck) {
    const int k = ck * KC;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) c.w[j][h] = *(const u32x4*)(wr[j] + k + h * 64);
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      if (b >= nb) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) c.x[b][h] = *(const u32x4*)(xr[b] + k + h * 64);
      c.xs[b] = xsr[b][ck];
    }
#pragma unroll
    for (int h = 0; h < NS; ++h) c.ws[h] = wsr[h][ck];
  };
  f32x4 acc[NB][TB];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[j][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto use = [&](const Chunk& c) {
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      if (b >= nb) continue;
      const i32x8 xf = join(c.x[b][0], c.x[b][1]);
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const i32x8 wf = join(c.w[j][0], c.w[j][1]);
        const float ws = c.ws[SWIGLU ? j / 2 : 0];
        if constexpr (P2) {
          acc[j][b] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, xf, acc[j][b], 0, 0, 0, (int)e8m0_of(ws), 0,
                                                                       (int)e8m0_of(c.xs[b]));
        } else {
          const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
          const f32x4 v = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, xf, z, 0, 0, 0, 127, 0, 127);
          const float s = ws * c.xs[b];
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[j][b][q] = __builtin_fmaf(v[q], s, acc[j][b][q]);
        }
      }
    }
  };
  {
    Chunk c0, c1;
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      c0.x[b][0] = c0.x[b][1] = c1.x[b][0] = c1.x[b][1] = u32x4{0u, 0u, 0u, 0u};
      c0.xs[b] = c1.xs[b] = 0.0f;
    }
    // the loop's loads are unconditional, so that the waits count them; the last one or two chunks follow
    if (kw < nkb) load(c0, kw);
    int ck = kw;
    for (; ck + 2 * KW < nkb; ck += 2 * KW) {
      load(c1, ck + KW);
      use(c0);
      load(c0, ck + 2 * KW);
      use(c1);
    }
    if (ck + KW < nkb) {
      load(c1, ck + KW);
      use(c0);
      use(c1);
    } else if (ck < nkb) {
      use(c0);
    }
  }

  // ---- add the second half's sums, then the epilogue in the first half's waves.  acc[j][b][q] of lane l
  // is row 16 b + l % 16, column 16 j' + 4 (l / 16) + q of the wave's quarter.
  if (kw == 1) {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int b = 0; b < TB; ++b) part[cw][j * TB + b][lane] = acc[j][b];
  }
  __syncthreads();
  if (kw == 0) {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int b = 0; b < TB; ++b) acc[j][b] += part[cw][j * TB + b][lane];
  }
  if constexpr (!SWIGLU) {
    if (kw != 0) return;
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      const int row = r0 + b * 16 + l16;
      if (row >= r1) continue;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const f32x4 v = acc[j][b];
        *(bf16x4*)(p.out + (int64_t)row * p.N + nt * 128 + cw * 32 + j * 16 + 4 * kq) =
            bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
      }
    }
  } else {
    f32x4 y[2][TB];
    if (kw == 0) {
#pragma unroll
      for (int b = 0; b < TB; ++b) {
        float m = 0.0f;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            y[j][b][q] = swiglu_fast(acc[j][b][q], acc[2 + j][b][q]);
            m = fmaxf(m, fabsf(y[j][b][q]));
          }
        m = fmaxf(m, __shfl_xor(m, 16));
        m = fmaxf(m, __shfl_xor(m, 32));
        if (kq == 0) s_amax[b * 16 + l16][cw] = m;
      }
    }
    __syncthreads();
    if (kw != 0) return;
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      const int row = r0 + b * 16 + l16;
      const float* mx = s_amax[b * 16 + l16];
      const float amax = fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]));
      // the scale and the multiply by its reciprocal of the 256-row kernels
      float sc, inv;
      if constexpr (P2) {
        sc = p2_scale(amax);
        inv = __builtin_amdgcn_ldexpf(1.0f, 127 - (int)e8m0_of(sc));
      } else {
        sc = amax / 448.0f;
        if (sc == 0.0f) sc = 1.0f;
        inv = 1.0f / sc;
      }
      if (row >= r1) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const f32x4 v = y[j][b];
        const int64_t o = (int64_t)row * p.I + nt * 128 + cw * 32 + j * 16 + 4 * kq;
        *(uint32_t*)(p.outq + o) = e4m3_pack4(v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv);
        if (p.out) *(bf16x4*)(p.out + o) = bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
      }
      if (cw == 0 && kq == 0) p.outs[(int64_t)row * nn + nt] = sc;
    }
  }
}

template <bool SWIGLU, bool P2, int TB>
static int launch(const Fp8ThinArgs& a, int64_t grid, hipStream_t st) {
  hipLaunchKernelGGL((gmm_fp8_thin_kernel<SWIGLU, P2, TB>), dim3((unsigned)grid), dim3(NT), 0, st, a);
  return check_launch();
}

}  // namespace f8thin

// Up to 12 rows per group on average.  128 groups, 2048 x 2*768 with SwiGLU and 768 x 2048, us here
// and in the 256-row kernel: 8 rows 19.5 / 30.8 and 6.8 / 16.6, 488 rows 73 / 107 and 41 / 61 (5.4 and
// 4.7 TB/s of weights), 1024 rows x 2048 x 1536 plain 77 / 109.  At 2048 rows, a mean of 16, popular
// groups take several m-tiles: 2048 x 1536 plain with Zipf loads 107 / 104 (uniform 97 / 112); at 4096
// rows the 256-row kernel is ahead, 110 against about 200.
constexpr int64_t kFp8ThinMaxMean = 12;

static int64_t fp8_thin_mt(int64_t M, int64_t E) { return M <= 2 * E ? 16 : 32; }

// Up to 2^19 outputs (SwiGLU: gate and up columns) it is ahead wherever the rows are, or within 6 % (128
// groups, 768 x 2048, 256 rows uniform / all on one group: 32 / 56 us and 11 / 17 here / there).  Beyond, the
// group sizes decide (256 groups, 512 x 4096, 256 rows on one group 27 / 14, uniform 70 / 104), but not with
// short reductions in a large grid, whose workgroups all end at once if the other kernel has the call
// (256 groups, 512 x 7168, 256 rows on one 23 / 15).
FewRowsMode fp8_thin_mode(int64_t M, int64_t E, int64_t K, int64_t N, int64_t I) {
  if (!(M >= 1 && M < (1 << 20) && E >= 1 && E <= 1024 && M <= E * kFp8ThinMaxMean)) return FEW_NEVER;
  if (M * N <= 1 << 19) return FEW_ALWAYS;
  const FewRows r = fp8_thin_rule(M, E, N, I);
  if ((E < M ? E : M) * r.cols < 192) return FEW_NEVER;
  return K < 2048 && (int64_t)r.max_tiles * r.cols > 4096 ? FEW_NEVER : FEW_BY_SIZES;
}

FewRows fp8_thin_rule(int64_t M, int64_t E, int64_t N, int64_t I) {
  const int64_t mt = fp8_thin_mt(M, E);
  return {(int)mt, (int)((I > 0 ? I : N) / 128), (int)thin_max_tiles(M, E, mt)};
}

int launch_fp8_thin(const Fp8ThinArgs& a, bool p2, hipStream_t st) {
  const int64_t MT = fp8_thin_mt(a.M, a.E);
  const int64_t mtiles = thin_max_tiles(a.M, a.E, MT);
  const int64_t grid = mtiles * ((a.I > 0 ? a.I : a.N) / 128);
#define MTX_F8THIN(S, P) (MT == 16 ? f8thin::launch<S, P, 1>(a, grid, st) : f8thin::launch<S, P, 2>(a, grid, st))
  if (a.I > 0) return p2 ? MTX_F8THIN(true, true) : MTX_F8THIN(true, false);
  return p2 ? MTX_F8THIN(false, true) : MTX_F8THIN(false, false);
#undef MTX_F8THIN
}

}  // namespace mtx
