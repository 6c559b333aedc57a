// bf16 grouped GEMM (forward, and forward + SwiGLU) for groups of few rows: decoding, where every
// expert of the batch has a handful of tokens and the time is that of streaming the weights once.
//
// The 256-row ring kernel (gmm.hip) reads W through LDS with one workgroup per CU and a tile per 256
// columns: 48 workgroups for one token of 8 experts of 2048 x 1536, which leaves most of the chip
// idle, behind a launch that builds the tile list.  Here a workgroup owns 128 columns of one group
// and its NW waves split the reduction: wave w takes the 32-k chunks w, w + NW, ... .  W goes from
// memory to registers (8 loads of 16 bytes per lane and chunk: 4 rows of 256 bytes each), the next
// chunk in flight while this one is used, and is turned into MFMA operands in registers (8x8
// transposes, 32 byte permutes per chunk).  No LDS and no barrier until the waves' partial sums are
// added, in wave order, so the result does not depend on timing.  Each workgroup finds its rows from
// group_sizes itself: no tile list, no launch before this one.
#include "common.h"
#include "gmm_thin.h"
#include "thin_rows.h"

namespace mtx {
namespace thin {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;

constexpr int BN = 128;        // W columns per wave
constexpr int KC = 32;         // reduction elements per chunk
constexpr int PADN = BN + 4;   // floats per token row of a wave's partial tile in LDS

// Column J of an 8x8 bf16 block whose row i is in[i]: eight k of one n, an MFMA operand.
template <int J>
__device__ __forceinline__ bf16x8 column(const u32x4 (&in)[8]) {
  constexpr uint32_t sel = (J & 1) ? 0x07060302u : 0x05040100u;
  u32x4 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = __builtin_amdgcn_perm(in[2 * q + 1][J / 2], in[2 * q][J / 2], sel);
  return __builtin_bit_cast(bf16x8, v);
}

// How a workgroup's columns map to its waves.  PLAIN: 128 columns, all waves.  NARROW: 64 gate and
// the matching 64 up columns, all waves.  WIDE: 128 gate columns in the first half of the waves, the
// matching 128 up columns in the second half; the reduction is split over half the waves.
enum { PLAIN = 0, NARROW = 1, WIDE = 2 };

// TB: 16-row blocks per m-tile; NW: waves per workgroup; STREAM: non-temporal loads of W.
template <int FORM, int TB, int NW, bool STREAM>
__global__ __launch_bounds__(NW * 64) void gmm_thin_kernel(ThinArgs p) {
  constexpr int MT = 16 * TB, NT = NW * 64;
  constexpr bool SWIGLU = FORM != PLAIN;
  constexpr int KW = FORM == WIDE ? NW / 2 : NW;  // waves that share a reduction
  __shared__ __attribute__((aligned(16))) float part[NW][16][PADN];
  if (p.take && *p.take == 0) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ocols = SWIGLU ? p.I : p.N;
  constexpr int OB = FORM == NARROW ? BN / 2 : BN;  // output columns per workgroup
  const int nn = (ocols + OB - 1) / OB;
  const int mt = blockIdx.x / nn, nt = blockIdx.x % nn;

  const ThinRows rows = thin_rows<MT, NT>(p.gs, p.E, p.M, mt);
  const int e = rows.e, r0 = rows.r0, r1 = rows.r1;
  if (e == -2) return;
  if (e < 0) {
    for (int i = tid; i < MT * OB; i += NT) {
      const int r = r0 + i / OB, c = nt * OB + i % OB;
      if (r < r1 && c < ocols) p.C[(int64_t)r * ocols + c] = 0;
    }
    return;
  }
  const int nb = (r1 - r0 + 15) >> 4;  // 16-row blocks with rows

  // ---- lane's sources: W columns col .. col+7 of k rows 8*kq .. 8*kq+7 of a chunk (columns past the
  // end re-read the last chunk of the row and are not stored), x rows of the lane's tokens
  const int l16 = lane & 15, kq = lane >> 4;
  int col;
  const int kw = FORM == WIDE ? wave % KW : wave;
  if (FORM == NARROW) col = (l16 < 8 ? 0 : p.I) + min(nt * 64 + (l16 & 7) * 8, p.I - 8);
  else if (FORM == WIDE) col = (wave < KW ? 0 : p.I) + min(nt * BN + l16 * 8, p.I - 8);
  else col = min(nt * BN + l16 * 8, p.N - 8);
  const uint16_t* We = p.W + (int64_t)e * p.Kred * p.N;
  const uint16_t* xr[TB];
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    int r = min(r0 + b * 16 + l16, r1 - 1);
    if (p.gather) r = min(max(p.gather[r], 0) / p.gather_div, p.gather_rows - 1);
    xr[b] = p.A + (int64_t)r * p.Kred;
  }
  const int nk = (p.Kred + KC - 1) / KC;

  // a chunk's operands: the 8-k part of lane group kq is past the end in a short last chunk; it
  // re-reads the last one and is zeroed in both operands at its use
  struct Chunk {
    u32x4 w[8];
    u32x4 x[TB];
  };
  auto load = [&](Chunk& c, int ck) {
    const int k = min(ck * KC + kq * 8, p.Kred - 8);
    const uint16_t* wp = We + (int64_t)k * p.N + col;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const u32x4* q = (const u32x4*)(wp + (int64_t)i * p.N);
      c.w[i] = STREAM ? __builtin_nontemporal_load(q) : *q;
    }
#pragma unroll
    for (int b = 0; b < TB; ++b)
      if (b < nb) c.x[b] = *(const u32x4*)(xr[b] + k);
  };
  f32x4 acc[8][TB];
#pragma unroll
  for (int f = 0; f < 8; ++f)
#pragma unroll
    for (int b = 0; b < TB; ++b) acc[f][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto use = [&](Chunk& c, int ck) {
    if (ck * KC + KC > p.Kred) {
      const uint32_t keep = ck * KC + kq * 8 < p.Kred ? 0xFFFFFFFFu : 0u;
#pragma unroll
      for (int i = 0; i < 8; ++i) c.w[i] &= keep;
#pragma unroll
      for (int b = 0; b < TB; ++b) c.x[b] &= keep;
    }
    bf16x8 wf[8] = {column<0>(c.w), column<1>(c.w), column<2>(c.w), column<3>(c.w),
                    column<4>(c.w), column<5>(c.w), column<6>(c.w), column<7>(c.w)};
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      if (b >= nb) continue;
      const bf16x8 xf = __builtin_bit_cast(bf16x8, c.x[b]);
#pragma unroll
      for (int f = 0; f < 8; ++f) acc[f][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[f], xf, acc[f][b], 0, 0, 0);
    }
  };
  {
    Chunk c0, c1;
#pragma unroll
    for (int b = 0; b < TB; ++b) c0.x[b] = c1.x[b] = u32x4{0u, 0u, 0u, 0u};
    // the loop's loads are unconditional, so that the waits count them; the last one or two chunks follow
    if (kw < nk) load(c0, kw);
    int ck = kw;
    for (; ck + 2 * KW < nk; ck += 2 * KW) {
      load(c1, ck + KW);
      use(c0, ck);
      load(c0, ck + 2 * KW);
      use(c1, ck + KW);
    }
    if (ck + KW < nk) {
      load(c1, ck + KW);
      use(c0, ck);
      use(c1, ck + KW);
    } else if (ck < nk) {
      use(c0, ck);
    }
  }

  // ---- add the waves' partial tiles, 16 rows at a time.  acc[f][b][r] of lane l is the output of token
  // 16 b + l % 16 at workgroup column 8 (4 (l / 16) + r) + f: eight consecutive columns over f.
#pragma unroll
  for (int b = 0; b < TB; ++b) {
    if (b >= nb) break;
    if (b > 0) __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float* o = &part[wave][l16][8 * (4 * kq + r)];
      *(f32x4*)o = f32x4{acc[0][b][r], acc[1][b][r], acc[2][b][r], acc[3][b][r]};
      *(f32x4*)(o + 4) = f32x4{acc[4][b][r], acc[5][b][r], acc[6][b][r], acc[7][b][r]};
    }
    __syncthreads();
    auto sum4 = [&](int w0, int tok, int c) {
      f32x4 v = *(const f32x4*)&part[w0][tok][c];
#pragma unroll
      for (int w = 1; w < KW; ++w) v += *(const f32x4*)&part[w0 + w][tok][c];
      return v;
    };
    for (int i = tid; i < 16 * OB / 4; i += NT) {
      const int tok = i / (OB / 4), c = (i % (OB / 4)) * 4;
      const int row = r0 + b * 16 + tok, oc = nt * OB + c;
      if (row >= r1 || oc >= ocols) continue;
      f32x4 v = sum4(0, tok, c);
      if (SWIGLU) {
        const f32x4 u = FORM == WIDE ? sum4(KW, tok, c) : sum4(0, tok, 64 + c);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = p.fast_silu ? swiglu_fast(v[q], u[q]) : silu_f32(v[q]) * u[q];
      }
      *(bf16x4*)(p.C + (int64_t)row * ocols + oc) = bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
    }
  }
}

template <int FORM, int TB, int NW>
static int launch(const ThinArgs& a, int64_t grid, bool stream, hipStream_t st) {
  if (stream)
    hipLaunchKernelGGL((gmm_thin_kernel<FORM, TB, NW, true>), dim3((unsigned)grid), dim3(NW * 64), 0, st, a);
  else
    hipLaunchKernelGGL((gmm_thin_kernel<FORM, TB, NW, false>), dim3((unsigned)grid), dim3(NW * 64), 0, st, a);
  return check_launch();
}

}  // namespace thin

// Up to 16 rows per group on average.  128 groups, 2048 x 1536 with SwiGLU / 768 x 2048, us here and
// in the ring kernel: 8 rows 12.3 / 35.0 and 7.8 / 27.6, 512 rows 116 / 141 and 63 / 118 (6.7 and 6.2
// TB/s), 2048 rows (a mean of 16) 129 / 147 and 79 / 119, the same with Zipf loads 154 / 158 and
// 77 / 124, but 6144 rows 251 / 155: groups then outgrow the m-tile of 32 rows and stream their
// weights again.  8 groups, 4096 x 2*14336 and 14336 x 4096: 74 rows 306 / 344 and 144 / 226, 400 rows
// 525 / 372.
constexpr int64_t kThinMaxMean = 16;

static int64_t thin_mt(int64_t M, int64_t E) { return M <= 2 * E ? 16 : 32; }

// Without a look at the group sizes it takes the calls in which it is ahead wherever the rows are: up to 16
// rows (an m-tile for each group), and short reductions while the output is small, where even all rows in
// one group stream little (2^19 outputs, SwiGLU 2^18 gate and up columns; uniform / all on one group against
// the ring kernel, us: 256 groups, 4096 x 4096 plain, 128 rows 520 / 604 and 26 / 47, but 512 rows on two groups
// 109 / 74).  A plain store's reduction past 4096 is split over the chip by the ring kernel, which then leads
// when few groups have rows (8 groups, 14336 x 4096, 32 rows on one 109 / 79, on all 147 / 228).
// Elsewhere the group sizes decide, where that costs little beside what it can gain: not on a SwiGLU of
// less than 128 MB of weights (32 groups, 512 x 1536, 512 rows 24 / 20), nor with short reductions in a large
// grid, whose workgroups all end at once if the ring kernel has the call (256 groups, 512 x 7168, 256 rows on
// one 25 / 20), nor on a long plain reduction that fills the chip in the ring kernel too (32 groups,
// 14336 x 4096, 64 rows 540 / 501).
FewRowsMode gmm_thin_mode(int64_t M, int64_t E, int64_t Kred, int64_t N, int64_t I) {
  if (M < 1 || M >= (1 << 20) || E < 1 || E > 1024) return FEW_NEVER;
  if (Kred < 8 || Kred % 8 || N < 8 || N % 8 || I % 8) return FEW_NEVER;
  if (M > E * kThinMaxMean) return FEW_NEVER;
  if (M <= 16 && (I > 0 || Kred <= 8192)) return FEW_ALWAYS;
  if (Kred <= 4096 && M * N <= (I > 0 ? 1 << 18 : 1 << 19)) return FEW_ALWAYS;
  const FewRows r = gmm_thin_rule(M, E, N, I);
  const int64_t groups = E < M ? E : M;
  if (groups * r.cols < 192) return FEW_NEVER;
  if (I > 0 && groups * Kred * N * 2 < (int64_t)128 << 20) return FEW_NEVER;
  if (Kred < 2048 && (int64_t)r.max_tiles * r.cols > 4096) return FEW_NEVER;
  if (I == 0 && Kred > 8192 && groups * r.cols > 256) return FEW_NEVER;
  return FEW_BY_SIZES;
}

FewRows gmm_thin_rule(int64_t M, int64_t E, int64_t N, int64_t I) {
  const int64_t mt = thin_mt(M, E);
  return {(int)mt, (int)ceil_div(I > 0 ? I : N, 128), (int)thin_max_tiles(M, E, mt)};
}

int launch_gmm_thin(const ThinArgs& a, hipStream_t st) {
  // rows per m-tile: 16 when the groups hold a row or two on average, else 32
  const int64_t MT = thin_mt(a.M, a.E);
  const int64_t mtiles = thin_max_tiles(a.M, a.E, MT);
  const int64_t bytes = mtiles * a.Kred * a.N * 2;                   // of weights, at most
  // Half the 256 MB memory-side cache or more: nothing of the weights is found there again by the
  // time they are next used, and loads that do not allocate in it run at 6.2-6.7 TB/s instead of
  // 5.2-5.9 (512 rows of 128 groups, 2048 x 1536: 132 -> 121 us).  Below that the plain loads keep
  // what does fit (8 rows: 12.6 against 18.1 us).
  const bool stream = bytes >= (int64_t)128 << 20;
  // SwiGLU: 256-byte row pieces of W instead of 128-byte ones (74 rows of 8 groups, 4096 x 2*14336:
  // 335 -> 306 us), once that leaves enough to do for each wave (64 rows of 128 groups, 2048 x 1536, 69
  // m-tiles, 434 MB: 66 against 59 us; 2 rows of 8 groups of 4096 x 28672, 705 MB: 77 against 90)
  const bool wide = a.I > 0 && bytes >= (int64_t)512 << 20;
  const int64_t nn = wide ? ceil_div(a.I, 128) : a.I > 0 ? ceil_div(a.I, 64) : ceil_div(a.N, 128);
  const int64_t grid = mtiles * nn;
  // few workgroups: eight waves in each instead of four, so that more of the chip's loads are in
  // flight (64 rows of 128 groups, 768 x 2048, 1104 workgroups: 35 us with eight, 31 with four)
  const bool eight = grid < 768;
#define MTX_THIN(F)                                                                                              \
  (MT == 16 ? (eight ? thin::launch<F, 1, 8>(a, grid, stream, st) : thin::launch<F, 1, 4>(a, grid, stream, st))  \
            : (eight ? thin::launch<F, 2, 8>(a, grid, stream, st) : thin::launch<F, 2, 4>(a, grid, stream, st)))
  return wide ? MTX_THIN(thin::WIDE) : a.I > 0 ? MTX_THIN(thin::NARROW) : MTX_THIN(thin::PLAIN);
#undef MTX_THIN
}

}  // namespace mtx
