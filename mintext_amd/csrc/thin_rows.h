// The rows of one m-tile, found by the workgroup itself from group_sizes (the kernels for groups of
// few rows, which have no tile-list launch before them).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace mtx {

struct ThinRows {
  int e, r0, r1;  // group (-1: rows past the last group, -2: no such m-tile) and its rows [r0, r1)
};

// m-tiles: the groups in order, ceil(size / MT) each, then the rows past the last group.  Called by
// all NT threads of the workgroup; thread t scans the groups [t*per, (t+1)*per).  32-bit sums: at
// most 1024 groups, each clamped to M < 2^20 rows.
template <int MT, int NT>
__device__ __forceinline__ ThinRows thin_rows(const int32_t* __restrict__ gs, int E, int M, int mt) {
  constexpr int NW = NT / 64;
  __shared__ int s_tiles[NW], s_rows[NW], s_found[3];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per = (E + NT - 1) / NT;
  const int e0 = min(tid * per, E), e1 = min(e0 + per, E);
  int tiles = 0, rows = 0;
  for (int e = e0; e < e1; ++e) {
    const int g = min(max(gs[e], 0), M);
    tiles += (g + MT - 1) / MT;
    rows += g;
  }
  int ti = tiles, ri = rows;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int a = __shfl_up(ti, off), b = __shfl_up(ri, off);
    if (lane >= off) {
      ti += a;
      ri += b;
    }
  }
  if (lane == 63) {
    s_tiles[wave] = ti;
    s_rows[wave] = ri;
  }
  if (tid == 0) s_found[0] = -2;
  __syncthreads();
  int t0 = ti - tiles, r0 = ri - rows, tsum = 0, rsum = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const int a = s_tiles[w], b = s_rows[w];
    if (w < wave) {
      t0 += a;
      r0 += b;
    }
    tsum += a;
    rsum += b;
  }
  if (mt >= t0 && mt < t0 + tiles) {
    int t = t0, r = r0;
    for (int e = e0; e < e1; ++e) {
      const int g = min(max(gs[e], 0), M), n = (g + MT - 1) / MT;
      if (mt < t + n) {
        const int b = r + (mt - t) * MT;
        s_found[0] = e;
        s_found[1] = min(b, M);
        s_found[2] = min(min(b + MT, r + g), M);
        break;
      }
      t += n;
      r += g;
    }
  }
  if (tid == 0 && mt >= tsum) {
    const int b = min(rsum, M) + (mt - tsum) * MT;
    if (b < M) {
      s_found[0] = -1;
      s_found[1] = b;
      s_found[2] = min(b + MT, M);
    }
  }
  __syncthreads();
  const ThinRows t{s_found[0], s_found[1], s_found[2]};
  return t.e == -2 || t.r0 >= t.r1 ? ThinRows{-2, 0, 0} : t;
}

// A call that the few-row kernel may take: its m-tile rows (0: the call is not offered to it), its
// 128-column output tiles and the m-tiles its grid has room for.
struct FewRows {
  int mt, cols, max_tiles;
};

// Whether the few-row kernel is to take the call, from the group sizes: it streams the weights of a group
// once for each of its m-tiles, and needs enough of them to fill the chip.  Asked by the tile-list
// kernels (all 1024 threads, rows: of the thread's group), which then list no tiles; the few-row kernel,
// launched behind them, ends at once otherwise.  Where the rows are on a few groups the 256-row kernels
// are ahead by up to 4.7 times (256 groups of 7168 x 4096, 4096 rows on one of them: 955 / 203 us, on all: 2330
// / 2437); the choice costs the call one tile list and an empty launch, 5 to 8 us.
// The lines: 1.25 m-tiles a group (2 m-tiles a group lose up to 2 times, 1 never more than the few-row kernel
// does by itself), 192 column tiles of 256 CUs (128: 75 us here, 62 there for 256 rows on 8 of 32 groups, SwiGLU of
// 4096 x 4096), and a quarter of the grid's m-tiles in use (8 of 137: its empty workgroups take as long as the
// call, 24 us here, 14 there for 128 rows on one of 256 groups, fp8, 512 x 7168).
__device__ __forceinline__ bool few_rows_take(const FewRows& f, int rows) {
  __shared__ int s_tiles;
  if (f.mt == 0) return false;
  if (threadIdx.x == 0) s_tiles = 0;
  const int groups = __syncthreads_count(rows > 0);
  if (rows > 0) atomicAdd(&s_tiles, (rows + f.mt - 1) / f.mt);
  __syncthreads();
  const int t = s_tiles;
  return 4 * t <= 5 * groups && t * f.cols >= 192 && 4 * t >= f.max_tiles;
}

// m-tiles of MT rows that M rows in E groups can make: groups with rows, full tiles, the rest.
inline int64_t thin_max_tiles(int64_t M, int64_t E, int64_t MT) { return (E < M ? E : M) + M / MT + 1; }

}  // namespace mtx
