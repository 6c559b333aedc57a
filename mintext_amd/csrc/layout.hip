// Expert weight layouts on gfx950: batched transpose-copy between HF's per-expert [out, in]
// weights and the fused [in, out] layout the grouped GEMMs read (bzantium/mintext
// mintext/checkpoint/conversion.py:80-166: _import_expert_weights / _export_expert_weights).
//
// out[b][c][r] = in[b][r][c] for r < R, c < C, with independent batch and row strides on both
// sides, so that one call writes the gate half and one the up half of a fused gate_up tensor
// (column offset = pointer offset, row stride 2I), or reads them back.  Element size 2 or 4
// bytes.  HBM-bound: 2 * B * R * C * elem bytes per call.
//
// Whole wave tiles (64x64 bf16, 32x32 f32; 16-byte aligned) of large calls turn in registers; the rest
// takes transpose_batched_kernel.  There a workgroup moves one 64x64 tile: 16-byte coalesced loads of 64 input rows into LDS, then
// 16-byte coalesced stores of 64 output rows read down the LDS columns (rows padded by one
// 16-byte chunk so that the column reads spread over the banks).  Tiles that are ragged or not
// 16-byte aligned take a per-element path.
#include "common.h"

namespace mtx {
namespace lay {

typedef __attribute__((ext_vector_type(4))) unsigned int u32x4;
constexpr int TILE = 64;

// 16 bytes from 8 bf16 / 4 f32 elements
__device__ __forceinline__ u32x4 pack16(const uint16_t (&v)[8]) {
  return u32x4{v[0] | ((uint32_t)v[1] << 16), v[2] | ((uint32_t)v[3] << 16), v[4] | ((uint32_t)v[5] << 16),
               v[6] | ((uint32_t)v[7] << 16)};
}
__device__ __forceinline__ u32x4 pack16(const float (&v)[4]) {
  return u32x4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])};
}

template <typename T>
__global__ __launch_bounds__(256) void transpose_batched_kernel(const T* __restrict__ in, int64_t R, int64_t C,
                                                                int64_t in_bs, int64_t in_ld, T* __restrict__ out,
                                                                int64_t out_bs, int64_t out_ld, int64_t tiles_c,
                                                                int vec_ok) {
  constexpr int EPC = 16 / sizeof(T);           // elements per 16-byte chunk
  constexpr int CPR = TILE / EPC;               // chunks per tile row
  constexpr int LD = TILE + EPC;                // padded LDS row (elements)
  __shared__ __attribute__((aligned(16))) T tile[TILE * LD];
  const int64_t b = blockIdx.z;
  const int64_t r0 = (int64_t)blockIdx.y * TILE, c0 = (int64_t)(blockIdx.x % tiles_c) * TILE;
  const T* src = in + b * in_bs;
  T* dst = out + b * out_bs;
  const bool full = vec_ok && r0 + TILE <= R && c0 + TILE <= C;
  if (full) {
    for (int q = threadIdx.x; q < TILE * CPR; q += blockDim.x) {
      const int r = q / CPR, ch = q % CPR;
      const u32x4 v = *(const u32x4*)(src + (r0 + r) * in_ld + c0 + ch * EPC);
      *(u32x4*)(tile + r * LD + ch * EPC) = v;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < TILE * CPR; q += blockDim.x) {
      const int c = q / CPR, ch = q % CPR;  // output row c (input column), chunk of input rows
      T v[EPC];
#pragma unroll
      for (int e = 0; e < EPC; ++e) v[e] = tile[(ch * EPC + e) * LD + c];
      *(u32x4*)(dst + (c0 + c) * out_ld + r0 + ch * EPC) = pack16(v);
    }
  } else {
    for (int q = threadIdx.x; q < TILE * TILE; q += blockDim.x) {
      const int r = q / TILE, c = q % TILE;
      if (r0 + r < R && c0 + c < C) tile[r * LD + c] = src[(r0 + r) * in_ld + c0 + c];
    }
    __syncthreads();
    for (int q = threadIdx.x; q < TILE * TILE; q += blockDim.x) {
      const int c = q / TILE, r = q % TILE;
      if (r0 + r < R && c0 + c < C) dst[(c0 + c) * out_ld + r0 + r] = tile[r * LD + c];
    }
  }
}

// Whole tiles through registers.  HBM-bound: a wave moves 64 x 64 bf16 (32 x 32 f32) as an 8 x 8 grid
// of lanes, each with an 8 x 8 (4 x 4) block.  Eight lanes load a 128-byte line of an input row and
// eight store one of an output row; the block turns in registers (byte permutes), so there is no LDS,
// no barrier, and all of a wave's loads are in flight at once.  Waves are numbered along the input's
// rows (512 contiguous bytes per workgroup) with none idle at a row's end.  Both sides bypass the
// caches, which data read and written once would only sweep.
// 64 x [1408, 2048] bf16 into rows of 2816: LDS tiles 148 us, this with 2 x 2 waves 138 (cached loads 140,
// cached stores 145), with four along a row 131 (5.6 TB/s; a plain copy reaches 5.9-6.1), down a column 150.
__device__ __forceinline__ void transpose_block(const u32x4 (&in)[8], u32x4 (&out)[8]) {
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
#pragma unroll
    for (int q = 0; q < 4; ++q) out[j][q] = __builtin_amdgcn_perm(in[2 * q + 1][j / 2], in[2 * q][j / 2], sel);
  }
}
__device__ __forceinline__ void transpose_block(const u32x4 (&in)[4], u32x4 (&out)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) out[j][q] = in[q][j];
}
template <typename T>
__global__ __launch_bounds__(256) void transpose_tiles_kernel(const T* __restrict__ in, int64_t in_bs, int64_t in_ld,
                                                              T* __restrict__ out, int64_t out_bs, int64_t out_ld,
                                                              int tiles_r, int tiles_c) {
  constexpr int B = 16 / (int)sizeof(T), WT = 8 * B;  // block and wave-tile side
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int id = blockIdx.x * 4 + wave;
  if (id >= tiles_r * tiles_c) return;
  const int64_t r = (int64_t)(id / tiles_c) * WT, c = (int64_t)(id % tiles_c) * WT;
  u32x4 v[B], w[B];
  const T* src = in + blockIdx.z * in_bs + (r + (lane >> 3) * B) * in_ld + c + (lane & 7) * B;
#pragma unroll
  for (int i = 0; i < B; ++i) v[i] = __builtin_nontemporal_load((const u32x4*)(src + i * in_ld));
  transpose_block(v, w);
  T* dst = out + blockIdx.z * out_bs + (c + (lane & 7) * B) * out_ld + r + (lane >> 3) * B;
#pragma unroll
  for (int j = 0; j < B; ++j) __builtin_nontemporal_store(w[j], (u32x4*)(dst + j * out_ld));
}

}  // namespace lay
}  // namespace mtx

using namespace mtx;

extern "C" int mtx_transpose_batched(const void* in, int dtype, int64_t B, int64_t R, int64_t C, int64_t in_batch_stride,
                                     int64_t in_ld, void* out, int64_t out_batch_stride, int64_t out_ld,
                                     void* stream) {
  if (dtype != MTX_F32 && dtype != MTX_BF16) return MTX_ERR_ARG;
  if (B < 0 || R < 0 || C < 0) return MTX_ERR_ARG;
  if (B == 0 || R == 0 || C == 0) return MTX_OK;
  if (!in || !out || in_ld < C || out_ld < R) return MTX_ERR_ARG;
  if (B > 65535 || ceil_div(R, lay::TILE) > 65535) return MTX_ERR_ARG;
  const int64_t es = dtype == MTX_F32 ? 4 : 2;
  const int64_t epc = 16 / es;
  const bool vec_ok = ((uintptr_t)in % 16 == 0) && ((uintptr_t)out % 16 == 0) && in_ld % epc == 0 &&
                      out_ld % epc == 0 && in_batch_stride % epc == 0 && out_batch_stride % epc == 0;
  const int64_t tiles_c = ceil_div(C, lay::TILE);
  if (tiles_c > INT32_MAX) return MTX_ERR_ARG;
  hipStream_t st = (hipStream_t)stream;
  // Whole tiles of 128 MB (half the memory-side cache) or more: streamed through registers.  Below that
  // the next reader finds the data in the cache, and the LDS tiles are ahead at most sizes.  A whole
  // import with its fp8 codes, bf16, E x D x I, us with LDS / register tiles: 36 x 768 x 768 (85 MB a
  // transpose) 88.8 / 95.9, 64 x 768 x 640 (126 MB) 121 / 130, 88 x 384 x 512 (69 MB) 75.5 / 79.0, but
  // 64 x 512 x 512 (67 MB) 72.5 / 69.9 and 8 x 1024 x 1024 (34 MB) 47.9 / 42.3; above the line
  // 64 x 1024 x 768 (201 MB) 221 / 196, 64 x 2048 x 1408 (738 MB) 744 / 685.
  const int64_t wt = 8 * epc, wtiles = ceil_div(R, wt) * ceil_div(C, wt);  // wave tiles
  if (vec_ok && R % wt == 0 && C % wt == 0 && wtiles <= INT32_MAX - 3 && 2 * B * R * C * es >= (int64_t)128 << 20) {
    dim3 tiles((unsigned)ceil_div(wtiles, 4), 1, (unsigned)B);
    if (dtype == MTX_F32)
      hipLaunchKernelGGL(lay::transpose_tiles_kernel<float>, tiles, dim3(256), 0, st, (const float*)in, in_batch_stride,
                         in_ld, (float*)out, out_batch_stride, out_ld, (int)(R / wt), (int)(C / wt));
    else
      hipLaunchKernelGGL(lay::transpose_tiles_kernel<uint16_t>, tiles, dim3(256), 0, st, (const uint16_t*)in,
                         in_batch_stride, in_ld, (uint16_t*)out, out_batch_stride, out_ld, (int)(R / wt), (int)(C / wt));
    return check_launch();
  }
  dim3 grid((unsigned)tiles_c, (unsigned)ceil_div(R, lay::TILE), (unsigned)B);
  if (dtype == MTX_F32)
    hipLaunchKernelGGL(lay::transpose_batched_kernel<float>, grid, dim3(256), 0, st, (const float*)in, R, C,
                       in_batch_stride, in_ld, (float*)out, out_batch_stride, out_ld, tiles_c, vec_ok ? 1 : 0);
  else
    hipLaunchKernelGGL(lay::transpose_batched_kernel<uint16_t>, grid, dim3(256), 0, st, (const uint16_t*)in, R, C,
                       in_batch_stride, in_ld, (uint16_t*)out, out_batch_stride, out_ld, tiles_c, vec_ok ? 1 : 0);
  return check_launch();
}
