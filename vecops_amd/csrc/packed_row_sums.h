// Sums over the rows of an int8 operand packed by launch_pack_b: the correction terms of unsigned and runtime-quantised
// activations.
#pragma once
#include "row_work_split.h"
#include "tile_gemm.h"
#include "tile_gemm_packed.h"

namespace vecops_hip {

// out[b * n + row] = scale * sum_k B[row,k] (+ add[b * add_bs + row], add may be null) for b < batch, wrapping.
struct PackedRowSums {
  const void* packed;
  int32_t n, k, batch;
  uint32_t scale;
  const int32_t* add;
  int64_t add_bs;
  int32_t* out;
};

__host__ __device__ inline int64_t packed_row_sums_blocks(const PackedRowSums& a) {
  return a.n <= 0 || a.batch <= 0 ? 0 : packed_sums_blocks(a.n, a.k);
}

__device__ __forceinline__ void add_signed_bytes(int32_t& sum, const u32x4& v) {
#pragma unroll
  for (int w = 0; w < 4; ++w) sum = __builtin_amdgcn_sdot4(static_cast<int32_t>(v[w]), 0x01010101, sum, false);
}

__device__ __forceinline__ void packed_row_sum_out(const PackedRowSums& a, int64_t row, int32_t sum) {
  const uint32_t total = static_cast<uint32_t>(sum) * a.scale;
  for (int32_t b = 0; b < a.batch; ++b)
    a.out[static_cast<int64_t>(b) * a.n + row] = static_cast<int32_t>(total + (a.add ? static_cast<uint32_t>(a.add[b * a.add_bs + row]) : 0u));
}

// Both bound by reading the packed bytes once.
// Few panels: a workgroup of 256 lanes takes eight rows - a quarter of a panel, the 128 contiguous bytes a k-half holds of
// them - and walks 32 k-halves a step, four steps in flight; a wavefront a panel left 4096 x 4096 to 128 wavefronts that
// each walked 128 KiB one load after the other (40.7 us, behind a quantisation of 7.4; the 512 workgroups of the quarters in
// one launch with the quantisation of 1000 x 4096 fp32 elements: 7.9 us for both, 4.7 TB/s).
// (block: the workgroup's number among packed_row_sums_blocks; 256 lanes)
__device__ __forceinline__ void packed_row_sums_by_quarter(const PackedRowSums& a, uint32_t block) {
  __shared__ int32_t wave_sums[4][8];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row_in = threadIdx.x & 7, slot = threadIdx.x >> 3;      // 8 rows x 32 k-halves
  const int64_t halves = packed_k_steps(a.k, 16) * 2;               // k-halves of a panel: 32 rows x 16 bytes each
  const uint32_t panel = block >> 2, quarter = block & 3;
  const u32x4* src = static_cast<const u32x4*>(a.packed) + panel * halves * 32 + quarter * 8 + row_in;
  int32_t sum = 0;
  int64_t h = slot;
  for (; h + 96 < halves; h += 128) {
    u32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = src[(h + i * 32) * 32];
#pragma unroll
    for (int i = 0; i < 4; ++i) add_signed_bytes(sum, v[i]);
  }
  for (; h < halves; h += 32) add_signed_bytes(sum, src[h * 32]);
#pragma unroll
  for (int off = 8; off < 64; off <<= 1) sum += __shfl_xor(sum, off, 64);
  if (lane < 8) wave_sums[wave][lane] = sum;
  __syncthreads();
  const int64_t row = static_cast<int64_t>(block) * 8 + threadIdx.x;
  if (threadIdx.x < 8 && row < a.n)
    packed_row_sum_out(a, row, wave_sums[0][threadIdx.x] + wave_sums[1][threadIdx.x] + wave_sums[2][threadIdx.x] + wave_sums[3][threadIdx.x]);
}

// Many panels: a wavefront takes one and walks its k-steps as one contiguous stream, four in flight; lanes l and l + 32 hold
// the two halves of a row.  (A workgroup for eight rows leaves most of its lanes idle where K is short.)
__device__ __forceinline__ void packed_row_sums_by_panel(const PackedRowSums& a, uint32_t block) {
  const int lane = threadIdx.x & 63;
  const int64_t panel = static_cast<int64_t>(block) * 4 + (threadIdx.x >> 6);
  if (panel * 32 >= a.n) return;
  const int64_t k_steps = packed_k_steps(a.k, 16);                  // a multiple of four
  const u32x4* src = static_cast<const u32x4*>(a.packed) + panel * k_steps * 64 + lane;
  int32_t sum = 0;
  for (int64_t ks = 0; ks < k_steps; ks += 4) {
    u32x4 v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = src[(ks + i) * 64];
#pragma unroll
    for (int i = 0; i < 4; ++i) add_signed_bytes(sum, v[i]);
  }
  sum += __shfl_xor(sum, 32, 64);
  const int64_t row = panel * 32 + lane;
  if (lane < 32 && row < a.n) packed_row_sum_out(a, row, sum);
}

__device__ __forceinline__ void packed_row_sums(const PackedRowSums& a, uint32_t block) {
  if (packed_sums_by_panel(a.n, a.k)) packed_row_sums_by_panel(a, block);
  else packed_row_sums_by_quarter(a, block);
}

hipError_t launch_packed_row_sums(const PackedRowSums& sums, hipStream_t stream);
// the quantisation of launch_quantize_rows and these sums as one launch (both must have work)
hipError_t launch_quantize_and_packed_row_sums(const float* x, int32_t batch, int32_t rows, int32_t k, int64_t xbs, int64_t xrs,
                                               int64_t xks, const float* multipliers, int64_t mult_bs, int32_t zero_point,
                                               uint32_t flip, uint8_t* q, int64_t qbs, int64_t qrs, int64_t qks,
                                               const PackedRowSums& sums, hipStream_t stream);

}  // namespace vecops_hip
