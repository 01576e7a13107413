// Tile GEMM instances that take a prepacked B operand, and the packing kernel.
#include "packed_row_sums.h"
#include "tile_gemm_packed_launch.h"
namespace vecops_hip {
hipError_t launch_tile_gemm_packed_b(int src, const TileGemmParams& p, int tile_m, int tile_n, int vector_a,
                                     hipStream_t stream) {
  switch (src) {
    case SRC_BF16: return launch_packed_bf16(p, tile_m, tile_n, vector_a, stream);
    case SRC_F16: return launch_packed_f16(p, tile_m, tile_n, vector_a, stream);
    case SRC_F32_AS_BF16: return launch_packed_f32_as_bf16(p, tile_m, tile_n, vector_a, stream);
    case SRC_F32: return launch_packed_f32(p, tile_m, tile_n, vector_a, stream);
    case SRC_I8: return launch_packed_i8(p, tile_m, tile_n, vector_a, stream);
    // unsigned A: xored on its way into LDS, so never by the loads that write LDS themselves
    case SRC_I8_FLIP: return launch_packed_i8_flip(p, tile_m, tile_n, vector_a ? 1 : 0, stream);
    default: return hipErrorInvalidValue;
  }
}

__global__ __launch_bounds__(256) void packed_row_sums_kernel(const PackedRowSums a) { packed_row_sums(a, blockIdx.x); }

hipError_t launch_packed_row_sums(const PackedRowSums& sums, hipStream_t stream) {
  const int64_t blocks = packed_row_sums_blocks(sums);
  if (blocks == 0) return hipSuccess;
  hipLaunchKernelGGL(packed_row_sums_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, sums);
  return hipGetLastError();
}

hipError_t launch_pack_b(int src, const PackBParams& p, hipStream_t stream) {
  const int epc = src == SRC_I8 ? 16 : src == SRC_F32 ? 4 : 8;
  const int64_t chunks = packed_b_bytes(p.n, p.k, epc) / 16;
  if (chunks == 0) return hipSuccess;
  int64_t blocks = (chunks + 255) / 256;
  if (blocks > 256 * 64) blocks = 256 * 64;
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  switch (src) {
    case SRC_BF16: hipLaunchKernelGGL(pack_b_kernel<SRC_BF16>, grid, block, 0, stream, p); break;
    case SRC_F32_AS_BF16: hipLaunchKernelGGL(pack_b_kernel<SRC_F32_AS_BF16>, grid, block, 0, stream, p); break;
    case SRC_F32: hipLaunchKernelGGL(pack_b_kernel<SRC_F32>, grid, block, 0, stream, p); break;
    case SRC_I8: hipLaunchKernelGGL(pack_b_kernel<SRC_I8>, grid, block, 0, stream, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_unpack_b(int src, const PackBParams& p, hipStream_t stream) {
  const int epc = src == SRC_I8 ? 16 : src == SRC_F32 ? 4 : 8;
  const int64_t chunks = packed_b_bytes(p.n, p.k, epc) / 16;
  if (chunks == 0) return hipSuccess;
  int64_t blocks = (chunks + 255) / 256;
  if (blocks > 256 * 64) blocks = 256 * 64;
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  switch (src) {
    case SRC_BF16: hipLaunchKernelGGL(unpack_b_kernel<SRC_BF16>, grid, block, 0, stream, p); break;
    case SRC_F32: hipLaunchKernelGGL(unpack_b_kernel<SRC_F32>, grid, block, 0, stream, p); break;
    case SRC_I8: hipLaunchKernelGGL(unpack_b_kernel<SRC_I8>, grid, block, 0, stream, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace vecops_hip
