// int8 x int8 tile GEMM instances of the grouped launch.
#include "tile_gemm_launch.h"
namespace vecops_hip {
hipError_t launch_tile_gemm_grouped_i8(const GroupLaunch& t, int32_t workgroups, int tile, int mode, hipStream_t stream) {
  return launch_grouped_class<SRC_I8>(t, workgroups, tile, mode, stream);
}
}  // namespace vecops_hip
