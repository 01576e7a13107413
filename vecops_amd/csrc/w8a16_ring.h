// Host side of w8a16_ring.hip: weight-only products of up to 16 rows on rings of LDS stages.
#ifndef VECOPS_HIP_W8A16_RING_H
#define VECOPS_HIP_W8A16_RING_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "skinny_w8a16.h"

namespace vecops_hip {

// bn: weight rows of a workgroup, 16, 32, 48 or 64.  Groups of 64, 128 or 256.
bool launch_w8a16_ring_serves(const SkinnyW8A16Params& p, int bn);
hipError_t launch_w8a16_ring(const SkinnyW8A16Params& p, int bn, hipStream_t stream);

}  // namespace vecops_hip
#endif
