// Tile GEMM instances for 8-bit integer operands with an unsigned side, and the
// row-sum kernel that produces their epilogue terms.
#include "packed_row_sums.h"
#include "row_work_split.h"
#include "tile_gemm_launch.h"
namespace vecops_hip {
hipError_t launch_tile_gemm_i8_flip(const TileGemmParams& p, int tile_m, int tile_n, int mode, hipStream_t stream) {
  return launch_tile_class<SRC_I8_FLIP>(p, tile_m, tile_n, mode, stream);
}

// out[b][r] = scale * sum_k int8(x[b][r][k] xor flip) (+ add[b * add_bs + r])  (wrapping): the per-row and
// per-column terms of SRC_I8_FLIP.  One wavefront per row, any strides; 16 bytes per lane and step
// when the row is contiguous and aligned.
struct ByteRowSums {
  const uint8_t* x;
  int32_t batch, rows, k;
  int64_t bs, rs, ks;
  uint32_t flip, scale;
  const int32_t* add;
  int64_t add_bs;
  int32_t* out;
};

// (block: the workgroup's number among those that sum rows)
__device__ __forceinline__ void byte_row_sums(const ByteRowSums& a, int64_t block) {
  const uint8_t* x = a.x;
  const int32_t batch = a.batch, rows = a.rows, k = a.k;
  const int64_t bs = a.bs, rs = a.rs, ks = a.ks, add_bs = a.add_bs;
  const uint32_t flip = a.flip, scale = a.scale;
  const int32_t* add = a.add;
  int32_t* out = a.out;
  const int lane = threadIdx.x & 63;
  const int64_t row = block * 4 + (threadIdx.x >> 6);
  if (row >= static_cast<int64_t>(batch) * rows) return;
  const int64_t b = row / rows, r = row - b * rows;
  const uint8_t* src = x + b * bs + r * rs;
  int32_t sum = 0;
  int done = 0;
  if (ks == 1 && (reinterpret_cast<uintptr_t>(src) & 15u) == 0) {
    const int chunks = k / 16;
    for (int ch = lane; ch < chunks; ch += 64) {
      const u32x4 v = reinterpret_cast<const u32x4*>(src)[ch];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int32_t word = static_cast<int32_t>(v[w] ^ flip);
        sum += (word << 24 >> 24) + (word << 16 >> 24) + (word << 8 >> 24) + (word >> 24);
      }
    }
    done = chunks * 16;
  }
  for (int kk = done + lane; kk < k; kk += 64) sum += static_cast<int8_t>(src[kk * ks] ^ static_cast<uint8_t>(flip));
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
  if (lane == 0) out[row] = static_cast<int32_t>(static_cast<uint32_t>(sum) * scale + (add ? static_cast<uint32_t>(add[b * add_bs + r]) : 0u));
}

__global__ __launch_bounds__(256) void byte_row_sums_kernel(const ByteRowSums a) { byte_row_sums(a, blockIdx.x); }

// q[b][r][k] = u8(x[b][r][k] * multipliers[b * mult_bs + r] + float(zero_point)): vecops'
// RuntimePerRowAsymmetricQuantizeTransform (matmul/Quantization.h:91-146) and the conversion of its fp32
// result to the uint8 compute type - a multiply and an add, each rounded (the file is compiled without
// contraction), truncation toward zero, NaN and values outside int32 to INT32_MIN, saturation to 0..255.
// Rows contiguous on both sides: by pieces of kQuantizePiece elements, a workgroup each (two quads a lane, each one 16-byte
// load and one 4-byte store at whatever alignment; no division per lane, and workgroups enough that their loads overlap), or
// by quads over all rows; row_work_split.h says which.  Bound by the bytes.
// Other strides: one thread per four consecutive k, a quad at a time on the side that is contiguous.  flip (0 or 0x80) is
// xored into every byte.
struct QuantizeRows {
  const float* x;
  int32_t batch, rows, k;
  int64_t xbs, xrs, xks;
  const float* multipliers;
  int64_t mult_bs;
  float zero_point;
  uint32_t flip;
  uint8_t* q;
  int64_t qbs, qrs, qks;
  QuantizeWalk walk;  // by quads
};

struct __attribute__((packed, aligned(4))) FloatQuad { float v[4]; };
struct __attribute__((packed, aligned(1))) ByteQuad { uint32_t v; };

// Four consecutive elements of a contiguous row at any element's address, or the first `left` of them where fewer are left
// (none: zero or less).
__device__ __forceinline__ FloatQuad load_quad(const float* src, int left) {
  FloatQuad quad;
  if (left >= 4) {
    quad = *reinterpret_cast<const FloatQuad*>(src);
  } else {
    for (int e = 0; e < 4; ++e) quad.v[e] = e < left ? src[e] : 0.0f;
  }
  return quad;
}

// The quad's four bytes, the first the lowest.
__device__ __forceinline__ uint32_t quantize_quad_word(const QuantizeRows& a, const FloatQuad& quad, float mult) {
  uint32_t word = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float scaled = quad.v[e] * mult;
    word |= (narrow_to_byte(scaled + a.zero_point, false) ^ a.flip) << (8 * e);  // flip 0x80: the byte as q - 128 in int8
  }
  return word;
}

__device__ __forceinline__ void quantize_quad_out(const QuantizeRows& a, const FloatQuad& quad, float mult, uint8_t* dst, int left) {
  const uint32_t word = quantize_quad_word(a, quad, mult);
  if (left >= 4) {
    reinterpret_cast<ByteQuad*>(dst)->v = word;
  } else {
    for (int e = 0; e < left; ++e) dst[e] = static_cast<uint8_t>(word >> (8 * e));
  }
}

// (block: the workgroup's number among those that quantise; xks == qks == 1; batch * rows is at most INT32_MAX)
__device__ __forceinline__ void quantize_by_pieces(const QuantizeRows& a, uint32_t block) {
  const uint32_t pieces = static_cast<uint32_t>(quantize_pieces(a.k));
  const uint32_t row = block / pieces, piece = block - row * pieces;
  const uint32_t b = row / static_cast<uint32_t>(a.rows), r = row - b * static_cast<uint32_t>(a.rows);
  const float* src = a.x + b * a.xbs + r * a.xrs;
  uint8_t* dst = a.q + b * a.qbs + r * a.qrs;
  const float mult = a.multipliers[b * a.mult_bs + r];
  FloatQuad quad[kQuantizeQuads];
#pragma unroll
  for (int i = 0; i < kQuantizeQuads; ++i) {
    const int k = quantize_quad(piece, threadIdx.x, i);
    quad[i] = load_quad(src + k, a.k - k);
  }
#pragma unroll
  for (int i = 0; i < kQuantizeQuads; ++i) {
    const int k = quantize_quad(piece, threadIdx.x, i);
    quantize_quad_out(a, quad[i], mult, dst + k, a.k - k);
  }
}

__device__ __forceinline__ void quantize_by_quads(const QuantizeRows& a, uint32_t block) {
  const int64_t rows = static_cast<int64_t>(a.batch) * a.rows;
  for (QuantizeQuad at = quantize_first(a.walk, block * 256 + threadIdx.x); at.row < rows; at = quantize_next(a.walk, at)) {
    const uint32_t row = static_cast<uint32_t>(at.row);
    const uint32_t b = a.batch == 1 ? 0 : row / static_cast<uint32_t>(a.rows), r = row - b * static_cast<uint32_t>(a.rows);
    const int k = static_cast<int>(at.quad) * 4;
    const FloatQuad quad = load_quad(a.x + b * a.xbs + r * a.xrs + k, a.k - k);
    quantize_quad_out(a, quad, a.multipliers[b * a.mult_bs + r], a.q + b * a.qbs + r * a.qrs + k, a.k - k);
  }
}

// (block of blocks: the workgroup's number among those that quantise, and how many they are; any strides)
__device__ __forceinline__ void quantize_strided(const QuantizeRows& a, int64_t block, int64_t blocks) {
  const int32_t batch = a.batch, rows = a.rows, k = a.k;
  const int64_t xks = a.xks, qks = a.qks;
  const int64_t quads_per_row = (static_cast<int64_t>(k) + 3) / 4;
  const int64_t total = static_cast<int64_t>(batch) * rows * quads_per_row;
  for (int64_t idx = block * 256ll + threadIdx.x; idx < total; idx += blocks * 256ll) {
    const int64_t row = idx / quads_per_row;                 // batch * rows + r
    const int k0 = static_cast<int>(idx - row * quads_per_row) * 4;
    const int64_t b = row / rows, r = row - b * rows;
    const float* src = a.x + b * a.xbs + r * a.xrs + k0 * xks;
    uint8_t* dst = a.q + b * a.qbs + r * a.qrs + k0 * qks;
    const float mult = a.multipliers[b * a.mult_bs + r];
    const int left = min(4, k - k0);
    FloatQuad quad;
    if (xks == 1) {
      quad = load_quad(src, left);
    } else {
      // (one load after the other: four at a time walk 8192 x 11008 from [K,M] 5 % slower, 1290 us against 1225)
      f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int e = 0; e < left; ++e) v[e] = src[e * xks];
      quad = {{v[0], v[1], v[2], v[3]}};
    }
    if (qks == 1) {
      quantize_quad_out(a, quad, mult, dst, left);
    } else {
      const uint32_t word = quantize_quad_word(a, quad, mult);
      for (int e = 0; e < left; ++e) dst[e * qks] = static_cast<uint8_t>(word >> (8 * e));
    }
  }
}

// One kernel a way, because the ways' registers and code would weigh on each other (32768 x 2049 by pieces 75 us in one kernel
// with the strided way, 70 alone).
enum QuantizeWay : int { QUANTIZE_PIECES, QUANTIZE_QUADS, QUANTIZE_STRIDED };

template <int WAY>
__device__ __forceinline__ void quantize_rows(const QuantizeRows& a, uint32_t block, uint32_t blocks) {
  if constexpr (WAY == QUANTIZE_PIECES) quantize_by_pieces(a, block);
  else if constexpr (WAY == QUANTIZE_QUADS) quantize_by_quads(a, block);
  else quantize_strided(a, block, blocks);
}

template <int WAY>
__global__ __launch_bounds__(256) void quantize_rows_kernel(const QuantizeRows a) { quantize_rows<WAY>(a, blockIdx.x, gridDim.x); }

// Both preparations of a runtime-quantised product in one launch: the first quantize_blocks workgroups quantise the
// activations, the others sum the weight rows (two memory-bound kernels of about 10 us each, neither of which needs the
// other: one launch saves a launch gap and lets their tails overlap).
template <int WAY>
__global__ __launch_bounds__(256) void quantize_and_row_sums_kernel(const QuantizeRows qa, const ByteRowSums sa, uint32_t quantize_blocks) {
  if (blockIdx.x < quantize_blocks) quantize_rows<WAY>(qa, blockIdx.x, quantize_blocks);
  else byte_row_sums(sa, blockIdx.x - quantize_blocks);
}

// The same with the weights packed.
template <int WAY>
__global__ __launch_bounds__(256) void quantize_and_packed_row_sums_kernel(const QuantizeRows qa, const PackedRowSums sa, uint32_t quantize_blocks) {
  if (blockIdx.x < quantize_blocks) quantize_rows<WAY>(qa, blockIdx.x, quantize_blocks);
  else packed_row_sums(sa, blockIdx.x - quantize_blocks);
}

namespace {
// Workgroups of the quantisation, 0 when there is nothing to quantise; says which way it goes and fills in the walk.
int64_t quantize_blocks_for(QuantizeRows& a, QuantizeWay* way) {
  const int64_t rows = static_cast<int64_t>(a.batch) * a.rows;
  if (rows <= 0 || a.k <= 0) return 0;
  if (a.xks == 1 && a.qks == 1) {
    const int64_t blocks = quantize_blocks(rows, a.k);
    *way = quantize_by_pieces(rows, a.k) ? QUANTIZE_PIECES : QUANTIZE_QUADS;
    if (*way == QUANTIZE_QUADS) a.walk = quantize_walk(a.k, static_cast<uint32_t>(blocks));
    return blocks;
  }
  *way = QUANTIZE_STRIDED;
  const int64_t blocks = (rows * ((static_cast<int64_t>(a.k) + 3) / 4) + 255) / 256;
  return blocks > 256 * 32 ? 256 * 32 : blocks;
}

// launch(way as a constant)
template <typename F>
hipError_t launch_way(QuantizeWay way, F&& launch) {
  switch (way) {
    case QUANTIZE_PIECES: launch(std::integral_constant<int, QUANTIZE_PIECES>{}); break;
    case QUANTIZE_QUADS: launch(std::integral_constant<int, QUANTIZE_QUADS>{}); break;
    default: launch(std::integral_constant<int, QUANTIZE_STRIDED>{}); break;
  }
  return hipGetLastError();
}
}  // namespace

hipError_t launch_quantize_rows(const float* x, int32_t batch, int32_t rows, int32_t k, int64_t xbs, int64_t xrs,
                                int64_t xks, const float* multipliers, int64_t mult_bs, int32_t zero_point, uint32_t flip,
                                uint8_t* q, int64_t qbs, int64_t qrs, int64_t qks, hipStream_t stream) {
  QuantizeRows a{x, batch, rows, k, xbs, xrs, xks, multipliers, mult_bs, static_cast<float>(zero_point), flip & 0xffu, q, qbs, qrs, qks, {}};
  QuantizeWay way = QUANTIZE_STRIDED;
  const int64_t blocks = quantize_blocks_for(a, &way);
  if (blocks == 0) return hipSuccess;
  return launch_way(way, [&](auto w) {
    hipLaunchKernelGGL(quantize_rows_kernel<decltype(w)::value>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, a);
  });
}

hipError_t launch_byte_row_sums(const void* x, int32_t batch, int32_t rows, int32_t k, int64_t bs, int64_t rs,
                                int64_t ks, uint32_t flip, uint32_t scale, const int32_t* add, int64_t add_bs, int32_t* out,
                                hipStream_t stream) {
  const int64_t total = static_cast<int64_t>(batch) * rows;
  if (total <= 0) return hipSuccess;
  const int64_t blocks = (total + 3) / 4;
  if (blocks > kMostBlocks) return hipErrorInvalidConfiguration;
  const ByteRowSums a{static_cast<const uint8_t*>(x), batch, rows, k, bs, rs, ks, flip, scale, add, add_bs, out};
  hipLaunchKernelGGL(byte_row_sums_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, a);
  return hipGetLastError();
}

// launch_quantize_rows and launch_byte_row_sums as one launch (both must have work: the caller checks).
hipError_t launch_quantize_and_row_sums(const float* x, int32_t batch, int32_t rows, int32_t k, int64_t xbs, int64_t xrs,
                                        int64_t xks, const float* multipliers, int64_t mult_bs, int32_t zero_point, uint32_t flip,
                                        uint8_t* q, int64_t qbs, int64_t qrs, int64_t qks, const void* w, int32_t w_batch,
                                        int32_t w_rows, int64_t w_bs, int64_t w_rs, int64_t w_ks, uint32_t w_flip, uint32_t scale,
                                        const int32_t* add, int64_t add_bs, int32_t* out, hipStream_t stream) {
  QuantizeRows qa{x, batch, rows, k, xbs, xrs, xks, multipliers, mult_bs, static_cast<float>(zero_point), flip & 0xffu, q, qbs, qrs, qks, {}};
  const int64_t sums = static_cast<int64_t>(w_batch) * w_rows;
  QuantizeWay way = QUANTIZE_STRIDED;
  const int64_t q_blocks = quantize_blocks_for(qa, &way), s_blocks = (sums + 3) / 4;
  if (q_blocks <= 0 || sums <= 0) return hipErrorInvalidValue;
  if (q_blocks + s_blocks > kMostBlocks) return hipErrorInvalidConfiguration;
  const ByteRowSums sa{static_cast<const uint8_t*>(w), w_batch, w_rows, k, w_bs, w_rs, w_ks, w_flip, scale, add, add_bs, out};
  return launch_way(way, [&](auto w) {
    hipLaunchKernelGGL(quantize_and_row_sums_kernel<decltype(w)::value>, dim3(static_cast<unsigned>(q_blocks + s_blocks)), dim3(256), 0, stream,
                       qa, sa, static_cast<uint32_t>(q_blocks));
  });
}

// launch_quantize_rows and launch_packed_row_sums as one launch (both must have work).
hipError_t launch_quantize_and_packed_row_sums(const float* x, int32_t batch, int32_t rows, int32_t k, int64_t xbs, int64_t xrs,
                                               int64_t xks, const float* multipliers, int64_t mult_bs, int32_t zero_point,
                                               uint32_t flip, uint8_t* q, int64_t qbs, int64_t qrs, int64_t qks,
                                               const PackedRowSums& sums, hipStream_t stream) {
  QuantizeRows qa{x, batch, rows, k, xbs, xrs, xks, multipliers, mult_bs, static_cast<float>(zero_point), flip & 0xffu, q, qbs, qrs, qks, {}};
  QuantizeWay way = QUANTIZE_STRIDED;
  const int64_t q_blocks = quantize_blocks_for(qa, &way), s_blocks = packed_row_sums_blocks(sums);
  if (q_blocks <= 0 || s_blocks <= 0) return hipErrorInvalidValue;
  if (q_blocks + s_blocks > kMostBlocks) return hipErrorInvalidConfiguration;
  return launch_way(way, [&](auto w) {
    hipLaunchKernelGGL(quantize_and_packed_row_sums_kernel<decltype(w)::value>, dim3(static_cast<unsigned>(q_blocks + s_blocks)), dim3(256), 0, stream,
                       qa, sums, static_cast<uint32_t>(q_blocks));
  });
}
}  // namespace vecops_hip
