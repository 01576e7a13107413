// How the byte preparations of a product are dealt to workgroups of 256 lanes: arithmetic on whole numbers only, compiled
// into the kernels and into the CPU test of the positions.
#pragma once
#include <cstdint>

namespace vecops_hip {

// Quantisation of contiguous rows: a workgroup takes one piece of a row, a lane two quads of it, 1024 elements apart.
constexpr int kQuantizePiece = 2048;
constexpr int kQuantizeQuads = kQuantizePiece / 1024;

constexpr int64_t quantize_pieces(int64_t k) { return (k + kQuantizePiece - 1) / kQuantizePiece; }

// First element of a lane's i-th quad, and whether all four of them lie in a row of k.  64 bits: a row may have INT32_MAX
// elements, and the last quad of its last piece ends past what 32 bits hold.
constexpr int64_t quantize_quad(int64_t piece, int lane, int i) { return piece * kQuantizePiece + i * 1024 + lane * 4; }
constexpr bool quantize_quad_is_whole(int64_t quad, int64_t k) { return quad + 4 <= k; }

}  // namespace vecops_hip
