// How the byte preparations of a product are dealt to workgroups of 256 lanes: arithmetic on whole numbers only, compiled
// into the kernels, their launches and the CPU test of both.
#pragma once
#include <cstdint>

namespace vecops_hip {

// A launch has fewer than 2^32 lanes.
constexpr int64_t kMostBlocks = (int64_t{1} << 24) - 1;

// Quantisation of contiguous rows, by pieces: a workgroup takes one piece of a row, a lane two quads of it, 1024 elements
// apart.  By quads: the quads of all rows are one sequence, a lane takes one and then the one a launch's lanes further on.
// Short rows go by quads, because the lanes past a row's end would idle (1048576 x 64 fp32: 937 us by pieces, 59 by quads,
// 131072 x 512 119 and 58, 65536 x 1000 67 and 57; 65536 x 4096 230 and 277), and so does what has more pieces than a
// launch may have workgroups.
constexpr int kQuantizePiece = 2048;
constexpr int kQuantizeQuads = kQuantizePiece / 1024;
constexpr int kQuantizeShortRow = 1024;
constexpr int64_t kMostPieces = 1 << 23;
constexpr int64_t kMostQuadBlocks = 8192;

constexpr int64_t quantize_pieces(int64_t k) { return (k + kQuantizePiece - 1) / kQuantizePiece; }
constexpr bool quantize_by_pieces(int64_t rows, int64_t k) { return k > kQuantizeShortRow && rows * quantize_pieces(k) <= kMostPieces; }
constexpr int64_t quantize_blocks(int64_t rows, int64_t k) {
  if (quantize_by_pieces(rows, k)) return rows * quantize_pieces(k);
  const int64_t blocks = (rows * ((k + 3) / 4) + 255) / 256;
  return blocks < kMostQuadBlocks ? blocks : kMostQuadBlocks;
}

// By pieces: where a lane's i-th quad begins.  It fits 32 bits in a row of INT32_MAX elements, up to 2047 past its end; where
// the quad ends need not (what is left of the row is compared, which may be less than nothing).
constexpr int quantize_quad(uint32_t piece, int lane, int i) { return static_cast<int>(piece) * kQuantizePiece + i * 1024 + lane * 4; }

// By quads.  The way of a lane over the quads of all rows: its first one, and the next, a launch's lanes further on.  That
// step is divided into whole rows and quads once, for the launch; the first quad's number fits 32 bits, all quads together
// need not.
struct QuantizeWalk {
  uint32_t quads;  // of a row
  uint32_t step_rows, step_quads;
};
constexpr QuantizeWalk quantize_walk(int64_t k, uint32_t blocks) {
  const uint32_t quads = static_cast<uint32_t>((k + 3) / 4);
  return {quads, blocks * 256 / quads, blocks * 256 % quads};
}
struct QuantizeQuad {
  int64_t row;
  uint32_t quad;
};
constexpr QuantizeQuad quantize_first(const QuantizeWalk& w, uint32_t lane) { return {lane / w.quads, lane % w.quads}; }
constexpr QuantizeQuad quantize_next(const QuantizeWalk& w, const QuantizeQuad& at) {
  const uint32_t quad = at.quad + w.step_quads;
  return quad < w.quads ? QuantizeQuad{at.row + w.step_rows, quad} : QuantizeQuad{at.row + w.step_rows + 1, quad - w.quads};
}

// Sums over the rows of a packed operand (panels of 32 rows): a panel is a wavefront's, or its quarters of eight rows are a
// workgroup's each (packed_row_sums.h).  By panel where the panels are many and K is short, because the lanes of a workgroup
// past a quarter's K would idle (the unsigned 17 x 262144 x 64 product 34 us by quarter, 26 by panel, 131072 x 256 29 and 27;
// 131072 x 512 level; 256 x 11008 x 4096 57 and 88), and where the quarters are more than a launch should have workgroups.
constexpr int64_t kShortKPanels = 2048, kPanelShortK = 512, kLongKPanels = 1 << 18;
constexpr bool packed_sums_by_panel(int64_t n, int64_t k) { return (n + 31) / 32 >= (k <= kPanelShortK ? kShortKPanels : kLongKPanels); }
constexpr int64_t packed_sums_blocks(int64_t n, int64_t k) {
  return packed_sums_by_panel(n, k) ? ((n + 31) / 32 + 3) / 4 : (n + 7) / 8;
}

}  // namespace vecops_hip
