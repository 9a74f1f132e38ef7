// Which 16 x 16 output blocks of a 64 x 64 tile each of its four waves computes (gemm.hip).
#pragma once

namespace ccx {

// Rows r0 .. r0 + 16 ni and columns c0 .. c0 + 16 nj of the tile, ni and nj 0, 1 or 2 (0: nothing).
struct WaveBlocks {
  int r0, c0, ni, nj;
};

// Wave w of a tile whose rb x cb (1 .. 4 each) first blocks hold outputs. Only those are computed, and where a side
// has at most two of them the four waves share them out: an o-wide side (o = 9, 13) would otherwise spend 4 to 16
// times its flops (Lambda at o=13 v=101: 2.26 to 2.11 ms). A wave's rows and columns never reach past the rb x cb
// blocks, so whoever reads ni and nj blocks of the operands stays inside the tile.
constexpr WaveBlocks wave_blocks(int rb, int cb, int w) {
  return rb <= 2 && cb > 2   ? (w < cb ? WaveBlocks{0, 16 * w, rb, 1} : WaveBlocks{0, 0, 0, 0})
         : cb <= 2 && rb > 2 ? (w < rb ? WaveBlocks{16 * w, 0, 1, cb} : WaveBlocks{0, 0, 0, 0})
         : rb <= 2           ? ((w >> 1) < rb && (w & 1) < cb ? WaveBlocks{16 * (w >> 1), 16 * (w & 1), 1, 1}
                                                              : WaveBlocks{0, 0, 0, 0})
                             : WaveBlocks{32 * (w >> 1), 32 * (w & 1), rb - 2 * (w >> 1) < 2 ? rb - 2 * (w >> 1) : 2,
                                          cb - 2 * (w & 1) < 2 ? cb - 2 * (w & 1) : 2};
}

}  // namespace ccx
