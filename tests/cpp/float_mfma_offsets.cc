// The loads that the floating-point dense product makes of its weight tiles, by the loop of its kernel: every chunk's weights
// are asked for while the chunk before is multiplied, and with an even number of chunks those behind the last one, too.  All of
// them must lie inside the tiles as prepare lays them out, and a row block's own must be read once each.
// Prints "ok", or what does not.
#include <cstdio>
#include <vector>

#include "sparse_conv_kernels.h"

int main() {
  for (int pieces = 1; pieces <= 2; ++pieces)
    for (int blocks = 1; blocks <= 3; ++blocks)
      for (int chunks = 1; chunks <= 9; ++chunks) {
        const int steps = pl::kFloatMfmaChunk / 16;
        const uint64_t block_bytes = static_cast<uint64_t>(chunks) * steps * pieces * 1024, all = blocks * block_bytes + pl::FloatMfmaWeightTail(pieces);
        std::vector<int> asked = {0};  // before the loop; in it pairs of chunks, behind it the last one, which asks for nothing
        for (int chunk = 0; chunk + 2 <= chunks; chunk += 2) {
          asked.push_back(chunk + 1);
          asked.push_back(chunk + 2);
        }
        for (int block = 0; block < blocks; ++block) {
          std::vector<int> reads(block_bytes / 1024, 0);
          for (int c : asked)
            for (int step = 0; step < steps; ++step)
              for (int piece = 0; piece < pieces; ++piece) {
                const uint64_t tile = pl::FloatMfmaWeightTile(c, step, pieces, piece);
                if (tile < block_bytes) ++reads[tile / 1024];
                if (block * block_bytes + tile + 64 * 16 > all) {
                  std::printf("chunk %d of %d, block %d of %d, step %d, piece %d: %llu of %llu\n", c, chunks, block, blocks, step, piece, (unsigned long long)(block * block_bytes + tile), (unsigned long long)all);
                  return 1;
                }
              }
          for (int r : reads)
            if (r != 1) {
              std::printf("%d chunks: a tile is read %d times\n", chunks, r);
              return 1;
            }
        }
      }
  std::printf("ok\n");
  return 0;
}
