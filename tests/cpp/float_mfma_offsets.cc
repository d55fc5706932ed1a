// The loads that the floating-point dense product makes of its weight tiles, by the loop of its kernel: every chunk's weights
// are asked for while the chunk before is multiplied, so those behind the last chunk too where the loop does not know yet that it
// ends.  A lane's bytes must lie inside its row block's tiles, or outside a buffer whose size is not below the scalar offset.
// Prints "ok", or what lies elsewhere.
#include <cstdio>

#include "sparse_conv_kernels.h"

int main() {
  for (int pieces = 1; pieces <= 2; ++pieces)
    for (int chunks = 1; chunks <= 9; ++chunks) {
      const uint32_t steps = pl::kFloatMfmaChunk / 16, size = (uint32_t)chunks * steps * (uint32_t)pieces * 1024u;
      uint64_t seen = 0;
      // chunk 0 before the loop, in the loop the one behind a chunk; pairs of chunks, then one
      const int last_asked = chunks % 2 == 0 ? chunks : chunks - 1;
      for (int chunk = 0; chunk <= last_asked; ++chunk)
        for (int step = 0; step < (int)steps; ++step)
          for (int piece = 0; piece < pieces; ++piece)
            for (uint32_t lane = 0; lane < 64; ++lane) {
              const uint64_t own = 16 * lane, tile = pl::FloatMfmaWeightTile(chunk, chunks, step, pieces, piece), bytes = pl::FloatMfmaWeightBytes(chunk, chunks, pieces);
              const bool inside = bytes == size && own + tile + 16 <= bytes;
              const bool outside = tile <= bytes && own >= bytes - tile;
              if (inside == outside || inside != (chunk < chunks)) {
                std::printf("chunk %d of %d, step %d, piece %d, lane %u: %llu + %llu of %u\n", chunk, chunks, step, piece, lane, (unsigned long long)own, (unsigned long long)tile, size);
                return 1;
              }
              if (inside) seen += 16;
            }
      if (seen != size) {
        std::printf("%llu of %u bytes read\n", (unsigned long long)seen, size);
        return 1;
      }
    }
  std::printf("ok\n");
  return 0;
}
