// The loads that the floating-point dense product makes of its weight tiles, by the loops of its two kernels: weights are asked
// for ahead of the multiplies, and those behind the last chunk, too.  All of them must lie inside the tiles as prepare lays them out,
// and a row block's own must be read once each.
// Prints "ok", or what does not.
#include <cstdio>
#include <vector>

#include "sparse_conv_kernels.h"

namespace {

struct Reads {
  std::vector<int> cells;  // of 16 bytes, of one row block
  uint64_t block_at, all;
  bool inside = true;

  void Load(uint64_t at) {
    if (block_at + at + 16 > all) inside = false;
    if (at / 16 < cells.size()) ++cells[at / 16];
  }
};

// Wavefronts that load and multiply: 64 channels a chunk, every chunk's weights asked for while the chunk before is multiplied.  Lane (n, half)
// holds eight channels of row n of a step of 16.
void Steps16(int pieces, int chunks, Reads* r) {
  std::vector<int> asked = {0};  // before the loop; in it pairs of chunks, behind it the last one, which asks for nothing
  for (int chunk = 0; chunk + 2 <= chunks; chunk += 2) {
    asked.push_back(chunk + 1);
    asked.push_back(chunk + 2);
  }
  for (int c : asked)
    for (int step = 0; step < pl::kFloatMfmaChunk / 16; ++step)
      for (int piece = 0; piece < pieces; ++piece)
        for (int lane = 0; lane < 64; ++lane) {
          const int n = lane & 31, half = lane >> 5;
          r->Load((n >> 4) * (pieces * 1024) + 256 * half + 16 * (n & 15) + pl::FloatMfmaWeightTile(c, step & ~1, pieces, piece) + 512 * (step & 1));
        }
}

// Wavefronts of their own for the inputs: 128 channels a chunk, the weights of a step of 32 asked for two steps ahead, as far as there are channels.
void Steps32(int channels, Reads* r) {
  auto load = [&](int chunk, int ks) {
    for (int t = 0; t < 2; ++t)
      for (int piece = 0; piece < 2; ++piece)
        for (int lane = 0; lane < 64; ++lane) r->Load(lane * 16 + pl::FloatMfmaWeightTile(0, 2 * (chunk * 4 + ks) + t, 2, piece));
  };
  load(0, 0);
  load(0, 1);
  const int chunks = (channels + 127) / 128;
  for (int chunk = 0; chunk < chunks; ++chunk)
    for (int ks = 0; ks < 4; ++ks) {
      const bool last = chunk + 1 == chunks;
      if (last && ks > 0 && 32 * (4 * chunk + ks) >= channels) break;
      if (!last || ks + 2 < 4) load(chunk, ks + 2);
    }
}

}  // namespace

int main() {
  for (int form = 0; form <= 2; ++form)  // fp16, fp32, fp32 with wavefronts of their own
    for (int blocks = 1; blocks <= 3; ++blocks)
      for (int channels = 8; channels <= 9 * 64; channels += 8) {
        const int pieces = form == 0 ? 1 : 2, chunks = (channels + pl::kFloatMfmaChunk - 1) / pl::kFloatMfmaChunk;
        const uint64_t block_bytes = static_cast<uint64_t>(chunks) * (pl::kFloatMfmaChunk / 16) * pieces * 1024;
        for (int block = 0; block < blocks; ++block) {
          Reads r{std::vector<int>(block_bytes / 16, 0), block * block_bytes, blocks * block_bytes + pl::FloatMfmaWeightTail(pieces)};
          if (form == 2) {
            Steps32(channels, &r);
          } else {
            Steps16(pieces, chunks, &r);
          }
          if (!r.inside) {
            std::printf("form %d, %d channels, block %d of %d: a load behind the tiles\n", form, channels, block, blocks);
            return 1;
          }
          // cells of steps of 32 channels that hold any of the layer's: a step's 16 rows, twice, in every piece
          const size_t used = form == 2 ? static_cast<size_t>((channels + 31) / 32) * 2 * pieces * 64 : r.cells.size();
          for (size_t i = 0; i < r.cells.size(); ++i)
            if (i < used ? r.cells[i] != 1 : r.cells[i] > 1) {
              std::printf("form %d, %d channels: cell %zu is read %d times\n", form, channels, i, r.cells[i]);
              return 1;
            }
        }
      }
  std::printf("ok\n");
  return 0;
}
