// Chunk MFMA: int8 sparse 1x1 convolution as a dense product on the matrix cores that takes the input channels chunk
// by chunk, for layers with many channels and for calls of few positions.
//
// One workgroup of eight wavefronts makes a tile of 128 output rows x up to 64 NW positions; wavefront w multiplies
// one tile of 16 rows with all of them.  Per chunk of 512 / NW channels a thread loads, for 16 consecutive channels,
// the dword (four positions) of one position quad, turns the 16 x 4 bytes into four 16-byte operand cells (16
// channels of one position) with two stages of byte permutes and writes them to one of two 32 KB LDS buffers.  The
// accumulators stay in registers over all chunks.  While a chunk is multiplied (v_mfma_i32_16x16x64_i8) the next one
// is written to the other buffer, a quarter behind each of the first multiplies, and the loads of the one three
// ahead are issued; the weights (dense tiles in operand order, straight into registers: every wavefront needs its own
// rows only) are requested one chunk ahead.  One barrier per chunk.
//
// What bounds it: on a full chip no unit by itself.  2048 -> 2048 @14x14 x 16 (one workgroup per CU, 16 chunks) takes 51 K clocks,
// 3.2 K per chunk, of which by counters and device rates LDS is busy for 1.6 K (every wavefront reads the whole chunk, 256 KB at
// 235 bytes per clock and CU; 32 KB of writes at 71), the matrix cores of a SIMD for 1.0 K and its vector ALU for 0.6 K; L2 serves
// 176 MB of reads per launch, 73 % of its requests from its own lines.  With two wavefronts per SIMD and a barrier per chunk these
// overlap in part only.  A workgroup whose wavefronts own two or four row tiles and split the channels halves the LDS reads and was
// no faster there (25.4 us against 24.6).  A call of one chunk is its chain of one load, transpose, multiply and store.
// us per launch, buffers rotating over 320 MB, the kernel that ran before / this one: that layer (the block kernel) 31.5 / 24.7,
// on buffers that stay in the last-level cache 31.4 / 22.5; 512 -> 512 @14x14 on one image 6.4 / 4.4; 2048 -> 512 @7x7 on 16 images
// 30.0 / 10.9.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "epilogue.h"
#include "kernarg_head.h"
#include "launch_lds.h"
#include "sparse_conv_kernels.h"

namespace pl {
namespace {

using epilogue::ActivateT;
using epilogue::ActQuantF;
using epilogue::DispatchAct;
using epilogue::TruncPackI8x4;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

// what the first loads need arrives in registers: with the scales and biases requested behind the first loads, 146 random
// calls take 0.94 of the time on average, 2048 -> 2048 @14x14 x 16 22.5 -> 21.9 us
PL_IN_HEAD(ChunkMfmaParams, x);
PL_IN_HEAD(ChunkMfmaParams, wtiles);
PL_IN_HEAD(ChunkMfmaParams, K);
PL_IN_HEAD(ChunkMfmaParams, hw);
PL_IN_HEAD(ChunkMfmaParams, qpi);
PL_IN_HEAD(ChunkMfmaParams, total_quads);
PL_IN_HEAD(ChunkMfmaParams, tile_quads);
PL_IN_HEAD(ChunkMfmaParams, tiles);
PL_IN_HEAD(ChunkMfmaParams, row_groups);
PL_IN_HEAD(ChunkMfmaParams, row_tiles);
PL_IN_HEAD(ChunkMfmaParams, padded_ksteps);
PL_IN_HEAD(ChunkMfmaParams, chunks);

constexpr int kBufCells = 2048;  // 16-byte cells of one chunk: (channel group of 16, position of the tile)

template <int NW, int OUT>
__device__ __forceinline__ void ChunkBody(const ChunkMfmaParams& p, uint4* xt) {
  constexpr int QT = 16 * NW;    // position quads a tile has room for
  constexpr int NG = 512 / QT;   // channel groups of a chunk
  constexpr int KS = NG / 4;     // 64-channel steps of a chunk
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // each XCD owns a contiguous range of tiles, the row groups of one tile follow each other there
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int first_tile = (xcd * p.tiles) >> 3, last_tile = ((xcd + 1) * p.tiles) >> 3;
  const int tile = first_tile + slot / p.row_groups, rg = slot % p.row_groups;
  if (tile >= last_tile) return;

  // the thread's part of a chunk: quad j, channel group kgl; a partial quad (the end of an image whose size is not
  // a multiple of 4) is read from the last four positions of its channel row and shifted, threads behind the tile's or
  // the tensor's last quad repeat that one
  const int j = tid & (QT - 1), kgl = tid / QT;
  const uint32_t tile_quad0 = (uint32_t)tile * (uint32_t)p.tile_quads;
  const uint32_t quad = min(tile_quad0 + (uint32_t)min(j, p.tile_quads - 1), p.total_quads - 1u);
  const uint32_t img = quad / (uint32_t)p.qpi;
  const int pp = 4 * (int)(quad - img * (uint32_t)p.qpi);
  const int first = min(pp, p.hw - 4), shift = 8 * (pp - first);
  const uint32_t vbase = img * (uint32_t)p.K * (uint32_t)p.hw + (uint32_t)first;
  uint32_t r[2][16];
  // loads [4 piece, 4 piece + 4) of the thread's 16 of a chunk
  auto issue = [&](uint32_t (&rd)[16], int chunk, int piece) {
    // the last group of a channel count that is no multiple of 16 holds the last 16 channels; groups behind it repeat
    // it against weights of zero
    const uint32_t voff = vbase + (uint32_t)(min(chunk * 16 * NG + 16 * kgl, p.K - 16) * p.hw);
    const int8_t* base = p.x + (size_t)(4 * piece) * p.hw;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rd[4 * piece + i] = *reinterpret_cast<const uint32_t*>(base + voff);
      base += p.hw;
    }
  };
  auto issue_all = [&](uint32_t (&rd)[16], int chunk) {
#pragma unroll
    for (int piece = 0; piece < 4; ++piece) issue(rd, chunk, piece);
  };
  // Two stages of byte permutes, in four pieces: bytes of neighbouring channels paired up for positions 0 and 1, their
  // cells made and written, then the same for positions 2 and 3.
  uint4* const cells = xt + kgl * (4 * QT) + j;
  uint32_t pair[4][2];
  auto commit = [&](uint32_t (&rd)[16], int buf, int piece) {
    if (piece == 0 && !p.quad_aligned) {
#pragma unroll
      for (int i = 0; i < 16; ++i) rd[i] >>= shift;
    }
    if ((piece & 1) == 0) {
      const uint32_t sel = piece == 0 ? 0x05010400u : 0x07030602u;
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4) {
        pair[b4][0] = __builtin_amdgcn_perm(rd[4 * b4 + 1], rd[4 * b4], sel);
        pair[b4][1] = __builtin_amdgcn_perm(rd[4 * b4 + 3], rd[4 * b4 + 2], sel);
      }
    } else {
      uint4* dst = cells + buf * kBufCells;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const uint32_t sel = c ? 0x07060302u : 0x05040100u;
        dst[(piece - 1 + c) * QT] = make_uint4(__builtin_amdgcn_perm(pair[0][1], pair[0][0], sel), __builtin_amdgcn_perm(pair[1][1], pair[1][0], sel),
                                               __builtin_amdgcn_perm(pair[2][1], pair[2][0], sel), __builtin_amdgcn_perm(pair[3][1], pair[3][0], sel));
      }
    }
  };
  auto commit_all = [&](uint32_t (&rd)[16], int buf) {
#pragma unroll
    for (int piece = 0; piece < 4; ++piece) commit(rd, buf, piece);
  };

  // the wavefront's row tile (past the last one: the last one again, not stored)
  const int rt = rg * 8 + wave;
  const v4i* const wt = static_cast<const v4i*>(p.wtiles) + (size_t)min(rt, p.row_tiles - 1) * p.padded_ksteps * 64 + lane;
  v4i a[KS];
  auto load_weights = [&](int chunk, int ks) { a[ks] = wt[(chunk * KS + ks) * 64]; };
  const int n = lane & 15, kq = lane >> 4;
  const uint4* const operand = xt + kq * (4 * QT) + n;
  v4i acc[NW][4];
#pragma unroll
  for (int w = 0; w < NW; ++w)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[w][c] = v4i{0, 0, 0, 0};

  // One chunk: eight (step, window of 16 quads) pairs of four multiplies.  The operand cells are read from LDS PF cells
  // ahead.  Behind the first four pairs the next chunk's activations go to the other buffer, so that the vector ALU
  // and the LDS writes work while the matrix cores do; behind the last four the loads of the chunk three ahead are
  // issued into the registers this frees.  The weights of a step are requested for the next chunk as soon as the
  // step has used their registers.  AHEAD: 1 there are such chunks, 0 there are none, 2 maybe; a condition around
  // loads makes the wait for older ones wait for these too, hence only near the end.
  constexpr int PF = 8;
  auto run_chunk = [&](auto ahead_c, int chunk, uint32_t (&rn)[16]) {
    constexpr int AHEAD = decltype(ahead_c)::value;
    const uint4* const cells_in = operand + (chunk & 1) * kBufCells;
    uint4 b[PF + 1];
    auto read = [&](int v) {
      const int u = v >> 2, c = v & 3;
      b[v % (PF + 1)] = cells_in[(u / NW) * 4 * (4 * QT) + c * QT + 16 * (u % NW)];
    };
#pragma unroll
    for (int d = 0; d < PF; ++d) read(d);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int ks = u / NW, w = u % NW;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int v = 4 * u + c;
        if (v + PF < 32) read(v + PF);
        __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the multiply
        const uint4 q = b[v % (PF + 1)];
        acc[w][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[ks], v4i{(int)q.x, (int)q.y, (int)q.z, (int)q.w}, acc[w][c], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (w == NW - 1 && (AHEAD == 1 || chunk + 1 < p.chunks)) load_weights(chunk + 1, ks);
      if (u < 4) {
        if (AHEAD == 1 || chunk + 1 < p.chunks) commit(rn, (chunk + 1) & 1, u);
      } else if (AHEAD == 1 || (AHEAD == 2 && chunk + 3 < p.chunks)) {
        issue(rn, chunk + 3, u - 4);
      }
    }
    __syncthreads();
  };
  issue_all(r[0], 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) load_weights(0, ks);
  __builtin_amdgcn_sched_barrier(0);
  // scales and biases behind the first loads: the epilogue of a small call would begin with a wait for memory
  const int row0 = rt * 16 + 4 * kq;
  float sc[4], bi[4];
  if (OUT != kOutAcc32) {
    // arrays are padded to a multiple of 32 rows
    const int row = min(rt, p.row_tiles - 1) * 16 + 4 * kq;
    const float4 s4 = *reinterpret_cast<const float4*>(p.scale + row), b4 = *reinterpret_cast<const float4*>(p.bias + row);
    sc[0] = s4.x, sc[1] = s4.y, sc[2] = s4.z, sc[3] = s4.w;
    bi[0] = b4.x, bi[1] = b4.y, bi[2] = b4.z, bi[3] = b4.w;
  }
  __builtin_amdgcn_sched_barrier(0);
  if (p.chunks >= 3) {
    issue_all(r[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    commit_all(r[0], 0);
    issue_all(r[0], 2);
  } else {
    if (p.chunks == 2) issue_all(r[1], 1);
    commit_all(r[0], 0);
  }
  __syncthreads();
  using Always = std::integral_constant<int, 1>;
  using Maybe = std::integral_constant<int, 2>;
  using Never = std::integral_constant<int, 0>;
  int chunk = 0;
  for (; chunk + 5 <= p.chunks; chunk += 2) {
    run_chunk(Always(), chunk, r[1]);
    run_chunk(Always(), chunk + 1, r[0]);
  }
  // one to four chunks are left
  run_chunk(Maybe(), chunk, r[1]);
  if (chunk + 1 < p.chunks) {
    run_chunk(Maybe(), chunk + 1, r[0]);
    if (chunk + 2 < p.chunks) {
      run_chunk(Never(), chunk + 2, r[1]);
      if (chunk + 3 < p.chunks) run_chunk(Never(), chunk + 3, r[0]);
    }
  }

  // epilogue: lane (n, kq) holds rows 4 kq .. 4 kq + 3 of the row tile at the four positions of quad 16 w + n
  if (row0 >= p.M) return;
  constexpr uint32_t kElem = OUT == kOutI8 ? 1u : 4u;
  // output rows that start on 64-byte boundaries are stored as streaming data; others share sectors with their
  // neighbours, which merge in L2 only if stored plainly (384 -> 384 @28x28 x 16, fp32: 9.2 against 12.2 us;
  // 192 -> 384 @17x17 x 64: 16.2 against 13.4)
  const bool stream = OUT != kOutI8 && (p.hw & 15) == 0;
  DispatchAct(OUT == kOutAcc32 ? 0 : epilogue::LeakyAsMax(p.act), [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
    char* dst[NW];
    int valid[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const uint32_t q = tile_quad0 + 16u * w + (uint32_t)n;
      const uint32_t on = q / (uint32_t)p.qpi;
      const int opp = 4 * (int)(q - on * (uint32_t)p.qpi);
      valid[w] = 16 * w + n >= p.tile_quads || q >= p.total_quads ? 0 : min(4, p.hw - opp);
      dst[w] = static_cast<char*>(p.out) + (((size_t)on * p.M + row0) * p.hw + opp) * kElem;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        if (row0 + i < p.M) {
          u4 v;
          if (OUT == kOutAcc32) {
            v = u4{(uint32_t)acc[w][0][i], (uint32_t)acc[w][1][i], (uint32_t)acc[w][2][i], (uint32_t)acc[w][3][i]};
          } else {
            float f[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) f[c] = __builtin_fmaf((float)acc[w][c][i], sc[i], bi[i]);
            if (OUT == kOutI8) {
              v = u4{TruncPackI8x4(ActQuantF<ACT>(f[0], p.act), ActQuantF<ACT>(f[1], p.act), ActQuantF<ACT>(f[2], p.act), ActQuantF<ACT>(f[3], p.act)), 0u, 0u, 0u};
            } else {
#pragma unroll
              for (int c = 0; c < 4; ++c) f[c] = ActivateT<ACT>(f[c], p.act);
              v = u4{__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3])};
            }
          }
          if (valid[w] == 4) {
            if (OUT == kOutI8) {
              *reinterpret_cast<uint32_t*>(dst[w]) = v.x;
            } else if (stream) {
              __builtin_nontemporal_store(v, reinterpret_cast<u4*>(dst[w]));
            } else {
              *reinterpret_cast<u4*>(dst[w]) = v;
            }
          } else {
#pragma unroll
            for (int c = 0; c < 3; ++c) {
              if (c < valid[w]) {
                if (OUT == kOutI8) {
                  reinterpret_cast<int8_t*>(dst[w])[c] = static_cast<int8_t>(v.x >> (8 * c));
                } else {
                  reinterpret_cast<uint32_t*>(dst[w])[c] = v[c];
                }
              }
            }
          }
        }
        dst[w] += (size_t)p.hw * kElem;
      }
    }
  });
}

// The form for many channels: 256 rows x eight blocks of 16 positions, 256 channels a chunk, twelve wavefronts.  Eight multiply, two row
// tiles with all positions each, so that nobody else loads their weights and an operand cell feeds two matrix instructions.  Four bring in
// the activations: a thread loads 16 positions of eight channels with 16-byte loads (a block behind the last whole one of a channel row is
// the row's last 16 positions; what the block before it holds as well is computed twice and stored once), two chunks ahead of
// the one that it turns into cells.
//
// Why twelve: wavefronts issue in order and loads return in order, so a wavefront that does everything waits for its activations, which
// come from memory, before it gets at weights that L2 has had for long, and a full queue of loads holds its matrix instructions
// back.  2048 -> 2048 @14x14 x 16 with eight wavefronts that do both, in this shape, 21.6 us, in 128 x 256 21.1; this 19.1; the kernel above
// 21.9 (128 x 256 in this form 22.6).  A 16-byte load takes a CU 7.0 ns, as long as an 8-byte one and less than two 4-byte
// ones (3.7), so bytes come in twice as fast as dword by dword.
// What bounds it: the matrix instructions, 0.85 of 1.2 us a chunk, beside 0.9 us in which the 96 KB of a chunk come in; around the
// chunks 9.9 us (launch, first chunk, 2.5 us of stores).  Without any loads 17.3 us, without the multiplies 17.0.
constexpr int kSplitQuads = 32;                   // position quads of a tile
constexpr int kSplitRowTiles = 16;
constexpr int kSplitCells = 16 * 4 * kSplitQuads;  // 16-byte cells of a chunk: (channel group of 16, position of the quad, quad)
constexpr int kSplitSteps = 4;                    // 64-channel steps of a chunk
constexpr int kSplitThreads = 768;

// Where a quad's cells lie: the quads of a block turned round by the block's number over four and the channel group's parity, so that lanes
// that write the same quad of neighbouring blocks (64 bytes apart) and of two groups use all banks.
__device__ __forceinline__ int QuadSlot(int group, int block, int quad) { return 4 * block + ((quad + (block >> 2) + 2 * (group & 1)) & 3); }

template <int OUT>
__device__ __forceinline__ void ChunkSplitBody(const ChunkMfmaParams& p, uint4* xt) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // each XCD owns a contiguous range of tiles, the row groups of one tile follow each other there
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int first_tile = (xcd * p.tiles) >> 3, last_tile = ((xcd + 1) * p.tiles) >> 3;
  const int tile = first_tile + slot / p.row_groups, rg = slot % p.row_groups;
  if (tile >= last_tile) return;

  const uint32_t blocks_per_image = (uint32_t)p.qpi >> 2, tile_block0 = (uint32_t)tile * ((uint32_t)p.tile_quads >> 2);
  const uint32_t total_blocks = p.total_quads >> 2;
  float* const table = reinterpret_cast<float*>(xt + 2 * kSplitCells);
  if (wave >= 8) {
    // the thread's part of a chunk: eight channels (half of group kg) of block j; threads behind the tile's or the tensor's last
    // block repeat that one
    const int j = tid & 7, kg = (tid >> 4) & 15, half = (tid >> 3) & 1;
    const uint32_t block = min(tile_block0 + (uint32_t)min(j, (p.tile_quads >> 2) - 1), total_blocks - 1u);
    const uint32_t img = block / blocks_per_image;
    const int first = min(16 * (int)(block - img * blocks_per_image), p.hw - 16);
    const uint32_t vbase = img * (uint32_t)p.K * (uint32_t)p.hw + (uint32_t)first;
    u4 r[2][8];
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.x), 0, (int)((uint32_t)p.batch * (uint32_t)p.K * (uint32_t)p.hw), 0x00020000);
    auto issue = [&](u4 (&rd)[8], int chunk) {
      // The last group of a channel count that is no multiple of 16 holds the last 16 channels.  Groups behind it meet weights of zero:
      // they lie outside the buffer, so nothing is fetched for them, and no condition around the loads makes the wait for older ones wait for these too.
      const int k = chunk * (64 * kSplitSteps) + 16 * kg;
      const uint32_t voff = k < p.K ? vbase + (uint32_t)((min(k, p.K - 16) + 8 * half) * p.hw) : 0x80000000u;
#pragma unroll
      for (int i = 0; i < 8; ++i) rd[i] = __builtin_amdgcn_raw_buffer_load_b128(xbuf, (int)voff, i * p.hw, 0);
    };
    // two stages of byte permutes: pairs of channels, then the eight bytes of each position
    char* const cells = reinterpret_cast<char*>(xt + kg * (4 * kSplitQuads)) + 8 * half;
    auto commit = [&](u4 (&rd)[8], int buf) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        char* const dst = cells + (buf * kSplitCells + QuadSlot(kg, j, t)) * 16;
#pragma unroll
        for (int pos = 0; pos < 4; pos += 2) {
          uint32_t pair[4];
#pragma unroll
          for (int m = 0; m < 4; ++m) pair[m] = __builtin_amdgcn_perm(rd[2 * m + 1][t], rd[2 * m][t], pos ? 0x07030602u : 0x05010400u);
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const uint32_t sel = c ? 0x07060302u : 0x05040100u;
            *reinterpret_cast<uint2*>(dst + (pos + c) * (kSplitQuads * 16)) = make_uint2(__builtin_amdgcn_perm(pair[1], pair[0], sel), __builtin_amdgcn_perm(pair[3], pair[2], sel));
          }
        }
      }
    };
    issue(r[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    issue(r[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    commit(r[0], 0);
    issue(r[0], 2);
    __syncthreads();
    int chunk = 0;
    for (; chunk + 2 < p.chunks; chunk += 2) {
      commit(r[1], 1);
      issue(r[1], chunk + 3);
      __syncthreads();
      commit(r[0], 0);
      issue(r[0], chunk + 4);
      __syncthreads();
    }
    if (chunk + 1 < p.chunks) {
      commit(r[1], 1);
      __syncthreads();
    }
    __syncthreads();
    return;
  }

  // the wavefront's row tiles (past the last one: the last one again, not stored)
  const int rt = rg * kSplitRowTiles + 2 * wave;
  const int n = lane & 15, kq = lane >> 4;
  const v4i* const wt0 = static_cast<const v4i*>(p.wtiles) + (size_t)min(rt, p.row_tiles - 1) * p.padded_ksteps * 64 + lane;
  const v4i* const wt1 = static_cast<const v4i*>(p.wtiles) + (size_t)min(rt + 1, p.row_tiles - 1) * p.padded_ksteps * 64 + lane;
  v4i a[kSplitSteps][2];
  auto load_weights = [&](int chunk, int ks) {
    a[ks][0] = wt0[(chunk * kSplitSteps + ks) * 64];
    a[ks][1] = wt1[(chunk * kSplitSteps + ks) * 64];
  };
  const uint4* const operand0 = xt + kq * (4 * kSplitQuads) + QuadSlot(kq, n >> 2, n & 3);
  const uint4* const operand1 = xt + kq * (4 * kSplitQuads) + QuadSlot(kq, 4 + (n >> 2), n & 3);
  v4i acc[2][2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int w = 0; w < 2; ++w)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[t][w][c] = v4i{0, 0, 0, 0};

  // One chunk: eight (step, window) pairs of eight multiplies, operand cells read PF cells ahead.  The weights of a step are requested for
  // the next chunk as soon as the step has used their registers.
  constexpr int PF = 4;
  auto run_chunk = [&](auto last_c, int chunk) {
    constexpr bool LAST = decltype(last_c)::value;
    const uint4* const in0 = operand0 + (chunk & 1) * kSplitCells;
    const uint4* const in1 = operand1 + (chunk & 1) * kSplitCells;
    uint4 b[PF + 1];
    auto read = [&](int v) { b[v % (PF + 1)] = (v >> 2 & 1 ? in1 : in0)[(v >> 3) * (16 * kSplitQuads) + (v & 3) * kSplitQuads]; };
#pragma unroll
    for (int d = 0; d < PF; ++d) read(d);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int ks = u >> 1, w = u & 1;
      if (LAST && w == 0 && 64 * (kSplitSteps * chunk + ks) >= p.K) break;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int v = 4 * u + c;
        if (v + PF < 32) read(v + PF);
        __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the multiply
        const uint4 q = b[v % (PF + 1)];
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t][w][c] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[ks][t], v4i{(int)q.x, (int)q.y, (int)q.z, (int)q.w}, acc[t][w][c], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (w == 1 && !LAST) load_weights(chunk + 1, ks);
    }
    __syncthreads();
  };
#pragma unroll
  for (int ks = 0; ks < kSplitSteps; ++ks) load_weights(0, ks);
  // scales and biases of the workgroup's rows wait in LDS (the arrays are padded to a multiple of 32 rows)
  if (OUT != kOutAcc32) {
    const int row = min(rg * (16 * kSplitRowTiles) + (tid & 255), 16 * p.row_tiles - 1);
    table[tid] = tid < 256 ? p.scale[row] : p.bias[row];
  }
  __syncthreads();
  int chunk = 0;
  for (; chunk + 1 < p.chunks; ++chunk) run_chunk(std::false_type(), chunk);
  run_chunk(std::true_type(), chunk);

  // epilogue: lane (n, kq) holds rows 4 kq .. 4 kq + 3 of the row tiles at the four positions of quad n of the windows
  const int row0 = rt * 16 + 4 * kq;
  if (row0 >= p.M) return;
  constexpr uint32_t kElem = OUT == kOutI8 ? 1u : 4u;
  const bool stream = OUT != kOutI8 && (p.hw & 15) == 0;  // as in ChunkBody
  DispatchAct(OUT == kOutAcc32 ? 0 : epilogue::LeakyAsMax(p.act), [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
    char* dst[2];
    int own[2];  // the quad's first position that no block before it holds
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const int bj = 4 * w + (n >> 2);
      const uint32_t ob = tile_block0 + (uint32_t)bj, on = ob / blocks_per_image;
      const int from = 16 * (int)(ob - on * blocks_per_image), opp = min(from, p.hw - 16) + 4 * (n & 3);
      own[w] = bj >= (p.tile_quads >> 2) || ob >= total_blocks ? 4 : min(4, max(0, from - opp));
      dst[w] = static_cast<char*>(p.out) + (((size_t)on * p.M + row0) * p.hw + opp) * kElem;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float s[4], o[4];
      if (OUT != kOutAcc32) {
        const float* const at = table + 32 * wave + 16 * t + 4 * kq;
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = at[i], o[i] = at[256 + i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool row = row0 + 16 * t + i < p.M;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
          if (row) {
            u4 v;
            if (OUT == kOutAcc32) {
              v = u4{(uint32_t)acc[t][w][0][i], (uint32_t)acc[t][w][1][i], (uint32_t)acc[t][w][2][i], (uint32_t)acc[t][w][3][i]};
            } else {
              float f[4];
#pragma unroll
              for (int c = 0; c < 4; ++c) f[c] = __builtin_fmaf((float)acc[t][w][c][i], s[i], o[i]);
              if (OUT == kOutI8) {
                v = u4{TruncPackI8x4(ActQuantF<ACT>(f[0], p.act), ActQuantF<ACT>(f[1], p.act), ActQuantF<ACT>(f[2], p.act), ActQuantF<ACT>(f[3], p.act)), 0u, 0u, 0u};
              } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) f[c] = ActivateT<ACT>(f[c], p.act);
                v = u4{__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3])};
              }
            }
            if (own[w] == 0) {
              if (OUT == kOutI8) {
                *reinterpret_cast<uint32_t*>(dst[w]) = v.x;
              } else if (stream) {
                __builtin_nontemporal_store(v, reinterpret_cast<u4*>(dst[w]));
              } else {
                *reinterpret_cast<u4*>(dst[w]) = v;
              }
            } else {
#pragma unroll
              for (int c = 1; c < 4; ++c) {
                if (c >= own[w]) {
                  if (OUT == kOutI8) {
                    reinterpret_cast<int8_t*>(dst[w])[c] = static_cast<int8_t>(v.x >> (8 * c));
                  } else {
                    reinterpret_cast<uint32_t*>(dst[w])[c] = v[c];
                  }
                }
              }
            }
          }
          dst[w] += (size_t)p.hw * kElem;
        }
      }
#pragma unroll
      for (int w = 0; w < 2; ++w) dst[w] += (size_t)(12 * p.hw) * kElem;
    }
  });
}

template <int OUT>
__global__ void __launch_bounds__(kSplitThreads, 3) ChunkSplitKernel(PL_HEAD_PARAMS, const ChunkMfmaParams block) {
  const ChunkMfmaParams p = WithHead(block, PL_HEAD_ARGS);
  extern __shared__ uint4 xt[];
  ChunkSplitBody<OUT>(p, xt);
}

template <int NW, int OUT>
__global__ void __launch_bounds__(512, 2) ChunkMfmaKernel(PL_HEAD_PARAMS, const ChunkMfmaParams block) {
  const ChunkMfmaParams p = WithHead(block, PL_HEAD_ARGS);
  extern __shared__ uint4 xt[];
  ChunkBody<NW, OUT>(p, xt);
}

template <int OUT>
hipError_t Launch(const ChunkMfmaPlan& plan, const ChunkMfmaParams& p, dim3 grid, hipStream_t s) {
  const dim3 block(512);
  if (plan.split) return LaunchWithHead(ChunkSplitKernel<OUT>, grid, dim3(kSplitThreads), (size_t)2 * kSplitCells * 16 + 2048, s, p);
  const size_t lds = 2 * kBufCells * 16;
  if (plan.nw == 4) return LaunchWithHead(ChunkMfmaKernel<4, OUT>, grid, block, lds, s, p);
  if (plan.nw == 2) return LaunchWithHead(ChunkMfmaKernel<2, OUT>, grid, block, lds, s, p);
  return LaunchWithHead(ChunkMfmaKernel<1, OUT>, grid, block, lds, s, p);
}

}  // namespace

int ChunkMfmaPaddedSteps(int K) { return (K + 511) / 512 * 8; }
bool ChunkMfmaFits(int K, int hw) { return K >= 16 && hw >= 4; }

static ChunkMfmaPlan PlanChunkSplit(int K, int M, int hw, int batch) {
  ChunkMfmaPlan p{};
  p.split = true;
  p.tile_quads = kSplitQuads;
  p.tiles = (int)(((int64_t)batch * ((hw + 15) / 16) + kSplitQuads / 4 - 1) / (kSplitQuads / 4));
  p.row_groups = ((M + 15) / 16 + kSplitRowTiles - 1) / kSplitRowTiles;
  p.chunks = ((K + 63) / 64 + kSplitSteps - 1) / kSplitSteps;
  p.workgroups = 8ll * p.row_groups * ((p.tiles + 7) / 8);
  return p;
}

// Where the form with twelve wavefronts is expected to be ahead of the tile width `plan` chose: a CU holds one of its workgroups, which takes
// about 4.4 us and 1.1 us per chunk of 256 channels.  us, the width chosen / this: 2048 -> 2048 @14x14 x 16 22.0 / 19.0, 1024 -> 512 @17x17 x 32
// 18.4 / 14.5, 900 -> 384 @13x13 x 60 15.5 / 13.0, 1024 -> 2048 @14x14 x 64 51.4 / 46.1; not taken: 192 -> 384 @17x17 x 64 (304
// workgroups) 12 / 15, 1024 -> 1024 @14x14 x 16 (half the CUs) 11.3 / 12.6, 1500 -> 700 @10x10 x 20 9.5 / 13.6.
// In place of a single round of 128 positions, which take as many chunks, it must be expected to take less than 0.9 of the time: of 17 calls between that
// and level 16 were slower, 1.09 times in the middle (1590 -> 1406 @40x40 11.6 / 13.1), in place of 256 positions none of 38 (162 -> 1888 @11x11 x 20
// 11.1 / 8.6).  Over more rounds 5 of 1388 calls are, to 1.14 (1169 -> 125 @14x14 x 1583).
static bool SplitPays(int cus, const ChunkMfmaPlan& plan, const ChunkMfmaPlan& split) {
  const int64_t rounds = (plan.workgroups + cus - 1) / cus, others = rounds * (300 + 135 * plan.chunks), own = (split.workgroups + cus - 1) / cus * (440 + 110 * split.chunks);
  return rounds == 1 && plan.nw == 2 ? own * 10 < others * 9 : own < others;
}

ChunkMfmaPlan PlanChunkMfma(int out_kind, int cus, int tile_positions, int split, int K, int M, int hw, int batch) {
  const bool split_fits = split != 0 && hw >= 16;
  if (split_fits && split == 2) return PlanChunkSplit(K, M, hw, batch);
  const int qpi = (hw + 3) / 4, ksteps = (K + 63) / 64;
  const int64_t total_quads = (int64_t)batch * qpi;
  auto plan_for = [&](int nw) {
    ChunkMfmaPlan p{};
    p.nw = nw;
    // whole images per tile where they fit: their channel rows lie back to back, so no line is fetched in parts
    p.tile_quads = qpi <= 16 * nw ? 16 * nw / qpi * qpi : 16 * nw;
    p.tiles = (int)((total_quads + p.tile_quads - 1) / p.tile_quads);
    p.row_groups = ((M + 15) / 16 + 7) / 8;
    p.chunks = (ksteps + 8 / nw - 1) / (8 / nw);
    p.workgroups = 8ll * p.row_groups * ((p.tiles + 7) / 8);
    return p;
  };
  if (tile_positions != 0) return plan_for(tile_positions / 64);  // a width that is asked for is that of the form above
  // The tile width: a CU holds one workgroup, a workgroup takes about 3 us and 1.35 us per chunk, so the fewest rounds
  // times that, rounds being what the XCD with the most workgroups needs.  2048 -> 2048 @14x14 x 16: 256 positions 24.7 us
  // (one round of 16 chunks), 128 36.6 (two of 8), 64 44.7 (four of 4); 1024 -> 256 @14x14 x 32: 14.6, 12.7 and 9.9 (one
  // round each); 608 -> 736 @9x8 x 42: 11.4 (one round), 13.2 and 12.9 (two).
  const ChunkMfmaPlan widest = plan_for(4);
  ChunkMfmaPlan best{};
  int64_t least = 0;
  for (int nw : {1, 2, 4}) {
    const ChunkMfmaPlan p = nw == 4 ? widest : plan_for(nw);
    const int64_t cost = (p.workgroups + cus - 1) / cus * (300 + 135 * p.chunks);
    if (nw == 1 || cost < least) least = cost, best = p;
  }
  // Over several rounds what all workgroups together read counts more than how full the last round is, and the widest
  // tile reads the weights the fewest times: it from a round and a half of its workgroups on (with one-byte output and on
  // ragged maps, where whole images leave up to a fifth of a tile empty, beyond two and a half).  us with the width of the
  // formula above / the widest: 2048 -> 2048 @14x14 x 64 131 / 98 (int8 output 111 / 89), 1280 -> 2048 @14x14 x 128 195 /
  // 149, 2048 -> 1024 @28x28 x 24 96 / 84; at two and a half rounds 768 -> 1024 @14x14 x 80 with int8 output 35.0 / 36.6,
  // 2048 -> 1024 @7x7 x 300 101 / 112.
  const bool few_rounds_count = out_kind == kOutI8 || hw % 4 != 0;
  if (few_rounds_count ? 2 * widest.workgroups > 5ll * cus : 2 * widest.workgroups >= 3ll * cus) best = widest;
  if (split_fits) {
    const ChunkMfmaPlan own = PlanChunkSplit(K, M, hw, batch);
    if (SplitPays(cus, best, own)) return own;
  }
  return best;
}

hipError_t LaunchChunkMfma(int out_kind, int cus, int tile_positions, int split, const ChunkMfmaParams& p, hipStream_t stream) {
  if (p.batch <= 0 || p.M <= 0) return hipSuccess;
  if (!ChunkMfmaFits(p.K, p.hw)) return hipErrorInvalidValue;
  const int64_t positions = (int64_t)p.batch * p.hw;
  // tensor offsets are kept in 32 bits
  if (positions * p.K >= (1ll << 31) || positions >= (1ll << 31) - 512) return hipErrorInvalidValue;
  const ChunkMfmaPlan plan = PlanChunkMfma(out_kind, cus, tile_positions, split, p.K, p.M, p.hw, p.batch);
  ChunkMfmaParams q = p;
  q.qpi = plan.split ? 4 * ((p.hw + 15) / 16) : (p.hw + 3) / 4;
  q.quad_aligned = p.hw % 4 == 0;
  q.total_quads = (uint32_t)p.batch * (uint32_t)q.qpi;
  q.row_tiles = (p.M + 15) / 16;
  q.padded_ksteps = ChunkMfmaPaddedSteps(p.K);
  q.row_groups = plan.row_groups;
  q.tile_quads = plan.tile_quads;
  q.tiles = plan.tiles;
  q.chunks = plan.chunks;
  if (plan.workgroups > (1ll << 30)) return hipErrorInvalidValue;
  const dim3 grid((uint32_t)plan.workgroups);
  switch (out_kind) {
    case kOutF32:
      return Launch<kOutF32>(plan, q, grid, stream);
    case kOutI8:
      return Launch<kOutI8>(plan, q, grid, stream);
    case kOutAcc32:
      return Launch<kOutAcc32>(plan, q, grid, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace pl
