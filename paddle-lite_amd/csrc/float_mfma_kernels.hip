// Floating-point sparse 1x1 convolution as a dense product on the matrix cores (v_mfma_f32_32x32x16_f16), the channels
// taken chunk by chunk, for the calls whose nonzeros cost a walk more than all weights cost here.
//
// One workgroup of eight wavefronts makes a tile of WR x 32 output rows x 128 positions (32 quads).  Per chunk of 64
// channels a thread loads four channels of one position quad, turns them into operand cells (eight channels of one
// position, 16 bytes) and writes these to one of two LDS buffers while the other one is multiplied; a wavefront owns 32
// rows (WR = 8), or shares them with KH - 1 others that take the other channels of every chunk (WR = 4, 2).  Weights
// come straight into registers, a chunk ahead.  One barrier per chunk.  The vector ALU's share of a step is spread
// between its matrix instructions: wavefronts issue in order, and both of a SIMD are at the same place.
//
// fp16: products and sums are exact to fp32, rounded to half precision once before the activation, which runs in half
// precision as in the walks (against 64 bits 2.1e-4 in 2-norm, the walks, whose sums are binary16, 8e-4 .. 2.6e-3).
// fp32: inputs and weights as two binary16 pieces each, the second one times 2^11, and three of the four products.  A
// row's weights are scaled by a power of two at prepare, a position's inputs by one that follows the largest of them seen
// so far.  A scaled value of 2^-13 and more is within 2^-23 of its pieces' sum, which is 2^-25 of its position's largest; a smaller one
// keeps an absolute error of 2^-36.  The products with a low piece have sums of their own: the matrix cores cut sums off instead
// of rounding them, and every addition to the large sum costs up to an ulp of it (512 channels, 85 % zeros, against 64
// bits: 2.2e-7 in 2-norm with one sum, 1.4e-7 with two; the walks 1.6e-7).  Products with a zero weight add nothing, whatever the
// input (a sum is cut off below its largest product that is not zero).
//
// What a dense product would get wrong is walked nonzero by nonzero at the end: outputs that an infinity or a NaN reached
// through a zero weight, and in fp32 outputs too small for the absolute error of the small inputs of their position.  The quads
// that hold such an input, or whose scale went down by more than 2^64, are marked; the error of a row there is at most 2^-36 of the sum of its scaled weights'
// magnitudes, so a result of 2^-13 of that sum and more is within 2^-23, and anything less is walked.
//
// What bounds it: no unit alone.  64 x 512 -> 512 @14x14 in fp32, per CU (counters): matrix cores busy 49 % of the time, vector ALU 24 %
// beside the matrix instructions' issue, LDS 26 %, 36 KB per us from L2 (47 - 53 inside the loop: a chunk of the widest form is 96 KB in
// fp32, 64 of them weights, and half in fp16, and takes 2.0 and 0.9 us, its matrix instructions alone 1.35 and 0.45).  One barrier per chunk
// keeps the wavefronts in step, so that the vector ALU's work adds to the rest: the search for small inputs, three of
// eleven instructions per pair of values, costs 2 - 3 % with 256 rows and 4 % with 64 (13 % there at 32 chunks).  More chunks
// in flight gain nothing (four instead of two: fp16 15.0 -> 16.9 us, the first chunk only arrives later).
// Hence 256 rows x 128 positions (128 x 256 has every weight fetched by two wavefronts: fp16 20.0 against 17.1 us at the
// time), hence nothing staged twice.  us per launch, buffers rotating over 320 MB, the walk that ran before / this one:
// fp16 64 x 512 -> 512 @14x14, 85 % zeros 29.1 / 14.4; fp16 8 x 128 -> 256 @55x55, row pairs, 70 % 20.7 / 9.5; fp32 64 x 512 -> 512
// @14x14, 85 % 33.0 / 25.4; fp32 64 x 1024 -> 1024 @7x7, row pairs, 70 % 61.0 / 28.8.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "epilogue.h"
#include "half_act.h"
#include "kernarg_head.h"
#include "launch_lds.h"
#include "sparse_conv_kernels.h"

namespace pl {
namespace {

using epilogue::ActivateT;
using epilogue::DispatchAct;
using half_act::ActivateH;
using half_act::h1;
using half_act::h2;

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v2f __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));

constexpr int kChunk = kFloatMfmaChunk;  // channels of a chunk
constexpr int kSteps = kChunk / 16;      // matrix instructions' channel steps of a chunk
constexpr int kQuads = 32;               // position quads of a tile
constexpr int kThreads = 512;
constexpr int kGroups = kChunk / 8;      // operand cells of a position and chunk (eight channels each)
// A scaled input is kept times kFloatMfmaLow.  A new scale from kPeak on; a mark below kSmallBits, which is kFloatMfmaSmall
// as the inputs are compared: bits without the sign, less one, so that zero is the largest.
constexpr float kPeak = 0x1p15f * kFloatMfmaLow;
constexpr uint32_t kSmallBits = (125u << 24) - 1u;
static_assert(kFloatMfmaSmall * kFloatMfmaLow == 0x1p-2f, "kSmallBits");

// what the first loads need arrives in registers
PL_IN_HEAD(FloatMfmaParams, x);
PL_IN_HEAD(FloatMfmaParams, wtiles);
PL_IN_HEAD(FloatMfmaParams, K);
PL_IN_HEAD(FloatMfmaParams, hw);
PL_IN_HEAD(FloatMfmaParams, batch);
PL_IN_HEAD(FloatMfmaParams, qpi);
PL_IN_HEAD(FloatMfmaParams, total_quads);
PL_IN_HEAD(FloatMfmaParams, chunks);
PL_IN_HEAD(FloatMfmaParams, tiles);
PL_IN_HEAD(FloatMfmaParams, row_groups);
PL_IN_HEAD(FloatMfmaParams, row_blocks);

// Four neighbouring positions of one channel.
template <bool F32>
using Quad = std::conditional_t<F32, u4, u2>;

// What the nonzeros at .. of a row's list (every step-th from there on) add to four neighbouring positions of x.
// Eight entries at a time: their channels and weights first, then the inputs; the list's padding reads channel 0 and adds nothing.
template <bool F32>
__device__ __forceinline__ void WalkRow(const FloatMfmaParams& p, const char* x, int row, uint32_t at, uint32_t step, float (&acc)[4]) {
  constexpr int kBatch = 8;
  constexpr uint32_t kElem = F32 ? 4u : 2u;
  const DevGroup g = p.groups[p.nr == 2 ? row >> 1 : row];
  const int r = row - g.row0;
  for (uint32_t e = at; e < g.count; e += kBatch * step) {
    uint32_t k[kBatch], w[kBatch];
    Quad<F32> v[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const uint32_t from = g.first + min(e + (uint32_t)u * step, g.count - 1u);
      k[u] = p.kidx[from];
      w[u] = F32 ? p.wts[(size_t)from * p.nr + r] : p.wts[from] >> (16 * r);
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (e + (uint32_t)u * step >= g.count) k[u] = (uint32_t)p.K;
      __builtin_memcpy(&v[u], x + (size_t)(k[u] < (uint32_t)p.K ? k[u] : 0u) * ((uint32_t)p.hw * kElem), sizeof(v[u]));
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      if (k[u] >= (uint32_t)p.K) continue;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if constexpr (F32) {
          acc[c] = __builtin_fmaf(__uint_as_float(v[u][c]), __uint_as_float(w[u]), acc[c]);
        } else {
          const uint32_t word = v[u][c >> 1];
          acc[c] = __builtin_fmaf((float)half_act::HalfBits((uint16_t)(word >> (16 * (c & 1)))), (float)half_act::HalfBits((uint16_t)w[u]), acc[c]);
        }
      }
    }
  }
}

// LDS: two buffers of operand cells, or what the wavefronts of a row block hand to each other at the end; behind either
// (a wavefront may still look at a flag when another has begun to hand over), for fp32, the positions' maxima, the two
// flags, the marks of the quads and the positions' first scales.
constexpr int kF32Tables = (4 * kQuads + 4 + kQuads + 4 * kQuads) * 4;
constexpr int LdsTables(int wr, bool f32) {
  const int cells = 2 * (f32 ? 2 : 1) * kGroups * 4 * kQuads * 16, trade = 8 * (64 - 8 * wr) * 64 * 4;
  return cells > trade ? cells : trade;
}

// Bias, activation and store of the positions of a quad that `bits` names; the quad's first output in row 0 of its image lies `to` elements into out.
template <bool F32>
__device__ __forceinline__ void StoreWalked(const FloatMfmaParams& p, const float (&acc)[4], uint32_t bits, int row, uint32_t to) {
  constexpr uint32_t kElem = F32 ? 4u : 2u;
  char* const dst = static_cast<char*>(p.out) + ((size_t)to + (size_t)(uint32_t)row * (uint32_t)p.hw) * kElem;
  DispatchAct(p.act.type, [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
    const uint32_t h0 = p.act_h_words[0], h1w = p.act_h_words[1];
    const DevActH act_h = {ACT, (uint16_t)h0, (uint16_t)(h0 >> 16), (uint16_t)h1w, (uint16_t)(h1w >> 16)};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if ((bits >> c & 1u) == 0) continue;
      if constexpr (F32) {
        reinterpret_cast<float*>(dst)[c] = ActivateT<ACT>(acc[c] + (p.bias ? static_cast<const float*>(p.bias)[row] : 0.0f), p.act);
      } else {
        const h1 v = (h1)(acc[c] + (p.bias ? (float)static_cast<const h1*>(p.bias)[row] : 0.0f));
        reinterpret_cast<h1*>(dst)[c] = ActivateH<ACT>(h2{v, v}, act_h).x;
      }
    }
  });
}

// The outputs that the product could not give, by the whole wavefront: lane (n, half) brings the bits of its own (4 i + c: row
// first_row + 8 (i / 4) + 4 half + i % 4, position c of quad n).  A row with many such quads
// is walked by two lanes per quad, others by sixteen lanes per row and quad, four of these at a time.
// What bounds it: with few quads two memory round trips per sixteen lanes' entries, with all of them the inputs, which every
// row's nonzeros fetch again from L1 and L2.  fp32 16 x 512 -> 512 @14x14, 85 % zeros, one NaN / a NaN in every position: every lane
// its own outputs, one value after the other, 108 / 436 us; this 23 / 70 (without any 14, the walk 15).
template <bool F32>
__device__ __forceinline__ void WalkOutputs(const FloatMfmaParams& p, uint64_t walk, int fin, int first_row, uint32_t first_quad) {
  constexpr uint32_t kElem = F32 ? 4u : 2u;
  constexpr int kManyQuads = 8;
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), n = lane & 31, half = lane >> 5;  // not held in a register meanwhile
  const uint32_t image = (first_quad + (uint32_t)n) / (uint32_t)p.qpi;
  const int position = 4 * (int)(first_quad + (uint32_t)n - image * (uint32_t)p.qpi);
  const uint32_t inside = (uint32_t)min(position, p.hw - 4);
  const uint32_t from_own = image * (uint32_t)p.K * (uint32_t)p.hw + inside, to_own = image * (uint32_t)p.M * (uint32_t)p.hw + inside;
  int next = 0, row = 0, half_of = 0;
  uint32_t quads = 0, bits = 0;  // of the present row: quads left; the lane's own four bits
  for (;;) {
    int taken = 0, quad = 0, item_row = 0;
    uint32_t item_bits = 0;
    bool many = false;
    while (taken < 4) {
      if (quads == 0) {
        if (next == 2 * fin) break;
        const int i = next >> 1;
        half_of = next & 1;
        ++next;
        bits = half == half_of ? (uint32_t)(walk >> (4 * i)) & 15u : 0u;
        quads = (uint32_t)(__ballot(bits != 0) >> (32 * half_of));
        row = first_row + 8 * (i >> 2) + 4 * half_of + (i & 3);
        continue;
      }
      if (__popc(quads) > kManyQuads) {
        if (taken != 0) break;  // the next time
        many = true;
        quads = 0;
        quad = n, item_row = row, item_bits = (uint32_t)__shfl((int)bits, n + 32 * half_of);
        break;
      }
      const int q = __ffs(quads) - 1;
      quads &= quads - 1;
      const uint32_t b = (uint32_t)__shfl((int)bits, q + 32 * half_of);
      if (lane >> 4 == taken) quad = q, item_row = row, item_bits = b;
      ++taken;
    }
    if (taken == 0 && !many) break;
    const uint32_t from = (uint32_t)__shfl((int)from_own, quad), to = (uint32_t)__shfl((int)to_own, quad);
    const uint32_t at = many ? half : lane & 15;
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (item_bits != 0) WalkRow<F32>(p, static_cast<const char*>(p.x) + (size_t)from * kElem, item_row, at, many ? 2 : 16, acc);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (many) {
        acc[c] += __shfl_xor(acc[c], 32);
      } else {
#pragma unroll
        for (int m = 8; m >= 1; m >>= 1) acc[c] += __shfl_xor(acc[c], m);
      }
    }
    if (item_bits == 0 || at != 0) continue;
    StoreWalked<F32>(p, acc, item_bits, item_row, to);
  }
}

// The same for wavefronts whose lanes hold 16 quads (n) in four parts (kq): the lane's row i is row first_row + 16 (i / 4) + 4 kq + i % 4.  Up to
// kStagedQuads quads of which eight rows and more are walked have their inputs brought to LDS: from memory every nonzero of every row fetches
// a line of its own for them, and one CU does the work of 256 rows.  Two positions of up to 2048 channels at a time, those without such an output
// left out.  Eight rows at a time, two by sixteen lanes.
// Of more quads every lane walks its own rows where more than half of the lanes have such outputs in their rows i, else sixteen lanes walk one row
// for one quad, four of these at a time.
// What bounds it: with one quad its inputs and lists on the one CU, with all of them the inputs.  Time with one NaN / one in every position, of that
// with the form above (119 calls of 400 - 2048 channels that the rule gives to this one): 0.84 / 1.00 at
// the median, 0.93 / 1.36 at most; with every row's inputs from memory 1.24 / 1.01, 1.63 / 1.48 at most.
constexpr int kStagedBytes = 16 * 1024, kStagedFirst = 8 * 1024, kStagedQuads = 6;  // of a wavefront; those in the first of its two parts of LDS; quads
constexpr int kStagedSums = 33 * 8;  // zeros and a wavefront's sums
__device__ __forceinline__ void WalkOutputs16(const FloatMfmaParams& p, uint32_t walk, int first_row, uint32_t first_quad, const void* part0, const void* part1, const void* part2) {
  const int lane = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), n = lane & 15;
  const uint32_t image = (first_quad + (uint32_t)n) / (uint32_t)p.qpi;
  const int position = 4 * (int)(first_quad + (uint32_t)n - image * (uint32_t)p.qpi);
  const uint32_t inside = (uint32_t)min(position, p.hw - 4);
  const uint32_t from_own = image * (uint32_t)p.K * (uint32_t)p.hw + inside, to_own = image * (uint32_t)p.M * (uint32_t)p.hw + inside;

  int rows_of_quad = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) rows_of_quad += (walk >> (4 * i) & 15u) != 0;
  rows_of_quad += __shfl_xor(rows_of_quad, 16);
  rows_of_quad += __shfl_xor(rows_of_quad, 32);
  uint32_t staged = (uint32_t)__ballot(rows_of_quad >= 8) & 0xffffu;
  if (__popc(staged) > kStagedQuads) staged = 0;
  const uint32_t few = staged >> n & 1u ? 0u : walk;
  // two positions at a time
  constexpr int W = 2, CELLS = kStagedBytes / (4 * W), LOADS = 16, BATCH = 8;
  typedef __attribute__((address_space(3))) v2f lds;
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(part0)), apart = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(part1)) - base - kStagedFirst;
  auto at_lds = [&](uint32_t i) { return reinterpret_cast<lds*>(base + i * (4u * W) + (i >= kStagedFirst / (4u * W) ? apart : 0u)); };
  lds* const zeros = reinterpret_cast<lds*>(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(part2)));
  lds* const sums = zeros + 1;
  *zeros = v2f{0.0f, 0.0f};
#pragma unroll 1
  for (int item = 0; staged != 0; ++item) {
    const int q = __ffs(staged) - 1, c = W * (item & 1);
    if ((item & 1) != 0) staged &= staged - 1;
    if (__ballot(n == q && (walk & 0x33333333u << c) != 0) == 0) continue;
    const char* const x = static_cast<const char*>(p.x) + ((size_t)(uint32_t)__shfl((int)from_own, q) + (uint32_t)c) * 4;
    const uint32_t to = (uint32_t)__shfl((int)to_own, q) + (uint32_t)c;
#pragma unroll 1
    for (int c0 = 0; c0 < p.K; c0 += CELLS) {
#pragma unroll 1
      for (int i = 0; i < CELLS && c0 + i < p.K; i += 64 * LOADS) {
        v2f v[LOADS];
#pragma unroll
        for (int u = 0; u < LOADS; ++u) __builtin_memcpy(&v[u], x + (size_t)min(c0 + i + 64 * u + lane, p.K - 1) * ((uint32_t)p.hw * 4u), 4 * W);
#pragma unroll
        for (int u = 0; u < LOADS; ++u) *at_lds(i + 64 * u + lane) = v[u];
      }
      const uint32_t present = (uint32_t)min(CELLS, p.K - c0);
      // lanes read what others wrote; LDS serves a wavefront in order
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll 1
      for (int pass = 0; pass < 4; ++pass) {
        uint32_t bits[2], first[2], count[2], most = 0;
        int of[2];
        float acc[2][W];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int r = 8 * pass + 2 * (lane >> 4) + j;  // of the wavefront's 32
          bits[j] = (uint32_t)__shfl((int)walk, q + 16 * (r >> 2 & 3)) >> (4 * (4 * (r >> 4) + (r & 3)) + c) & ((1u << W) - 1u);
          const int row = bits[j] != 0 ? first_row + r : 0;
          const DevGroup g = p.groups[p.nr == 2 ? row >> 1 : row];
          const bool any = bits[j] != 0 && g.count != 0;
          first[j] = any ? g.first : 0u, count[j] = any ? g.count : 0u, of[j] = any ? row - g.row0 : 0;
          most = max(most, count[j]);
          const v2f before = c0 != 0 && n == 0 ? sums[r] : v2f{0.0f, 0.0f};
#pragma unroll
          for (int i = 0; i < W; ++i) acc[j][i] = before[i];
        }
        for (uint32_t e = (uint32_t)n; e < most; e += BATCH * 16) {
          uint32_t k[2][BATCH], w[2][BATCH];
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
              const uint32_t entry = first[j] + min(e + 16u * u, max(count[j], 1u) - 1u);
              k[j][u] = p.kidx[entry];
              w[j][u] = p.wts[(size_t)entry * p.nr + of[j]];
            }
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int u = 0; u < BATCH; ++u) {
              // zeros for what is not there: channels of another window, what pads the lists
              const uint32_t at = k[j][u] - (uint32_t)c0;
              const v2f in = *(e + 16u * u < count[j] && at < present ? at_lds(at) : zeros);
#pragma unroll
              for (int i = 0; i < W; ++i) acc[j][i] = __builtin_fmaf(in[i], __uint_as_float(w[j][u]), acc[j][i]);
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < W; ++i)
#pragma unroll
            for (int m = 8; m >= 1; m >>= 1) acc[j][i] += __shfl_xor(acc[j][i], m);
        if (n == 0) {
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            const int r = 8 * pass + 2 * (lane >> 4) + j;
            if (c0 + CELLS < p.K) {
              sums[r] = v2f{acc[j][0], acc[j][1]};
            } else if (bits[j] != 0) {
              const float out[4] = {acc[j][0], acc[j][1]};
              StoreWalked<true>(p, out, bits[j], first_row + r, to);
            }
          }
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
  }
#pragma unroll 1
  for (int i = 0; i < 8; ++i) {
    const uint32_t bits = (few >> (4 * i)) & 15u;
    uint64_t left = __ballot(bits != 0);
    const int row0 = first_row + 16 * (i >> 2) + (i & 3);
    if (__popcll(left) > 32) {
      float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (bits != 0) {
        WalkRow<true>(p, static_cast<const char*>(p.x) + (size_t)from_own * 4, row0 + 4 * (lane >> 4), 0, 1, acc);
        StoreWalked<true>(p, acc, bits, row0 + 4 * (lane >> 4), to_own);
      }
      continue;
    }
    while (left != 0) {
      int from = lane;
      bool taken = false;
#pragma unroll
      for (int item = 0; item < 4; ++item) {
        if (left == 0) break;
        const int of = __ffsll((unsigned long long)left) - 1;
        left &= left - 1;
        if (lane >> 4 == item) from = of, taken = true;
      }
      const uint32_t item_bits = (uint32_t)__shfl((int)bits, from), at = (uint32_t)__shfl((int)from_own, from), to = (uint32_t)__shfl((int)to_own, from);
      const int row = row0 + 4 * (from >> 4);
      float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      if (taken) WalkRow<true>(p, static_cast<const char*>(p.x) + (size_t)at * 4, row, n, 16, acc);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int m = 8; m >= 1; m >>= 1) acc[c] += __shfl_xor(acc[c], m);
      if (taken && n == 0) StoreWalked<true>(p, acc, item_bits, row, to);
    }
  }
}

template <int WR, bool F32, bool RAGGED>
__device__ __forceinline__ void FloatMfmaBody(const FloatMfmaParams& p, uint4* xt) {
  constexpr int QT = kQuads;               // position quads of a tile
  constexpr int UC = 4;                    // channels a thread brings in of a chunk: half a cell
  constexpr int KH = 8 / WR;               // wavefronts that share a row block, each with its part of a chunk's steps
  constexpr int STEPS = kSteps / KH;       // steps of one of them
  constexpr int FIN = 16 / KH;             // rows per lane that a wavefront finishes
  constexpr int PIECES = F32 ? 2 : 1;      // binary16 pieces of a value
  constexpr int DEPTH = 2;                 // chunks of activations in registers
  constexpr int ADEPTH = 1;                // chunks of weights in registers
  constexpr int kCells = kGroups * 4 * QT; // cells of a chunk and piece
  constexpr int kBuf = PIECES * kCells;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // each XCD owns a contiguous range of tiles, the row groups of one tile follow each other there
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int first_tile = (xcd * p.tiles) >> 3, last_tile = ((xcd + 1) * p.tiles) >> 3;
  const int tile = first_tile + slot / p.row_groups, rg = slot % p.row_groups;
  if (tile >= last_tile) return;

  // the thread's part of a chunk: UC channels of quad j; a partial quad (the end of an image whose size is not a multiple
  // of 4) is the last four positions of its channel row, the first of which belong to the quad before; threads behind the tensor's last quad
  // repeat that one
  const int part = (tid / QT) & 1, j = tid & (QT - 1), kg = tid / (QT * 2);
  const uint32_t tile_quad0 = (uint32_t)tile * (uint32_t)QT;
  const uint32_t quad = min(tile_quad0 + (uint32_t)j, p.total_quads - 1u);
  const uint32_t img = quad / (uint32_t)p.qpi;
  const int pp = 4 * (int)(quad - img * (uint32_t)p.qpi);
  const int first = min(pp, p.hw - 4);
  constexpr uint32_t kElem = F32 ? 4u : 2u;
  const uint32_t vbase = img * (uint32_t)p.K * (uint32_t)p.hw + (uint32_t)first;
  Quad<F32> r[DEPTH][UC];
  // Loads of one chunk.  The last group of a channel count that is no multiple of 8 holds the last eight channels,
  // groups behind it repeat it against weights of zero.  Chunks behind the last one lie outside the buffer: nothing is
  // fetched for them, and no condition around the loads makes the wait for older ones wait for these too.
  const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), 0, (int)((uint32_t)p.batch * (uint32_t)p.K * (uint32_t)p.hw * kElem), 0x00020000);
  const int pitch_in = p.hw * (int)kElem;
  auto issue = [&](Quad<F32> (&rd)[UC], int chunk) {
    const uint32_t k = (uint32_t)(min(chunk * kChunk + 8 * kg, p.K - 8) + UC * part);
    const uint32_t voff = chunk < p.chunks ? (vbase + k * (uint32_t)p.hw) * kElem : kFloatMfmaOutside;
#pragma unroll
    for (int i = 0; i < UC; ++i) {
      if constexpr (F32) {
        rd[i] = __builtin_amdgcn_raw_buffer_load_b128(xbuf, (int)voff, i * pitch_in, 0);
      } else {
        rd[i] = __builtin_amdgcn_raw_buffer_load_b64(xbuf, (int)voff, i * pitch_in, 0);
      }
    }
  };
  // the operand cells of position c of the quad: eight channels
  char* const cells = reinterpret_cast<char*>(xt + kg * (4 * QT) + j) + 2 * UC * part;
  // fp32: every position's inputs are scaled by a power of two that follows the largest of them seen so far (below); this is
  // kFloatMfmaLow times that
  [[maybe_unused]] float scale[4];
  [[maybe_unused]] float peak = 0.0f;
  [[maybe_unused]] uint32_t low = 0xffffffffu;  // the smallest magnitude but zero, as kSmallBits
  auto put = [](char* dst, const uint32_t (&d)[UC / 2]) {
    *reinterpret_cast<u2*>(dst) = u2{d[0], d[1]};
  };
  auto commit = [&](Quad<F32> (&rd)[UC], int buf, int c) {
    char* dst = cells + (buf * kBuf + c * QT) * 16;
    if constexpr (F32) {
      uint32_t hi[UC / 2], lo[UC / 2];
#pragma unroll
      for (int i = 0; i < UC / 2; ++i) {
        // the first pieces are one mixed-precision multiply-add each
        const float a = __uint_as_float(rd[2 * i][c]) * scale[c], b = __uint_as_float(rd[2 * i + 1][c]) * scale[c];
        peak = fmaxf(fmaxf(peak, fabsf(a)), fabsf(b));
        low = min(min(low, (__float_as_uint(a) << 1) - 1u), (__float_as_uint(b) << 1) - 1u);
        const h2 both = {(h1)__builtin_fmaf(a, 1.0f / kFloatMfmaLow, 0.0f), (h1)__builtin_fmaf(b, 1.0f / kFloatMfmaLow, 0.0f)};
        uint32_t word = __builtin_bit_cast(uint32_t, both);
        asm("" : "+v"(word));  // the second value is taken from the word, not converted again
        const h2 h = __builtin_bit_cast(h2, word);
        const h2 l = __builtin_convertvector((v2f{__builtin_fmaf((float)h.x, -kFloatMfmaLow, a), __builtin_fmaf((float)h.y, -kFloatMfmaLow, b)}), h2);
        hi[i] = __builtin_bit_cast(uint32_t, h), lo[i] = __builtin_bit_cast(uint32_t, l);
      }
      put(dst, hi);
      put(dst + kCells * 16, lo);
    } else {
      const uint32_t sel = c & 1 ? 0x07060302u : 0x05040100u;
      uint32_t d[UC / 2];
#pragma unroll
      for (int i = 0; i < UC / 2; ++i) d[i] = __builtin_amdgcn_perm(rd[2 * i + 1][c >> 1], rd[2 * i][c >> 1], sel);
      put(dst, d);
    }
  };

  // the wavefront's row block (past the last one: the last one again, not stored) and window of 32 quads
  const int rb = rg * WR + wave % WR, kh = wave / WR;
  const int n = lane & 31, half = lane >> 5;
  const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(p.wtiles)) + (size_t)min(rb, p.row_blocks - 1) * p.padded_ksteps * (1024 * PIECES), 0,
                                                                        (int)(FloatMfmaWeightTile(p.chunks, 0, PIECES, 0) + FloatMfmaWeightTail(PIECES)), 0x00020000);
  const int weight_lane = (n >> 4) * (PIECES * 1024) + 256 * half + 16 * (n & 15);
  h8 a[ADEPTH][STEPS][PIECES];
  auto load_weights = [&](h8 (&dst)[PIECES], int chunk, int ks) {
#pragma unroll
    for (int q = 0; q < PIECES; ++q) {
      const int step = kh * STEPS + ks;  // of 16 channels: half of two tiles
      dst[q] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(wbuf, weight_lane, (int)FloatMfmaWeightTile(chunk, step & ~1, PIECES, q) + 512 * (step & 1), 0));
    }
  };
  const uint4* const operand = xt + (2 * STEPS * kh + half) * (4 * QT) + n;
  // fp32: the products of two high pieces, and those of a high and a low one, which would otherwise each round the sum
  // of the former (the matrix cores cut sums off rather than round them)
  v16f acc[4];
  [[maybe_unused]] v16f rest[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[c][i] = 0.0f, rest[c][i] = 0.0f;

  // The scales of fp32.  colmax holds the bits of the largest magnitude of every position; its exponent gives the scale
  // that takes it to [2^12, 2^13).  A chunk with a value beyond 2^15 after scaling raises its flag; then everyone
  // takes the new maxima, brings the sums so far to the new scales and writes that chunk's cells again.  Even and odd
  // chunks have a flag each: a wavefront may be behind the barrier of one chunk and at its look at that chunk's flag
  // while another is through the next chunk's values.
  uint32_t* const colmax = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(xt) + LdsTables(WR, F32));
  uint32_t* const flags = colmax + 4 * QT;
  uint32_t* const marks = flags + 4;
  uint32_t* const first_exp = marks + QT;  // of the positions' first scales
  const uint32_t* const own_max = colmax + 4 * n;  // of the positions whose sums the lane holds
  [[maybe_unused]] uint32_t own_exps = 0;  // a byte each: four registers do not fit beside the sums
  auto own_exp = [&](int c) { return (int)(own_exps >> (8 * c) & 0xffu); };
  auto scale_exp = [](uint32_t bits) { return max(1, min(243, 266 - (int)(bits >> 23))); };
  auto collect = [&](Quad<F32> (&rd)[UC]) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float m = 0.0f;
#pragma unroll
      for (int i = 0; i < UC; ++i) m = fmaxf(m, fabsf(__uint_as_float(rd[i][c])));
      atomicMax(&colmax[4 * j + c], __float_as_uint(m));
    }
  };
  auto rescale = [&](Quad<F32> (&rd)[UC], int buf) {
    collect(rd);
    __syncthreads();
    if (tid == 0) flags[buf] = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const uint32_t m = colmax[4 * j + c], om = own_max[c];
      if (__uint_as_float(m) * scale[c] >= kPeak) scale[c] = __uint_as_float((uint32_t)(scale_exp(m) + 11) << 23);
      const int before = own_exp(c);
      if (__uint_as_float(om) * __uint_as_float((uint32_t)before << 23) >= 0x1p15f) {
        const int e = scale_exp(om);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[c][i] = __builtin_amdgcn_ldexpf(acc[c][i], e - before), rest[c][i] = __builtin_amdgcn_ldexpf(rest[c][i], e - before);
        own_exps = (own_exps & ~(0xffu << (8 * c))) | (uint32_t)e << (8 * c);
        // unmarked, every term of a sum was 2^-48 or more when it was added: 2^64 less is far from the subnormal numbers
        if ((int)first_exp[4 * n + c] - e > 64) marks[n] = 1;
      }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) commit(rd, buf, c);
    __syncthreads();
  };

  // One chunk: kSteps x 4 cells.  Behind the multiplies of a step the next chunk's cells of one position go to the
  // other buffer; then the loads of the chunk DEPTH behind that one are issued into the registers this frees.
  constexpr int PF = F32 ? 2 : 3;  // operand cells in flight
  auto run_chunk = [&](auto slot_c, auto last_c, int chunk) {
    constexpr bool LAST = decltype(last_c)::value;  // no chunk is left to load
    constexpr int S = decltype(slot_c)::value, NEXT = (S + 1) % DEPTH, AS = S % ADEPTH;
    const uint4* const cells_in = operand + (S & 1) * kBuf;
    uint4 b[PF + 1][PIECES];
    auto read = [&](int v) {
#pragma unroll
      for (int q = 0; q < PIECES; ++q) b[v % (PF + 1)][q] = cells_in[q * kCells + (v >> 2) * 2 * (4 * QT) + (v & 3) * QT];
    };
#pragma unroll
    for (int d = 0; d < PF; ++d) read(d);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < STEPS; ++ks) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int v = 4 * ks + c;
        if (v + PF < 4 * STEPS) read(v + PF);
        const h8 xh = __builtin_bit_cast(h8, b[v % (PF + 1)][0]);
        acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[AS][ks][0], xh, acc[c], 0, 0, 0);
        if constexpr (F32) {
          const h8 xl = __builtin_bit_cast(h8, b[v % (PF + 1)][PIECES - 1]);
          rest[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[AS][ks][PIECES - 1], xh, rest[c], 0, 0, 0);
          rest[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[AS][ks][0], xl, rest[c], 0, 0, 0);
        }
      }
      if (!LAST) load_weights(a[AS][ks], chunk + ADEPTH, ks);
#pragma unroll
      for (int c = 0; c < KH; ++c) commit(r[NEXT], (S + 1) & 1, KH * ks + c);
      // the vector ALU's share of a step goes between its matrix instructions: a wavefront issues in order
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (4 * ks + c + PF < 4 * STEPS) __builtin_amdgcn_sched_group_barrier(0x100, PIECES, 0);
#pragma unroll
        for (int q = 0; q < (F32 ? 3 : 1); ++q) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x002, F32 ? 2 * KH : KH, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (F32) {
      if (peak >= kPeak || low < kSmallBits) {  // one branch for both
        if (peak >= kPeak) flags[(S + 1) & 1] = 1;
        if (low < kSmallBits) marks[j] = 1;
      }
      peak = 0.0f;
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(flags[(S + 1) & 1]) != 0) rescale(r[NEXT], (S + 1) & 1);
      if (!LAST) issue(r[NEXT], chunk + 1 + DEPTH);
    } else {
      if (!LAST) issue(r[NEXT], chunk + 1 + DEPTH);
      __syncthreads();
    }
  };
  static_assert(kSteps == 4 && STEPS >= 1, "KH positions of the quads are written per step");
  static_assert(DEPTH == 2 && DEPTH % ADEPTH == 0, "the buffer and the weights' registers follow from the slot");
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    issue(r[d], d);
    __builtin_amdgcn_sched_barrier(0);
    if (d < ADEPTH) {
#pragma unroll
      for (int ks = 0; ks < STEPS; ++ks) load_weights(a[d % ADEPTH][ks], d, ks);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (F32) {
    for (int i = tid; i < kF32Tables / 4; i += kThreads) colmax[i] = 0;  // and the flags and marks
    __syncthreads();
    collect(r[0]);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      scale[c] = __uint_as_float((uint32_t)(scale_exp(colmax[4 * j + c]) + 11) << 23);
      own_exps |= (uint32_t)scale_exp(own_max[c]) << (8 * c);
    }
    if (tid < 4 * QT) first_exp[tid] = (uint32_t)scale_exp(colmax[tid]);
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) commit(r[0], 0, c);
  if constexpr (F32) {
    if (low < kSmallBits) marks[j] = 1;
    peak = 0.0f;
  }
  issue(r[0], DEPTH);
  __syncthreads();
  using More = std::false_type;
  using Last = std::true_type;
  int chunk = 0;
  for (; chunk + DEPTH <= p.chunks; chunk += DEPTH) {
    run_chunk(std::integral_constant<int, 0>(), More(), chunk);
    run_chunk(std::integral_constant<int, 1>(), More(), chunk + 1);
  }
  if (chunk < p.chunks) run_chunk(std::integral_constant<int, 0>(), Last(), chunk);

  // Lane (n, half) holds rows 8 (i / 4) + 4 half + i % 4 (i = 0 .. 15) of the row block at the four positions of quad n.
  // Wavefronts that share a row block finish FIN of the sixteen each, from what the others hand over through LDS.
  float fin[4][FIN];
  auto total = [&](int c, int i) { return F32 ? __builtin_fmaf(rest[c][i], 1.0f / kFloatMfmaLow, acc[c][i]) : acc[c][i]; };
  if constexpr (KH == 1) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) fin[c][i] = total(c, i);
  } else {
    // [row block][finishing part][part it comes from, without its own][value][lane]
    float* const trade = reinterpret_cast<float*>(xt) + (wave % WR) * (KH * (KH - 1) * 4 * FIN * 64) + lane;
    auto slot_of = [](int to, int from) { return (to * (KH - 1) + (from < to ? from : from - 1)) * (4 * FIN * 64); };
#pragma unroll
    for (int to = 0; to < KH; ++to) {
      if (to == kh) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int i = 0; i < FIN; ++i) fin[c][i] = total(c, to * FIN + i);
      } else {
        float* const dst = trade + slot_of(to, kh);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int i = 0; i < FIN; ++i) dst[(c * FIN + i) * 64] = total(c, to * FIN + i);
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KH - 1; ++k) {
      const float* const src = trade + (kh * (KH - 1) + k) * (4 * FIN * 64);
#pragma unroll
      for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int i = 0; i < FIN; ++i) fin[c][i] += src[(c * FIN + i) * 64];
    }
  }
  // An infinity or a NaN among the inputs of a position reaches every row of the product through the zero weights.  Such
  // quads are walked below, in fp32 those and the marked ones output by output.
  float poison = 0.0f;
#pragma unroll
  for (int c = 0; c < 4; ++c) poison = __builtin_fmaf(fin[c][0], 0.0f, poison);
  const int row_in_block = 4 * half + (32 / KH) * kh, row0 = rb * 32 + row_in_block;
  const uint32_t oq = tile_quad0 + (uint32_t)n;
  const uint32_t on = oq / (uint32_t)p.qpi;
  const int opp = 4 * (int)(oq - on * (uint32_t)p.qpi), ofirst = min(opp, p.hw - 4);
  const bool present = oq < p.total_quads;
  const int own = RAGGED ? opp - ofirst : 0;  // the first position of the quad that is not one of the quad before
  bool suspect = poison != poison;
  const int table = min(rb, p.row_blocks - 1) * 32 + row_in_block;
  if constexpr (F32) {
    if (marks[n] != 0) {  // most marked quads hold no output that is too small
#pragma unroll
      for (int b = 0; b < FIN / 4; ++b) {
        const v4f reach = *reinterpret_cast<const v4f*>(p.row_exp + 32 * p.row_blocks + table + 8 * b);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int c = 0; c < 4; ++c) suspect = suspect || fabsf(fin[c][4 * b + i]) < reach[i];
      }
    }
  }
  suspect = suspect && present;
  float bias[FIN];
  [[maybe_unused]] int row_exp[FIN];
#pragma unroll
  for (int b = 0; b < FIN / 4; ++b) {
    if constexpr (F32) {
      const v4f v = p.bias ? *reinterpret_cast<const v4f*>(static_cast<const float*>(p.bias) + table + 8 * b) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
      const int4 e = *reinterpret_cast<const int4*>(p.row_exp + table + 8 * b);
      bias[4 * b] = v.x, bias[4 * b + 1] = v.y, bias[4 * b + 2] = v.z, bias[4 * b + 3] = v.w;
      row_exp[4 * b] = e.x, row_exp[4 * b + 1] = e.y, row_exp[4 * b + 2] = e.z, row_exp[4 * b + 3] = e.w;
    } else {
      const u2 v = p.bias ? *reinterpret_cast<const u2*>(static_cast<const h1*>(p.bias) + table + 8 * b) : u2{0u, 0u};
      const uint32_t d0 = v.x, d1 = v.y;
      const h2 lo = __builtin_bit_cast(h2, d0), hi = __builtin_bit_cast(h2, d1);
      bias[4 * b] = (float)lo.x, bias[4 * b + 1] = (float)lo.y, bias[4 * b + 2] = (float)hi.x, bias[4 * b + 3] = (float)hi.y;
    }
  }
  // Stores past the end of the buffer are dropped, so lanes and rows without an output need no branch.
  constexpr uint32_t kOutside = kFloatMfmaOutside;
  const __amdgpu_buffer_rsrc_t obuf = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)((uint32_t)p.batch * (uint32_t)p.M * (uint32_t)p.hw * kElem), 0x00020000);
  const uint32_t pitch = (uint32_t)p.hw * kElem;
  const uint32_t obase = ((on * (uint32_t)p.M + (uint32_t)row0) * (uint32_t)p.hw + (uint32_t)ofirst) * kElem;
  auto finish = [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
    const uint32_t h0 = p.act_h_words[0], h1w = p.act_h_words[1];
    const DevActH act_h = {ACT, (uint16_t)h0, (uint16_t)(h0 >> 16), (uint16_t)h1w, (uint16_t)(h1w >> 16)};
#pragma unroll
    for (int i = 0; i < FIN; ++i) {
      const int rr = 8 * (i >> 2) + (i & 3);
      const uint32_t at = row0 + rr < p.M && present ? obase + (uint32_t)rr * pitch : kOutside;
      const int whole = (int)(own == 0 ? at : kOutside);
      if constexpr (F32) {
        u4 o;
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] = __float_as_uint(ActivateT<ACT>(__builtin_amdgcn_ldexpf(fin[c][i], row_exp[i] + 127 - own_exp(c)) + bias[i], p.act));
        __builtin_amdgcn_raw_buffer_store_b128(o, obuf, whole, 0, 0);
        if constexpr (RAGGED) {
#pragma unroll
          for (int c = 1; c < 4; ++c) __builtin_amdgcn_raw_buffer_store_b32(o[c], obuf, (int)(own != 0 && c >= own ? at + 4 * c : kOutside), 0, 0);
        }
      } else {
        const h2 o0 = ActivateH<ACT>(__builtin_convertvector((v2f{fin[0][i] + bias[i], fin[1][i] + bias[i]}), h2), act_h);
        const h2 o1 = ActivateH<ACT>(__builtin_convertvector((v2f{fin[2][i] + bias[i], fin[3][i] + bias[i]}), h2), act_h);
        const u2 o = {__builtin_bit_cast(uint32_t, o0), __builtin_bit_cast(uint32_t, o1)};
        __builtin_amdgcn_raw_buffer_store_b64(o, obuf, whole, 0, 0);
        if constexpr (RAGGED) {
#pragma unroll
          for (int c = 1; c < 4; ++c) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(o[c >> 1] >> (16 * (c & 1))), obuf, (int)(own != 0 && c >= own ? at + 2 * c : kOutside), 0, 0);
        }
      }
    }
  };
  if (row0 < p.M) DispatchAct(p.act.type, finish);
  if (__ballot(suspect) == 0) return;
  uint64_t walk = 0;  // bit 4 i + c: the output of row i at position c is walked
  if (suspect) {
#pragma unroll
    for (int i = 0; i < FIN; ++i) {
      const int rr = 8 * (i >> 2) + (i & 3);
      if (row0 + rr >= p.M) break;
      const float reach = F32 ? reinterpret_cast<const float*>(p.row_exp + 32 * p.row_blocks)[table + rr] : 0.0f;
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (c >= own && (!F32 || !(fabsf(fin[c][i]) >= reach))) walk |= 1ull << (4 * i + c);
    }
  }
  // other lanes write these outputs again: what this wavefront has stored must have arrived
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  WalkOutputs<F32>(p, walk, FIN, rb * 32 + (32 / KH) * kh, tile_quad0);
}

template <int WR, bool F32, bool RAGGED>
__global__ void __launch_bounds__(kThreads, F32 ? 2 : 4) FloatMfmaKernel(PL_HEAD_PARAMS, const FloatMfmaParams block) {
  const FloatMfmaParams p = WithHead(block, PL_HEAD_ARGS);
  extern __shared__ uint4 xt[];
  FloatMfmaBody<WR, F32, RAGGED>(p, xt);
}

// fp32 with wavefronts of their own for the inputs: 256 rows x 64 positions, 128 channels a chunk, twelve wavefronts.  Eight multiply 32 rows
// with all positions (16 x 16 x 32 matrix instructions: half of the sums' registers of FloatMfmaBody's wavefronts, which three wavefronts
// per SIMD leave).  Four turn inputs into operand cells: a thread loads eight channels of a position quad, two chunks ahead of the one that
// it writes, so the conversions, eleven instructions per pair of values, run beside the multiplies instead of between them.  us per call among
// others, FloatMfmaBody / this: 64 x 1024 -> 1024 @7x7, row pairs, 70 % zeros 26.7 / 23.0; 32 x 512 -> 512 @14x14 16.1 / 14.8; 4 x 1248 -> 1024
// @29x29 30.7 / 25.4.  With 128 rows x 128 positions, 64 channels a chunk, the first takes 25.3 (every input converted twice as
// often).  What bounds it: nothing alone; 2.2 us a chunk, of which its matrix instructions take 1.4 at the rate they reach on such data
// (32 x 32 x 16 ones 1.7: 18 ns against twice 7.7 for half the products) and its 80 KB 0.6.
constexpr int kSplitThreads = 768;
constexpr int kSplitQuads = 16;                                // position quads of a tile
constexpr int kSplitChunk = 128;                               // channels of a chunk
constexpr int kSplitCells = kSplitChunk / 8 * 4 * kSplitQuads;  // cells of a chunk and piece
constexpr int kSplitRowBlocks = 8;

template <bool RAGGED>
__device__ __forceinline__ void FloatSplitBody(const FloatMfmaParams& p, uint4* xt) {
  constexpr int QT = kSplitQuads, CHUNK = kSplitChunk, STEPS = CHUNK / 32, PIECES = 2, kCells = kSplitCells, kBuf = PIECES * kCells;
  constexpr uint32_t kElem = 4u;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // each XCD owns a contiguous range of tiles, the row groups of one tile follow each other there
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int first_tile = (xcd * p.tiles) >> 3, last_tile = ((xcd + 1) * p.tiles) >> 3;
  const int tile = first_tile + slot / p.row_groups, rg = slot % p.row_groups;
  if (tile >= last_tile) return;
  const uint32_t tile_quad0 = (uint32_t)tile * (uint32_t)QT;
  const int chunks = (p.K + CHUNK - 1) / CHUNK;

  // the scales of fp32, as in FloatMfmaBody
  uint32_t* const colmax = reinterpret_cast<uint32_t*>(xt + 2 * kBuf);
  uint32_t* const flags = colmax + 4 * QT;
  uint32_t* const marks = flags + 4;
  uint32_t* const first_exp = marks + QT;
  auto scale_exp = [](uint32_t bits) { return max(1, min(243, 266 - (int)(bits >> 23))); };
  for (int i = tid; i < kF32Tables / 4; i += kSplitThreads) colmax[i] = 0;
  __syncthreads();

  if (wave >= 8) {
    const int j = tid & (QT - 1), kg = (tid >> 4) & 15;
    const uint32_t quad = min(tile_quad0 + (uint32_t)j, p.total_quads - 1u);
    const uint32_t img = quad / (uint32_t)p.qpi;
    const int first = min(4 * (int)(quad - img * (uint32_t)p.qpi), p.hw - 4);
    const uint32_t vbase = img * (uint32_t)p.K * (uint32_t)p.hw + (uint32_t)first;
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p.x), 0, (int)((uint32_t)p.batch * (uint32_t)p.K * (uint32_t)p.hw * kElem), 0x00020000);
    const int pitch_in = p.hw * (int)kElem;
    u4 r[2][8];
    // The last group of a channel count that is no multiple of 8 holds the last eight channels.  Groups behind it lie outside the buffer:
    // they read as zeros, and no condition around the loads makes the wait for older ones wait for these too.
    auto issue = [&](u4 (&rd)[8], int chunk) {
      const int k = chunk * CHUNK + 8 * kg;
      const uint32_t voff = k < p.K ? (vbase + (uint32_t)min(k, p.K - 8) * (uint32_t)p.hw) * kElem : kFloatMfmaOutside;
#pragma unroll
      for (int i = 0; i < 8; ++i) rd[i] = __builtin_amdgcn_raw_buffer_load_b128(xbuf, (int)voff, i * pitch_in, 0);
    };
    uint4* const cells = xt + kg * (4 * QT) + j;
    float scale[4], peak = 0.0f;
    uint32_t low = 0xffffffffu;  // the smallest magnitude but zero, as kSmallBits
    auto commit = [&](u4 (&rd)[8], int buf) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // the first pieces are one mixed-precision multiply-add each
          const float a = __uint_as_float(rd[2 * i][c]) * scale[c], b = __uint_as_float(rd[2 * i + 1][c]) * scale[c];
          peak = fmaxf(fmaxf(peak, fabsf(a)), fabsf(b));
          low = min(min(low, (__float_as_uint(a) << 1) - 1u), (__float_as_uint(b) << 1) - 1u);
          const h2 both = {(h1)__builtin_fmaf(a, 1.0f / kFloatMfmaLow, 0.0f), (h1)__builtin_fmaf(b, 1.0f / kFloatMfmaLow, 0.0f)};
          uint32_t word = __builtin_bit_cast(uint32_t, both);
          asm("" : "+v"(word));  // the second value is taken from the word, not converted again
          const h2 h = __builtin_bit_cast(h2, word);
          const h2 l = __builtin_convertvector((v2f{__builtin_fmaf((float)h.x, -kFloatMfmaLow, a), __builtin_fmaf((float)h.y, -kFloatMfmaLow, b)}), h2);
          hi[i] = word, lo[i] = __builtin_bit_cast(uint32_t, l);
        }
        uint4* const dst = cells + buf * kBuf + c * QT;
        *dst = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        dst[kCells] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      }
    };
    auto collect = [&](u4 (&rd)[8]) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float m = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(__uint_as_float(rd[i][c])));
        atomicMax(&colmax[4 * j + c], __float_as_uint(m));
      }
    };
    // the cells of chunk `to` (its loads are rd), the barrier behind them, the loads of the chunk two behind it
    auto bring = [&](u4 (&rd)[8], int buf, int to) {
      commit(rd, buf);
      if (peak >= kPeak || low < kSmallBits) {  // one branch for both
        if (peak >= kPeak) flags[buf] = 1;
        if (low < kSmallBits) marks[j] = 1;
      }
      peak = 0.0f;
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(flags[buf]) != 0) {
        collect(rd);
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t m = colmax[4 * j + c];
          if (__uint_as_float(m) * scale[c] >= kPeak) scale[c] = __uint_as_float((uint32_t)(scale_exp(m) + 11) << 23);
        }
        commit(rd, buf);
        if (low < kSmallBits) marks[j] = 1;
        peak = 0.0f;
        __syncthreads();
      }
      issue(rd, to + 2);
    };
    issue(r[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    issue(r[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    collect(r[0]);
    __syncthreads();
#pragma unroll
    for (int c = 0; c < 4; ++c) scale[c] = __uint_as_float((uint32_t)(scale_exp(colmax[4 * j + c]) + 11) << 23);
    commit(r[0], 0);
    if (low < kSmallBits) marks[j] = 1;
    peak = 0.0f;
    issue(r[0], 2);
    __syncthreads();
    int chunk = 0;
    for (; chunk + 2 < chunks; chunk += 2) {
      bring(r[1], 1, chunk + 1);
      bring(r[0], 0, chunk + 2);
    }
    if (chunk + 1 < chunks) bring(r[1], 1, chunk + 1);
    __syncthreads();  // the last chunk is multiplied
    return;
  }

  // the wavefront's row block (past the last one: the last one again, not stored)
  const int rb = rg * kSplitRowBlocks + wave;
  const int n = lane & 15, kq = lane >> 4;
  const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(static_cast<const char*>(p.wtiles)) + (size_t)min(rb, p.row_blocks - 1) * p.padded_ksteps * (1024 * PIECES), 0,
                                                                        (int)(FloatMfmaWeightTile(p.chunks, 0, PIECES, 0) + FloatMfmaWeightTail(PIECES)), 0x00020000);
  constexpr int AHEAD = 2;  // steps of weights in registers
  h8 a[AHEAD][2][PIECES];
  auto load_weights = [&](int chunk, int ks) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < PIECES; ++q) a[ks % AHEAD][t][q] = __builtin_bit_cast(h8, __builtin_amdgcn_raw_buffer_load_b128(wbuf, lane * 16, (int)FloatMfmaWeightTile(0, 2 * (chunk * STEPS + ks) + t, PIECES, q), 0));
  };
  const uint4* const operand = xt + kq * (4 * QT) + n;
  // fp32: the products of two high pieces, and those of a high and a low one, which would otherwise each round the sum
  // of the former (the matrix cores cut sums off rather than round them)
  v4f acc[2][4], rest[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[t][c] = rest[t][c] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  uint32_t own_exps = 0;  // a byte each
  auto own_exp = [&](int c) { return (int)(own_exps >> (8 * c) & 0xffu); };
  const uint32_t* const own_max = colmax + 4 * n;

  // The matrix cores cut sums off, so a long sum is off by more: behind half of the chunks the sums are added, rounded, to those that wait
  // in LDS and begin anew (1024 channels 1.6e-7 in 2-norm, as FloatMfmaBody's two sums of 512 each; one sum 2.1e-7; four of 256
  // 1.3e-7 and 0.8 us more on 64 x 1024 -> 1024 @7x7).
  v4f* const waiting = reinterpret_cast<v4f*>(reinterpret_cast<char*>(colmax) + kF32Tables) + wave * (8 * 64) + lane;
#pragma unroll
  for (int i = 0; i < 8; ++i) waiting[64 * i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  auto add_waiting = [&](auto keep_c) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const v4f sum = acc[t][c] + waiting[64 * (4 * t + c)];
        if constexpr (decltype(keep_c)::value) {
          waiting[64 * (4 * t + c)] = sum;
          acc[t][c] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        } else {
          acc[t][c] = sum;
        }
      }
  };

  // One chunk: STEPS x 4 cells, two tiles each, cells read PF ahead.  The weights of a step are requested as soon as the one two before it
  // has used their registers.
  constexpr int PF = 4;
  auto run_chunk = [&](auto last_c, int chunk) {
    constexpr bool LAST = decltype(last_c)::value;
    const uint4* const in = operand + (chunk & 1) * kBuf;
    uint4 b[PF + 1][PIECES];
    auto read = [&](int v) {
#pragma unroll
      for (int q = 0; q < PIECES; ++q) b[v % (PF + 1)][q] = in[q * kCells + (v >> 2) * 4 * (4 * QT) + (v & 3) * QT];
    };
#pragma unroll
    for (int d = 0; d < PF; ++d) read(d);
#pragma unroll
    for (int ks = 0; ks < STEPS; ++ks) {
      if (LAST && ks > 0 && 32 * (STEPS * chunk + ks) >= p.K) break;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int v = 4 * ks + c;
        if (v + PF < 4 * STEPS) read(v + PF);
        __builtin_amdgcn_sched_barrier(0);  // the reads stay ahead of the multiply
        const h8 xh = __builtin_bit_cast(h8, b[v % (PF + 1)][0]), xl = __builtin_bit_cast(h8, b[v % (PF + 1)][1]);
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[ks % AHEAD][t][0], xh, acc[t][c], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t) rest[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[ks % AHEAD][t][1], xh, rest[t][c], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < 2; ++t) rest[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[ks % AHEAD][t][0], xl, rest[t][c], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (!LAST || ks + AHEAD < STEPS) load_weights(chunk, ks + AHEAD);
    }
    __syncthreads();
    if constexpr (!LAST) {
      const int next = (chunk + 1) & 1;
      if (__builtin_amdgcn_readfirstlane(flags[next]) != 0) {
        __syncthreads();
        if (tid == 0) flags[next] = 0;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t om = own_max[c];
          const int before = own_exp(c);
          if (__uint_as_float(om) * __uint_as_float((uint32_t)before << 23) >= 0x1p15f) {
            const int e = scale_exp(om);
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
              for (int i = 0; i < 4; ++i)
                acc[t][c][i] = __builtin_amdgcn_ldexpf(acc[t][c][i], e - before), rest[t][c][i] = __builtin_amdgcn_ldexpf(rest[t][c][i], e - before);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
              v4f sum = waiting[64 * (4 * t + c)];
#pragma unroll
              for (int i = 0; i < 4; ++i) sum[i] = __builtin_amdgcn_ldexpf(sum[i], e - before);
              waiting[64 * (4 * t + c)] = sum;
            }
            own_exps = (own_exps & ~(0xffu << (8 * c))) | (uint32_t)e << (8 * c);
            // unmarked, every term of a sum was 2^-48 or more when it was added: 2^64 less is far from the subnormal numbers
            if ((int)first_exp[4 * n + c] - e > 64) marks[n] = 1;
          }
        }
        __syncthreads();
      }
    }
  };
#pragma unroll
  for (int ks = 0; ks < AHEAD; ++ks) load_weights(0, ks);
  __syncthreads();  // the first chunk's maxima
#pragma unroll
  for (int c = 0; c < 4; ++c) own_exps |= (uint32_t)scale_exp(own_max[c]) << (8 * c);
  if (tid < 4 * QT) first_exp[tid] = (uint32_t)scale_exp(colmax[tid]);
  __syncthreads();
  int chunk = 0;
  const int half = chunks >> 1;
  for (int begun = 0; chunk + 1 < chunks; begun = chunk) {
    const int until = min(chunk + half, chunks - 1);
    for (; chunk < until; ++chunk) run_chunk(std::false_type(), chunk);
    if (chunk - begun == half) add_waiting(std::true_type());
  }
  run_chunk(std::true_type(), chunk);
  add_waiting(std::false_type());

  // Lane (n, kq) holds rows 4 kq .. 4 kq + 3 of its tiles at the four positions of quad n.
  constexpr int ROWS = 8;  // row i of a lane is row 16 (i / 4) + i % 4 behind its first
  auto total = [&](int c, int i) { return __builtin_fmaf(rest[i >> 2][c][i & 3], 1.0f / kFloatMfmaLow, acc[i >> 2][c][i & 3]); };
  auto row_of = [](int i) { return 16 * (i >> 2) + (i & 3); };
  const int row0 = rb * 32 + 4 * kq, table = min(rb, p.row_blocks - 1) * 32 + 4 * kq;
  const uint32_t oq = tile_quad0 + (uint32_t)n, on = oq / (uint32_t)p.qpi;
  const int opp = 4 * (int)(oq - on * (uint32_t)p.qpi), ofirst = min(opp, p.hw - 4);
  const bool present = oq < p.total_quads;
  const int own = RAGGED ? opp - ofirst : 0;  // the first position of the quad that is not one of the quad before
  // An infinity or a NaN among the inputs of a position reaches every row of the product through the zero weights.  Such
  // quads are walked below, those and the marked ones output by output.
  float poison = 0.0f;
#pragma unroll
  for (int c = 0; c < 4; ++c) poison = __builtin_fmaf(total(c, 0), 0.0f, poison);
  bool suspect = poison != poison;
  if (marks[n] != 0) {  // most marked quads hold no output that is too small
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const v4f reach = *reinterpret_cast<const v4f*>(p.row_exp + 32 * p.row_blocks + table + 16 * b);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) suspect = suspect || fabsf(total(c, 4 * b + i)) < reach[i];
    }
  }
  suspect = suspect && present;
  float bias[ROWS];
  int row_exp[ROWS];
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const v4f v = p.bias ? *reinterpret_cast<const v4f*>(static_cast<const float*>(p.bias) + table + 16 * b) : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    const int4 e = *reinterpret_cast<const int4*>(p.row_exp + table + 16 * b);
    bias[4 * b] = v.x, bias[4 * b + 1] = v.y, bias[4 * b + 2] = v.z, bias[4 * b + 3] = v.w;
    row_exp[4 * b] = e.x, row_exp[4 * b + 1] = e.y, row_exp[4 * b + 2] = e.z, row_exp[4 * b + 3] = e.w;
  }
  // Stores past the end of the buffer are dropped, so lanes and rows without an output need no branch.
  constexpr uint32_t kOutside = kFloatMfmaOutside;
  const __amdgpu_buffer_rsrc_t obuf = __builtin_amdgcn_make_buffer_rsrc(p.out, 0, (int)((uint32_t)p.batch * (uint32_t)p.M * (uint32_t)p.hw * kElem), 0x00020000);
  const uint32_t pitch = (uint32_t)p.hw * kElem;
  const uint32_t obase = ((on * (uint32_t)p.M + (uint32_t)row0) * (uint32_t)p.hw + (uint32_t)ofirst) * kElem;
  auto finish = [&](auto act_c) {
    constexpr int ACT = decltype(act_c)::value;
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const uint32_t at = row0 + row_of(i) < p.M && present ? obase + (uint32_t)row_of(i) * pitch : kOutside;
      u4 o;
#pragma unroll
      for (int c = 0; c < 4; ++c) o[c] = __float_as_uint(ActivateT<ACT>(__builtin_amdgcn_ldexpf(total(c, i), row_exp[i] + 127 - own_exp(c)) + bias[i], p.act));
      __builtin_amdgcn_raw_buffer_store_b128(o, obuf, (int)(own == 0 ? at : kOutside), 0, 0);
      if constexpr (RAGGED) {
#pragma unroll
        for (int c = 1; c < 4; ++c) __builtin_amdgcn_raw_buffer_store_b32(o[c], obuf, (int)(own != 0 && c >= own ? at + 4 * c : kOutside), 0, 0);
      }
    }
  };
  if (row0 < p.M) DispatchAct(p.act.type, finish);
  if (__ballot(suspect) == 0) return;
  uint32_t walk = 0;  // bit 4 i + c: the output of row i at position c is walked
  if (suspect) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const v4f reach = *reinterpret_cast<const v4f*>(p.row_exp + 32 * p.row_blocks + table + 16 * b);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          if (row0 + 16 * b + i < p.M && c >= own && !(fabsf(total(c, 4 * b + i)) >= reach[i])) walk |= 1u << (16 * b + 4 * i + c);
    }
  }
  // other lanes write these outputs again: what this wavefront has stored must have arrived
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // the cells are multiplied and the sums that waited are taken: a part of either for every wavefront
  static_assert(2 * kBuf * 16 == 8 * kStagedFirst && kStagedBytes - kStagedFirst <= 8 * 64 * 16, "LDS of a wavefront");
  char* const sums = reinterpret_cast<char*>(colmax) + kF32Tables + 8 * 8 * 64 * 16;
  WalkOutputs16(p, walk, rb * 32, tile_quad0, reinterpret_cast<const char*>(xt) + wave * kStagedFirst, waiting - lane, sums + wave * kStagedSums);
}

template <bool RAGGED>
__global__ void __launch_bounds__(kSplitThreads, 3) FloatSplitKernel(PL_HEAD_PARAMS, const FloatMfmaParams block) {
  const FloatMfmaParams p = WithHead(block, PL_HEAD_ARGS);
  extern __shared__ uint4 xt[];
  FloatSplitBody<RAGGED>(p, xt);
}

template <int WR, bool F32>
hipError_t Launch(const FloatMfmaParams& p, dim3 grid, hipStream_t s) {
  const dim3 block(kThreads);
  constexpr size_t lds = LdsTables(WR, F32) + (F32 ? kF32Tables : 0);
  return p.quad_aligned ? LaunchWithHead(FloatMfmaKernel<WR, F32, false>, grid, block, lds, s, p) : LaunchWithHead(FloatMfmaKernel<WR, F32, true>, grid, block, lds, s, p);
}

hipError_t LaunchSplit(const FloatMfmaParams& p, dim3 grid, hipStream_t s) {
  const dim3 block(kSplitThreads);
  constexpr size_t lds = 2 * 2 * kSplitCells * 16 + kF32Tables + 8 * 8 * 64 * 16 + 8 * kStagedSums;
  return p.quad_aligned ? LaunchWithHead(FloatSplitKernel<false>, grid, block, lds, s, p) : LaunchWithHead(FloatSplitKernel<true>, grid, block, lds, s, p);
}

}  // namespace

int FloatMfmaPaddedSteps(int K) { return (K + kChunk - 1) / kChunk * kSteps; }
bool FloatMfmaFits(bool f32, int K, int M, int hw, int64_t positions) {
  // offsets are kept in 32 bits, and the half above 2^31 stands for what is left out
  const int64_t values = (1ll << 31) / (f32 ? 4 : 2);
  return K >= 8 && hw >= 4 && positions * K < values && positions * M < values && ((int64_t)K + kChunk) * (M + 31) * 2 < values;
}

// The rows a workgroup takes: the least of the times fitted to 5600 random calls in fp32 and 4600 in fp16 (32 - 2048
// channels and rows, 50 - 100 000 positions, 256 CUs); the form picked takes 0.1 % (fp32) and 1.2 % (fp16) longer than the
// fastest on average.  Many rows per workgroup fetch the inputs the fewest times, few rows let small calls fill the chip
// and halve the chain of a chunk: 64 x 1024 -> 1024 @7x7
// fp32 256 rows 37.3, 128 rows 29.4, 64 rows 40.9; 64 x 512 -> 512 @14x14 25.9, 34.1, 47.7; one image 96 -> 192 @56x56 8.0, 6.9, 6.4.
static FloatMfmaPlan PlanRows(bool f32, int cus, int row_blocks, int K, int M, int hw, int batch) {
  const int64_t tiles = ((int64_t)batch * ((hw + 3) / 4) + kQuads - 1) / kQuads;
  const int chunks = (K + kChunk - 1) / kChunk;
  // us: a launch, a chunk of it; a full chip and a chunk of it; every workgroup beyond one per CU and a chunk of it (fp16,
  // where two share a CU); every further round of workgroups and a chunk of it; outputs
  struct Cost {
    double launch, chunk, full, full_chunk, over, over_chunk, round, round_chunk, out;
  };
  // the last one for layers of at most 64 rows, of which there were hardly any among those calls (1802 of 8 - 64 rows; another
  // 884 take 0.91 .. 1.08 of what it says, and by the one before 1.13 times as long in the middle)
  static constexpr Cost kF32[4] = {
      {4.5, 1.56, 2.9, 0.89, 0, 0, 4.8, 2.1, 0}, {4.6, 0.98, 2.0, 0.56, 0, 0, 5.0, 1.22, 0}, {4.5, 0.74, 1.2, 0.4, 0, 0, 4.4, 0.82, 0}, {3.9, 0.91, 1.65, 0.58, 0, 0, 5.0, 1.02, 0}};
  // maps of whole and of ragged quads
  static constexpr Cost kF16[2][3] = {
      {{3.1, 0.57, 0, 0.34, 0.57, 0.27, 0.023, 0.79, 0.4}, {3.7, 0.38, 0, 0.33, 0.43, 0.41, 0.74, 0.36, 0.31}, {3.6, 0.31, 0.8, 0.21, 0.84, 0.23, 2.1, 0.32, 0}},
      {{3.8, 0.66, 0, 0.28, 0.13, 0.34, 0, 0.91, 0.59}, {4.1, 0.47, 0, 0.3, 0.4, 0.33, 0.68, 0.5, 0.43}, {3.8, 0.39, 0.42, 0.26, 0.52, 0.25, 2.5, 0.32, 0.13}}};
  const double positions = (double)batch * hw;
  FloatMfmaPlan best{};
  for (int i = 0; i < 3; ++i) {
    const int wr = 8 >> i;
    if (row_blocks != 0 ? wr != row_blocks : wr > 2 && f32 && M <= 64) continue;
    FloatMfmaPlan p{};
    p.wr = wr;
    p.row_groups = ((M + 31) / 32 + wr - 1) / wr;
    p.tiles = (int)tiles;
    p.workgroups = 8ll * p.row_groups * ((tiles + 7) / 8);
    const Cost& c = f32 ? kF32[M <= 64 && wr == 2 ? 3 : i] : kF16[hw % 4 != 0][i];
    const int64_t used = f32 ? p.workgroups : p.row_groups * tiles;  // fp16: without those of the last eight tiles that return at once
    const double per_cu = (double)used / cus, over = per_cu > 1.0 ? per_cu - 1.0 : 0.0, rounds = (double)((used + cus - 1) / cus - 1);
    p.us = c.launch + c.chunk * chunks + (per_cu < 1.0 ? per_cu : 1.0) * (c.full + c.full_chunk * chunks) + over * (c.over + c.over_chunk * chunks) + rounds * (c.round + c.round_chunk * chunks) +
           1e-6 * c.out * positions * M * 256.0 / cus;
    if (best.wr == 0 || p.us < best.us) best = p;
  }
  return best;
}

// The form with wavefronts of their own for the inputs (fp32).  us: fitted to 150 random calls that it makes one round of workgroups of (64 - 2048
// channels, 33 - 2048 rows), within 7 % for two of three, and 0.8 for the sums that wait.
static FloatMfmaPlan PlanFloatSplit(int cus, int K, int M, int hw, int batch) {
  FloatMfmaPlan p{};
  p.wr = kSplitRowBlocks;
  p.split = true;
  p.row_groups = ((M + 31) / 32 + kSplitRowBlocks - 1) / kSplitRowBlocks;
  p.tiles = (int)(((int64_t)batch * ((hw + 3) / 4) + kSplitQuads - 1) / kSplitQuads);
  p.workgroups = 8ll * p.row_groups * ((p.tiles + 7) / 8);
  const double chunks = (K + kSplitChunk - 1) / kSplitChunk, full = (double)p.workgroups / cus;
  p.us = 4.5 + 1.57 * chunks + full * (1.73 + 0.71 * chunks);
  return p;
}

FloatMfmaPlan PlanFloatMfma(bool f32, int cus, int row_blocks, int split, int K, int M, int hw, int batch) {
  if (f32 && split == 2) return PlanFloatSplit(cus, K, M, hw, batch);
  const FloatMfmaPlan plan = PlanRows(f32, cus, row_blocks, K, M, hw, batch);
  // One round of workgroups of 256 rows x 64 positions where that is expected to take 0.88 of the time (of 11 of 150 random calls at 0.97 two were
  // slower, 1536 -> 352 @11x11 x 37 31.5 / 33.4, the others 0.85 - 0.97); over more rounds it is 1.1 times as long
  // (64 x 512 -> 512 @14x14 23.9 / 26.2).  Not in place of 64 rows per workgroup, whose four sums per output are closer to 64 bits (1024
  // channels 1.3e-7), nor of up to 384 channels, where halves of the sums would not be chunks, nor of a number of rows that is asked for.
  if (f32 && split == 1 && row_blocks == 0 && plan.wr >= 4 && K > 3 * kSplitChunk) {
    const FloatMfmaPlan own = PlanFloatSplit(cus, K, M, hw, batch);
    if (own.workgroups <= cus && own.us < 0.88 * plan.us) return own;
  }
  return plan;
}

hipError_t LaunchFloatMfma(bool f32, int cus, int row_blocks, int split, const FloatMfmaParams& p, hipStream_t stream) {
  if (p.batch <= 0 || p.M <= 0) return hipSuccess;
  if (!FloatMfmaFits(f32, p.K, p.M, p.hw, (int64_t)p.batch * p.hw)) return hipErrorInvalidValue;
  const FloatMfmaPlan plan = PlanFloatMfma(f32, cus, row_blocks, split, p.K, p.M, p.hw, p.batch);
  FloatMfmaParams q = p;
  q.qpi = (p.hw + 3) / 4;
  q.quad_aligned = p.hw % 4 == 0;
  q.total_quads = (uint32_t)p.batch * (uint32_t)q.qpi;
  q.row_blocks = (p.M + 31) / 32;
  q.row_groups = plan.row_groups;
  q.chunks = (p.K + kChunk - 1) / kChunk;
  q.padded_ksteps = FloatMfmaPaddedSteps(p.K);
  q.tiles = plan.tiles;
  if (plan.workgroups > (1ll << 30)) return hipErrorInvalidValue;
  const dim3 grid((uint32_t)plan.workgroups);
  if (plan.split) return LaunchSplit(q, grid, stream);
  switch (plan.wr) {
    case 8:
      return f32 ? Launch<8, true>(q, grid, stream) : Launch<8, false>(q, grid, stream);
    case 4:
      return f32 ? Launch<4, true>(q, grid, stream) : Launch<4, false>(q, grid, stream);
    case 2:
      return f32 ? Launch<2, true>(q, grid, stream) : Launch<2, false>(q, grid, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace pl
