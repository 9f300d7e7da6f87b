// dispatch.hpp -- the rules on sizes that choose between the library's
// kernels and work decompositions: host arithmetic on the shape and the number
// of CUs alone, no HIP, so that they compile and can be checked without a GPU.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "swamp_qmm.h"

namespace swamp {

// Full tile (tokens, weight rows) and K step of the fused bf16 GEMM.
constexpr int kGemmTokens = 256, kGemmRows = 256, kGemmK = 64;

// Work decomposition of one bf16 GEMM call.
//  kSmall  at most 64 tokens: 64-token tiles (a quarter of the MFMA work of
//          a full tile for the same weight stream), split along K into up
//          to 8 pieces while they fill at most half the CUs;
//  kSplit  at most half a round of tiles: full tiles, 128-token halves or
//          64-token quarters, those that hold tokens split along K into up to 8
//          pieces while they fit one round, whichever is estimated fastest;
//  kRounds full tiles in complete rounds, a last round at most half full as
//          128-token halves (no partial sums).
// Split pieces write partial tiles to scratch, summed in piece order by a
// second kernel (deterministic).  Without scratch the pieces add into
// zeroed y with float atomics (and kSplit takes halves).
// The kSplit estimate is fitted to the measured times of every part size and
// piece count of 3052 shapes (65 to 2048 tokens, 1024 to 28672 rows, 1024 to 28672
// weights, all formats; it meets those near the best of their shape within 3%
// rms): 13 us to fill a whole tile's stages and store it, the K steps below
// while a round is full (0.78 of a step when few tiles are in flight), 5.7 us for
// the second kernel and 3.4 TB/s for its partial sums, written and read.  The
// choice is within 0.5% of the best on average, 16% at worst.  An
// estimate from single shapes (2.04 us a step, 2 us for the second kernel) had
// split where it does not pay and taken halves where whole tiles in two pieces
// are faster: us, that choice / this one, 256 tokens x 4096 x 1024 Q4_0 19.2 /
// 15.4 (quarters, 2 pieces / 1), 300 x 14336 x 5120 Q8_0 109.9 / 90.4 (halves /
// whole tiles in 2 pieces), 640 x 8192 x 5120 Q8_0 107.9 / 87.3.  The choice of
// full tiles or halves in at most 4 pieces, both halves of a tile counted, that
// was there before either: 100 x 6144 x 4096 Q4_K 31.3, now 25.4, 300 x 6144 x
// 4096 47.0, now 35.7, 120 x 3000 x 28672 88.1, now 54.5.
struct GemmPlan {
  enum Kind { kSmall, kSplit, kRounds } kind;
  int parts;      // kSplit: tiles run whole (1), as halves (2) or quarters (4)
  int pieces;     // K pieces (1: none)
  int kps;        // K steps per piece
  int half_pieces, half_kps;  // kSplit fallback without scratch: halves
  size_t part_bytes;          // scratch for the pieces' partial sums
};

// us of one K step of a whole tile, a half, a quarter, in a full round (fitted
// with the rest of the estimate, above).
constexpr double gemm_step_us(uint32_t dt, int parts) {
  return dt == SWAMP_Q6_K   ? (parts == 1 ? 1.96 : 1.58)
         : dt == SWAMP_Q8_0 ? (parts == 1 ? 1.66 : parts == 2 ? 1.28 : 1.10)
                            : (parts == 1 ? 1.42 : parts == 2 ? 0.98 : 0.78);
}

inline GemmPlan plan_gemm_bf16(uint32_t dt, int m, int n_rows, int n_cols, int cus) {
  constexpr int kBM = kGemmTokens;
  const int tiles_m = (m + kBM - 1) / kBM, tiles_n = (n_rows + kGemmRows - 1) / kGemmRows;
  const int tiles = tiles_m * tiles_n, KT = n_cols / kGemmK;
  const size_t mn = size_t(m) * size_t(n_rows);
  auto piece_len = [&](int splits) {  // K steps per piece (whole 256-weight blocks)
    int kps = (KT + splits - 1) / splits;
    if (dt == SWAMP_Q4_K || dt == SWAMP_Q6_K) kps = (kps + 3) / 4 * 4;
    return kps;
  };
  GemmPlan p{GemmPlan::kRounds, 1, 1, KT, 1, KT, 0};
  if (m <= kBM / 4) {
    p.kind = GemmPlan::kSmall;
    int pieces = 2 * tiles <= cus ? std::max(1, std::min({cus / tiles, 8, KT / 8})) : 1;
    p.kps = piece_len(pieces);
    p.pieces = (KT + p.kps - 1) / p.kps;
  } else if (2 * tiles <= cus) {
    p.kind = GemmPlan::kSplit;
    const int hs = 4 * tiles <= cus ? std::max(1, std::min({cus / (2 * tiles), 4, KT / 8})) : 1;
    p.half_kps = piece_len(hs);
    p.half_pieces = (KT + p.half_kps - 1) / p.half_kps;
    // Calls that the allocation-free entry point's scratch holds keep fitting: a
    // split takes no more than that leaves beside the bf16 x, or than the
    // simpler choice of whole tiles or halves (2.0 and 1.3 us a step) would.
    const int fs = std::min({cus / tiles, 8, KT / 8});
    auto plain_us = [&](double step, int n) {
      return piece_len(n) * step + (n > 1 ? (2.0 * n + 1.0) * double(mn) * 4.0 / 6e6 : 0.0);
    };
    const int plain = piece_len(fs >= 2 && plain_us(2.0, fs) < plain_us(1.3, hs) ? fs : hs);
    const size_t xb = size_t(m) * size_t(n_cols) * 2 + 512;
    const size_t cap = std::max(plain < KT ? size_t((KT + plain - 1) / plain) * mn * sizeof(float) : 0,
                                SWAMP_NOALLOC_SCRATCH_BYTES -
                                    std::min(xb, SWAMP_NOALLOC_SCRATCH_BYTES));
    double best = 0;
    for (int parts = 1; parts <= (dt == SWAMP_Q6_K ? 2 : 4); parts *= 2) {
      const int rows = kBM / parts, units = (m + rows - 1) / rows * tiles_n;
      int last = 0;  // pieces of the previous candidate (rounding repeats them)
      for (int want = 1; want <= std::max(1, std::min(8, KT / 8)); want++) {
        const int kps = piece_len(want), pieces = (KT + kps - 1) / kps;
        if (pieces == last) continue;
        last = pieces;
        if (pieces > 1 && units * pieces > cus) break;
        const size_t part = pieces > 1 ? size_t(pieces) * mn * sizeof(float) : 0;
        if (part > cap) break;
        const double fill = double(units) * pieces / cus, rounds = std::ceil(fill);
        double t =
            13.0 / parts + kps * gemm_step_us(dt, parts) * rounds * (0.78 + 0.22 * fill / rounds);
        if (pieces > 1) t += 5.7 + 1.75 * pieces * double(mn) * 4.0 / 6e6;
        if (best == 0 || t < best) {
          best = t;
          p.parts = parts;
          p.pieces = pieces;
          p.kps = kps;
        }
      }
    }
  }
  p.part_bytes = p.pieces > 1 ? size_t(p.pieces) * mn * sizeof(float) : 0;
  return p;
}

// Shapes the fused Q6_K GEMM takes: it reads rows of whole block pairs
// (dword-aligned); at most 64 tokens it would run its 64-token tiles, where the
// dequantization of a tile's weights is not spread over enough tokens.
inline bool q6k_gemm_fusable(int m, int n_cols) { return m > 64 && n_cols % 512 == 0; }

// Whether a bf16 GEMM dequantizes its weights to memory once and multiplies
// them with the plain bf16 GEMM, instead of the fused kernel.
inline bool gemm_dequantize_once(uint32_t dtype, int m, int n_rows, int n_cols, int cus) {
  const long tiles = long((m + 255) / 256) * long((n_rows + 255) / 256);
  if (dtype == SWAMP_Q6_K) {
    // Q6_K's fused dequantization takes twice the vector work of the others
    // per matrix instruction, once per token tile; this route instead writes
    // and re-reads 2 bytes per weight, once.  Fused where that traffic counts
    // most -- one token tile, or two, or long rows whose tiles split along K --
    // and enough tiles are left to split.  Timed on 2146 shapes; us, fused /
    // this route.  One token tile: 65 x 4096 x 4096 25.9 / 30.1, 128 x 28672 x
    // 4096 74 / 141, 256 x 4096 x 14336 71 / 82, but with 8 or 4 tiles 65 x 2048 x
    // 14336 53 / 46, 256 x 1024 x 8192 36 / 33.  Two: 512 x 28672 x 4096 149 /
    // 183, 350 x 3584 x 6144 45 / 52, 512 x 4096 x 4096 46 / 46, 300 x 14336 x
    // 4096 88 / 86, but 512 x 3000 x 8192 (24 tiles) 65 / 59, 512 x 2048 x 1024
    // 26 / 22; over 8192 weights 16 tiles do: 450 x 3584 x 10240 71 / 79.  More:
    // 777 x 4096 x 14336 143 / 158, 700 x 7168 x 10240 153 / 191, 777 x 2048 x
    // 28672 150 / 164, but 1300 x 4096 x 8192 141 / 117, 1000 x 6144 x 4096 102 /
    // 75, and past half a round 1300 x 6144 x 14336 394 / 339.
    if (!q6k_gemm_fusable(m, n_cols)) return true;
    if (m <= 256) return 16 * tiles < cus;
    if (m <= 512) return (n_cols > 8192 ? 16 : 10) * tiles < cus;
    return n_cols <= 8192 || 2 * tiles > cus || (n_cols >= 20480 ? 16 : 8) * tiles < cus;
  }
  // The fused kernel reads 0.56-1.06 bytes per weight per tile, the plain
  // bf16 GEMM 2 (its loads from L2 bound it, not the dequantization), so the
  // fused kernel is faster wherever its 256 x 256 tiles fill whole rounds of
  // the CUs or split along K.  Between half a round and one round they leave
  // CUs idle, and the plain GEMM's 256-token x 192-row tiles fill them: this
  // route, once every weight meets enough tokens to repay the dequantization.
  // `bench.py --route-crossover` (8B shapes, us, fused / this route, Q4_0):
  // 2048 tokens qkv 113.1 / 109.4, gate_up 514.0 / 599.1, down 253.0 / 324.4,
  // o_proj 76.5 / 84.9; Q8_0 qkv 128.7 / 112.8; Q4_K qkv 116.8 / 111.4.
  if (m < 1024 || n_cols < 1024) return false;
  return 2 * tiles > cus && tiles < cus;
}

// Rows of a tile of the small-batch kernels, and of a workgroup of 16 tiles.
constexpr int kBatchTileRows = 16, kBatchGroupRows = 256;

// Whether a small-batch pass splits K over workgroups (each stages a range of x;
// the partial sums go to scratch and a second kernel adds them), instead of
// staging all of x into every workgroup in K phases.  It takes at most half the
// CUs in row groups, and activations worth splitting: from 16384 values, but not
// where a pass of phases is short.  Timed on 8164 shapes; us, phases / K groups:
//  * up to 1024 weights, two phases at most: 17 x 6144 x 1024 Q8_0 8.1 / 9.4, 32 x
//    4096 x 1024 Q4_0 7.9 / 8.9, 63 x 14337 x 1024 12.2 / 18.9; only 33 tokens
//    and more on few rows gain (64 x 4096 x 1024 11.1 / 10.9);
//  * up to 2048 weights and 32 tokens: many rows leave only 4 or 5 groups (32 x
//    12288 x 2048 Q4_K 12.4 / 13.3, 17 x 12288 x 1536 Q4_0 10.2 / 10.5), and at
//    most 16 tokens stage quickly (16 x 4096 x 2048 Q4_K 7.3 / 8.1, 16 x 2048 x
//    2048 Q4_0 6.9 / 8.0; but 16 x 4096 x 1536 Q4_K, no whole number of the phases'
//    granules, 8.3 / 7.8, 16 x 4096 x 1792 8.5 / 7.8);
//  * beyond, groups gain: 16 x 4096 x 4096 Q4_K 10.0 / 8.8, 32 x 4096 x 2048 Q6_K
//    12.7 / 11.9, 48 x 1024 x 4096 Q4_0 24.7 / 11.2.
inline bool small_batch_k_groups(int n_tok, int n_rows, int n_cols, int cus) {
  const int groups = (n_rows + kBatchGroupRows - 1) / kBatchGroupRows;
  if (2 * groups > cus || long(n_tok) * n_cols < 16384) return false;
  if (n_cols <= 1024) return n_tok > 32 && 16 * groups <= cus;
  if (n_cols <= 2048 && n_tok <= 32)
    return 32 * groups <= 5 * cus && (n_tok > 16 || n_cols % 1024 != 0);
  return true;
}

// Small-batch passes that take gemv_xs_kernel, which loads each wave's share of
// x into registers, instead of gemv_batched_kernel, which stages x through LDS.
// Every workgroup of the former converts all of x for itself, so it is faster
// only while tokens times row length are few.  Measured over 10000 shapes, 1 to
// 16 tokens x 256 to 32768 rows x 256 to 32768 weights; us, staged / registers:
//  * One tile per workgroup (rows <= 16 x the CUs): 16 waves take up to 4096
//    weights in one pass (rows of 14336 lose, 14.5 / 22.0).  Q6_K gains up to 32768 x
//    values: 1024 x 4096 at 5 tokens 10.4 / 8.3, 4096 x 2048 at 16 9.9 / 8.9.
//    Q8_0 4096 x 4096 at 5 9.9 / 8.6, but 4096 x 2560 at 12 8.8 / 9.1; Q4_0 4096 x
//    4096 at 5 8.0 / 7.6, at 8 8.1 / 9.0.  Rows of 2048 weights are one phase of
//    the staged kernel: Q8_0 4096 x 2048 at 8 8.2 / 7.6, at 14 8.4 / 8.9, Q4_0 at 6
//    6.8 / 6.5, at 12 7.1 / 7.5.
//  * Q4_K's scale unpacking makes the line fall faster than the token count
//    rises: 4096 x 4096 at 5 7.9 / 7.5, at 6 8.0 / 8.4, at 8 8.1 / 10.1; 4096 x
//    2048 at 8 7.1 / 7.7, at 16 7.5 / 11.7.  Rows that are not whole 1024-weight
//    granules of the staged kernel leave more room, most on few tiles: 4096 x
//    1280 at 12 8.1 / 7.7, 512 x 1280 at 14 7.2 / 6.2.
//  * Rows of 256 weights gain nothing (5.1 / 5.3).
//  * More rows take 2 to 8 tiles per workgroup, whose 8 waves are all busy when
//    the row is whole 2048-weight passes; each pass beyond the second costs
//    more than staging: Q4_K 14336 x 4096 at 5 16.0 / 14.4, but 5120 x 8192 at
//    4 12.7 / 16.2 and 5120 x 14336 at 2 16.7 / 23.4; Q4_0 5120 x 28672 at 1
//    25.0 / 39.0.  Q8_0 and Q6_K stream enough weights behind their x for that
//    at 4 tiles: 14336 x 8192 at 4 34.9 / 33.4, 14336 x 6144 at 5 27.6 / 25.2.
//  * 5 and 6 tiles run the instance of 8, whose idle tiles cost the nibble
//    formats more than they gain: 20480 x 2048 at 16 Q4_K 13.4 / 14.8, but 28672
//    x 2048 at 8 14.9 / 13.8.  So does a single token on 4 tiles: 13.7 / 14.5.
inline bool small_batch_in_registers(uint32_t dtype, int n_tok, int n_rows, int n_cols, int cus) {
  const int n_tiles = (n_rows + kBatchTileRows - 1) / kBatchTileRows;
  const int nt = (n_tiles + cus - 1) / cus;  // tiles per workgroup
  const long nx = long(n_tok) * n_cols;
  const bool nibbles = dtype == SWAMP_Q4_0 || dtype == SWAMP_Q4_K, q8 = dtype == SWAMP_Q8_0;
  if (n_tok > 16 || n_cols % 256 != 0 || n_cols < 512) return false;
  if (nt <= 1) {
    if (n_cols > 4096 || (n_cols == 2048 && n_tok > (nibbles ? 6 : q8 ? 9 : 16))) return false;
    if (dtype == SWAMP_Q4_K) {
      if (n_cols % 1024 == 0) return nx * n_tok <= (n_cols > 1024 ? 131072 : 98304);
      if (n_cols < 2048 && 4 * n_tiles <= cus) return true;
      return nx <= 21504 && nx * n_tok <= (8 * n_tiles <= 5 * cus ? 262144 : 196608);
    }
    return nx <= (q8 ? 28672 : nibbles ? 27648 : 32768);
  }
  if (nt > 8 || n_cols % 2048 != 0) return false;
  if (nibbles) {
    if (n_tok < (nt <= 3 ? 2 : 3) || nt == 5 || nt == 6) return false;
    if (n_cols == 2048) return n_tok <= (nt == 2 ? 9 : 12);
    return n_cols == 4096 && nt <= 4 && nx <= (nt == 2 ? 28672 : 32768);
  }
  if (n_cols == 2048) return n_tok <= (q8 && nt == 2 ? 13 : 16);
  if (n_cols == 4096) return nx <= (nt >= 3 ? 57344 : 32768);
  return n_cols <= 8192 && nt >= 4 && nt <= (q8 ? 5 : 4) && nx <= 32768;
}

// Whether the decode GEMV behind SwiGLU forms silu(gate) * up once per
// workgroup while staging, instead of staging gate and up and multiplying in
// every row set.  The product is formed sooner, but with Q8_0 and Q6_K rows of
// 4097 to 8192 weights (two waves per row) matrices of more than one tile per
// row set measured slower behind it (the tile loop is the same code; in the
// other form each wave reaches it at its own time): Q8_0 beyond 8 rows of 8192
// weights per CU, Q6_K beyond 8 rows per CU, 12 when it adds to y.  us, both staged /
// product: Q8_0 2048 x 8192 8.0 / 7.7, 2100 x 8192 8.2 / 8.6, 2816 x 5632 8.1 /
// 8.0, 5120 x 5632 9.6 / 10.5, 6144 x 8192 13.2 / 14.6, 8192 15.6 / 17.1; Q6_K
// 1900 x 5632 8.4 / 7.2, 2304 8.7 / 8.9, 4096 x 8192 11.3 / 12.8, added 2560 x
// 8192 10.1 / 9.3, 4096 12.2 / 12.9; Q4_K 4096 x 8192 8.9 / 8.2, 8192 x 8192 12.2 /
// 12.0.  Other row lengths gain everywhere: Q8_0 8192 x 4096 10.4 / 9.6, 8192 x
// 14336 27.3 / 24.8, Q6_K 8192 x 8704 31.3 / 24.9.
inline bool swiglu_product_staged(uint32_t dtype, int n_rows, int n_cols, bool accumulate,
                                  int cus) {
  if (dtype == SWAMP_Q4_0 || dtype == SWAMP_Q4_K || n_cols <= 4096 || n_cols > 8192) return true;
  if (dtype == SWAMP_Q8_0) return long(n_rows) * n_cols <= 8L * 8192 * cus;
  return n_rows <= (accumulate ? 12 : 8) * cus;
}

}  // namespace swamp
