// Block tile of a 16-bit product by its sizes, type and epilogue, for the
// pipelined kernels (gemm_pipe.hip).  Host arithmetic only
// (tests/cxx/gemm_tiles_check.cpp).
#pragma once

namespace mh {

// Epilogue: no more than a bias; an activation with exponentials; a residual;
// packed rows in the general program (a ReLU, an activation without a bias).
enum TileEpi { TILE_PLAIN, TILE_GELU, TILE_RESID, TILE_GENERAL };

// A tile's time over n = its tiles in the product: rounds(n) (k K + epi[type]) +
// launch, in us, where a round is per_cu tiles on each of 256 CUs and a last
// partial round takes `half` of one up to one tile per CU and then
// `over` to 1 (per_cu = 1: `half` to 1).  Fitted to 16 (N, K) of 512 to 8192 by
// 9 M of 500 to 8192, three epilogues and both types (weights and rows in L2
// or not as they fit): 2 to 4% rms per tile, and the tile of least predicted time
// takes 0.4% longer than the fastest on average, 9% at worst.  The general program
// counts as a residual in bf16 and as a GELU in fp16, whose roundings it makes
// value by value (ReLU, 10 products of K 64 to 2048: 1.4% and 2.1% over the
// fastest on average; as no more than a bias fp16 11%, 1100 x 8192 x 512 37.9 us
// on 256x192 against 24.6 on 128x64).
struct TileTime {
  int tile, bm, bn, per_cu;
  double half, over, k, epi[3][2], launch;  // epi[TileEpi below TILE_GENERAL][fp16]
};
constexpr TileTime kTileTimes[6] = {
    {0, 128, 128, 2, 0.50, 0.80, 0.0143, {{3.6, 4.9}, {4.7, 19.8}, {6.3, 9.1}}, 5.5},
    {1, 128, 64, 2, 0.45, 0.90, 0.0092, {{1.8, 2.4}, {2.0, 7.0}, {3.1, 4.1}}, 4.7},
    {3, 128, 96, 2, 0.50, 0.80, 0.0115, {{3.4, 4.3}, {4.2, 14.6}, {5.4, 7.4}}, 4.6},
    {9, 128, 128, 2, 0.65, 0.80, 0.0127, {{4.1, 5.2}, {4.3, 20.4}, {7.2, 9.4}}, 4.4},
    {16, 256, 192, 1, 0.80, 1.00, 0.0163, {{7.8, 8.7}, {8.3, 33.5}, {15.5, 14.7}}, 2.9},
    {19, 128, 288, 1, 0.70, 1.00, 0.0240, {{0.0, 0.7}, {0.1, 18.8}, {4.6, 4.2}}, 2.7},  // whole tiles only
};

inline double tile_time(const TileTime &t, int M, int N, int K, int batch, bool f16, TileEpi epi) {
  const long n = long((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * batch, round = 256L * t.per_cu, rem = n % round;
  double rounds = double(n / round);
  if (rem && t.per_cu == 1) rounds += t.half + (1 - t.half) * double(rem) / 256;
  else if (rem) rounds += rem <= 256 ? t.half : t.over + (1 - t.over) * double(rem - 256) / 256;
  const TileEpi cost = epi != TILE_GENERAL ? epi : f16 ? TILE_GELU : TILE_RESID;
  return rounds * (t.k * K + t.epi[cost][f16]) + t.launch;
}

// Output rows that cannot be stored four at a time (N % 4 != 0, a destination or
// residual off 8 bytes): the epilogue goes value by value and takes longer than
// most loops, so that tiles whose workgroups overlap it, several to a CU, win
// over the wide ones until the loop is long.  Register-staged 64x64 for short
// loops (always at K <= 128, fp16 longer, as its roundings are), 128x64 between,
// 128x128 for the long ones; at up to 256 128x128 tiles the many-stage 128x128
// for the long ones.  Us, 64x64 | 128x64 | 128x128 | two-stage 128x128 | 256x192:
// bf16 GELU, 1100 x 8193 x 256 22.3 | 22.2 | 30.4 | 28.4 | 51.4; fp16 bias, 2000 x
// 5001 x 512 33.5 | 35.0 | 48.2 | 48.0 | 67.8, 1100 x 8193 x 128 20.4 | 22.7 | 35.2 |
// 33.2 | 59.8; bf16 bias, 4096 x 4098 x 2048 114 | 101 | 94 | 99 | 113; 1500 x 2049 x
// 2048 30.2 | 27.1 | 27.1, many-stage 22.8.
inline int unpacked_tile(bool f16, TileEpi epi, int K, long t128) {
  const bool slow = epi == TILE_RESID || (f16 && epi == TILE_GELU);
  if (t128 <= 256) return K < (f16 ? 2049 : 1024) ? 2 : 27;
  if (t128 >= 512 && K >= (slow ? 4096 : 2048)) return 0;
  return K <= 128 || (f16 && K < 2048 && (slow || K <= 512)) ? 2 : 1;
}

// dma: the operands allow direct-to-LDS loads (K % 64 == 0).  packed: output rows
// are stored four values at a time (more than 128 128x128 tiles that are not:
// unpacked_tile).  Tile codes as in gemm_pipe.hpp.
//  * M tiling evenly by 256 and N by 192 into 232..256 tiles (the decoder's FFN
//    up, 4096 x 3072: 256): direct-to-LDS 256x192 with eight waves, one
//    workgroup per CU (FFN up in the forward 33.1 -> 31.1 us; QKV, 192 tiles,
//    28.3 -> 29.5 us, so it stays below);
//  * M tiling by 128 and N by 288 into 232..256 tiles (QKV, 4096 x 2304):
//    direct-to-LDS 128x288, eight waves of 32x144, one workgroup per CU
//    (forward 1.620 -> 1.609 ms against the register-staged 128x96, whose
//    768 tiles take three rounds of two workgroups per CU);
//  * N tiling evenly by 96 with at most one tile per CU (N = 768: FFN down,
//    attention out-projection): direct-to-LDS 128x96, 4 stages, eight waves
//    (one workgroup per CU, so deep stages and two waves per SIMD hide the
//    memory latency; out-projection 13.9 -> 12.9 us against four waves);
//  * 129 to 256 128x128 tiles: direct-to-LDS 128x128, eight waves and four
//    stages (27; gemm_pipe_deep.hip), with a GELU too (bf16, 128x64 | 27, us:
//    2048 x 2048 x 512 11.1 | 10.1, 1100 x 3072 x 768 13.3 | 11.5, 500 x 8192 x
//    2048 25.9 | 22.4, 2048 x 2048 x 8192 81.7 | 61.8), but for fp16's GELU, whose
//    half-away roundings take longer than a short loop: there 64x64, whose four
//    workgroups per CU overlap one's epilogue with another's loop, below K = 768
//    and to K = 2048 at up to 192 tiles (64x64 | 27: 2048 x 2048 x 512 16.3 | 17.2,
//    1000 x 2500 x 1024 17.8 | 19.5, 1536 x 2500 x 1024 21.7 | 21.0, 2000 x 2048 x
//    2048 33.6 | 29.2);
//    At K = 64, one step of the loop, 64x64 whatever the type (27 | 64x64:
//    2048 x 2048 bias 7.1 | 6.3, 1100 x 2048 bias 6.6 | 5.2, fp16 residual at 256
//    tiles 8.7 | 8.1);
//  * more, with K <= 768 and N tiling evenly by 96 into at most two tiles per CU:
//    register-staged 128x96, unless fp16's GELU or general program (the sizes that the model below
//    knows least: its loops are longer, and 128x288 filling half the chip had
//    one shape.  The model's | 128x96, us: 8192 x 768 x 256 bias, fp16 12.2 |
//    10.9, 4096 x 1152 x 512 bf16 GELU 14.1 | 12.5; bf16 GELU at K = 768 17.1 |
//    17.5);
//  * more: the least of kTileTimes (bf16 with a residual, 4096 x 5000 x 512:
//    128x128 37.2, 256x192 50.3; fp16 GELU, 1100 x 5000 x 512: 128x64 22.3,
//    two-stage 128x128 27.6);
//  * K % 64 != 0, register-staged: 128x128 when N tiles evenly by 128 and there
//    are >= 2.5 tiles per CU, 128x96 when N tiles evenly by 96, else 128x128 /
//    128x64 / 64x64 by tile count.
// (The vocabulary head, a non-temporal output, takes direct-to-LDS 128x128
// with two stages.)
inline int auto_tile(bool dma, bool packed, bool f16, TileEpi epi, int M, int N, int K, int batch) {
  const long t128 = long((M + 127) / 128) * ((N + 127) / 128) * batch;
  const long t96 = long((M + 127) / 128) * ((N + 95) / 96) * batch;
  const long t64 = long((M + 127) / 128) * ((N + 63) / 64) * batch;
  if (dma && !packed && t128 > 128) return unpacked_tile(f16, epi, K, t128);
  const long t192w = long(M / 256) * (N / 192) * batch;
  if (dma && M % 256 == 0 && N % 192 == 0 && t192w >= 232 && t192w <= 256) return 16;
  const long t288 = long(M / 128) * (N / 288) * batch;
  if (dma && M % 128 == 0 && N % 288 == 0 && t288 >= 232 && t288 <= 256) return 19;
  if (dma && N % 96 == 0 && t96 <= 256) return 17;
  if (dma && t128 > 128 && t128 <= 256 && K <= 64) return 2;
  if (dma && t128 > 128 && t128 <= 256)
    return f16 && epi == TILE_GELU && (K < 768 || (K < 2048 && t128 <= 192)) ? 2 : 27;
  if (dma && t128 > 256 && K <= 768 && N % 96 == 0 && t96 <= 512 && !(f16 && (epi == TILE_GELU || epi == TILE_GENERAL))) return 3;
  if (dma && t128 > 256) {
    int best = 9;
    double best_t = 1e30;
    for (const TileTime &t : kTileTimes) {
      if (t.tile == 19 && (M % 128 || N % 288)) continue;
      const double us = tile_time(t, M, N, K, batch, f16, epi);
      if (us < best_t) {
        best_t = us;
        best = t.tile;
      }
    }
    return best;
  }
  if (N % 128 == 0 && t128 >= 640) return 0;
  if (N % 96 == 0) return 3;
  return (t128 >= 640 || (K >= 2048 && t128 >= 128)) ? 0 : (t64 >= 256 ? 1 : 2);
}

// Of a product that the many-stage tiles could take: whether its K is too short
// for them to fill their stages, so that register-staged 64x64 is faster.  One
// step (K = 64): yes (many-stage | 64x64, us, bf16 1 x 64 3.1 | 2.7, 2000 x 512
// 4.2 | 3.5, 500 x 2048 4.2 | 3.5), but with fp16's roundings in the epilogue only
// from about a tile per CU.  Two and three steps: from there too (K = 128 by up
// to 7%, 192 by 4%), below it the smaller many-stage tiles use more CUs.  Rows
// that are not packed: from about a tile per CU at K = 64 (16 x 250 x 250, bf16 6.5 |
// 5.9), and instead of the largest many-stage tile, 128x64, to a longer K,
// as 64x64 overlaps their epilogues (500 x 2049 x 64, fp16 bias 16% faster, bf16
// 11%; even at K = 512 in bf16 and 1024 in fp16).
inline bool short_loop(bool packed, bool f16, TileEpi epi, int M, int N, int K, int batch) {
  const long t = long((M + 63) / 64) * ((N + 63) / 64) * batch;
  if (!packed) return t > 256 ? K < (f16 ? 1024 : 512) : t > 200 && K <= 64;
  return (K <= 64 && (!f16 || epi == TILE_PLAIN)) || (K <= 192 && t > 200);
}

}  // namespace mh
