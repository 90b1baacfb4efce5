// Host run of csrc/gemm_tiles.hpp (tests/test_launch_shapes.py): tiles that
// were measured well ahead of the ones they displaced, and a defined choice
// over the range.  Prints "ok" or the first fault.
#include <cstdio>
#include <initializer_list>

#include "gemm_tiles.hpp"

using namespace mh;

int main() {
  // the tile chosen is one of `a` and `b` (within the runs' noise of each other)
  const struct { bool f16; TileEpi epi; int M, N, K, a, b; } want[] = {
      {false, TILE_GELU, 2048, 2048, 8192, 27, 27}, {false, TILE_GELU, 500, 8192, 2048, 27, 27},
      {false, TILE_GELU, 1100, 3072, 768, 27, 27},  {true, TILE_GELU, 2000, 2048, 8192, 27, 27},
      {true, TILE_GELU, 2048, 2048, 512, 2, 2},     {true, TILE_GELU, 1100, 5000, 512, 1, 2},
      {true, TILE_GELU, 8192, 4096, 512, 1, 1},     {true, TILE_GELU, 8192, 8192, 2048, 0, 9},
      {false, TILE_RESID, 4096, 5000, 512, 0, 9},   {false, TILE_RESID, 2000, 5000, 512, 1, 0},
      {false, TILE_RESID, 8192, 2500, 1024, 0, 9},  {true, TILE_GELU, 8192, 2048, 8192, 9, 16},
      {false, TILE_PLAIN, 2048, 2048, 64, 2, 2},    {true, TILE_RESID, 2048, 2048, 64, 2, 2},
      {true, TILE_PLAIN, 8192, 768, 256, 3, 3},     {false, TILE_PLAIN, 8192, 768, 128, 3, 3},
      {true, TILE_GELU, 8192, 768, 256, 1, 2},      {false, TILE_GELU, 4096, 1152, 512, 3, 3},
      {true, TILE_GENERAL, 1100, 8192, 512, 1, 2},  {true, TILE_GENERAL, 4096, 4096, 512, 1, 1}, {true, TILE_GENERAL, 2048, 2048, 512, 27, 27},
      {false, TILE_GENERAL, 1100, 8192, 256, 1, 2}};
  for (const auto &w : want) {
    const int t = auto_tile(true, true, w.f16, w.epi, w.M, w.N, w.K, 1);
    if (t != w.a && t != w.b) {
      std::printf("%d x %d x %d f16 %d epi %d: tile %d\n", w.M, w.N, w.K, w.f16, w.epi, t);
      return 1;
    }
  }
  // rows that are stored value by value
  const struct { bool f16; TileEpi epi; int M, N, K, a, b; } odd[] = {
      {false, TILE_GELU, 1100, 8193, 256, 1, 2}, {true, TILE_PLAIN, 1100, 8193, 128, 2, 2}, {true, TILE_PLAIN, 2000, 5001, 512, 1, 2},
      {true, TILE_RESID, 4096, 4098, 2048, 1, 2}, {false, TILE_PLAIN, 4096, 4098, 2048, 0, 0}, {true, TILE_GELU, 1100, 2501, 2048, 2, 2},
      {false, TILE_PLAIN, 1500, 2049, 2048, 27, 27}};
  for (const auto &w : odd) {
    const int t = auto_tile(true, false, w.f16, w.epi, w.M, w.N, w.K, 1);
    if (t != w.a && t != w.b) {
      std::printf("%d x %d x %d f16 %d epi %d, value by value: tile %d\n", w.M, w.N, w.K, w.f16, w.epi, t);
      return 1;
    }
  }
  // where the many-stage tiles give way to 64x64
  const struct { bool f16; TileEpi epi; int M, N, K; bool yes; } shorter[] = {
      {false, TILE_PLAIN, 1, 64, 64, true},     {false, TILE_GELU, 500, 2048, 64, true}, {true, TILE_PLAIN, 33, 96, 64, true},
      {true, TILE_GELU, 33, 96, 64, false},     {true, TILE_GELU, 500, 2048, 64, true},  {false, TILE_PLAIN, 2000, 512, 192, true},
      {false, TILE_PLAIN, 2000, 512, 256, false}, {false, TILE_PLAIN, 1, 64, 128, false}, {false, TILE_PLAIN, 33, 97, 64, false},
      {true, TILE_PLAIN, 500, 2049, 512, true}, {true, TILE_PLAIN, 500, 2049, 1024, false},
      {false, TILE_PLAIN, 4000, 250, 64, true}, {false, TILE_PLAIN, 4000, 250, 128, false}};
  for (const auto &w : shorter)
    if (short_loop(w.N % 4 == 0, w.f16, w.epi, w.M, w.N, w.K, 1) != w.yes) {
      std::printf("%d x %d x %d f16 %d epi %d: short loop %d\n", w.M, w.N, w.K, w.f16, w.epi, !w.yes);
      return 1;
    }
  for (int M : {1, 129, 4096, 100000})
    for (int N : {1, 288, 5000, 100000})
      for (int K : {64, 512, 8192, 1 << 20})
        for (int e = 0; e < 32; ++e) {
          const int t = auto_tile(e & 1, e < 16, e & 2, TileEpi(e / 4 % 4), M, N, K, 3);
          if ((t == 19 && (M % 128 || N % 288)) || ((t >= 7) && !(e & 1))) {
            std::printf("tile %d for %d x %d x %d\n", t, M, N, K);
            return 1;
          }
        }
  std::printf("ok\n");
}
