// Launch shapes and row walks that must hold for every row count that the
// calls admit (just below 2^31, far past what a test can allocate).  Kept free
// of device code, so that the host compiler can run them over those counts
// (tests/cxx/launch_shapes_check.cpp).
#pragma once

#include <algorithm>

namespace mh {

// f(r) for r = first, first + step, ... below rows.  64 bits: a step of 2^23
// past a row count near 2^31 leaves the range of int.
template <class F>
__host__ __device__ __forceinline__ void walk_rows(long first, long step, long rows, F f) {
  for (long r = first; r < rows; r += step) f(r);
}

// f(row0, n) for the launches that cover rows with one workgroup of `threads`
// per row: a launch's work-items must fit in 32 bits.
template <class F> inline void split_rows(long rows, int threads, F f) {
  const long cap = 0xffffffffL / threads;
  for (long r = 0; r < rows; r += cap) f(r, int(std::min(cap, rows - r)));
}

// Threads per row of an argmax of rows of n loads (values or 16-byte chunks): a
// wave up to 256 (four per lane), and up to 2048 where the rows alone fill the
// chip; 1024 threads for the longest rows and for few long ones.  64 | 256 |
// 1024 threads, bf16, us: chunks, 20000 rows of n = 256 14.9 | 20.2 | 70.8, 4096
// of 2048 23.1 | 22.9 | 24.7, 33 of 4000 8.5 | 4.9 | 4.6, 1000 of 4000 12.7 |
// 12.4 | 14.3; values, 4096 of 1025 3.7 | 5.9 | 17.5, 1000 of
// 50257 68.8 | 24.1 | 19.2.
inline int argmax_threads(long rows, int n) {
  if (n <= 256 || (rows >= 2048 && n <= 2048)) return 64;
  return n >= 4096 || (n >= 2048 && rows <= std::max(256, n / 8)) ? 1024 : 256;
}

// Implicit-GEMM convolution: the input row, within its image, that the offsets
// of a block of output pixels start from, for a first pixel in output row oh.
__host__ __device__ __forceinline__ int conv_base_row(int oh, int iH, int s, int p) {
  const int r = oh * s - p;
  return r < 0 ? 0 : r < iH ? r : iH - 1;
}
// No fewer than the input rows, over all images, from there to the last one that
// `pix` consecutive output pixels touch: they lie in (pix - 2) / oW + 2 output
// rows, which start s input rows apart, or what an image leaves below its last.
inline long conv_row_span(int pix, long B, long iH, long oH, long oW, long kH, long s, long p) {
  const long step = std::max(s, iH - (oH - 1) * s);
  return std::min(((pix - 2) / std::max(1L, oW) + 1) * step + kH + p, B * iH);
}

// Row-broadcast kernel: tpr threads per row, rpb rows per 256-thread
// workgroup, gx x gy workgroups for rows of cpr 16-byte chunks; up to 32768
// workgroups of one row in flight per thread, or 8192 of kRowsInFlight.
constexpr int kRowsInFlight = 4;
struct RowBcastShape {
  int tpr, rpb, gx, gy, u;
};
inline RowBcastShape row_bcast_shape(long rows, int cpr, bool f16) {
  RowBcastShape s;
  // Several rows in flight only where the chunks outnumber the threads that the
  // chip holds: below that each is a longer chain in one thread of an idle chip
  // (one | four rows, us: 300 x 256 bf16 2.4 | 3.1, fp16 2.8 | 4.8, 4096 x 1000
  // 4.2 | 4.3 and 5.9 | 6.8; 4096 x 50256 bf16 170 | 149, 20000 x 768 fp16 16.1 |
  // 15.7, 20000 x 256 fp32 7.3 | 6.5).
  s.u = rows * cpr >= (f16 ? 3L : 2L) << 19 ? kRowsInFlight : 1;
  s.tpr = std::min(cpr, 256);
  s.rpb = 256 / s.tpr;
  s.gy = (cpr + s.tpr - 1) / s.tpr;
  const long per = long(s.u) * s.rpb;
  s.gx = int(std::max(1L, std::min((rows + per - 1) / per, long((s.u == 1 ? 32768 : 8192) / s.gy))));
  return s;
}

// Whether a batch of transposes takes one workgroup per slice (slices of at most
// transpose_flat_max values with fewer than 16 rows or columns) instead of
// 64x64 tiles, `es` bytes a value, `vec` where the tiles load and store chunks.
// A slice takes its workgroup about 2.1 us + 0.17 ns per byte, the tiles 2.3 to
// 4.3 us + 1.2 ns per tile over the whole batch (slices | tiles, fp32, us: 32 of
// 64 x 9 2.4 | 4.1, 2 of 8 x 1000 7.3 | 2.4, 2 of 1 x 8000 7.7 | 3.4, 128 of them 8.6 |
// 21.2, 128 of 3 x 1024 4.4 | 4.8, 64 of 512 x 15 7.9 | 4.6, 512 of them 10.7 |
// 14.9; bf16 32 of 3 x 1024 3.4 | 3.2, 512 of 8 x 1000 7.5 | 6.8).
constexpr int transpose_flat_max = 8192;
inline bool transpose_flat(long batch, long rows, long cols, int es, bool vec) {
  const long n = rows * cols, tiles = batch * ((rows + 63) / 64) * ((cols + 63) / 64);
  if (batch <= 1 || (rows >= 16 && cols >= 16) || n > transpose_flat_max) return false;
  // (a launch of tiles holds at most 65535 slices)
  return n <= 1024 || batch > 65535 || (!vec && n * es <= 4096 + 7 * tiles);
}

// Whether attention over T keys in `blocks` (batch, head) blocks takes one wave
// per query instead of the flash kernels, which do a whole 64-key tile for any
// T and a few us for the smallest call.  Rows | tiles, us: fp32, 2400 blocks, hd
// 8: T = 1 6.4 | 20.6, T = 8 15.8 | 20.2; hd 128: T = 1 17.9 | 62.6, T = 3 56.3 |
// 64.4, T = 4 85.5 | 64.1 (textbook keys 71.6 | 82.4); 512 blocks, hd 128, T = 4
// 18.1 | 15.3 (14.1 | 19.5); bf16, 2400 blocks, hd 96: T = 2 19.6 | 27.1, 16000
// blocks of T = 3 187 | 166; fp16 187 | 259; 512 blocks, hd 96, T = 1 14.4 | 8.6.
// (16-bit heads of 64 have always run on tiles; the rows' launch holds 65535
// blocks.)
inline bool attention_by_rows(bool f32, bool f16, bool textbook, int T, int hd, long blocks) {
  if (blocks > 65535 || (!f32 && hd == 64)) return false;
  if (long(T) * hd <= (f32 ? 64 : f16 ? 32 : 24)) return true;
  if (f32) return textbook ? T <= 4 && blocks >= 256 : T <= (hd <= 96 ? 4 : 3) && blocks >= 1024;
  return T <= (f16 && hd > 64 ? 4 : 2) && blocks >= 1024;
}

}  // namespace mh
