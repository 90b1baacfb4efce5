// Host run of csrc/launch_shapes.hpp over row counts up to the largest that
// the calls admit (tests/test_launch_shapes.py compiles and runs it under the
// undefined-behaviour sanitizer).  Prints "ok" or the first fault.
#include <cstdio>
#include <initializer_list>
#include <cstdlib>
#include <vector>

#include "launch_shapes.hpp"

static void fail(const char *what, long a, long b, long c) {
  std::printf("%s: %ld %ld %ld\n", what, a, b, c);
  std::exit(1);
}

// Every row that any thread of the row-broadcast launch loads or stores.
static void row_bcast(long rows, int cpr, bool f16) {
  const mh::RowBcastShape s = mh::row_bcast_shape(rows, cpr, f16);
  if (s.tpr < 1 || s.rpb < 1 || s.gx < 1 || s.gy < 1 || s.gx > 32768 || s.tpr * s.gy < cpr) fail("shape", rows, cpr, s.gx);
  // one row per thread until the chip is full
  if (rows * cpr < 1 << 20 && (s.u != 1 || long(s.gx) * s.rpb < std::min(rows, 32768L * s.rpb / s.gy - s.rpb)))
    fail("rows in flight", rows, cpr, s.u);
  const long step = long(s.gx) * s.rpb, U = s.u;
  const bool all = rows <= 100000;
  std::vector<int> seen(all ? rows : 0, 0);
  auto thread = [&](long first) {
    long trips = 0, last = -1;
    mh::walk_rows(first, U * step, rows, [&](long r) {
      if (r < 0 || r >= rows || r <= last || ++trips > rows) fail("row", rows, cpr, r);
      last = r;
      for (long u = 0; u < U; ++u)
        if (all && r + u * step < rows) ++seen[r + u * step];
    });
    const long want = first < rows ? (rows - first + U * step - 1) / (U * step) : 0;
    if (trips != want) fail("trips", rows, first, trips);
  };
  if (all) {
    for (long f = 0; f < step; ++f) thread(f);
    for (long r = 0; r < rows; ++r)
      if (seen[r] != 1) fail("covered", rows, r, seen[r]);
  } else {
    for (long f : {0L, step / 2, step - 1}) thread(f);
  }
}

// The launches of one workgroup per row: consecutive, all rows, 32-bit sizes.
static void split(long rows, int threads) {
  long next = 0;
  mh::split_rows(rows, threads, [&](long r, int n) {
    if (r != next || n < 1 || long(n) * threads > 0xffffffffL) fail("launch", rows, r, n);
    next = r + n;
  });
  if (next != rows) fail("rows", rows, threads, next);
}

// Every valid input row that any 64 consecutive output pixels touch lies within
// the span from their base row.
static void conv(int B, int iH, int iW, int k, int s, int p) {
  const int oH = (iH + 2 * p - k) / s + 1, oW = (iW + 2 * p - k) / s + 1;
  if (iH + 2 * p < k || iW + 2 * p < k) return;
  const long M = long(B) * oH * oW, span = mh::conv_row_span(64, B, iH, oH, oW, k, s, p);
  for (long m0 = 0; m0 < M; ++m0) {
    const long b0 = m0 / (oH * oW), base = b0 * iH + mh::conv_base_row(int(m0 % (oH * oW) / oW), iH, s, p);
    if (base < b0 * iH || base >= (b0 + 1) * iH) fail("base row", m0, base, iH);
    for (long m = m0; m < m0 + 64 && m < M; ++m)
      for (int kh = 0; kh < k; ++kh) {
        const long ih = m % (oH * oW) / oW * s - p + kh, r = m / (oH * oW) * iH + ih;
        if (ih >= 0 && ih < iH && (r < base || r >= base + span)) fail("row span", m0, r - base, span);
      }
  }
}

int main() {
  for (int B : {1, 3})
    for (int iH : {1, 2, 5, 8, 17})
      for (int iW : {1, 3, 7, 31, 64, 100})
        for (int k : {1, 2, 3, 5, 7})
          for (int s : {1, 2, 3, 4})
            for (int p : {0, 1, 2, 3, 6}) conv(B, iH, iW, k, s, p);
  // an image of 1 GiB, 64 floats at 2048 x 2048, a few rows of which a tile sees
  if (mh::conv_row_span(64, 4, 2048, 2048, 2048, 3, 1, 1) * 2048 * 64 * 4 > 1 << 24) fail("large image", 0, 0, 0);
  const long rows[] = {1, 2, 3, 5, 255, 1024, 1025, 65537, 99999, 8388609, 2139095040, 2139095041, 2147483000, 2147483646};
  for (long r : rows)
    for (int cpr : {1, 2, 3, 8, 100, 255, 256, 257, 5000, 3000000})
      if (r * cpr < (1L << 35)) {  // 512 GiB operands and below
        row_bcast(r, cpr, false);
        row_bcast(r, cpr, true);
      }
  // many rows on a wave each, few long ones on a workgroup
  const struct { long rows; int n, th; } am[] = {{20000, 1025, 64}, {4096, 2048, 64}, {4, 64, 64}, {1, 257, 256},
                                                 {1000, 512, 256}, {4, 4000, 1024}, {4096, 4000, 256}, {1000, 50257, 1024}};
  for (const auto &a : am)
    if (mh::argmax_threads(a.rows, a.n) != a.th) fail("argmax", a.rows, a.n, mh::argmax_threads(a.rows, a.n));
  // few long slices in tiles, many or short ones flat
  const struct { long b, r, c; int es; bool vec, flat; } tr[] = {
      {128, 64, 9, 4, false, true}, {2, 8, 1000, 4, true, false}, {3, 1, 8000, 4, false, false}, {128, 1, 8000, 4, false, true},
      {4, 15, 400, 4, false, false}, {2, 8, 1000, 2, true, false}, {1, 64, 9, 4, false, false}, {512, 16, 16, 4, false, false},
      {70000, 2, 1000, 4, true, true}};
  for (const auto &t : tr)
    if (mh::transpose_flat(t.b, t.r, t.c, t.es, t.vec) != t.flat) fail("transpose", t.b, t.r, t.c);
  // a few keys of many heads by rows; long ones, and 16-bit heads of 64, by tiles
  if (!mh::attention_by_rows(true, false, false, 1, 128, 2400) || !mh::attention_by_rows(true, false, true, 4, 64, 512) ||
      !mh::attention_by_rows(false, true, false, 3, 96, 16000) || !mh::attention_by_rows(false, false, false, 3, 8, 2) ||
      mh::attention_by_rows(false, false, false, 3, 96, 16000) || mh::attention_by_rows(false, false, false, 1, 64, 2400) ||
      mh::attention_by_rows(true, false, false, 5, 64, 2400) || mh::attention_by_rows(true, false, false, 1, 8, 65536))
    fail("attention", 0, 0, 0);
  for (long r : {1L, 67108863L, 4194303L, 4194304L, 16777216L, 67108864L, 2147483647L})
    for (int threads : {64, 256, 1024}) split(r, threads);
  std::printf("ok\n");
}
