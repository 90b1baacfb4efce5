// fp32 MFMA GEMM and implicit-GEMM convolution for gfx950: C[M,N] = A[M,K] *
// Bt[N,K]^T with the fused epilogue of gemm_common.hpp, full fp32 products
// and sums (v_mfma_f32_16x16x4f32).  Operands in whole 16-byte chunks (K, the
// row strides and a convolution's channels multiples of 4, 16-byte aligned)
// with less than 2 GiB under a tile's rows; every other fp32 product runs on
// gemm.hip's general kernel.
//
// Bound: the fp32 matrix rate, 1/16 of the bf16 one (157 TFLOP/s nominal; a
// register-only loop of this instruction reaches 154, a large library product
// 140 to 154).  A 128-byte slab of K is 8 MFMAs of 32 cycles per 16x16
// fragment, so what decides is that no wave waits between slabs, and how
// evenly the tiles spread over 256 CUs:
//   * slabs double-buffered in LDS, the two after next in registers; every
//     load is unconditional, through buffer resources that return zeros for
//     what lies outside; one barrier per slab, waiting for LDS only, with the second half's
//     MFMAs after it while the next slab's fragments are read;
//   * the four MFMAs of a 16-byte chunk interleaved over all fragments;
//   * tiles 64x64, 32x64 and 32x32 on four waves, by the work of the busiest
//     CU (auto_tile).  128x128 and 128x64 tiles, on four or eight waves,
//     were no faster on 4096 x 4096 x 1024 and behind on every smaller product
//     (fewer, coarser tiles), and four slabs in registers changed nothing.
// On 4096 x 4096 x 1024 (128 TFLOP/s) the matrix cores were busy 76% of the
// kernel before the buffer resources replaced 20 VALU instructions per slab
// (287 -> 269 us).
// Measured against the 64x64 general kernel that these products ran on
// (conditional loads, one slab ahead): 2000 x 1536 x 512 42.3 -> 35 us, 2000
// x 512 x 2048 55.8 -> 40.5, 1000 x 5000 x 768 93 -> 68; the convolution 16 x 56
// x 56 x 64 -> 128 146 -> 86.
//
// Convolution: the A loader gathers im2col chunks (4 channels of one filter
// tap) from the NHWC activation; a thread stages the same K column of one or
// two output pixels and steps its (tap, channel) state by 32 channels per slab
// without dividing.
#include <algorithm>

#include "mh_common.hpp"
#include "mh_kernels.hpp"
#include "gemm_common.hpp"
#include "launch_shapes.hpp"

namespace mh {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// Barrier between LDS writers and readers that leaves global loads in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int V> struct Set { static constexpr int value = V; };

// Steps of an im2col column by one slab (32 values): channels, and whole taps.
struct ConvStep {
  int dic = 0, dkh = 0, dkw = 0;
};

template <int BM, int BN, int WGM, int WGN, bool CONV>
__global__ void __launch_bounds__(WGM * WGN * 64)
gemm_f32_kernel(const float *__restrict__ A, const float *__restrict__ Bt, int M, int N, int K, long lda, long ldb,
                long sa, long sb, long sc, EpiArgs ep, ConvArgs cv, ConvStep cs) {
  constexpr int NT = WGM * WGN * 64, BK = 32;
  constexpr int WTM = BM / WGM, WTN = BN / WGN, FM = WTM / 16, FN = WTN / 16;
  constexpr int ACH = BM * 8 / NT, BCH = BN * 8 / NT;
  static_assert(ACH >= 1 && BCH >= 1 && FM >= 1 && FN >= 1, "tile does not fit the thread count");
  __shared__ u32x4 lds[2][(BM + BN) * 8];  // [buf][A rows | Bt rows][8 chunks], chunk c of row r at c ^ (r & 7)

  // tile order: each XCD a contiguous eighth of the tiles, in groups of 8 tile rows
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN, ntiles = tiles_m * tiles_n;
  int pid = blockIdx.x;
  if ((ntiles & 7) == 0) pid = (pid & 7) * (ntiles >> 3) + (pid >> 3);
  const int span = 8 * tiles_n, gid = pid / span, fm = gid * 8, gs = min(tiles_m - fm, 8);
  const int m0 = (fm + (pid % span) % gs) * BM, n0 = ((pid % span) / gs) * BN;

  const int z = blockIdx.z;
  A += z * sa;
  Bt += z * sb;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / WGN, wn = wave % WGN, li = lane & 15, lg = lane >> 4;

  // staging: chunk c of rows r0 + i NT / 8 of A and of Bt, by 32-bit byte
  // offsets into buffer resources over the tile's rows (rows past M / N are
  // clamped: they feed outputs that are not stored).  What lies outside (K's
  // tail, slabs past the end, padding taps) gets an offset past the resource's
  // end, which the hardware returns as zeros: no select per value, and a slab
  // adds a scalar.  (Selects beside the load waited for it at once, a memory
  // latency on every slab; beside the LDS store they took as many VALU
  // instructions as there are MFMAs.)
  constexpr uint32_t kOut = 0x80000000u;
  const int r0 = tid >> 3, c = tid & 7;
  uint32_t ao[ACH], bo[BCH];
  int ih0[ACH], iw0[ACH];
  long abase, alen;
  if constexpr (CONV) {
    const int img = cv.oH * cv.oW, b0 = m0 / img;
    const int row0 = conv_base_row((m0 - b0 * img) / cv.oW, cv.iH, cv.s, cv.p);
    abase = (long(b0) * cv.iH + row0) * cv.iW * cv.ldx;
    alen = long(cv.B) * cv.iH * cv.iW * cv.ldx - (cv.ldx - cv.iC) - abase;
#pragma unroll
    for (int i = 0; i < ACH; ++i) {
      const int m = min(m0 + r0 + i * (NT / 8), M - 1);
      const int ow = m % cv.oW, t = m / cv.oW, oh = t % cv.oH, b = t / cv.oH;
      ih0[i] = oh * cv.s - cv.p;
      iw0[i] = ow * cv.s - cv.p;
      // element offset of tap (0, 0) (it may lie before the base; modulo 2^32)
      ao[i] = ((uint32_t(b - b0) * uint32_t(cv.iH) + uint32_t(ih0[i] - row0)) * uint32_t(cv.iW) + uint32_t(iw0[i])) *
              uint32_t(cv.ldx);
    }
  } else {
    abase = long(m0) * lda;
    alen = long(min(BM, M - m0) - 1) * lda + K;
#pragma unroll
    for (int i = 0; i < ACH; ++i) ao[i] = (uint32_t(min(r0 + i * (NT / 8), M - 1 - m0)) * uint32_t(lda) + c * 4) * 4;
  }
#pragma unroll
  for (int i = 0; i < BCH; ++i) bo[i] = (uint32_t(min(r0 + i * (NT / 8), N - 1 - n0)) * uint32_t(ldb) + c * 4) * 4;
  const __amdgpu_buffer_rsrc_t ares = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(A + abase), 0,
                                                                        int(min(alen * 4, 0x7fffffffL)), 0x00020000);
  const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(Bt + long(n0) * ldb), 0, int(min((long(min(BN, N - n0) - 1) * ldb + K) * 4, 0x7fffffffL)), 0x00020000);
  int ks = 0;  // first K column of the slab loaded next
  int ic = 0, kh = 0, kw = 0;
  if constexpr (CONV) {
    const int tap = c * 4 / cv.iC;
    ic = c * 4 - tap * cv.iC;
    kh = tap / cv.kW;
    kw = tap - kh * cv.kW;
  }
  // Slab s is held in set s % 2, requested two steps before it is stored.
  u32x4 ra[2][ACH], rb[2][BCH];
  auto gload = [&](auto setc) {
    constexpr int d = decltype(setc)::value;
    const bool in = ks + c * 4 < K;  // K % 4 == 0: a chunk is inside or past the end
    if constexpr (CONV) {
      const uint32_t toff = (uint32_t(kh) * uint32_t(cv.iW) + uint32_t(kw)) * uint32_t(cv.ldx) + ic;
#pragma unroll
      for (int i = 0; i < ACH; ++i) {
        const bool ok = in && unsigned(ih0[i] + kh) < unsigned(cv.iH) && unsigned(iw0[i] + kw) < unsigned(cv.iW);
        ra[d][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ares, ok ? (ao[i] + toff) * 4 : kOut, 0, 0));
      }
    } else {
#pragma unroll
      for (int i = 0; i < ACH; ++i)
        ra[d][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ares, in ? ao[i] : kOut, ks * 4, 0));
    }
#pragma unroll
    for (int i = 0; i < BCH; ++i)
      rb[d][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(bres, in ? bo[i] : kOut, ks * 4, 0));
    ks += BK;
    if constexpr (CONV) {
      ic += cs.dic;
      int carry = cs.dkw;
      if (ic >= cv.iC) {
        ic -= cv.iC;
        ++carry;
      }
      kw += carry;
      kh += cs.dkh;
      if (kw >= cv.kW) {
        kw -= cv.kW;
        ++kh;
      }
    }
  };
  auto sstore = [&](u32x4 *buf, auto setc) {
    constexpr int d = decltype(setc)::value;
#pragma unroll
    for (int i = 0; i < ACH; ++i) {
      const int r = r0 + i * (NT / 8);
      buf[r * 8 + (c ^ (r & 7))] = ra[d][i];
    }
#pragma unroll
    for (int i = 0; i < BCH; ++i) {
      const int r = r0 + i * (NT / 8);
      buf[BM * 8 + r * 8 + (c ^ (r & 7))] = rb[d][i];
    }
  };

  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // fragments of half KS (16 K values) of the slab in buf
  auto frags = [&](const u32x4 *buf, int ks, u32x4 (&af)[FM], u32x4 (&bf)[FN]) {
    const int ch = ks * 4 + lg;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int r = wm * WTM + i * 16 + li;
      af[i] = buf[r * 8 + (ch ^ (r & 7))];
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int r = wn * WTN + j * 16 + li;
      bf[j] = buf[BM * 8 + r * 8 + (ch ^ (r & 7))];
    }
  };
  auto mma = [&](const u32x4 (&af)[FM], const u32x4 (&bf)[FN]) {
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(bf[j][e]), __uint_as_float(af[i][e]),
                                                           acc[i][j], 0, 0, 0);
  };
  constexpr int NM = 4 * FM * FN, NR = FM + FN, NS = ACH + BCH;
  const int KT = (K + BK - 1) / BK;
  u32x4 af0[FM], bf0[FN], af1[FM], bf1[FN];
  gload(Set<0>{});
  gload(Set<1>{});
  sstore(lds[0], Set<0>{});
  gload(Set<0>{});
  lds_barrier();
  frags(lds[0], 0, af0, bf0);
  // step kt of slab kt in lds[U & 1], U = kt & 1
  auto step = [&](auto uc) {
    constexpr int U = decltype(uc)::value;
    const u32x4 *cur = lds[U];
    u32x4 *nxt = lds[U ^ 1];
    // phase A: the first half's MFMAs beside the second half's fragment reads,
    // slab kt + 1 into the other buffer, whose last reads were before the
    // previous barrier, and the request for slab kt + 3; slabs past the
    // end are zeros
    frags(cur, 1, af1, bf1);
    mma(af0, bf0);
    sstore(nxt, Set<U ^ 1>{});
    gload(Set<U ^ 1>{});
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      constexpr int PER = (NR + 2 * NS + NM - 1) / NM;  // memory operations per MFMA
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
      for (int u = i * PER; u < (i + 1) * PER; ++u) {
        if (u < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        else if (u < NR + NS) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        else if (u < NR + 2 * NS) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
      }
    }
    // (left to the scheduler, the barrier and its wait for LDS moved up among
    // the MFMAs that are to cover them)
    __builtin_amdgcn_sched_barrier(0);
    lds_barrier();
    // phase B: the second half's MFMAs beside the next slab's first fragments
    frags(nxt, 0, af0, bf0);
    mma(af1, bf1);
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      constexpr int PER = (NR + NM - 1) / NM;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
      for (int u = i * PER; u < (i + 1) * PER; ++u)
        if (u < NR) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // (an odd slab count runs one more step on a slab of zeros: with an exit
  // between the steps the accumulators changed registers from step to step)
  for (int kt = 0; kt < KT; kt += 2) {
    step(Set<0>{});
    step(Set<1>{});
  }
  lds_barrier();
  store_tile<F32, BM, BN, WTM, WTN, FM, FN, WGM * WGN>(acc, reinterpret_cast<float *>(&lds[0][0]), ep, m0 + wm * WTM,
                                                      n0 + wn * WTN, M, N, wave, lane,
                                                      ep.mode == EPI_ROWMAJOR ? z * sc : 0);
}

template <int BM, int BN, int WGM, int WGN>
void launch(const float *A, const float *Bt, int M, int N, int K, long lda, long ldb, int batch, long sa, long sb,
            long sc, const EpiArgs &ep, const ConvArgs *cv, hipStream_t st) {
  const dim3 grid(unsigned(((M + BM - 1) / BM) * ((N + BN - 1) / BN)), 1, unsigned(batch)), block(WGM * WGN * 64);
  ConvStep cs;
  if (cv) {
    const int dtap = 32 / cv->iC;
    cs.dic = 32 % cv->iC;
    cs.dkh = dtap / cv->kW;
    cs.dkw = dtap % cv->kW;
    hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, WGM, WGN, true>), grid, block, 0, st, A, Bt, M, N, K, lda, ldb, sa, sb, sc,
                       ep, *cv, cs);
  } else {
    hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, WGM, WGN, false>), grid, block, 0, st, A, Bt, M, N, K, lda, ldb, sa, sb,
                       sc, ep, ConvArgs{}, cs);
  }
}

struct Tile {
  int bm, bn;
  double per;  // time per unit of tile area against 64x64 (a smaller tile reads more operands per output)
};
const Tile kTiles[3] = {{64, 64, 1.0}, {32, 64, 1.07}, {32, 32, 1.12}};

// The tile whose busiest CU has the least to do: whole tiles per CU times the
// tile's area (a CU runs its resident tiles side by side on the same matrix
// cores).  Both sides: 4096 x 4096 x 1024 in 64x64 tiles 269 us, 32x64 288,
// 32x32 302 (the weights of kTiles); 2048 x 768 x 3072 is 1.5 64x64 tiles per
// CU, 106 us, or three 32x64, 85; 300 x 512 x 512 40 / 80 / 160 tiles, 12.9 /
// 8.6 / 8.1.
int auto_tile(int M, int N, int batch) {
  int best = 0;
  double best_t = 1e30;
  for (int i = 0; i < 3; ++i) {
    const long tiles = long((M + kTiles[i].bm - 1) / kTiles[i].bm) * ((N + kTiles[i].bn - 1) / kTiles[i].bn) * batch;
    const double t = double((tiles + 255) / 256) * kTiles[i].bm * kTiles[i].bn * kTiles[i].per;
    if (t < best_t) {
      best_t = t;
      best = i;
    }
  }
  return best;
}

}  // namespace

bool gemm_f32_ok(const void *A, const void *Bt, int K, long lda, long ldb, long sa, long sb, const ConvArgs *cv) {
  const bool b = K > 0 && K % 4 == 0 && ldb % 4 == 0 && sb % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)Bt % 16 == 0;
  // 32-bit byte offsets within a tile's 64 rows (a convolution's: within the
  // input rows that 64 output pixels touch), below the out-of-range offset 2^31
  const long rows = 64 * 4, lim = 0x7fffffffL;
  if (!b || long(ldb) * rows > lim || ldb < 0) return false;
  if (!cv) return lda % 4 == 0 && sa % 4 == 0 && lda >= 0 && lda * rows <= lim;
  const long span = conv_row_span(64, cv->B, cv->iH, cv->oH, cv->oW, cv->kH, cv->s, cv->p);
  return cv->iC % 4 == 0 && cv->ldx % 4 == 0 && span * cv->iW * cv->ldx * 4 <= lim;
}

hipError_t gemm_f32(const float *A, const float *Bt, int M, int N, int K, long lda, long ldb, int batch, long sa,
                    long sb, long sc, const EpiArgs &ep, const ConvArgs *cv, int tile, hipStream_t st) {
  if (M <= 0 || N <= 0 || batch <= 0) return hipSuccess;
  if (tile < 0 || tile > 2) tile = auto_tile(M, N, batch);
  switch (tile) {
  case 0: launch<64, 64, 2, 2>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, cv, st); break;
  case 1: launch<32, 64, 2, 2>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, cv, st); break;
  default: launch<32, 32, 2, 2>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, cv, st); break;
  }
  return hipGetLastError();
}

}  // namespace mh
