// Direct-to-LDS pipelined kernels on small block tiles with many stages, for
// products whose tiles do not fill the chip (a prompt's or a small batch's
// layer GEMMs): at most one workgroup per CU, so its LDS is all stages.
//
// What bounds such a product is the memory latency: with S stages, S - 1 slabs
// of K are in flight and a 64-wide step takes latency / (S - 1), but no less
// than about 0.11 us (the waits, the barrier and the fragment reads of one
// step).  The block tiles of the full-chip products ran them at 0.4 us per
// step (three or four stages) on a few dozen of the 256 CUs.  Measured against
// those (bf16, weights cold in L2, us): 237 x 768 x 768 8.5 -> 5.4, 237 x 768 x
// 3072 20.2 -> 10.0, 237 x 2304 x 768 8.9 -> 6.9, 512 x 2048 x 2048 14.5 ->
// 10.9, 500 x 2048 x 8192 59 -> 34.5, 2048 x 1024 x 4096 33 -> 23.7.  More stages
// than here (13 instead of 10 at 32x64, 9 instead of 8 at 64x64) changed
// nothing; K split over a workgroup's waves with fragments straight from
// memory was slower than three stages (the MFMA operand layout puts sixteen
// rows in each quarter of a load).
// 27 is the 128x128 tile of products of 129 to 256 such tiles, eight waves and
// four stages: two waves per SIMD and three slabs in flight where the
// register-staged four-wave tile has one of each (bf16, us: 2000 x 2048 x 8192
// 87.4 -> 74.5, 2000 x 2048 x 2048 23.9 -> 21.8, 4096 x 1024 x 4096 44.4 -> 40.3,
// 4096 x 1024 x 1024 15.5 -> 13.7; fp16 2000 x 2048 x 2048 28.9 -> 24.3; four waves
// on four stages 80.6, 21.2, 40.4, 13.7 and 26.5).
// Tiles: 20 64x64, 21 64x48, 22 64x96, 23 32x64, 24 32x48, 25 128x64, 26 32x32,
// 27 128x128.
#include "gemm_pipe.hpp"

namespace mh {

namespace {

template <int DT, int EK>
hipError_t run(int tile, const void *A, const void *Bt, int M, int N, int K, long lda, long ldb, int batch, long sa,
               long sb, long sc, const EpiArgs &ep, hipStream_t st) {
  typedef PipeKindT<EK> KT;
  switch (tile) {
  case 20: launch_dma<DT, 64, 64, 2, 2, 8, EK>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st); break;
  case 22: launch_dma<DT, 64, 96, 2, 2, 7, EK>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st); break;
  case 25: launch_dma<DT, 128, 64, 4, 2, 6, EK>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st); break;
  case 27: launch_dma<DT, 128, 128, 4, 2, 4, EK>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st); break;
  // 48-column wave tiles, for LayerNorm partials of 48 columns
  case 21:
    if constexpr (KT::ST) launch_dma<DT, 64, 48, 4, 1, 10, EK>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st);
    else return hipErrorNotSupported;
    break;
  case 24:
    if constexpr (KT::ST) launch_dma<DT, 32, 48, 2, 1, 13, EK>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st);
    else return hipErrorNotSupported;
    break;
  // (a folded LayerNorm takes at most 4 threads per tile row)
  case 23:
    if constexpr (!KT::LN) launch_dma<DT, 32, 64, 2, 2, 10, EK>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st);
    else return hipErrorNotSupported;
    break;
  case 26:
    if constexpr (!KT::LN) launch_dma<DT, 32, 32, 2, 2, 16, EK>(A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st);
    else return hipErrorNotSupported;
    break;
  default: return hipErrorNotSupported;
  }
  return hipGetLastError();
}

}  // namespace

hipError_t gemm_pipe_deep(int dt, int kind, int tile, const void *A, const void *Bt, int M, int N, int K, long lda, long ldb,
                          int batch, long sa, long sb, long sc, const EpiArgs &ep, hipStream_t st) {
#define MH_RUN(DT, EK) \
  case EK: return run<DT, EK>(tile, A, Bt, M, N, K, lda, ldb, batch, sa, sb, sc, ep, st)
  if (dt == F16) {
    switch (kind) {
      MH_RUN(F16, PK_GENERAL);
      MH_RUN(F16, PK_PLAIN);
      MH_RUN(F16, PK_BIAS);
      MH_RUN(F16, PK_BIAS_GELU);
      MH_RUN(F16, PK_BIAS_RESID);
    default: return hipErrorNotSupported;
    }
  }
  switch (kind) {
    MH_RUN(BF16, PK_GENERAL);
    MH_RUN(BF16, PK_PLAIN);
    MH_RUN(BF16, PK_BIAS);
    MH_RUN(BF16, PK_BIAS_GELU);
    MH_RUN(BF16, PK_BIAS_RESID);
    MH_RUN(BF16, PK_LN_BIAS);
    MH_RUN(BF16, PK_LN_BIAS_GELU);
    MH_RUN(BF16, PK_BIAS_RESID_ST);
  default: return hipErrorNotSupported;
  }
#undef MH_RUN
}

}  // namespace mh
