// fp32 fused attention for gfx950 (the fp32 case of attention.hip: the core
// of nn::MultiHeadAttention, reference src/nn/attention.hpp:51-99, with
// MuNet's reading of k's buffer as a [hd, B*H*T] matrix, or textbook keys).
//
// Flash form on v_mfma_f32_16x16x4f32 (full fp32 products and sums): one
// workgroup of four waves per 64 queries of a (b, h) block, 64 keys per tile,
// each wave 16 queries.  S^T = K Q^T and O^T = V^T P^T, so every lane owns
// one query (its column of both products) and P goes from the S accumulators
// into the PV operand register for register.
//
// The matrix rows are spread over the lanes so that every LDS read is 16
// bytes and feeds four (PV: CW) MFMAs:
//   * k-slot lg of step (ks, e) of QK holds d = 16 ks + 4 lg + e;
//   * MuNet's K tile is [d][j]: row li of product x is key 4 li + x, so one
//     read of K[d][4 li ..] serves x = 0..3, and lane (li, lg) ends with keys
//     16 lg + 4 e + x of query li in s[x][e].  A textbook tile is [j][d]: one
//     read of K[16 x + li][16 ks + 4 lg ..] serves e = 0..3, and s[x][e] is
//     key 16 x + 4 lg + e;
//   * PV step (x, e) takes s[x][e] as it is: its k-slot lg is that key; row li
//     of product (g, w) is column CW (16 g + li) + w, so one read of CW floats
//     of V's row serves w = 0..CW-1 and each lane stores CW consecutive floats.
// HDP = 16 NG CW is hd rounded up to 32, 64, 96 or 128; Q and K past hd are
// zero.  A ragged last tile's K columns may hold what follows in the buffer
// (masked after the product); V rows past T are zero.
//
// The work is bound by the fp32 matrix rate (64 keys x 16 queries x hd 64:
// 128 MFMAs of 32 cycles beside about 250 VALU instructions), so the tiles
// are single-buffered in LDS with the next tile in registers: 32 KB at hd 64
// leaves room for several workgroups per CU.  Encoder layer of 8 x 250 tokens,
// 8 heads of 64: the block took 382 us with the one-wave-per-query kernel that
// this replaces, 215 us with this one (the other kernels as they were).
//
// Precision: exp(v - m) with m the exact running row max, its base-2 argument
// carried in two floats (the one-float product loses |v - m| 2^-24); row sums in
// doubles, scores and outputs each in two accumulators (even and odd elements
// d, even and odd keys), which halves the variance of a long sum, and one rounding of
// their double sum over the row sum.  Against float64 that is 0.66 to 0.88 of
// the error of the one-wave-per-query kernel, whose exponentials, sum and
// division are doubles, over 2 to 4000 keys, heads of 8 to 128 and scores of 0.25
// to 9; with one accumulator each and fp32 row sums it had been 1.00 to 1.26
// of it.  Time: up to 6% more than that form (8 x 250 keys, 8 heads of 64 19.5
// -> 20.2 us).
#include "mh_common.hpp"
#include "mh_kernels.hpp"

namespace mh {
namespace {

constexpr int KB = 64;

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// exp(x) for x <= 0 (-inf gives 0, NaN stays NaN): 2^(hi + lo) with x log2(e)
// = hi + lo
__device__ __forceinline__ float exp_neg(float x) {
  constexpr float kL = 1.44269502162933349609375f, kLlo = 1.92596303e-8f, kLn2 = 0.693147181f;
  x = x < -200.f ? -200.f : x;
  const float hi = __fmul_rn(x, kL);
  const float lo = __fmaf_rn(x, kLlo, __fmaf_rn(x, kL, -hi));
  const float p = __builtin_amdgcn_exp2f(hi);
  return __fmaf_rn(p, __fmul_rn(lo, kLn2), p);
}

// One causal row again, over keys 0..qi alone, by one wave (see the end of the
// kernel): lane j of a group of 64 keys takes key j's p against the row's max m,
// then lanes d and d + 64 the output columns.
template <bool TXT>
__device__ __forceinline__ void causal_row(const float *q, const float *Kb, const float *Vb, float *dst, int qi, int hd,
                                           long N, float scale, float m, double inv) {
  const int lane = threadIdx.x & 63;
  float a0 = 0.f, a1 = 0.f;
  for (int j0 = 0; j0 <= qi; j0 += 64) {
    const int j = min(j0 + lane, qi);
    float acc = 0.f;
    for (int d = 0; d < hd; ++d) acc = __fmaf_rn(q[d], TXT ? Kb[long(j) * hd + d] : Kb[d * N + j], acc);
    const float p = exp_neg(__fmul_rn(acc, scale) - m);
    for (int k = 0; k < 64 && j0 + k <= qi; ++k) {
      const float pk = __shfl(p, k, 64);
      const float *vr = Vb + long(j0 + k) * hd;
      if (lane < hd) a0 = __fmaf_rn(pk, vr[lane], a0);
      if (lane + 64 < hd) a1 = __fmaf_rn(pk, vr[lane + 64], a1);
    }
  }
  if (lane < hd) dst[lane] = float(double(a0) * inv);
  if (lane + 64 < hd) dst[lane + 64] = float(double(a1) * inv);
}

template <int NG, int CW, bool TXT>
__global__ void __launch_bounds__(256, NG * CW == 2 ? (TXT ? 3 : 4) : NG * CW == 4 ? (TXT ? 2 : 3) : 2)
flash_attn_f32_kernel(const float *__restrict__ Q, const float *__restrict__ K, const float *__restrict__ V,
                      float *__restrict__ O, int B, int H, int T, int hd, int causal, float scale) {
  constexpr int HDP = NG * 16 * CW, KS = HDP / 16, VC = HDP / 4;  // VC: 16-byte chunks of a V row
  constexpr int NL = HDP / 16;                                     // chunks each thread stages of a K or V tile
  typedef float vcw __attribute__((ext_vector_type(CW)));
  __shared__ __attribute__((aligned(16))) float ks_[64 * HDP], vs_[64 * HDP];

  const int BH = B * H, nq = (T + KB - 1) / KB;
  const int lvl = blockIdx.x / BH, bh = blockIdx.x - lvl * BH;
  const int q0 = (causal ? nq - 1 - lvl : lvl) * KB;  // causal: longest rows first
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lg = lane >> 4;
  const long N = long(BH) * T;
  const float *Kb = TXT ? K + long(bh) * T * hd : K + long(bh) * T;
  const float *Vb = V + long(bh) * T * hd;
  const float *kend = K + N * hd;
  const int wrow0 = q0 + wave * 16, i = wrow0 + li;

  f32x4 qf[KS];
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    const int d = 16 * ks + 4 * lg;
    qf[ks] = d < hd ? *reinterpret_cast<const f32x4 *>(Q + (long(bh) * T + min(i, T - 1)) * hd + d)
                    : f32x4{0.f, 0.f, 0.f, 0.f};
  }
  f32x4 o[2][NG][CW];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int w = 0; w < CW; ++w) o[h][g][w] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -3.4028234e38f;
  double l = 0.0;

  // staging: chunk id = tid + 256 n of a tile.  Where 256 chunks are whole rows
  // (kEven) the n-th chunk lies a fixed distance from the first, and so do the
  // rows of MuNet's keys: one pointer for all (an array of them cost 50
  // registers and hd 128 its second wave per SIMD).
  constexpr bool kEven = 256 % VC == 0;
  constexpr int NP = kEven ? 1 : NL, RS = 256 / VC;
  const float *kp[TXT ? NP : 1], *vp[NP];
  int kst[TXT ? NP : 1], vst[NP], vrow[NP];
  bool vin[NP];  // (textbook keys: in the same way)
#pragma unroll
  for (int n = 0; n < NP; ++n) {
    const int id = tid + 256 * n, row = id / VC, c = id % VC;
    vrow[n] = row;
    vin[n] = 4 * c < hd;
    const long voff = long(row) * hd + (vin[n] ? 4 * c : 0);
    vp[n] = Vb + voff;
    vst[n] = row * HDP + 4 * c;
    if constexpr (TXT) {
      kp[n] = Kb + voff;
      kst[n] = row * HDP + 4 * (c ^ (row & 7));
    }
  }
  const int kd = tid >> 4;  // MuNet's keys: row kd + 16 n of the tile
  if constexpr (!TXT) {
    kp[0] = Kb + kd * N + 4 * (tid & 15);
    kst[0] = kd * KB + 4 * (tid & 15);
  }
  // index and row distance of the n-th chunk
  auto pi = [](int n) { return kEven ? 0 : n; };
  auto rs = [](int n) { return kEven ? n * RS : 0; };
  auto kin = [&](int n) { return TXT ? vin[pi(n)] : kd + 16 * n < hd; };
  auto kptr = [&](int n) { return TXT ? kp[pi(n)] + long(rs(n)) * hd : kp[0] + 16 * n * N; };
  auto vptr = [&](int n) { return vp[pi(n)] + long(rs(n)) * hd; };
  auto kdst = [&](int n) { return ks_ + (TXT ? kst[pi(n)] + rs(n) * HDP : kst[0] + 16 * n * KB); };
  auto vdst = [&](int n) { return vs_ + vst[pi(n)] + rs(n) * HDP; };
#pragma unroll
  for (int n = 0; n < NL; ++n)
    if (!kin(n)) *reinterpret_cast<f32x4 *>(kdst(n)) = f32x4{0.f, 0.f, 0.f, 0.f};
  const long kstep = TXT ? long(KB) * hd : KB, vstep = long(KB) * hd;
  f32x4 kr[NL], vr[NL];
  auto gload = [&](int j0) {
    if (j0 + KB <= T) {
#pragma unroll
      for (int n = 0; n < NL; ++n) {
        if constexpr (TXT) kr[n] = *reinterpret_cast<const f32x4 *>(kptr(n));
        else if (kin(n)) kr[n] = *reinterpret_cast<const f32x4_any *>(kptr(n));
        vr[n] = *reinterpret_cast<const f32x4 *>(vptr(n));
      }
    } else {
#pragma unroll
      for (int n = 0; n < NL; ++n) {
        const bool in = j0 + vrow[pi(n)] + rs(n) < T;
        const f32x4 vv = *reinterpret_cast<const f32x4 *>(in ? vptr(n) : Vb);
#pragma unroll
        for (int e = 0; e < 4; ++e) vr[n][e] = in ? vv[e] : 0.f;
        if constexpr (TXT) {
          const f32x4 kv = *reinterpret_cast<const f32x4 *>(in ? kptr(n) : Kb);
#pragma unroll
          for (int e = 0; e < 4; ++e) kr[n][e] = in ? kv[e] : 0.f;
        } else if (kin(n)) {
          const long left = kend - kptr(n);
          if (left >= 4) {
            kr[n] = *reinterpret_cast<const f32x4_any *>(kptr(n));
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) kr[n][e] = left > e ? kptr(n)[e] : 0.f;
          }
        }
      }
    }
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      if constexpr (TXT) kp[n] += kstep;
      vp[n] += vstep;
    }
    if constexpr (!TXT) kp[0] += kstep;
  };

  const int kv_end = causal ? min(T, q0 + KB) : T;
  const int ntiles = (kv_end + KB - 1) / KB;
  gload(0);
  for (int t = 0; t < ntiles; ++t) {
    const int j0 = t * KB;
    __syncthreads();  // the previous tile has been read
#pragma unroll
    for (int n = 0; n < NL; ++n) {
      if (kin(n)) *reinterpret_cast<f32x4 *>(kdst(n)) = kr[n];
      if (vin[pi(n)]) *reinterpret_cast<f32x4 *>(vdst(n)) = vr[n];
    }
    __syncthreads();
    if (t + 1 < ntiles) gload(j0 + KB);

    f32x4 s[4], s1[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) s[x] = s1[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (TXT) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        f32x4 kf[4];
#pragma unroll
        for (int x = 0; x < 4; ++x)
          kf[x] = *reinterpret_cast<const f32x4 *>(ks_ + (16 * x + li) * HDP + 4 * ((4 * ks + lg) ^ (li & 7)));
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            f32x4 &c = (e & 1 ? s1 : s)[x];
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[x][e], qf[ks][e], c, 0, 0, 0);
          }
      }
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4 kf = *reinterpret_cast<const f32x4 *>(ks_ + (16 * ks + 4 * lg + e) * KB + 4 * li);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            f32x4 &c = (e & 1 ? s1 : s)[x];
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[x], qf[ks][e], c, 0, 0, 0);
          }
        }
    }

    const bool edge = j0 + KB > T || (causal && j0 + KB - 1 > wrow0);  // wave-uniform
    const int lim = (causal ? min(T - 1, i) : T - 1) - j0;             // last unmasked key of this query
    float mx = -INFINITY;
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float v = __fmul_rn(__fadd_rn(s[x][e], s1[x][e]), scale);
        if (edge && (TXT ? 16 * x + 4 * lg + e : 16 * lg + 4 * e + x) > lim) v = -INFINITY;
        s[x][e] = v;
        mx = fmaxf(mx, v);
      }
    mx = xor32_max(xor16_max(mx));
    if (__any(mx > m)) {
      const float mnew = fmaxf(m, mx), alpha = exp_neg(m - mnew);
      m = mnew;
      l *= alpha;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int g = 0; g < NG; ++g)
#pragma unroll
          for (int w = 0; w < CW; ++w) o[h][g][w] *= alpha;
    }
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[x][e] = exp_neg(s[x][e] - m);
        l += double(s[x][e]);
      }
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = TXT ? 16 * x + 4 * lg + e : 16 * lg + 4 * e + x;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
          const vcw vf = *reinterpret_cast<const vcw *>(vs_ + row * HDP + CW * (16 * g + li));
#pragma unroll
          for (int w = 0; w < CW; ++w) {
            f32x4 &c = o[(TXT ? e : x) & 1][g][w];  // neighbouring keys apart
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[w], s[x][e], c, 0, 0, 0);
          }
        }
      }
  }

  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  const double inv = 1.0 / l;
  const int b = bh / H, h = bh - b * H;
  float *const out = O + long(b) * T * (long(H) * hd) + long(h) * hd;
  // An infinity or NaN in a masked row of V reaches the queries before it in
  // its tile as 0 * inf: a row with a NaN that its scores do not account for is
  // summed again over its own keys.
  if (causal) {
    bool nan = false;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (CW * (16 * g + 4 * lg + e) < hd)
#pragma unroll
          for (int w = 0; w < CW; ++w) {
            const float v = o[0][g][w][e] + o[1][g][w][e];
            nan |= v != v;
          }
    uint64_t rows = __ballot(nan && i < T && l == l);
    rows |= rows >> 32;
    rows = (rows | rows >> 16) & 0xffff;
    const bool redo = rows >> li & 1;
    for (; rows; rows &= rows - 1) {
      const int row = __builtin_ctzll(rows), qi = wrow0 + row;
      causal_row<TXT>(Q + (long(bh) * T + qi) * hd, Kb, Vb, out + qi * (long(H) * hd), qi, hd, N, scale,
                      __shfl(m, row, 64), __shfl(inv, row, 64));
    }
    if (redo) return;
  }
  if (i >= T) return;
  float *dst = out + i * (long(H) * hd);
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int d = CW * (16 * g + 4 * lg + e);
      if (d >= hd) continue;
      vcw w4;
#pragma unroll
      for (int w = 0; w < CW; ++w) w4[w] = float((double(o[0][g][w][e]) + double(o[1][g][w][e])) * inv);
      *reinterpret_cast<vcw *>(dst + d) = w4;
    }
}

}  // namespace

bool attention_f32_ok(int hd, const void *ctx) { return hd > 0 && hd <= 128 && hd % 4 == 0 && (uintptr_t)ctx % 16 == 0; }

hipError_t attention_f32(const float *q, const float *k, const float *v, float *ctx, int B, int H, int T, int hd,
                         int causal, float scale, int textbook, hipStream_t st) {
  const long items = long((T + KB - 1) / KB) * B * H;
  if (items > 0x7fffffffL || !attention_f32_ok(hd, ctx)) return hipErrorInvalidValue;
  const dim3 grid{unsigned(items)};
#define MH_AF(NG, CW)                                                                                             \
  {                                                                                                               \
    if (textbook) hipLaunchKernelGGL((flash_attn_f32_kernel<NG, CW, true>), grid, dim3(256), 0, st, q, k, v, ctx, \
                                     B, H, T, hd, causal, scale);                                                 \
    else hipLaunchKernelGGL((flash_attn_f32_kernel<NG, CW, false>), grid, dim3(256), 0, st, q, k, v, ctx, B, H,   \
                            T, hd, causal, scale);                                                                \
  }
  if (hd <= 32) MH_AF(1, 2)
  else if (hd <= 64) MH_AF(1, 4)
  else if (hd <= 96) MH_AF(3, 2)
  else MH_AF(2, 4)
#undef MH_AF
  return hipGetLastError();
}

}  // namespace mh
