// Batched dense complex FP64 linear algebra for gfx950: GEMM on FP64 MFMA
// (v_mfma_f64_16x16x4f64), blocked LU with partial pivoting and the two
// triangular solves.  These carry the mode-matching solves and the cascade
// products of the layer-stack solve (rcwa/RCWASolver.cpp:378-614).
#include <algorithm>
#include <cstdlib>

#include "engine.h"

namespace orcwa {

typedef double v4d __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// GEMM: 64x64 output tile per workgroup (4 waves, 32x32 each = 2x2 MFMA
// 16x16 sub-tiles), K staged through LDS 16 at a time (32 spills registers
// and is slower), re/im split into separate LDS planes so each MFMA reads one
// double per lane.  Complex
// products in three real MFMAs (Gauss); the launch bound asks for two
// workgroups per CU, which keeps the 64x64 tile's accumulators in VGPRs
// without spilling.
// MFMA f64 16x16x4 lane layout (measured on gfx950): A[i][k] in lane i+16k,
// B[k][j] in lane j+16k, D[i][j] in lane j+16(i%4), element i/4.
// ---------------------------------------------------------------------------
// TM x TN output tile (TM, TN in {16, 32, 64}): 4 waves in WR x WC, each wave
// (TM/WR) x (TN/WC) = BI x BJ MFMA 16 x 16 blocks.
#ifndef GEMM_KS
#define GEMM_KS 16
#endif
#ifndef GEMM_PAD
#define GEMM_PAD 1
#endif
#ifndef ORCWA_GEMM_XCD
#define ORCWA_GEMM_XCD 1
#endif
#ifndef ORCWA_GEMM_XCD_MIN
#define ORCWA_GEMM_XCD_MIN 64
#endif

template <int TM, int TN>
struct TileShape {
  static constexpr int WR = (TM >= 32 && TN >= 32) ? 2 : (TN == 16 ? 4 : 1);
  static constexpr int WC = 4 / WR;
  static constexpr int BI = TM / (16 * WR), BJ = TN / (16 * WC);
  static constexpr int LA = TM * GEMM_KS / 256, LB = TN * GEMM_KS / 256;  // loads per thread per K step
  static_assert(BI >= 1 && BJ >= 1 && WR * WC == 4, "tile shape");
};

// Tile and batch entry of this workgroup.  Workgroups go to the 8 XCDs
// round-robin by linear id: for large batches give each XCD whole matrices so
// one L2 serves all tiles of a product (a few big products are better spread
// over every XCD).
__device__ __forceinline__ void tile_of_block(int& bx, int& by, int& b) {
  bx = blockIdx.x;
  by = blockIdx.y;
  b = blockIdx.z;
#if ORCWA_GEMM_XCD
  if (gridDim.z >= ORCWA_GEMM_XCD_MIN) {
    const unsigned T = gridDim.x * gridDim.y, Bt = gridDim.z;
    const unsigned w = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const unsigned full = (Bt / 8) * 8 * T;
    unsigned tile;
    if (w < full) {
      const unsigned slot = w / 8;
      tile = slot % T;
      b = (int)((slot / T) * 8 + (w % 8));
    } else {
      const unsigned r = w - full;
      tile = r % T;
      b = (int)((Bt / 8) * 8 + r / T);
    }
    bx = (int)(tile % gridDim.x);
    by = (int)(tile / gridDim.x);
  }
#endif
}

template <bool BETA0, int TM, int TN>
__global__ __launch_bounds__(256, 2) void k_zgemm(
    int M, int N, int K, cd alpha, cd beta,
    const cd* const* __restrict__ Ap, long long offA, long long rsA, long long csA, int conjA,
    const cd* const* __restrict__ Bp, long long offB, long long rsB, long long csB, int conjB,
    cd* const* __restrict__ Cp, long long offC, long long rsC, long long csC, int kup) {
  using TS = TileShape<TM, TN>;
  constexpr int BI = TS::BI, BJ = TS::BJ, LA = TS::LA, LB = TS::LB, WC = TS::WC;
  // rows padded by one double: the k-fast stores (16 lanes down one column)
  // then fall in distinct banks
  __shared__ double sAr[GEMM_KS][TM + GEMM_PAD];
  __shared__ double sAi[GEMM_KS][TM + GEMM_PAD];
  __shared__ double sBr[GEMM_KS][TN + GEMM_PAD];
  __shared__ double sBi[GEMM_KS][TN + GEMM_PAD];

  int bx, by, b;
  tile_of_block(bx, by, b);
  const cd* __restrict__ A = gptr(Ap[b]) + offA;
  const cd* __restrict__ B = gptr(Bp[b]) + offB;
  cd* __restrict__ C = gptr(Cp[b]) + offC;
  const int m0 = bx * TM, n0 = by * TN;
  // op(B) upper triangular from diagonal kup on: its rows past this tile's
  // last column + kup are zero, so the K range ends there
  if (kup >= 0) K = min(K, n0 + TN + kup);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave / WC) * (16 * BI), wn = (wave % WC) * (16 * BJ);
  const double sa = conjA ? -1.0 : 1.0, sb = conjB ? -1.0 : 1.0;

  // global loads run along whichever index of an operand has unit stride
  const bool a_mfast = (rsA == 1), b_kfast = (rsB == 1);
  int amm[LA], akk[LA], bkk[LB], bnn[LB];
  long long pa[LA], pb[LB];
  bool aok[LA], bok[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int e = tid + 256 * j;
    amm[j] = a_mfast ? (e % TM) : (e / GEMM_KS);
    akk[j] = a_mfast ? (e / TM) : (e % GEMM_KS);
    aok[j] = (m0 + amm[j] < M);
    pa[j] = (long long)(m0 + amm[j]) * rsA + (long long)akk[j] * csA;
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    const int e = tid + 256 * j;
    bkk[j] = b_kfast ? (e % GEMM_KS) : (e / TN);
    bnn[j] = b_kfast ? (e / GEMM_KS) : (e % TN);
    bok[j] = (n0 + bnn[j] < N);
    pb[j] = (long long)bkk[j] * rsB + (long long)(n0 + bnn[j]) * csB;
  }
  const long long stepA = GEMM_KS * csA, stepB = GEMM_KS * rsB;
  cd ra[LA], rb[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) ra[j] = (aok[j] && akk[j] < K) ? A[pa[j]] : mk(0.0, 0.0);
#pragma unroll
  for (int j = 0; j < LB; ++j) rb[j] = (bok[j] && bkk[j] < K) ? B[pb[j]] : mk(0.0, 0.0);

  // Gauss form: T1 = ar br, T2 = ai bi, T3 = (ar + ai)(br + bi);
  // re = T1 - T2, im = T3 - T1 - T2 (three real MFMAs per complex product)
  v4d acc1[BI][BJ], acc2[BI][BJ], acc3[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      acc1[i][j] = (v4d){0.0, 0.0, 0.0, 0.0};
      acc2[i][j] = (v4d){0.0, 0.0, 0.0, 0.0};
      acc3[i][j] = (v4d){0.0, 0.0, 0.0, 0.0};
    }

  for (int k0 = 0; k0 < K; k0 += GEMM_KS) {
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      sAr[akk[j]][amm[j]] = ra[j].re;
      sAi[akk[j]][amm[j]] = sa * ra[j].im;
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      sBr[bkk[j]][bnn[j]] = rb[j].re;
      sBi[bkk[j]][bnn[j]] = sb * rb[j].im;
    }
    __syncthreads();
    // next K step in flight while this one runs on the MFMA units
    if (k0 + GEMM_KS < K) {
#pragma unroll
      for (int j = 0; j < LA; ++j) {
        pa[j] += stepA;
        ra[j] = (aok[j] && k0 + GEMM_KS + akk[j] < K) ? A[pa[j]] : mk(0.0, 0.0);
      }
#pragma unroll
      for (int j = 0; j < LB; ++j) {
        pb[j] += stepB;
        rb[j] = (bok[j] && k0 + GEMM_KS + bkk[j] < K) ? B[pb[j]] : mk(0.0, 0.0);
      }
    }
#pragma unroll
    for (int kq = 0; kq < GEMM_KS; kq += 4) {
      const int ka = kq + (lane >> 4);
      double ar[BI], ai[BI], br[BJ], bi[BJ];
#pragma unroll
      for (int i = 0; i < BI; ++i) {
        ar[i] = sAr[ka][wm + 16 * i + (lane & 15)];
        ai[i] = sAi[ka][wm + 16 * i + (lane & 15)];
      }
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        br[j] = sBr[ka][wn + 16 * j + (lane & 15)];
        bi[j] = sBi[ka][wn + 16 * j + (lane & 15)];
      }
      double as[BI], bs[BJ];
#pragma unroll
      for (int i = 0; i < BI; ++i) as[i] = ar[i] + ai[i];
#pragma unroll
      for (int j = 0; j < BJ; ++j) bs[j] = br[j] + bi[j];
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
          acc1[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[i], br[j], acc1[i][j], 0, 0, 0);
          acc2[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[i], bi[j], acc2[i][j], 0, 0, 0);
          acc3[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(as[i], bs[j], acc3[i][j], 0, 0, 0);
        }
    }
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + wm + 16 * i + (lane >> 4) + 4 * r;
        const int gn = n0 + wn + 16 * j + (lane & 15);
        if (gm < M && gn < N) {
          const double t1 = acc1[i][j][r], t2 = acc2[i][j][r];
          cd v = alpha * mk(t1 - t2, acc3[i][j][r] - t1 - t2);
          cd* p = C + gm * rsC + gn * csC;
          if (!BETA0) v += beta * (*p);
          *p = v;
        }
      }
}

// ---------------------------------------------------------------------------
// Reduced-precision complex GEMMs for the cascade (star-product) products,
// same operands, tiles and XCD mapping as k_zgemm.  Products run on FP32 or
// BF16 MFMA with FP32 accumulation inside one K step; each K step's partial
// sums are added into FP64 accumulators, so only the operand rounding and
// the short in-step sums are reduced-precision.
//   FP32:    operands rounded to FP32, MFMA 16x16x4 f32, Gauss three-product
//            complex form (as k_zgemm).
//   BF16xS:  each FP64 operand split into S BF16 slices x = x0 + x1 + ...
//            (x0 = bf16(x), x1 = bf16(x - x0), ...; 8 significant bits each),
//            the slice products with i + j < S kept (S = 2: 3 products, about
//            16 significant bits; S = 3: 6 products, about 24 -- the second
//            level refines the first by the products of the next slice),
//            MFMA 16x16x32 bf16, four-product complex form.
// MFMA f32 16x16x4 lane layout: A[i][k] in lane i + 16k, B[k][j] in lane
// j + 16k, D[i][j] in lane j + 16 (i / 4), element i % 4.  MFMA 16x16x32 bf16:
// A[i][k] in lane i + 16 (k / 8), element k % 8; B[k][j] in lane j + 16 (k / 8),
// element k % 8; D as f32.
// ---------------------------------------------------------------------------
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v8s __attribute__((ext_vector_type(8)));

template <bool BETA0, int TM, int TN>
__global__ __launch_bounds__(256, 2) void k_zgemm_f32(
    int M, int N, int K, cd alpha, cd beta,
    const cd* const* __restrict__ Ap, long long offA, long long rsA, long long csA, int conjA,
    const cd* const* __restrict__ Bp, long long offB, long long rsB, long long csB, int conjB,
    cd* const* __restrict__ Cp, long long offC, long long rsC, long long csC, int kup) {
  constexpr int KS = 16;
  constexpr int WR = (TM >= 32 && TN >= 32) ? 2 : (TN == 16 ? 4 : 1), WC = 4 / WR;
  constexpr int BI = TM / (16 * WR), BJ = TN / (16 * WC);
  constexpr int LA = TM * KS / 256, LB = TN * KS / 256;
  __shared__ float sAr[KS][TM + 1], sAi[KS][TM + 1];
  __shared__ float sBr[KS][TN + 1], sBi[KS][TN + 1];
  int bx, by, b;
  tile_of_block(bx, by, b);
  const cd* __restrict__ A = gptr(Ap[b]) + offA;
  const cd* __restrict__ B = gptr(Bp[b]) + offB;
  cd* __restrict__ C = gptr(Cp[b]) + offC;
  const int m0 = bx * TM, n0 = by * TN;
  // op(B) upper triangular from diagonal kup on: its rows past this tile's
  // last column + kup are zero, so the K range ends there
  if (kup >= 0) K = min(K, n0 + TN + kup);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave / WC) * (16 * BI), wn = (wave % WC) * (16 * BJ);
  const double sa = conjA ? -1.0 : 1.0, sb = conjB ? -1.0 : 1.0;
  const bool a_mfast = (rsA == 1), b_kfast = (rsB == 1);
  int amm[LA], akk[LA], bkk[LB], bnn[LB];
  long long pa[LA], pb[LB];
  bool aok[LA], bok[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int e = tid + 256 * j;
    amm[j] = a_mfast ? (e % TM) : (e / KS);
    akk[j] = a_mfast ? (e / TM) : (e % KS);
    aok[j] = (m0 + amm[j] < M);
    pa[j] = (long long)(m0 + amm[j]) * rsA + (long long)akk[j] * csA;
  }
#pragma unroll
  for (int j = 0; j < LB; ++j) {
    const int e = tid + 256 * j;
    bkk[j] = b_kfast ? (e % KS) : (e / TN);
    bnn[j] = b_kfast ? (e / KS) : (e % TN);
    bok[j] = (n0 + bnn[j] < N);
    pb[j] = (long long)bkk[j] * rsB + (long long)(n0 + bnn[j]) * csB;
  }
  const long long stepA = KS * csA, stepB = KS * rsB;
  cd ra[LA], rb[LB];
#pragma unroll
  for (int j = 0; j < LA; ++j) ra[j] = (aok[j] && akk[j] < K) ? A[pa[j]] : mk(0.0, 0.0);
#pragma unroll
  for (int j = 0; j < LB; ++j) rb[j] = (bok[j] && bkk[j] < K) ? B[pb[j]] : mk(0.0, 0.0);

  double d1[BI][BJ][4], d2[BI][BJ][4], d3[BI][BJ][4];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) d1[i][j][r] = d2[i][j][r] = d3[i][j][r] = 0.0;

  for (int k0 = 0; k0 < K; k0 += KS) {
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      sAr[akk[j]][amm[j]] = (float)ra[j].re;
      sAi[akk[j]][amm[j]] = (float)(sa * ra[j].im);
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      sBr[bkk[j]][bnn[j]] = (float)rb[j].re;
      sBi[bkk[j]][bnn[j]] = (float)(sb * rb[j].im);
    }
    __syncthreads();
    if (k0 + KS < K) {
#pragma unroll
      for (int j = 0; j < LA; ++j) {
        pa[j] += stepA;
        ra[j] = (aok[j] && k0 + KS + akk[j] < K) ? A[pa[j]] : mk(0.0, 0.0);
      }
#pragma unroll
      for (int j = 0; j < LB; ++j) {
        pb[j] += stepB;
        rb[j] = (bok[j] && k0 + KS + bkk[j] < K) ? B[pb[j]] : mk(0.0, 0.0);
      }
    }
    v4f p1[BI][BJ], p2[BI][BJ], p3[BI][BJ];
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        p1[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
        p2[i][j] = p1[i][j];
        p3[i][j] = p1[i][j];
      }
#pragma unroll
    for (int kq = 0; kq < KS; kq += 4) {
      const int ka = kq + (lane >> 4);
      float ar[BI], ai[BI], as[BI], br[BJ], bi[BJ], bs[BJ];
#pragma unroll
      for (int i = 0; i < BI; ++i) {
        ar[i] = sAr[ka][wm + 16 * i + (lane & 15)];
        ai[i] = sAi[ka][wm + 16 * i + (lane & 15)];
        as[i] = ar[i] + ai[i];
      }
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        br[j] = sBr[ka][wn + 16 * j + (lane & 15)];
        bi[j] = sBi[ka][wn + 16 * j + (lane & 15)];
        bs[j] = br[j] + bi[j];
      }
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) {
          p1[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ar[i], br[j], p1[i][j], 0, 0, 0);
          p2[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(ai[i], bi[j], p2[i][j], 0, 0, 0);
          p3[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(as[i], bs[j], p3[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          d1[i][j][r] += (double)p1[i][j][r];
          d2[i][j][r] += (double)p2[i][j][r];
          d3[i][j][r] += (double)p3[i][j][r];
        }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
        const int gn = n0 + wn + 16 * j + (lane & 15);
        if (gm < M && gn < N) {
          const double t1 = d1[i][j][r], t2 = d2[i][j][r];
          cd v = alpha * mk(t1 - t2, d3[i][j][r] - t1 - t2);
          cd* p = C + gm * rsC + gn * csC;
          if (!BETA0) v += beta * (*p);
          *p = v;
        }
      }
}

// x -> S BF16 slices (round to nearest at each level)
template <int S>
__device__ __forceinline__ void bf16_split(double x, __bf16 (&out)[S]) {
#pragma unroll
  for (int q = 0; q < S; ++q) {
    const __bf16 h = (__bf16)(float)x;
    out[q] = h;
    x -= (double)(float)h;
  }
}

__device__ __forceinline__ v8bf bf16_neg(v8bf x) {
  v8s t = __builtin_bit_cast(v8s, x);
  t ^= (v8s)((short)0x8000);
  return __builtin_bit_cast(v8bf, t);
}

template <bool BETA0, int TM, int TN, int S>
__global__ __launch_bounds__(256, 2) void k_zgemm_bf16(
    int M, int N, int K, cd alpha, cd beta,
    const cd* const* __restrict__ Ap, long long offA, long long rsA, long long csA, int conjA,
    const cd* const* __restrict__ Bp, long long offB, long long rsB, long long csB, int conjB,
    cd* const* __restrict__ Cp, long long offC, long long rsC, long long csC, int kup) {
  constexpr int KS = 32, LDK = KS + 8;        // k-fastest rows, padded by 8 (16 bytes)
  constexpr int WR = (TM >= 32 && TN >= 32) ? 2 : (TN == 16 ? 4 : 1), WC = 4 / WR;
  constexpr int BI = TM / (16 * WR), BJ = TN / (16 * WC);
  constexpr int LA = TM * KS / 256, LB = TN * KS / 256;
  // [re/im][slice][row][k]
  __shared__ __attribute__((aligned(16))) __bf16 sA[2][S][TM][LDK];
  __shared__ __attribute__((aligned(16))) __bf16 sB[2][S][TN][LDK];
  int bx, by, b;
  tile_of_block(bx, by, b);
  const cd* __restrict__ A = gptr(Ap[b]) + offA;
  const cd* __restrict__ B = gptr(Bp[b]) + offB;
  cd* __restrict__ C = gptr(Cp[b]) + offC;
  const int m0 = bx * TM, n0 = by * TN;
  // op(B) upper triangular from diagonal kup on: its rows past this tile's
  // last column + kup are zero, so the K range ends there
  if (kup >= 0) K = min(K, n0 + TN + kup);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave / WC) * (16 * BI), wn = (wave % WC) * (16 * BJ);
  const double sa = conjA ? -1.0 : 1.0, sb = conjB ? -1.0 : 1.0;
  const bool a_mfast = (rsA == 1), b_kfast = (rsB == 1);
  // element j of this thread's share of a tile: (row, k) of A and (k, col) of
  // B, recomputed from the thread index (fewer live registers than tables)
  auto a_at = [&](int j, int& mm, int& kk) {
    const int e = tid + 256 * j;
    mm = a_mfast ? (e % TM) : (e / KS);
    kk = a_mfast ? (e / TM) : (e % KS);
  };
  auto b_at = [&](int j, int& kk, int& nn) {
    const int e = tid + 256 * j;
    kk = b_kfast ? (e % KS) : (e / TN);
    nn = b_kfast ? (e / KS) : (e % TN);
  };

  double dre[BI][BJ][4], dim_[BI][BJ][4];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) dre[i][j][r] = dim_[i][j][r] = 0.0;

  for (int k0 = 0; k0 < K; k0 += KS) {
    // no register prefetch (the slices need the registers); the second
    // workgroup on the CU covers the load latency
#pragma unroll
    for (int j = 0; j < LA; ++j) {
      int mm, kk;
      a_at(j, mm, kk);
      const cd v = (m0 + mm < M && k0 + kk < K)
                       ? A[(long long)(m0 + mm) * rsA + (long long)(k0 + kk) * csA]
                       : mk(0.0, 0.0);
      __bf16 xr[S], xi[S];
      bf16_split<S>(v.re, xr);
      bf16_split<S>(sa * v.im, xi);
#pragma unroll
      for (int q = 0; q < S; ++q) {
        sA[0][q][mm][kk] = xr[q];
        sA[1][q][mm][kk] = xi[q];
      }
    }
#pragma unroll
    for (int j = 0; j < LB; ++j) {
      int kk, nn;
      b_at(j, kk, nn);
      const cd v = (n0 + nn < N && k0 + kk < K)
                       ? B[(long long)(k0 + kk) * rsB + (long long)(n0 + nn) * csB]
                       : mk(0.0, 0.0);
      __bf16 xr[S], xi[S];
      bf16_split<S>(v.re, xr);
      bf16_split<S>(sb * v.im, xi);
#pragma unroll
      for (int q = 0; q < S; ++q) {
        sB[0][q][nn][kk] = xr[q];
        sB[1][q][nn][kk] = xi[q];
      }
    }
    __syncthreads();
    const int kl = 8 * (lane >> 4), rl = lane & 15;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int j = 0; j < BJ; ++j) {
        v4f pre = (v4f){0.f, 0.f, 0.f, 0.f}, pim = pre;
#pragma unroll
        for (int qa = 0; qa < S; ++qa) {
          const v8bf a_r = *(const v8bf*)&sA[0][qa][wm + 16 * i + rl][kl];
          const v8bf a_i = *(const v8bf*)&sA[1][qa][wm + 16 * i + rl][kl];
          const v8bf a_in = bf16_neg(a_i);
#pragma unroll
          for (int qb = 0; qb + qa < S; ++qb) {
            const v8bf b_r = *(const v8bf*)&sB[0][qb][wn + 16 * j + rl][kl];
            const v8bf b_i = *(const v8bf*)&sB[1][qb][wn + 16 * j + rl][kl];
            // re += ar br - ai bi, im += ar bi + ai br
            pre = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_r, b_r, pre, 0, 0, 0);
            pre = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_in, b_i, pre, 0, 0, 0);
            pim = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_r, b_i, pim, 0, 0, 0);
            pim = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_i, b_r, pim, 0, 0, 0);
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          dre[i][j][r] += (double)pre[r];
          dim_[i][j][r] += (double)pim[r];
        }
      }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
        const int gn = n0 + wn + 16 * j + (lane & 15);
        if (gm < M && gn < N) {
          cd v = alpha * mk(dre[i][j][r], dim_[i][j][r]);
          cd* p = C + gm * rsC + gn * csC;
          if (!BETA0) v += beta * (*p);
          *p = v;
        }
      }
}

template <int TM, int TN>
static void zgemm_launch(hipStream_t s, int M, int N, int K, cd alpha, const cd* const* A,
                         long long offA, long long rsA, long long csA, int conjA,
                         const cd* const* B, long long offB, long long rsB, long long csB,
                         int conjB, cd beta, cd* const* C, long long offC, long long rsC,
                         long long csC, int batch, int prec, int kup) {
  if (M <= 0 || N <= 0) return;
  dim3 grid((M + TM - 1) / TM, (N + TN - 1) / TN, batch);
  const bool b0 = (beta.re == 0.0 && beta.im == 0.0);
#define ORCWA_GEMM_ARGS                                                                        \
  grid, dim3(256), 0, s, M, N, K, alpha, beta, A, offA, rsA, csA, conjA, B, offB, rsB, csB,   \
      conjB, C, offC, rsC, csC, kup
  switch (prec) {
    case GEMM_FP32:
      if (b0) hipLaunchKernelGGL((k_zgemm_f32<true, TM, TN>), ORCWA_GEMM_ARGS);
      else hipLaunchKernelGGL((k_zgemm_f32<false, TM, TN>), ORCWA_GEMM_ARGS);
      break;
    case GEMM_BF16X3:
      if (b0) hipLaunchKernelGGL((k_zgemm_bf16<true, TM, TN, 2>), ORCWA_GEMM_ARGS);
      else hipLaunchKernelGGL((k_zgemm_bf16<false, TM, TN, 2>), ORCWA_GEMM_ARGS);
      break;
    case GEMM_BF16X6:
      if (b0) hipLaunchKernelGGL((k_zgemm_bf16<true, TM, TN, 3>), ORCWA_GEMM_ARGS);
      else hipLaunchKernelGGL((k_zgemm_bf16<false, TM, TN, 3>), ORCWA_GEMM_ARGS);
      break;
    default:
      if (b0) hipLaunchKernelGGL((k_zgemm<true, TM, TN>), ORCWA_GEMM_ARGS);
      else hipLaunchKernelGGL((k_zgemm<false, TM, TN>), ORCWA_GEMM_ARGS);
  }
#undef ORCWA_GEMM_ARGS
}

// main-block tile of the GEMMs issued by this thread (set_gemm_tile)
static thread_local int g_gemm_tile = GEMM_TILE_64x64;
void set_gemm_tile(int tile) { g_gemm_tile = tile; }
int gemm_tile() { return g_gemm_tile; }

// rows of a strip narrower than 64: the smallest tile height that covers them
template <int TN>
static void zgemm_rows(hipStream_t s, int M, int N, int K, cd alpha, const cd* const* A,
                       long long offA, long long rsA, long long csA, int conjA, const cd* const* B,
                       long long offB, long long rsB, long long csB, int conjB, cd beta,
                       cd* const* C, long long offC, long long rsC, long long csC, int batch,
                       int prec, int kup) {
  // (a 4-wave tile needs at least four 16 x 16 blocks)
  if constexpr (TN == 64) {
    if (M <= 16) {
      zgemm_launch<16, 64>(s, M, N, K, alpha, A, offA, rsA, csA, conjA, B, offB, rsB, csB, conjB,
                           beta, C, offC, rsC, csC, batch, prec, kup);
      return;
    }
  }
  if constexpr (TN >= 32) {
    if (M <= 32) {
      zgemm_launch<32, TN>(s, M, N, K, alpha, A, offA, rsA, csA, conjA, B, offB, rsB, csB, conjB,
                           beta, C, offC, rsC, csC, batch, prec, kup);
      return;
    }
  }
  zgemm_launch<64, TN>(s, M, N, K, alpha, A, offA, rsA, csA, conjA, B, offB, rsB, csB, conjB,
                       beta, C, offC, rsC, csC, batch, prec, kup);
}

void zgemm_batched_prec(int prec, hipStream_t s, int M, int N, int K, cd alpha,
                        const cd* const* A, long long offA, long long rsA, long long csA,
                        int conjA, const cd* const* B, long long offB, long long rsB,
                        long long csB, int conjB, cd beta, cd* const* C, long long offC,
                        long long rsC, long long csC, int batch, int kup) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  // 64 x 64 tiles over the largest multiple-of-64 block, narrower tiles on the
  // remaining row and column strips (n = 450: 448 + a 2-wide strip, instead
  // of a 64-wide tile row and column that are 97 % padding)
  const int M0 = (M / 64) * 64, N0 = (N / 64) * 64, mr = M - M0, nr = N - N0;
  if (M0 > 0 && N0 > 0) {
    // the main block's tile: the autotuned preference of the calling thread's
    // current plan (64 x 64 unless set)
    if (g_gemm_tile == GEMM_TILE_32x64)
      zgemm_launch<32, 64>(s, M0, N0, K, alpha, A, offA, rsA, csA, conjA, B, offB, rsB, csB,
                           conjB, beta, C, offC, rsC, csC, batch, prec, kup);
    else if (g_gemm_tile == GEMM_TILE_64x32)
      zgemm_launch<64, 32>(s, M0, N0, K, alpha, A, offA, rsA, csA, conjA, B, offB, rsB, csB,
                           conjB, beta, C, offC, rsC, csC, batch, prec, kup);
    else
      zgemm_launch<64, 64>(s, M0, N0, K, alpha, A, offA, rsA, csA, conjA, B, offB, rsB, csB,
                           conjB, beta, C, offC, rsC, csC, batch, prec, kup);
  }
  if (mr > 0 && N0 > 0)     // bottom strip
    zgemm_rows<64>(s, mr, N0, K, alpha, A, offA + M0 * rsA, rsA, csA, conjA, B, offB, rsB, csB,
                   conjB, beta, C, offC + M0 * rsC, rsC, csC, batch, prec, kup);
  if (nr > 0) {             // right strip, all rows (corner included)
    const long long oB = offB + N0 * csB, oC = offC + N0 * csC;
    const int kr = kup >= 0 ? kup + N0 : -1;   // the strip's column 0 is column N0
    if (nr <= 16)
      zgemm_rows<16>(s, M, nr, K, alpha, A, offA, rsA, csA, conjA, B, oB, rsB, csB, conjB, beta, C,
                     oC, rsC, csC, batch, prec, kr);
    else if (nr <= 32)
      zgemm_rows<32>(s, M, nr, K, alpha, A, offA, rsA, csA, conjA, B, oB, rsB, csB, conjB, beta, C,
                     oC, rsC, csC, batch, prec, kr);
    else
      zgemm_rows<64>(s, M, nr, K, alpha, A, offA, rsA, csA, conjA, B, oB, rsB, csB, conjB, beta, C,
                     oC, rsC, csC, batch, prec, kr);
  }
}

void zgemm_batched(hipStream_t s, int M, int N, int K, cd alpha,
                   const cd* const* A, long long offA, long long rsA, long long csA, int conjA,
                   const cd* const* B, long long offB, long long rsB, long long csB, int conjB,
                   cd beta, cd* const* C, long long offC, long long rsC, long long csC,
                   int batch) {
  zgemm_batched_prec(GEMM_FP64, s, M, N, K, alpha, A, offA, rsA, csA, conjA, B, offB, rsB, csB,
                     conjB, beta, C, offC, rsC, csC, batch);
}

void zgemm_batched_upper_b(hipStream_t s, int M, int N, int K, cd alpha,
                           const cd* const* A, long long offA, long long rsA, long long csA,
                           int conjA, const cd* const* B, long long offB, long long rsB,
                           long long csB, int conjB, cd beta, cd* const* C, long long offC,
                           long long rsC, long long csC, int batch) {
  zgemm_batched_prec(GEMM_FP64, s, M, N, K, alpha, A, offA, rsA, csA, conjA, B, offB, rsB, csB,
                     conjB, beta, C, offC, rsC, csC, batch, 0);
}

// ---------------------------------------------------------------------------
// LU with partial pivoting, right-looking, panel width NB.
// ---------------------------------------------------------------------------
static constexpr int NB = 32;

// Panel factorisation of columns [k0, k0+nb) over rows [k0, n), one
// workgroup per matrix, in global memory.  Row swaps are applied inside the
// panel only.
__global__ __launch_bounds__(256) void k_getf2_panel(int n, int k0, int nb, cd* const* Ap,
                                                     int* ipiv, int* info, const int* info_map) {
  __shared__ double s_val[256];
  __shared__ int s_idx[256];
  __shared__ cd s_inv;
  __shared__ int s_piv;
  __shared__ cd s_u[NB];
  const int b = blockIdx.x;
  cd* __restrict__ A = gptr(Ap[b]);
  const int tid = threadIdx.x;
  for (int j = 0; j < nb; ++j) {
    const int c = k0 + j;
    // pivot search: max cabs1 over rows c..n-1 of column c (first index wins ties)
    double best = -1.0;
    int bi = c;
    for (int i = c + tid; i < n; i += 256) {
      double v = cabs1(A[i + (long long)c * n]);
      if (v > best) { best = v; bi = i; }
    }
    s_val[tid] = best;
    s_idx[tid] = bi;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
      if (tid < st) {
        double o = s_val[tid + st];
        int oi = s_idx[tid + st];
        if (o > s_val[tid] || (o == s_val[tid] && oi < s_idx[tid])) {
          s_val[tid] = o;
          s_idx[tid] = oi;
        }
      }
      __syncthreads();
    }
    if (tid == 0) {
      int p = s_idx[0];
      s_piv = p;
      ipiv[(long long)b * n + c] = p;
      cd pv = A[p + (long long)c * n];
      if (pv.re == 0.0 && pv.im == 0.0) {
        atomicOr(&info[info_map ? info_map[b] : b], ORCWA_STATUS_SINGULAR);
        s_inv = mk(0.0, 0.0);
      } else {
        s_inv = cinv(pv);
      }
    }
    __syncthreads();
    const int p = s_piv;
    if (p != c) {
      for (int jj = tid; jj < nb; jj += 256) {
        const long long col = (long long)(k0 + jj) * n;
        cd t = A[c + col];
        A[c + col] = A[p + col];
        A[p + col] = t;
      }
    }
    __syncthreads();
    // the pivot row's entries right of column c, staged for every thread
    const int ncol = nb - j - 1;
    for (int jj = tid; jj < ncol; jj += 256) s_u[jj] = A[c + (long long)(c + 1 + jj) * n];
    __syncthreads();
    // scale column c below the pivot and apply the rank-1 update, one row per
    // thread (its multiplier read once)
    const cd inv = s_inv;
    for (int i = c + 1 + tid; i < n; i += 256) {
      const cd l = A[i + (long long)c * n] * inv;
      A[i + (long long)c * n] = l;
      for (int jj = 0; jj < ncol; ++jj) A[i + (long long)(c + 1 + jj) * n] -= l * s_u[jj];
    }
    __syncthreads();
  }
}

// The same panel factorization held in registers, for panels of at most
// GF_T rows: thread t owns one row of the nb <= NB panel columns.  The rows do
// not move: a thread keeps the position that the interchanges give its row and
// stores it there at the end.  Per column one barrier: every wave reduces its
// pivot candidate with DPP moves (no LDS round trips) and puts that row in LDS
// beside the others', so that after the barrier each thread finds the winner
// and reads its row from the wave's buffer.  (Rows exchanged through LDS, two
// barriers and shuffled reductions took 2.4 us a column at n = 450, this 1.5.)
// The column steps are instantiated one by one (template recursion) so that
// every register index is a constant.
constexpr int GF_T = 512, GF_T2 = 1024, NB2 = 16;

// T threads (rows), WB panel columns: 512 x 32, or 1024 x 16 (a thread's row
// then fits the 128 registers it has)
template <int T, int WB>
struct GetrfRegState {
  cd (*s_row)[T / 64][WB];       // [parity][wave]: the wave's candidate row
  double (*s_wv)[T / 64];
  int (*s_wp)[T / 64];
  int n, k0, nb, lane, wave, b;
  int pos;                          // position of this thread's row (n: no row)
  int* ipiv;
  int* info;
  const int* info_map;
};

// maximum over the first 16 lanes, in every lane
__device__ __forceinline__ double dpp_row_max(double v) {
  return lane_value(dpp_row_reduce_max(v), 15);
}

template <int J, int T, int WB>
__device__ __forceinline__ void getrf_reg_step(GetrfRegState<T, WB>& S, cd (&a)[WB]) {
  if constexpr (J < WB) {
    if (J < S.nb) {
      const int c = S.k0 + J, par = J & 1;
      // the wave's pivot: max cabs1 over its rows at positions c..n-1 (-1: it
      // has none; a NaN counts as 0), the lowest position on ties
      const bool in = S.pos >= c && S.pos < S.n;
      const double v0 = cabs1(a[J]);
      const double v = in ? (v0 == v0 ? v0 : 0.0) : -1.0;
      const double best = wave_max(v);
      if (best >= 0.0) {
        unsigned long long who = __ballot(v == best);
        int bl = __ffsll(who) - 1, bp = __builtin_amdgcn_readlane(S.pos, bl);
        for (who &= who - 1; who; who &= who - 1) {
          const int l = __ffsll(who) - 1, p = __builtin_amdgcn_readlane(S.pos, l);
          if (p < bp) {
            bp = p;
            bl = l;
          }
        }
        if (S.lane == bl) {
          S.s_wp[par][S.wave] = bp;
#pragma unroll
          for (int jj = J; jj < WB; ++jj) lds_st(&S.s_row[par][S.wave][jj], a[jj]);
        }
      }
      if (S.lane == 0) S.s_wv[par][S.wave] = best;
      __syncthreads();
      // the winner among the waves' candidates, lane w holding wave w's
      const double cv = S.lane < T / 64 ? S.s_wv[par][S.lane] : -1.0;
      const int cp = S.s_wp[par][S.lane & (T / 64 - 1)];
      const double top = dpp_row_max(cv);
      unsigned long long won = __ballot(cv == top);
      int bw = __ffsll(won) - 1, bi = __builtin_amdgcn_readlane(cp, bw);
      for (won &= won - 1; won; won &= won - 1) {
        const int w = __ffsll(won) - 1, q = __builtin_amdgcn_readlane(cp, w);
        if (q < bi) {
          bi = q;
          bw = w;
        }
      }
      const cd* prow = S.s_row[par][bw];
      const cd pv = lds_ld(&prow[J]);
      const bool zero = (pv.re == 0.0 && pv.im == 0.0);
      if (threadIdx.x == 0) {
        S.ipiv[(long long)S.b * S.n + c] = bi;
        if (zero) atomicOr(&S.info[S.info_map ? S.info_map[S.b] : S.b], ORCWA_STATUS_SINGULAR);
      }
      const cd inv = cinv(pv);
      // rows c and bi trade positions
      S.pos = S.pos == bi ? c : (S.pos == c ? bi : S.pos);
      if (S.pos > c && S.pos < S.n) {
        a[J] = zero ? mk(0.0, 0.0) : a[J] * inv;
#pragma unroll
        for (int jj = J + 1; jj < WB; ++jj) a[jj] = cfnma(a[jj], a[J], lds_ld(&prow[jj]));
      }
      // (the candidates alternate by column parity: the next column writes the
      // other half, and the one after writes this half only after every thread
      // has passed the next column's barrier)
      getrf_reg_step<J + 1, T, WB>(S, a);
    }
  }
}

template <int T, int WB>
__global__ __launch_bounds__(T) void k_getf2_reg(int n, int k0, int nb, cd* const* Ap,
                                                    int* ipiv, int* info, const int* info_map) {
  __shared__ alignas(16) cd s_row[2][T / 64][WB];
  __shared__ double s_wv[2][T / 64];
  __shared__ int s_wp[2][T / 64];
  GetrfRegState<T, WB> S;
  S.s_row = s_row;
  S.s_wv = s_wv;
  S.s_wp = s_wp;
  S.n = n;
  S.k0 = k0;
  S.nb = nb;
  S.b = blockIdx.x;
  S.lane = threadIdx.x & 63;
  S.wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = k0 + threadIdx.x;
  const bool live = r < n;
  S.pos = live ? r : n;
  S.ipiv = ipiv;
  S.info = info;
  S.info_map = info_map;
  cd* __restrict__ A = gptr(Ap[S.b]);
  cd a[WB];
#pragma unroll
  for (int j = 0; j < WB; ++j)
    a[j] = (live && j < nb) ? A[r + (long long)(k0 + j) * n] : mk(0.0, 0.0);
  getrf_reg_step<0, T, WB>(S, a);
#pragma unroll
  for (int j = 0; j < WB; ++j)
    if (live && j < nb) A[S.pos + (long long)(k0 + j) * n] = a[j];
}

// Apply row swaps ipiv[k0..k0+nb) (in order) to columns [c0, c1) of an
// n-row matrix with leading dimension n (one thread per column).
__global__ void k_laswp(int n, int ncols_total, int k0, int nb, int c0, int c1, cd* const* Ap,
                        const int* ipiv) {
  const int b = blockIdx.y;
  const int col = c0 + blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= c1 || col >= ncols_total) return;
  cd* __restrict__ A = gptr(Ap[b]) + (long long)col * n;
  const int* pv = ipiv + (long long)b * n;
  for (int j = 0; j < nb; ++j) {
    const int r = k0 + j;
    const int p = pv[r];
    if (p != r) {
      cd t = A[r];
      A[r] = A[p];
      A[p] = t;
    }
  }
}

// The interchanges of one panel (rows k0..k0+nb-1 with their pivot rows,
// applied in order) as a single gather on the columns left and right of it: one
// wave composes them on the <= 2 nb rows they touch (lane s holds row R; after
// the swaps it holds the original row of lane src), in registers (in LDS by one
// thread it took most of the kernel's 21 us); the workgroup then stages those
// rows of its 16 columns in LDS and writes back the moved ones.
constexpr int LASWP_MAXS = 64, LASWP_NC = 16;
static_assert(2 * NB <= LASWP_MAXS, "one lane per touched row");
__global__ __launch_bounds__(256) void k_laswp_panel(int n, int k0, int nb, cd* const* Ap,
                                                     const int* ipiv) {
  __shared__ int s_R[LASWP_MAXS], s_src[LASWP_MAXS];
  __shared__ int s_ns;
  __shared__ alignas(16) cd tile[LASWP_MAXS][LASWP_NC];
  const int b = blockIdx.y;
  const int* pv = ipiv + (long long)b * n;
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const int piv = lane < nb ? pv[k0 + lane] : -1;
    int R = lane < nb ? k0 + lane : -1, src = lane, ns = nb;
    for (int j = 0; j < nb; ++j) {
      const int p = __builtin_amdgcn_readlane(piv, j);
      const unsigned long long m = __ballot(R == p);
      int sp = ns;
      if (m) sp = __ffsll(m) - 1;
      else {
        if (lane == ns) R = p;
        ++ns;
      }
      const int sj = __builtin_amdgcn_readlane(src, j), ss = __builtin_amdgcn_readlane(src, sp);
      if (lane == j) src = ss;
      if (lane == sp) src = sj;
    }
    s_R[lane] = R;
    s_src[lane] = src;
    if (lane == 0) s_ns = ns;
  }
  __syncthreads();
  const int ns = s_ns;
  const int c = threadIdx.x % LASWP_NC, sg = threadIdx.x / LASWP_NC;
  const int idx = blockIdx.x * LASWP_NC + c, col = idx < k0 ? idx : idx + nb;
  cd* __restrict__ A = gptr(Ap[b]) + (long long)col * n;
  if (col < n)
    for (int t = sg; t < ns; t += 256 / LASWP_NC) lds_st(&tile[t][c], A[s_R[t]]);
  __syncthreads();
  if (col < n)
    for (int t = sg; t < ns; t += 256 / LASWP_NC)
      if (s_src[t] != t) A[s_R[t]] = lds_ld(&tile[s_src[t]][c]);
}

// perm[r] = the original row that ends in row r after all n interchanges (one
// wave per matrix, up to PERM_MB matrices per workgroup, in LDS)
constexpr int PERM_MB = 4;
__global__ __launch_bounds__(64 * PERM_MB) void k_ipiv_to_perm(int n, const int* ipiv, int* perm,
                                                               int batch) {
  extern __shared__ int sp[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int b = blockIdx.x * (blockDim.x >> 6) + wave;
  if (b >= batch) return;
  int* q = sp + (long long)wave * n;
  const int* pv = ipiv + (long long)b * n;
  for (int r = lane; r < n; r += 64) q[r] = r;
  wave_fence();
  for (int k0 = 0; k0 < n; k0 += 64)
    compose_swaps(k0, min(64, n - k0), k0 + lane < n ? pv[k0 + lane] : 0, q);
  wave_fence();
  int* out = perm + (long long)b * n;
  for (int r = lane; r < n; r += 64) out[r] = q[r];
}

// B <- P^T B as a gather through LDS: ncw (<= PERM_NC) columns per workgroup
constexpr int PERM_NC = 4;
__global__ __launch_bounds__(256) void k_apply_perm(int n, int nrhs, int ncw, const int* perm,
                                                    cd* const* Bp) {
  extern __shared__ cd X[];   // [ncw][n]
  const int b = blockIdx.y;
  const int c0 = blockIdx.x * ncw;
  cd* __restrict__ B = gptr(Bp[b]);
  const int* pm = perm + (long long)b * n;
  const int nc = min(ncw, nrhs - c0);
  for (int e = threadIdx.x; e < nc * n; e += 256) {
    const int c = e / n, r = e % n;
    X[c * n + r] = B[r + (long long)(c0 + c) * n];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < nc * n; e += 256) {
    const int c = e / n, r = e % n;
    B[r + (long long)(c0 + c) * n] = X[c * n + pm[r]];
  }
}

// X <- L11^{-1} X for the nb x ncols block of rows [k0, k0+nb), columns
// [c0, c0+ncols) of X (ld = n), L11 unit lower at (k0,k0) of L (ld = n); with
// UNIT_LOWER false, U11^{-1} X for the upper, non-unit block.  One column per
// thread; the block moves between HBM and registers through LDS in slabs of
// TR_SLAB rows, so that consecutive threads touch consecutive rows of a
// column (a column's 32-row segment is 512 contiguous bytes; read directly,
// the lanes of a wave would each touch another column).  All slabs are loaded
// before the first is staged: one memory latency instead of four.
// 256 columns a workgroup, also where few workgroups result: 64 took as long or
// longer from 1 to 1024 matrices (four LUs and solves of a cascade, ms by 256 / 64:
// n = 98, 1 matrix 2.14 / 2.16, 128: 2.50 / 2.61; n = 450, 1: 13.1 / 13.2, 256:
// 62.7 / 65.0; n = 722, 1: 23.7 / 24.0, 1024: 851 / 863).
constexpr int TR_SLAB = 8, TR_COLS = 256;
template <bool UNIT_LOWER>
__global__ __launch_bounds__(TR_COLS) void k_trsm_block(int n, int k0, int nb, int c0, int ncols,
                                                        const cd* const* Lp, cd* const* Xp) {
  constexpr int TPB = TR_COLS;
  __shared__ alignas(16) cd sT[NB][NB];
  __shared__ alignas(16) cd sX[TPB][TR_SLAB + 1];
  const int b = blockIdx.y;
  const cd* __restrict__ Lm = gptr(Lp[b]);
  cd* __restrict__ X = gptr(Xp[b]);
  const int tid = threadIdx.x;
  const int cb = blockIdx.x * TPB;   // this workgroup's first column (from c0)
  const int rr0 = tid % TR_SLAB;
  cd r[NB];
#pragma unroll
  for (int e = 0; e < NB; ++e) {
    const int cc = tid / TR_SLAB + (TPB / TR_SLAB) * (e % TR_SLAB), row = TR_SLAB * (e / TR_SLAB) + rr0;
    r[e] = (cb + cc < ncols && row < nb) ? X[(long long)(c0 + cb + cc) * n + k0 + row]
                                         : mk(0.0, 0.0);
  }
  // (zero outside nb x nb, so the unrolled products below need no guard)
  for (int e = tid; e < NB * NB; e += TPB) {
    const int i = e % NB, j = e / NB;
    sT[i][j] = (i < nb && j < nb) ? Lm[(k0 + i) + (long long)(k0 + j) * n] : mk(0.0, 0.0);
  }
#pragma unroll
  for (int q = 0; q < NB / TR_SLAB; ++q) {
#pragma unroll
    for (int i = 0; i < TR_SLAB; ++i)
      lds_st(&sX[tid / TR_SLAB + (TPB / TR_SLAB) * i][rr0], r[TR_SLAB * q + i]);
    __syncthreads();
#pragma unroll
    for (int rr = 0; rr < TR_SLAB; ++rr) r[TR_SLAB * q + rr] = lds_ld(&sX[tid][rr]);
    __syncthreads();
  }
  // (columns past ncols hold zeros and are not stored)
  if (UNIT_LOWER) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (i < nb) {
#pragma unroll
        for (int k = 0; k < NB; ++k)
          if (k < i) r[i] = cfnma(r[i], lds_ld(&sT[i][k]), r[k]);
      }
    }
  } else {  // upper, non-unit
#pragma unroll
    for (int ii = NB - 1; ii >= 0; --ii) {
      if (ii < nb) {
#pragma unroll
        for (int k = ii + 1; k < NB; ++k) r[ii] = cfnma(r[ii], lds_ld(&sT[ii][k]), r[k]);
        cd d = sT[ii][ii];
        if (d.re != 0.0 || d.im != 0.0) r[ii] = cdiv(r[ii], d);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < NB / TR_SLAB; ++q) {
#pragma unroll
    for (int rr = 0; rr < TR_SLAB; ++rr) lds_st(&sX[tid][rr], r[TR_SLAB * q + rr]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < TR_SLAB; ++i) {
      const int cc = tid / TR_SLAB + (TPB / TR_SLAB) * i, row = TR_SLAB * q + rr0;
      if (cb + cc < ncols && row < nb)
        X[(long long)(c0 + cb + cc) * n + k0 + row] = lds_ld(&sX[cc][rr0]);
    }
    __syncthreads();
  }
}

template <bool UNIT_LOWER>
static void trsm_block(hipStream_t s, int n, int k0, int nb, int c0, int ncols,
                       const cd* const* L, cd* const* X, int batch) {
  hipLaunchKernelGGL((k_trsm_block<UNIT_LOWER>), dim3((ncols + TR_COLS - 1) / TR_COLS, batch),
                     dim3(TR_COLS), 0, s, n, k0, nb, c0, ncols, L, X);
}

void zgetrf_batched(hipStream_t s, int n, cd* const* A, int* ipiv, int* info,
                    const int* info_map, int batch) {
  if (n <= 0 || batch <= 0) return;
  const cd* const* Ac = (const cd* const*)A;
  for (int k0 = 0, nb; k0 < n; k0 += nb) {
    const int rows = n - k0;
    // Panels of 513 to 1024 rows are kept in registers, 16 columns at a time:
    // four LUs and their solves of a cascade, ms so / by k_getf2_panel: n = 578, 1
    // matrix 18.0 / 19.4, 64: 41.8 / 41.8, 256: 120.6 / 118.8; n = 798, 1: 28.5 /
    // 33.4, 32: 59.1 / 60.7, 64: 93.8 / 90.2, 256: 300 / 277; n = 1058, 1: 43.2 /
    // 52.8, 256: 617 / 571.  Many matrices pay for twice the passes over the
    // trailing part, but there the eigen solves take most of the time; and by the
    // row count alone, because a matrix has to get the same factors in any batch.
    const bool half = rows > GF_T && rows <= GF_T2;
    nb = std::min(half ? NB2 : NB, rows);
    if (rows <= GF_T)
      hipLaunchKernelGGL((k_getf2_reg<GF_T, NB>), dim3(batch), dim3(GF_T), 0, s, n, k0, nb, A, ipiv,
                         info, info_map);
    else if (half)
      hipLaunchKernelGGL((k_getf2_reg<GF_T2, NB2>), dim3(batch), dim3(GF_T2), 0, s, n, k0, nb, A,
                         ipiv, info, info_map);
    else
      hipLaunchKernelGGL(k_getf2_panel, dim3(batch), dim3(256), 0, s, n, k0, nb, A, ipiv, info,
                         info_map);
    // swaps on the columns left and right of the panel
    if (n > nb)
      hipLaunchKernelGGL(k_laswp_panel, dim3((n - nb + LASWP_NC - 1) / LASWP_NC, batch), dim3(256),
                         0, s, n, k0, nb, A, (const int*)ipiv);
    const int rest = n - k0 - nb;
    if (rest > 0) {
      trsm_block<true>(s, n, k0, nb, k0 + nb, rest, Ac, A, batch);
      // A22 -= L21 * U12
      zgemm_batched(s, rest, rest, nb, mk(-1.0, 0.0), Ac, (long long)(k0 + nb) + (long long)k0 * n,
                    1, n, 0, Ac, (long long)k0 + (long long)(k0 + nb) * n, 1, n, 0, mk(1.0, 0.0), A,
                    (long long)(k0 + nb) + (long long)(k0 + nb) * n, 1, n, batch);
    }
  }
}

// Two-level blocking: 32-row triangular blocks inside 128-row outer blocks;
// the updates inside an outer block touch its 128 rows only, and the rows
// outside get one rank-128 GEMM update per outer block, so the right-hand
// side streams through HBM n/128 times per sweep instead of n/32.
static constexpr int OB = 128;

void zgetrs_batched(hipStream_t s, int n, int nrhs, const cd* const* LU, const int* ipiv,
                    cd* const* B, int batch, int* perm_ws) {
  if (n <= 0 || nrhs <= 0 || batch <= 0) return;
  const cd* const* Bc = (const cd* const*)B;
  const cd one = mk(1.0, 0.0), mone = mk(-1.0, 0.0);
  // all row interchanges: composed once per matrix and applied as a gather
  // (when a workspace of batch x n ints is given), else swap by swap; the
  // matrices per workgroup (composition) and columns per workgroup (gather)
  // shrink with n so that each stays within 64 KB of LDS
  constexpr size_t kPermLds = 64 * 1024;
  const int mb = (int)std::min<size_t>(PERM_MB, kPermLds / ((size_t)n * sizeof(int)));
  const int ncw = (int)std::min<size_t>(PERM_NC, kPermLds / ((size_t)n * sizeof(cd)));
  if (perm_ws && mb >= 1 && ncw >= 1) {
    hipLaunchKernelGGL(k_ipiv_to_perm, dim3((batch + mb - 1) / mb), dim3(64 * mb),
                       (size_t)mb * n * sizeof(int), s, n, ipiv, perm_ws, batch);
    hipLaunchKernelGGL(k_apply_perm, dim3((nrhs + ncw - 1) / ncw, batch), dim3(256),
                       (size_t)ncw * n * sizeof(cd), s, n, nrhs, ncw, (const int*)perm_ws, B);
  } else {
    hipLaunchKernelGGL(k_laswp, dim3((nrhs + 127) / 128, batch), dim3(128), 0, s, n, nrhs, 0, n, 0,
                       nrhs, B, ipiv);
  }
  // forward substitution with unit L
  for (int o0 = 0; o0 < n; o0 += OB) {
    const int oe = std::min(n, o0 + OB);
    for (int k0 = o0; k0 < oe; k0 += NB) {
      const int nb = std::min(NB, oe - k0);
      trsm_block<true>(s, n, k0, nb, 0, nrhs, LU, B, batch);
      const int rin = oe - k0 - nb;
      if (rin > 0)
        zgemm_batched(s, rin, nrhs, nb, mone, LU, (long long)(k0 + nb) + (long long)k0 * n, 1, n,
                      0, Bc, (long long)k0, 1, n, 0, one, B, (long long)(k0 + nb), 1, n, batch);
    }
    if (oe < n)
      zgemm_batched(s, n - oe, nrhs, oe - o0, mone, LU, (long long)oe + (long long)o0 * n, 1, n, 0,
                    Bc, (long long)o0, 1, n, 0, one, B, (long long)oe, 1, n, batch);
  }
  // backward substitution with U
  const int nob = (n + OB - 1) / OB;
  for (int ob = nob - 1; ob >= 0; --ob) {
    const int o0 = ob * OB, oe = std::min(n, o0 + OB);
    const int nib = (oe - o0 + NB - 1) / NB;
    for (int ib = nib - 1; ib >= 0; --ib) {
      const int k0 = o0 + ib * NB, nb = std::min(NB, oe - k0);
      trsm_block<false>(s, n, k0, nb, 0, nrhs, LU, B, batch);
      if (k0 > o0)
        zgemm_batched(s, k0 - o0, nrhs, nb, mone, LU, (long long)o0 + (long long)k0 * n, 1, n, 0,
                      Bc, (long long)k0, 1, n, 0, one, B, (long long)o0, 1, n, batch);
    }
    if (o0 > 0)
      zgemm_batched(s, o0, nrhs, oe - o0, mone, LU, (long long)o0 * n, 1, n, 0, Bc, (long long)o0,
                    1, n, 0, one, B, 0, 1, n, batch);
  }
}

// ---------------------------------------------------------------------------
// elementwise
// ---------------------------------------------------------------------------
__global__ void k_set_identity(int n, cd* const* Ap) {
  cd* A = gptr(Ap[blockIdx.y]);
  const long long nn = (long long)n * n;
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < nn;
       e += (long long)gridDim.x * blockDim.x) {
    const long long i = e % n, j = e / n;
    A[e] = (i == j) ? mk(1.0, 0.0) : mk(0.0, 0.0);
  }
}

__global__ void k_axpby(long long count, cd a, const cd* const* Ap, cd bb, const cd* const* Bp,
                        cd* const* Cp) {
  const cd* A = gptr(Ap[blockIdx.y]);
  const cd* B = gptr(Bp[blockIdx.y]);
  cd* C = gptr(Cp[blockIdx.y]);
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < count;
       e += (long long)gridDim.x * blockDim.x)
    C[e] = a * A[e] + bb * B[e];
}

__global__ void k_copy(long long count, const cd* const* Ap, cd* const* Bp) {
  const cd* A = gptr(Ap[blockIdx.y]);
  cd* B = gptr(Bp[blockIdx.y]);
  for (long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x; e < count;
       e += (long long)gridDim.x * blockDim.x)
    B[e] = A[e];
}

static inline int grid1d(long long count) {
  long long g = (count + 255) / 256;
  return (int)(g > 1024 ? 1024 : (g < 1 ? 1 : g));
}

void set_identity_batched(hipStream_t s, int n, cd* const* A, int batch) {
  if (batch <= 0) return;
  hipLaunchKernelGGL(k_set_identity, dim3(grid1d((long long)n * n), batch), dim3(256), 0, s, n, A);
}

void axpby_batched(hipStream_t s, int n, cd a, const cd* const* A, cd b, const cd* const* B,
                   cd* const* C, int batch) {
  if (batch <= 0) return;
  const long long cnt = (long long)n * n;
  hipLaunchKernelGGL(k_axpby, dim3(grid1d(cnt), batch), dim3(256), 0, s, cnt, a, A, b, B, C);
}

void copy_batched(hipStream_t s, long long count, const cd* const* A, cd* const* B, int batch) {
  if (batch <= 0) return;
  hipLaunchKernelGGL(k_copy, dim3(grid1d(count), batch), dim3(256), 0, s, count, A, B);
}

}  // namespace orcwa
