// Small f32 GEMM on the FMA units: C = alpha op(A) op(B) + beta C (the fp32
// model's projections, gemm_f32.hip; the training products too small for
// the matrix cores, train.hip).
//
// One wave per workgroup owns an 8R x 8R output tile, lane (ty, tx) the outputs
// of rows ty + 8 i and columns tx + 8 j. Both operand tiles sit in LDS as rows of
// KT + 4 floats along k (the pad puts the eight rows a 16-byte read touches in
// different banks; an operand stored across k is transposed on the way), and the
// next KT columns' loads are in flight in registers during the current ones'
// FMAs; with one wave there is no barrier to wait at. An output is one serial
// chain of FMAs over k in order, whatever the tile, so the tile size changes no
// bits. At the sizes it is used for that chain and the launch are the bound, so
// the tile is as small as fills the chip. Against one 64 x 64 tile per 256 threads:
// M 32: 768 x 256 19.9 -> 4.1 us, 256 x 1024 70.7 -> 10.8, 4096 x 256 20.2 -> 5.5;
// 64 x 1536 x 512 with B across k 53 -> 8.9, 204 x 768 x 32768 5330 -> 870.
#pragma once

#include "common.hpp"

namespace sm {
namespace {

typedef float f32x4w __attribute__((ext_vector_type(4)));

// One operand's tile: rows r0 .. r0 + 8R of op(X), KT columns from k0. KC: element
// (r, k) at X[r * ld + k], else X[k * ld + r]; vec: its 16-byte loads are aligned
// and whole (R and K limits multiples of 4 along the contiguous dimension).
template <bool KC, int R, int KT>
struct WaveTile {
  static constexpr int ROWS = 8 * R, RS = KT + 4, NL = ROWS * KT / 256;
  const float* X;
  int64_t ld;
  int r0, rows, K, vec;
  f32x4w v[NL];
  __device__ inline void load(int k0, int l) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = i * 64 + l;
      const int r = r0 + (KC ? c / (KT / 4) : 4 * (c % (2 * R)));
      const int k = k0 + (KC ? 4 * (c % (KT / 4)) : c / (2 * R));
      f32x4w t = {0.f, 0.f, 0.f, 0.f};
      if (r < rows && k < K) {
        const float* q = X + (KC ? (int64_t)r * ld + k : (int64_t)k * ld + r);
        if (vec) {
          t = *reinterpret_cast<const f32x4w*>(q);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (KC ? k + e < K : r + e < rows) t[e] = q[e];
        }
      }
      v[i] = t;
    }
  }
  __device__ inline void store(float* lds, int l) const {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = i * 64 + l;
      if constexpr (KC) {
        *reinterpret_cast<f32x4w*>(lds + c / (KT / 4) * RS + 4 * (c % (KT / 4))) = v[i];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) lds[(4 * (c % (2 * R)) + e) * RS + c / (2 * R)] = v[i][e];
      }
    }
  }
};

template <bool TA, bool TB, int R, int KT>
__global__ __launch_bounds__(64) void gemm_wave_kernel(const float* __restrict__ A, int64_t lda,
                                                       const float* __restrict__ B, int64_t ldb,
                                                       float* __restrict__ C, int64_t ldc, int M,
                                                       int N, int K, float alpha, float beta,
                                                       int vec_a, int vec_b, int ntn) {
  using TileA = WaveTile<!TA, R, KT>;
  using TileB = WaveTile<TB, R, KT>;
  constexpr int ROWS = 8 * R, RS = KT + 4;
  __shared__ __attribute__((aligned(16))) float as[ROWS * RS];
  __shared__ __attribute__((aligned(16))) float bs[ROWS * RS];
  const int l = threadIdx.x, tx = l % 8, ty = l / 8;
  const int m0 = (int)(blockIdx.x / ntn) * ROWS, n0 = (int)(blockIdx.x % ntn) * ROWS;
  TileA ta{A, lda, m0, M, K, vec_a};
  TileB tb{B, ldb, n0, N, K, vec_b};
  float acc[R][R] = {};
  ta.load(0, l);
  tb.load(0, l);
  for (int k0 = 0; k0 < K; k0 += KT) {
    ta.store(as, l);
    tb.store(bs, l);
    __syncthreads();
    if (k0 + KT < K) {
      ta.load(k0 + KT, l);
      tb.load(k0 + KT, l);
    }
#pragma unroll 4
    for (int k = 0; k < KT; k += 4) {
      f32x4w a[R], b[R];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        a[i] = *reinterpret_cast<const f32x4w*>(as + (ty + 8 * i) * RS + k);
        b[i] = *reinterpret_cast<const f32x4w*>(bs + (tx + 8 * i) * RS + k);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int j = 0; j < R; ++j) acc[i][j] = fmaf(a[i][e], b[j][e], acc[i][j]);
    }
    __syncthreads();  // the tiles are read before the next ones are written
  }
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int gm = m0 + ty + 8 * i;
    if (gm >= M) continue;
#pragma unroll
    for (int j = 0; j < R; ++j) {
      const int gn = n0 + tx + 8 * j;
      if (gn >= N) continue;
      float* cp = C + (int64_t)gm * ldc + gn;
      *cp = alpha * acc[i][j] + (beta != 0.f ? beta * *cp : 0.f);
    }
  }
}

template <bool TA, bool TB, int R, int KT>
void launch_gemm_wave(const float* A, int64_t lda, const float* B, int64_t ldb, float* C,
                      int64_t ldc, int64_t M, int64_t N, int64_t K, float alpha, float beta,
                      hipStream_t st) {
  auto vec = [&](const float* X, int64_t ld, int64_t along) {
    return along % 4 == 0 && ld % 4 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0 ? 1 : 0;
  };
  const int64_t ntn = ceil_div(N, 8 * R);
  gemm_wave_kernel<TA, TB, R, KT><<<(unsigned)(ceil_div(M, 8 * R) * ntn), 64, 0, st>>>(
      A, lda, B, ldb, C, ldc, (int)M, (int)N, (int)K, alpha, beta, vec(A, lda, TA ? M : K),
      vec(B, ldb, TB ? K : N), (int)ntn);
}

// The tile by the number of 8 x 8 ones (us for 8 / 16 / 32-row tiles, both
// operands along k): up to 16 waves per CU the smallest wins (M 128, N 2048, K
// 256: 8.5 / 8.8 / 15.7; M 1024, N 256, K 1024: 26 / 28 / 55), then its repeated
// operand reads cost more than the shorter chains save (M 1024, N 768: 20 / 12.9 /
// 16.5), and from 64 per CU on the 32-row tile reads least (M 512, N 4096: 50 / 31
// / 23).
template <bool TA, bool TB>
void gemm_wave(const float* A, int64_t lda, const float* B, int64_t ldb, float* C, int64_t ldc,
               int64_t M, int64_t N, int64_t K, float alpha, float beta, hipStream_t st) {
  const int64_t tiles = ceil_div(M, 8) * ceil_div(N, 8);
  if (tiles <= 4096)
    launch_gemm_wave<TA, TB, 1, 128>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
  else if (tiles <= 16384)
    launch_gemm_wave<TA, TB, 2, 64>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
  else
    launch_gemm_wave<TA, TB, 4, 32>(A, lda, B, ldb, C, ldc, M, N, K, alpha, beta, st);
}

}  // namespace
}  // namespace sm
