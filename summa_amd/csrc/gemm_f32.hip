// Dense fp32 matmul y = x . W^T for fp32 models (config[0]: the reference CPU
// path's precision, summa-llm/src/model/matmul.rs:57-66 with F32 weights),
// plus the SwiGLU combine of a [gate | value] projection (ffn.rs:854-886).
//
// Used for the tiny fp32 model, whose decode batches have a few rows; the
// quantized path uses q4.hip.
#include "common.hpp"

namespace sm {
namespace {

// One wave per workgroup owns an 8R x 8R output tile, lane (ty, tx) the outputs
// of rows ty + 8 i and columns tx + 8 j. Both operand tiles sit in LDS as rows of
// KT + 4 floats along k (the pad puts the eight rows a 16-byte read touches in
// different banks), and the next KT columns' loads are in flight in registers
// during the current ones' FMAs; with one wave there is no barrier to wait at.
// An output is one serial chain of FMAs over k in order, whatever the tile, so
// the tile size changes no bits. At decode sizes that chain and the launch are
// the bound, so the tile is as small as fills the chip. M 32, against one
// 64 x 64 tile per 256 threads (4 to 64 workgroups): 768 x 256 19.9 -> 4.1 us,
// 256 x 1024 70.7 -> 10.8, 4096 x 256 20.2 -> 5.5.
template <bool ADD, int R, int KT>
__global__ __launch_bounds__(64) void gemm_f32_wave_kernel(const float* __restrict__ w,
                                                           const float* __restrict__ x,
                                                           float* __restrict__ y, int M, int N,
                                                           int K, int ldx, int ldy, int vec,
                                                           int ntn) {
  constexpr int ROWS = 8 * R, RS = KT + 4, NL = ROWS * KT / 256;  // float4 loads per operand
  typedef float f4 __attribute__((ext_vector_type(4)));
  __shared__ __attribute__((aligned(16))) float xs[ROWS * RS];
  __shared__ __attribute__((aligned(16))) float ws[ROWS * RS];
  const int l = threadIdx.x, tx = l % 8, ty = l / 8;
  const int m0 = (int)(blockIdx.x / ntn) * ROWS, n0 = (int)(blockIdx.x % ntn) * ROWS;
  f4 rx[NL], rw[NL];
  auto fetch = [&](const float* p, size_t ld, int row, int rows, int k) -> f4 {
    f4 v = {0.f, 0.f, 0.f, 0.f};
    if (row >= rows || k >= K) return v;
    const float* q = p + (size_t)row * ld + k;
    if (vec) return *reinterpret_cast<const f4*>(q);  // K % 4 == 0, aligned rows
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (k + e < K) v[e] = q[e];
    return v;
  };
  auto gload = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = i * 64 + l, r = c / (KT / 4), k = k0 + 4 * (c % (KT / 4));
      rx[i] = fetch(x, (size_t)ldx, m0 + r, M, k);
      rw[i] = fetch(w, (size_t)K, n0 + r, N, k);
    }
  };
  float acc[R][R] = {};
  gload(0);
  for (int k0 = 0; k0 < K; k0 += KT) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = i * 64 + l, r = c / (KT / 4), k = 4 * (c % (KT / 4));
      *reinterpret_cast<f4*>(xs + r * RS + k) = rx[i];
      *reinterpret_cast<f4*>(ws + r * RS + k) = rw[i];
    }
    __syncthreads();
    if (k0 + KT < K) gload(k0 + KT);
#pragma unroll 4
    for (int k = 0; k < KT; k += 4) {
      f4 a[R], b[R];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        a[i] = *reinterpret_cast<const f4*>(xs + (ty + 8 * i) * RS + k);
        b[i] = *reinterpret_cast<const f4*>(ws + (tx + 8 * i) * RS + k);
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
      float* o = y + (size_t)gm * ldy + gn;
      if (ADD) *o += acc[i][j]; else *o = acc[i][j];
    }
  }
}

template <int R, int KT>
void launch_gemm_f32(const float* w, const float* x, float* y, int64_t M, int64_t N, int64_t K,
                     int64_t ldx, int64_t ldy, bool add, hipStream_t st) {
  const int vec = K % 4 == 0 && ldx % 4 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 &&
                  reinterpret_cast<uintptr_t>(x) % 16 == 0;
  const int64_t ntn = ceil_div(N, 8 * R);
  const unsigned grid = (unsigned)(ceil_div(M, 8 * R) * ntn);
  if (add)
    gemm_f32_wave_kernel<true, R, KT><<<grid, 64, 0, st>>>(w, x, y, (int)M, (int)N, (int)K,
                                                           (int)ldx, (int)ldy, vec, (int)ntn);
  else
    gemm_f32_wave_kernel<false, R, KT><<<grid, 64, 0, st>>>(w, x, y, (int)M, (int)N, (int)K,
                                                            (int)ldx, (int)ldy, vec, (int)ntn);
}

__global__ void swiglu_f32_kernel(const float* __restrict__ gv, int64_t rows, int F,
                                  float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * F) return;
  const int64_t r = i / F;
  const int c = i % F;
  const float g = gv[r * 2 * F + c], v = gv[r * 2 * F + F + c];
  out[i] = g / (1.f + expf(-g)) * v;
}

}  // namespace
}  // namespace sm

using namespace sm;

extern "C" int sm_gemm_f32(const float* w, int64_t N, int64_t K, const float* x, int64_t M,
                           int64_t ldx, float* y, int64_t ldy, int epilogue, void* stream) {
  SM_REQUIRE(w && x && y, "sm_gemm_f32: null buffer");
  SM_REQUIRE(N > 0 && K > 0 && M >= 0 && ldx >= K && ldy >= N, "sm_gemm_f32: bad shape");
  SM_REQUIRE(M <= 0x7fffffff && N <= 0x7fffffff, "sm_gemm_f32: shape too large");
  SM_REQUIRE(epilogue == SM_EPI_STORE_F32 || epilogue == SM_EPI_ADD_F32,
             "sm_gemm_f32: epilogue must be SM_EPI_STORE_F32 or SM_EPI_ADD_F32");
  if (M == 0) return SM_OK;
  // The tile by the number of 8 x 8 ones (us for 8 / 16 / 32-row tiles): up to
  // 16 waves per CU the smallest wins (M 128, N 2048, K 256: 8.5 / 8.8 / 15.7;
  // M 1024, N 256, K 1024: 26 / 28 / 55), then its repeated operand reads cost
  // more than the shorter chains save (M 1024, N 768: 20 / 12.9 / 16.5), and from
  // 64 per CU on the 32-row tile reads least (M 512, N 4096: 50 / 31 / 23).
  const int64_t tiles = ceil_div(M, 8) * ceil_div(N, 8);
  const bool add = epilogue == SM_EPI_ADD_F32;
  hipStream_t st = as_stream(stream);
  if (tiles <= 4096) launch_gemm_f32<1, 128>(w, x, y, M, N, K, ldx, ldy, add, st);
  else if (tiles <= 16384) launch_gemm_f32<2, 64>(w, x, y, M, N, K, ldx, ldy, add, st);
  else launch_gemm_f32<4, 32>(w, x, y, M, N, K, ldx, ldy, add, st);
  SM_LAUNCH_CHECK();
  return SM_OK;
}

extern "C" int sm_swiglu_f32(const float* gate_value, int64_t rows, int64_t F, float* out,
                             void* stream) {
  SM_REQUIRE(gate_value && out, "sm_swiglu_f32: null buffer");
  SM_REQUIRE(rows >= 0 && F > 0, "sm_swiglu_f32: bad shape");
  const int64_t n = rows * F;
  if (n == 0) return SM_OK;
  swiglu_f32_kernel<<<(unsigned)ceil_div(n, 256), 256, 0, as_stream(stream)>>>(gate_value, rows,
                                                                              (int)F, out);
  SM_LAUNCH_CHECK();
  return SM_OK;
}
