// Dense fp32 matmul y = x . W^T for fp32 models (config[0]: the reference CPU
// path's precision, summa-llm/src/model/matmul.rs:57-66 with F32 weights),
// plus the SwiGLU combine of a [gate | value] projection (ffn.rs:854-886).
//
// Used for the tiny fp32 model, whose decode batches have a few rows (the GEMM is
// gemm_wave.hpp's); the quantized path uses q4.hip.
#include "common.hpp"
#include "gemm_wave.hpp"

namespace sm {
namespace {

// A decode batch's projection with the step that follows in its epilogue: SwiGLU
// of [gate | value] columns, or RoPE and the cache append of a qkv projection. A
// decode step of the tiny model is 23 launches of 4 to 11 us, most of that the
// launch itself; this takes out two a layer (32 rollouts x 32 tokens, two layers:
// 3.36 -> 3.18 ms). The projection and the epilogues are gemm_wave_kernel's,
// swiglu_f32_kernel's and rope_append_kernel's: the same bits. (The RMSNorm before
// them as well, each workgroup normalising its own rows, cost as much as its
// launch: 3.35 ms against 3.36.)
struct FusedGemm {
  const float *x, *w;
  int M, N, K, ntn, vec;  // N: output columns (SwiGLU: of each half)
  float* y;  // SwiGLU
  const float2* rope;  // RoPE, to the end
  const int32_t* pos0;
  int L, H, KVH, hd, cap;
  float *q, *kc, *vc;
};

template <bool SWIGLU>
__global__ __launch_bounds__(64) void fused_gemm_kernel(FusedGemm g) {
  constexpr int KT = 128, RS = KT + 4;
  using Tile = WaveTile<true, 1, KT>;
  __shared__ __attribute__((aligned(16))) float as[8 * RS];
  __shared__ __attribute__((aligned(16))) float bs[SWIGLU ? 2 : 1][8 * RS];
  const int l = threadIdx.x, tx = l % 8, ty = l / 8;
  const int m0 = (int)(blockIdx.x / g.ntn) * 8, n0 = (int)(blockIdx.x % g.ntn) * 8;
  Tile ta{g.x, g.K, m0, g.M, g.K, g.vec}, tb{g.w, g.K, n0, g.N, g.K, g.vec};
  Tile tv{g.w + (int64_t)g.N * g.K, g.K, n0, g.N, g.K, g.vec};
  auto load = [&](int k0) {
    ta.load(k0, l);
    tb.load(k0, l);
    if constexpr (SWIGLU) tv.load(k0, l);
  };
  load(0);
  float acc = 0.f, val = 0.f;
  for (int k0 = 0; k0 < g.K; k0 += KT) {
    ta.store(as, l);
    tb.store(bs[0], l);
    if constexpr (SWIGLU) tv.store(bs[1], l);
    __syncthreads();
    if (k0 + KT < g.K) load(k0 + KT);
#pragma unroll 8
    for (int k = 0; k < KT; k += 4) {
      const f32x4w a = *reinterpret_cast<const f32x4w*>(as + ty * RS + k);
      const f32x4w b = *reinterpret_cast<const f32x4w*>(bs[0] + tx * RS + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = fmaf(a[e], b[e], acc);
      if constexpr (SWIGLU) {
        const f32x4w c = *reinterpret_cast<const f32x4w*>(bs[1] + tx * RS + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) val = fmaf(a[e], c[e], val);
      }
    }
    __syncthreads();
  }
  const int row = m0 + ty, col = n0 + tx;
  const float other = SWIGLU ? 0.f : dpp_f32<kDppXor1>(acc);  // the pair's other column
  if (row >= g.M || col >= g.N) return;
  if constexpr (SWIGLU) {
    g.y[(int64_t)row * g.N + col] = acc / (1.f + expf(-acc)) * val;
  } else {
    const int s = row / g.L, pos = g.pos0[s] + row % g.L;
    if (pos < 0 || pos >= g.cap) return;
    const int slot = col / g.hd, e = col % g.hd;
    const float a = col & 1 ? other : acc, b = col & 1 ? acc : other;
    if (slot >= g.H + g.KVH) {  // value: no rotation
      g.vc[(((int64_t)s * g.KVH + slot - g.H - g.KVH) * g.cap + pos) * g.hd + e] = acc;
      return;
    }
    const float2 cs = g.rope[(int64_t)pos * (g.hd / 2) + e / 2];  // (cos, sin)
    const float ra = a * cs.x - b * cs.y;
    const float rb = b * cs.x + a * cs.y;
    float* dst = slot < g.H
                     ? g.q + ((int64_t)row * g.H + slot) * g.hd + e
                     : g.kc + (((int64_t)s * g.KVH + slot - g.H) * g.cap + pos) * g.hd + e;
    *dst = col & 1 ? rb : ra;
  }
}

template <bool SWIGLU>
int launch_fused_gemm(FusedGemm g, hipStream_t st) {
  g.ntn = (int)ceil_div(g.N, 8);
  g.vec = g.K % 4 == 0 && reinterpret_cast<uintptr_t>(g.x) % 16 == 0 &&
          reinterpret_cast<uintptr_t>(g.w) % 16 == 0;
  fused_gemm_kernel<SWIGLU><<<(unsigned)(ceil_div(g.M, 8) * g.ntn), 64, 0, st>>>(g);
  SM_LAUNCH_CHECK();
  return SM_OK;
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

// Whether the fused forms below take a projection of M rows and N columns: the
// sizes of gemm_wave's smallest tile.
bool f32_fused_fits(int64_t M, int64_t N) { return ceil_div(M, 8) * ceil_div(N, 8) <= 4096; }

int f32_swiglu(const float* w, const float* x, int64_t M, int64_t F, int64_t K, float* y,
               hipStream_t st) {
  FusedGemm g{x, w, (int)M, (int)F, (int)K};
  g.y = y;
  return launch_fused_gemm<true>(g, st);
}

int f32_qkv_rope(const float* w, const float* x, int64_t S, int64_t L, int64_t H, int64_t KVH,
                 int64_t hd, int64_t K, const float* rope, const int32_t* pos0, int64_t cap,
                 float* q, float* kc, float* vc, hipStream_t st) {
  FusedGemm g{x, w, (int)(S * L), (int)((H + 2 * KVH) * hd), (int)K};
  g.rope = reinterpret_cast<const float2*>(rope);
  g.pos0 = pos0;
  g.L = (int)L;
  g.H = (int)H;
  g.KVH = (int)KVH;
  g.hd = (int)hd;
  g.cap = (int)cap;
  g.q = q;
  g.kc = kc;
  g.vc = vc;
  return launch_fused_gemm<false>(g, st);
}

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
  gemm_wave<false, true>(x, ldx, w, K, y, ldy, M, N, K, 1.f,
                         epilogue == SM_EPI_ADD_F32 ? 1.f : 0.f, as_stream(stream));
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
