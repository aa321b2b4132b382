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
