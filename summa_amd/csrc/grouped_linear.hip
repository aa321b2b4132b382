// Float-weight grouped expert projections and the MoE row permutation at the
// reference's dispatch seam:
//   * GroupedLinearBackend::grouped_linear_inner / _backward
//     (summa-llm/src/model/grouped_linear.rs:23-60, 65-86): input [routes,
//     d_in] with its rows grouped by expert (counts[e] consecutive rows of
//     expert e, in expert order), weight [E, d_in, d_out] row-major, output
//     [routes, d_out] = each expert's rows times its matrix; the backward
//     gives grad_input = grad W_e^T per expert and grad_weight[e] =
//     input_e^T grad_e (zero for an expert without rows);
//   * grouped_swiglu_mlp_inner / _backward (grouped_linear.rs:40-60, 89-111,
//     779-826): projected = grouped_linear(input, in_weight) as [gate |
//     value] (fused_swiglu.rs:30-42), hidden = silu(gate) * value, output =
//     grouped_linear(hidden, down_weight); the backward chains the two
//     grouped backwards through the SwiGLU backward;
//   * RowPermutationBackend::row_permute_inner (row_permute.rs:33-41): out[i]
//     = input[order[i]] (float_select over rows; the backward is the same
//     selection by the inverse permutation).
// The counts are host values, as grouped_linear_inner takes them (Vec<usize>;
// the CUDA path reads device counts back to the host before its grouped GEMM,
// grouped_linear.rs:787).
//
// With a workspace (the _ws entries) a projection is one f32-grade launch over
// all experts on operands split once into three exact bf16 planes (gemm_pairs.hip): a
// launch per expert left the chip with one expert's few tiles at a time (24 to
// 100 workgroups on 256 CUs; the weight gradients, K = an expert's rows, ran on
// 24-48). 8192 tokens, top-2 of 8 experts, d 512, width 768, forward and
// backward: 4.81 -> 1.25 ms. Without one, or for few experts and small products
// (grouped_split_sizes), each expert with rows is one sm_gemm_ex, in expert order.
#include <algorithm>

#include "common.hpp"
#include "gemm_pairs.hpp"

extern "C" {
int sm_gemm_ex(int, int, int64_t, int64_t, int64_t, float, const float*, int64_t, const float*,
               int64_t, float, float*, int64_t, void*);
int sm_swiglu(const void*, int, int64_t, int64_t, void*, void*);
int sm_swiglu_backward(const void*, const void*, int, int64_t, int64_t, void*, void*);
}

namespace sm {
namespace {

// out row i = in row order[i] (16-byte chunks when rows allow, else 4-byte
// words or 2-byte elements); an order entry outside [0, rows) gives a zero row.
template <typename T>
__global__ __launch_bounds__(256) void row_permute_kernel(const T* __restrict__ in,
                                                          const int32_t* __restrict__ order,
                                                          int64_t rows, int64_t units,
                                                          T* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= rows * units) return;
  const int64_t r = i / units, u = i % units;
  const int32_t src = order[r];
  T v{};
  if (src >= 0 && src < rows) v = in[(int64_t)src * units + u];
  out[i] = v;
}

__global__ void zero_f32_kernel(float* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

int check_counts(const int64_t* counts, int64_t experts, int64_t routes, const char* who) {
  SM_REQUIRE(counts, "%s: null counts", who);
  int64_t sum = 0;
  for (int64_t e = 0; e < experts; ++e) {
    SM_REQUIRE(counts[e] >= 0, "%s: negative count for expert %lld", who, (long long)e);
    sum += counts[e];
  }
  SM_REQUIRE(sum == routes, "%s: route counts must cover the input (%lld != %lld)", who,
             (long long)sum, (long long)routes);
  return SM_OK;
}

// The workspace of a projection: the rows, the weights and, in the backward, the
// two run-padded transposes, all as three exact bf16 planes: a row whose factor in a
// sum is zero may hold any finite values. (f16 pairs on one power-of-two scale per
// row or column took half the products but lost the small rows to a large one.)
constexpr Split kForm = Split::kBf16x3;
struct GroupedWs {
  void* p;
  int64_t bytes;
};

// Whether a projection is one launch over all experts on split operands, or a launch
// per expert. One launch costs 20 to 30 us forward and 35 to 60 backward however little
// it does (the splits, and one tile's serial K); the others 4 to 8 us an expert and then
// their arithmetic, on the FMA units below 2^27 multiply-adds. Forward / backward us,
// one launch against one per expert: 8 experts of 64 rows, 256 x 256 25 / 35 against 42 /
// 61, of 2048 rows, 512 x 1536 222 / 501 against 357 / 2107; 6 of 128 rows, 256 x 256 25 /
// 47 against 28 / 51 (2^25.6 in all); 4 of 512 rows, 256 x 512 28 / 82 against 39 / 87
// (2^28), of 256 rows 27 / 64 against 26 / 61; 1 of 1024 rows, 512 x 512 32 / 80 against
// 39 / 122, of 256 rows, 256 x 512 21 / 48 against 7 / 16. Few experts with narrow sides
// have few tiles for long sums: 4 of 16384 rows, 64 x 128 47 / 812 against 43 / 689.
bool grouped_split_sizes(int64_t routes, int64_t d_in, int64_t d_out, int64_t experts) {
  const int64_t narrow = std::min(d_in, d_out), madds = routes * d_in * d_out;
  if (!pairs_fit(d_in) || !pairs_fit(d_out) || !pairs_fit(routes + 64 * experts) ||
      experts * std::max(d_in, d_out) >= (1 << 30) || experts >= (1 << 16))
    return false;
  return experts >= 6 ? narrow >= 32 && madds >= ((int64_t)1 << 25)
                      : narrow >= 128 && madds >= ((int64_t)1 << 28);
}

int64_t forward_bytes(int64_t experts, int64_t routes, int64_t d_in, int64_t d_out) {
  if (!grouped_split_sizes(routes, d_in, d_out, experts)) return 0;
  return split_bytes(kForm, routes, d_in) + split_bytes(kForm, experts * d_out, d_in);
}

int64_t backward_bytes(int64_t experts, int64_t routes, int64_t d_in, int64_t d_out) {
  if (!grouped_split_sizes(routes, d_in, d_out, experts)) return 0;
  const int64_t kp = routes + 64 * experts;  // every run padded to whole 64s
  return std::max(split_bytes(kForm, routes, d_out) + split_bytes(kForm, experts * d_in, d_out),
                  split_bytes(kForm, d_in, kp) + split_bytes(kForm, d_out, kp));
}

bool use_split(const GroupedWs& ws, int64_t need) {
  return ws.p && need > 0 && need <= ws.bytes && reinterpret_cast<uintptr_t>(ws.p) % 16 == 0;
}

// Experts e0 .. e0 + kMaxRuns - 1 as runs of the grouped rows.
Runs runs_of(const int64_t* counts, int64_t experts, int64_t e0, int64_t off) {
  Runs r{};
  r.n = (int)std::min<int64_t>(kMaxRuns, experts - e0);
  for (int i = 0; i < r.n; ++i) {
    r.off[i] = (int)off;
    r.cnt[i] = (int)counts[e0 + i];
    off += counts[e0 + i];
  }
  return r;
}

// y = x B_e^T per expert, from split rows x and weights [E][n] split along k
int grouped_rows(const SplitOperand& x, const SplitOperand& w, const int64_t* counts,
                 int64_t experts, int64_t n, float* y, hipStream_t st) {
  int64_t off = 0;
  for (int64_t e0 = 0; e0 < experts; e0 += kMaxRuns) {
    const Runs r = runs_of(counts, experts, e0, off);
    SplitOperand b = w;
    b.data += e0 * n * w.row_bytes();
    SM_TRY(gemm_pairs_rows(x, b, n, n, r, y, n, st));
    off = r.off[r.n - 1] + r.cnt[r.n - 1];
  }
  return SM_OK;
}

// y = x W_e per expert (x rows grouped by expert, W [E, d_in, d_out])
int grouped_forward(const float* x, const float* w, const int64_t* counts, int64_t experts,
                    int64_t routes, int64_t d_in, int64_t d_out, float* y, const GroupedWs& ws,
                    void* stream) {
  if (use_split(ws, forward_bytes(experts, routes, d_in, d_out))) {
    hipStream_t st = as_stream(stream);
    const SplitOperand a = split_place(kForm, routes, d_in, ws.p);
    const SplitOperand b =
        split_place(kForm, experts * d_out, d_in,
                    static_cast<char*>(ws.p) + split_bytes(kForm, routes, d_in));
    SM_TRY(split_operand(a, x, d_in, true, d_in, st));
    SM_TRY(split_operand(b, w, d_out, false, d_in, st, nullptr, experts));
    return grouped_rows(a, b, counts, experts, d_out, y, st);
  }
  int64_t off = 0;
  for (int64_t e = 0; e < experts; ++e) {
    const int64_t c = counts[e];
    if (c > 0)
      SM_TRY(sm_gemm_ex(0, 0, c, d_out, d_in, 1.f, x + off * d_in, d_in,
                        w + e * d_in * d_out, d_out, 0.f, y + off * d_out, d_out, stream));
    off += c;
  }
  return SM_OK;
}

// The same two gradients as one launch each.
int grouped_backward_split(const float* x, const float* w, const float* grad,
                           const int64_t* counts, int64_t experts, int64_t routes, int64_t d_in,
                           int64_t d_out, float* grad_x, float* grad_w, void* ws,
                           hipStream_t st) {
  char* at = static_cast<char*>(ws);
  if (grad_x) {
    const SplitOperand g = split_place(kForm, routes, d_out, at);
    const SplitOperand b = split_place(kForm, experts * d_in, d_out,
                                       at + split_bytes(kForm, routes, d_out));
    SM_TRY(split_operand(g, grad, d_out, true, d_out, st));
    SM_TRY(split_operand(b, w, d_out, true, d_out, st));
    SM_TRY(grouped_rows(g, b, counts, experts, d_in, grad_x, st));
  }
  if (grad_w) {
    int64_t off = 0;
    for (int64_t e0 = 0; e0 < experts; e0 += kMaxRuns) {
      const Runs r = runs_of(counts, experts, e0, off);
      int64_t kp = 0;
      for (int i = 0; i < r.n; ++i) kp += ceil_div(r.cnt[i], 64) * 64;
      const SplitOperand a = split_place(kForm, d_in, kp, at);
      const SplitOperand b =
          split_place(kForm, d_out, kp, at + split_bytes(kForm, d_in, kp));
      const int64_t rows = r.off[r.n - 1] + r.cnt[r.n - 1] - r.off[0];
      Runs local = r;
      for (int i = 0; i < r.n; ++i) local.off[i] -= r.off[0];
      SM_TRY(split_operand(a, x + off * d_in, d_in, false, rows, st, &local));
      SM_TRY(split_operand(b, grad + off * d_out, d_out, false, rows, st, &local));
      SM_TRY(gemm_pairs_ks(a, b, d_in, d_out, r, grad_w + e0 * d_in * d_out, d_out,
                           d_in * d_out, st));
      off += rows;
    }
  }
  return SM_OK;
}

// grad_x = grad W_e^T; grad_w[e] = x_e^T grad_e (zero without rows)
int grouped_backward(const float* x, const float* w, const float* grad, const int64_t* counts,
                     int64_t experts, int64_t routes, int64_t d_in, int64_t d_out, float* grad_x,
                     float* grad_w, const GroupedWs& ws, void* stream) {
  hipStream_t st = as_stream(stream);
  if (use_split(ws, backward_bytes(experts, routes, d_in, d_out)))
    return grouped_backward_split(x, w, grad, counts, experts, routes, d_in, d_out, grad_x, grad_w,
                                  ws.p, st);
  int64_t off = 0;
  for (int64_t e = 0; e < experts; ++e) {
    const int64_t c = counts[e];
    float* gw = grad_w ? grad_w + e * d_in * d_out : nullptr;
    if (c > 0) {
      if (grad_x)
        SM_TRY(sm_gemm_ex(0, 1, c, d_in, d_out, 1.f, grad + off * d_out, d_out,
                          w + e * d_in * d_out, d_out, 0.f, grad_x + off * d_in, d_in, stream));
      if (gw)
        SM_TRY(sm_gemm_ex(1, 0, d_in, d_out, c, 1.f, x + off * d_in, d_in, grad + off * d_out,
                          d_out, 0.f, gw, d_out, stream));
    } else if (gw) {
      zero_f32_kernel<<<(unsigned)ceil_div(d_in * d_out, 256), 256, 0, st>>>(gw, d_in * d_out);
      SM_LAUNCH_CHECK();
    }
    off += c;
  }
  return SM_OK;
}

}  // namespace
}  // namespace sm

using namespace sm;

extern "C" int sm_row_permute(const void* input, int dtype, int64_t rows, int64_t cols,
                              const int32_t* order, void* out, void* stream) {
  SM_REQUIRE(input && order && out, "sm_row_permute: null buffer");
  SM_REQUIRE(rows >= 0 && cols > 0, "sm_row_permute: bad shape");
  SM_REQUIRE(dtype == SM_F32 || dtype == SM_BF16 || dtype == SM_F16,
             "sm_row_permute: dtype must be SM_F32, SM_BF16 or SM_F16");
  SM_REQUIRE(input != out, "sm_row_permute: out must not alias input");
  if (rows == 0) return SM_OK;
  hipStream_t st = as_stream(stream);
  const int64_t bytes = cols * (dtype == SM_F32 ? 4 : 2);
  const bool a16 = bytes % 16 == 0 && reinterpret_cast<uintptr_t>(input) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const bool a4 = bytes % 4 == 0 && reinterpret_cast<uintptr_t>(input) % 4 == 0 &&
                  reinterpret_cast<uintptr_t>(out) % 4 == 0;
  if (a16) {
    const int64_t units = bytes / 16;
    row_permute_kernel<u32x4><<<(unsigned)ceil_div(rows * units, 256), 256, 0, st>>>(
        static_cast<const u32x4*>(input), order, rows, units, static_cast<u32x4*>(out));
  } else if (a4) {
    const int64_t units = bytes / 4;
    row_permute_kernel<uint32_t><<<(unsigned)ceil_div(rows * units, 256), 256, 0, st>>>(
        static_cast<const uint32_t*>(input), order, rows, units, static_cast<uint32_t*>(out));
  } else {
    const int64_t units = bytes / 2;
    row_permute_kernel<uint16_t><<<(unsigned)ceil_div(rows * units, 256), 256, 0, st>>>(
        static_cast<const uint16_t*>(input), order, rows, units, static_cast<uint16_t*>(out));
  }
  SM_LAUNCH_CHECK();
  return SM_OK;
}

extern "C" int64_t sm_grouped_linear_workspace_bytes(int64_t experts, int64_t routes,
                                                     int64_t d_in, int64_t d_out, int backward) {
  if (experts <= 0 || routes < 0 || d_in <= 0 || d_out <= 0) return -1;
  return backward ? backward_bytes(experts, routes, d_in, d_out)
                  : forward_bytes(experts, routes, d_in, d_out);
}

extern "C" int64_t sm_grouped_swiglu_mlp_workspace_bytes(int64_t experts, int64_t routes,
                                                         int64_t d, int64_t intermediate,
                                                         int64_t d_out, int backward) {
  if (experts <= 0 || routes < 0 || d <= 0 || intermediate <= 0 || d_out <= 0) return -1;
  if (backward)
    return std::max(backward_bytes(experts, routes, intermediate, d_out),
                    backward_bytes(experts, routes, d, 2 * intermediate));
  return std::max(forward_bytes(experts, routes, d, 2 * intermediate),
                  forward_bytes(experts, routes, intermediate, d_out));
}

extern "C" int sm_grouped_linear_ws(const float* input, const float* weight,
                                    const int64_t* counts, int64_t experts, int64_t routes,
                                    int64_t d_in, int64_t d_out, float* out, void* workspace,
                                    int64_t workspace_bytes, void* stream) {
  SM_REQUIRE(input && weight && out, "sm_grouped_linear: null buffer");
  SM_REQUIRE(experts > 0 && routes >= 0 && d_in > 0 && d_out > 0, "sm_grouped_linear: bad shape");
  SM_TRY(check_counts(counts, experts, routes, "sm_grouped_linear"));
  return grouped_forward(input, weight, counts, experts, routes, d_in, d_out, out,
                         {workspace, workspace_bytes}, stream);
}

extern "C" int sm_grouped_linear(const float* input, const float* weight, const int64_t* counts,
                                 int64_t experts, int64_t routes, int64_t d_in, int64_t d_out,
                                 float* out, void* stream) {
  return sm_grouped_linear_ws(input, weight, counts, experts, routes, d_in, d_out, out, nullptr, 0,
                              stream);
}

extern "C" int sm_grouped_linear_backward_ws(const float* input, const float* weight,
                                             const float* grad, const int64_t* counts,
                                             int64_t experts, int64_t routes, int64_t d_in,
                                             int64_t d_out, float* grad_input,
                                             float* grad_weight, void* workspace,
                                             int64_t workspace_bytes, void* stream) {
  SM_REQUIRE(input && weight && grad && (grad_input || grad_weight),
             "sm_grouped_linear_backward: null buffer");
  SM_REQUIRE(experts > 0 && routes >= 0 && d_in > 0 && d_out > 0,
             "sm_grouped_linear_backward: bad shape");
  SM_TRY(check_counts(counts, experts, routes, "sm_grouped_linear_backward"));
  return grouped_backward(input, weight, grad, counts, experts, routes, d_in, d_out, grad_input,
                          grad_weight, {workspace, workspace_bytes}, stream);
}

extern "C" int sm_grouped_linear_backward(const float* input, const float* weight,
                                          const float* grad, const int64_t* counts,
                                          int64_t experts, int64_t routes, int64_t d_in,
                                          int64_t d_out, float* grad_input, float* grad_weight,
                                          void* stream) {
  return sm_grouped_linear_backward_ws(input, weight, grad, counts, experts, routes, d_in, d_out,
                                       grad_input, grad_weight, nullptr, 0, stream);
}

extern "C" int sm_grouped_swiglu_mlp_ws(const float* input, const float* in_weight,
                                        const float* down_weight, const int64_t* counts,
                                        int64_t experts, int64_t routes, int64_t d,
                                        int64_t intermediate, int64_t d_out, float* out,
                                        float* projected, float* hidden, void* workspace,
                                        int64_t workspace_bytes, void* stream) {
  SM_REQUIRE(input && in_weight && down_weight && out && projected && hidden,
             "sm_grouped_swiglu_mlp: null buffer");
  SM_REQUIRE(experts > 0 && routes >= 0 && d > 0 && intermediate > 0 && d_out > 0,
             "sm_grouped_swiglu_mlp: bad shape");
  SM_TRY(check_counts(counts, experts, routes, "sm_grouped_swiglu_mlp"));
  if (routes == 0) return SM_OK;
  const GroupedWs ws{workspace, workspace_bytes};
  SM_TRY(grouped_forward(input, in_weight, counts, experts, routes, d, 2 * intermediate, projected,
                         ws, stream));
  SM_TRY(sm_swiglu(projected, SM_F32, routes, intermediate, hidden, stream));
  return grouped_forward(hidden, down_weight, counts, experts, routes, intermediate, d_out, out, ws,
                         stream);
}

extern "C" int sm_grouped_swiglu_mlp(const float* input, const float* in_weight,
                                     const float* down_weight, const int64_t* counts,
                                     int64_t experts, int64_t routes, int64_t d,
                                     int64_t intermediate, int64_t d_out, float* out,
                                     float* projected, float* hidden, void* stream) {
  return sm_grouped_swiglu_mlp_ws(input, in_weight, down_weight, counts, experts, routes, d,
                                  intermediate, d_out, out, projected, hidden, nullptr, 0, stream);
}

extern "C" int sm_grouped_swiglu_mlp_backward_ws(
    const float* input, const float* in_weight, const float* down_weight, const int64_t* counts,
    int64_t experts, int64_t routes, int64_t d, int64_t intermediate, int64_t d_out,
    const float* projected, const float* hidden, const float* grad, float* grad_input,
    float* grad_in_weight, float* grad_down_weight, float* scratch, void* workspace,
    int64_t workspace_bytes, void* stream) {
  SM_REQUIRE(input && in_weight && down_weight && projected && hidden && grad && grad_input &&
                 grad_in_weight && grad_down_weight && scratch,
             "sm_grouped_swiglu_mlp_backward: null buffer");
  SM_REQUIRE(experts > 0 && routes >= 0 && d > 0 && intermediate > 0 && d_out > 0,
             "sm_grouped_swiglu_mlp_backward: bad shape");
  SM_TRY(check_counts(counts, experts, routes, "sm_grouped_swiglu_mlp_backward"));
  const GroupedWs ws{workspace, workspace_bytes};
  // scratch: grad_hidden [routes, I] then grad_projected [routes, 2I]
  float* grad_hidden = scratch;
  float* grad_projected = scratch + routes * intermediate;
  SM_TRY(grouped_backward(hidden, down_weight, grad, counts, experts, routes, intermediate, d_out,
                          grad_hidden, grad_down_weight, ws, stream));
  if (routes > 0)
    SM_TRY(sm_swiglu_backward(projected, grad_hidden, SM_F32, routes, intermediate,
                              grad_projected, stream));
  return grouped_backward(input, in_weight, grad_projected, counts, experts, routes, d,
                          2 * intermediate, grad_input, grad_in_weight, ws, stream);
}

extern "C" int sm_grouped_swiglu_mlp_backward(const float* input, const float* in_weight,
                                              const float* down_weight, const int64_t* counts,
                                              int64_t experts, int64_t routes, int64_t d,
                                              int64_t intermediate, int64_t d_out,
                                              const float* projected, const float* hidden,
                                              const float* grad, float* grad_input,
                                              float* grad_in_weight, float* grad_down_weight,
                                              float* scratch, void* stream) {
  return sm_grouped_swiglu_mlp_backward_ws(input, in_weight, down_weight, counts, experts, routes,
                                           d, intermediate, d_out, projected, hidden, grad,
                                           grad_input, grad_in_weight, grad_down_weight, scratch,
                                           nullptr, 0, stream);
}
