// Fused linear head + cross-entropy (the LinearCrossEntropyBackend seam).
//
// Forward: per chunk of `chunk` token rows, logits = hidden[rows] . W^T (+ b)
// into a workspace slab of [chunk, stored_vocab] f32 (the full [tokens, V]
// logits never exist), then the row kernel of sm_ce_rows (online max / sum,
// token log-prob, padded columns never read); the loss is -mean(lp) over
// every token, one fixed-order reduction. Backward: the same logits per
// chunk, the row kernel's gradient in place scaled by grad_output / tokens
// (read on the device), then dhidden[rows] = G . W, dW (+)= G^T . hidden[rows]
// and db (+)= column sums of G, so padded rows of dW and db stay exactly 0.
// The GEMMs are f32-grade: sm_gemm_ex, or the same plane products over operands that
// were split once into their bf16 planes (gemm_pairs.hip), where that is the faster
// one and the workspace has room. The backward's dhidden and dW always are at
// matrix-core sizes: dhidden's few tiles have K = V, which is split over the chip
// (4096 x 768 x 32768, chunk 1024, with bias: backward 11.98 -> 4.45 ms, dhidden's
// error against float64 2.3e-6 -> 3.8e-7). The logits are where their bias then needs
// no pass of its own or the weight is large (lce_split).
//
// Reference: LinearCrossEntropyBackend (summa-llm/src/model/linear_cross_entropy/mod.rs:33-57),
// chunked_loss / chunked_backward (reference.rs:42-159), fused_loss /
// fused_backward (gpu.rs:264-426).
#include <algorithm>

#include "common.hpp"
#include "gemm_pairs.hpp"

namespace sm {
namespace {

constexpr size_t kLceAlign = 256;
size_t lce_align(size_t v) { return (v + kLceAlign - 1) / kLceAlign * kLceAlign; }

// Workspace layout: logits [chunk, Vs] f32 | lp [tokens] f32 | row scale
// [chunk] f32 | bias-gradient partials [kColParts, Vs] f32.
constexpr int kColParts = 64;

struct LceLayout {
  size_t logits, lp, rscale, parts, total;
};

LceLayout lce_layout(int64_t tokens, int64_t stored, int64_t chunk, bool use_bias) {
  LceLayout l{};
  const int64_t rows = std::min(chunk, tokens);
  l.logits = 0;
  l.lp = l.logits + lce_align((size_t)rows * stored * 4);
  l.rscale = l.lp + lce_align((size_t)tokens * 4);
  l.parts = l.rscale + lce_align((size_t)rows * 4);
  l.total = l.parts + (use_bias ? lce_align((size_t)kColParts * stored * 4) : 0);
  return l;
}

// The split operands and the split-K partial sums behind the chunk's buffers:
// W [V, d] and W^T [d, V], hidden [tokens, d], and per chunk hidden^T, G and G^T.
// Three exact bf16 planes each: a vocabulary row or a token whose factor in a sum
// is zero (padding, a softmax saturated on its target) may hold any finite values,
// and planes of every element's own leave the others' bits alone. (f16 pairs on one
// power-of-two scale per row took half the products but lost the small rows to a
// large one.)
constexpr Split kForm = Split::kBf16x3;
struct LceSplit {
  bool logits, grads;  // which products run on split operands
  SplitOperand w, h;   // the logits'
  SplitOperand wt, ht, g, gt;
  float* part;
  int64_t part_floats;
  size_t forward, total;  // bytes with which the forward, the backward does so
};

// the products sm_gemm_ex would run on the matrix cores
bool lce_split_sizes(int64_t rows, int64_t d, int64_t stored) {
  return d >= 32 && rows >= 32 && pairs_fit(d) && pairs_fit(rows) && pairs_fit(stored) &&
         rows * stored >= (int64_t)128 * 128 * 16 &&
         rows * stored * d >= ((int64_t)1 << 27);
}

LceSplit lce_split(int64_t tokens, int64_t d, int64_t stored, int64_t chunk, bool use_bias,
                   size_t start, char* ws) {
  const int64_t rows = std::min(chunk, tokens);
  LceSplit l{};
  size_t at = start;
  auto place = [&](int64_t r, int64_t k) {
    const SplitOperand o = split_place(kForm, r, k, ws + at);
    at += (size_t)split_bytes(kForm, r, k);
    return o;
  };
  l.grads = lce_split_sizes(rows, d, stored);
  // The split of W pays from about 1024 tokens on, and then through the bias (added
  // in the epilogue, not by a pass over the logits) or a weight of some 2^27
  // elements. Forward, split against in-loop, us: with bias 1024 x 768 x 32768 332 /
  // 355, 4096 x 768 x 32768 1206 / 1413, 4096 x 256 x 4096 134 / 178, but 512 x 1024 x
  // 32768 252 / 226; without 4096 x 768 x 32768 1192 / 1221, 2048 x 1024 x 32768 812 /
  // 779, 1024 x 2048 x 65536 1582 / 1638, 4096 x 2048 x 65536 5753 / 6546, but 128 x
  // 2048 x 65536 481 / 213.
  l.logits = l.grads && tokens >= 1024 && (use_bias || d * stored >= ((int64_t)1 << 27));
  if (l.logits) {
    l.w = place(stored, d);
    l.h = place(tokens, d);
  }
  l.forward = l.total = at;
  if (!l.grads) return l;
  l.wt = place(d, stored);
  l.ht = place(d, rows);
  l.g = split_place(kForm, rows, stored, ws + at);  // G, then G^T in its place
  l.gt = split_place(kForm, stored, rows, ws + at);
  at += (size_t)std::max(split_bytes(kForm, rows, stored), split_bytes(kForm, stored, rows));
  auto parts = [](int64_t m, int64_t n, int64_t k) {
    return gemm_pairs_part_floats(kForm, kForm, m, n, k);
  };
  const int64_t last = tokens % rows;  // the last chunk may choose other splits
  for (int64_t r : {rows, last})
    if (r > 0)
      l.part_floats = std::max({l.part_floats, parts(r, d, stored), parts(stored, d, r)});
  l.part = reinterpret_cast<float*>(ws + at);
  l.total = at + lce_align((size_t)l.part_floats * 4);
  return l;
}

// rows [start, start + n) of a row-split operand
SplitOperand lce_rows(SplitOperand o, int64_t start, int64_t n) {
  o.data += start * o.row_bytes();
  o.rows = n;
  return o;
}

// logits[r, c] += bias[c] over the stored columns.
__global__ void add_bias_kernel(float* __restrict__ logits, const float* __restrict__ bias,
                                int64_t rows, int64_t stored) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * stored) return;
  logits[i] += bias[i % stored];
}

// scale[r] = grad_output[0] / tokens for the chunk's rows.
__global__ void fill_scale_kernel(float* __restrict__ scale, int64_t rows,
                                  const float* __restrict__ grad_output, float inv_tokens) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < rows) scale[i] = grad_output[0] * inv_tokens;
}

// Column sums of G [rows, Vs] in kColParts row slices (part p sums rows
// p, p + kColParts, ... in order), then db (+)= the parts summed in order:
// deterministic, no atomics.
__global__ void colsum_parts_kernel(const float* __restrict__ g, int64_t rows, int64_t stored,
                                    float* __restrict__ parts) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int p = blockIdx.y;
  if (c >= stored) return;
  float acc = 0.f;
  for (int64_t r = p; r < rows; r += kColParts) acc += g[r * stored + c];
  parts[(int64_t)p * stored + c] = acc;
}

__global__ void colsum_finish_kernel(const float* __restrict__ parts, int64_t stored,
                                     int accumulate, float* __restrict__ db) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= stored) return;
  float acc = 0.f;
  for (int p = 0; p < kColParts; ++p) acc += parts[(int64_t)p * stored + c];
  db[c] = accumulate ? db[c] + acc : acc;
}

// loss = -mean(lp) over every token (f64, fixed order).
__global__ __launch_bounds__(1024) void lce_mean_neg_kernel(const float* __restrict__ lp,
                                                            int64_t n, float* __restrict__ loss) {
  __shared__ double part[1024 / kWave];
  double acc = 0.0;
  for (int64_t i = threadIdx.x; i < n; i += 1024) acc += (double)lp[i];
  acc = wave_sum_f64(acc);
  if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < 1024 / kWave; ++w) t += part[w];
    loss[0] = (float)(-t / (double)n);
  }
}

int lce_check(const float* hidden, const float* weight, const float* bias,
              const int32_t* targets, int64_t tokens, int64_t d, int64_t stored,
              int64_t logical, int64_t chunk, int use_bias, void* ws, int64_t ws_bytes,
              const char* who) {
  SM_REQUIRE(hidden && weight && targets && ws, "%s: null argument", who);
  SM_REQUIRE(chunk > 0, "linear cross-entropy chunk size must be positive");
  SM_REQUIRE(tokens > 0, "linear cross-entropy requires at least one token");
  SM_REQUIRE(d > 0 && d < (1 << 30) && stored > 0 && stored < (1 << 30), "%s: bad shape", who);
  SM_REQUIRE(logical > 0 && logical <= stored, "logical vocabulary %lld must be in 1..=%lld",
             (long long)logical, (long long)stored);
  SM_REQUIRE(!use_bias || bias, "%s: use_bias needs a bias vector", who);
  SM_REQUIRE(reinterpret_cast<uintptr_t>(ws) % kLceAlign == 0, "%s: workspace must be 256-byte aligned",
             who);
  const LceLayout l = lce_layout(tokens, stored, chunk, use_bias != 0);
  SM_REQUIRE(ws_bytes >= 0 && (size_t)ws_bytes >= l.total,
             "%s: workspace holds %lld bytes, %zu needed (sm_linear_cross_entropy_workspace_bytes)",
             who, (long long)ws_bytes, l.total);
  return SM_OK;
}

// logits of rows [start, start + rows) into the workspace slab (+ bias), from the
// split operands where `l` says so (K is not split: where sm_gemm_ex is on the matrix
// cores, the same bits).
int lce_logits(const LceSplit& l, const float* hidden, const float* weight, const float* bias,
               int64_t start, int64_t rows, int64_t d, int64_t stored, int use_bias,
               float* logits, hipStream_t st) {
  if (l.logits)
    return gemm_pairs(lce_rows(l.h, start, rows), l.w, rows, stored, 1.f, 0.f,
                      use_bias ? bias : nullptr, logits, stored, nullptr, 0, st);
  SM_TRY(sm_gemm_ex(0, 1, rows, stored, d, 1.0f, hidden + start * d, d, weight, d, 0.0f, logits,
                    stored, st));
  if (use_bias) {
    const int64_t n = rows * stored;
    add_bias_kernel<<<(unsigned)ceil_div(n, 256), 256, 0, st>>>(logits, bias, rows, stored);
    SM_LAUNCH_CHECK();
  }
  return SM_OK;
}

}  // namespace
}  // namespace sm

using namespace sm;

extern "C" int64_t sm_linear_cross_entropy_workspace_bytes(int64_t tokens, int64_t d,
                                                           int64_t stored_vocab, int64_t chunk,
                                                           int use_bias) {
  if (tokens <= 0 || d <= 0 || stored_vocab <= 0 || chunk <= 0) return -1;
  const size_t n = lce_layout(tokens, stored_vocab, chunk, use_bias != 0).total;
  return (int64_t)lce_split(tokens, d, stored_vocab, chunk, use_bias != 0, n, nullptr).total;
}

extern "C" int64_t sm_linear_cross_entropy_forward_workspace_bytes(int64_t tokens, int64_t d,
                                                                   int64_t stored_vocab,
                                                                   int64_t chunk, int use_bias) {
  if (tokens <= 0 || d <= 0 || stored_vocab <= 0 || chunk <= 0) return -1;
  const size_t n = lce_layout(tokens, stored_vocab, chunk, use_bias != 0).total;
  return (int64_t)lce_split(tokens, d, stored_vocab, chunk, use_bias != 0, n, nullptr).forward;
}

extern "C" int sm_linear_cross_entropy(const float* hidden, const float* weight,
                                       const float* bias, const int32_t* targets, int64_t tokens,
                                       int64_t d, int64_t stored_vocab, int64_t logical_vocab,
                                       int64_t chunk, int use_bias, float* loss,
                                       float* token_logprob, void* workspace,
                                       int64_t workspace_bytes, void* stream) {
  SM_TRY(lce_check(hidden, weight, bias, targets, tokens, d, stored_vocab, logical_vocab, chunk,
                   use_bias, workspace, workspace_bytes, "sm_linear_cross_entropy"));
  SM_REQUIRE(loss, "sm_linear_cross_entropy: null loss");
  hipStream_t st = as_stream(stream);
  const LceLayout l = lce_layout(tokens, stored_vocab, chunk, use_bias != 0);
  char* ws = static_cast<char*>(workspace);
  float* logits = reinterpret_cast<float*>(ws + l.logits);
  float* lp = token_logprob ? token_logprob : reinterpret_cast<float*>(ws + l.lp);
  LceSplit sp = lce_split(tokens, d, stored_vocab, chunk, use_bias != 0, l.total, ws);
  if ((size_t)workspace_bytes < sp.forward) sp = {};
  if (sp.logits) {
    SM_TRY(split_operand(sp.w, weight, d, true, d, st));
    SM_TRY(split_operand(sp.h, hidden, d, true, d, st));
  }
  for (int64_t s0 = 0; s0 < tokens; s0 += chunk) {
    const int64_t rows = std::min(chunk, tokens - s0);
    SM_TRY(lce_logits(sp, hidden, weight, bias, s0, rows, d, stored_vocab, use_bias, logits, st));
    SM_TRY(sm_ce_rows(logits, SM_F32, targets + s0, rows, stored_vocab, logical_vocab, lp + s0,
                      nullptr, nullptr, 1.0f, nullptr, nullptr, st));
  }
  lce_mean_neg_kernel<<<1, 1024, 0, st>>>(lp, tokens, loss);
  SM_LAUNCH_CHECK();
  return SM_OK;
}

extern "C" int sm_linear_cross_entropy_backward(
    const float* hidden, const float* weight, const float* bias, const int32_t* targets,
    const float* grad_output, int64_t tokens, int64_t d, int64_t stored_vocab,
    int64_t logical_vocab, int64_t chunk, int use_bias, float* grad_hidden, float* grad_weight,
    float* grad_bias, void* workspace, int64_t workspace_bytes, void* stream) {
  SM_TRY(lce_check(hidden, weight, bias, targets, tokens, d, stored_vocab, logical_vocab, chunk,
                   use_bias, workspace, workspace_bytes, "sm_linear_cross_entropy_backward"));
  SM_REQUIRE(grad_output && grad_hidden && grad_weight,
             "sm_linear_cross_entropy_backward: null gradient buffer");
  SM_REQUIRE(!use_bias || grad_bias, "sm_linear_cross_entropy_backward: use_bias needs grad_bias");
  hipStream_t st = as_stream(stream);
  const LceLayout l = lce_layout(tokens, stored_vocab, chunk, use_bias != 0);
  char* ws = static_cast<char*>(workspace);
  float* logits = reinterpret_cast<float*>(ws + l.logits);
  float* lp = reinterpret_cast<float*>(ws + l.lp);
  float* rscale = reinterpret_cast<float*>(ws + l.rscale);
  float* parts = reinterpret_cast<float*>(ws + l.parts);
  const float inv_tokens = (float)(1.0 / (double)tokens);
  LceSplit sp = lce_split(tokens, d, stored_vocab, chunk, use_bias != 0, l.total, ws);
  if ((size_t)workspace_bytes < sp.total) sp = {};
  if (sp.logits) {
    SM_TRY(split_operand(sp.w, weight, d, true, d, st));
    SM_TRY(split_operand(sp.h, hidden, d, true, d, st));
  }
  if (sp.grads) SM_TRY(split_operand(sp.wt, weight, d, false, stored_vocab, st));
  for (int64_t s0 = 0; s0 < tokens; s0 += chunk) {
    const int64_t rows = std::min(chunk, tokens - s0);
    const bool first = s0 == 0;
    SM_TRY(lce_logits(sp, hidden, weight, bias, s0, rows, d, stored_vocab, use_bias, logits, st));
    fill_scale_kernel<<<(unsigned)ceil_div(rows, 256), 256, 0, st>>>(rscale, rows, grad_output,
                                                                     inv_tokens);
    SM_LAUNCH_CHECK();
    // G = (softmax - onehot) * grad_output / tokens in place; padded columns 0
    SM_TRY(sm_ce_rows(logits, SM_F32, targets + s0, rows, stored_vocab, logical_vocab, lp + s0,
                      nullptr, logits, 1.0f, rscale, nullptr, st));
    // dhidden[rows] = G . W          ([rows, Vs] x [Vs, d])
    // dW (+)= G^T . hidden[rows]     ([Vs, rows] x [rows, d])
    if (sp.grads) {
      const SplitOperand g = split_place(kForm, rows, stored_vocab, sp.g.data);
      const SplitOperand gt = split_place(kForm, stored_vocab, rows, sp.gt.data);
      const SplitOperand ht = split_place(kForm, d, rows, sp.ht.data);
      SM_TRY(split_operand(g, logits, stored_vocab, true, stored_vocab, st));
      SM_TRY(gemm_pairs(g, sp.wt, rows, d, 1.f, 0.f, nullptr, grad_hidden + s0 * d, d, sp.part,
                        sp.part_floats, st));
      SM_TRY(split_operand(gt, logits, stored_vocab, false, rows, st));
      SM_TRY(split_operand(ht, hidden + s0 * d, d, false, rows, st));
      SM_TRY(gemm_pairs(gt, ht, stored_vocab, d, 1.f, first ? 0.f : 1.f, nullptr, grad_weight, d,
                        sp.part, sp.part_floats, st));
    } else {
      SM_TRY(sm_gemm_ex(0, 0, rows, d, stored_vocab, 1.0f, logits, stored_vocab, weight, d, 0.0f,
                        grad_hidden + s0 * d, d, st));
      SM_TRY(sm_gemm_ex(1, 0, stored_vocab, d, rows, 1.0f, logits, stored_vocab, hidden + s0 * d,
                        d, first ? 0.0f : 1.0f, grad_weight, d, st));
    }
    if (use_bias) {
      const dim3 grid((unsigned)ceil_div(stored_vocab, 256), kColParts);
      colsum_parts_kernel<<<grid, 256, 0, st>>>(logits, rows, stored_vocab, parts);
      colsum_finish_kernel<<<(unsigned)ceil_div(stored_vocab, 256), 256, 0, st>>>(
          parts, stored_vocab, first ? 0 : 1, grad_bias);
      SM_LAUNCH_CHECK();
    }
  }
  return SM_OK;
}
