// Internal interface of the pre-split matrix-core GEMM (gemm_pairs.hip).
#pragma once

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

namespace sm {

// How a split operand holds its values: the leading one, two or three bf16 planes
// of x (one: rounded to bf16; three: exact).
enum class Split { kBf16, kBf16x2, kBf16x3 };
constexpr int planes_of(Split f) {
  return f == Split::kBf16x3 ? 3 : f == Split::kBf16x2 ? 2 : 1;
}

// Consecutive runs of the grouped forms: run i covers `cnt[i]` rows (or k)
// from `off[i]` of the dense operand.
constexpr int kMaxRuns = 64;
struct Runs {
  int n;
  int off[kMaxRuns], cnt[kMaxRuns];
};

// op(X) of `rows` rows and K columns in split form, k padded with zeros to whole
// 64s, in the caller's buffer of split_bytes() (16-byte aligned).
struct SplitOperand {
  Split form;
  char* data;
  int64_t rows, kp;
  int64_t row_bytes() const { return kp * 2 * planes_of(form); }
};
int64_t split_bytes(Split form, int64_t rows, int64_t K);
SplitOperand split_place(Split form, int64_t rows, int64_t K, void* buf);

// Whether K is in the kernel's range (a tile's rows lie within 4 GB).
bool pairs_fit(int64_t K);

// Fills `o` from X: element (r, k) at X[r * ld + k] (kc) or X[k * ld + r]. With
// `runs` (not kc), the runs' k follow each other, each padded with zeros to whole
// 64s. With `batch` > 1 (not kc), X holds that many matrices,
// K * ld apart, whose rows / batch rows each follow each other.
int split_operand(const SplitOperand& o, const float* X, int64_t ld, bool kc, int64_t K,
                  hipStream_t st, const Runs* runs = nullptr, int64_t batch = 1);

// C = alpha A B^T + beta C (+ bias along n) from split operands: each form with
// itself, or kBf16x3 with kBf16x2. Without `part`, gemm_planes' sums bit for bit. With
// it, three planes' sums as exact as they come: the lower planes' products apart from
// hi.hi, and K split where the plan says so and part_floats are room for the parts.
int gemm_pairs(const SplitOperand& A, const SplitOperand& B, int64_t M, int64_t N, float alpha,
               float beta, const float* bias, float* C, int64_t ldc, float* part,
               int64_t part_floats, hipStream_t st);
// Floats of `part` that let gemm_pairs split K as it would choose to.
int64_t gemm_pairs_part_floats(Split a, Split b, int64_t M, int64_t N, int64_t K);
// Rows of A in runs, run e against B[e] (`bstride` rows of B apart, N used):
// C rows off[e] .. = A rows off[e] .. times B_e^T.
int gemm_pairs_rows(const SplitOperand& A, const SplitOperand& B, int64_t bstride, int64_t N,
                    const Runs& runs, float* C, int64_t ldc, hipStream_t st);
// k in runs: C_e (`cstride` floats apart) = A[:, run e] B[:, run e]^T, zero for
// an empty run.
int gemm_pairs_ks(const SplitOperand& A, const SplitOperand& B, int64_t M, int64_t N,
                  const Runs& runs, float* C, int64_t ldc, int64_t cstride, hipStream_t st);

}  // namespace sm
