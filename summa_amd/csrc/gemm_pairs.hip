// Matrix-core GEMM over operands that were split once into 16-bit planes: the
// large f32 products of training (the policy's forward, data and weight
// gradients, the linear head + cross-entropy, the MoE expert projections).
//
// Forms: one, two or three unscaled bf16 planes, the plane products of
// gemm_mfma.hip with the split taken out of the K loop, in its order (the same bits)
// unless the caller lets the sums be more exact. Three planes hold every f32 exactly,
// whatever its row holds beside it. (Two f16 planes on a power-of-two scale of the row
// or column took three products instead of six, and 0.7 of the time, but held 22 bits,
// and fewer of values below 2^-18 of their row's largest: a row that a zero factor
// took out of the sum erased the others.)
//
// Layout of a split operand: per row, one plane: its k in order; more: per 32 k
// the planes' 64 bytes one after the other. A stage of the K loop then reads
// whole lines.
//
// gemm_pairs_kernel: a BM x BN tile per workgroup, 8 waves (4 for the dense 128 x 128,
// two of which share a CU where their planes leave the LDS for it); two LDS stages
// filled by global_load_lds (16 bytes a lane, no registers): the next stage's copies
// are issued right after the barrier and land during the current one's MFMAs. 16-byte chunk c of row r lies at
// c ^ f(r), f chosen so that the 32-row fragment reads spread over all banks;
// the copy permutes its global addresses instead, as its LDS side is always
// consecutive.
#include "gemm_pairs.hpp"

#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace sm {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kCUs = 256;

// ------------------------------------------------------------------ split --

// 8 consecutive values of a row at k (a multiple of 8) -> 16 bytes per plane
template <Split F>
__device__ inline void store8(char* row, int64_t k, const float* v) {
  constexpr int P = planes_of(F);
  u32x4 w[P];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
#pragma unroll
    for (int p = 0; p < P; ++p) {
      w[p][i] = pack_bf16x2(a, b);
      a -= bf16lo(w[p][i]);
      b -= bf16hi(w[p][i]);
    }
  }
  char* o = row + (P == 1 ? k * 2 : k / 32 * (64 * P) + k % 32 * 2);
#pragma unroll
  for (int p = 0; p < P; ++p) *reinterpret_cast<u32x4*>(o + 64 * p) = w[p];
}

// k contiguous: T threads per row (one wave, or the workgroup for long rows),
// 8 k per thread and step, 4 steps in flight. HBM-bound: 4 bytes read and 2 per
// plane written a value.
template <Split F, int T>
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ X, int64_t ld,
                                                         int64_t R, int64_t K, int64_t Kp,
                                                         char* __restrict__ out,
                                                         int64_t row_bytes, int vec) {
  constexpr int NR = 4;
  const int64_t r = (int64_t)blockIdx.x * (256 / T) + threadIdx.x / T;
  if (r >= R) return;
  const float* x = X + r * ld;
  char* row = out + r * row_bytes;
  for (int64_t k0 = 8 * (threadIdx.x % T); k0 < Kp; k0 += 8 * T * NR) {
    float v[NR][8];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int64_t k = k0 + 8 * T * i;
      if (k >= Kp) continue;
      if (vec && k + 8 <= K) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(x + k);
        const f32x4 b = *reinterpret_cast<const f32x4*>(x + k + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[i][e] = a[e];
          v[i][4 + e] = b[e];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = k + e < K ? x[k + e] : 0.f;
      }
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int64_t k = k0 + 8 * T * i;
      if (k < Kp) store8<F>(row, k, v[i]);
    }
  }
}

// The rows [k0, k1) of X behind 64-k block kb of the split operand.
__device__ inline void block_rows(int64_t kb, int64_t K, int use_runs, const Runs& runs,
                                  int64_t& k0, int64_t& k1) {
  k0 = kb * 64;
  k1 = K;
  if (!use_runs) return;
  int e = 0;
  while (kb >= (runs.cnt[e] + 63) / 64) kb -= (runs.cnt[e++] + 63) / 64;
  k0 = runs.off[e] + kb * 64;
  k1 = runs.off[e] + runs.cnt[e];
}

// k across rows: 64 k x 64 r tiles through LDS; reads are 64 consecutive r a
// wave, writes 8 consecutive chunks (whole lines) of a row. With runs, 64-k
// block b of the output is the next 64 k of its run (zeros past its end).
template <Split F>
__global__ __launch_bounds__(256) void split_cols_kernel(const float* __restrict__ X, int64_t ld,
                                                         int64_t R, int64_t K,
                                                         char* __restrict__ out,
                                                         int64_t row_bytes, int use_runs,
                                                         Runs runs) {
  __shared__ float t[64][65];  // [k][r]
  const int64_t kb = blockIdx.x, r0 = (int64_t)blockIdx.y * 64;
  X += blockIdx.z * K * ld;
  out += blockIdx.z * R * row_bytes;
  int64_t k0, k1;
  block_rows(kb, K, use_runs, runs, k0, k1);
  const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
#pragma unroll 4
  for (int i = ty; i < 64; i += 4) {
    const int64_t k = k0 + i, r = r0 + tx;
    t[i][tx] = (k < k1 && r < R) ? X[k * ld + r] : 0.f;
  }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = (int)threadIdx.x + 256 * h, rl = c / 8, kl = (c % 8) * 8;
    if (r0 + rl >= R) continue;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = t[kl + e][rl];
    store8<F>(out + (r0 + rl) * row_bytes, kb * 64 + kl, v);
  }
}

// ------------------------------------------------------------------- GEMM --

struct PairArgs {
  const char *A, *B;
  int64_t rowA, rowB;  // bytes
  int rowsA;
  float* C;
  int64_t ldc;
  int M, N, nst;  // nst: K stages
  float alpha, beta;
  const float* bias;
  int ntm, ntn, splits;
  float* part;     // [splits][M][N] when splits > 1
  int64_t stride;  // run forms: B rows (kRows) or C floats (kKs) per run
  Runs runs;
};
enum Mode { kPlain, kRows, kKs };

// Tile order: workgroups go to the 8 XCDs in turn, each XCD gets a consecutive
// range of tiles, and within it four tile rows are walked column by column, so
// that the tiles an XCD works on at once share operand rows in its L2.
__device__ inline void tile_of(int id, int total, int ntm, int ntn, int& tm, int& tn) {
  const int per = total / 8, rem = total % 8, x = id % 8, i = id / 8;
  const int t = x * per + min(x, rem) + i;
  constexpr int G = 4;
  const int band = t / (G * ntn), m0 = band * G, gm = min(G, ntm - m0), in = t - band * G * ntn;
  tm = m0 + in % gm;
  tn = in / gm;
}

// plane pairs (a, b) of each product, smallest weight first
template <int PA, int PB> struct Products;
template <> struct Products<3, 3> {
  static constexpr int n = 6, a[6] = {2, 1, 0, 1, 0, 0}, b[6] = {0, 1, 2, 0, 1, 0};
};
template <> struct Products<3, 2> {
  static constexpr int n = 5, a[5] = {2, 1, 1, 0, 0}, b[5] = {0, 1, 0, 1, 0};
};
template <> struct Products<2, 2> {
  static constexpr int n = 3, a[3] = {1, 0, 0}, b[3] = {0, 1, 0};
};
template <> struct Products<1, 1> { static constexpr int n = 1, a[1] = {0}, b[1] = {0}; };

__device__ inline f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// TWO: the products of lower planes, all but hi.hi, are summed apart and added last.
// An addition rounds at the size of the sum, so five of three planes' six additions
// then round at 2^-8 of it: at the same time, a third to two thirds of the error
// against float64 (K 512, 768, 1536: 3.4e-7, 4.2e-7, 6.0e-7 -> 1.3e-7, 1.6e-7, 2.3e-7;
// K 32768 in 10 splits 6.5e-7 -> 3.8e-7).
template <int PA, int PB, int BM, int BN, int BK, int WM, int WN, Mode MODE, bool TWO>
__global__ __launch_bounds__(WM * WN * 64, 2) void gemm_pairs_kernel(PairArgs g) {
  static_assert((PA == 1 || BK == 32) && (PB == 1 || BK == 32), "");
  constexpr int NW = WM * WN;
  constexpr int CR = BK / 8;                           // chunks per row, plane and stage
  constexpr int SA = PA * BM * CR, SB = PB * BN * CR;  // chunks per stage
  constexpr int NA = SA / (64 * NW), NB = SB / (64 * NW);  // copies per wave
  static_assert(SA % (64 * NW) == 0 && SB % (64 * NW) == 0, "");
  constexpr int MB = BM / WM / 32, NBk = BN / WN / 32;  // 32 x 32 blocks per wave
  constexpr int kStage = (SA + SB) * 16;
  __shared__ __attribute__((aligned(16))) char lds[2 * kStage];
  const int lane = threadIdx.x % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int wm = wave / WN, wn = wave % WN;

  int tm, tn, z = 0, M = g.M, s0 = 0, s1 = g.nst, arow0 = 0;
  const char* Bp = g.B;
  float* C = g.C;
  if constexpr (MODE == kPlain) {
    const int per = g.ntm * g.ntn;
    z = blockIdx.x / per;
    tile_of(blockIdx.x % per, per, g.ntm, g.ntn, tm, tn);
    if (g.splits > 1) {
      s0 = (int)((int64_t)g.nst * z / g.splits);
      s1 = (int)((int64_t)g.nst * (z + 1) / g.splits);
    }
  } else if constexpr (MODE == kRows) {
    int t = blockIdx.x / g.ntn, e = 0;
    while (t >= (g.runs.cnt[e] + BM - 1) / BM) t -= (g.runs.cnt[e++] + BM - 1) / BM;
    tm = t;
    tn = blockIdx.x % g.ntn;
    M = g.runs.cnt[e];
    arow0 = g.runs.off[e];
    Bp += (int64_t)e * g.stride * g.rowB;
    C += (int64_t)arow0 * g.ldc;
  } else {
    const int per = g.ntm * g.ntn, e = blockIdx.x / per;
    tm = blockIdx.x % per / g.ntn;
    tn = blockIdx.x % per % g.ntn;
    for (int i = 0; i < e; ++i) s0 += (g.runs.cnt[i] + 63) / 64 * (64 / BK);
    s1 = s0 + (g.runs.cnt[e] + 63) / 64 * (64 / BK);
    C += (int64_t)e * g.stride;
  }
  const int m0 = tm * BM, n0 = tn * BN;

  // copy j of this wave: chunks (NW j + wave) 64 + lane of the stage, at a fixed
  // offset from the tile's first row; the rows' bases advance with the stages
  uint32_t src[NA + NB];
  auto swz = [](int r) { return CR == 4 ? (r >> 2) & 3 : (r >> 1) & 7; };
#pragma unroll
  for (int j = 0; j < NA + NB; ++j) {
    const bool isA = j < NA;
    const int c = (NW * (isA ? j : j - NA) + wave) * 64 + lane;
    const int rows = isA ? BM : BN;
    const int p = c / (rows * CR), r = c / CR % rows, k = (c % CR) ^ swz(r);
    const int rr = min(r, isA ? g.rowsA - arow0 - m0 - 1 : g.N - n0 - 1);  // rows past the end
    src[j] = (uint32_t)rr * (uint32_t)(isA ? g.rowA : g.rowB) + p * (BK * 2) + k * 16;
  }
  const char* at = g.A + (int64_t)(arow0 + m0) * g.rowA + (int64_t)s0 * (BK * 2 * PA);
  const char* bt = Bp + (int64_t)n0 * g.rowB + (int64_t)s0 * (BK * 2 * PB);
  auto fetch = [&](int buf) {
#if defined(__HIP_DEVICE_COMPILE__)  // (the host pass does not emit the launch stub otherwise)
#pragma unroll
    for (int j = 0; j < NA + NB; ++j) {
      const int to = buf * kStage + (j < NA ? 0 : SA * 16) +
                     (NW * (j < NA ? j : j - NA) + wave) * 1024;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) char*)(j < NA ? at : bt) + src[j],
          (__attribute__((address_space(3))) char*)lds + to, 16, 0, 0);
    }
#endif
    at += BK * 2 * PA;
    bt += BK * 2 * PB;
  };

  f32x16 acc[MB][NBk], low[TWO ? MB : 1][TWO ? NBk : 1];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NBk; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        acc[i][j][e] = 0.f;
        if constexpr (TWO) low[i][j][e] = 0.f;
      }
  // fragment of lane l: row l % 32 of the block, chunk 2 ks + l / 32
  const int fr = lane % 32, fs = swz(fr);  // blocks start at multiples of 32
  const int fa = (wm * (BM / WM) + fr) * CR * 16, fb = (wn * (BN / WN) + fr) * CR * 16;

  if (s0 < s1) fetch(0);
  for (int s = s0; s < s1; ++s) {
    const int buf = (s - s0) & 1;
    // this wave's copies of stage s have landed, and behind the barrier every
    // wave's; every wave has also read all it needs of the other buffer
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + 1 < s1) fetch(buf ^ 1);
    const char* As = lds + buf * kStage;
    const char* Bs = As + SA * 16;
    // the fragments of the next 16 k are read between the MFMAs of these
    u32x4 a[2][PA][MB], b[2][PB][NBk];
    auto frags = [&](int ks) {
      const int co = ((2 * ks + lane / 32) ^ fs) * 16;
#pragma unroll
      for (int p = 0; p < PA; ++p)
#pragma unroll
        for (int i = 0; i < MB; ++i)
          a[ks & 1][p][i] =
              *reinterpret_cast<const u32x4*>(As + (p * BM + i * 32) * CR * 16 + fa + co);
#pragma unroll
      for (int p = 0; p < PB; ++p)
#pragma unroll
        for (int i = 0; i < NBk; ++i)
          b[ks & 1][p][i] =
              *reinterpret_cast<const u32x4*>(Bs + (p * BN + i * 32) * CR * 16 + fb + co);
    };
    frags(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      if (ks + 1 < BK / 16) frags(ks + 1);
      using Pr = Products<PA, PB>;
#pragma unroll
      for (int q = 0; q < Pr::n; ++q)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int j = 0; j < NBk; ++j) {
            f32x16& c = TWO && q + 1 < Pr::n ? low[TWO ? i : 0][TWO ? j : 0] : acc[i][j];
            c = mfma(a[ks & 1][Pr::a[q]][i], b[ks & 1][Pr::b[q]][j], c);
          }
      if (ks + 1 < BK / 16) {
        constexpr int nr = PA * MB + PB * NBk, nm = Pr::n * MB * NBk;
#pragma unroll
        for (int r = 0; r < nr; ++r) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
          __builtin_amdgcn_sched_group_barrier(0x008, nm / nr > 0 ? nm / nr : 1, 0);  // MFMAs
        }
        __builtin_amdgcn_sched_group_barrier(0x008, nm, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // acc[i][j][e]: row 8 (e / 4) + 4 (lane / 32) + e % 4, column lane % 32
  auto emit = [&](auto whole) {  // whole: no row or column of the tile is past the end
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int rb = m0 + wm * (BM / WM) + i * 32 + 4 * (lane / 32);
#pragma unroll
      for (int j = 0; j < NBk; ++j) {
        const int col = n0 + wn * (BN / WN) + j * 32 + fr;
        if (!whole && col >= g.N) continue;
        const float bias = g.bias ? g.bias[col] : 0.f;
        float old[16];  // read together: a read behind a write of C waits for it
        if (g.beta != 0.f && !(MODE == kPlain && g.splits > 1)) {
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            const int row = rb + 8 * (e / 4) + e % 4;
            if (whole || row < M) old[e] = C[(int64_t)row * g.ldc + col];
          }
        }
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = rb + 8 * (e / 4) + e % 4;
          if (!whole && row >= M) continue;
          const float v = TWO ? acc[i][j][e] + low[TWO ? i : 0][TWO ? j : 0][e] : acc[i][j][e];
          if (MODE == kPlain && g.splits > 1) {
            g.part[((int64_t)z * M + row) * g.N + col] = v;
            continue;
          }
          const float w = g.beta == 0.f ? g.alpha * v : fmaf(g.alpha, v, g.beta * old[e]);
          C[(int64_t)row * g.ldc + col] = g.bias ? w + bias : w;
        }
      }
    }
  };
  if (m0 + BM <= M && n0 + BN <= g.N) emit(std::true_type{});
  else emit(std::false_type{});
}

// C = alpha sum_z part[z] + beta C (+ bias), z in order
__global__ __launch_bounds__(256) void pairs_reduce_kernel(const float* __restrict__ part,
                                                           int splits, int64_t M, int64_t N,
                                                           float alpha, float beta,
                                                           const float* __restrict__ bias,
                                                           float* __restrict__ C, int64_t ldc) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= M * N) return;
  float v = part[i];
  for (int z = 1; z < splits; ++z) v += part[z * M * N + i];
  float* o = C + i / N * ldc + i % N;
  const float w = beta == 0.f ? alpha * v : fmaf(alpha, v, beta * *o);
  *o = bias ? w + bias[i % N] : w;
}

// ---------------------------------------------------------------- dispatch --

// (the grouped modes and TWO take three planes only)
template <Mode MODE, int BM, int BN, int WM, int WN, bool TWO>
int launch(const SplitOperand& A, const SplitOperand& B, PairArgs& g, int64_t wgs,
           hipStream_t st) {
  if (wgs == 0) return SM_OK;
  SM_REQUIRE(wgs * 512 < ((int64_t)1 << 32) && pairs_fit(A.kp) && A.kp == B.kp,
             "gemm_pairs: shape out of range");
#define SM_GP(PA, PB, BK) \
  gemm_pairs_kernel<PA, PB, BM, BN, BK, WM, WN, MODE, TWO>  \
      <<<(unsigned)wgs, WM * WN * 64, 0, st>>>(g)
  g.nst = (int)(A.kp / (A.form == Split::kBf16 ? 64 : 32));
  if constexpr (TWO) {
    SM_GP(3, 3, 32);
  } else {
    if constexpr (BM * BN <= 256 * 128) {  // (three planes of a larger tile overflow LDS)
      if (A.form == Split::kBf16x3) {
        if (B.form == Split::kBf16x3) SM_GP(3, 3, 32);
        else SM_GP(3, 2, 32);
      }
    }
    if (A.form == Split::kBf16x2) SM_GP(2, 2, 32);
    else if (A.form == Split::kBf16) SM_GP(1, 1, 64);
  }
#undef SM_GP
  SM_LAUNCH_CHECK();
  return SM_OK;
}

PairArgs pair_args(const SplitOperand& A, const SplitOperand& B) {
  PairArgs g{};
  g.A = A.data;
  g.B = B.data;
  g.rowA = A.row_bytes();
  g.rowB = B.row_bytes();
  g.rowsA = (int)A.rows;
  g.alpha = 1.f;
  g.splits = 1;
  return g;
}

// The tile and the K splits of an M x N x K product: rounds of workgroups over
// the chip times the time of a round, ns per k measured at full rounds (`ns1` for
// one product, `ns3` for three, more in proportion;
// 1.05-1.2 PF/s of MFMA work, set by power rather than by the tile), less where
// a round leaves CUs idle (0.6 of it for the large tiles with few busy, half for
// the 128 x 128 ones, two of which share a CU). A split writes and reads its
// partial sums. Three products, us: 8192 x 8192 x 4096 256 x 256 1378, 128 x 256
// 1493, 128 x 128 1558; 2048 x 2048 x 8184 500, 288, 208. Six: 1024 x 768 x 32768 (24
// tiles of 128 x 256) in 10 splits 291. One bf16 product: 4096 x 2048 x 65536 1598,
// 1350, 1112.
struct Tile {
  int bm, bn, slots;  // slots: workgroups the chip runs at once
  double ns1, ns3;
};
constexpr Tile kTiles[] = {
    {256, 256, kCUs, 34, 85}, {128, 256, kCUs, 20, 46}, {128, 128, 2 * kCUs, 18.5, 47.5}};
struct Plan {
  int tile, splits;
};
Plan pair_plan(Split a, Split b, int64_t M, int64_t N, int64_t K, bool split_k) {
  const bool three = a == Split::kBf16x3;
  const double products = !three ? 1.0 : b == Split::kBf16x3 ? 2.0 : 5.0 / 3.0;
  Plan best{0, 1};
  double least = 0;
  for (int i = three ? 1 : 0; i < 3; ++i) {
    const Tile& t = kTiles[i];
    const int64_t tiles = ceil_div(M, t.bm) * ceil_div(N, t.bn);
    const int slots = three ? kCUs : t.slots;  // (three planes: one workgroup's LDS per CU)
    const double half = t.slots / slots;
    for (int s = 1; s <= 32; ++s) {
      if (s > 1 && (!split_k || K / s < 512 || tiles * s > 4 * slots)) break;
      const double rounds = (double)ceil_div(tiles * s, slots);
      const double full = tiles * s / (rounds * slots);
      const double part = slots > kCUs ? std::max(0.53, 0.1 + 0.9 * full) : 0.6 + 0.4 * full;
      const double per_k = (a == Split::kBf16 ? t.ns1 : t.ns3) * products / half * part;
      const double ns = rounds * ((double)K / s * per_k + 4000) +
                        (s > 1 ? (double)s * M * N * 8 / 4000 + 5000 : 0);
      if (least == 0 || ns < 0.98 * least) {
        least = ns;
        best = {i, s};
      }
    }
  }
  return best;
}

}  // namespace

bool pairs_fit(int64_t K) { return K <= ((int64_t)1 << 21); }

int64_t split_bytes(Split form, int64_t rows, int64_t K) {
  return ceil_div(rows * split_place(form, rows, K, nullptr).row_bytes(), 256) * 256;
}

SplitOperand split_place(Split form, int64_t rows, int64_t K, void* buf) {
  return {form, static_cast<char*>(buf), rows, ceil_div(K, 64) * 64};
}

namespace {
template <Split F>
int split_fill(const SplitOperand& o, const float* X, int64_t ld, bool kc, int64_t K,
               hipStream_t st, const Runs* runs, int64_t batch) {
  const int64_t R = o.rows / batch, rb = o.row_bytes();
  if (kc) {
    const int vec = ld % 4 == 0 && reinterpret_cast<uintptr_t>(X) % 16 == 0;
    if (o.kp <= 2048)
      split_rows_kernel<F, 64><<<(unsigned)ceil_div(R, 4), 256, 0, st>>>(X, ld, R, K, o.kp,
                                                                         o.data, rb, vec);
    else
      split_rows_kernel<F, 256><<<(unsigned)R, 256, 0, st>>>(X, ld, R, K, o.kp, o.data, rb, vec);
  } else {
    const dim3 grid((unsigned)(o.kp / 64), (unsigned)ceil_div(R, 64), (unsigned)batch);
    split_cols_kernel<F><<<grid, 256, 0, st>>>(X, ld, R, K, o.data, rb,
                                               runs ? 1 : 0, runs ? *runs : Runs{});
  }
  SM_LAUNCH_CHECK();
  return SM_OK;
}
}  // namespace

int split_operand(const SplitOperand& o, const float* X, int64_t ld, bool kc, int64_t K,
                  hipStream_t st, const Runs* runs, int64_t batch) {
  if (o.rows == 0 || o.kp == 0) return SM_OK;
  switch (o.form) {
    case Split::kBf16: return split_fill<Split::kBf16>(o, X, ld, kc, K, st, runs, batch);
    case Split::kBf16x2: return split_fill<Split::kBf16x2>(o, X, ld, kc, K, st, runs, batch);
    default: return split_fill<Split::kBf16x3>(o, X, ld, kc, K, st, runs, batch);
  }
}

int64_t gemm_pairs_part_floats(Split a, Split b, int64_t M, int64_t N, int64_t K) {
  const Plan p = pair_plan(a, b, M, N, ceil_div(K, 64) * 64, true);  // as gemm_pairs sees it
  return p.splits == 1 ? 0 : p.splits * M * N;
}

int gemm_pairs(const SplitOperand& A, const SplitOperand& B, int64_t M, int64_t N, float alpha,
               float beta, const float* bias, float* C, int64_t ldc, float* part,
               int64_t part_floats, hipStream_t st) {
  if (M == 0 || N == 0) return SM_OK;
  PairArgs g = pair_args(A, B);
  Plan p = pair_plan(A.form, B.form, M, N, A.kp, part != nullptr);
  if (p.splits * M * N > part_floats) p.splits = 1;
  g.C = C;
  g.ldc = ldc;
  g.M = (int)M;
  g.N = (int)N;
  g.alpha = alpha;
  g.beta = beta;
  g.bias = bias;
  g.splits = p.splits;
  g.part = part;
  g.ntm = (int)ceil_div(M, kTiles[p.tile].bm);
  g.ntn = (int)ceil_div(N, kTiles[p.tile].bn);
  const int64_t wgs = (int64_t)g.ntm * g.ntn * p.splits;
  if (part && B.form == Split::kBf16x3) {
    if (p.tile == 1) SM_TRY((launch<kPlain, 128, 256, 2, 4, true>(A, B, g, wgs, st)));
    else SM_TRY((launch<kPlain, 128, 128, 2, 4, true>(A, B, g, wgs, st)));
  } else if (p.tile == 0) {
    SM_TRY((launch<kPlain, 256, 256, 2, 4, false>(A, B, g, wgs, st)));
  } else if (p.tile == 1) {
    SM_TRY((launch<kPlain, 128, 256, 2, 4, false>(A, B, g, wgs, st)));
  } else {
    SM_TRY((launch<kPlain, 128, 128, 2, 2, false>(A, B, g, wgs, st)));
  }
  if (p.splits > 1) {
    pairs_reduce_kernel<<<(unsigned)ceil_div(M * N, 256), 256, 0, st>>>(part, p.splits, M, N, alpha,
                                                                        beta, bias, C, ldc);
    SM_LAUNCH_CHECK();
  }
  return SM_OK;
}

// The grouped forms' tile is 128 x 128 with eight waves: three planes of it fill the
// CU's LDS, so four waves would be one per SIMD (8 experts of 512 rows, 512 x 1536,
// forward / backward: 79 / 176 us, with eight 71 / 163; 128 x 256 tiles are within 4 %
// of it either way from two rounds on).
int gemm_pairs_rows(const SplitOperand& A, const SplitOperand& B, int64_t bstride, int64_t N,
                    const Runs& runs, float* C, int64_t ldc, hipStream_t st) {
  PairArgs g = pair_args(A, B);
  g.C = C;
  g.ldc = ldc;
  g.N = (int)N;
  g.stride = bstride;
  g.runs = runs;
  int64_t tm = 0;
  for (int i = 0; i < runs.n; ++i) tm += ceil_div(runs.cnt[i], 128);
  g.ntn = (int)ceil_div(N, 128);
  return launch<kRows, 128, 128, 2, 4, true>(A, B, g, tm * g.ntn, st);
}

int gemm_pairs_ks(const SplitOperand& A, const SplitOperand& B, int64_t M, int64_t N,
                  const Runs& runs, float* C, int64_t ldc, int64_t cstride, hipStream_t st) {
  PairArgs g = pair_args(A, B);
  g.C = C;
  g.ldc = ldc;
  g.M = (int)M;
  g.N = (int)N;
  g.stride = cstride;
  g.runs = runs;
  g.ntm = (int)ceil_div(M, 128);
  g.ntn = (int)ceil_div(N, 128);
  return launch<kKs, 128, 128, 2, 4, true>(A, B, g, (int64_t)runs.n * g.ntm * g.ntn, st);
}

}  // namespace sm
