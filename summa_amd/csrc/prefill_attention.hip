// Causal flash attention for prefill and log-prob recompute (16-bit MFMA;
// q and cache bf16 or f16).
//
// Semantics: Transformer full-sequence attention (sdpa with causal mask,
// summa-llm/src/model/attention.rs:216-298; CubeK flash forward
// cube_attention.rs:127-220): query row r of sequence s sits at absolute
// position pos0[s] + r and attends keys 0..=pos0[s]+r of the cache, scale
// 1/sqrt(hd), GQA head h -> KV head h / (H/KVH).
//
// Tiling: one workgroup per (128 query rows, head, sequence), 4 waves x 32 query
// rows, two workgroups per CU. 64-key tiles of K [64][hd] and V transposed
// [hd][64] sit in two LDS buffers (rows padded by 8 elements: the 16-byte
// fragment reads of 32 rows spread over all banks); the next tile's global loads
// go out into registers before the current tile's math and are stored to the
// other buffer after it, one barrier per tile.
// The tile math is transposed so that each lane owns one query, and P never
// leaves the registers:
//   S^T = K.Q^T  (v_mfma_f32_32x32x16_{bf16,f16}; A = K rows from LDS, B = the
//                 wave's Q fragments, kept in registers for the whole sweep):
//                 lane (j, h) receives keys 8 i + 4 h + 0..3 of query j;
//   softmax      running max / sum per lane in raw-score units, the scale folded
//                into one FMA before exp2; the max crosses lanes by one shuffle
//                (lanes j, j + 32), the sum once after the sweep; the causal mask
//                runs on the diagonal tiles only;
//   O^T += V^T.P^T  P as an f16 pair (hi + lo, ~21 significant bits), two f16
//                MFMAs per 16 keys. The order of the contraction is free, so a
//                lane's eight scores of 16 keys are its B operand as they are,
//                and V^T is stored with each 16 keys in that order (0-3, 8-11,
//                4-7, 12-15); V is f16 as stored, or bf16 -> f16 while staging
//                (exact for |v| < 65504 and above the f16 subnormal range).
//                Lane (j, h) accumulates dims 8 i + 4 h + 0..3 of query j, so
//                rescaling needs no cross-lane traffic and stores are 8 bytes.
// The workgroups that share K and V (a KV head's query heads and row tiles) are
// consecutive on one XCD where there are KV heads for all of them (prefill_map.hpp).
// 16-query waves on the 16 x 16 x 32 form read every K and V fragment for half as
// many queries and passed P through LDS: bf16, 32 x 512, 16 / 4 heads of 128: 130 ->
// 94 us; 64 x 1024 974 -> 644; 128 x 383, 12 heads of 64 137 -> 105.
// A wave skips the key tiles past its last row's position (fully masked for
// it). Without the causal mask (AttentionBackend::attention_inner with
// causal = false) every query attends keys 0..L-1. q and out are addressed
// through element strides (sequence, position, head), so the same kernel
// serves the model's [S, L, H, hd] rows and the reference's [B, H, S, hd]
// tensors. The f16 pair keeps P.V at fp32-like precision, so the prefill path
// matches the decode path's fp32 probabilities; a single bf16 or f16 P costs
// measurable log-prob accuracy.
#include <algorithm>
#include <cmath>

#include "attn_common.hpp"
#include "common.hpp"
#include "prefill_map.hpp"

namespace sm {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <bool KF16>
__device__ inline f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (KF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8, a),
                                                  __builtin_bit_cast(h8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a),
                                                   __builtin_bit_cast(bf8, b), c, 0, 0, 0);
}

constexpr int kRows = 128;  // query rows per workgroup

template <int HD, bool KF16, int OM>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ kc,
    const uint16_t* __restrict__ vc, const int32_t* __restrict__ pos0,
    void* __restrict__ out, float* __restrict__ lse, int S, int L, int H, int KVH, int cap,
    float scale, AttnStrides qs, AttnStrides os, int causal, int nqt) {
  constexpr int KS = HD / 16, DB = HD / 32;  // MFMA steps of a score, 32-dim blocks of O
  constexpr int KP = HD + 8, VP = 64 + 8;    // padded LDS rows (elements)
  constexpr int CH = HD / 8;                 // 16-byte chunks per key row
  constexpr int KPT = 64 * CH / 256;         // K chunks per thread
  constexpr int VU = 16 * CH;                // V units: 4 keys x 8 dims
  constexpr int VPT = (VU + 255) / 256;
  __shared__ __attribute__((aligned(16))) uint16_t ks[2][64 * KP];
  __shared__ __attribute__((aligned(16))) _Float16 vts[2][HD * VP];

  // the row tiles with the most keys first
  const int rep = H / KVH;
  const PrefillMap map((uint32_t)S * KVH, (uint32_t)rep * nqt);
  uint32_t grp, place;
  if (!map.at(blockIdx.y * gridDim.x + blockIdx.x, grp, place)) return;  // (uniform)
  const int s = (int)(grp / KVH), kvh = (int)(grp % KVH);
  const int qt = nqt - 1 - (int)(place / rep), h = kvh * rep + (int)(place % rep);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int j = lane % 32, hf = lane / 32;
  const int p0 = pos0 ? pos0[s] : 0;
  const int r0 = qt * kRows + wave * 32;  // first query row of this wave
  const size_t kv_base = ((size_t)s * KVH + kvh) * cap * HD;

  // Q fragments (B operand): lane (query j, half hf)
  u32x4 qa[KS];
#pragma unroll
  for (int st = 0; st < KS; ++st)
    qa[st] = r0 + j < L
                 ? *reinterpret_cast<const u32x4*>(q + qs.at(s, r0 + j, h) + st * 16 + hf * 8)
                 : u32x4{0u, 0u, 0u, 0u};
  f32x16 o[DB];  // o[d][e]: query j, dim 32 d + 8 (e / 4) + 4 hf + e % 4
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int e = 0; e < 16; ++e) o[d][e] = 0.f;
  float m = -INFINITY, l = 0.f;  // running max; this lane's part of the sum
  const float c2 = scale * 1.44269504088896340736f;  // scale * log2(e)
  const int qpos = p0 + r0 + j;                       // this lane's query position

  const int last_row = min(qt * kRows + kRows - 1, L - 1);
  // keys [0, kend) needed by this workgroup (all L of them without the mask)
  const int kend = causal ? p0 + last_row + 1 : L;
  // keys this wave attends to: [0, p0 + its last row]; later tiles are fully
  // masked for it (they would leave m, l and o bit-for-bit unchanged) and skipped
  const int wave_kmax = (r0 < L) ? (causal ? p0 + min(r0 + 31, L - 1) : L - 1) : -1;

  u32x4 kreg[KPT], vreg[VPT][4];
  auto load_tile = [&](int kt) {
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int c = i * 256 + threadIdx.x, key = kt + c / CH;
      kreg[i] = u32x4{0u, 0u, 0u, 0u};
      if (key < kend && key < cap)
        kreg[i] = *reinterpret_cast<const u32x4*>(kc + kv_base + (size_t)key * HD + (c % CH) * 8);
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int u = i * 256 + threadIdx.x;
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const int key = kt + 4 * (u % 16) + y;
        vreg[i][y] = u32x4{0u, 0u, 0u, 0u};
        if (u < VU && key < kend && key < cap)
          vreg[i][y] = *reinterpret_cast<const u32x4*>(vc + kv_base + (size_t)key * HD +
                                                       (u / 16) * 8);
      }
    }
  };
  auto store_tile = [&](int buf) {
#pragma unroll
    for (int i = 0; i < KPT; ++i) {
      const int c = i * 256 + threadIdx.x;
      *reinterpret_cast<u32x4*>(&ks[buf][(c / CH) * KP + (c % CH) * 8]) = kreg[i];
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int u = i * 256 + threadIdx.x;
      if (u >= VU) continue;
      // keys 4 kq .. + 3: quarter kq % 4 of its 16 keys, stored as quarter 0, 2, 1, 3
      const int kq = u % 16, at = 16 * (kq / 4) + 8 * (kq % 2) + 4 * (kq % 4 / 2);
      float f[4][8];
#pragma unroll
      for (int y = 0; y < 4; ++y) unpack8<KF16>(vreg[i][y], f[y]);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        *reinterpret_cast<h4*>(&vts[buf][((u / 16) * 8 + e) * VP + at]) =
            h4{(_Float16)f[0][e], (_Float16)f[1][e], (_Float16)f[2][e], (_Float16)f[3][e]};
    }
  };

  load_tile(0);
  store_tile(0);
  __syncthreads();
  for (int kt = 0, buf = 0; kt < kend; kt += 64, buf ^= 1) {
    const bool more = kt + 64 < kend;
    if (more) load_tile(kt + 64);
    if (kt <= wave_kmax) {  // uniform per wave
      f32x16 sc[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[kb][e] = 0.f;
#pragma unroll
        for (int st = 0; st < KS; ++st) {
          const u32x4 kf = *reinterpret_cast<const u32x4*>(
              &ks[buf][(kb * 32 + j) * KP + st * 16 + hf * 8]);
          sc[kb] = mfma32<KF16>(kf, qa[st], sc[kb]);
        }
      }
      // causal mask (only tiles that reach past the wave's first query)
      if (kt + 63 > (causal ? p0 + r0 : L - 1)) {
        const int lim = (causal ? qpos : L - 1) - kt - 4 * hf;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int e = 0; e < 16; ++e)
            if (kb * 32 + 8 * (e / 4) + e % 4 > lim) sc[kb][e] = -INFINITY;
      }
      // online softmax of query j (32 keys here, 32 in lane j + 32)
      float mx = sc[0][0];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sc[kb][e]);
      mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
      const float mnew = fmaxf(m, mx);  // finite: key 0 <= every query position
      const float alpha = __builtin_amdgcn_exp2f((m - mnew) * c2);
      const float mc = mnew * c2;
      float sum = 0.f;
      u32x4 ph[2][2], pl[2][2];  // P^T of 16 keys each, hi and lo
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {  // (pairs: one packed conversion each for hi and lo)
            f32x2_t p;
#pragma unroll
            for (int y = 0; y < 2; ++y) {
              p[y] = __builtin_amdgcn_exp2f(fmaf(sc[kb][8 * i + 2 * e + y], c2, -mc));
              sum += p[y];
            }
            const h2 x = __builtin_convertvector(p, h2);
            const f32x2_t r = {p[0] - (float)x[0], p[1] - (float)x[1]};
            ph[kb][i][e] = __builtin_bit_cast(uint32_t, x);
            pl[kb][i][e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, h2));
          }
        }
      l = l * alpha + sum;
      m = mnew;
      if (__ballot(alpha != 1.f)) {  // a factor of 1 would leave O unchanged
#pragma unroll
        for (int d = 0; d < DB; ++d)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[d][e] *= alpha;
      }
      // O^T += V^T P^T, 16 keys at a time
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int d = 0; d < DB; ++d) {
            const u32x4 vb = *reinterpret_cast<const u32x4*>(
                &vts[buf][(d * 32 + j) * VP + kb * 32 + i * 16 + hf * 8]);
            o[d] = mfma32<true>(vb, ph[kb][i], o[d]);
            o[d] = mfma32<true>(vb, pl[kb][i], o[d]);
          }
    }
    if (more) store_tile(buf ^ 1);  // last read before the previous barrier
    __syncthreads();
  }
  const int row = r0 + j;
  l += __shfl_xor(l, 32, kWave);
  if (row >= L) return;
  // log-sum-exp of the scaled, masked scores, [S*H, L] (fused_attention.rs:166-172)
  if (lse && hf == 0) lse[((size_t)s * H + h) * L + row] = m * scale + logf(l);
  const float inv = 1.f / l;
  const size_t orow = (size_t)s * L + row;  // f16-pair rows: [S * L, 2 * H * hd]
  const int width = H * HD;
  const size_t obase = os.at(s, row, h);
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int dim = d * 32 + 8 * i + 4 * hf;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = o[d][4 * i + e] * inv;
      if constexpr (OM == 2) {
        h4 hi, lo;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          _Float16 x, y;
          split_f16(v[e], x, y);
          hi[e] = x;
          lo[e] = y;
        }
        _Float16* base = static_cast<_Float16*>(out) + orow * 2 * width + h * HD + dim;
        *reinterpret_cast<h4*>(base) = hi;
        *reinterpret_cast<h4*>(base + width) = lo;
      } else if constexpr (OM == 1) {
        *reinterpret_cast<h4*>(static_cast<_Float16*>(out) + obase + dim) =
            h4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
      } else {
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + obase + dim) =
            uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
    }
}

}  // namespace

int attn_prefill_16(const uint16_t* q, const uint16_t* kc, const uint16_t* vc,
                    const int32_t* pos0, void* out, float* lse, bool kf16, int om, int S, int L,
                    int H, int KVH, int cap, int hd, hipStream_t st, const AttnStrides* qs_in,
                    const AttnStrides* os_in, bool causal) {
  if (S > 65535 || H > 65535) {
    set_error("sm_attn_prefill: S and H must be <= 65535");
    return SM_ERR_UNSUPPORTED;
  }
  const int64_t nqt = ceil_div(L, kRows);
  const int64_t most = (int64_t)1 << 31;
  int64_t wgs = most;
  if ((int64_t)S * KVH < most && (H / KVH) * nqt < most)
    wgs = PrefillMap((uint32_t)S * KVH, (uint32_t)(H / KVH) * nqt).workgroups();
  // (a grid dimension holds less than 2^24 workgroups of 256 threads)
  const int64_t wide = std::min<int64_t>(wgs, (int64_t)1 << 23), tall = ceil_div(wgs, wide);
  if (wgs >= most) {
    set_error("sm_attn_prefill: problem too large");
    return SM_ERR_UNSUPPORTED;
  }
  const dim3 grid((unsigned)wide, (unsigned)tall);
  const float scale = 1.0f / sqrtf((float)hd);
  const AttnStrides rows = AttnStrides::rows(L, H, hd);  // [S, L, H, hd]
  const AttnStrides qs = qs_in ? *qs_in : rows, os = os_in ? *os_in : rows;
  const int cz = causal ? 1 : 0;
#define SM_PF3(HD, KF, OM)                                                                \
  attn_prefill_kernel<HD, KF, OM><<<grid, 256, 0, st>>>(q, kc, vc, pos0, out, lse, S, L, H, KVH, \
                                                        cap, scale, qs, os, cz, (int)nqt)
#define SM_PF2(HD, KF)                          \
  do {                                          \
    if (om == 2) SM_PF3(HD, KF, 2);             \
    else if (om == 1) SM_PF3(HD, KF, 1);        \
    else SM_PF3(HD, KF, 0);                     \
  } while (0)
#define SM_PF(HD)                               \
  do {                                          \
    if (kf16) SM_PF2(HD, true);                 \
    else SM_PF2(HD, false);                     \
  } while (0)
  if (hd == 64) SM_PF(64);
  else SM_PF(128);
#undef SM_PF
#undef SM_PF2
#undef SM_PF3
  SM_LAUNCH_CHECK();
  return SM_OK;
}

}  // namespace sm
