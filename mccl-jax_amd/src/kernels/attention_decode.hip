// Attention forward for few queries (at most 16 per head, no causal mask)
// behind mk_sdpa_fwd: new tokens of running sequences against their key /
// value caches.
//
// Bound: HBM, one read of K and V.  A workgroup of 4 waves takes one head's
// keys, or one of `slices` runs of them where the heads alone would leave
// CUs idle; its waves take steps of 32 keys round-robin, several steps ahead
// in registers, with their own online softmax, and are merged through LDS.
// Slices leave (max, sum, O) in the workspace, merged by a second launch.
//
// Nothing is staged in LDS.  Per step and wave, with v_mfma_f32_16x16x32_bf16
// (lane l: c = l % 16, g = l / 16):
//   S^T = K Q^T: K rows are the first operand (row c of 16 keys, 8 d per
//     lane, one 16-byte load), queries the columns, so lane (c, g) ends with
//     query c's scores of keys 16 t + 4 g + r (t = 0, 1; r = 0 .. 3);
//   O^T += V^T P^T: those 8 probabilities, packed, are the lane's second
//     operand as they stand when k slot 8 g + 4 t + r means key 16 t + 4 g +
//     r.  The lane loads D / 16 consecutive d of the 8 V rows of its keys (16
//     lanes cover a row), and operand j pairs element j of two rows per word
//     (v_perm_b32): its row c is d = (D / 16) c + j.
// Scores, max, sum and O are fp32; probabilities are rounded to bf16 and the
// sum adds the rounded values, as in the other forward kernels, and the max
// is raised only when a score exceeds it by 2^8.
//
// Measured against the 128-query-tile kernel, 1 query, D 128, a call: B 8 x H 16
// x 4096 keys (268 MB) 83 -> 51 us, 47.5 of it this kernel (5.6 TB/s); B 1 x H
// 8 x 16384 keys 252 -> 22.6 us; B 32 x H 16 x 4096 keys, 4 queries (1.07 GB)
// 221 -> 173 us.
#include "attn_common.h"

#include <algorithm>

namespace mk {
namespace {

using namespace attn;

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kNW = 4;         // waves per workgroup (one per lane group g in the merge)
constexpr int kMaxQ = 16;      // queries per head
constexpr int kStepKeys = 32;

struct DecodeArgs {
  const uint16_t *q, *k, *v;
  uint16_t* o;
  float* lse;
  float* part;  // slices > 1: [head][slice] of Sq x (D values, max, sum)
  int64_t q_bs, q_hs, q_ss, k_bs, k_hs, k_ss, v_bs, v_hs, v_ss, o_bs, o_hs, o_ss;
  int H, Sq, Sk, slices, slice_keys;
  float scale_log2;
};

// what sums taken at max m are worth at max top (>= m); no score above -inf: 0
__device__ inline float weight(float m, float top) { return m == -INFINITY ? 0.f : exp2f(m - top); }

// one query's D outputs from weighted partial rows: out(i) = sum_w wt_w O_w[i]
// / l, thread-strided; shared by the in-workgroup and the slice merge
template <int D>
__device__ inline void store_out(const DecodeArgs& p, int bh, int q, int d, float o, float l, float m) {
  const int64_t at = int64_t(bh / p.H) * p.o_bs + int64_t(bh % p.H) * p.o_hs + int64_t(q) * p.o_ss;
  p.o[at + d] = f32_to_bf16(l > 0.f ? o / l : __builtin_nanf(""));
  if (p.lse && d == 0)
    p.lse[int64_t(bh) * p.Sq + q] = l > 0.f ? (m + log2f(l)) * 0.69314718055994531f : -INFINITY;
}

template <int D>
__global__ __launch_bounds__(64 * kNW, 2) void sdpa_decode_kernel(const DecodeArgs p) {
  constexpr int KK = D / 32;      // MFMAs over d per 16 keys
  constexpr int VJ = D / 16;      // d per lane of a V row
  constexpr int kD = D == 128 ? 2 : 3;  // steps in flight
  // rows of O 4 floats past a multiple of the banks: the 16 queries' lanes
  // write 16 bytes each to different ones
  __shared__ __attribute__((aligned(16))) float os[kNW][kMaxQ][D + 4];
  __shared__ float ms[kNW][kMaxQ], ls[kNW][kMaxQ], fs[kNW][kMaxQ], tops[kMaxQ];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int bh = blockIdx.x / p.slices, slice = blockIdx.x % p.slices;
  const int b = bh / p.H, h = bh % p.H;
  const int key_lo = slice * p.slice_keys, key_hi = min(key_lo + p.slice_keys, p.Sk);
  const uint16_t* kb = p.k + b * p.k_bs + h * p.k_hs + 8 * g;
  const uint16_t* vb = p.v + b * p.v_bs + h * p.v_hs + VJ * c;

  u32x4_t qf[KK];
  {
    const uint16_t* qr = p.q + b * p.q_bs + h * p.q_hs + int64_t(min(c, p.Sq - 1)) * p.q_ss + 8 * g;
#pragma unroll
    for (int i = 0; i < KK; ++i) qf[i] = *reinterpret_cast<const u32x4_t*>(qr + 32 * i);
  }
  struct Step {
    u32x4_t k[2][KK];
    uint32_t v[8][VJ / 2];
  };
  // rows past the last key repeat it; their probabilities are zero and
  // (in that step) their V rows are cleared
  auto load = [&](Step& s, int key0) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint16_t* kr = kb + int64_t(min(key0 + 16 * t + c, p.Sk - 1)) * p.k_ss;
#pragma unroll
      for (int i = 0; i < KK; ++i) s.k[t][i] = *reinterpret_cast<const u32x4_t*>(kr + 32 * i);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint16_t* vr = vb + int64_t(min(key0 + 16 * (u / 4) + 4 * g + u % 4, p.Sk - 1)) * p.v_ss;
      if constexpr (VJ == 8) {
        const u32x4_t w = *reinterpret_cast<const u32x4_t*>(vr);
#pragma unroll
        for (int e = 0; e < 4; ++e) s.v[u][e] = w[e];
      } else {
        const uint2 w = *reinterpret_cast<const uint2*>(vr);
        s.v[u][0] = w.x;
        s.v[u][1] = w.y;
      }
    }
  };
  f32x4_t acc[VJ] = {};
  float m = -INFINITY, l = 0.f;  // the max is -inf until a score above it is seen
  auto use = [&](Step& s, int key0) __attribute__((always_inline)) {
    float x[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4_t st = {};
#pragma unroll
      for (int i = 0; i < KK; ++i)
        st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(s.k[t][i]), as_bf16x8(qf[i]), st, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) x[4 * t + r] = st[r] * p.scale_log2;
    }
    if (key0 + kStepKeys > key_hi) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (key0 + 16 * (u / 4) + 4 * g + u % 4 >= key_hi) {
          x[u] = -INFINITY;
#pragma unroll
          for (int e = 0; e < VJ / 2; ++e) s.v[u][e] = 0;
        }
    }
    float top = x[0];
#pragma unroll
    for (int u = 1; u < 8; ++u) top = fmaxf(top, x[u]);
    if (__any(top > m + 8.f)) {
      float nm = fmaxf(m, top);
      nm = fmaxf(nm, __shfl_xor(nm, 16, 64));
      nm = fmaxf(nm, __shfl_xor(nm, 32, 64));
      const float f = weight(m, nm);
      m = nm;
      l *= f;
#pragma unroll
      for (int j = 0; j < VJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[j][r] *= f;
    }
    const float base = m == -INFINITY ? 0.f : m;
    float e[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) e[u] = __builtin_amdgcn_exp2f(x[u] - base);
    const bf16x8_t pr = pack8(e[0], e[1], e[2], e[3], e[4], e[5], e[6], e[7]);
    const u32x4_t pw = __builtin_bit_cast(u32x4_t, pr);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w = pw[i];
      l += __builtin_bit_cast(float, w << 16) + __builtin_bit_cast(float, w & 0xFFFF0000u);
    }
#pragma unroll
    for (int j = 0; j < VJ; ++j) {
      u32x4_t w;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        w[i] = __builtin_amdgcn_perm(s.v[2 * i + 1][j / 2], s.v[2 * i][j / 2], j % 2 ? 0x07060302u : 0x05040100u);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(w), pr, acc[j], 0, 0, 0);
    }
  };

  // this wave's steps; unconditional loads in the steady loop (a branch
  // around them would make the compiler wait for all of them at its head)
  const int steps = (key_hi - key_lo + kStepKeys - 1) / kStepKeys;
  const int n = steps > wave ? (steps - wave + kNW - 1) / kNW : 0;
  Step s[kD];
  auto key_of = [&](int i) { return key_lo + kStepKeys * (wave + kNW * i); };
  if (n >= kD) {
    int i = 0;
#pragma unroll
    for (int d = 0; d < kD; ++d) load(s[d], key_of(d));
    for (; i + 2 * kD <= n; i += kD) {
#pragma unroll
      for (int d = 0; d < kD; ++d) {
        use(s[d], key_of(i + d));
        load(s[d], key_of(i + kD + d));
      }
    }
#pragma unroll
    for (int d = 0; d < kD; ++d) {
      use(s[d], key_of(i + d));
      if (i + kD + d < n) load(s[d], key_of(i + kD + d));
    }
#pragma unroll
    for (int d = 0; d < kD; ++d)
      if (i + kD + d < n) use(s[d], key_of(i + kD + d));
  } else {
#pragma unroll
    for (int d = 0; d < kD - 1; ++d)
      if (d < n) load(s[d], key_of(d));
#pragma unroll
    for (int d = 0; d < kD - 1; ++d)
      if (d < n) use(s[d], key_of(d));
  }

  // acc[j] reg r of lane (c, g): query c, d = VJ (4 g + r) + j
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (c < p.Sq) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int j = 0; j < VJ; j += 4)
        *reinterpret_cast<f32x4_t*>(&os[wave][c][VJ * (4 * g + r) + j]) =
            f32x4_t{acc[j][r], acc[j + 1][r], acc[j + 2][r], acc[j + 3][r]};
    if (g == 0) ms[wave][c] = m, ls[wave][c] = l;
  }
  __syncthreads();
  // each wave's weight of each query, once
  if (wave == 0 && c < p.Sq) {
    float top = ms[0][c];
#pragma unroll
    for (int w = 1; w < kNW; ++w) top = fmaxf(top, ms[w][c]);
    fs[g][c] = weight(ms[g][c], top);
    if (g == 0) tops[c] = top;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < p.Sq * D; e += 64 * kNW) {
    const int q = e / D, d = e % D;
    const float top = tops[q];
    float o = 0.f, sum = 0.f;
#pragma unroll
    for (int w = 0; w < kNW; ++w) {
      o += fs[w][q] * os[w][q][d];
      sum += fs[w][q] * ls[w][q];
    }
    if (p.slices == 1) {
      store_out<D>(p, bh, q, d, o, sum, top);
    } else {
      float* row = p.part + (int64_t(blockIdx.x) * p.Sq + q) * (D + 2);
      row[d] = o;
      if (d == 0) row[D] = top, row[D + 1] = sum;
    }
  }
}

// the slices of each (head, query), in slice order
template <int D>
__global__ __launch_bounds__(D) void sdpa_decode_merge_kernel(const DecodeArgs p) {
  const int bh = blockIdx.x / p.Sq, q = blockIdx.x % p.Sq, d = threadIdx.x;
  const float* rows = p.part + (int64_t(bh) * p.slices * p.Sq + q) * (D + 2);
  const int64_t pitch = int64_t(p.Sq) * (D + 2);
  float top = rows[D];
#pragma unroll 4
  for (int s = 1; s < p.slices; ++s) top = fmaxf(top, rows[s * pitch + D]);
  float o = 0.f, sum = 0.f;
#pragma unroll 4
  for (int s = 0; s < p.slices; ++s) {
    const float f = weight(rows[s * pitch + D], top);
    o += f * rows[s * pitch + d];
    sum += f * rows[s * pitch + D + 1];
  }
  store_out<D>(p, bh, q, d, o, sum, top);
}

}  // namespace

// The 128-query-tile kernel keeps calls of few heads, one or two key steps and
// many queries' values to merge over the waves: D 128, 64 heads, 16 queries, 64
// keys 4.8 us there and 5.5 here (6.4 before the merge's padded rows and its
// weights computed once); 10 queries 4.9 and 5.0, 16 queries and 128 keys 6.5 and 6.1.
bool sdpa_decode_fits(int64_t BH, int64_t Sq, int64_t Sk, int64_t D, int causal) {
  return Sq <= kMaxQ && Sk >= 1 && !causal && !(BH <= 256 && Sk <= 64 && Sq * D > 1280);
}

int64_t sdpa_decode_slices(int64_t BH, int64_t Sk, int64_t D) {
  // Two workgroups of 4 waves per CU (256 CUs), each with at least 256 keys
  // (two steps per wave), where that gains more than the partial results and
  // the second launch cost, 2 - 6 us.  One run / cut, caches not in the L2s, us:
  // D 128, 64 heads x 1024 keys 15.0 / 11.6, 128 x 1024 16.8 / 17.3, 128 x 4096
  // 60.8 / 53.3, 170 x 2048 33.2 / 37.0, 256 x 1024 26.9 / 29.8 (16 queries 28.1 /
  // 33.0); D 64, 64 heads x 768 8.6 / 9.2.  More than 128 heads never gain.
  if (BH > 128 || Sk < (BH <= 64 ? (D == 128 ? 768 : 1024) : 16 * BH)) return 1;
  return std::max<int64_t>(1, std::min<int64_t>({512 / std::max<int64_t>(BH, 1), Sk / 256, 64}));
}

size_t sdpa_decode_workspace(int64_t BH, int64_t Sq, int64_t Sk, int64_t D) {
  const int64_t slices = sdpa_decode_slices(BH, Sk, D);
  return slices == 1 ? 0 : size_t(BH * slices * Sq * (D + 2) * 4);
}

int sdpa_decode(hipStream_t s, int64_t B, int64_t H, int64_t Sq, int64_t Sk, int64_t D,
                const void* q, int64_t q_bs, int64_t q_hs, int64_t q_ss,
                const void* k, int64_t k_bs, int64_t k_hs, int64_t k_ss,
                const void* v, int64_t v_bs, int64_t v_hs, int64_t v_ss,
                void* o, int64_t o_bs, int64_t o_hs, int64_t o_ss, float scale, float* lse, void* workspace) {
  const int64_t slices = workspace ? sdpa_decode_slices(B * H, Sk, D) : 1;
  const int64_t keys = ((Sk + slices - 1) / slices + kStepKeys - 1) / kStepKeys * kStepKeys;
  DecodeArgs a{(const uint16_t*)q, (const uint16_t*)k, (const uint16_t*)v, (uint16_t*)o, lse, (float*)workspace,
               q_bs, q_hs, q_ss, k_bs, k_hs, k_ss, v_bs, v_hs, v_ss, o_bs, o_hs, o_ss,
               int(H), int(Sq), int(Sk), int((Sk + keys - 1) / keys), int(keys), scale * 1.4426950408889634f};
  const dim3 g{unsigned(B * H * a.slices)};
  if (D == 128) hipLaunchKernelGGL((sdpa_decode_kernel<128>), g, dim3(64 * kNW), 0, s, a);
  else hipLaunchKernelGGL((sdpa_decode_kernel<64>), g, dim3(64 * kNW), 0, s, a);
  if (a.slices > 1) {
    const dim3 gm{unsigned(B * H * Sq)};
    if (D == 128) hipLaunchKernelGGL((sdpa_decode_merge_kernel<128>), gm, dim3(128), 0, s, a);
    else hipLaunchKernelGGL((sdpa_decode_merge_kernel<64>), gm, dim3(64), 0, s, a);
  }
  return check_launch("mk_sdpa_fwd");
}

}  // namespace mk
