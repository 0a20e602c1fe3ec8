// GEMM with few rows (M <= 64) behind mk_gemm: a layer of a model applied to
// a few tokens, where reading B (the weights) once is the work.
//   C[b] = A[b] · B[b] (+ bias)(ReLU), bf16 or fp32 operands, fp32 accumulate.
//
// Bound: HBM, K N elements of B.  A workgroup owns NT = 16 VN columns of C
// and all M rows; its NW waves take the k axis in steps of 32, round-robin,
// so a workgroup reads one stretch of B at a time, several steps ahead per
// wave, and no two workgroups read the same part of B.  The waves' sums are
// added through LDS in wave order (deterministic).
//
// One CU takes in about one line every 8 clocks from HBM whatever the loads'
// width (a probe with this access pattern: 35 GB/s per CU with 128-byte rows,
// 17.6 with 64-byte ones), so N / 64 workgroups below the 256 CUs cannot
// reach the chip's rate; the split-K entry then also cuts k over workgroups
// (W slices of fp32 partial sums, added in slice order by splitk_sum).
//
// B goes from memory straight into the registers the MFMA reads, in either
// orientation.  A lane (c, g) of v_mfma_f32_16x16x32_bf16 supplies column c
// and k = 8 g .. 8 g + 7:
//   k-contiguous (B stored as [n][k]): MFMA j takes column n0 + 16 j + c, one
//     load of 8 k;
//   n-contiguous: the lane loads VN consecutive columns n0 + VN c .. of 8
//     k-rows and MFMA j takes column n0 + VN c + j, which is a permutation of
//     the tile's columns; pairing two k of a column is one v_perm_b32.  A row
//     of the tile is 128 bytes (bf16) or 128 / 256 (fp32): whole lines.
// fp32 operands use v_mfma_f32_16x16x4_f32, one k per lane, with the k of a
// step dealt the same way (lane group g: k = 8 g + u in MFMA u), so A's 8 k
// are contiguous too.  Loads need element alignment only.
//
// Measured against the 128 x 128-tile kernel, which runs N / 128 workgroups
// and pads M to 128, at 16 x 4096 x 16384 and 16 x 16384 x 4096 bf16 (M x K x
// N; one MLP, 268 MB of weights): 100 and 377 us -> 27.4 (4.9 TB/s) and 28.3 +
// 3.9 us for the sum of 4 slices (72 us unsliced).
#include "mk_common.h"

#include <algorithm>
#include <type_traits>

namespace mk {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kKU = 8, kKS = 32;  // k per lane and step, k per step

struct SkinnyArgs {
  const void* A;
  const void* B;
  void* C;
  const void* bias;
  int64_t M, N, K;
  int64_t a_bs, a_ms, b_bs, b_rs, b_cs, c_bs, c_ms;  // B element (k, n): k * b_rs + n * b_cs
  int epilogue;
  int c_type;
  int slices;  // > 1: workgroup row blockIdx.y takes every slices-th step of k and writes C + blockIdx.y * c_bs
};

// W 32-bit words from an element-aligned address
template <typename T, int W>
__device__ inline void load_words(const T* p, uint32_t (&w)[W]) {
  struct __attribute__((packed, aligned(sizeof(T)))) Pack { uint32_t w[W]; };
  const Pack q = *reinterpret_cast<const Pack*>(p);
#pragma unroll
  for (int i = 0; i < W; ++i) w[i] = q.w[i];
}
// elements 0 .. n - 1 of a run of 32-bit words' worth, zeros past them
template <typename T, int W>
__device__ inline void load_words_upto(const T* p, int64_t n, uint32_t (&w)[W]) {
  constexpr int E = W * 4 / int(sizeof(T));
  T e[E];
#pragma unroll
  for (int i = 0; i < E; ++i) e[i] = i < n ? p[i] : T(0);
  __builtin_memcpy(w, e, sizeof(w));
}

template <typename T, bool B_KC, int VN, int MT, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_skinny_kernel(const SkinnyArgs p) {
  constexpr int NT = 16 * VN;
  constexpr int WK = kKU * int(sizeof(T)) / 4;  // words of 8 k
  constexpr int WN = VN * int(sizeof(T)) / 4;   // words of VN columns
  static_assert(B_KC || WN > 0, "whole words of columns");
  __shared__ __attribute__((aligned(16))) float red[NW][16][NT];
  const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, g = lane >> 4;
  const int64_t n0 = int64_t(blockIdx.x) * NT;
  const int64_t bz = p.slices > 1 ? 0 : blockIdx.y, slice = p.slices > 1 ? blockIdx.y : 0;
  const T* A = reinterpret_cast<const T*>(p.A) + bz * p.a_bs + kKU * g;
  const T* B = reinterpret_cast<const T*>(p.B) + bz * p.b_bs + kKU * g * p.b_rs;
  // rows past M repeat row M - 1 and are not stored
  const T* ap[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int64_t row = 16 * m + c;
    ap[m] = A + (row < p.M ? row : p.M - 1) * p.a_ms;
  }
  // columns past N: an n-contiguous lane whose columns cross N takes the last
  // VN columns (the ones it repeats are computed from the same values in the
  // same order), a k-contiguous one repeats column N - 1
  const T* bp[B_KC ? VN : 1];
  if constexpr (B_KC) {
#pragma unroll
    for (int j = 0; j < VN; ++j) {
      const int64_t n = n0 + 16 * j + c;
      bp[j] = B + (n < p.N ? n : p.N - 1) * p.b_cs;
    }
  } else {
    const int64_t n = n0 + VN * c;
    bp[0] = B + (n + VN <= p.N ? n : p.N - VN);
  }

  struct Step {
    uint32_t a[MT][WK];
    uint32_t b[B_KC ? VN : kKU][B_KC ? WK : (WN > 0 ? WN : 1)];
  };
  auto load = [&](Step& s, int64_t step) __attribute__((always_inline)) {
    const int64_t k0 = step * kKS;
    if constexpr (B_KC) {
#pragma unroll
      for (int j = 0; j < VN; ++j) load_words(bp[j] + k0, s.b[j]);
    } else {
#pragma unroll
      for (int u = 0; u < kKU; ++u) load_words(bp[0] + (k0 + u) * p.b_rs, s.b[u]);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) load_words(ap[m] + k0, s.a[m]);
  };
  f32x4_t acc[MT][VN] = {};
  auto multiply = [&](const Step& s) __attribute__((always_inline)) {
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int j = 0; j < VN; ++j) {
        u32x4_t w;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if constexpr (B_KC) w[q] = s.b[j][q];
          else w[q] = __builtin_amdgcn_perm(s.b[2 * q + 1][j / 2], s.b[2 * q][j / 2], j % 2 ? 0x07060302u : 0x05040100u);
        }
        const bf16x8_t bj = __builtin_bit_cast(bf16x8_t, w);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          const u32x4_t a = {s.a[m][0], s.a[m][1], s.a[m][2], s.a[m][3]};
          acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), bj, acc[m][j], 0, 0, 0);
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < kKU; ++u)
#pragma unroll
        for (int j = 0; j < VN; ++j) {
          const uint32_t w = B_KC ? s.b[j][B_KC ? u : 0] : s.b[B_KC ? 0 : u][B_KC ? 0 : j];
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const uint32_t a = s.a[m][u];
            acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, a), __builtin_bit_cast(float, w),
                                                            acc[m][j], 0, 0, 0);
          }
        }
    }
  };

  // kD steps in flight per wave.  The loop's loads are unconditional: with a
  // branch around them the compiler waits for every load at the loop head.
  constexpr int kWords = int(sizeof(Step)) / 4, kFit = (NW == 16 ? 64 : 112) / kWords;
  constexpr int kD = kFit < 2 ? 2 : kFit > 6 ? 6 : kFit;
  const int64_t full = p.K / kKS;
  const int64_t first = wave + NW * slice, pace = NW * p.slices;   // this wave's steps
  const int64_t n = full > first ? (full - first + pace - 1) / pace : 0;
  Step s[kD];
  auto fetch = [&](int d, int64_t i) __attribute__((always_inline)) { load(s[d], first + pace * i); };
  if (n >= kD) {
    int64_t i = 0;
#pragma unroll
    for (int d = 0; d < kD; ++d) fetch(d, d);
    for (; i + 2 * kD <= n; i += kD) {
#pragma unroll
      for (int d = 0; d < kD; ++d) {
        multiply(s[d]);
        fetch(d, i + kD + d);
      }
    }
#pragma unroll
    for (int d = 0; d < kD; ++d) {
      multiply(s[d]);
      if (i + kD + d < n) fetch(d, i + kD + d);
    }
#pragma unroll
    for (int d = 0; d < kD; ++d)
      if (i + kD + d < n) multiply(s[d]);
  } else {
#pragma unroll
    for (int d = 0; d < kD - 1; ++d)
      if (d < n) fetch(d, d);
#pragma unroll
    for (int d = 0; d < kD - 1; ++d)
      if (d < n) multiply(s[d]);
  }
  // the last K % 32: zeros past K in both operands
  if (p.K % kKS != 0 && full % pace == first) {
    const int64_t k0 = full * kKS, left = p.K - k0 - kKU * g;  // of this lane's 8 k (may be <= 0)
    if constexpr (B_KC) {
#pragma unroll
      for (int j = 0; j < VN; ++j) load_words_upto(bp[j] + k0, left, s[0].b[j]);
    } else {
#pragma unroll
      for (int u = 0; u < kKU; ++u) {
#pragma unroll
        for (int w = 0; w < WN; ++w) s[0].b[u][w] = 0;
        if (u < left) load_words(bp[0] + (k0 + u) * p.b_rs, s[0].b[u]);
      }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) load_words_upto(ap[m] + k0, left, s[0].a[m]);
    multiply(s[0]);
  }

  // acc[m][j] reg r: row 16 m + 4 g + r, the column that lane c's operand j
  // held: LDS column 16 j + c (k-contiguous) or VN c + j
  char* C = reinterpret_cast<char*>(p.C);
  const int64_t c_at = int64_t(blockIdx.y) * p.c_bs;
  for (int m = 0; m < MT; ++m) {
    if (m > 0) __syncthreads();
#pragma unroll
    for (int mm = 0; mm < MT; ++mm) {
      if (mm != m) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int j = 0; j < VN; ++j) red[wave][4 * g + r][B_KC ? 16 * j + c : VN * c + j] = acc[mm][j][r];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * NT; e += 64 * NW) {
      const int row = e / NT, col = e % NT;
      float v = red[0][row][col];
#pragma unroll
      for (int w = 1; w < NW; ++w) v += red[w][row][col];
      int64_t n = n0 + col;
      bool live = n < p.N;
      if constexpr (!B_KC) {
        const int64_t lane_n = n0 + col / VN * VN;  // the lane's columns, moved back where they crossed N
        live = lane_n < p.N;
        if (lane_n + VN > p.N) n = p.N - VN + col % VN;
      }
      const int64_t mrow = 16 * m + row;
      if (!live || mrow >= p.M) continue;
      if (p.epilogue != 0) v += load_as_f32(p.bias, n, (p.epilogue & 4) ? MK_F32 : p.c_type);
      if ((p.epilogue & 3) == 2) v = fmaxf(v, 0.f);
      store_from_f32(C, c_at + mrow * p.c_ms + n, p.c_type, v);
    }
  }
}

template <int V> using Int = std::integral_constant<int, V>;

template <typename T, bool B_KC, int VN>
void launch(hipStream_t s, const SkinnyArgs& a, int64_t batch) {
  const dim3 grid{unsigned((a.N + 16 * VN - 1) / (16 * VN)), unsigned(batch)};
  auto go = [&](auto mt) {
    constexpr int MT = decltype(mt)::value;
    // sixteen waves where two steps in flight and the accumulators fit 128 registers, else eight
    constexpr int NW = MT == 1 && VN * sizeof(T) <= 8 ? 16 : 8;
    hipLaunchKernelGGL((gemm_skinny_kernel<T, B_KC, VN, MT, NW>), grid, dim3(64 * NW), 0, s, a);
  };
  if (a.M <= 16) go(Int<1>{});
  else if (a.M <= 32) go(Int<2>{});
  else go(Int<4>{});
}

}  // namespace

// N: a workgroup of 1024 threads per 64 columns, and HIP refuses grids of 2^32
// threads
bool gemm_skinny_fits(int64_t M, int64_t N, int64_t K, int64_t a_ks, int64_t b_ks, int64_t b_ns) {
  return M <= 64 && N >= 16 && N <= (int64_t(1) << 27) && K >= 1 && a_ks == 1 && (b_ks == 1 || b_ns == 1);
}

bool gemm_skinny_pays(int ab_type, int64_t batch, int64_t M, int64_t N, int64_t K, bool b_kc, bool b_aligned) {
  // A workgroup of this kernel fills a CU and takes 2 - 5 us however short k
  // is (the first loads, the waves' sums through LDS: MT 16-row blocks of
  // them), so it pays where its workgroups are few or k is long.  Up to one
  // workgroup of either kernel per CU it is always ahead, but for 33 - 64 rows
  // at k of a few steps.  Past that the two were timed on 3000 products
  // (batches up to 4096, 16 - 131072 columns, k 8 - 4096): the least k from
  // which this kernel is no slower grows with MT, is shorter where the general
  // kernel's last 128-column tile is half empty, and is longer where that
  // kernel is at its best, k-contiguous bf16 on the 16-byte grid.  4096 x 64 x
  // 8 x 512 (batch x M x K x N), bf16: general 313 us, this kernel 608; 4096 x
  // 64 x 128 x 128 k-contiguous 90 and 163; 512 x 64 x 512 x 64: 38 and 20.
  const int64_t tiles = (N + 127) / 128 * batch, mine = (N + 63) / 64 * batch, mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  if (mine <= 256) return true;
  if (tiles <= 256) return K >= 32 * mt;
  const bool half = 2 * mine < 3 * tiles;
  if (ab_type != MK_BF16) return K >= (!b_aligned ? 32 : half ? 16 : b_kc ? 96 : 64) * mt;
  if (!b_aligned) return K >= (b_kc ? 96 : 32) * mt;
  return K >= (b_kc ? (half ? 128 : 2048) : (half ? 64 : 256)) * mt;
}

int64_t gemm_skinny_slices(int ab_type, int64_t M, int64_t N, int64_t K, bool b_kc, int64_t most) {
  // A workgroup's time is its lines at 8 clocks each, one 128-byte line per
  // k-row of bf16, two of fp32; the slices' second pass costs about 4 us.  Timed
  // on 1000 products, in one launch and in slices: slices gain from 2048 lines
  // on (16 x 2048 x 768 bf16: 9.0 -> 7.1 us, 16 x 16384 x 4096: 47.9 -> 26.3), but
  // not where only two find CUs, unless a workgroup's rows are many (n-contiguous
  // 16 x 2048 x 6000: 10.8 -> 12.1), and with at most 16 rows of k-contiguous B only
  // from 4096 lines below 2560 columns: its 16-column workgroups fill the chip
  // alone (1 x 4096 x 4096: 8.6 -> 10.5).
  const int64_t tiles = (N + 63) / 64, lines = ab_type == MK_BF16 ? K : 2 * K;
  const bool few = M <= 16;
  if (tiles >= (b_kc ? (few ? 40 : 192) : (ab_type == MK_BF16 && !few ? 192 : 86))) return 1;
  if (lines < (b_kc && few ? 4096 : 2048)) return 1;
  return std::max<int64_t>(1, std::min({most, 256 / tiles, K / 512, int64_t(16)}));
}

int gemm_skinny(hipStream_t s, int ab_type, int c_type, int64_t batch, int64_t M, int64_t N, int64_t K,
                const void* A, int64_t a_bs, int64_t a_ms, int64_t a_ks, const void* B, int64_t b_bs, int64_t b_ks,
                int64_t b_ns, void* C, int64_t c_bs, int64_t c_ms, const void* bias, int epilogue, int64_t slices) {
  if (!gemm_skinny_fits(M, N, K, a_ks, b_ks, b_ns)) return -1;
  const bool kc = b_ks == 1;
  SkinnyArgs a{A, B, C, bias, M, N, K, a_bs, a_ms, b_bs, b_ks, b_ns, c_bs, c_ms, epilogue, c_type, int(slices)};
  // 64 columns per workgroup where that fills the chip's 256 CUs; fewer where
  // it does not, as far as a row of the tile stays whole lines
  const bool wide = (N + 63) / 64 * batch * slices >= 192;
  const int64_t rows = slices > 1 ? slices : batch;
  if (ab_type == MK_BF16) {
    if (kc) wide ? launch<uint16_t, true, 4>(s, a, rows) : launch<uint16_t, true, 1>(s, a, rows);
    else launch<uint16_t, false, 4>(s, a, rows);
  } else {
    if (kc) wide ? launch<float, true, 4>(s, a, rows) : launch<float, true, 1>(s, a, rows);
    else wide ? launch<float, false, 4>(s, a, rows) : launch<float, false, 2>(s, a, rows);
  }
  return check_launch("mk_gemm");
}

}  // namespace mk
