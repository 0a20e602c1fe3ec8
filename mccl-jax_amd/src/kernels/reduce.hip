// Row-wise reductions over the innermost axis: reduce (sum/max/min/prod),
// fused max+argmax (bit-exact), LayerNorm and softmax.
//
// Layout: x is [rows, cols] row-major.  One wave64 owns one row; each lane
// reads 16-byte vectors (8 bf16 / 4 fp32) so a 2 KiB bf16 row is exactly two
// dwordx4 loads per lane and every HBM line is fully used.  Cross-lane
// combination is a 6-step butterfly.  Rows never interact, so the grid is
// rows/4 workgroups of 4 waves — tens of thousands of waves for 65536 rows,
// enough to keep all 256 CUs streaming.  Few or long rows take 4 or 16 waves
// each (team_waves).
#include "mk_common.h"

#include <algorithm>
#include <type_traits>
#include <cmath>

namespace mk {
namespace {

constexpr int kWavesPerBlock = 4;
constexpr int kBlock = kWavesPerBlock * kWave;

template <typename T> struct Vec;
template <> struct Vec<uint16_t> { static constexpr int N = 8; using V = u16x8; };
template <> struct Vec<float> { static constexpr int N = 4; using V = f32x4; };

template <typename T> __device__ inline float to_f32(T v);
template <> __device__ inline float to_f32<float>(float v) { return v; }
template <> __device__ inline float to_f32<uint16_t>(uint16_t v) { return bf16_to_f32(v); }

// Input element types handled by the templated row kernels: bf16 (uint16_t
// bits, IS_F16=false), f16 (uint16_t bits, IS_F16=true) and f32.
template <typename T, bool IS_F16>
__device__ inline float ld(T v) {
  if constexpr (IS_F16) return f16_to_f32(v);
  else return to_f32<T>(v);
}

template <int OP> __device__ inline float combine(float a, float b) {
  if constexpr (OP == 0) return a + b;
  else if constexpr (OP == 1) return fmaxf(a, b);
  else if constexpr (OP == 2) return fminf(a, b);
  else return a * b;
}
template <int OP> __device__ inline float wave_combine(float v) {
  if constexpr (OP == 0) return wave_sum(v);
  else if constexpr (OP == 1) return wave_max(v);
  else if constexpr (OP == 2) return wave_min(v);
  else return wave_prod(v);
}
template <int OP> __device__ inline float identity() {
  if constexpr (OP == 0) return 0.f;
  else if constexpr (OP == 1) return -INFINITY;
  else if constexpr (OP == 2) return INFINITY;
  else return 1.f;
}

// A row of any length at any element-aligned address, shared by the W waves
// of a team (W = 1: four rows per 256-thread workgroup; W = 4, 16: one row
// per workgroup): 16-byte vectors t, t + 64 W, ... for team lane t, then the
// up to N - 1 elements past the last whole vector, one per lane.  A row of
// odd length starts off the 16-byte grid; the vector loads need element
// alignment only (global accesses of any alignment are one instruction on
// gfx950), so such rows keep the full load width.
template <typename T> struct __attribute__((packed, aligned(sizeof(T)))) Unaligned16 { u32x4_t v; };
template <typename T> __device__ inline u32x4_t ld_row(const T* p) { return reinterpret_cast<const Unaligned16<T>*>(p)->v; }
template <typename T> __device__ inline void st_row(T* p, u32x4_t v) { reinterpret_cast<Unaligned16<T>*>(p)->v = v; }

template <int W> constexpr int kTeamBlock = W > kWavesPerBlock ? W * kWave : kBlock;

template <int W>
struct Team {
  static constexpr int kRows = kTeamBlock<W> / (W * kWave);  // rows per workgroup
  static constexpr int kLanes = W * kWave;
  int wave, t;
  int64_t row;
  __device__ inline Team() {
    wave = int(threadIdx.x) / kWave;
    t = int(threadIdx.x) % kLanes;
    row = int64_t(blockIdx.x) * kRows + int(threadIdx.x) / kLanes;
  }
  // v, already combined over each wave, over the team's waves in wave order
  template <typename V, class F>
  __device__ inline V combine(V v, V* lds, F f) const {
    if constexpr (W == 1) return v;
    if ((threadIdx.x & (kWave - 1)) == 0) lds[wave] = v;
    __syncthreads();
    V r = lds[0];
#pragma unroll
    for (int w = 1; w < W; ++w) r = f(r, lds[w]);
    return r;
  }
};

// What a row's lanes read (one wave per row only, but for kLoop): kElements
// one or two elements and no vector (nv 0), kOne at most one vector, kLoop any
// number of them.  Rows of at most 64 elements, or 128 where they are no whole
// vectors, are read by element: more lanes share the arithmetic; and without
// the loop a short row's wave is a few instructions shorter (65536 rows, bf16, in
// us with vectors and the loop / so: sum of 7 9.6 / 8.4, max of 100 13.0 / 10.5,
// softmax of 64 18.4 / 13.0, LayerNorm of 65 25.1 / 18.0).
enum RowPath { kElements, kOne, kLoop };

// f(i, vector i) for the lane's vectors of a row in order, 4 loads in flight.
// The last up to 4 per lane are loaded together too, lanes past the end the
// last vector: with a branch per lane around them a wave waited up to three
// times (argmax of 4096 x 2000 bf16: 6.4 us, 5.1 now).
template <int W, typename T, class F>
__device__ inline void for_vectors(const T* xr, int64_t nv, int t, F f) {
  constexpr int S = W * kWave, N = Vec<T>::N;
  int64_t base = 0;
  for (; base + 4 * S <= nv; base += 4 * S) {
    const T* p = xr + (base + t) * N;
    const u32x4_t a = ld_row(p), b = ld_row(p + S * N), c = ld_row(p + 2 * S * N), d = ld_row(p + 3 * S * N);
    f(base + t, a);
    f(base + t + S, b);
    f(base + t + 2 * S, c);
    f(base + t + 3 * S, d);
  }
  const int64_t i = base + t;
  auto rest = [&](auto count) __attribute__((always_inline)) {
    constexpr int C = decltype(count)::value;
    u32x4_t v[C];
#pragma unroll
    for (int k = 0; k < C; ++k) v[k] = ld_row(xr + (i + k * S < nv ? i + k * S : nv - 1) * N);
#pragma unroll
    for (int k = 0; k < C; ++k)
      if (i + k * S < nv) f(i + k * S, v[k]);
  };
  const int64_t left = nv - base;  // uniform
  if (left > 2 * S) rest(std::integral_constant<int, 4>{});
  else if (left > S) rest(std::integral_constant<int, 2>{});
  else if (left > 0) rest(std::integral_constant<int, 1>{});
}

template <int W, RowPath PATH, typename T, class F>
__device__ inline void row_vectors(const T* xr, int64_t nv, int t, F f) {
  if constexpr (PATH == kLoop) for_vectors<W>(xr, nv, t, f);
  else if constexpr (PATH == kOne) {
    if (t < nv) f(int64_t(t), ld_row(xr + t * Vec<T>::N));
  }
}

// f(c) for the lane's elements past the vectors, the first of them at c
template <int W, RowPath PATH, class F>
__device__ inline void row_elements(int64_t c, int64_t cols, F f) {
  if (c < cols) f(c);
  if constexpr (PATH == kElements)
    if (c + W * kWave < cols) f(c + W * kWave);
}

// element j of a 16-byte vector as fp32
template <typename T, bool IS_F16>
__device__ inline float elem(const u32x4_t& v, int j) {
  if constexpr (sizeof(T) == 4) {
    const uint32_t w = v[j];
    return __builtin_bit_cast(float, w);
  } else {
    const uint32_t w = v[j / 2];
    return ld<T, IS_F16>(uint16_t(j % 2 ? w >> 16 : w));
  }
}

// StableHLO max/min propagate NaN; fmaxf/fminf drop it, so NaN is tracked
// separately for OP 1/2.
template <typename T, bool IS_F16, int OP, int W, RowPath PATH>
__global__ __launch_bounds__(kTeamBlock<W>) void row_reduce_kernel(const T* __restrict__ x, int64_t rows,
                                                                   int64_t cols, int64_t nv, float init, void* y,
                                                                   int out_type) {
  __shared__ float red[W];
  __shared__ int red_nan[W];
  const Team<W> tm;
  if (W == 1 && tm.row >= rows) return;
  const T* xr = x + tm.row * cols;
  constexpr int N = Vec<T>::N;
  float acc = identity<OP>();
  bool nan = false;
  auto take = [&](float f) {
    nan |= (f != f);
    acc = combine<OP>(acc, f);
  };
  row_vectors<W, PATH>(xr, nv, tm.t, [&](int64_t, const u32x4_t& v) {
#pragma unroll
    for (int j = 0; j < N; ++j) take(elem<T, IS_F16>(v, j));
  });
  row_elements<W, PATH>(nv * N + tm.t, cols, [&](int64_t c) { take(ld<T, IS_F16>(xr[c])); });
  acc = tm.combine(wave_combine<OP>(acc), red, [](float a, float b) { return combine<OP>(a, b); });
  // the vote must run with the whole wave active, before the lane-0 branch
  const int any_nan = tm.combine(int(__any(nan)), red_nan, [](int a, int b) { return a | b; });
  if (tm.t == 0) {
    float r = combine<OP>(acc, init);
    if constexpr (OP == 1 || OP == 2) {
      if (any_nan || init != init) r = __builtin_nanf("");
    }
    store_from_f32(y, tm.row, out_type, r);
  }
}

// Argmax / argmin with XLA's variadic-reduce semantics: larger value wins for
// argmax (smaller for argmin), every NaN beats every number, -0 == +0, ties
// go to the lower index.  Each element becomes an unsigned key that orders
// the values that way.
typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));

// two 16-bit floats (bf16, f16; INF the infinity's bits) at once with packed
// 16-bit integer ops
template <bool IS_MIN, uint32_t INF>
__device__ inline uint32_t order_keys(uint32_t w) {
  constexpr unsigned short kNan = INF + 1;  // smallest NaN magnitude
  const u16x2_t mag = __builtin_bit_cast(u16x2_t, w & 0x7FFF7FFFu);
  const u16x2_t magc = __builtin_elementwise_min(mag, u16x2_t{kNan, kNan});  // NaN -> kNan
  // bit 15 of mag + (0x8000 - kNan) is set exactly for NaN halves
  const uint32_t nanb =
      __builtin_bit_cast(uint32_t, mag + u16x2_t{0x8000 - kNan, 0x8000 - kNan}) & 0x80008000u;
  const uint32_t sgn = w & 0x80008000u;
  // halves whose key is 0x8000 - magnitude: negative numbers for argmax,
  // positive numbers for argmin; the other halves (NaN included) take
  // 0x8000 + magnitude
  const uint32_t low = IS_MIN ? (~(sgn | nanb) & 0x80008000u) : (sgn & ~nanb);
  const uint32_t mask = (low >> 15) * 0xFFFFu;
  const uint32_t kp = __builtin_bit_cast(uint32_t, magc + u16x2_t{0x8000, 0x8000});
  const uint32_t kn = __builtin_bit_cast(uint32_t, u16x2_t{0x8000, 0x8000} - magc);
  return (mask & kn) | (~mask & kp);
}
// one fp32
template <bool IS_MIN>
__device__ inline uint32_t order_key32(uint32_t w) {
  const uint32_t mag = w & 0x7FFFFFFFu;
  if (mag > 0x7F800000u) return 0xFFFFFFFFu;
  return ((w >> 31) != 0) != IS_MIN ? 0x80000000u - mag : 0x80000000u + mag;
}

// Rows of at most 65536 16-bit floats (NARROW): an element is the word
// (key << 16) | (0xFFFF - index), so the row winner is the unsigned max of
// the words.  Otherwise key and index are kept apart; a lane visits its
// elements in increasing index, so only a larger key replaces its winner.
template <typename T, bool IS_F16, bool IS_MIN, typename IdxT, bool NARROW, int W, RowPath PATH>
__global__ __launch_bounds__(kTeamBlock<W>) void row_argmax_kernel(const T* __restrict__ x, int64_t rows,
                                                                   int64_t cols, int64_t nv, T* __restrict__ values,
                                                                   IdxT* __restrict__ indices) {
  constexpr uint32_t kInf = IS_F16 ? 0x7C00u : 0x7F80u;
  constexpr int N = Vec<T>::N;
  __shared__ uint32_t red_key[W];
  __shared__ int64_t red_at[W];
  const Team<W> tm;
  if (W == 1 && tm.row >= rows) return;
  const T* xr = x + tm.row * cols;
  const int64_t tail = nv * N + tm.t;
  uint32_t best = 0;  // below every element's word; at or below every key
  int64_t at = INT64_MAX;
  if constexpr (NARROW) {
    static_assert(sizeof(T) == 2, "16-bit floats");
    row_vectors<W, PATH>(xr, nv, tm.t, [&](int64_t i, const u32x4_t& v) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t k = order_keys<IS_MIN, kInf>(v[j]);
        const uint32_t e = 0xFFFFu - (8u * uint32_t(i) + 2 * j);  // complement of the low half's index
        const uint32_t p0 = (k << 16) | e, p1 = (k & 0xFFFF0000u) | (e - 1u);
        best = max(best, max(p0, p1));
      }
    });
    row_elements<W, PATH>(tail, cols, [&](int64_t c) {
      best = max(best, (order_keys<IS_MIN, kInf>(xr[c]) << 16) | (0xFFFFu - uint32_t(c)));
    });
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) best = max(best, uint32_t(__shfl_xor(int(best), m, kWave)));
    best = tm.combine(best, red_key, [](uint32_t a, uint32_t b) { return max(a, b); });
    at = int64_t(0xFFFFu - (best & 0xFFFFu));
  } else {
    auto take = [&](uint32_t key, int64_t i) {
      if (key > best || at == INT64_MAX) best = key, at = i;
    };
    row_vectors<W, PATH>(xr, nv, tm.t, [&](int64_t i, const u32x4_t& v) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (sizeof(T) == 2) {
          const uint32_t k = order_keys<IS_MIN, kInf>(v[j]);
          take(k & 0xFFFFu, i * N + 2 * j);
          take(k >> 16, i * N + 2 * j + 1);
        } else {
          take(order_key32<IS_MIN>(v[j]), i * N + j);
        }
      }
    });
    row_elements<W, PATH>(tail, cols, [&](int64_t c) {
      if constexpr (sizeof(T) == 2) take(order_keys<IS_MIN, kInf>(xr[c]) & 0xFFFFu, c);
      else take(order_key32<IS_MIN>(__builtin_bit_cast(uint32_t, xr[c])), c);
    });
    // lanes without an element hold (0, INT64_MAX) and lose every tie
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
      const uint32_t ok = __shfl_xor(best, m, kWave);
      const int64_t oi = __shfl_xor(at, m, kWave);
      if (ok > best || (ok == best && oi < at)) best = ok, at = oi;
    }
    if constexpr (W > 1) {
      if ((threadIdx.x & (kWave - 1)) == 0) red_key[tm.wave] = best, red_at[tm.wave] = at;
      __syncthreads();
      if (tm.t != 0) return;
      for (int w = 1; w < W; ++w)
        if (red_key[w] > best || (red_key[w] == best && red_at[w] < at)) best = red_key[w], at = red_at[w];
    }
  }
  if (tm.t == 0) {
    if (values) values[tm.row] = xr[at];  // the winner's own bits (NaN payloads included)
    indices[tm.row] = IdxT(at);
  }
}

// LayerNorm: one wave per row, the whole row held in registers (up to
// kLnMaxPerLane fp32 per lane), two-pass mean/variance, single store.
constexpr int kLnMaxVecs = 8;  // 8 × 8 bf16 = 64 elements per lane → cols ≤ 4096 in registers

// TO: the stored type (T, or bf16 for fp32 rows: four values as one 8-byte
// store, y rows 8-byte aligned).  ADD (fp32 rows): the row is x + x2 (one
// fp32 add per element, the residual stream's update), stored to xsum and
// normalised.
template <typename T, typename TO = T, bool ADD = false>
__global__ __launch_bounds__(kBlock) void layernorm_reg_kernel(const T* __restrict__ x,
                                                               const T* __restrict__ gamma,
                                                               const T* __restrict__ beta,
                                                               int64_t rows, int cols, float eps,
                                                               TO* __restrict__ y, const T* __restrict__ x2 = nullptr,
                                                               T* __restrict__ xsum = nullptr) {
  using V = typename Vec<T>::V;
  constexpr int N = Vec<T>::N;
  static_assert(!ADD || sizeof(T) == 4, "the fused residual add is for fp32 rows");
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t row = int64_t(blockIdx.x) * kWavesPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int nv = cols / N;  // vectors per row; host guarantees nv ≤ kLnMaxVecs * 64
  const V* xv = reinterpret_cast<const V*>(x + row * int64_t(cols));
  float r[kLnMaxVecs][N];
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < kLnMaxVecs; ++k) {
    int i = lane + k * kWave;
    if (i < nv) {
      V a = xv[i];
      if constexpr (ADD) {
        const V b = reinterpret_cast<const V*>(x2 + row * int64_t(cols))[i];
#pragma unroll
        for (int j = 0; j < N; ++j) a.v[j] = a.v[j] + b.v[j];
        reinterpret_cast<V*>(xsum + row * int64_t(cols))[i] = a;
      }
#pragma unroll
      for (int j = 0; j < N; ++j) {
        r[k][j] = to_f32<T>(a.v[j]);
        s += r[k][j];
      }
    }
  }
  const float inv_n = 1.f / float(cols);
  const float mean = wave_sum(s) * inv_n;
  float q = 0.f;
#pragma unroll
  for (int k = 0; k < kLnMaxVecs; ++k) {
    if (lane + k * kWave < nv) {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        float d = r[k][j] - mean;
        q += d * d;
      }
    }
  }
  const float var = wave_sum(q) * inv_n;
  const float rstd = 1.f / sqrtf(var + eps);
  const V* gv = reinterpret_cast<const V*>(gamma);
  const V* bv = reinterpret_cast<const V*>(beta);
  constexpr bool kNarrow = sizeof(TO) < sizeof(T);
  static_assert(!kNarrow || N == 4, "narrowing store: fp32 rows to bf16");
  using VO = std::conditional_t<kNarrow, uint2, V>;
  VO* yv = reinterpret_cast<VO*>(y + row * int64_t(cols));
#pragma unroll
  for (int k = 0; k < kLnMaxVecs; ++k) {
    int i = lane + k * kWave;
    if (i < nv) {
      V g{}, b{};
      float o[N];
      if (gamma) g = gv[i];
      if (beta) b = bv[i];
#pragma unroll
      for (int j = 0; j < N; ++j) {
        float gj = gamma ? to_f32<T>(g.v[j]) : 1.f;
        float bj = beta ? to_f32<T>(b.v[j]) : 0.f;
        o[j] = (r[k][j] - mean) * rstd * gj + bj;
      }
      if constexpr (kNarrow) {
        yv[i] = uint2{uint32_t(f32_to_bf16(o[0])) | (uint32_t(f32_to_bf16(o[1])) << 16),
                      uint32_t(f32_to_bf16(o[2])) | (uint32_t(f32_to_bf16(o[3])) << 16)};
      } else {
        V ov;
#pragma unroll
        for (int j = 0; j < N; ++j) {
          if constexpr (sizeof(T) == 2) ov.v[j] = f32_to_bf16(o[j]);
          else ov.v[j] = o[j];
        }
        yv[i] = ov;
      }
    }
  }
}

// bf16 -> fp32 widening of the low / high half of a packed word, spelled
// three ways (shift, byte permute, funnel shift).  The LayerNorm passes each
// use their own spelling, so the compiler cannot merge them into one widened
// copy of the row kept live across the passes: the row stays packed (8 bf16
// per 16-byte vector), fewer registers, more rows in flight.
__device__ inline float lo_a(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ inline float hi_a(uint32_t w) { return __builtin_bit_cast(float, w & 0xFFFF0000u); }
__device__ inline float lo_b(uint32_t w) { return __builtin_bit_cast(float, __builtin_amdgcn_perm(w, 0u, 0x05040C0Cu)); }
__device__ inline float hi_b(uint32_t w) { return __builtin_bit_cast(float, __builtin_amdgcn_perm(w, 0u, 0x07060C0Cu)); }
__device__ inline float lo_c(uint32_t w) { return __builtin_bit_cast(float, __builtin_amdgcn_alignbit(w, 0u, 16u)); }
__device__ inline float hi_c(uint32_t w) { return __builtin_bit_cast(float, __builtin_amdgcn_perm(0u, w, 0x03020C0Cu)); }

// LayerNorm for bf16 rows split over WPR waves of a 256-thread workgroup
// (4 / WPR rows per workgroup): lane t of the row's WPR*64 lanes holds the
// 16-byte vectors t, t + 64 WPR, ... (KV of them), so a row of 4096 needs
// 8 / WPR registers' worth of vectors per lane and many more waves fit on a
// CU than with a whole row per wave.  The two row sums are combined across
// the row's waves through LDS; mean and variance are two-pass as in
// layernorm_reg_kernel.  Rows past the end still take part in the barriers.
template <int WPR, int KV>
__global__ __launch_bounds__(kBlock) void layernorm_bf16_split_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ gamma, const uint16_t* __restrict__ beta,
    int64_t rows, int cols, float eps, uint16_t* __restrict__ y) {
  constexpr int RPB = kWavesPerBlock / WPR;  // rows per workgroup
  __shared__ float red[2][kWavesPerBlock];
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x >> 6;
  const int rloc = wave / WPR, part = wave % WPR;
  const int64_t row = int64_t(blockIdx.x) * RPB + rloc;
  const bool live = row < rows;
  const int nv = cols / 8;
  const int t0 = part * kWave + lane;
  constexpr int kStride = WPR * kWave;
  const u32x4_t* xv = reinterpret_cast<const u32x4_t*>(x + (live ? row : 0) * cols);
  u32x4_t v[KV];
#pragma unroll
  for (int k = 0; k < KV; ++k)
    if (live && t0 + k * kStride < nv) v[k] = xv[t0 + k * kStride];
  const float inv_n = 1.f / float(cols);
  float s = 0.f;
#pragma unroll
  for (int k = 0; k < KV; ++k)
    if (live && t0 + k * kStride < nv)
#pragma unroll
      for (int j = 0; j < 4; ++j) s += lo_a(v[k][j]) + hi_a(v[k][j]);
  s = wave_sum(s);
  if constexpr (WPR > 1) {
    if (lane == 0) red[0][wave] = s;
    __syncthreads();
    s = 0.f;
#pragma unroll
    for (int w = 0; w < WPR; ++w) s += red[0][rloc * WPR + w];
  }
  const float mean = s * inv_n;
  float q = 0.f;
#pragma unroll
  for (int k = 0; k < KV; ++k)
    if (live && t0 + k * kStride < nv)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float d0 = lo_b(v[k][j]) - mean, d1 = hi_b(v[k][j]) - mean;
        q += d0 * d0 + d1 * d1;
      }
  q = wave_sum(q);
  if constexpr (WPR > 1) {
    if (lane == 0) red[1][wave] = q;
    __syncthreads();
    q = 0.f;
#pragma unroll
    for (int w = 0; w < WPR; ++w) q += red[1][rloc * WPR + w];
  }
  if (!live) return;
  const float rstd = 1.f / sqrtf(q * inv_n + eps);
  u32x4_t* yv = reinterpret_cast<u32x4_t*>(y + row * cols);
#pragma unroll
  for (int k = 0; k < KV; ++k) {
    const int i = t0 + k * kStride;
    if (i < nv) {
      const u32x4_t one4 = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
      const u32x4_t gk = gamma ? reinterpret_cast<const u32x4_t*>(gamma)[i] : one4;
      const u32x4_t bk = beta ? reinterpret_cast<const u32x4_t*>(beta)[i] : u32x4_t{0u, 0u, 0u, 0u};
      u32x4_t o;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x2_t e = {(lo_c(v[k][j]) - mean) * rstd * lo_a(gk[j]) + lo_a(bk[j]),
                           (hi_c(v[k][j]) - mean) * rstd * hi_a(gk[j]) + hi_a(bk[j])};
        o[j] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e, bf16x2_t));
      }
      yv[i] = o;
    }
  }
}

// A lane's share of a team's row: KV 16-byte vectors (vector t + 64 W k; nv
// whole ones in the row) and the row's element nv N + t past them.  The loads
// are unconditional (vector 0 where the row has no such vector), so all of
// them are in flight together.  KV = 0: no vectors, the row's elements t and
// t + 64 W.
template <typename T, int W, int KV>
struct RowShare {
  static constexpr int N = Vec<T>::N, S = W * kWave, E = KV > 0 ? 1 : 2;
  u32x4_t v[KV > 0 ? KV : 1];
  float tail[E];
  int64_t nv, cols;
  int t;
  __device__ inline RowShare(const T* xr, int64_t cols_, int t_) : cols(cols_), t(t_) {
    nv = KV > 0 ? cols / N : 0;
    if (nv > 0) {
#pragma unroll
      for (int k = 0; k < KV; ++k) v[k] = ld_row(xr + (has(k) ? t + k * S : 0) * int64_t(N));
    }
#pragma unroll
    for (int e = 0; e < E; ++e) tail[e] = has_tail(e) ? to_f32<T>(xr[tail_at(e)]) : 0.f;
  }
  __device__ inline bool has(int k) const { return t + k * S < nv; }
  __device__ inline float at(int k, int j) const { return elem<T, false>(v[k], j); }
  __device__ inline int64_t tail_at(int e) const { return nv * N + t + e * S; }
  __device__ inline bool has_tail(int e) const { return tail_at(e) < cols; }
};

template <typename T>
__device__ inline T narrow(float f) {
  if constexpr (sizeof(T) == 2) return f32_to_bf16(f);
  else return f;
}
// N fp32 values to TO elements at an element-aligned address
template <typename TO, int N>
__device__ inline void st_values(TO* p, const float (&o)[N]) {
  struct __attribute__((packed, aligned(sizeof(TO)))) Pack { TO e[N]; };
  Pack q;
#pragma unroll
  for (int j = 0; j < N; ++j) q.e[j] = narrow<TO>(o[j]);
  *reinterpret_cast<Pack*>(p) = q;
}

// LayerNorm of rows off the 16-byte grid or wider than the kernels above
// hold: the row in the registers of a team of W waves (KV vectors per lane),
// one read of x, the same two-pass statistics.  With x2 (fp32 rows) the row
// is x + x2, written to xsum.  Against three element-wise passes over the
// row: 8192 x 4095 bf16 114 -> 29.9 us, 8192 x 4096 fp32 114 -> 50.5 us (5.3
// TB/s), 30000 x 300 bf16 26.3 -> 12.8 us.
template <typename T, typename TO, int W, int KV>
__global__ __launch_bounds__(kTeamBlock<W>) void layernorm_team_kernel(
    const T* __restrict__ x, const T* __restrict__ gamma, const T* __restrict__ beta, int64_t rows, int64_t cols,
    float eps, TO* __restrict__ y, const T* __restrict__ x2, T* __restrict__ xsum) {
  using R = RowShare<T, W, KV>;
  constexpr int N = R::N;
  __shared__ float red[2][W];
  const Team<W> tm;
  if (W == 1 && tm.row >= rows) return;
  R r(x + tm.row * cols, cols, tm.t);
  if constexpr (sizeof(T) == 4) {
    if (x2) {
      const R r2(x2 + tm.row * cols, cols, tm.t);
      T* sr = xsum + tm.row * cols;
#pragma unroll
      for (int k = 0; k < KV; ++k) {
        float o[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
          o[j] = r.at(k, j) + r2.at(k, j);
          r.v[k][j] = __builtin_bit_cast(uint32_t, o[j]);
        }
        if (r.has(k)) st_values<T, N>(sr + int64_t(tm.t + k * R::S) * N, o);
      }
#pragma unroll
      for (int e = 0; e < R::E; ++e) {
        r.tail[e] += r2.tail[e];
        if (r.has_tail(e)) sr[r.tail_at(e)] = r.tail[e];
      }
    }
  }
  auto add = [](float a, float b) { return a + b; };
  const float inv_n = 1.f / float(cols);
  float s = r.tail[0];
#pragma unroll
  for (int e = 1; e < R::E; ++e) s += r.tail[e];
#pragma unroll
  for (int k = 0; k < KV; ++k)
    if (r.has(k))
#pragma unroll
      for (int j = 0; j < N; ++j) s += r.at(k, j);
  const float mean = tm.combine(wave_sum(s), red[0], add) * inv_n;
  float q = 0.f;
#pragma unroll
  for (int e = 0; e < R::E; ++e)
    if (r.has_tail(e)) q += (r.tail[e] - mean) * (r.tail[e] - mean);
#pragma unroll
  for (int k = 0; k < KV; ++k)
    if (r.has(k))
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const float d = r.at(k, j) - mean;
        q += d * d;
      }
  const float rstd = 1.f / sqrtf(tm.combine(wave_sum(q), red[1], add) * inv_n + eps);
  TO* yr = y + tm.row * cols;
#pragma unroll
  for (int k = 0; k < KV; ++k) {
    if (!r.has(k)) continue;
    const int64_t c = int64_t(tm.t + k * R::S) * N;
    const u32x4_t g = gamma ? ld_row(gamma + c) : u32x4_t{0u, 0u, 0u, 0u};
    const u32x4_t b = beta ? ld_row(beta + c) : u32x4_t{0u, 0u, 0u, 0u};
    float o[N];
#pragma unroll
    for (int j = 0; j < N; ++j)
      o[j] = (r.at(k, j) - mean) * rstd * (gamma ? elem<T, false>(g, j) : 1.f) + elem<T, false>(b, j);
    st_values<TO, N>(yr + c, o);
  }
#pragma unroll
  for (int e = 0; e < R::E; ++e) {
    if (!r.has_tail(e)) continue;
    const int64_t c = r.tail_at(e);
    yr[c] = narrow<TO>((r.tail[e] - mean) * rstd * (gamma ? to_f32<T>(gamma[c]) : 1.f) +
                       (beta ? to_f32<T>(beta[c]) : 0.f));
  }
}

// LayerNorm of rows longer than a 16-wave team holds: three passes over the
// row.  With x2: as above; each lane reads back only what it wrote to xsum.
template <typename T, typename TO = T>
__global__ __launch_bounds__(kTeamBlock<16>) void layernorm_loop_kernel(
    const T* __restrict__ x, const T* __restrict__ gamma, const T* __restrict__ beta, int64_t rows, int64_t cols,
    float eps, TO* __restrict__ y, const T* x2, T* xsum) {
  constexpr int N = Vec<T>::N;
  __shared__ float red[2][16];
  const Team<16> tm;
  const T* xr = x + tm.row * cols;
  const int64_t nv = cols / N, tail = nv * N + tm.t;
  const bool has_tail = tail < cols;
  if constexpr (sizeof(T) == 4) {
    if (x2) {
      T* sr = xsum + tm.row * cols;
      for_vectors<16>(xr, nv, tm.t, [&](int64_t i, const u32x4_t& v) {
        const u32x4_t v2 = ld_row(x2 + tm.row * cols + i * N);
        float o[N];
#pragma unroll
        for (int j = 0; j < N; ++j) o[j] = elem<T, false>(v, j) + elem<T, false>(v2, j);
        st_values<T, N>(sr + i * N, o);
      });
      if (has_tail) sr[tail] = xr[tail] + x2[tm.row * cols + tail];
      xr = sr;
    }
  }
  auto add = [](float a, float b) { return a + b; };
  float s = has_tail ? to_f32<T>(xr[tail]) : 0.f;
  for_vectors<16>(xr, nv, tm.t, [&](int64_t, const u32x4_t& v) {
#pragma unroll
    for (int j = 0; j < N; ++j) s += elem<T, false>(v, j);
  });
  const float mean = tm.combine(wave_sum(s), red[0], add) / float(cols);
  float q = has_tail ? (to_f32<T>(xr[tail]) - mean) * (to_f32<T>(xr[tail]) - mean) : 0.f;
  for_vectors<16>(xr, nv, tm.t, [&](int64_t, const u32x4_t& v) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float d = elem<T, false>(v, j) - mean;
      q += d * d;
    }
  });
  const float rstd = 1.f / sqrtf(tm.combine(wave_sum(q), red[1], add) / float(cols) + eps);
  TO* yr = y + tm.row * cols;
  for_vectors<16>(xr, nv, tm.t, [&](int64_t i, const u32x4_t& v) {
    const u32x4_t g = gamma ? ld_row(gamma + i * N) : u32x4_t{0u, 0u, 0u, 0u};
    const u32x4_t b = beta ? ld_row(beta + i * N) : u32x4_t{0u, 0u, 0u, 0u};
    float o[N];
#pragma unroll
    for (int j = 0; j < N; ++j)
      o[j] = (elem<T, false>(v, j) - mean) * rstd * (gamma ? elem<T, false>(g, j) : 1.f) + elem<T, false>(b, j);
    st_values<TO, N>(yr + i * N, o);
  });
  if (has_tail)
    yr[tail] = narrow<TO>((to_f32<T>(xr[tail]) - mean) * rstd * (gamma ? to_f32<T>(gamma[tail]) : 1.f) +
                          (beta ? to_f32<T>(beta[tail]) : 0.f));
}

// Softmax with the row in a team's registers: one read of x, the exponentials
// kept for the division.  Against three element-wise passes over the row:
// 65536 x 1024 bf16 171 -> 46.5 us (5.8 TB/s), 2048 x 50257 921 -> 118 us.
template <typename T, int W, int KV>
__global__ __launch_bounds__(kTeamBlock<W>) void softmax_team_kernel(const T* __restrict__ x, int64_t rows,
                                                                     int64_t cols, T* __restrict__ y) {
  using R = RowShare<T, W, KV>;
  constexpr int N = R::N;
  __shared__ float red[2][W];
  const Team<W> tm;
  if (W == 1 && tm.row >= rows) return;
  const R r(x + tm.row * cols, cols, tm.t);
  float m = -INFINITY;
#pragma unroll
  for (int e = 0; e < R::E; ++e)
    if (r.has_tail(e)) m = fmaxf(m, r.tail[e]);
#pragma unroll
  for (int k = 0; k < KV; ++k)
    if (r.has(k))
#pragma unroll
      for (int j = 0; j < N; ++j) m = fmaxf(m, r.at(k, j));
  m = tm.combine(wave_max(m), red[0], [](float a, float b) { return fmaxf(a, b); });
  float e[KV > 0 ? KV : 1][N], s = 0.f;
#pragma unroll
  for (int k = 0; k < KV; ++k)
    if (r.has(k))
#pragma unroll
      for (int j = 0; j < N; ++j) {
        e[k][j] = __expf(r.at(k, j) - m);
        s += e[k][j];
      }
  float et[R::E];
#pragma unroll
  for (int k = 0; k < R::E; ++k) {
    et[k] = __expf(r.tail[k] - m);
    if (r.has_tail(k)) s += et[k];
  }
  const float inv = 1.f / tm.combine(wave_sum(s), red[1], [](float a, float b) { return a + b; });
  T* yr = y + tm.row * cols;
#pragma unroll
  for (int k = 0; k < KV; ++k) {
    if (!r.has(k)) continue;
#pragma unroll
    for (int j = 0; j < N; ++j) e[k][j] *= inv;
    st_values<T, N>(yr + int64_t(tm.t + k * R::S) * N, e[k]);
  }
#pragma unroll
  for (int k = 0; k < R::E; ++k)
    if (r.has_tail(k)) yr[r.tail_at(k)] = narrow<T>(et[k] * inv);
}

// Softmax of rows longer than a 16-wave team holds: max pass, sum-of-exp
// pass, normalise pass.
template <typename T>
__global__ __launch_bounds__(kTeamBlock<16>) void softmax_loop_kernel(const T* __restrict__ x, int64_t rows,
                                                                      int64_t cols, T* __restrict__ y) {
  constexpr int N = Vec<T>::N;
  __shared__ float red[2][16];
  const Team<16> tm;
  const T* xr = x + tm.row * cols;
  const int64_t nv = cols / N, tail = nv * N + tm.t;
  const bool has_tail = tail < cols;
  const float xt = has_tail ? to_f32<T>(xr[tail]) : -INFINITY;
  float m = xt;
  for_vectors<16>(xr, nv, tm.t, [&](int64_t, const u32x4_t& v) {
#pragma unroll
    for (int j = 0; j < N; ++j) m = fmaxf(m, elem<T, false>(v, j));
  });
  m = tm.combine(wave_max(m), red[0], [](float a, float b) { return fmaxf(a, b); });
  float s = has_tail ? __expf(xt - m) : 0.f;
  for_vectors<16>(xr, nv, tm.t, [&](int64_t, const u32x4_t& v) {
#pragma unroll
    for (int j = 0; j < N; ++j) s += __expf(elem<T, false>(v, j) - m);
  });
  const float inv = 1.f / tm.combine(wave_sum(s), red[1], [](float a, float b) { return a + b; });
  T* yr = y + tm.row * cols;
  for_vectors<16>(xr, nv, tm.t, [&](int64_t i, const u32x4_t& v) {
    float o[N];
#pragma unroll
    for (int j = 0; j < N; ++j) o[j] = __expf(elem<T, false>(v, j) - m) * inv;
    st_values<T, N>(yr + i * N, o);
  });
  if (has_tail) yr[tail] = narrow<T>(__expf(xt - m) * inv);
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

inline unsigned grid_for_rows(int64_t rows) {
  return unsigned((rows + kWavesPerBlock - 1) / kWavesPerBlock);
}

// Waves per row.  A wave per row when there are rows enough to fill the chip
// and a lane's share is at most 8 vectors; four or sixteen waves for longer
// rows, and for few rows, whose time is one wave's serial chain of loads
// (argmax of 32 rows of 50257 bf16: 161 us a call with a wave per row and
// 2-byte loads, 11.8 us with sixteen, most of that the call itself).
inline int team_waves(int64_t rows, int64_t vecs) {
  if (vecs > 2048 || (rows < 512 && vecs > 512)) return 16;
  if (vecs > 512 || (rows < 2048 && vecs > 64)) return 4;
  return 1;
}
template <int W> using Waves = std::integral_constant<int, W>;
template <RowPath P> using Path = std::integral_constant<RowPath, P>;
// f(Waves<W>{}) with W = waves
template <class F>
void with_waves(int waves, F f) {
  switch (waves) {
    case 1: f(Waves<1>{}); break;
    case 4: f(Waves<4>{}); break;
    default: f(Waves<16>{}); break;
  }
}
// whether rows are read by element (RowPath)
template <typename T> bool short_row(int64_t cols) { return cols <= (cols % Vec<T>::N == 0 ? 64 : 128); }
// f(Waves<W>{}, Path<P>{}, whole vectors per row) for the kernels that loop over a
// row of any length (reduce, argmax).  With 2048 rows or more the chip is full
// with one wave each, or four where a wave's share is long; fewer rows as
// team_waves.  argmax of 8192 x 16384 fp32, us with 1 / 4 / 16 waves: 106 / 90 /
// 114, 65536 x 2052: 92 / 110 / 437; sum of 4096 x 32768 bf16: 46.2 / 39.8 / 38.9.
template <typename T, class F>
void with_loop(int64_t rows, int64_t cols, F f) {
  const int64_t vecs = cols / Vec<T>::N;
  if (short_row<T>(cols)) return f(Waves<1>{}, Path<kElements>{}, int64_t(0));
  const int w = rows >= 4096 && vecs <= 1024 ? 1 : rows >= 2048 ? (vecs > 512 ? 4 : 1) : team_waves(rows, vecs);
  if (w == 1 && vecs <= kWave) f(Waves<1>{}, Path<kOne>{}, vecs);
  else if (w == 1) f(Waves<1>{}, Path<kLoop>{}, vecs);
  else if (w == 4) f(Waves<4>{}, Path<kLoop>{}, vecs);
  else f(Waves<16>{}, Path<kLoop>{}, vecs);
}
template <int W> dim3 team_grid(int64_t rows) { return dim3(unsigned((rows + Team<W>::kRows - 1) / Team<W>::kRows)); }
// f(first row, rows) in runs that a launch takes: HIP refuses grids of 2^32
// threads, 2^22 rows of a 16-wave team
template <int W, class F>
void for_row_runs(int64_t rows, F f) {
  constexpr int64_t kMost = (int64_t(1) << 32) / (W * kWave) - Team<W>::kRows;
  for (int64_t r = 0; r < rows; r += kMost) f(r, std::min(kMost, rows - r));
}

template <typename T, bool IS_F16, int OP>
void launch_reduce_op(hipStream_t s, int64_t rows, int64_t cols, const void* x, float init, void* y, int out_type) {
  with_loop<T>(rows, cols, [&](auto w, auto path, int64_t nv) {
    constexpr int W = decltype(w)::value;
    for_row_runs<W>(rows, [&](int64_t r, int64_t n) {
      hipLaunchKernelGGL((row_reduce_kernel<T, IS_F16, OP, W, decltype(path)::value>), team_grid<W>(n), dim3(kTeamBlock<W>), 0, s,
                         reinterpret_cast<const T*>(x) + r * cols, n, cols, nv, init,
                         static_cast<void*>(static_cast<char*>(y) + r * dtype_bytes(out_type)), out_type);
    });
  });
}

template <typename T, bool IS_F16>
int launch_reduce(hipStream_t s, int op, int64_t rows, int64_t cols, const void* x, float init,
                  void* y, int out_type) {
  switch (op) {
    case 0: launch_reduce_op<T, IS_F16, 0>(s, rows, cols, x, init, y, out_type); break;
    case 1: launch_reduce_op<T, IS_F16, 1>(s, rows, cols, x, init, y, out_type); break;
    case 2: launch_reduce_op<T, IS_F16, 2>(s, rows, cols, x, init, y, out_type); break;
    case 3: launch_reduce_op<T, IS_F16, 3>(s, rows, cols, x, init, y, out_type); break;
    default: return fail(MK_ERR_INVALID, "mk_row_reduce: op must be 0..3");
  }
  return check_launch("mk_row_reduce");
}

template <typename T, bool IS_F16, bool IS_MIN, typename IdxT>
int launch_argmax_as(hipStream_t s, int64_t rows, int64_t cols, const void* x, void* values, void* indices) {
  with_loop<T>(rows, cols, [&](auto w, auto path, int64_t nv) {
    constexpr int W = decltype(w)::value;
    constexpr RowPath P = decltype(path)::value;
    auto go = [&](auto kernel) {
      for_row_runs<W>(rows, [&](int64_t r, int64_t n) {
        T* v = reinterpret_cast<T*>(values);
        hipLaunchKernelGGL(kernel, team_grid<W>(n), dim3(kTeamBlock<W>), 0, s, reinterpret_cast<const T*>(x) + r * cols,
                           n, cols, nv, v ? v + r : v, reinterpret_cast<IdxT*>(indices) + r);
      });
    };
    if constexpr (sizeof(T) == 2) {
      if (cols <= 65536) return go(row_argmax_kernel<T, IS_F16, IS_MIN, IdxT, true, W, P>);
    }
    go(row_argmax_kernel<T, IS_F16, IS_MIN, IdxT, false, W, P>);
  });
  return check_launch("mk_row_argmax");
}

template <typename T, bool IS_F16, bool IS_MIN>
int launch_argmax(hipStream_t s, int64_t rows, int64_t cols, const void* x, void* values,
                  int index_type, void* indices) {
  return index_type == MK_S32 ? launch_argmax_as<T, IS_F16, IS_MIN, int32_t>(s, rows, cols, x, values, indices)
                              : launch_argmax_as<T, IS_F16, IS_MIN, int64_t>(s, rows, cols, x, values, indices);
}

// f(Waves<KV>{}) with the vectors per lane of a team of W waves
template <class F>
void with_share(int64_t vecs, int waves, F f) {
  const int64_t per = (vecs + 64 * waves - 1) / (64 * waves);
  if (per <= 2) f(Waves<2>{});
  else if (per <= 4) f(Waves<4>{});
  else f(Waves<8>{});
}
constexpr int64_t kTeamMaxVecs = 16 * kWave * 8;  // vectors a 16-wave team's registers hold

// LayerNorm on the kernels that take any width and alignment
template <typename T, typename TO>
void launch_layernorm_any(hipStream_t s, int64_t rows, int64_t cols, const T* x, const T* gamma, const T* beta,
                          float eps, TO* y, const T* x2 = nullptr, T* xsum = nullptr) {
  const int64_t vecs = cols / Vec<T>::N;
  auto go = [&](auto w, auto kernel) {
    constexpr int W = decltype(w)::value;
    for_row_runs<W>(rows, [&](int64_t r, int64_t n) {
      const int64_t at = r * cols;
      hipLaunchKernelGGL(kernel, team_grid<W>(n), dim3(kTeamBlock<W>), 0, s, x + at, gamma, beta, n, cols, eps, y + at,
                         x2 ? x2 + at : x2, xsum ? xsum + at : xsum);
    });
  };
  if (vecs > kTeamMaxVecs) return go(Waves<16>{}, layernorm_loop_kernel<T, TO>);
  if (short_row<T>(cols)) return go(Waves<1>{}, layernorm_team_kernel<T, TO, 1, 0>);
  with_waves(team_waves(rows, vecs), [&](auto w) {
    constexpr int W = decltype(w)::value;
    with_share(vecs, W, [&](auto kv) { go(w, layernorm_team_kernel<T, TO, W, decltype(kv)::value>); });
  });
}

template <typename T>
void launch_softmax(hipStream_t s, int64_t rows, int64_t cols, const T* x, T* y) {
  const int64_t vecs = cols / Vec<T>::N;
  auto go = [&](auto w, auto kernel) {
    constexpr int W = decltype(w)::value;
    for_row_runs<W>(rows, [&](int64_t r, int64_t n) {
      hipLaunchKernelGGL(kernel, team_grid<W>(n), dim3(kTeamBlock<W>), 0, s, x + r * cols, n, cols, y + r * cols);
    });
  };
  if (vecs > kTeamMaxVecs) return go(Waves<16>{}, softmax_loop_kernel<T>);
  if (short_row<T>(cols)) return go(Waves<1>{}, softmax_team_kernel<T, 1, 0>);
  with_waves(team_waves(rows, vecs), [&](auto w) {
    constexpr int W = decltype(w)::value;
    with_share(vecs, W, [&](auto kv) { go(w, softmax_team_kernel<T, W, decltype(kv)::value>); });
  });
}

}  // namespace
}  // namespace mk

using namespace mk;

extern "C" int mk_row_reduce(void* stream, int in_type, int out_type, int op, int64_t rows,
                             int64_t cols, const void* x, float init, void* y) {
  clear_error();
  if (rows < 0 || cols < 0) return fail(MK_ERR_INVALID, "mk_row_reduce: negative shape");
  if (out_type != MK_F32 && out_type != MK_BF16 && out_type != MK_F16)
    return fail(MK_ERR_UNSUPPORTED, "mk_row_reduce: out_type must be f32/bf16/f16");
  if (rows == 0) return MK_OK;
  if (!x || !y) return fail(MK_ERR_INVALID, "mk_row_reduce: null pointer");
  hipStream_t s = as_stream(stream);
  switch (in_type) {
    case MK_BF16: return launch_reduce<uint16_t, false>(s, op, rows, cols, x, init, y, out_type);
    case MK_F16: return launch_reduce<uint16_t, true>(s, op, rows, cols, x, init, y, out_type);
    case MK_F32: return launch_reduce<float, false>(s, op, rows, cols, x, init, y, out_type);
    default: return fail(MK_ERR_UNSUPPORTED, "mk_row_reduce: in_type must be bf16/f16/f32");
  }
}

extern "C" int mk_row_argmax(void* stream, int in_type, int is_min, int64_t rows, int64_t cols,
                             const void* x, void* values, int index_type, void* indices) {
  clear_error();
  if (rows < 0 || cols <= 0)
    return fail(MK_ERR_INVALID, "mk_row_argmax: need rows >= 0 and cols >= 1");
  if (index_type != MK_S32 && index_type != MK_S64)
    return fail(MK_ERR_UNSUPPORTED, "mk_row_argmax: index_type must be s32/s64");
  if (rows == 0) return MK_OK;
  if (!x || !indices) return fail(MK_ERR_INVALID, "mk_row_argmax: null pointer");
  hipStream_t s = as_stream(stream);
  switch (in_type) {
    case MK_BF16:
      return is_min ? launch_argmax<uint16_t, false, true>(s, rows, cols, x, values, index_type, indices)
                    : launch_argmax<uint16_t, false, false>(s, rows, cols, x, values, index_type, indices);
    case MK_F16:
      return is_min ? launch_argmax<uint16_t, true, true>(s, rows, cols, x, values, index_type, indices)
                    : launch_argmax<uint16_t, true, false>(s, rows, cols, x, values, index_type, indices);
    case MK_F32:
      return is_min ? launch_argmax<float, false, true>(s, rows, cols, x, values, index_type, indices)
                    : launch_argmax<float, false, false>(s, rows, cols, x, values, index_type, indices);
    default: return fail(MK_ERR_UNSUPPORTED, "mk_row_argmax: in_type must be bf16/f16/f32");
  }
}

extern "C" int mk_layernorm(void* stream, int io_type, int64_t rows, int64_t cols, const void* x,
                            const void* gamma, const void* beta, float eps, void* y) {
  clear_error();
  if (rows < 0 || cols <= 0) return fail(MK_ERR_INVALID, "mk_layernorm: bad shape");
  if (rows == 0) return MK_OK;
  if (!x || !y) return fail(MK_ERR_INVALID, "mk_layernorm: null pointer");
  hipStream_t s = as_stream(stream);
  dim3 g(grid_for_rows(rows)), b(kBlock);
  auto vec_ok = [&](int n) {
    return (cols % n) == 0 && cols / n <= int64_t(kLnMaxVecs) * kWave && aligned16(x) &&
           aligned16(y) && (!gamma || aligned16(gamma)) && (!beta || aligned16(beta));
  };
  if (io_type == MK_BF16) {
    using T = uint16_t;
    const T *xp = (const T*)x, *gp = (const T*)gamma, *bp = (const T*)beta;
    // rows of up to 4096 / 8192 / 16384 stay in registers over 1 / 2 / 4 waves
    const bool vec = cols % 8 == 0 && cols <= 16384 && rows < (int64_t(1) << 31) && aligned16(x) &&
                     aligned16(y) && (!gamma || aligned16(gamma)) && (!beta || aligned16(beta));
    if (vec && cols <= 4096)
      hipLaunchKernelGGL((layernorm_bf16_split_kernel<1, 8>), g, b, 0, s, xp, gp, bp, rows, int(cols), eps, (T*)y);
    else if (vec && cols <= 8192)
      hipLaunchKernelGGL((layernorm_bf16_split_kernel<2, 8>), dim3(unsigned((rows + 1) / 2)), b, 0, s, xp, gp,
                         bp, rows, int(cols), eps, (T*)y);
    else if (vec && cols <= 16384)
      hipLaunchKernelGGL((layernorm_bf16_split_kernel<4, 8>), dim3(unsigned(rows)), b, 0, s, xp, gp, bp, rows,
                         int(cols), eps, (T*)y);
    else
      launch_layernorm_any<T, T>(s, rows, cols, xp, gp, bp, eps, (T*)y);
  } else if (io_type == MK_F32) {
    using T = float;
    const T *xp = (const T*)x, *gp = (const T*)gamma, *bp = (const T*)beta;
    if (vec_ok(4))
      hipLaunchKernelGGL(layernorm_reg_kernel<T>, g, b, 0, s, xp, gp, bp, rows, int(cols), eps, (T*)y);
    else
      launch_layernorm_any<T, T>(s, rows, cols, xp, gp, bp, eps, (T*)y);
  } else {
    return fail(MK_ERR_UNSUPPORTED, "mk_layernorm: io_type must be bf16/f32");
  }
  return check_launch("mk_layernorm");
}

extern "C" int mk_layernorm_typed(void* stream, int in_type, int out_type, int64_t rows, int64_t cols,
                                  const void* x, const void* gamma, const void* beta, float eps, void* y) {
  if (in_type == out_type) return mk_layernorm(stream, in_type, rows, cols, x, gamma, beta, eps, y);
  clear_error();
  if (in_type != MK_F32 || out_type != MK_BF16)
    return fail(MK_ERR_UNSUPPORTED, "mk_layernorm_typed: (in, out) must be (bf16, bf16), (f32, f32) or (f32, bf16)");
  if (rows < 0 || cols <= 0) return fail(MK_ERR_INVALID, "mk_layernorm_typed: bad shape");
  if (rows == 0) return MK_OK;
  if (!x || !y) return fail(MK_ERR_INVALID, "mk_layernorm_typed: null pointer");
  hipStream_t s = as_stream(stream);
  dim3 g(grid_for_rows(rows)), b(kBlock);
  const float *xp = (const float*)x, *gp = (const float*)gamma, *bp = (const float*)beta;
  const bool vec = cols % 4 == 0 && cols / 4 <= int64_t(kLnMaxVecs) * kWave && aligned16(x) &&
                   (reinterpret_cast<uintptr_t>(y) & 7u) == 0 && (!gamma || aligned16(gamma)) &&
                   (!beta || aligned16(beta));
  if (vec)
    hipLaunchKernelGGL((layernorm_reg_kernel<float, uint16_t>), g, b, 0, s, xp, gp, bp, rows, int(cols), eps,
                       (uint16_t*)y);
  else
    launch_layernorm_any<float, uint16_t>(s, rows, cols, xp, gp, bp, eps, (uint16_t*)y);
  return check_launch("mk_layernorm_typed");
}

extern "C" int mk_add_layernorm_typed(void* stream, int in_type, int out_type, int64_t rows, int64_t cols,
                                      const void* a, const void* b, const void* bias, const void* gamma,
                                      const void* beta, float eps, void* sum_out, void* y) {
  if (in_type == MK_BF16 && out_type == MK_BF16)
    return mk_add_layernorm(stream, rows, cols, a, b, bias, gamma, beta, eps, sum_out, y);
  clear_error();
  if (in_type != MK_F32 || (out_type != MK_F32 && out_type != MK_BF16))
    return fail(MK_ERR_UNSUPPORTED, "mk_add_layernorm_typed: (in, out) must be (bf16, bf16), (f32, f32) or (f32, bf16)");
  if (bias) return fail(MK_ERR_UNSUPPORTED, "mk_add_layernorm_typed: no bias for fp32 rows (add it to b)");
  if (rows < 0 || cols <= 0) return fail(MK_ERR_INVALID, "mk_add_layernorm_typed: bad shape");
  if (rows == 0) return MK_OK;
  if (!a || !b || !sum_out || !y) return fail(MK_ERR_INVALID, "mk_add_layernorm_typed: null pointer");
  hipStream_t s = as_stream(stream);
  dim3 g(grid_for_rows(rows)), blk(kBlock);
  const float *ap = (const float*)a, *bp = (const float*)b, *gp = (const float*)gamma, *tp = (const float*)beta;
  float* sp = (float*)sum_out;
  const uintptr_t ymask = out_type == MK_BF16 ? 7u : 15u;
  const bool vec = cols % 4 == 0 && cols / 4 <= int64_t(kLnMaxVecs) * kWave && aligned16(a) && aligned16(b) &&
                   aligned16(sum_out) && (reinterpret_cast<uintptr_t>(y) & ymask) == 0 && (!gamma || aligned16(gamma)) &&
                   (!beta || aligned16(beta));
  if (out_type == MK_BF16) {
    if (vec)
      hipLaunchKernelGGL((layernorm_reg_kernel<float, uint16_t, true>), g, blk, 0, s, ap, gp, tp, rows, int(cols), eps,
                         (uint16_t*)y, bp, sp);
    else
      launch_layernorm_any<float, uint16_t>(s, rows, cols, ap, gp, tp, eps, (uint16_t*)y, bp, sp);
  } else {
    if (vec)
      hipLaunchKernelGGL((layernorm_reg_kernel<float, float, true>), g, blk, 0, s, ap, gp, tp, rows, int(cols), eps,
                         (float*)y, bp, sp);
    else
      launch_layernorm_any<float, float>(s, rows, cols, ap, gp, tp, eps, (float*)y, bp, sp);
  }
  return check_launch("mk_add_layernorm_typed");
}

extern "C" int mk_softmax_rows(void* stream, int io_type, int64_t rows, int64_t cols,
                               const void* x, void* y) {
  clear_error();
  if (rows < 0 || cols <= 0) return fail(MK_ERR_INVALID, "mk_softmax_rows: bad shape");
  if (rows == 0) return MK_OK;
  if (!x || !y) return fail(MK_ERR_INVALID, "mk_softmax_rows: null pointer");
  hipStream_t s = as_stream(stream);
  if (io_type == MK_BF16)
    launch_softmax(s, rows, cols, (const uint16_t*)x, (uint16_t*)y);
  else if (io_type == MK_F32)
    launch_softmax(s, rows, cols, (const float*)x, (float*)y);
  else
    return fail(MK_ERR_UNSUPPORTED, "mk_softmax_rows: io_type must be bf16/f32");
  return check_launch("mk_softmax_rows");
}
