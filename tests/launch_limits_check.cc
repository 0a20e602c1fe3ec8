// The host side of the row kernels (src/kernels/reduce.hip), the GEMMs and
// the attention backward against a HIP runtime that only writes down its
// launches: the largest shapes the entry points take must stay within the
// 2^32 - 1 threads per grid axis that HIP launches, and products of few rows
// must run on the kernel that the dispatch rule names (attention of few queries too).  Nothing is allocated and
// nothing runs on a GPU.  Prints "ok".
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <string>
#include <utility>
#include <vector>

#include "mk_kernels.h"

namespace mk {
bool gemm_tiled_streams(int64_t batch, int64_t M, int64_t N, int64_t K, bool side_output);  // gemm_tiled.hip
}

namespace {
struct Launch {
  const void* kernel;       // its host stub
  uint64_t threads, grid;   // along x
  std::vector<void*> args;  // the first g_args arguments' first 8 bytes
};
std::vector<Launch> g_launches;
int g_args = 4;
dim3 g_grid, g_block;

void expect(bool ok, const std::string& what) {
  if (ok) return;
  std::printf("FAILED: %s\n", what.c_str());
  std::exit(1);
}
void* ptr(uint64_t v) { return reinterpret_cast<void*>(v); }

// every launch within the limit
void limits(const std::string& what, int rc) {
  expect(rc == MK_OK && !g_launches.empty(), what + ": not launched");
  for (const Launch& l : g_launches)
    expect(l.threads < (uint64_t(1) << 32), what + ": " + std::to_string(l.threads) + " threads along x");
}
// the launches' rows (argument rows_arg), each from where the one before ended
// (argument 0, a row being row_bytes), are all `rows` rows
void covers(const std::string& what, int rc, uint64_t x, int64_t rows, uint64_t row_bytes, int rows_arg) {
  limits(what, rc);
  uint64_t at = 0;
  for (const Launch& l : g_launches) {
    expect(reinterpret_cast<uint64_t>(l.args[0]) == x + at * row_bytes, what + ": a gap in the rows");
    at += reinterpret_cast<uint64_t>(l.args[rows_arg]);
  }
  expect(at == uint64_t(rows), what + ": " + std::to_string(at) + " rows of " + std::to_string(rows));
  g_launches.clear();
}
}  // namespace

// ---------------------------------------------------------------- the runtime
extern "C" {
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
void** __hipRegisterFatBinary(const void*) { return nullptr; }
void __hipRegisterFunction(void**, const void*, char*, const char*, unsigned, void*, void*, void*, void*, int*) {}
void __hipUnregisterFatBinary(void**) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t, hipStream_t) { return g_grid = g, g_block = b, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
  return *g = g_grid, *b = g_block, *lds = 0, *s = nullptr, hipSuccess;
}
hipError_t hipLaunchKernel(const void* kernel, dim3 g, dim3 b, void** args, size_t, hipStream_t) {
  Launch l{kernel, uint64_t(g.x) * b.x, g.x, {}};
  expect(g.x > 0 && g.y > 0 && g.z > 0 && g.y < 65536 && g.z < 65536, "an empty or too large grid");
  for (int i = 0; i < g_args; ++i) l.args.push_back(*static_cast<void**>(args[i]));
  return g_launches.push_back(l), hipSuccess;
}
}

namespace mk {
int sdpa_bwd_flash(hipStream_t, int64_t B, int64_t H, int64_t Sq, int64_t Sk, int64_t D, const void*, int64_t, int64_t,
                   int64_t, const void*, int64_t, int64_t, int64_t, const void*, int64_t, int64_t, int64_t, const void*,
                   int64_t, int64_t, int64_t, const void*, int64_t, int64_t, int64_t, const float*, void*, int64_t,
                   int64_t, int64_t, void*, int64_t, int64_t, int64_t, void*, int64_t, int64_t, int64_t, float, int,
                   void*);
void clear_error() {}
int fail(int code, const std::string& what) { return std::printf("%s\n", what.c_str()), code; }
int check_launch(const char*) { return MK_OK; }
}  // namespace mk

int main() {
  const uint64_t X = uint64_t(1) << 44, Y = uint64_t(1) << 46;  // never touched
  // rows at the teams' limits (2^22, 2^24 and 2^26 rows of 16, 4 and 1 waves), lengths of each team
  for (int64_t rows : {int64_t(1) << 22, (int64_t(1) << 24) - 1, (int64_t(1) << 24) + 3, (int64_t(1) << 26) - 1,
                       (int64_t(1) << 26) + 5})
    for (int64_t cols : {7, 2048, 4104, 16400, 70001, 530000})
      for (int t : {MK_BF16, MK_F32}) {
        const uint64_t row = uint64_t(cols) * (t == MK_BF16 ? 2 : 4);
        const std::string at = " of " + std::to_string(rows) + " x " + std::to_string(cols);
        covers("sum" + at, mk_row_reduce(nullptr, t, MK_F32, 0, rows, cols, ptr(X), 0.f, ptr(Y)), X, rows, row, 1);
        covers("argmax" + at, mk_row_argmax(nullptr, t, 0, rows, cols, ptr(X), nullptr, MK_S32, ptr(Y)), X, rows, row, 1);
        covers("softmax" + at, mk_softmax_rows(nullptr, t, rows, cols, ptr(X), ptr(Y)), X, rows, row, 1);
        // + 2 / 4: rows off the 16-byte grid, on the kernels that take any alignment
        covers("LayerNorm" + at, mk_layernorm(nullptr, t, rows, cols, ptr(X + (t == MK_BF16 ? 2 : 4)), nullptr, nullptr,
                                              1e-5f, ptr(Y)), X + (t == MK_BF16 ? 2 : 4), rows, row, 3);
        if (t == MK_F32)
          covers("add + LayerNorm" + at, mk_add_layernorm_typed(nullptr, t, MK_BF16, rows, cols, ptr(X + 4), ptr(X), nullptr,
                                                                nullptr, nullptr, 1e-5f, ptr(Y), ptr(Y)), X + 4, rows, row, 3);
      }

  // reduce and argmax: waves per row by rows and length, and no vectors (argument
  // 3) in short rows
  struct { int64_t rows, cols; int type; int64_t waves, vectors; } teams[] = {
      {8192, 16384, MK_F32, 4, 4096}, {65536, 2052, MK_F32, 1, 513},   {4096, 8192, MK_BF16, 1, 1024},
      {4096, 8200, MK_BF16, 4, 1025}, {4095, 4096, MK_BF16, 1, 512},   {4095, 4104, MK_BF16, 4, 513},
      {32, 50257, MK_BF16, 16, 6282}, {65536, 64, MK_BF16, 1, 0},      {65536, 100, MK_BF16, 1, 0},
      {65536, 128, MK_BF16, 1, 16},   {65536, 7, MK_F32, 1, 0},        {65536, 130, MK_F32, 1, 32}};
  for (const auto& t : teams) {
    const std::string at = " of " + std::to_string(t.rows) + " x " + std::to_string(t.cols);
    const uint64_t threads = t.waves == 1 ? (t.rows + 3) / 4 * 256 : uint64_t(t.rows) * 64 * t.waves;
    for (bool argmax : {false, true}) {
      limits("row", argmax ? mk_row_argmax(nullptr, t.type, 0, t.rows, t.cols, ptr(X), nullptr, MK_S32, ptr(Y))
                           : mk_row_reduce(nullptr, t.type, MK_F32, 1, t.rows, t.cols, ptr(X), 0.f, ptr(Y)));
      expect(g_launches[0].threads == threads, "waves per row" + at);
      expect(g_launches[0].args[3] == ptr(t.vectors), "vectors" + at);
      g_launches.clear();
    }
  }

  // the backward's row statistics: 8 or 16 lanes a row
  g_args = 0;
  for (int64_t D : {64, 128}) {
    const int64_t H = 1 << 18, Sq = D == 64 ? 2048 : 1024, n = Sq * D, z = 64 * D;
    float* lse = static_cast<float*>(ptr(X));
    limits("attention backward, head_dim " + std::to_string(D),
           mk::sdpa_bwd_flash(nullptr, 1, H, Sq, 64, D, ptr(X), 0, n, D, ptr(X), 0, z, D, ptr(X), 0, z, D, ptr(X), 0, n,
                              D, ptr(X), 0, n, D, lse, ptr(Y), 0, n, D, ptr(Y), 0, z, D, ptr(Y), 0, z, D, 1.f, 0,
                              ptr(Y)));
    g_launches.clear();
  }

  // few rows and any number of columns: up to the 2^31 (bf16) and 2^30 (fp32)
  // that 256 and 512 threads per 128 columns allow
  for (int64_t M : {1, 16, 17, 64})
    for (int64_t N : {(int64_t(1) << 28) - 1, (int64_t(1) << 28) + 1, (int64_t(1) << 29) + 5, (int64_t(1) << 30) - 128})
      for (int64_t K : {1, 64, 512, 16384})
        for (int t : {MK_BF16, MK_F32})
          for (bool kc : {false, true}) {
            limits("few rows, N " + std::to_string(N) + ", K " + std::to_string(K),
                   mk_gemm(nullptr, t, t, 1, M, N, K, ptr(X), 0, K, 1, ptr(X), 0, kc ? 1 : N, kc ? K : 1, ptr(Y), 0, N,
                           nullptr, 0));
            g_launches.clear();
          }

  // few rows: many short products stay on the 128-column tiles, deep or few
  // ones run on the kernel that reads B once (16- to 64-column workgroups)
  struct { int64_t batch, M, N, K; int type; bool kc, tiles; } routes[] = {
      {4096, 64, 512, 8, MK_BF16, false, true},    {4096, 64, 128, 128, MK_BF16, true, true},
      {512, 64, 256, 64, MK_F32, false, true},     {1, 33, 65536, 16, MK_BF16, true, true},
      {4096, 1, 1024, 128, MK_BF16, true, true},   {1, 16, 16384, 4096, MK_BF16, false, false},
      {512, 64, 64, 512, MK_BF16, false, false},   {1, 64, 4096, 8, MK_F32, true, false},
      {4096, 16, 192, 64, MK_F32, false, false},    {512, 8, 128, 2048, MK_BF16, true, false},
      {2, 64, 16384, 96, MK_F32, false, true},     {2, 64, 16384, 128, MK_F32, false, false}};
  for (const auto& r : routes) {
    limits("few rows", mk_gemm(nullptr, r.type, r.type, r.batch, r.M, r.N, r.K, ptr(X), r.M * r.K, r.K, 1, ptr(X),
                               r.K * r.N, r.kc ? 1 : r.N, r.kc ? r.K : 1, ptr(Y), r.M * r.N, r.N, nullptr, 0));
    const uint64_t tiles = (r.N + 127) / 128, block = r.type == MK_BF16 ? 256 : 512;
    expect((g_launches[0].grid == tiles && g_launches[0].threads == tiles * block) == r.tiles,
           "the kernel of " + std::to_string(r.batch) + " x " + std::to_string(r.M) + " x " + std::to_string(r.K) +
               " x " + std::to_string(r.N));
    g_launches.clear();
  }

  // tile shapes of large products: the grid's tiles name them
  struct { int64_t M, N, K; int c_type; int64_t tm, tn; } tiles[] = {
      {8192, 8192, 4096, MK_BF16, 256, 256}, {8192, 50264, 768, MK_BF16, 128, 192}, {3248, 2112, 1344, MK_F32, 128, 128},
      {15336, 416, 1408, MK_F32, 128, 128},  {8192, 6144, 2048, MK_BF16, 256, 256}, {8192, 768, 3072, MK_BF16, 128, 192},
      {1024, 8192, 2048, MK_BF16, 128, 128}, {4096, 4096, 4096, MK_BF16, 256, 256}};
  for (const auto& t : tiles) {
    limits("tiled", mk_gemm(nullptr, MK_BF16, t.c_type, 1, t.M, t.N, t.K, ptr(X), 0, t.K, 1, ptr(X), 0, t.N, 1, ptr(Y), 0,
                            t.N, nullptr, 0));
    expect(g_launches[0].grid == uint64_t((t.M + t.tm - 1) / t.tm * ((t.N + t.tn - 1) / t.tn)),
           "the tile shape of " + std::to_string(t.M) + " x " + std::to_string(t.N) + " x " + std::to_string(t.K));
    g_launches.clear();
  }

  // a 16-bit result that the next product reads is stored into the caches
  struct { int64_t batch, M, N, K; bool side, streams; } results[] = {
      {1, 2048, 4096, 1024, false, false},   {1, 256, 8192, 2048, false, false}, {1, 2300, 40000, 768, false, false},
      {12, 1024, 1024, 64, false, false},    {1, 8192, 768, 1536, false, false}, {1, 1024, 768, 3072, false, false},
      {1, 8192, 50264, 768, false, true},    {1, 2048, 4096, 1024, true, true},  {1, 8192, 768, 3072, false, true},
      {64, 2048, 2048, 128, false, true}};
  for (const auto& r : results)
    expect(mk::gemm_tiled_streams(r.batch, r.M, r.N, r.K, r.side) == r.streams,
           "the stores of " + std::to_string(r.M) + " x " + std::to_string(r.N) + " x " + std::to_string(r.K));

  // few queries, many of them beside few keys: the query-tile kernel of 17 queries
  auto kernel = [&](int64_t BH, int64_t Sq, int64_t Sk, int64_t D, int causal) {
    limits("attention", mk_sdpa_fwd(nullptr, 1, BH, Sq, Sk, D, ptr(X), 0, Sq * D, D, ptr(X), 0, Sk * D, D, ptr(X), 0,
                                    Sk * D, D, ptr(Y), 0, Sq * D, D, 1.f, causal, nullptr));
    const void* k = g_launches[0].kernel;
    return g_launches.clear(), k;
  };
  g_args = 1;
  const void *tile = kernel(64, 17, 64, 128, 0), *few = kernel(64, 1, 4096, 128, 0);
  expect(tile != few && kernel(64, 16, 64, 128, 0) == tile && kernel(256, 11, 1, 128, 0) == tile &&
             kernel(64, 10, 64, 128, 0) == few && kernel(64, 16, 65, 128, 0) == few &&
             kernel(257, 16, 64, 128, 0) == few && kernel(64, 16, 64, 64, 0) == kernel(64, 1, 4096, 64, 0) &&
             kernel(64, 1, 64, 128, 1) != few,
         "the kernel of few queries");
  expect(mk_sdpa_fwd_workspace_bytes(1, 64, 16, 64, 128, 0) == 0, "no workspace for the query-tile kernel");
  // runs of keys: heads, keys, head_dim, how many
  const int64_t runs[][4] = {{256, 1024, 128, 1}, {129, 16384, 64, 1}, {128, 2047, 128, 1}, {128, 2048, 128, 4},
                             {96, 1536, 64, 5},   {64, 767, 128, 1},   {64, 768, 128, 3},   {64, 1000, 64, 1},
                             {64, 1024, 64, 4},   {1, 16384, 128, 64}, {8, 16384, 64, 64}};
  for (const auto& r : runs)
    expect(mk_sdpa_fwd_workspace_bytes(1, r[0], 2, r[1], r[2], 0) == (r[3] == 1 ? 0 : uint64_t(r[0] * r[3] * 2 * (r[2] + 2) * 4)),
           "runs of " + std::to_string(r[1]) + " keys of " + std::to_string(r[0]) + " heads");
  std::printf("ok\n");
}
