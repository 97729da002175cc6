// C ABI glue: error text, the expert-linear entry points (kernel selection,
// bias gradient) and the host-count upload.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>

#include "gemm.h"

namespace fmoe {

static thread_local char g_err[512] = "";
// What fmoe_set_gemm_path() selected, per calling thread (a testing aid; every
// thread starts with the automatic choice).
static thread_local int g_gemm_path = 0;   // 0 = automatic, 1 = scalar kernel only
static thread_local int g_tile = 0;        // 1..4 = one MFMA tile configuration forced
static thread_local bool g_fuse_fwd_act = true;  // false: the forward activation stays a kernel

int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

// ------------------------------------------------------------ bias gradient
// db[e][c] = sum over the rows of expert e of dy[r][c], fp32 accumulation
// (fp64 for doubles).  Block = 16 column groups x 16 row lanes; a thread adds
// VEC adjacent columns of every 16th row, four independent rows in flight per
// step, then the 16 row lanes meet in LDS.  HBM-bound: reads dy once.
constexpr int kBgCols = 16, kBgRows = 16, kBgUnroll = 4;
template <typename T, int VEC>
__global__ __launch_bounds__(kBgCols * kBgRows) void bias_grad_kernel(
    const T* __restrict__ dy, const int32_t* __restrict__ seg_off,
    T* __restrict__ db, int out_feat) {
  using acc_t = typename Elem<T>::acc_t;
  struct alignas(sizeof(T) * VEC) Pk { T v[VEC]; };
  __shared__ acc_t part[kBgRows][kBgCols * VEC + 1];
  const int e = blockIdx.y;
  const int cx = threadIdx.x % kBgCols, ry = threadIdx.x / kBgCols;
  const int c0 = (blockIdx.x * kBgCols + cx) * VEC;
  const int r_begin = seg_off[e], r_end = seg_off[e + 1];
  acc_t acc[VEC];
#pragma unroll
  for (int v = 0; v < VEC; ++v) acc[v] = 0;
  if (c0 < out_feat) {
    const T* col = dy + c0;
    int r = r_begin + ry;
    for (; r + (kBgUnroll - 1) * kBgRows < r_end; r += kBgUnroll * kBgRows) {
      Pk p[kBgUnroll];
#pragma unroll
      for (int u = 0; u < kBgUnroll; ++u)
        p[u] = *reinterpret_cast<const Pk*>(col + (int64_t)(r + u * kBgRows) * out_feat);
#pragma unroll
      for (int u = 0; u < kBgUnroll; ++u)
#pragma unroll
        for (int v = 0; v < VEC; ++v) acc[v] += Elem<T>::to_acc(p[u].v[v]);
    }
    for (; r < r_end; r += kBgRows) {
      const Pk p = *reinterpret_cast<const Pk*>(col + (int64_t)r * out_feat);
#pragma unroll
      for (int v = 0; v < VEC; ++v) acc[v] += Elem<T>::to_acc(p.v[v]);
    }
  }
#pragma unroll
  for (int v = 0; v < VEC; ++v) part[ry][cx * VEC + v] = acc[v];
  __syncthreads();
  for (int c = threadIdx.x; c < kBgCols * VEC; c += kBgCols * kBgRows) {
    acc_t s = 0;
#pragma unroll
    for (int y = 0; y < kBgRows; ++y) s += part[y][c];
    const int col = blockIdx.x * kBgCols * VEC + c;
    if (col < out_feat) db[(int64_t)e * out_feat + col] = Elem<T>::from_acc(s);
  }
}

template <typename T>
static int launch_bias_grad(const void* dy, const int32_t* seg_off, void* db,
                            int out_feat, int n_expert, hipStream_t s) {
  constexpr int kVec = 16 / sizeof(T);
  const bool vec = out_feat % kVec == 0 && ((uintptr_t)dy % 16) == 0;
  if (vec) {
    dim3 grid(ceil_div(out_feat, kBgCols * kVec), n_expert);
    hipLaunchKernelGGL((bias_grad_kernel<T, kVec>), grid, dim3(kBgCols * kBgRows), 0, s,
                       (const T*)dy, seg_off, (T*)db, out_feat);
  } else {
    dim3 grid(ceil_div(out_feat, kBgCols), n_expert);
    hipLaunchKernelGGL((bias_grad_kernel<T, 1>), grid, dim3(kBgCols * kBgRows), 0, s,
                       (const T*)dy, seg_off, (T*)db, out_feat);
  }
  FMOE_LAUNCH_CHECK("bias_grad");
  return FMOE_OK;
}

// ------------------------------------------------------- host-count upload
struct OffChunk { int32_t v[512]; };
__global__ void write_offsets_kernel(OffChunk c, int32_t* dst, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = c.v[i];
}

static int check_linear(const char* who, int64_t n_rows, int64_t in_feat,
                        int64_t out_feat, int64_t n_expert, int dtype) {
  FMOE_REQUIRE(dtype_size(dtype) != 0, FMOE_ERR_INVALID, "%s: unknown dtype %d",
               who, dtype);
  FMOE_REQUIRE(n_rows >= 0 && in_feat >= 1 && out_feat >= 1 && n_expert >= 1,
               FMOE_ERR_INVALID,
               "%s: bad sizes rows=%lld in=%lld out=%lld experts=%lld", who,
               (long long)n_rows, (long long)in_feat, (long long)out_feat,
               (long long)n_expert);
  FMOE_REQUIRE(n_rows < ((int64_t)1 << 31) && in_feat < ((int64_t)1 << 31) &&
                   out_feat < ((int64_t)1 << 31) && n_expert <= 65535,
               FMOE_ERR_UNSUPPORTED, "%s: size exceeds the int32 index range", who);
  return FMOE_OK;
}

// Which family of kernels runs a product (fmoe_set_gemm_path may force one).
enum Family { kScalar, kWide, kPlain, kBig };

// `lead`: microseconds by which the 256-row kernels are behind to begin with.
static Family fwd_family(const GemmArgs& g, int dtype, double lead) {
  if (g_gemm_path != 0) return kScalar;
  const bool plain = gemm_plain_supported(g, dtype);
  if (gemm_mfma_supported(GEMM_FWD, g, dtype))
    return plain && gemm_plain_fwd_preferred(g, dtype, lead) ? kPlain : kBig;
  if (plain) return kPlain;
  return gemm_mfma_wide_supported(GEMM_FWD, g, dtype) ? kWide : kScalar;
}

// dX (gd) and dW (gw), either of which may be absent (c null).
static Family bwd_family(const GemmArgs& gd, const GemmArgs& gw, int dtype, double lead) {
  if (g_gemm_path != 0) return kScalar;
  const bool plain = gemm_plain_supported(gd, dtype) && gemm_plain_supported(gw, dtype);
  if ((!gd.c || gemm_mfma_supported(GEMM_DGRAD, gd, dtype)) &&
      (!gw.c || gemm_mfma_supported(GEMM_WGRAD, gw, dtype)))
    return plain && gemm_plain_bwd_preferred(gd, gw, dtype, lead) ? kPlain : kBig;
  if (plain) return kPlain;
  return gemm_mfma_wide_supported(GEMM_DGRAD, gd, dtype) &&
                 gemm_mfma_wide_supported(GEMM_WGRAD, gw, dtype) ? kWide : kScalar;
}

static int run_fwd(Family family, const GemmArgs& g, int dtype, hipStream_t s) {
  switch (family) {
    case kBig: return launch_gemm_mfma(GEMM_FWD, g, dtype, s);
    case kPlain: return launch_gemm_plain_fwd(g, dtype, s);
    case kWide: return launch_gemm_mfma_wide(GEMM_FWD, g, dtype, s);
    default: return launch_gemm_simt(GEMM_FWD, g, dtype, s);
  }
}

static int run_bwd(Family family, const GemmArgs& gd, const GemmArgs& gw, int dtype,
                   hipStream_t s) {
  if (family == kPlain) return launch_gemm_plain_bwd(gd, gw, dtype, s);
  if (family == kBig && gd.c && gw.c) return launch_gemm_mfma_bwd(gd, gw, dtype, s);
  for (int mode : {GEMM_DGRAD, GEMM_WGRAD}) {
    const GemmArgs& g = mode == GEMM_DGRAD ? gd : gw;
    if (!g.c) continue;
    const int rc = family == kBig ? launch_gemm_mfma(mode, g, dtype, s)
                   : family == kWide ? launch_gemm_mfma_wide(mode, g, dtype, s)
                                     : launch_gemm_simt(mode, g, dtype, s);
    if (rc) return rc;
  }
  return FMOE_OK;
}

// Up to this many values the small 16-bit tiles look the activation up in its table in
// memory while they store; a bigger product leaves it to the activation kernel, which
// keeps the table in LDS.  ReLU needs no table and always runs in the tiles (top-1 layer
// of 4096 tokens, 768 -> 3072: 178 -> 168 us).
constexpr int64_t kTableInMemoryMax = 4 << 20;

// Which kernels take an activation into their tiles.
// 256-row tiles forward: worth it from about 768 rows per expert on (measured: 12 % of GEMM +
// activation kernel at 1024 rows per expert, 5 % at 4096, level at 512, where half of the
// tiles are remainder tiles that pay the table and the second store for few rows).  Small
// tiles: f32 always (the activation costs what evaluating it costs either way, and the
// pass over memory is saved).  A forced tile shape (tests, tuning) fuses at any size.
static bool fwd_act_fused(Family family, int act, int dtype, int64_t n_rows, int64_t out_feat,
                          int64_t n_expert) {
  if (!g_fuse_fwd_act) return false;
  if (family == kBig) return dtype == FMOE_BF16 && (g_tile != 0 || n_rows >= 768 * n_expert);
  return family == kPlain && (dtype == FMOE_F32 || act == FMOE_ACT_RELU || g_tile != 0 ||
                              n_rows * out_feat <= kTableInMemoryMax);
}
static bool bwd_act_fused(Family family, int act, int dtype, int64_t n_rows, int64_t in_feat) {
  if (family == kBig) return dtype == FMOE_BF16;
  // (f16 GELU: the activation kernel rounds its product once, not through f32 first)
  return family == kPlain && (dtype != FMOE_F16 || act == FMOE_ACT_RELU) &&
         (dtype == FMOE_F32 || act == FMOE_ACT_RELU || g_tile != 0 ||
          n_rows * in_feat <= kTableInMemoryMax);
}
// A 16-bit activation as a kernel of its own: a launch and its passes over memory (measured
// 5.6 us for 64 x 4096 values, 87 for 134 million of which half are live, 60 for 92 million
// with the live rows in the last-level cache).
static double act_kernel_us(int64_t values, int passes) {
  return 5 + 2.0 * passes * (double)values / 5e6;
}

// The tables of a 16-bit GELU (a ReLU needs none, so that its first call may be captured).
static int act_tables(int act, int dtype, hipStream_t s, GemmArgs* g, bool fwd) {
  if (act != FMOE_ACT_GELU || (dtype != FMOE_BF16 && dtype != FMOE_F16)) return FMOE_OK;
  return fwd ? gelu_fwd_table(dtype, s, &g->act_fwd_table) : gelu_bwd_table(dtype, s, &g->act_table);
}

}  // namespace fmoe

using namespace fmoe;

#ifndef FMOE_SOURCE_HASH
#define FMOE_SOURCE_HASH "unknown"
#endif
// the build script puts a digest of the sources behind the "fmoe-src:" marker, so
// that a loader can tell a library built from other sources without loading it
extern "C" const char* fmoe_version(void) {
  return "fastmoe_amd 0.2 (gfx950) fmoe-src:" FMOE_SOURCE_HASH;
}
extern "C" const char* fmoe_last_error(void) { return g_err; }

// One-time set-up of the current GPU, all of which the entry points otherwise do
// at their first call: the address of fmoe_route_static's built-in buffer and the
// activation tables of the 16-bit kernels (built on `stream`, waited for).
extern "C" int fmoe_init(void* stream) {
  int rc = route_static_init();
  if (rc) return rc;
  const uint16_t* fwd = nullptr;
  const float* bwd = nullptr;
  rc = gelu_fwd_table(FMOE_BF16, (hipStream_t)stream, &fwd);
  if (rc) return rc;
  return gelu_bwd_table(FMOE_BF16, (hipStream_t)stream, &bwd);
}

extern "C" int fmoe_set_gemm_path(int path) {
  FMOE_REQUIRE(path >= 0 && path <= 12 && path != 7 && path != 10, FMOE_ERR_INVALID,
               "gemm path must be 0..6, 8, 9, 11 or 12");
  // 2..5: tile configuration 1..4 forced (16-bit types: 256 rows; 128; 64 with 128-row dW; 256
  // with K slices of 64 in two stages; f32 and odd feature sizes: their larger, smaller shape);
  // 6: automatic, but the forward activation runs as a kernel of its own behind the GEMM;
  // 8, 9: configurations 5 and 6 (16-bit types: 64 rows throughout; 128 x 256 backward)
  // 11, 12: configurations 7 and 8 (16-bit types: forward tiles of few rows, 32 x 64, 64 x 128)
  g_gemm_path = path == 1 ? 1 : 0;
  g_tile = path >= 2 && path <= 5 ? path - 1 : path >= 11 ? path - 4 : path >= 8 ? path - 3 : 0;
  g_fuse_fwd_act = path != 6;
  return FMOE_OK;
}

extern "C" int fmoe_seg_off_from_host_counts(const int64_t* expert_count_host,
                                             int64_t n_expert, int32_t* seg_off,
                                             void* stream) {
  FMOE_REQUIRE(expert_count_host && seg_off && n_expert >= 1, FMOE_ERR_INVALID,
               "seg_off_from_host_counts: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  // offsets travel as kernel arguments: no staging copy, nothing to keep alive
  int64_t run = 0;
  int64_t done = 0;  // entries of seg_off already written
  OffChunk chunk;
  int fill = 0;
  for (int64_t e = 0; e <= n_expert; ++e) {
    FMOE_REQUIRE(run >= 0 && run < ((int64_t)1 << 31), FMOE_ERR_INVALID,
                 "seg_off_from_host_counts: counts negative or too large");
    chunk.v[fill++] = (int32_t)run;
    if (e < n_expert) {
      FMOE_REQUIRE(expert_count_host[e] >= 0, FMOE_ERR_INVALID,
                   "seg_off_from_host_counts: negative count for expert %lld",
                   (long long)e);
      run += expert_count_host[e];
    }
    if (fill == 512 || e == n_expert) {
      hipLaunchKernelGGL(write_offsets_kernel, dim3(2), dim3(256), 0, s, chunk,
                         seg_off + done, fill);
      FMOE_LAUNCH_CHECK("write_offsets");
      done += fill;
      fill = 0;
    }
  }
  return FMOE_OK;
}

// Forward of the grouped linear layer, with the weights (and the bias) as one
// [E, ...] array or as tables of per-expert pointers, and optionally an activation
// behind it: y_act = act(y) from the same tiles where the kernel can, by the activation
// kernel over y otherwise.  With an activation y may be null (not kept).
static int linear_fwd(const char* who, const void* x, const void* w, const void* const* w_table,
                      const void* bias, const void* const* bias_table, const int32_t* seg_off,
                      void* y, void* y_act, int act, int64_t n_rows, int64_t in_feat,
                      int64_t out_feat, int64_t n_expert, int dtype, void* stream) {
  int rc = check_linear(who, n_rows, in_feat, out_feat, n_expert, dtype);
  if (rc) return rc;
  FMOE_REQUIRE(act >= FMOE_ACT_NONE && act <= FMOE_ACT_RELU, FMOE_ERR_INVALID,
               "%s: unknown activation %d", who, act);
  if (n_rows == 0) return FMOE_OK;
  FMOE_REQUIRE(x && (w || w_table) && seg_off && (act ? y_act : y), FMOE_ERR_INVALID,
               "%s: null pointer", who);
  hipStream_t s = (hipStream_t)stream;
  GemmArgs g{x, w, y ? y : y_act, bias, seg_off, n_rows, (int)in_feat, (int)out_feat, (int)n_expert, g_tile};
  g.w_table = w_table;
  g.bias_table = bias_table;
  // the tiles that leave the activation to its kernel pay for that in the choice: 800 rows
  // through 8 experts, 2048 -> 1024, are level in the estimate without it (and 64 x 64 tiles take
  // 15.3 us, 256-row ones 19.6) and 16.5 to 25.1 us with a GELU
  double lead = 0;
  if (act) {
    const double us = act_kernel_us(n_rows * out_feat, 2);
    lead = (fwd_act_fused(kBig, act, dtype, n_rows, out_feat, n_expert) ? 0 : us) -
           (fwd_act_fused(kPlain, act, dtype, n_rows, out_feat, n_expert) ? 0 : us);
  }
  Family family = fwd_family(g, dtype, lead);
  if (!act) return run_fwd(family, g, dtype, s);
  bool fused = (uintptr_t)y_act % 16 == 0 &&
               fwd_act_fused(family, act, dtype, n_rows, out_feat, n_expert);
  // A pre-activation whose sign is decided in its last bit switches a whole gradient on or
  // off behind a ReLU: feature sizes off the 8-element grid keep the sums in ascending order.
  if (act == FMOE_ACT_RELU && dtype != FMOE_F32 && family == kPlain &&
      !gemm_mfma_supported(GEMM_FWD, g, dtype)) {
    family = kScalar;
    fused = false;
  }
  if (fused) {
    g.act = act;
    g.act_out = y_act;
    g.c = y;
    rc = act_tables(act, dtype, s, &g, true);
    if (rc) return rc;
    return run_fwd(family, g, dtype, s);
  }
  rc = run_fwd(family, g, dtype, s);
  if (rc) return rc;
  if (act == FMOE_ACT_RELU)
    return relu_fwd(g.c, y_act, n_rows * out_feat, seg_off + n_expert, out_feat, dtype, s);
  return fmoe_gelu_fwd(g.c, y_act, n_rows * out_feat, seg_off + n_expert, out_feat, dtype, stream);
}

extern "C" int fmoe_grouped_linear_fwd(const void* x, const void* w,
                                       const void* bias, const int32_t* seg_off,
                                       void* y, int64_t n_rows, int64_t in_feat,
                                       int64_t out_feat, int64_t n_expert,
                                       int dtype, void* stream) {
  return linear_fwd("grouped_linear_fwd", x, w, nullptr, bias, nullptr, seg_off, y, nullptr,
                    FMOE_ACT_NONE, n_rows, in_feat, out_feat, n_expert, dtype, stream);
}

extern "C" int fmoe_grouped_linear_fwd_act(const void* x, const void* w, const void* bias,
                                           const int32_t* seg_off, void* y, void* y_act,
                                           int64_t n_rows, int64_t in_feat, int64_t out_feat,
                                           int64_t n_expert, int dtype, void* stream) {
  FMOE_REQUIRE(n_rows == 0 || y != nullptr, FMOE_ERR_INVALID, "grouped_linear_fwd_act: y is null");
  return linear_fwd("grouped_linear_fwd_act", x, w, nullptr, bias, nullptr, seg_off, y, y_act,
                    FMOE_ACT_GELU, n_rows, in_feat, out_feat, n_expert, dtype, stream);
}

extern "C" int fmoe_grouped_linear_fwd_ptrs(const void* x, const void* const* w_ptrs,
                                            const void* const* bias_ptrs,
                                            const int32_t* seg_off, void* y, void* y_act,
                                            int64_t n_rows, int64_t in_feat, int64_t out_feat,
                                            int64_t n_expert, int dtype, void* stream) {
  FMOE_REQUIRE(n_rows == 0 || y != nullptr, FMOE_ERR_INVALID,
               "grouped_linear_fwd_ptrs: y is null");
  return linear_fwd("grouped_linear_fwd_ptrs", x, nullptr, w_ptrs, nullptr, bias_ptrs, seg_off, y,
                    y_act, y_act ? FMOE_ACT_GELU : FMOE_ACT_NONE, n_rows, in_feat, out_feat, n_expert, dtype, stream);
}

extern "C" int fmoe_expert_linear_fwd(const void* x, const void* w, const void* const* w_ptrs,
                                      const void* bias, const void* const* bias_ptrs,
                                      const int32_t* seg_off, void* y, void* y_act, int act,
                                      int64_t n_rows, int64_t in_feat, int64_t out_feat,
                                      int64_t n_expert, int dtype, void* stream) {
  return linear_fwd("expert_linear_fwd", x, w, w_ptrs, bias, bias_ptrs, seg_off, y, y_act, act,
                    n_rows, in_feat, out_feat, n_expert, dtype, stream);
}

// A device array of pointers from a host array, written by a small kernel that
// carries the values as its arguments: no staging copy, nothing to keep alive, no
// host synchronisation.
struct PtrChunk { const void* v[256]; };
__global__ void write_pointers_kernel(PtrChunk c, const void** dst, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = c.v[i];
}

extern "C" int fmoe_pointer_table(const void* const* host_ptrs, int64_t n, const void** table,
                                  void* stream) {
  FMOE_REQUIRE(host_ptrs && table && n >= 1, FMOE_ERR_INVALID, "pointer_table: bad arguments");
  hipStream_t s = (hipStream_t)stream;
  for (int64_t done = 0; done < n; done += 256) {
    PtrChunk chunk;
    const int fill = (int)std::min<int64_t>(256, n - done);
    for (int i = 0; i < fill; ++i) chunk.v[i] = host_ptrs[done + i];
    hipLaunchKernelGGL(write_pointers_kernel, dim3(1), dim3(256), 0, s, chunk, table + done, fill);
    FMOE_LAUNCH_CHECK("write_pointers");
  }
  return FMOE_OK;
}

// Backward of the grouped linear layer; with act_pre, dx is further multiplied
// by act'(act_pre): inside the dX tiles where the kernel can, by the activation kernel over
// dx otherwise.  ReLU: act_pre may be the activation itself.
static int linear_bwd(const void* dy, const void* x, const void* w, const void* const* w_table,
                      const int32_t* seg_off, const void* act_pre, int act, void* dx, void* dw,
                      void* dbias, int64_t n_rows, int64_t in_feat, int64_t out_feat,
                      int64_t n_expert, int dtype, void* stream) {
  int rc = check_linear("grouped_linear_bwd", n_rows, in_feat, out_feat, n_expert, dtype);
  if (rc) return rc;
  FMOE_REQUIRE(seg_off != nullptr, FMOE_ERR_INVALID,
               "grouped_linear_bwd: seg_off is null");
  FMOE_REQUIRE(n_rows == 0 || dy != nullptr, FMOE_ERR_INVALID,
               "grouped_linear_bwd: dy is null");
  FMOE_REQUIRE(n_rows == 0 || !dx || w || w_table, FMOE_ERR_INVALID,
               "grouped_linear_bwd: w is null");
  FMOE_REQUIRE(n_rows == 0 || !dw || x, FMOE_ERR_INVALID, "grouped_linear_bwd: x is null");
  hipStream_t s = (hipStream_t)stream;
  if (n_rows == 0) dx = nullptr;   // (dw runs all the same: experts without rows get zeros)
  GemmArgs gw{dy, x, dw, nullptr, seg_off, n_rows, (int)in_feat, (int)out_feat, (int)n_expert, g_tile};
  GemmArgs gd{dy, w, dx, nullptr, seg_off, n_rows, (int)in_feat, (int)out_feat, (int)n_expert, g_tile};
  gd.w_table = w_table;
  double lead = 0;
  if (act_pre && dx) {
    const double us = act_kernel_us(n_rows * in_feat, 3);
    lead = (bwd_act_fused(kBig, act, dtype, n_rows, in_feat) ? 0 : us) -
           (bwd_act_fused(kPlain, act, dtype, n_rows, in_feat) ? 0 : us);
  }
  const Family family = bwd_family(gd, gw, dtype, lead);
  // The matrix-core kernels for 16-bit types and f32 sum the columns of dY inside their dW
  // tiles; f64 and the scalar kernel leave the bias gradient to the reduction kernel below.
  if (dw && dbias && (family == kBig || family == kPlain)) {
    gw.bias = dbias;
    dbias = nullptr;
  }
  const bool act_fused = act_pre && dx && (uintptr_t)act_pre % 16 == 0 &&
                         bwd_act_fused(family, act, dtype, n_rows, in_feat);
  if (act_fused) {
    gd.act = act;
    gd.act_pre = act_pre;
    rc = act_tables(act, dtype, s, &gd, false);
    if (rc) return rc;
  }
  if (dx || dw) {
    rc = run_bwd(family, gd, gw, dtype, s);
    if (rc) return rc;
  }
  if (dbias) {
    switch (dtype) {
      case FMOE_F32: rc = launch_bias_grad<float>(dy, seg_off, dbias, (int)out_feat, (int)n_expert, s); break;
      case FMOE_F64: rc = launch_bias_grad<double>(dy, seg_off, dbias, (int)out_feat, (int)n_expert, s); break;
      case FMOE_F16: rc = launch_bias_grad<__half>(dy, seg_off, dbias, (int)out_feat, (int)n_expert, s); break;
      default: rc = launch_bias_grad<__hip_bfloat16>(dy, seg_off, dbias, (int)out_feat, (int)n_expert, s); break;
    }
    if (rc) return rc;
  }
  if (act_pre && !act_fused && dx) {
    // rows of experts only: the device-side row total is the table's last entry
    if (act == FMOE_ACT_RELU)
      return relu_bwd(dx, act_pre, dx, n_rows * in_feat, seg_off + n_expert, in_feat, dtype, s);
    return fmoe_gelu_bwd(dx, act_pre, dx, n_rows * in_feat, seg_off + n_expert, in_feat, dtype,
                         stream);
  }
  return FMOE_OK;
}

extern "C" int fmoe_grouped_linear_bwd(const void* dy, const void* x,
                                       const void* w, const int32_t* seg_off,
                                       void* dx, void* dw, void* dbias,
                                       int64_t n_rows, int64_t in_feat,
                                       int64_t out_feat, int64_t n_expert,
                                       int dtype, void* stream) {
  return linear_bwd(dy, x, w, nullptr, seg_off, nullptr, FMOE_ACT_NONE, dx, dw, dbias, n_rows, in_feat,
                    out_feat, n_expert, dtype, stream);
}

extern "C" int fmoe_grouped_linear_bwd_act(const void* dy, const void* x,
                                           const void* w, const int32_t* seg_off,
                                           const void* act_pre, void* dx, void* dw,
                                           void* dbias, int64_t n_rows, int64_t in_feat,
                                           int64_t out_feat, int64_t n_expert,
                                           int dtype, void* stream) {
  FMOE_REQUIRE(act_pre != nullptr || n_rows == 0 || dx == nullptr, FMOE_ERR_INVALID,
               "grouped_linear_bwd_act: act_pre is null");
  return linear_bwd(dy, x, w, nullptr, seg_off, act_pre, FMOE_ACT_GELU, dx, dw, dbias, n_rows, in_feat,
                    out_feat, n_expert, dtype, stream);
}

extern "C" int fmoe_grouped_linear_bwd_ptrs(const void* dy, const void* x,
                                            const void* const* w_ptrs, const int32_t* seg_off,
                                            const void* act_pre, void* dx, void* dw,
                                            void* dbias, int64_t n_rows, int64_t in_feat,
                                            int64_t out_feat, int64_t n_expert,
                                            int dtype, void* stream) {
  FMOE_REQUIRE(w_ptrs != nullptr || dx == nullptr || n_rows == 0, FMOE_ERR_INVALID,
               "grouped_linear_bwd_ptrs: w_ptrs is null");
  return linear_bwd(dy, x, nullptr, w_ptrs, seg_off, act_pre, FMOE_ACT_GELU, dx, dw, dbias, n_rows, in_feat,
                    out_feat, n_expert, dtype, stream);
}

extern "C" int fmoe_expert_linear_bwd(const void* dy, const void* x, const void* w,
                                      const void* const* w_ptrs, const int32_t* seg_off,
                                      const void* act_pre, int act, void* dx, void* dw,
                                      void* dbias, int64_t n_rows, int64_t in_feat,
                                      int64_t out_feat, int64_t n_expert, int dtype,
                                      void* stream) {
  FMOE_REQUIRE(act >= FMOE_ACT_NONE && act <= FMOE_ACT_RELU, FMOE_ERR_INVALID,
               "expert_linear_bwd: unknown activation %d", act);
  FMOE_REQUIRE(act == FMOE_ACT_NONE || act_pre != nullptr || n_rows == 0 || dx == nullptr,
               FMOE_ERR_INVALID, "expert_linear_bwd: act_pre is null");
  return linear_bwd(dy, x, w, w_ptrs, seg_off, act == FMOE_ACT_NONE ? nullptr : act_pre, act, dx,
                    dw, dbias, n_rows, in_feat, out_feat, n_expert, dtype, stream);
}
