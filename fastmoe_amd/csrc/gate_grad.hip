// Gradients of the plain gate's linear map (fmoe/gates/naive_gate.py:31-38) from the routing
// results: the gradient of the logits is zero but for each token's top-k experts, so
//   dwg[e] = sum over the slots i of expert e of dl[i] * x[i / k],  dbg[e] = sum of dl[i]
// is a sum over the rows that the routing has already sorted by expert.  The dense products
// that torch makes of it leave most of the chip idle (few experts: 16384 tokens, 4096
// features, 8 experts ran on 64 workgroups) and cost four launches with the bias: 80 + 12 + 5
// us there, 86 + 15 + 5 for 8192 tokens, 2048 features, 128 experts, top-8.  Together with the
// gate's share of dx (dispatch.hip) a step of these two takes 1.2 and 2.2 % less (both sides in
// turn, within one run), one of 1000 tokens of 300 features 210 us instead of 252, of 512 of 128
// 213 instead of 248.
#include <algorithm>

#include "common.h"

namespace fmoe {
namespace {

constexpr int kThreads = 256, kWaves = 4, kWave = 64;
constexpr int kMinRows = 32;        // per workgroup
constexpr int kWantBlocks = 1024;   // four per CU: enough loads in flight for L2 and HBM
constexpr int kRowsInFlight = 8;

// Sorted rows per workgroup.
int64_t rows_per_chunk(int64_t slots, int64_t strips) {
  return std::max<int64_t>(kMinRows, std::min(slots, (slots * strips + kWantBlocks - 1) / kWantBlocks));
}

__device__ __forceinline__ float bcast(float v, int j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}
__device__ __forceinline__ double bcast(double v, int j) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), j);
  const int hi = __builtin_amdgcn_readlane((int)(b >> 32), j);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// dl[t][j] = score_j * (dscore_j - sum_i dscore_i * score_i), in the accumulation type
template <typename T>
__global__ __launch_bounds__(kThreads) void slot_grad_kernel(
    const T* __restrict__ dscore, const T* __restrict__ score,
    typename Elem<T>::acc_t* __restrict__ dl, int64_t n_tokens, int top_k) {
  using acc_t = typename Elem<T>::acc_t;
  const int64_t t = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (t >= n_tokens) return;
  acc_t dot = 0;
  for (int j = 0; j < top_k; ++j)
    dot += Elem<T>::to_acc(dscore[t * top_k + j]) * Elem<T>::to_acc(score[t * top_k + j]);
  for (int j = 0; j < top_k; ++j)
    dl[t * top_k + j] = Elem<T>::to_acc(score[t * top_k + j]) *
                        (Elem<T>::to_acc(dscore[t * top_k + j]) - dot);
}

// A workgroup adds `rows` consecutive sorted rows over a strip of 64 * VEC columns, whatever
// experts they belong to: equal work however uneven the experts are.  Chunk i leaves its sum
// for expert e in row i + e of the table of partial sums (both only grow along the rows, so no
// two meet).  A wave takes every fourth row, 64 row numbers and gradients per lane at a
// time and kRowsInFlight rows of x in flight.  Bound by the k reads of x (L2 / last-level
// cache).
template <typename T, int VEC>
__global__ __launch_bounds__(kThreads) void gate_wgrad_kernel(
    const T* __restrict__ x, const int64_t* __restrict__ pos, const int32_t* __restrict__ seg,
    const typename Elem<T>::acc_t* __restrict__ dl, typename Elem<T>::acc_t* __restrict__ part,
    typename Elem<T>::acc_t* __restrict__ part_b, int n_expert, int top_k, int64_t d, int rows) {
  using acc_t = typename Elem<T>::acc_t;
  struct alignas(sizeof(T) * VEC) Pk { T v[VEC]; };
  __shared__ acc_t sums[kWaves][kWave * VEC];
  __shared__ acc_t sums_b[kWaves];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t col0 = (int64_t)blockIdx.y * kWave * VEC;
  const int64_t col = col0 + lane * VEC;
  const bool in = col < d;             // d is a multiple of VEC
  const int live = seg[n_expert];
  int r = (int)std::min<int64_t>((int64_t)blockIdx.x * rows, live);
  const int r_end = (int)std::min<int64_t>((int64_t)blockIdx.x * rows + rows, live);
  if (r >= r_end) return;              // the same for the whole block
  int lo = 0, hi = n_expert;           // seg[lo] <= r < seg[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (seg[mid] <= r) lo = mid; else hi = mid;
  }
  for (int e = lo; r < r_end; ++e) {
    const int end = std::min(r_end, seg[e + 1]);
    if (end <= r) continue;
    acc_t acc[VEC], b = 0;
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = 0;
    for (int base = r + w; base < end; base += kWaves * kWave) {
      const int mine = base + lane * kWaves;
      int tok = 0;
      acc_t g = 0;
      if (mine < end) {
        const int64_t slot = pos[mine];
        tok = (int)(slot / top_k);
        g = dl[slot];
      }
      b += g;
      const int n = std::min(kWave, (end - base + kWaves - 1) / kWaves);
      for (int q = 0; q < n; q += kRowsInFlight) {
        // (other lanes' values are read by the whole wave: a lane beyond the last column holds
        // rows and gradients too, which a branch that leaves it out need not keep)
        Pk p[kRowsInFlight];
#pragma unroll
        for (int u = 0; u < kRowsInFlight; ++u) {
          const int row = __builtin_amdgcn_readlane(tok, q + u);
          if (q + u < n && in) p[u] = *reinterpret_cast<const Pk*>(x + (int64_t)row * d + col);
        }
#pragma unroll
        for (int u = 0; u < kRowsInFlight; ++u) {
          const acc_t gu = bcast(g, q + u);
          if (q + u < n && in) {
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] += gu * Elem<T>::to_acc(p[u].v[v]);
          }
        }
      }
    }
#pragma unroll
    for (int v = 0; v < VEC; ++v) sums[w][lane * VEC + v] = acc[v];
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) b += __shfl_xor(b, off, kWave);
    if (lane == 0) sums_b[w] = b;
    __syncthreads();
    const int64_t row = (int64_t)blockIdx.x + e;
    for (int c = threadIdx.x; c < kWave * VEC; c += kThreads)
      if (col0 + c < d)
        part[row * d + col0 + c] = (sums[0][c] + sums[1][c]) + (sums[2][c] + sums[3][c]);
    if (blockIdx.y == 0 && threadIdx.x == 0)
      part_b[row] = (sums_b[0] + sums_b[1]) + (sums_b[2] + sums_b[3]);
    __syncthreads();
    r = end;
  }
}

// The partial sums of every expert; experts without rows get zeros.
template <typename T>
__global__ __launch_bounds__(kThreads) void gate_wgrad_sum_kernel(
    const typename Elem<T>::acc_t* __restrict__ part,
    const typename Elem<T>::acc_t* __restrict__ part_b, const int32_t* __restrict__ seg,
    T* __restrict__ dwg, T* __restrict__ dbg, int64_t d, int rows) {
  using acc_t = typename Elem<T>::acc_t;
  const int e = blockIdx.y;
  const int64_t c = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int r0 = seg[e], r1 = seg[e + 1];
  const int first = r0 / rows + e, last = r1 > r0 ? (r1 - 1) / rows + e : first - 1;
  if (dwg && c < d) {
    acc_t sum = 0;
#pragma unroll 8
    for (int i = first; i <= last; ++i) sum += part[(int64_t)i * d + c];
    dwg[(int64_t)e * d + c] = Elem<T>::from_acc(sum);
  }
  if (dbg && c == 0) {
    acc_t sum = 0;
#pragma unroll 8
    for (int i = first; i <= last; ++i) sum += part_b[i];
    dbg[e] = Elem<T>::from_acc(sum);
  }
}

template <typename T>
int launch_slot_grad(const void* dscore, const void* score, void* dl, int64_t n_tokens, int top_k,
                     hipStream_t s) {
  hipLaunchKernelGGL(slot_grad_kernel<T>, dim3(ceil_div(n_tokens, kThreads)), dim3(kThreads), 0, s,
                     (const T*)dscore, (const T*)score, (typename Elem<T>::acc_t*)dl, n_tokens, top_k);
  FMOE_LAUNCH_CHECK("gate_slot_grad");
  return FMOE_OK;
}

// rows of the table of partial sums, and sorted rows per workgroup
struct Plan { int64_t vec, strips, rows, chunks, table; };
Plan make_plan(int64_t slots, int64_t d, int64_t n_expert, int dtype, const void* x) {
  const int64_t vec = 16 / (int64_t)dtype_size(dtype);
  Plan p;
  p.vec = d % vec == 0 && (uintptr_t)x % 16 == 0 ? vec : 1;
  p.strips = (d + kWave * p.vec - 1) / (kWave * p.vec);
  p.rows = rows_per_chunk(slots, p.strips);
  p.chunks = (slots + p.rows - 1) / p.rows;
  p.table = p.chunks + n_expert;
  return p;
}

template <typename T>
int launch_wgrad(const Plan& p, const void* x, const int64_t* pos, const int32_t* seg,
                 const void* dl, void* dwg, void* dbg, int top_k, int64_t d, int n_expert, void* ws,
                 hipStream_t s) {
  using acc_t = typename Elem<T>::acc_t;
  acc_t* part = (acc_t*)ws;
  acc_t* part_b = part + p.table * d;
  // (the bias alone needs one strip)
  const dim3 grid((unsigned)p.chunks, dwg ? (unsigned)p.strips : 1u);
  if (p.vec == 1)
    hipLaunchKernelGGL((gate_wgrad_kernel<T, 1>), grid, dim3(kThreads), 0, s, (const T*)x, pos, seg,
                       (const acc_t*)dl, part, part_b, n_expert, top_k, d, (int)p.rows);
  else
    hipLaunchKernelGGL((gate_wgrad_kernel<T, 16 / sizeof(T)>), grid, dim3(kThreads), 0, s,
                       (const T*)x, pos, seg, (const acc_t*)dl, part, part_b, n_expert, top_k, d,
                       (int)p.rows);
  FMOE_LAUNCH_CHECK("gate_wgrad");
  hipLaunchKernelGGL(gate_wgrad_sum_kernel<T>,
                     dim3(dwg ? (unsigned)ceil_div(d, kThreads) : 1u, (unsigned)n_expert),
                     dim3(kThreads), 0, s, part, part_b, seg, (T*)dwg, (T*)dbg, d, (int)p.rows);
  FMOE_LAUNCH_CHECK("gate_wgrad_sum");
  return FMOE_OK;
}

}  // namespace
}  // namespace fmoe

using namespace fmoe;

static int check_slots(const char* who, int64_t n_tokens, int64_t top_k, int dtype) {
  FMOE_REQUIRE(dtype_size(dtype) != 0, FMOE_ERR_INVALID, "%s: unknown dtype %d", who, dtype);
  FMOE_REQUIRE(n_tokens >= 0 && top_k >= 1 && top_k <= 64, FMOE_ERR_INVALID,
               "%s: bad sizes tokens=%lld top_k=%lld", who, (long long)n_tokens, (long long)top_k);
  FMOE_REQUIRE(n_tokens * top_k < ((int64_t)1 << 31), FMOE_ERR_UNSUPPORTED, "%s: too many slots",
               who);
  return FMOE_OK;
}

extern "C" int fmoe_gate_slot_grad(const void* dscore, const void* score, void* dslot,
                                   int64_t n_tokens, int64_t top_k, int dtype, void* stream) {
  const int rc = check_slots("gate_slot_grad", n_tokens, top_k, dtype);
  if (rc || n_tokens == 0) return rc;
  FMOE_REQUIRE(dscore && score && dslot, FMOE_ERR_INVALID, "gate_slot_grad: null pointer");
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case FMOE_F32: return launch_slot_grad<float>(dscore, score, dslot, n_tokens, (int)top_k, s);
    case FMOE_F64: return launch_slot_grad<double>(dscore, score, dslot, n_tokens, (int)top_k, s);
    case FMOE_F16: return launch_slot_grad<__half>(dscore, score, dslot, n_tokens, (int)top_k, s);
    default: return launch_slot_grad<__hip_bfloat16>(dscore, score, dslot, n_tokens, (int)top_k, s);
  }
}

static int check_linear_grad(int64_t n_tokens, int64_t top_k, int64_t d, int64_t n_expert, int dtype) {
  const int rc = check_slots("gate_linear_grad", n_tokens, top_k, dtype);
  if (rc) return rc;
  FMOE_REQUIRE(d >= 1 && d < ((int64_t)1 << 31) && n_expert >= 1 && n_expert <= 65535,
               FMOE_ERR_INVALID, "gate_linear_grad: bad sizes d=%lld experts=%lld", (long long)d,
               (long long)n_expert);
  // strips of 64 columns at the least
  FMOE_REQUIRE(d <= 65535 * 64, FMOE_ERR_UNSUPPORTED, "gate_linear_grad: d too large");
  return FMOE_OK;
}

extern "C" int64_t fmoe_gate_linear_grad_workspace_bytes(const void* x, int64_t n_tokens,
                                                         int64_t top_k, int64_t d, int32_t n_expert,
                                                         int dtype) {
  const int rc = check_linear_grad(n_tokens, top_k, d, n_expert, dtype);
  if (rc) return rc;
  const Plan p = make_plan(n_tokens * top_k, d, n_expert, dtype, x);
  return p.table * (d + 1) * (dtype == FMOE_F64 ? 8 : 4);
}

extern "C" int fmoe_gate_linear_grad(const void* x, const int64_t* pos, const int32_t* seg_off,
                                     const void* dslot, void* dwg, void* dbg, int64_t n_tokens,
                                     int64_t top_k, int64_t d, int32_t n_expert, void* workspace,
                                     int64_t workspace_bytes, int dtype, void* stream) {
  const int64_t need = fmoe_gate_linear_grad_workspace_bytes(x, n_tokens, top_k, d, n_expert, dtype);
  if (need < 0) return (int)need;
  if (!dwg && !dbg) return FMOE_OK;
  FMOE_REQUIRE(seg_off && workspace && workspace_bytes >= need && (uintptr_t)workspace % 8 == 0,
               FMOE_ERR_INVALID, "gate_linear_grad: no segments or workspace too small");
  FMOE_REQUIRE(n_tokens == 0 || (x && pos && dslot), FMOE_ERR_INVALID,
               "gate_linear_grad: null pointer");
  Plan p = make_plan(n_tokens * top_k, d, n_expert, dtype, x);
  p.chunks = std::max<int64_t>(p.chunks, 1);   // (no tokens: a block that finds no rows)
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case FMOE_F32: return launch_wgrad<float>(p, x, pos, seg_off, dslot, dwg, dbg, (int)top_k, d, n_expert, workspace, s);
    case FMOE_F64: return launch_wgrad<double>(p, x, pos, seg_off, dslot, dwg, dbg, (int)top_k, d, n_expert, workspace, s);
    case FMOE_F16: return launch_wgrad<__half>(p, x, pos, seg_off, dslot, dwg, dbg, (int)top_k, d, n_expert, workspace, s);
    default: return launch_wgrad<__hip_bfloat16>(p, x, pos, seg_off, dslot, dwg, dbg, (int)top_k, d, n_expert, workspace, s);
  }
}
