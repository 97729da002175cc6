// Top-k gate on gfx950: the k largest logits of every token and the softmax
// over those k values in one pass, and the matching backward pass.
//
// Replaces the torch.topk + F.softmax pair of fmoe/gates/naive_gate.py:31-38
// (and, in the backward, softmax-backward + zero-fill + scatter).  Results are
// ordered by descending logit; equal logits go to the lower expert index.
//
// A group of lanes shares a token.  Up to 512 experts the group (8 lanes, 32
// above 32 experts) holds all logits in registers and every one of the k
// rounds is a plain arg-max over what is still alive; above that each of 32
// lanes keeps the k best of its share as a sorted list and the rounds pop the
// overall winners.  The arrays are a few hundred KiB at most: the kernels are
// bound by launch latency and instruction count, not by memory.
#include <algorithm>

#include "common.h"

namespace fmoe {

constexpr int kGateThreads = 256;
// Lanes per token of the backward kernel: 8, and 32 from this many experts on.
constexpr int kGateWideFrom = 64;
constexpr int kGateChunk = 8;                       // logits a lane loads before it sorts them

// Order of the candidates: larger logit first, equal logits by expert index.
// A NaN logit ranks above every number (as torch.topk ranks it), so a diverged
// row selects its NaNs and its scores come out as NaN instead of being masked.
template <typename A>
__device__ __forceinline__ bool better(A v, int e, A w, int f) {
  const bool v_nan = v != v, w_nan = w != w;
  if (v_nan || w_nan) return v_nan && (!w_nan || e < f);
  return v > w || (v == w && e < f);
}

template <typename T, int KMAX, int LANES>
__global__ __launch_bounds__(kGateThreads) void topk_softmax_fwd_kernel(
    const T* __restrict__ logits, int64_t n_tokens, int n_expert, int top_k,
    int64_t* __restrict__ idx, T* __restrict__ score, float* __restrict__ zero_loss) {
  using acc_t = typename Elem<T>::acc_t;
  if (zero_loss && blockIdx.x == 0 && threadIdx.x == 0) *zero_loss = 0.f;
  const int g = threadIdx.x % LANES;
  const int64_t t = (int64_t)blockIdx.x * (kGateThreads / LANES) + threadIdx.x / LANES;
  const bool live = t < n_tokens;
  // local candidates, best first; empty slots hold (-inf, INT_MAX)
  acc_t val[KMAX];
  int id[KMAX];
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    val[j] = -INFINITY;
    id[j] = 0x7fffffff;
  }
  if (live) {
    const T* row = logits + t * n_expert;
    // kGateChunk loads in flight, then their insertions: one memory round trip
    // per chunk instead of one per logit
    for (int e0 = g; e0 < n_expert; e0 += LANES * kGateChunk) {
      T raw[kGateChunk];
#pragma unroll
      for (int u = 0; u < kGateChunk; ++u) {
        const int e = e0 + u * LANES;
        if (e < n_expert) raw[u] = row[e];
      }
#pragma unroll
      for (int u = 0; u < kGateChunk; ++u) {
        int ve = e0 + u * LANES;
        if (ve >= n_expert) break;
        acc_t v = Elem<T>::to_acc(raw[u]);
        // insertion into the sorted list: the displaced entry moves down
#pragma unroll
        for (int j = 0; j < KMAX; ++j) {
          if (better(v, ve, val[j], id[j])) {
            const acc_t tv = val[j];
            const int te = id[j];
            val[j] = v;
            id[j] = ve;
            v = tv;
            ve = te;
          }
        }
      }
    }
  }
  // k rounds: the best head of the LANES lists wins and is popped
  acc_t sel[KMAX];
  int sel_id[KMAX];
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    sel[j] = -INFINITY;
    sel_id[j] = 0;
    if (j < top_k) {
      acc_t bv = val[0];
      int be = id[0];
#pragma unroll
      for (int d = 1; d < LANES; d <<= 1) {
        const acc_t ov = __shfl_xor(bv, d, kWave);
        const int oe = __shfl_xor(be, d, kWave);
        if (better(ov, oe, bv, be)) {
          bv = ov;
          be = oe;
        }
      }
      sel[j] = bv;
      sel_id[j] = be;
      if (id[0] == be) {  // this lane held the winner: pop it
#pragma unroll
        for (int q = 0; q + 1 < KMAX; ++q) {
          val[q] = val[q + 1];
          id[q] = id[q + 1];
        }
        val[KMAX - 1] = -INFINITY;
        id[KMAX - 1] = 0x7fffffff;
      }
    }
  }
  if (!live || g != 0) return;
  // softmax over the winners; sel[0] is the largest
  acc_t p[KMAX];
  acc_t sum = 0;
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    p[j] = 0;
    if (j < top_k) {
      p[j] = exp(sel[j] - sel[0]);
      sum += p[j];
    }
  }
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    if (j < top_k) {
      idx[t * top_k + j] = sel_id[j];
      score[t * top_k + j] = Elem<T>::from_acc(p[j] / sum);
    }
  }
}

// Up to 512 experts: the LANES lanes of a token hold ALL its logits in
// registers, C each (element u of lane g is expert LANES u + g), and every
// round takes the best logit still alive: a scan of the lane's C values, a
// shuffle reduction over the group, and the owner retires the winner in a bit
// mask.  No sorted lists to maintain.
template <typename T, int LANES, int C>
__global__ __launch_bounds__(kGateThreads) void topk_softmax_fwd_flat_kernel(
    const T* __restrict__ logits, int64_t n_tokens, int n_expert, int top_k,
    int64_t* __restrict__ idx, T* __restrict__ score, float* __restrict__ zero_loss) {
  using acc_t = typename Elem<T>::acc_t;
  if (zero_loss && blockIdx.x == 0 && threadIdx.x == 0) *zero_loss = 0.f;
  constexpr int KMAX = FMOE_MAX_GATE_TOP_K;
  static_assert(C <= 32, "one bit per register in the alive mask");
  const int g = threadIdx.x % LANES;
  const int64_t t = (int64_t)blockIdx.x * (kGateThreads / LANES) + threadIdx.x / LANES;
  const bool live = t < n_tokens;
  acc_t v[C];
  uint32_t alive = 0;
#pragma unroll
  for (int u = 0; u < C; ++u) {
    const int e = u * LANES + g;
    v[u] = -INFINITY;
    if (live && e < n_expert) {
      v[u] = Elem<T>::to_acc(logits[t * n_expert + e]);
      alive |= 1u << u;
    }
  }
  acc_t sel[KMAX];
  int sel_id[KMAX];
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    sel[j] = -INFINITY;
    sel_id[j] = 0;
    if (j < top_k) {
      acc_t bv = -INFINITY;
      int be = 0x7fffffff;
#pragma unroll
      for (int u = 0; u < C; ++u) {
        const bool take = ((alive >> u) & 1u) && better(v[u], u * LANES + g, bv, be);
        bv = take ? v[u] : bv;
        be = take ? u * LANES + g : be;
      }
#pragma unroll
      for (int d = 1; d < LANES; d <<= 1) {
        const acc_t ov = __shfl_xor(bv, d, kWave);
        const int oe = __shfl_xor(be, d, kWave);
        const bool take = better(ov, oe, bv, be);
        bv = take ? ov : bv;
        be = take ? oe : be;
      }
      sel[j] = bv;
      sel_id[j] = be;
      if (be % LANES == g) alive &= ~(1u << ((be / LANES) & 31));  // no-op for "none left"
    }
  }
  if (!live || g != 0) return;
  acc_t p[KMAX];
  acc_t sum = 0;
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    p[j] = 0;
    if (j < top_k) {
      p[j] = exp(sel[j] - sel[0]);
      sum += p[j];
    }
  }
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    if (j < top_k) {
      idx[t * top_k + j] = sel_id[j];
      score[t * top_k + j] = Elem<T>::from_acc(p[j] / sum);
    }
  }
}

// dlogits[t][idx[t][j]] = score_j * (dscore_j - sum_i dscore_i * score_i), zero elsewhere.
template <typename T, int KMAX, int LANES>
__global__ __launch_bounds__(kGateThreads) void topk_softmax_bwd_kernel(
    const T* __restrict__ dscore, const T* __restrict__ score,
    const int64_t* __restrict__ idx, T* __restrict__ dlogits, int64_t n_tokens,
    int n_expert, int top_k) {
  using acc_t = typename Elem<T>::acc_t;
  const int g = threadIdx.x % LANES;
  const int64_t t = (int64_t)blockIdx.x * (kGateThreads / LANES) + threadIdx.x / LANES;
  if (t >= n_tokens) return;
  acc_t grad[KMAX];
  int id[KMAX];
  acc_t dot = 0;
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    grad[j] = 0;
    id[j] = -1;
    if (j < top_k) {
      const acc_t s = Elem<T>::to_acc(score[t * top_k + j]);
      const acc_t d = Elem<T>::to_acc(dscore[t * top_k + j]);
      dot += d * s;
      grad[j] = d;
      id[j] = (int)idx[t * top_k + j];
    }
  }
#pragma unroll
  for (int j = 0; j < KMAX; ++j)
    if (j < top_k) grad[j] = Elem<T>::to_acc(score[t * top_k + j]) * (grad[j] - dot);
  T* row = dlogits + t * n_expert;
  for (int e = g; e < n_expert; e += LANES) {
    acc_t v = 0;
#pragma unroll
    for (int j = 0; j < KMAX; ++j)
      if (id[j] == e) v = grad[j];
    row[e] = Elem<T>::from_acc(v);
  }
}

template <typename T, int KMAX>
static int launch_fwd(const void* logits, int64_t n_tokens, int n_expert, int top_k,
                      int64_t* idx, void* score, float* zero_loss, hipStream_t s) {
  const T* in = (const T*)logits;
  T* out = (T*)score;
#define FMOE_GATE_FLAT(LANES, C)                                                              \
  hipLaunchKernelGGL((topk_softmax_fwd_flat_kernel<T, LANES, C>),                             \
                     dim3(std::max(1, ceil_div(n_tokens, kGateThreads / LANES))), dim3(kGateThreads), 0, s, \
                     in, n_tokens, n_expert, top_k, idx, out, zero_loss)
  // measured at 128 experts, k = 8, 8192 tokens: 32 lanes x 4 registers 15 us,
  // 8 lanes x 16 registers 19 us (one wave per SIMD, nothing to overlap with),
  // the sorted lists 20 us
  if (n_expert <= 16) FMOE_GATE_FLAT(8, 2);
  else if (n_expert <= 32) FMOE_GATE_FLAT(8, 4);
  else if (n_expert <= 64) FMOE_GATE_FLAT(32, 2);
  else if (n_expert <= 128) FMOE_GATE_FLAT(32, 4);
  else if (n_expert <= 256) FMOE_GATE_FLAT(32, 8);
  else if (n_expert <= 512) FMOE_GATE_FLAT(32, 16);
  else
    hipLaunchKernelGGL((topk_softmax_fwd_kernel<T, KMAX, 32>),
                       dim3(std::max(1, ceil_div(n_tokens, kGateThreads / 32))), dim3(kGateThreads), 0, s, in,
                       n_tokens, n_expert, top_k, idx, out, zero_loss);
#undef FMOE_GATE_FLAT
  FMOE_LAUNCH_CHECK("topk_softmax_fwd");
  return FMOE_OK;
}

template <typename T, int KMAX>
static int launch_bwd(const void* dscore, const void* score, const int64_t* idx, void* dlogits,
                      int64_t n_tokens, int n_expert, int top_k, hipStream_t s) {
  if (n_expert >= kGateWideFrom)
    hipLaunchKernelGGL((topk_softmax_bwd_kernel<T, KMAX, 32>),
                       dim3(ceil_div(n_tokens, kGateThreads / 32)), dim3(kGateThreads), 0, s,
                       (const T*)dscore, (const T*)score, idx, (T*)dlogits, n_tokens, n_expert,
                       top_k);
  else
    hipLaunchKernelGGL((topk_softmax_bwd_kernel<T, KMAX, 8>),
                       dim3(ceil_div(n_tokens, kGateThreads / 8)), dim3(kGateThreads), 0, s,
                       (const T*)dscore, (const T*)score, idx, (T*)dlogits, n_tokens, n_expert,
                       top_k);
  FMOE_LAUNCH_CHECK("topk_softmax_bwd");
  return FMOE_OK;
}

// ------------------------------------------------------------ balance gates
// The two gates with a load-balance loss, each step of theirs that torch would run as a
// launch of its own (softmax, its mean over the tokens, the histogram, the loss) in two
// kernels forward and one backward, in f32:
//   GShard (fmoe/gates/gshard_gate.py): top-2 and the softmax over the two, loss
//     mean_e(share_e * mean_t p[t][e]) * E^2 with share_e = tokens whose first choice is e / T;
//   Switch (fmoe/gates/switch_gate.py): top-1 and its probability, loss
//     sum_e(share_e * sum_t p[t][e] / kept) * E with share_e = survivors of e / kept.
// p = softmax over all logits.  The loss's gradient reaches p[t][e] with one coefficient per
// expert (the shares are counts), which the statistics kernel leaves behind.
enum { GATE_GSHARD = FMOE_GATE_GSHARD, GATE_SWITCH = FMOE_GATE_SWITCH };
constexpr int kBalanceBlocks = 256;        // at most: rows of the table of partial sums
constexpr int kBalanceMaxExperts = 512;

// A token's logits, LANES lanes x C registers, their maximum and sum of exponentials.
template <typename T, int LANES, int C>
__device__ __forceinline__ void load_softmax(const T* logits, int64_t t, bool live, int n_expert,
                                             int g, float (&v)[C], float (&p)[C]) {
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < C; ++u) {
    const int e = u * LANES + g;
    v[u] = live && e < n_expert ? Elem<T>::to_acc(logits[t * n_expert + e]) : -INFINITY;
    m = fmaxf(m, v[u]);
  }
#pragma unroll
  for (int d = 1; d < LANES; d <<= 1) m = fmaxf(m, __shfl_xor(m, d, kWave));
  // The order of the sum is part of the result (callers compare the scores with a softmax
  // over the same logits): a wave's lane-wise halving over 64 (virtual) lanes, each summing
  // every 64th element in turn.  Registers u and u + C/2 of a lane are such a pair.
#pragma unroll
  for (int u = 0; u < C; ++u) p[u] = u * LANES + g < n_expert ? expf(v[u] - m) : 0.f;
  float sum = 0;
  if (LANES == 32) {
    float odd = 0;
#pragma unroll
    for (int u = 0; u < C; u += 2) {
      sum += p[u];
      odd += p[u + 1];
    }
    sum += odd;
  } else {
    sum = C == 4 ? (p[0] + p[C / 2]) + (p[1] + p[C - 1]) : p[0] + p[1];
  }
#pragma unroll
  for (int d = LANES / 2; d > 0; d >>= 1) sum += __shfl_xor(sum, d, kWave);
#pragma unroll
  for (int u = 0; u < C; ++u) p[u] = p[u] / sum;
}

template <typename T, int LANES, int C, int KIND>
__global__ __launch_bounds__(kGateThreads) void balance_gate_fwd_kernel(
    const T* __restrict__ logits, int64_t n_tokens, int n_expert, int64_t* __restrict__ idx,
    T* __restrict__ score, float* __restrict__ part_p, int32_t* __restrict__ part_n) {
  constexpr int kGroups = kGateThreads / LANES, K = KIND == GATE_GSHARD ? 2 : 1;
  const int g = threadIdx.x % LANES, group = threadIdx.x / LANES;
  float psum[C];
  int32_t first[C];
#pragma unroll
  for (int u = 0; u < C; ++u) {
    psum[u] = 0;
    first[u] = 0;
  }
  for (int64_t base = (int64_t)blockIdx.x * kGroups; base < n_tokens;
       base += (int64_t)gridDim.x * kGroups) {
    const int64_t t = base + group;
    const bool live = t < n_tokens;
    float v[C], p[C];
    load_softmax<T, LANES, C>(logits, t, live, n_expert, g, v, p);
    float sel[K];
    int sel_id[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
      float bv = -INFINITY;
      int be = 0x7fffffff;
#pragma unroll
      for (int u = 0; u < C; ++u) {
        const int e = u * LANES + g;
        // Switch picks among the probabilities: logits a rounding apart can share one
        const float key = KIND == GATE_SWITCH ? p[u] : v[u];
        const bool take = e < n_expert && (j == 0 || e != sel_id[0]) && better(key, e, bv, be);
        bv = take ? key : bv;
        be = take ? e : be;
      }
#pragma unroll
      for (int d = 1; d < LANES; d <<= 1) {
        const float ov = __shfl_xor(bv, d, kWave);
        const int oe = __shfl_xor(be, d, kWave);
        const bool take = better(ov, oe, bv, be);
        bv = take ? ov : bv;
        be = take ? oe : be;
      }
      sel[j] = bv;
      sel_id[j] = be;
    }
    if (live) {
#pragma unroll
      for (int u = 0; u < C; ++u) {
        psum[u] += p[u];
        first[u] += u * LANES + g == sel_id[0];
      }
      if (g == 0) {
        if (KIND == GATE_SWITCH) {
          idx[t] = sel_id[0];
          score[t] = Elem<T>::from_acc(sel[0]);
        } else {
          // (as topk_softmax_fwd_flat_kernel: the same bits)
          const float p1 = exp(sel[K - 1] - sel[0]), sum = exp(sel[0] - sel[0]) + p1;
          idx[2 * t] = sel_id[0];
          idx[2 * t + 1] = sel_id[K - 1];
          score[2 * t] = Elem<T>::from_acc(exp(sel[0] - sel[0]) / sum);
          score[2 * t + 1] = Elem<T>::from_acc(p1 / sum);
        }
      }
    }
  }
  // the groups' sums meet in LDS, in a fixed order
  __shared__ float s_p[kGroups][LANES * C];
  __shared__ int32_t s_n[kGroups][LANES * C];
#pragma unroll
  for (int u = 0; u < C; ++u) {
    s_p[group][u * LANES + g] = psum[u];
    s_n[group][u * LANES + g] = first[u];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < n_expert; e += kGateThreads) {
    float sp = 0;
    int32_t sn = 0;
    for (int q = 0; q < kGroups; ++q) {
      sp += s_p[q][e];
      sn += s_n[q][e];
    }
    part_p[(int64_t)blockIdx.x * n_expert + e] = sp;
    part_n[(int64_t)blockIdx.x * n_expert + e] = sn;
  }
}

// One block: the partial sums of all blocks -> loss and the coefficient of every expert.
constexpr int kStatThreads = 1024;
__global__ __launch_bounds__(kStatThreads) void balance_stat_kernel(
    const float* __restrict__ part_p, const int32_t* __restrict__ part_n, int n_blocks, int n_expert,
    int e_pad, int kind, int64_t n_tokens, int64_t capacity, float scale, float* __restrict__ loss,
    float* __restrict__ coef) {
  __shared__ float s_p[kStatThreads];
  __shared__ int32_t s_n[kStatThreads];
  __shared__ float s_loss[kStatThreads / kWave];
  __shared__ int32_t s_kept[kStatThreads / kWave];
  const int e = threadIdx.x % e_pad, q = threadIdx.x / e_pad, nq = kStatThreads / e_pad;
  float sp = 0;
  int32_t sn = 0;
  if (e < n_expert)
    for (int b = q; b < n_blocks; b += nq) {
      sp += part_p[(int64_t)b * n_expert + e];
      sn += part_n[(int64_t)b * n_expert + e];
    }
  s_p[threadIdx.x] = sp;
  s_n[threadIdx.x] = sn;
  __syncthreads();
  const bool owner = threadIdx.x < n_expert;   // thread e speaks for expert e from here on
  sp = 0;
  sn = 0;
  if (owner)
    for (int r = 0; r < nq; ++r) {
      sp += s_p[r * e_pad + threadIdx.x];
      sn += s_n[r * e_pad + threadIdx.x];
    }
  int32_t c = kind == GATE_SWITCH ? (int32_t)min((int64_t)sn, capacity) : sn;
  int32_t kept = c;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) kept += __shfl_xor(kept, d, kWave);
  if (threadIdx.x % kWave == 0) s_kept[threadIdx.x / kWave] = kept;
  __syncthreads();
  kept = 0;
  for (int w = 0; w < kStatThreads / kWave; ++w) kept += s_kept[w];
  // GShard: share = c / T, mean p = sp / T; Switch: both over what was kept
  const float n = kind == GATE_SWITCH ? (float)kept : (float)n_tokens;
  const float share = (float)c / n;
  float term = owner ? share * (sp / n) : 0.f;
  if (owner) coef[threadIdx.x] = share * scale / n;
#pragma unroll
  for (int d = 1; d < kWave; d <<= 1) term += __shfl_xor(term, d, kWave);
  if (threadIdx.x % kWave == 0) s_loss[threadIdx.x / kWave] = term;
  __syncthreads();
  if (threadIdx.x == 0) {
    float total = 0;
    for (int w = 0; w < kStatThreads / kWave; ++w) total += s_loss[w];
    *loss = total * scale;
  }
}

// dlogits of both paths, the selected scores' and the loss's.  dscore or dloss may be null.
template <typename T, int LANES, int C, int KIND>
__global__ __launch_bounds__(kGateThreads) void balance_gate_bwd_kernel(
    const T* __restrict__ logits, const float* __restrict__ coef, const float* __restrict__ dloss,
    const T* __restrict__ dscore, const T* __restrict__ score, const int64_t* __restrict__ idx,
    T* __restrict__ dlogits, int64_t n_tokens, int n_expert) {
  const int g = threadIdx.x % LANES;
  const int64_t t = (int64_t)blockIdx.x * (kGateThreads / LANES) + threadIdx.x / LANES;
  const bool live = t < n_tokens;
  float v[C], p[C], grad[C];
  load_softmax<T, LANES, C>(logits, t, live, n_expert, g, v, p);
  const float dl = dloss ? *dloss : 0.f;
  constexpr int K = KIND == GATE_GSHARD ? 2 : 1;
  int id[K];
  float ds[K];
#pragma unroll
  for (int j = 0; j < K; ++j) {
    id[j] = live ? (int)idx[t * K + j] : -1;
    ds[j] = live && dscore ? Elem<T>::to_acc(dscore[t * K + j]) : 0.f;
  }
  float dot = 0;
#pragma unroll
  for (int u = 0; u < C; ++u) {
    const int e = u * LANES + g;
    grad[u] = e < n_expert ? coef[e] * dl : 0.f;
    if (KIND == GATE_SWITCH && e == id[0]) grad[u] += ds[0];
    dot += p[u] * grad[u];
  }
#pragma unroll
  for (int d = 1; d < LANES; d <<= 1) dot += __shfl_xor(dot, d, kWave);
  float own[K] = {};
  if (KIND == GATE_GSHARD && live) {
    const float s0 = Elem<T>::to_acc(score[2 * t]), s1 = Elem<T>::to_acc(score[2 * t + 1]);
    const float both = ds[0] * s0 + ds[K - 1] * s1;
    own[0] = s0 * (ds[0] - both);
    own[K - 1] = s1 * (ds[K - 1] - both);
  }
  if (!live) return;
#pragma unroll
  for (int u = 0; u < C; ++u) {
    const int e = u * LANES + g;
    if (e >= n_expert) continue;
    float d = p[u] * (grad[u] - dot);
    if (KIND == GATE_GSHARD) d += e == id[0] ? own[0] : e == id[K - 1] ? own[K - 1] : 0.f;
    dlogits[t * n_expert + e] = Elem<T>::from_acc(d);
  }
}

static int64_t balance_blocks(int64_t n_tokens, int lanes) {
  const int64_t need = (n_tokens + kGateThreads / lanes - 1) / (kGateThreads / lanes);
  return std::max<int64_t>(1, std::min<int64_t>(need, kBalanceBlocks));
}

#define FMOE_BALANCE_SHAPE(CALL)                       \
  do {                                                 \
    if (n_expert <= 16) CALL(8, 2);                    \
    else if (n_expert <= 32) CALL(8, 4);               \
    else if (n_expert <= 64) CALL(32, 2);              \
    else if (n_expert <= 128) CALL(32, 4);             \
    else if (n_expert <= 256) CALL(32, 8);             \
    else CALL(32, 16);                                 \
  } while (0)

template <typename T, int KIND>
static int launch_balance_fwd(const void* logits, int64_t n_tokens, int n_expert, int64_t capacity,
                              int64_t* idx, void* score, float* loss, float* coef, void* ws,
                              hipStream_t s) {
  const int lanes = n_expert <= 32 ? 8 : 32;
  const int blocks = (int)balance_blocks(n_tokens, lanes);
  float* part_p = (float*)ws;
  int32_t* part_n = (int32_t*)(part_p + (int64_t)kBalanceBlocks * n_expert);
#define FMOE_CALL(LANES, C)                                                                  \
  hipLaunchKernelGGL((balance_gate_fwd_kernel<T, LANES, C, KIND>), dim3(blocks),             \
                     dim3(kGateThreads), 0, s, (const T*)logits, n_tokens, n_expert, idx,    \
                     (T*)score, part_p, part_n)
  FMOE_BALANCE_SHAPE(FMOE_CALL);
#undef FMOE_CALL
  FMOE_LAUNCH_CHECK("balance_gate_fwd");
  int e_pad = 1;
  while (e_pad < n_expert) e_pad *= 2;
  // GShard: mean over the experts of share * p, times E^2; Switch: their sum, times E
  hipLaunchKernelGGL(balance_stat_kernel, dim3(1), dim3(kStatThreads), 0, s, part_p, part_n, blocks,
                     n_expert, e_pad, KIND, n_tokens, capacity, (float)n_expert, loss, coef);
  FMOE_LAUNCH_CHECK("balance_stat");
  return FMOE_OK;
}

template <typename T, int KIND>
static int launch_balance_bwd(const void* logits, const float* coef, const float* dloss,
                              const void* dscore, const void* score, const int64_t* idx,
                              void* dlogits, int64_t n_tokens, int n_expert, hipStream_t s) {
#define FMOE_CALL(LANES, C)                                                                      \
  hipLaunchKernelGGL((balance_gate_bwd_kernel<T, LANES, C, KIND>),                               \
                     dim3(ceil_div(n_tokens, kGateThreads / LANES)), dim3(kGateThreads), 0, s,   \
                     (const T*)logits, coef, dloss, (const T*)dscore, (const T*)score, idx,      \
                     (T*)dlogits, n_tokens, n_expert)
  FMOE_BALANCE_SHAPE(FMOE_CALL);
#undef FMOE_CALL
  FMOE_LAUNCH_CHECK("balance_gate_bwd");
  return FMOE_OK;
}

static int check_balance(const char* who, int64_t n_tokens, int64_t n_expert, int kind, int dtype) {
  FMOE_REQUIRE(kind == GATE_GSHARD || kind == GATE_SWITCH, FMOE_ERR_INVALID, "%s: unknown gate %d",
               who, kind);
  FMOE_REQUIRE(n_tokens >= 1 && n_expert >= (kind == GATE_GSHARD ? 2 : 1), FMOE_ERR_INVALID,
               "%s: bad sizes tokens=%lld experts=%lld", who, (long long)n_tokens,
               (long long)n_expert);
  FMOE_REQUIRE(n_expert <= kBalanceMaxExperts && dtype != FMOE_F64 && dtype_size(dtype) != 0 &&
                   n_tokens < ((int64_t)1 << 31),
               FMOE_ERR_UNSUPPORTED, "%s: up to %d experts of f32, f16 or bf16", who,
               kBalanceMaxExperts);
  return FMOE_OK;
}

static int check_gate(const char* who, int64_t n_tokens, int64_t n_expert, int64_t top_k,
                      int dtype) {
  FMOE_REQUIRE(dtype_size(dtype) != 0, FMOE_ERR_INVALID, "%s: unknown dtype %d", who, dtype);
  FMOE_REQUIRE(n_tokens >= 0 && n_expert >= 1 && top_k >= 1, FMOE_ERR_INVALID,
               "%s: bad sizes tokens=%lld experts=%lld top_k=%lld", who, (long long)n_tokens,
               (long long)n_expert, (long long)top_k);
  FMOE_REQUIRE(top_k <= n_expert, FMOE_ERR_INVALID, "%s: top_k %lld exceeds %lld experts", who,
               (long long)top_k, (long long)n_expert);
  FMOE_REQUIRE(top_k <= FMOE_MAX_GATE_TOP_K, FMOE_ERR_UNSUPPORTED,
               "%s: top_k %lld exceeds FMOE_MAX_GATE_TOP_K (%d)", who, (long long)top_k,
               FMOE_MAX_GATE_TOP_K);
  FMOE_REQUIRE(n_expert < ((int64_t)1 << 31) &&
                   n_tokens < ((int64_t)1 << 31) * (kGateThreads / 32),
               FMOE_ERR_UNSUPPORTED, "%s: size exceeds the index range", who);
  return FMOE_OK;
}

}  // namespace fmoe

using namespace fmoe;

#define FMOE_GATE_DISPATCH(FN, T, ...)                         \
  (top_k <= 2 ? FN<T, 2>(__VA_ARGS__)                          \
              : top_k <= 4 ? FN<T, 4>(__VA_ARGS__)             \
                           : top_k <= 8 ? FN<T, 8>(__VA_ARGS__) : FN<T, 16>(__VA_ARGS__))

static int gate_fwd(const char* who, const void* logits, int64_t n_tokens, int32_t n_expert,
                    int32_t top_k, int64_t* idx, void* score, float* zero_loss, int dtype,
                    void* stream) {
  int rc = check_gate(who, n_tokens, n_expert, top_k, dtype);
  if (rc) return rc;
  if (n_tokens == 0 && zero_loss == nullptr) return FMOE_OK;
  FMOE_REQUIRE(n_tokens == 0 || (logits && idx && score), FMOE_ERR_INVALID, "%s: null pointer", who);
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case FMOE_F32: return FMOE_GATE_DISPATCH(launch_fwd, float, logits, n_tokens, n_expert, top_k, idx, score, zero_loss, s);
    case FMOE_F64: return FMOE_GATE_DISPATCH(launch_fwd, double, logits, n_tokens, n_expert, top_k, idx, score, zero_loss, s);
    case FMOE_F16: return FMOE_GATE_DISPATCH(launch_fwd, __half, logits, n_tokens, n_expert, top_k, idx, score, zero_loss, s);
    default: return FMOE_GATE_DISPATCH(launch_fwd, __hip_bfloat16, logits, n_tokens, n_expert, top_k, idx, score, zero_loss, s);
  }
}

extern "C" int fmoe_topk_softmax_fwd(const void* logits, int64_t n_tokens, int32_t n_expert,
                                     int32_t top_k, int64_t* idx, void* score, int dtype,
                                     void* stream) {
  return gate_fwd("topk_softmax_fwd", logits, n_tokens, n_expert, top_k, idx, score, nullptr, dtype,
                  stream);
}

extern "C" int fmoe_naive_gate_fwd(const void* logits, int64_t n_tokens, int32_t n_expert,
                                   int32_t top_k, int64_t* idx, void* score, float* zero_loss,
                                   int dtype, void* stream) {
  FMOE_REQUIRE(zero_loss != nullptr, FMOE_ERR_INVALID, "naive_gate_fwd: zero_loss is null");
  return gate_fwd("naive_gate_fwd", logits, n_tokens, n_expert, top_k, idx, score, zero_loss, dtype,
                  stream);
}

extern "C" int fmoe_topk_softmax_bwd(const void* dscore, const void* score, const int64_t* idx,
                                     void* dlogits, int64_t n_tokens, int32_t n_expert,
                                     int32_t top_k, int dtype, void* stream) {
  int rc = check_gate("topk_softmax_bwd", n_tokens, n_expert, top_k, dtype);
  if (rc) return rc;
  if (n_tokens == 0) return FMOE_OK;
  FMOE_REQUIRE(dscore && score && idx && dlogits, FMOE_ERR_INVALID,
               "topk_softmax_bwd: null pointer");
  hipStream_t s = (hipStream_t)stream;
  switch (dtype) {
    case FMOE_F32: return FMOE_GATE_DISPATCH(launch_bwd, float, dscore, score, idx, dlogits, n_tokens, n_expert, top_k, s);
    case FMOE_F64: return FMOE_GATE_DISPATCH(launch_bwd, double, dscore, score, idx, dlogits, n_tokens, n_expert, top_k, s);
    case FMOE_F16: return FMOE_GATE_DISPATCH(launch_bwd, __half, dscore, score, idx, dlogits, n_tokens, n_expert, top_k, s);
    default: return FMOE_GATE_DISPATCH(launch_bwd, __hip_bfloat16, dscore, score, idx, dlogits, n_tokens, n_expert, top_k, s);
  }
}

extern "C" int64_t fmoe_balance_gate_workspace_bytes(int32_t n_expert) {
  if (n_expert < 1) return FMOE_ERR_INVALID;
  return (int64_t)kBalanceBlocks * n_expert * 8;
}

#define FMOE_BALANCE_DISPATCH(FN, ...)                                                        \
  do {                                                                                        \
    switch (dtype) {                                                                          \
      case FMOE_F32:                                                                          \
        return kind == GATE_GSHARD ? FN<float, GATE_GSHARD>(__VA_ARGS__)                      \
                                   : FN<float, GATE_SWITCH>(__VA_ARGS__);                     \
      case FMOE_F16:                                                                          \
        return kind == GATE_GSHARD ? FN<__half, GATE_GSHARD>(__VA_ARGS__)                     \
                                   : FN<__half, GATE_SWITCH>(__VA_ARGS__);                    \
      default:                                                                                \
        return kind == GATE_GSHARD ? FN<__hip_bfloat16, GATE_GSHARD>(__VA_ARGS__)             \
                                   : FN<__hip_bfloat16, GATE_SWITCH>(__VA_ARGS__);            \
    }                                                                                         \
  } while (0)

extern "C" int fmoe_balance_gate_fwd(const void* logits, int64_t n_tokens, int32_t n_expert,
                                     int kind, int64_t capacity, int64_t* idx, void* score,
                                     float* loss, float* coef, void* workspace,
                                     int64_t workspace_bytes, int dtype, void* stream) {
  int rc = check_balance("balance_gate_fwd", n_tokens, n_expert, kind, dtype);
  if (rc) return rc;
  FMOE_REQUIRE(logits && idx && score && loss && coef, FMOE_ERR_INVALID,
               "balance_gate_fwd: null pointer");
  FMOE_REQUIRE(workspace && workspace_bytes >= fmoe_balance_gate_workspace_bytes(n_expert),
               FMOE_ERR_WORKSPACE, "balance_gate_fwd: workspace too small");
  hipStream_t s = (hipStream_t)stream;
  FMOE_BALANCE_DISPATCH(launch_balance_fwd, logits, n_tokens, n_expert, capacity, idx, score, loss,
                        coef, workspace, s);
}

extern "C" int fmoe_balance_gate_bwd(const void* logits, const float* coef, const float* dloss,
                                     const void* dscore, const void* score, const int64_t* idx,
                                     void* dlogits, int64_t n_tokens, int32_t n_expert, int kind,
                                     int dtype, void* stream) {
  int rc = check_balance("balance_gate_bwd", n_tokens, n_expert, kind, dtype);
  if (rc) return rc;
  FMOE_REQUIRE(logits && coef && (score || kind == GATE_SWITCH) && idx && dlogits,
               FMOE_ERR_INVALID, "balance_gate_bwd: null pointer");
  hipStream_t s = (hipStream_t)stream;
  FMOE_BALANCE_DISPATCH(launch_balance_bwd, logits, coef, dloss, dscore, score, idx, dlogits,
                        n_tokens, n_expert, s);
}
