// Grouped GEMM on the matrix cores for what the 256-row bf16/f16 kernels
// (gemm_mfma_impl.h) do not take, f32 of any shape and bf16/f16 whose feature sizes are
// even but no multiples of 8 (rows then start on 4-byte boundaries), and for bf16/f16 on
// 16-byte rows where the estimate at the end finds smaller tiles faster (few rows per
// expert, few tiles).
//
// One pipeline for all of them.  A workgroup of 4 waves (2 x 2) computes a BM x BN tile;
// a K slice is 128 BYTES of every operand row (32 values of f32, 64 of bf16/f16), or 64
// where that lets more workgroups share a CU; two to six LDS stages of it take turns,
// copied by `buffer_load ... lds` (16 or 4 bytes per lane, no staging registers), with one
// wait and one barrier per slice.  There is no interleaving plan as in the 256-row kernels:
// f32 MFMAs are 16 times slower, so one slice of a 64 x 128 tile is 2048 cycles of them per
// SIMD, and two to four workgroups per CU cover each other's barriers; with 4-byte copies
// (dword-aligned rows) the CU's address unit bounds the kernel (a quarter of a KiB per 20
// cycles).
//
// Both operand layouts are kept in LDS as they come:
//   K-contiguous rows  [row][128 bytes], 16-byte packs XORed by row bits;
//   K-strided          [k][rows], plain for f32, 32-byte segments XORed by k bits for
//                      bf16/f16 (ds_read_b64_tr_b16 transposes on the way to registers).
// f32 fragments: the 32x32x2 MFMA takes one value of K per lane, and WHICH value of a
// slice that is, and which row of the wave's patch, only has to agree with the other
// operand and the epilogue.  With 16-byte copies lane group g = l / 32 takes
// k = 8 s + 4 g + c in round c of group s, so a K-contiguous operand is one 16-byte read
// per four rounds; with 4-byte copies (feature sizes off the 16-byte grid) it takes
// k = 8 s + 2 c + g, i.e. the sums run over K in ascending order.  Both orders are those
// of the kernels that ran before, so results are the same bits (a ReLU behind the layer
// turns any difference of a sum around zero into a whole gradient).  Block i of lane l is
// row (l % 32) * blocks + i: a K-strided operand is then one read per round for all
// blocks, and a lane's blocks are adjacent columns of the output, so that 32 lanes store
// up to 256 contiguous bytes straight from the accumulators.
//
// Tile shape: the cost model and the measurements at the end.
#include <algorithm>
#include <climits>

#include "act_math.h"
#include "dma_desc.h"
#include "gemm_tiles.h"

namespace fmoe {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(4))) int i32x4_t;
typedef __attribute__((ext_vector_type(4))) short s16x4_t;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

constexpr int kThreads = 256, kWaves = 4;
constexpr int kSliceBytes = 128;               // of one operand row per K slice
constexpr int kRsrcFlags = 0x00020000;         // raw buffer, 32-bit data format

template <typename T> struct Half;             // the 16-bit types' instructions
template <> struct Half<__hip_bfloat16> {
  static __device__ __forceinline__ f32x4_t mma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ float add(uint32_t pair, float s) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair),
                                           __builtin_bit_cast(bf16x2_t, 0x3f803f80u), s, false);
  }
};
template <> struct Half<__half> {
  static __device__ __forceinline__ f32x4_t mma(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                  __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ float add(uint32_t pair, float s) {
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, pair),
                                  __builtin_bit_cast(f16x2_t, 0x3c003c00u), s, false);
  }
};

// One operand tile: R rows of the M or N index by one K slice.  ES bytes per element, BLOCKS
// 16-row blocks per wave, DMA bytes per lane and copy.
template <int R, int ES, int BLOCKS, bool KC, int DMA, int SB>
struct SliceTile {
  static constexpr int kBytes = R * SB;
  static constexpr int kBK = SB / ES;                 // values of K per slice
  static constexpr int kLoads = kBytes / (64 * DMA) / kWaves;  // copies per wave and slice
  static constexpr int kRowBytes = R * ES;                     // of a [k] row (not KC)
  static_assert(kBytes % (64 * DMA * kWaves) == 0 && kLoads >= 1, "tile must split evenly");

  // which of the 8 packs of a [row][128 bytes] row holds pack p: rows that the lanes of
  // one read touch together differ in the bits used here
  static __device__ __forceinline__ int row_swizzle(int row) {
    if (SB == 64) return ((row >> 4) & 1) | (((row >> 2) & 1) << 1);
    return (row / (ES == 4 ? BLOCKS : 2)) & 7;
  }
  // XOR of the 32-byte segment index of a [k] row (16-bit types)
  static __device__ __forceinline__ int k_swizzle(int k) {
    return ES == 2 ? (((k & 3) << 1) ^ ((k >> 3) & 1)) & (kRowBytes / 32 - 1) : 0;
  }

  uint32_t voff[kLoads];   // per lane: source offset of every copy
  i32x4_t rsrc;            // descriptor of the current slice; num_records ends the valid data
  int64_t remaining;       // bytes from the slice origin to the end of the valid data
  int step, k_left;

  // K value (inside the slice) of the bytes this lane copies in copy i (KC only)
  static __device__ __forceinline__ int copy_k(int i, int wave, int lane) {
    const int off = (wave * kLoads + i) * 64 * DMA + lane * DMA;
    const int row = off / SB, in = off % SB;
    return (((in / 16) ^ row_swizzle(row)) * 16 + in % 16) / ES;
  }

  __device__ __forceinline__ void init(const char* origin, int wave, int lane, int ld, int r_valid,
                                       int r_span, int k_total) {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const int off = (wave * kLoads + i) * 64 * DMA + lane * DMA;
      if (KC) {
        voff[i] = (uint32_t)(off / SB * ld + copy_k(i, wave, lane)) * ES;
      } else {
        const int k = off / kRowBytes, in = off % kRowBytes;
        const int r = (((in / 32) ^ k_swizzle(k)) * 32 + in % 32) / ES;
        voff[i] = r < r_valid ? (uint32_t)(k * ld + r) * ES : kDmaOutOfRange;
      }
    }
    int64_t bytes = 0;
    if (k_total > 0)
      bytes = KC ? ((int64_t)(r_valid - 1) * ld + k_total) * ES
                 : ((int64_t)(k_total - 1) * ld + r_span) * ES;
    remaining = ((int64_t)__builtin_amdgcn_readfirstlane((int)(bytes >> 32)) << 32) |
                (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bytes);
    step = __builtin_amdgcn_readfirstlane(KC ? SB : kBK * ld * ES);
    k_left = k_total;
    const uint64_t p = (uint64_t)origin;
    rsrc[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)p);
    rsrc[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(p >> 32) & 0xffff);
    rsrc[2] = dma_num_records(remaining);
    rsrc[3] = kRsrcFlags;
    mask_k_tail(wave, lane);
  }

  // the one slice that holds the end of K: what lies past it is pointed out of range for
  // good (the slices behind it are empty)
  __device__ __forceinline__ void mask_k_tail(int wave, int lane) {
    if (KC && k_left < kBK) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i)
        if (copy_k(i, wave, lane) >= k_left) voff[i] = kDmaOutOfRange;
    }
  }

  __device__ __forceinline__ void advance(int wave, int lane) {
    const uint64_t p = (((uint64_t)(uint32_t)rsrc[1] << 32) | (uint32_t)rsrc[0]) + (uint32_t)step;
    rsrc[0] = (int)(uint32_t)p;
    rsrc[1] = (int)(uint32_t)(p >> 32);
    remaining -= step;
    rsrc[2] = dma_num_records(remaining);
    k_left -= kBK;
    mask_k_tail(wave, lane);
  }

  // All copies of this wave for the current slice.  Inline assembly, so that the compiler
  // neither counts them nor waits for them at every LDS read: the kernel waits itself.
  __device__ __forceinline__ void issue(uint32_t tile_lds, int wave) const {
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const uint32_t dst = tile_lds + (uint32_t)(wave * kLoads + i) * (64 * DMA);
      if (DMA == 16)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     :: "s"(dst), "v"(voff[i]), "s"(rsrc) : "memory", "m0");
      else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
                     :: "s"(dst), "v"(voff[i]), "s"(rsrc) : "memory", "m0");
    }
  }

  // f32, K group s (8 values): f[c][i] = the value of K that round c multiplies, of row
  // row0 + (lane % 32) * BLOCKS + i
  static __device__ __forceinline__ void frags32(const char* lds, int row0, int s, int lane,
                                                 float (&f)[4][BLOCKS]) {
    const int a = lane & 31, g = lane >> 5;
    if (KC) {
#pragma unroll
      for (int i = 0; i < BLOCKS; ++i) {
        const int row = row0 + a * BLOCKS + i;
        const char* p = lds + row * SB;
        if (DMA == 16) {
          const f32x4_t v = *reinterpret_cast<const f32x4_t*>(p + (((s * 2 + g) ^ row_swizzle(row)) * 16));
#pragma unroll
          for (int c = 0; c < 4; ++c) f[c][i] = v[c];
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            f[c][i] = *reinterpret_cast<const float*>(
                p + (((s * 2 + c / 2) ^ row_swizzle(row)) * 16) + ((c & 1) * 2 + g) * 4);
        }
      }
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = s * 8 + (DMA == 16 ? 4 * g + c : 2 * c + g);
        const char* p = lds + k * kRowBytes + (row0 + a * BLOCKS) * 4;
        if (BLOCKS == 2) {
          const f32x2_t v = *reinterpret_cast<const f32x2_t*>(p);
#pragma unroll
          for (int i = 0; i < BLOCKS; ++i) f[c][i] = v[i];
        } else {
          f[c][0] = *reinterpret_cast<const float*>(p);
        }
      }
    }
  }

  // bf16 / f16, K group s (32 values): lane l holds row row16 + l % 16, values
  // 8 (l / 16) .. + 7 of the group
  static __device__ __forceinline__ uint4 frag16(const char* lds, int row16, int s, int lane) {
    if (KC) {
      const int row = row16 + (lane & 15);
      return *reinterpret_cast<const uint4*>(
          lds + row * SB + (((s * 4 + (lane >> 4)) ^ row_swizzle(row)) * 16));
    }
    const int k = s * 32 + 8 * (lane >> 4) + ((lane & 15) >> 2);
    const int m = row16 + 4 * (lane & 3);
    const char* p = lds + k * kRowBytes + ((m >> 4) ^ k_swizzle(k)) * 32 + (m & 15) * 2;
    const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4_t*)(p));
    const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4_t*)(p + 4 * kRowBytes));
    const uint2 l2 = __builtin_bit_cast(uint2, lo), h2 = __builtin_bit_cast(uint2, hi);
    return make_uint4(l2.x, l2.y, h2.x, h2.y);
  }
};

// A tile's shape and pipeline: BM x BN outputs, NS stages of SB bytes per operand row.
template <int BM_, int BN_, int NS_, int SB_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, NS = NS_, SB = SB_;
  // pipeline stages; the 16-bit epilogue stages an output tile in the same place
  static constexpr size_t kLds = std::max((size_t)NS * (BM + BN) * SB, (size_t)BM * (BN + 8) * 2);
};
// workgroups per CU that LDS allows, at most 4 (the registers are budgeted for them)
constexpr int workgroups_per_cu(size_t lds) {
  return std::min<int>(4, (int)(160 * 1024 / (lds + 128)));
}

// The activation behind the forward product and in front of the backward one.  GELU of the
// 16-bit types comes from the activation kernels' tables in memory (they stay in L2; these
// are small products), ReLU takes the activation itself as `pre`: its sign is all it needs.
// A NaN stays one in both directions, as in torch.
__device__ __forceinline__ float act_fwd(const GemmArgs& g, float v) {
  return g.act == FMOE_ACT_RELU ? (v < 0.f ? 0.f : v) : gelu_direct(v);
}
__device__ __forceinline__ float act_bwd(const GemmArgs& g, float d, float pre) {
  return g.act == FMOE_ACT_RELU ? (pre <= 0.f ? 0.f : d) : d * gelu_grad_direct(pre);
}
__device__ __forceinline__ uint16_t act_fwd16(const GemmArgs& g, uint16_t v) {
  return load_global<uint16_t>(g.act_fwd_table + v);
}
// (bf16; the derivative behind an f16 product is the activation kernel's)
__device__ __forceinline__ uint16_t gelu_bwd16(const GemmArgs& g, uint16_t d, uint16_t pre) {
  using B = __hip_bfloat16;
  const float n = load_global<float>(g.act_table + (pre & 0x7fffu));
  return __builtin_bit_cast(uint16_t, Elem<B>::from_acc(
      Elem<B>::to_acc(__builtin_bit_cast(B, d)) * ((pre & 0x8000u) ? n : 1.f - n)));
}

template <typename T, typename S, int MODE, int DMA>
__device__ __forceinline__ void plain_tile(const GemmArgs& g, char* smem, TileRows where,
                                           int n_origin) {
  constexpr int BM = S::BM, BN = S::BN, NS = S::NS, SB = S::SB;
  constexpr bool kF32 = std::is_same<T, float>::value;
  constexpr int ES = sizeof(T);
  // blocks of a wave: 32x32 for f32, 16x16 for the 16-bit types
  constexpr int TM = BM / 2 / (kF32 ? 32 : 16), TN = BN / 2 / (kF32 ? 32 : 16);
  using Acc = typename std::conditional<kF32, f32x16_t, f32x4_t>::type;
  constexpr bool A_KC = MODE != GEMM_WGRAD, B_KC = MODE == GEMM_FWD;
  using ATile = SliceTile<BM, ES, TM, A_KC, DMA, SB>;
  using BTile = SliceTile<BN, ES, TN, B_KC, DMA, SB>;
  constexpr int kStage = ATile::kBytes + BTile::kBytes;
  constexpr int kLoads = ATile::kLoads + BTile::kLoads;
  static_assert((NS - 2) * kLoads < 64, "vmcnt is a 6-bit counter");
  static_assert(!kF32 || (TM <= 2 && TN <= 2), "fragment reads cover 1 or 2 blocks");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m = wave >> 1, wave_n = wave & 1;
  const int in_f = g.in_feat, out_f = g.out_feat;
  const int e = __builtin_amdgcn_readfirstlane(where.e);
  const int row0 = __builtin_amdgcn_readfirstlane(where.row0);
  const int cnt = __builtin_amdgcn_readfirstlane(where.cnt);

  int M, N, K, lda, ldb, ldc;
  const T *A, *B;
  T* C;
  if (MODE == GEMM_FWD) {
    M = cnt; N = out_f; K = in_f;
    A = (const T*)g.a + (int64_t)row0 * in_f;                      lda = in_f;
    B = expert_operand<T>(g.b, g.w_table, e, (int64_t)out_f * in_f); ldb = in_f;
    C = (T*)g.c + (int64_t)row0 * out_f;                           ldc = out_f;
  } else if (MODE == GEMM_DGRAD) {
    M = cnt; N = in_f; K = out_f;
    A = (const T*)g.a + (int64_t)row0 * out_f;                     lda = out_f;
    B = expert_operand<T>(g.b, g.w_table, e, (int64_t)out_f * in_f); ldb = in_f;
    C = (T*)g.c + (int64_t)row0 * in_f;                            ldc = in_f;
  } else {
    M = out_f; N = in_f; K = cnt;
    A = (const T*)g.a + (int64_t)row0 * out_f;                     lda = out_f;
    B = (const T*)g.b + (int64_t)row0 * in_f;                      ldb = in_f;
    C = (T*)g.c + (int64_t)e * out_f * in_f;                       ldc = in_f;
  }
  const int m0 = __builtin_amdgcn_readfirstlane(where.m0);
  const int n0 = __builtin_amdgcn_readfirstlane(n_origin);
  if (m0 >= M || n0 >= N) return;   // the same for the whole block
  const int m_valid = min(BM, M - m0), n_valid = min(BN, N - n0);

  const uint32_t lds_base = (uint32_t)(size_t)(lds_ptr_t)smem;
  ATile ta;
  BTile tb;
  ta.init((const char*)(A_KC ? A + (int64_t)m0 * lda : A + m0), wave, lane, lda, m_valid, M - m0, K);
  tb.init((const char*)(B_KC ? B + (int64_t)n0 * ldb : B + n0), wave, lane, ldb, n_valid, N - n0, K);

  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = (Acc)(0.f);

  // dW tiles of the first column also sum the columns of dY: the bias gradient
  const bool colsum = MODE == GEMM_WGRAD && g.bias != nullptr && n0 == 0;
  float cs[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) cs[i] = 0.f;

  const int k_tiles = (K + ATile::kBK - 1) / ATile::kBK;
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) {
    ta.issue(lds_base + s * kStage, wave);
    tb.issue(lds_base + s * kStage + ATile::kBytes, wave);
    ta.advance(wave, lane);
    tb.advance(wave, lane);
  }
  int stage = 0;
  for (int kt = 0; kt < k_tiles; ++kt) {
    // slice kt has landed here (my share) and, behind the barrier, everywhere; behind it
    // nobody reads the stage of slice kt - 1 any more, which slice kt + NS - 1 takes
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * kLoads) : "memory");
    __syncthreads();
    const int free_stage = stage == 0 ? NS - 1 : stage - 1;
    ta.issue(lds_base + free_stage * kStage, wave);
    tb.issue(lds_base + free_stage * kStage + ATile::kBytes, wave);
    ta.advance(wave, lane);
    tb.advance(wave, lane);
    const char* la = smem + stage * kStage;
    const char* lb = la + ATile::kBytes;
    if constexpr (kF32) {
#pragma unroll
      for (int s = 0; s < SB / 32; ++s) {
        float fa[4][TM], fb[4][TN];
        ATile::frags32(la, wave_m * (BM / 2), s, lane, fa);
        BTile::frags32(lb, wave_n * (BN / 2), s, lane, fb);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[c][i], fb[c][j], acc[i][j], 0, 0, 0);
        }
        if (MODE == GEMM_WGRAD && colsum) {
#pragma unroll
          for (int i = 0; i < TM; ++i) cs[i] += (fa[0][i] + fa[1][i]) + (fa[2][i] + fa[3][i]);
        }
      }
    } else {
#pragma unroll
      for (int s = 0; s < SB / 64; ++s) {
        uint4 fa[TM], fb[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[i] = ATile::frag16(la, wave_m * (BM / 2) + i * 16, s, lane);
#pragma unroll
        for (int j = 0; j < TN; ++j) fb[j] = BTile::frag16(lb, wave_n * (BN / 2) + j * 16, s, lane);
        // operands swapped: a lane then owns 4 adjacent columns of a row of C
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = Half<T>::mma(fb[j], fa[i], acc[i][j]);
        if (MODE == GEMM_WGRAD && colsum) {
#pragma unroll
          for (int i = 0; i < TM; ++i) {
            cs[i] = Half<T>::add(fa[i].x, cs[i]);
            cs[i] = Half<T>::add(fa[i].y, cs[i]);
            cs[i] = Half<T>::add(fa[i].z, cs[i]);
            cs[i] = Half<T>::add(fa[i].w, cs[i]);
          }
        }
      }
    }
    stage = stage + 1 == NS ? 0 : stage + 1;
  }
  // the zero-filled slices past the end of K are still landing; behind the barrier the LDS
  // is free to stage an output tile
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  const int a = lane & (kF32 ? 31 : 15), gr = lane / (kF32 ? 32 : 16);
  if (MODE == GEMM_WGRAD && colsum) {
    T* db = (T*)const_cast<void*>(g.bias) + (int64_t)e * out_f;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      float total = cs[i] + __shfl_xor(cs[i], 32, 64);
      if (!kF32) total += __shfl_xor(total, 16, 64);
      const int m = m0 + wave_m * (BM / 2) + (kF32 ? a * TM + i : i * 16 + a);
      if (wave_n == 0 && gr == 0 && m < M) db[m] = Elem<T>::from_acc(total);
    }
  }

  const T* bias = MODE == GEMM_FWD ? expert_operand<T>(g.bias, g.bias_table, e, out_f) : nullptr;
  if constexpr (kF32) {
    // accumulator r of block (i, j): row (8 (r / 4) + 4 gr + r % 4) TM + i, column a TN + j
    struct alignas(DMA == 16 ? 4 * TN : 4) Vec { float v[TN]; };
    const int col = n0 + wave_n * (BN / 2) + a * TN;
    float bv[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
      bv[j] = bias && col + j < N ? load_global<float>(bias + col + j) : 0.f;
    const float* pre = MODE == GEMM_DGRAD ? (const float*)g.act_pre : nullptr;
    float* act_out = MODE == GEMM_FWD ? (float*)g.act_out : nullptr;
#pragma unroll
    for (int r = 0; r < 16; ++r)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = wave_m * (BM / 2) + (8 * (r / 4) + 4 * gr + r % 4) * TM + i;
        if (m >= m_valid || col >= N) continue;
        Vec o;
#pragma unroll
        for (int j = 0; j < TN; ++j) o.v[j] = acc[i][j][r] + bv[j];
        const int64_t at = (int64_t)(m0 + m) * ldc + col;
        const bool whole = DMA == 16 || col + TN <= N;   // 16-byte rows: N is a multiple of 4
        if (MODE == GEMM_DGRAD && pre) {
          const float* p = pre + (int64_t)row0 * ldc + at;
          Vec x;
          if (whole) {
            x = *reinterpret_cast<const Vec*>(p);
          } else {
#pragma unroll
            for (int j = 0; j < TN; ++j) x.v[j] = col + j < N ? p[j] : 0.f;
          }
#pragma unroll
          for (int j = 0; j < TN; ++j) o.v[j] = act_bwd(g, o.v[j], x.v[j]);
        }
        if (MODE == GEMM_FWD && g.c == nullptr) {   // only the activation is wanted
        } else if (whole) {
          *reinterpret_cast<Vec*>(C + at) = o;
        } else {
#pragma unroll
          for (int j = 0; j < TN; ++j)
            if (col + j < N) C[at + j] = o.v[j];
        }
        if (MODE == GEMM_FWD && act_out) {
          float* q = act_out + (int64_t)row0 * ldc + at;
#pragma unroll
          for (int j = 0; j < TN; ++j) o.v[j] = act_fwd(g, o.v[j]);
          if (whole) {
            *reinterpret_cast<Vec*>(q) = o;
          } else {
#pragma unroll
            for (int j = 0; j < TN; ++j)
              if (col + j < N) q[j] = o.v[j];
          }
        }
      }
  } else {
    // Accumulator r of block (i, j) is row 16 i + a, column 16 j + 4 gr + r of the patch: the
    // tile goes through LDS (rows padded by 16 bytes) and leaves in units of 16 bytes (4
    // where rows start on 4-byte boundaries), 128 to 256 contiguous bytes per row.
    constexpr int kLdc = BN + 8, kUnit = DMA / 2;             // elements
    constexpr int kRowUnits = BN / kUnit, kUnits = BM * kRowUnits / kThreads;
  
    using Unit = typename std::conditional<DMA == 16, uint4, uint32_t>::type;
    uint16_t* staged = reinterpret_cast<uint16_t*>(smem);
    // pre-activations (ReLU: activations) in front of the dX product: under way while the
    // tile is staged
    constexpr bool kDgrad = MODE == GEMM_DGRAD, kFwd = MODE == GEMM_FWD;
    const uint16_t* pre = kDgrad ? (const uint16_t*)g.act_pre : nullptr;
    Unit pv[kDgrad ? kUnits : 1];
    if (kDgrad && pre) {
#pragma unroll
      for (int u = 0; u < kUnits; ++u) {
        const int m = (tid + u * kThreads) / kRowUnits, c = (tid + u * kThreads) % kRowUnits * kUnit;
        pv[u] = Unit{};
        if (m < m_valid && c < n_valid)
          pv[u] = *reinterpret_cast<const Unit*>(pre + (int64_t)(row0 + m0 + m) * ldc + n0 + c);
      }
    }
    __syncthreads();
    // The branches on the activation stay outside the loops over elements: inside them they
    // cost more than a pass over memory (4096 x 3072 bf16 ReLU: 71 us, and 62 + 10 with a kernel
    // of its own).  A ReLU whose argument nobody wants is applied before the rounding: zero
    // for everything that rounds to a negative number or to either zero.
    const bool relu = g.act == FMOE_ACT_RELU, relu_early = kFwd && relu && g.c == nullptr;
    const float floor_v = relu_early ? 0.f : -INFINITY;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = wave_n * (BN / 2) + j * 16 + 4 * gr;
      float bv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        bv[r] = bias && n0 + col + r < N ? Elem<T>::to_acc(load_global<T>(bias + n0 + col + r)) : 0.f;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        struct alignas(8) Quad { T v[4]; } o;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
          const float v = kFwd ? acc[i][j][r] + bv[r] : acc[i][j][r];
          o.v[r] = Elem<T>::from_acc(kFwd && v <= floor_v ? floor_v : v);
        }
        *reinterpret_cast<Quad*>(staged + (wave_m * (BM / 2) + i * 16 + a) * kLdc + col) = o;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kUnits; ++u) {
      const int m = (tid + u * kThreads) / kRowUnits, c = (tid + u * kThreads) % kRowUnits * kUnit;
      if (m >= m_valid || c >= n_valid) continue;   // N is a multiple of the unit
      const int64_t at = (int64_t)(m0 + m) * ldc + n0 + c;
      union { Unit u; uint16_t h[kUnit]; } v, p;
      v.u = *reinterpret_cast<const Unit*>(staged + m * kLdc + c);
      if (kDgrad && pre) {
        p.u = pv[u];
        if (relu) {
#pragma unroll
          for (int q = 0; q < kUnit; ++q) v.h[q] = relu_bwd16<T>(v.h[q], p.h[q]);
        } else if constexpr (std::is_same<T, __hip_bfloat16>::value) {
#pragma unroll
          for (int q = 0; q < kUnit; ++q) v.h[q] = gelu_bwd16(g, v.h[q], p.h[q]);
        }
      }
      if (!kFwd || g.c) *reinterpret_cast<Unit*>(C + at) = v.u;
      if (kFwd && g.act_out) {
        if (relu) {
          if (!relu_early) {
#pragma unroll
            for (int q = 0; q < kUnit; ++q) v.h[q] = relu_fwd16<T>(v.h[q]);
          }
        } else {
#pragma unroll
          for (int q = 0; q < kUnit; ++q) v.h[q] = act_fwd16(g, v.h[q]);
        }
        *reinterpret_cast<Unit*>((uint16_t*)g.act_out + (int64_t)row0 * ldc + at) = v.u;
      }
    }
  }
}

template <typename T, typename S, int DMA>
__global__ __launch_bounds__(kThreads, (workgroups_per_cu(S::kLds))) void plain_fwd_kernel(
    GemmArgs g, int tiles_n) {
  extern __shared__ __attribute__((aligned(1024))) char plain_smem[];
  __shared__ int s_owner[4], s_wave_sum[2 * kWaves];
  RowTiles<S::BM, kOneHeight, kWaves> rows;
  rows.scan(g.seg_off, g.n_expert, s_wave_sum);
  const int live = rows.rows_f * tiles_n;
  if (live == 0) return;
  const int t = tile_number(blockIdx.x, live);
  if (t >= live) return;
  int v, n_tile;
  tile_order(t, rows.rows_f, tiles_n, v, n_tile);
  const TileRows where = rows.find(g.seg_off, v, false, s_owner);
  plain_tile<T, S, GEMM_FWD, DMA>(g, plain_smem, where, n_tile * S::BN);
}

// Forward product of few rows per expert on average, cut by the rows that each expert really
// has: tiles Low, but tiles High for experts of more than kFewRows rows where these fill the
// chip.  Low tiles of a long expert copy its weights into LDS again and again; while there are
// fewer High tiles than CUs, though, the wait for memory counts and not the copies, and Low
// tiles spread it wider.  Measured: see low_rows().
constexpr int kFewRows = 64, kCus = 256;
template <typename T, typename Low, typename High, int DMA>
__global__ __launch_bounds__(kThreads, (workgroups_per_cu(std::max(Low::kLds, High::kLds)))) void
plain_fwd_few_kernel(GemmArgs g, int tiles_n_low, int tiles_n_high) {
  extern __shared__ __attribute__((aligned(1024))) char plain_smem[];
  __shared__ int s_owner[4], s_wave_sum[2 * kWaves];
  RowTiles<High::BM, kTwoHeights, kWaves, Low::BM> rows;
  rows.low_most = kFewRows;
  rows.scan(g.seg_off, g.n_expert, s_wave_sum);
  if (rows.rows_f > 0 && rows.rows_f * tiles_n_high < kCus) {
    rows.low_most = INT_MAX;
    __syncthreads();   // the sums of the first scan have been read
    rows.scan(g.seg_off, g.n_expert, s_wave_sum);
  }
  const int live_high = rows.rows_f * tiles_n_high;
  const int live = live_high + rows.rows_s * tiles_n_low;
  if (live == 0) return;
  const int t = tile_number(blockIdx.x, live);
  if (t >= live) return;
  int v, n_tile;
  if (t < live_high) {
    tile_order(t, rows.rows_f, tiles_n_high, v, n_tile);
    const TileRows where = rows.find(g.seg_off, v, false, s_owner);
    plain_tile<T, High, GEMM_FWD, DMA>(g, plain_smem, where, n_tile * High::BN);
  } else {
    tile_order(t - live_high, rows.rows_s, tiles_n_low, v, n_tile);
    const TileRows where = rows.find(g.seg_off, v, true, s_owner);
    plain_tile<T, Low, GEMM_FWD, DMA>(g, plain_smem, where, n_tile * Low::BN);
  }
}

// dX (tiles D) and dW with the bias gradient (tiles W) in one launch, dX tiles first;
// either may be absent (no tiles).
template <typename T, typename D, typename W, int DMA>
__global__ __launch_bounds__(kThreads, (workgroups_per_cu(std::max(D::kLds, W::kLds)))) void
plain_bwd_kernel(GemmArgs gd, GemmArgs gw, int tiles_n_d, int tiles_n_w, int tiles_m_w) {
  extern __shared__ __attribute__((aligned(1024))) char plain_smem[];
  __shared__ int s_owner[4], s_wave_sum[2 * kWaves];
  RowTiles<D::BM, kOneHeight, kWaves> rows;
  rows.scan(gd.seg_off, gd.n_expert, s_wave_sum);
  const int live_d = rows.rows_f * tiles_n_d;
  const int per_expert_w = tiles_n_w * tiles_m_w;
  const int live = live_d + per_expert_w * gw.n_expert;
  if (live == 0) return;
  const int t = tile_number(blockIdx.x, live);
  if (t >= live) return;
  if (t >= live_d) {
    const int tw = t - live_d, e = tw / per_expert_w;
    int m_tile, n_tile;
    tile_order(tw % per_expert_w, tiles_m_w, tiles_n_w, m_tile, n_tile);
    const int row0 = gw.seg_off[e];
    plain_tile<T, W, GEMM_WGRAD, DMA>(
        gw, plain_smem, {e, m_tile * W::BM, row0, gw.seg_off[e + 1] - row0}, n_tile * W::BN);
    return;
  }
  int v, n_tile;
  tile_order(t, rows.rows_f, tiles_n_d, v, n_tile);
  const TileRows where = rows.find(gd.seg_off, v, false, s_owner);
  plain_tile<T, D, GEMM_DGRAD, DMA>(gd, plain_smem, where, n_tile * D::BN);
}

// ------------------------------------------------------------------ host side
int round_up_blocks(int64_t tiles, unsigned* blocks) {
  const int64_t b = ceil_div(tiles, 8 * kXcdRun) * (int64_t)(8 * kXcdRun);
  FMOE_REQUIRE(b < ((int64_t)1 << 31), FMOE_ERR_UNSUPPORTED, "grouped GEMM: too many tiles");
  *blocks = (unsigned)b;
  return FMOE_OK;
}

template <typename T, typename S, int DMA>
int launch_fwd(const GemmArgs& g, hipStream_t s) {
  auto kern = plain_fwd_kernel<T, S, DMA>;
  FMOE_SET_DYNAMIC_LDS_ONCE(kern, S::kLds);
  const int tiles_n = ceil_div(g.out_feat, S::BN);
  unsigned blocks = 0;
  const int rc = round_up_blocks(tiles_n * (g.n_rows / S::BM + (int64_t)g.n_expert), &blocks);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kThreads), S::kLds, s, g, tiles_n);
  FMOE_LAUNCH_CHECK("gemm_plain");
  return FMOE_OK;
}

template <typename T, typename Low, typename High, int DMA>
int launch_fwd_few(const GemmArgs& g, hipStream_t s) {
  static_assert(Low::BM <= High::BM && Low::BN <= High::BN, "Low must be the smaller tile");
  constexpr size_t lds = std::max(Low::kLds, High::kLds);
  auto kern = plain_fwd_few_kernel<T, Low, High, DMA>;
  FMOE_SET_DYNAMIC_LDS_ONCE(kern, lds);
  const int tiles_n_low = ceil_div(g.out_feat, Low::BN);
  const int tiles_n_high = ceil_div(g.out_feat, High::BN);
  unsigned blocks = 0;
  // (an expert in High tiles has no more of them than it would have of Low ones)
  const int rc = round_up_blocks(tiles_n_low * (g.n_rows / Low::BM + (int64_t)g.n_expert), &blocks);
  if (rc) return rc;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kThreads), lds, s, g, tiles_n_low, tiles_n_high);
  FMOE_LAUNCH_CHECK("gemm_plain");
  return FMOE_OK;
}

template <typename T, typename D, typename W, int DMA>
int launch_bwd(const GemmArgs& gd, const GemmArgs& gw, hipStream_t s) {
  constexpr size_t lds = std::max(D::kLds, W::kLds);
  auto kern = plain_bwd_kernel<T, D, W, DMA>;
  FMOE_SET_DYNAMIC_LDS_ONCE(kern, lds);
  const int tiles_n_d = gd.c ? ceil_div(gd.in_feat, D::BN) : 0;
  const int tiles_n_w = gw.c ? ceil_div(gw.in_feat, W::BN) : 0;
  const int tiles_m_w = ceil_div(gw.out_feat, W::BM);
  unsigned blocks = 0;
  const int rc = round_up_blocks(tiles_n_d * (gd.n_rows / D::BM + (int64_t)gd.n_expert) +
                                     (int64_t)tiles_n_w * tiles_m_w * gw.n_expert, &blocks);
  if (rc || blocks == 0) return rc;
  hipLaunchKernelGGL(kern, dim3(blocks), dim3(kThreads), lds, s, gd, gw, tiles_n_d, tiles_n_w,
                     tiles_m_w);
  FMOE_LAUNCH_CHECK("gemm_plain_bwd");
  return FMOE_OK;
}

// Tile shape: the matrix cores of a CU take `us` per K slice of a tile, whatever the
// number of workgroups that share them, and at least one whole tile is walked.  The tiles
// of a launch are dealt over 256 CUs, half-way between evenly and in whole rounds.  The
// shape with the least estimated time wins: the bigger one where there are enough tiles of
// it, the smaller one where the chip would idle.
struct Shape { int bm, bn; double us; };
double rounds(double tiles) { return std::max(1.0, 0.5 * (tiles / 256 + ceil(tiles / 256))); }

// every expert's last row tile is half empty on average
double row_tiles(const GemmArgs& g, int bm) {
  return (double)g.n_rows / bm + 0.5 * g.n_expert;
}

// Two stages and as many workgroups per CU as fit: they cover each other's waits better
// than more stages do.  Measured in f32, forward / dX + dW, us (4 stages of the 64 x 64
// tile, 2 of 128 x 128, 64 x 128, 64 x 64, against the register-staged 128 x 128 kernel
// before):
//   4 experts, 1024 rows, 128 -> 256       8.0/10.0  15.5/25.4  9.7/14.7  7.6/10.0  (26/50)
//   8 experts, 4000 rows, 512 -> 2048      106/169   118/208    90/163    88/151    (110/250)
//   8 experts, 4000 rows, 2048 -> 512      126/175   138/171    128/158   109/156   (160/255)
//   32 experts, 15567 rows, 512 -> 2176    393/642   336/619    300/560   320/588
//   64 experts, 32000 rows, 1024 -> 4096   2741/4897 2245/4288  2110/4261 2296/4460 (127 TFLOP/s)
constexpr Shape kShapesF32[2] = {{64, 128, 1.06}, {64, 64, 0.56}};
// bound by the address unit: 4-byte copies
constexpr Shape kShapes16[2] = {{128, 128, 1.36}, {64, 64, 0.42}};

int fwd_shape(const GemmArgs& g, const Shape (&shapes)[2], int es) {
  if (g.tile) return (g.tile - 1) % 2;   // forced (tests)
  const double slices = ceil_div((int64_t)g.in_feat * es, kSliceBytes);
  double cost[2];
  for (int i = 0; i < 2; ++i)
    cost[i] = rounds(row_tiles(g, shapes[i].bm) * ceil_div(g.out_feat, shapes[i].bn)) * slices *
              shapes[i].us;
  return cost[0] <= cost[1] ? 0 : 1;
}

// Both gradients share one shape: the estimate counts the tiles of both, each with its own
// number of slices.
int bwd_shape(const GemmArgs& gd, const GemmArgs& gw, const Shape (&shapes)[2], int es) {
  const int forced = gd.tile ? gd.tile : gw.tile;
  if (forced) return (forced - 1) % 2;
  const double ks_d = gd.c ? ceil_div((int64_t)gd.out_feat * es, kSliceBytes) : 0;
  const double ks_w = gw.c ? (double)gw.n_rows / gw.n_expert * es / kSliceBytes + 0.5 : 0;
  double cost[2];
  for (int i = 0; i < 2; ++i) {
    const double td = row_tiles(gd, shapes[i].bm) * ceil_div(gd.in_feat, shapes[i].bn);
    const double tw = (double)gw.n_expert * ceil_div(gw.out_feat, shapes[i].bm) *
                      ceil_div(gw.in_feat, shapes[i].bn);
    // (the last tiles to finish run alone for a while: a fifth of the longest)
    const double longest = std::max(ks_d, ks_w);
    cost[i] = std::max(longest, (td * ks_d + tw * ks_w) / 256 + 0.2 * longest) * shapes[i].us;
  }
  return cost[0] <= cost[1] ? 0 : 1;
}

// ---- bf16 / f16 on 16-byte rows: this file's tiles or the 256-row kernels?
//
// Estimated microseconds of a launch from the experts' average number of rows (and what
// random routing spreads around it).  Per tile: a fixed cost and a cost per K slice, alone
// on its CU or sharing it; per launch: what HBM needs for the operands and results.  The
// constants are fits to measured launches (us: 256-row kernels, 128 x 128, 64 x 64 tiles):
//   forward  16 experts,   64 rows, 1024 -> 4096     25   24   25
//            16,   64, 4096 -> 1024                  24   55   23
//             8,  128, 14336 -> 4096                179  221  162
//            32, 4096, 3072 -> 768                   81   41   49
//            16, 6002, 768 -> 3072                   52   53   75
//             8, 2000, 256 -> 1024                   13  8.4  7.2
//           128, 16376, 2048 -> 1408                190  235  270
//            32, 16000, 1024 -> 2048                 88  108  154
//   dX + dW (and 64 x 64 dX tiles with 128 x 128 dW tiles of half slices)
//            16,   64, 1024 -> 4096                  80   78   83  (61)
//             8,  128, 14336 -> 4096                470  521  632  (382)
//            32, 4096, 768 -> 3072                  143   92  140  (105)
//             4, 1000, 256 -> 512                    16  9.6  7.1  (8.2)
//             8, 8000, 512 -> 2048                   56   49   69  (71)
//            32, 16000, 1024 -> 2048                167  196  275
//          (128 x 256 tiles, dX + dW, against the best of the others)
//            64, 18790, 1152 -> 4032           627  581  648   543
//            32, 8307, 2304 -> 1536            221  210  237   186
//           128, 16376, 2048 -> 1408           469  513  511   446
//             8, 16620, 1664 -> 3328           355  377  474   370
//             4, 24620, 1600 -> 6400           960 1030 1404  1050
// The constants come from 38 such launches.  How much longer than the best of the five kinds
// the chosen one takes has not been measured since the 128 x 256 tiles came.
enum Kind { k256, k128, k64, kMixed, kTall };

struct Spread {   // rows of an expert: three equally spaced points and their weights
  double rows[3];
  explicit Spread(const GemmArgs& g) {
    const double r = (double)g.n_rows / g.n_expert, dev = std::max(sqrt(r), 0.03 * r);
    rows[0] = std::max(0.0, r - dev);
    rows[1] = r;
    rows[2] = r + dev;
  }
  template <typename F> double mean(F f) const {
    return 0.25 * f(rows[0]) + 0.5 * f(rows[1]) + 0.25 * f(rows[2]);
  }
};

// Work of one product over the experts' rows (forward or dX): CU microseconds over all
// tiles and the longest tile.  N columns, K values per sum.
struct Work { double total, longest, tiles; };
Work row_product(Kind kind, const GemmArgs& g, double N, double K, bool narrow_quarter) {
  const Spread sp(g);
  const double slices = ceil(K / 64);
  if (kind == k256) {
    const double cols = ceil(N / 128) / 2, tile = 8 + slices * 1.56;
    double full = 0, half = 0, quarter = 0;
    full = sp.mean([&](double r) { const double q = floor(r / 256); return q + (r - 256 * q > 128); });
    half = sp.mean([&](double r) { const double m = r - 256 * floor(r / 256); return m > 64 && m <= 128; });
    quarter = sp.mean([&](double r) { const double m = r - 256 * floor(r / 256); return m > 0 && m <= 64; });
    full *= g.n_expert * cols;
    half *= g.n_expert * cols;
    quarter *= g.n_expert * cols;
    Work w{full * tile + (half * 0.6 + quarter * 0.45) * tile, full > 0 ? tile : 0.6 * tile,
           full + half + quarter};
    if (K >= 2048 && half + quarter <= 128) {   // narrow remainder tiles
      const double f = narrow_quarter ? 4 : 2, narrow = 4 + slices * (narrow_quarter ? 0.31 : 0.4);
      w.total = full * tile + (half * 1.5 + quarter) * f * narrow;
      w.longest = full > 0 ? tile : narrow;
      w.tiles = full + (half + quarter) * f;
    }
    return w;
  }
  if (kind == kTall) {
    const double tiles = g.n_expert * sp.mean([&](double r) { return ceil(r / 128); }) * ceil(N / 256);
    return Work{tiles * (slices * 1.1 + 2.0), slices * 1.4, tiles};
  }
  const double side = kind == k128 ? 128 : 64;
  const double tiles = g.n_expert * sp.mean([&](double r) { return ceil(r / side); }) * ceil(N / side);
  return kind == k128 ? Work{tiles * (slices * 0.65 + 0.8), slices * 0.8, tiles}
                      : Work{tiles * (slices * 0.256 + 1.0), slices * 0.31, tiles};
}

// HBM time of one pass over the weights and `passes` over the rows of both sides; weights
// are read again for every further row tile of an expert as far as caches do not hold them
double memory_us(const GemmArgs& g, double weight_passes, double row_passes, double side) {
  const double tiles = ceil((double)g.n_rows / g.n_expert / side);
  const double again = std::min(2.0, 1 + 0.5 * std::max(0.0, tiles - 1));
  return 2.0 * ((double)g.n_expert * g.in_feat * g.out_feat * (weight_passes - 1 + again) +
                row_passes * g.n_rows * ((double)g.in_feat + g.out_feat)) / 5.3e6 + 3;
}

double launch_us(const Work& w, double tail) {
  return w.tiles <= 256 ? w.longest : std::max(w.longest, w.total / 256 + tail * w.longest);
}

double fwd_us(Kind kind, const GemmArgs& g) {
  const Work w = row_product(kind, g, g.out_feat, g.in_feat, true);
  const double side = kind == k256 ? 256 : kind == k128 ? 128 : 64;
  const double tiles = kind == k256 ? launch_us(w, 0.6) : 4 + launch_us(w, 0.15);
  return std::max(tiles, memory_us(g, 1, 1, side));
}

double bwd_us(Kind kind, const GemmArgs& gd, const GemmArgs& gw) {
  const double r = (double)gw.n_rows / gw.n_expert, E = gw.n_expert;
  Work w{0, 0, 0};
  if (gd.c) w = row_product(kind == kMixed ? k64 : kind, gd, gd.in_feat, gd.out_feat, false);
  if (gw.c) {
    const double side = kind == k256 ? 256 : kind == k64 ? 64 : 128;
    const double n = E * ceil(gw.out_feat / side) * ceil(gw.in_feat / (kind == kTall ? 256 : side));
    const double tile = kind == k256 ? 8.7 + ceil(r / 32) * 0.7
                        : kind == k128 ? 2.2 + ceil(r / 64) * 0.42
                        : kind == kTall ? 2.0 + ceil(r / 64) * 0.75
                        : kind == kMixed ? 1.45 + ceil(r / 32) * 0.23 : 0.9 + ceil(r / 64) * 0.15;
    w.total += n * tile;
    w.longest = std::max(w.longest, tile * (kind == k256 ? 1 : 2));
    w.tiles += n;
  }
  const double side = kind == k256 ? 256 : kind == k128 || kind == kTall ? 128 : 64;
  const double tiles = kind == k256 ? launch_us(w, 0.5) : 4 + launch_us(w, 0.3);
  return std::max(tiles, memory_us(gw, (gd.c ? 1 : 0) + (gw.c ? 1 : 0), 1.5, side));
}

Kind bwd_choice(const GemmArgs& gd, const GemmArgs& gw) {
  Kind best = k128;
  for (Kind kind : {kMixed, k64, kTall})
    if (bwd_us(kind, gd, gw) < bwd_us(best, gd, gw)) best = kind;
  return best;
}

// Forward product of few rows per expert (decode steps, many experts): the weights' way from
// HBM bounds it, and a tile higher than the experts spends copies, LDS reads and matrix
// instructions on rows that are not there.  32 x 64 tiles in three stages, four workgroups to
// a CU, while experts hold 32 rows (what random routing spreads around the average included);
// 64 x 128 in three stages in place of 128 x 128 while they hold 64.  Measured, us, routing
// near uniform (256-row kernels, 128 x 128, 64 x 64 and these):
//    16 experts,   64 rows, 1024 -> 4096     25   24   25     22.4
//     8,  128, 4096 -> 14336                183  170  167    162
//     8,  128, 14336 -> 4096                167  218  159    160
//    64,  512, 2048 -> 4096                 252  254  247    227
//   128,  256, 1408 -> 2048                 141  129  122    117
//   128, 2048, 1024 -> 2048                 115  108  115    100
//    64, 2560, 1024 -> 2048                  53   49   52     47.6
//    64, 2560, 2048 -> 1024                  47   44   47     43.6
// At 100 rows per expert the 64 x 128 tiles are behind (32, 3200, 2048 -> 4096: 145 against 152).
//
// With at most one 32 x 64 tile for each of the 256 CUs, three stages are too few bytes under way
// to HBM: six there.  (Weights from HBM each time, us, three stages and six: 16 experts, 64 rows,
// 4096 -> 1024 33.0 and 31.1; 8, 100, 2048 -> 1408 16.4 and 13.8; 32, 200, 3072 -> 512 23.6 and
// 21.1; with more tiles 24, 200, 2048 -> 768 21.4 and 25.0; 16, 256, 4096 -> 2048 62.6 and 77.6.)
//
// The host knows the average only.  Experts far above it are cut on the device
// (plain_fwd_few_kernel), into 64 x 64 and 128 x 128 tiles.  Skewed loads, weights from HBM each
// time, us: the choice before there were tiles for few rows, those tiles for all experts, as
// it is.  (Popularity p_e ~ e^-1.2; all rows on two experts; on one.)
//    64 experts, 1024 rows, 4096 -> 14336    1302 1353 1289    130 261 193    93 240 170
//   128, 3400, 2048 -> 1408                   164  166  168     45  51  43    44  50  42
//    64,  512, 2048 -> 4096                   225  165  175     45  31  22    43  23  19
//   128, 2048, 1024 -> 2048                   111  108  111     27  30  26    27  25  20
//     8,  128, 4096 -> 14336                  205  166  166     53  64  53    27  39  34
//     8,  128, 14336 -> 4096                  187  203  202     68  72  72    67  60  60
//    32, 1280, 4096 -> 4096                   284  239  228     80  75  63    77  72  62
//   128, 6000, 1408 -> 2048                   187  178  174     37  54  46    37  52  45
// Left behind: experts of 33 to 64 rows in two 32-row tiles where K is long (the sixth), and
// wide products with all rows on one or two of many experts, which the 256-row kernels run
// faster still; these take a seventh to a third of what the call takes under a uniform load.
enum Low { kLow32, kLow64, kNotLow };
Low low_rows(const GemmArgs& g) {
  const double most = Spread(g).rows[2];
  return most <= 32 ? kLow32 : most <= 64 ? kLow64 : kNotLow;
}

template <typename T, int DMA>
int fwd_typed(const GemmArgs& g, hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    return fwd_shape(g, kShapesF32, 4) == 0 ? launch_fwd<T, Tile<64, 128, 2, 128>, DMA>(g, s)
                                            : launch_fwd<T, Tile<64, 64, 2, 128>, DMA>(g, s);
  } else if constexpr (DMA == 16) {
    const Low low = g.tile == 7 ? kLow32 : g.tile == 8 ? kLow64 : g.tile ? kNotLow : low_rows(g);
    using Big = Tile<128, 128, 2, 128>;
    if (low == kLow32)
      return (int64_t)g.n_expert * ceil_div(g.out_feat, 64) <= kCus
                 ? launch_fwd<T, Tile<32, 64, 6, 128>, DMA>(g, s)
                 : launch_fwd_few<T, Tile<32, 64, 3, 128>, Tile<64, 64, 2, 128>, DMA>(g, s);
    const bool big = g.tile ? g.tile != 3 && g.tile != 5 : fwd_us(k128, g) <= fwd_us(k64, g);
    if (low == kLow64 && big) return launch_fwd_few<T, Tile<64, 128, 3, 128>, Big, DMA>(g, s);
    return big ? launch_fwd<T, Big, DMA>(g, s) : launch_fwd<T, Tile<64, 64, 4, 128>, DMA>(g, s);
  } else {
    return fwd_shape(g, kShapes16, 2) == 0 ? launch_fwd<T, Tile<128, 128, 2, 128>, DMA>(g, s)
                                           : launch_fwd<T, Tile<64, 64, 2, 128>, DMA>(g, s);
  }
}

template <typename T, int DMA>
int bwd_typed(const GemmArgs& gd, const GemmArgs& gw, hipStream_t s) {
  if constexpr (std::is_same<T, float>::value) {
    using Wide = Tile<64, 128, 2, 128>;
    using Small = Tile<64, 64, 2, 128>;
    return bwd_shape(gd, gw, kShapesF32, 4) == 0 ? launch_bwd<T, Wide, Wide, DMA>(gd, gw, s)
                                                 : launch_bwd<T, Small, Small, DMA>(gd, gw, s);
  } else if constexpr (DMA == 16) {
    const int forced = gd.tile ? gd.tile : gw.tile;
    const Kind kind = !forced ? bwd_choice(gd, gw)
                      : forced == 3 ? kMixed : forced == 5 ? k64 : forced == 6 ? kTall : k128;
    using Big = Tile<128, 128, 2, 128>;
    if (kind == k128) return launch_bwd<T, Big, Big, DMA>(gd, gw, s);
    // Experts of some hundred rows: dW tiles that are half output.  Twice the columns of the
    // 128 x 128 tile in three stages of half slices load a quarter less per product, and the
    // two workgroups of a CU store and multiply at the same time, which the one of the
    // 256-row kernels cannot.
    using Tall = Tile<128, 256, 3, 64>;
    if (kind == kTall) return launch_bwd<T, Tall, Tall, DMA>(gd, gw, s);
    // short dW sums: half as deep slices, so that four workgroups fit a CU and their output
    // stores (which bound such products) overlap
    if (kind == kMixed)
      return launch_bwd<T, Tile<64, 64, 2, 128>, Tile<128, 128, 2, 64>, DMA>(gd, gw, s);
    return launch_bwd<T, Tile<64, 64, 3, 128>, Tile<64, 64, 3, 128>, DMA>(gd, gw, s);
  } else {
    using Big = Tile<128, 128, 2, 128>;
    using Small = Tile<64, 64, 2, 128>;
    return bwd_shape(gd, gw, kShapes16, 2) == 0 ? launch_bwd<T, Big, Big, DMA>(gd, gw, s)
                                                : launch_bwd<T, Small, Small, DMA>(gd, gw, s);
  }
}

// bytes per lane of the copies: 16 where every row of every operand starts on a 16-byte
// boundary, 4 where it starts on a 4-byte one, 0 = not this kernel's
int copy_width(const GemmArgs& g, int dtype) {
  const int es = (int)dtype_size(dtype);
  const uintptr_t bases = (uintptr_t)g.a | (uintptr_t)g.b | (uintptr_t)g.c |
                          (uintptr_t)g.act_pre | (uintptr_t)g.act_out;
  const int64_t rows = ((int64_t)g.in_feat | g.out_feat) * es;
  if (rows % 16 == 0 && bases % 16 == 0) return 16;
  return rows % 4 == 0 && bases % 4 == 0 ? 4 : 0;
}

// Forced configurations (tests) that are this file's: 128 x 128 tiles; 64 x 64 with 128 x 128
// ones for dW; 64 x 64 for all; 128 x 128 forward with 128 x 256 backward; the forward tiles of
// few rows, 32 x 64 and 64 x 128, with 128 x 128 backward
bool forced_plain(int tile) { return tile == 2 || tile == 3 || tile >= 5; }

}  // namespace

bool gemm_plain_supported(const GemmArgs& g, int dtype) {
  if (dtype != FMOE_F32 && dtype != FMOE_BF16 && dtype != FMOE_F16) return false;
  // tile-relative byte offsets are 32-bit: 128 rows of f32 are the bytes of 256 of bf16
  if (!dma_ld_supported(g.in_feat) || !dma_ld_supported(g.out_feat)) return false;
  return copy_width(g, dtype) != 0;
}

bool gemm_plain_fwd_preferred(const GemmArgs& g, int dtype, double lead) {
  if (dtype == FMOE_F32 || !gemm_plain_supported(g, dtype)) return dtype == FMOE_F32;
  if (g.tile) return forced_plain(g.tile);
  const double plain = std::min(fwd_us(k128, g), fwd_us(k64, g)), wide = fwd_us(k256, g) + lead;
  // few rows: where the estimates meet at the time HBM needs, the lower tiles come closer to it
  // (copies of 4 bytes have none)
  if (copy_width(g, dtype) == 16) {
    const Low low = low_rows(g);
    if (low != kNotLow) return low == kLow32 || plain <= wide;
  }
  return plain < wide;
}

bool gemm_plain_bwd_preferred(const GemmArgs& gd, const GemmArgs& gw, int dtype, double lead) {
  if (dtype == FMOE_F32 || !gemm_plain_supported(gd, dtype) || !gemm_plain_supported(gw, dtype))
    return dtype == FMOE_F32;
  if (gd.tile) return forced_plain(gd.tile);
  return bwd_us(bwd_choice(gd, gw), gd, gw) < bwd_us(k256, gd, gw) + lead;
}

int launch_gemm_plain_fwd(const GemmArgs& g, int dtype, hipStream_t s) {
  if (!gemm_plain_supported(g, dtype))
    return set_error(FMOE_ERR_UNSUPPORTED, "grouped GEMM: rows not on 4-byte boundaries");
  switch (dtype) {
    case FMOE_F32:
      return copy_width(g, dtype) == 16 ? fwd_typed<float, 16>(g, s) : fwd_typed<float, 4>(g, s);
    case FMOE_F16:
      return copy_width(g, dtype) == 16 ? fwd_typed<__half, 16>(g, s) : fwd_typed<__half, 4>(g, s);
    default:
      return copy_width(g, dtype) == 16 ? fwd_typed<__hip_bfloat16, 16>(g, s)
                                        : fwd_typed<__hip_bfloat16, 4>(g, s);
  }
}

int launch_gemm_plain_bwd(const GemmArgs& gd, const GemmArgs& gw, int dtype, hipStream_t s) {
  if (!gemm_plain_supported(gd, dtype) || !gemm_plain_supported(gw, dtype))
    return set_error(FMOE_ERR_UNSUPPORTED, "grouped GEMM: rows not on 4-byte boundaries");
  switch (dtype) {
    case FMOE_F32:
      return copy_width(gd, dtype) == 16 && copy_width(gw, dtype) == 16
                 ? bwd_typed<float, 16>(gd, gw, s)
                 : bwd_typed<float, 4>(gd, gw, s);
    case FMOE_F16:
      return copy_width(gd, dtype) == 16 && copy_width(gw, dtype) == 16
                 ? bwd_typed<__half, 16>(gd, gw, s)
                 : bwd_typed<__half, 4>(gd, gw, s);
    default:
      return copy_width(gd, dtype) == 16 && copy_width(gw, dtype) == 16
                 ? bwd_typed<__hip_bfloat16, 16>(gd, gw, s)
                 : bwd_typed<__hip_bfloat16, 4>(gd, gw, s);
  }
}

}  // namespace fmoe
