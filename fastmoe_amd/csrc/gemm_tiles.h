// How the grouped GEMMs cut ragged expert rows into tiles and deal the tiles to
// workgroups: shared by the 16-bit matrix-core kernels (gemm_mfma_impl.h) and the
// plain-pipeline ones (gemm_plain.hip).
#pragma once
#include "gemm.h"

namespace fmoe {

// Tiles one XCD works on between two refills of its 32 CUs.
constexpr int kXcdRun = 32;

// Patch order over a rows x cols grid of tiles: bands of 16 rows, cut into
// blocks of 8 columns, cut into patches of 4 rows that are walked column by
// column.  32 consecutive numbers are a 4x8 patch (12 operand tiles for 32
// products), 256 consecutive ones a 16x16 region.  Ragged edges shrink the
// band, block or patch; the order stays a bijection.
// (The three sizes can be set at build time, for measurements of other walks: on the
// 16384-token, 4096 -> 14336, 8-expert layer a forward launch pulls 2.87 GiB through L2
// with 4 x 8 patches, 2.86 GiB with 8 x 4 and 4.19 GiB with 2 x 16.)
#ifndef FMOE_PATCH_ROWS
#define FMOE_PATCH_ROWS 4
#define FMOE_PATCH_COLS 8
#define FMOE_BAND_ROWS 16
#endif
__device__ __forceinline__ void tile_order(int t, int rows, int cols, int& row, int& col) {
  constexpr int kBand = FMOE_BAND_ROWS, kCols = FMOE_PATCH_COLS, kRows = FMOE_PATCH_ROWS;
  const int band = t / (kBand * cols);
  int r = t % (kBand * cols);
  const int band_rows = min(kBand, rows - band * kBand);
  const int blk = r / (band_rows * kCols);
  r %= band_rows * kCols;
  const int blk_cols = min(kCols, cols - blk * kCols);
  const int patch = r / (kRows * blk_cols);
  r %= kRows * blk_cols;
  const int patch_rows = min(kRows, band_rows - patch * kRows);
  row = band * kBand + patch * kRows + r % patch_rows;
  col = blk * kCols + r / patch_rows;
}

// Where a tile sits in the rows of its expert.
struct TileRows {
  int e;        // expert
  int m0;       // first row of the tile inside the expert
  int row0;     // first row of the expert
  int cnt;      // rows of the expert
};

// Remainder tiles (see the kernels below): 64 rows (the 4 waves side by side,
// K slices of 32 in 6 LDS stages: a slice is a quarter of the MFMA work of a
// 256-row one, so its copies need more slices of lead to cover the memory
// latency) or 128 rows (2 x 2 waves, 4 stages).
constexpr int kSmallRows = 64;
constexpr int kSmallBK = 32;
constexpr int kSmallStages = 6;

// How expert rows are cut into tiles.
// kOneHeight: tiles of BM rows.
// kRemainder: `full` tiles of BM rows from row 0 on
// and, for a remainder of at most BM / 2 rows, one remainder tile (`small` is
// 0 or 1) of 64 rows, or of 128 rows when the remainder is longer than 64;
// a remainder above BM / 2 rows takes one more BM tile.  Remainder tiles cost
// about 0.45 (64 rows) and 0.6 (128 rows) of a 256-row tile.
// kTwoHeights: an expert of up to `low_most` rows in `small` tiles of LOW rows, a longer one
// in tiles of BM rows.
enum Cut { kOneHeight, kRemainder, kTwoHeights };
template <int BM, Cut CUT, int LOW>
__device__ __forceinline__ void cut_rows(int cnt, int low_most, int& full, int& small) {
  full = (cnt + BM - 1) / BM;
  small = 0;
  if (CUT == kOneHeight) return;
  if (CUT == kTwoHeights) {
    if (cnt <= low_most) {
      full = 0;
      small = (cnt + LOW - 1) / LOW;
    }
    return;
  }
  full = cnt / BM;
  const int rem = cnt - full * BM;
  small = rem > 0 && rem <= BM / 2;
  if (rem > BM / 2) ++full;
}

// Position of a workgroup in the order in which tiles are handed out.
// The hardware gives consecutive workgroup ids to the 8 XCDs in turn, and each
// XCD has its own L2.  The live tiles are numbered 0..live-1 so that
// neighbours share operands (tile_order()); XCD x takes the runs
// [256 j + 32 x, +32) of that numbering (shorter runs when there are fewer than
// 256 tiles), one run per round of its 32 CUs, so the blocks that share an L2
// work on a 4x8 patch and the whole chip on a 16x16 one.  Blocks past the live
// range sit at the end of the launch order and exit at once (idle blocks
// interleaved with live ones were measured to delay live blocks of the same
// XCD by a whole tile time).
__device__ __forceinline__ int tile_number(int pid, int live) {
  const int run = max(1, min(kXcdRun, (live + 7) >> 3));  // fewer than 256 tiles: spread them
  const int slot = pid >> 3;                      // position in this XCD's queue
  return (slot / run) * (8 * run) + (pid & 7) * run + slot % run;
}

// Inclusive prefix sum over the 64 lanes of a wave with data-parallel-primitive
// moves (no trips through the LDS crossbar: every workgroup runs this before its
// first copy): shifts by 1, 2, 4, 8 inside each row of 16 lanes, then lane 15 of
// rows 0 and 2 added to rows 1 and 3, then lane 31 added to rows 2 and 3.  A lane
// without a source, or outside the row mask, adds the 0 passed as the old value.
__device__ __forceinline__ int wave_inclusive_sum(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31
  return x;
}

// Row tiles of a ragged product.  The BM-row tiles of all experts are numbered
// first, one expert after the other, the remainder (or lower) tiles behind them.
//
// Up to 64 experts: lane x of EVERY wave cuts the rows of expert x and a wave
// scan turns the counts into first-tile numbers, so no LDS and no barrier are
// involved and the owner of a tile is read from its lane.  More experts: each
// thread cuts the rows of a contiguous run of experts, the scan runs over the
// whole block through LDS, and the thread whose run contains a given row tile
// walks the run to find its owner.
template <int BM, Cut CUT, int NW, int LOW = BM>
struct RowTiles {
  bool by_lane;            // the up-to-64-experts scheme
  int x_lo, x_hi;          // this thread's run of experts
  int mine_f, mine_s;      // BM-row / small tiles in the run
  int first_f, first_s;    // number of the run's first tile of either kind
  int rows_f, rows_s;      // totals over all experts
  int my_row0, my_cnt;     // by_lane: the expert of this lane
  int low_most = BM;       // kTwoHeights: rows of the longest expert in small tiles

  // May contain a __syncthreads(); s_wave_sum has 2 * NW entries.
  __device__ __forceinline__ void scan(const int32_t* seg_off, int n_expert, int* s_wave_sum) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    by_lane = n_expert <= 64;
    mine_f = mine_s = 0;
    if (by_lane) {
      x_lo = lane;
      x_hi = lane < n_expert ? lane + 1 : lane;
      my_row0 = my_cnt = 0;
      if (lane < n_expert) {
        my_row0 = seg_off[lane];
        my_cnt = seg_off[lane + 1] - my_row0;
        cut_rows<BM, CUT, LOW>(my_cnt, low_most, mine_f, mine_s);
      }
    } else {
      const int per_thread = (n_expert + NW * 64 - 1) / (NW * 64);
      x_lo = min(tid * per_thread, n_expert);
      x_hi = min(x_lo + per_thread, n_expert);
      for (int x = x_lo; x < x_hi; ++x) {
        int f, sm;
        cut_rows<BM, CUT, LOW>(seg_off[x + 1] - seg_off[x], low_most, f, sm);
        mine_f += f;
        mine_s += sm;
      }
    }
    // inclusive scans inside the wave
    const int incl_f = wave_inclusive_sum(mine_f);
    const int incl_s = CUT != kOneHeight ? wave_inclusive_sum(mine_s) : 0;
    first_f = incl_f - mine_f;
    first_s = incl_s - mine_s;
    if (by_lane) {
      rows_f = __builtin_amdgcn_readlane(incl_f, 63);
      rows_s = __builtin_amdgcn_readlane(incl_s, 63);
      return;
    }
    if (lane == 63) {
      s_wave_sum[wave] = incl_f;
      s_wave_sum[NW + wave] = incl_s;
    }
    __syncthreads();
    rows_f = rows_s = 0;
#pragma unroll
    for (int w2 = 0; w2 < NW; ++w2) {
      const int wf = s_wave_sum[w2], ws = s_wave_sum[NW + w2];
      if (w2 < wave) {
        first_f += wf;
        first_s += ws;
      }
      rows_f += wf;
      rows_s += ws;
    }
  }

  // First row of an expert's tile `i` of its kind, behind `full` BM-row ones.
  static __device__ __forceinline__ int first_row(int i, int full, bool small) {
    if (CUT == kTwoHeights) return i * (small ? LOW : BM);
    return (small ? full : i) * BM;
  }

  // Owner of row tile v (of the small kind if `small`), v below the total
  // of its kind.  s_out has 4 entries; may contain a __syncthreads().
  __device__ __forceinline__ TileRows find(const int32_t* seg_off, int v, bool small,
                                           int* s_out) const {
    const int first = small ? first_s : first_f, mine = small ? mine_s : mine_f;
    const bool own = v >= first && v < first + mine;
    TileRows t;
    if (by_lane) {
      const int owner = __ffsll((unsigned long long)__ballot(own)) - 1;  // exactly one lane
      const int at = __builtin_amdgcn_readlane(first, owner);
      const int f = __builtin_amdgcn_readlane(mine_f, owner);
      t.e = owner;
      t.m0 = first_row(v - at, f, small);
      t.row0 = __builtin_amdgcn_readlane(my_row0, owner);
      t.cnt = __builtin_amdgcn_readlane(my_cnt, owner);
      return t;
    }
    if (own) {
      int at = first;
      for (int x = x_lo; x < x_hi; ++x) {
        const int r0 = seg_off[x], c = seg_off[x + 1] - r0;
        int f, sm;
        cut_rows<BM, CUT, LOW>(c, low_most, f, sm);
        const int tx = small ? sm : f;
        if (v < at + tx) {
          s_out[0] = x;
          s_out[1] = first_row(v - at, f, small);
          s_out[2] = r0;
          s_out[3] = c;
          break;
        }
        at += tx;
      }
    }
    __syncthreads();
    t.e = s_out[0];
    t.m0 = s_out[1];
    t.row0 = s_out[2];
    t.cnt = s_out[3];
    return t;
  }
};

}  // namespace fmoe
