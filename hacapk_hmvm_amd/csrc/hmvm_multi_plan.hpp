// hmvm_multi_plan.hpp -- host-side schedule of the products with several
// right-hand sides (no HIP dependency).
//
// The multi-RHS product has a schedule and a copy of the values of its own.
// A tile of the one-vector launches is one wavefront and leaves its rows in
// output slots that a further launch adds up, which with 16 to 64 right-hand
// sides moves more bytes than the matrix itself.  Here a workgroup owns rows
// of an output and its waves split the columns:
//   stage-1 groups  up to kMultiRows rank rows of a column cluster's stack;
//                   over all of its columns where these fit one group, whose
//                   rows then go straight to t, else one group per chunk of
//                   columns, whose rows go to slots that a t sum adds (the
//                   stacks of few columns are one wave each);
//   row groups      up to kMultiRows rows of y: the a2 factors and the dense
//                   leaves of every row cluster that meets these rows; the
//                   group writes y.
// A row group is cut so that no row cluster taller than a group starts or
// ends inside it, so such a cluster covers all of its rows.  The columns that
// all rows of a group have (those of tall clusters, and the dense leaves of
// one column cluster that together cover the group) are one list that the
// waves split evenly: the "kept" items, whose sums stay in registers until
// the waves add theirs through LDS.  Columns that only some of the rows have
// are items of one wave each, which leaves their rows in slots that the same
// workgroup adds to y.  Rows outside an item never meet its columns, so that
// a non-finite entry of X reaches the rows of its leaves alone.
//
// Columns are taken in slices of KS (4, BF16 8): a slice is KS columns of X or
// t whose rows follow each other, zero columns filling the last slice of a
// leaf or cluster; four slices, one per 16 lanes, are one batch of MFMA
// steps.  The values of an item are packed in the order its wave reads them:
// element (r, q) of slice s at
//   a0 + (s*H + q/E)*nrows*E + r*E + q%E,   E = 16 bytes, H = KS/E,
// so a lane's KS columns of its row are one or two 16-byte words, 16 lanes
// read 256 consecutive bytes, and a wave one contiguous stream.  Reading the
// one-vector layout instead (columns of a whole cluster apart) left lines
// partly used, and BF16 spent more time on bringing a row's columns together
// than on the products (N=101,250 cube, 32 right-hand sides: rows of y 413 / 310
// / 131 us for FP64 / FP32 / BF16, packed 370 / 206 / 98; HBM bytes of the packed
// launches 1.33 and 1.48 (FP64), 1.26 and 1.38 (FP32), 1.41 and 1.43 (BF16) times
// the matrix they read).
#pragma once

#include <cstdint>
#include <string>
#include <vector>

#include "hmvm_plan.hpp"

namespace hmvm {

constexpr int kMultiRows = 64;  // most rows of a group
constexpr int kMultiBatch = 4;  // slices per batch
constexpr int kMultiXcds = 8;   // XCDs of an MI355X

// Columns of a slice, and elements of a 16-byte word.
inline int multi_slice_cols(int storage) { return storage == kBF16 ? 8 : 4; }
inline int multi_word(int storage) { return storage == kF64 ? 2 : storage == kF32 ? 4 : 8; }

struct MultiSlice {
  int32_t v;     // row of X or t of the first column
  int32_t info;  // columns in use (0..KS), bit 8: rows of t (else X); BF16 stage 1: see below
};
constexpr int kSliceT = 1 << 8;

// Stage 1 of BF16 storage, whose t is rounded to BF16: a sum that lies next to
// a rounding boundary decides an element of t, so the order of its additions
// is part of the result (with one FP32 sum per wave, the elements of t rounded
// the other way moved elements of y by up to 1.5e-3 of their size).  The order
// is that of a tile of the one-vector launches at its default size: rank rows
// in groups of at most Plan::chunk_rows that end with a leaf, a group's columns
// in chunks (chunk_cols), a chunk one FP32 sum in steps of 16 columns
// (v_mfma_f32_16x16x16_bf16), and the chunks added in FP64, in registers, over
// the waves, and over a stack's groups.  A batch is two steps of 16 columns:
// its slice s takes columns 4s + 0..3 and, as its second half, those + 16; info
// holds the columns in use of each half (bits 0..3, 4..7) and whether the batch
// ends a chunk.
// Rows: 32, as a chunk's FP32 and FP64 sums of 64 rows and 64 right-hand sides
// would spill.  Product at N=50,021 (cube), 16 / 32 / 64 right-hand sides: the
// tile launches 122 / 145 / 371 us, one FP32 sum per wave 78 / 94 / 124, this
// 85 / 106 / 138 (one wave a chunk, all chunks through FP32 slots: 91 / 115 /
// 140, and N=4,096 29 / 40 / 46 instead of 16 / 16 / 21).
constexpr int kSliceEnd = 1 << 9;
constexpr int kOrderedRows = 32;
constexpr int kHalf = 4, kStep = 16;
constexpr int ordered_column(int slice, int q) {
  return slice / kMultiBatch * 2 * kStep + slice % kMultiBatch * kHalf + q % kHalf + q / kHalf * kStep;
}

// nbatch batches of slices from slice0, values from a0, over nrows rows.
// out: first slot (kItemSlot), offset in tmap (kItemT); a kept item's sum is
// added over the waves of its workgroup.
enum MultiItemKind : int { kItemSlot = 0, kItemT = 1, kItemKept = 2 };
struct MultiItem {
  int64_t a0;
  int32_t slice0, nbatch, nrows, out, kind, reserved;
};

// One workgroup, in dispatch order: wave w runs the items of waves[waves per
// group * g + w].  kind: where the rows of its kept items go (each wave's last
// item is then one), or that it has none (the waves are on their own); out:
// first row of y, offset in tmap, or first slot.
enum MultiKind : int { kMultiY = 0, kMultiT = 1, kMultiTSlot = 2, kMultiNone = 3 };
struct MultiGroup {
  int32_t nrows, kind, out, reserved;
};
struct MultiWave {
  int32_t item0, nitems;
};

// Packs rows x cols elements (r, c) = values[src + r + c*ld] as rows row0..
// of an item of nrows rows: columns from the item's slice at dst (the address
// of that slice), with zeros in the unused columns of the last slice and in
// `pad` further slices.
struct MultiPack {
  int64_t src, dst;
  int32_t ld, rows, cols, row0, nrows, pad;
  int32_t factor;  // BF16: the factor's scale goes into the values (-1: none)
  int32_t ordered; // column q of slice s is ordered_column(s, q), else s*KS + q
};

struct MultiOptions {
  int rows = kMultiRows;    // most rows of a row group
  int rows_a = kMultiRows;  // most rank rows of a stage-1 group
  int waves = 4;            // waves per workgroup
  int cols1 = 2048;         // most columns of a stage-1 group
  int wave_cols = 256;      // stage-1 stacks of at most so many columns are one wave's
};

struct MultiPlan {
  int waves = 4;
  int64_t nvals = 0;                       // packed values (elements)
  int64_t n_t = 0, n_slots = 0;            // t rows, slots (t partials, then partial items)
  std::vector<MultiSlice> slices;
  std::vector<MultiPack> pack;
  std::vector<MultiItem> items;
  std::vector<MultiGroup> groups_a, groups_b;  // stage 1; rows of y
  std::vector<MultiWave> waves_a, waves_b;
  std::vector<int32_t> tmap;               // t row of every row of the kMultiT groups
  std::vector<int32_t> t_factor;           // a1 factor of every t row (its a2 factor is the next id)
  struct TSum { int32_t first, nch, stride, entry; };
  std::vector<TSum> tsum;                  // t entry = sum of nch slots first + c*stride
  std::vector<int32_t> yptr;               // 2 per row of y: its slots are list[yptr[2r] .. yptr[2r+1]) + r
  std::vector<int32_t> ylist;
};

constexpr const char *kMultiTooLarge = "the matrix is too large for the multi-RHS schedule";

// P: the plan whose value layout (repack records) is read; nstrtl, nstrtt:
// first row and column of every leaf (1-based).  "" or an error message
// (kMultiTooLarge: offsets exceed int32).
std::string build_multi_plan(const Plan &P, int storage, const int *nstrtl, const int *nstrtt,
                             const MultiOptions &opt, MultiPlan *out);

// Every packed element written once and read by one item, every t row and y row
// written once, every address a kernel forms inside its buffer.
std::string verify_multi_plan(const Plan &P, int storage, const MultiPlan &M);

// For a plan that passed verify_multi_plan, element by element (4 bytes of host
// memory each; hmvm_plan_check does it up to kMultiCheckValues): every element
// of every leaf packed once, against its vector entry, into its row.
constexpr int64_t kMultiCheckValues = int64_t(1) << 28;
std::string verify_multi_values(const Plan &P, int storage, const int *nstrtl, const int *nstrtt, const MultiPlan &M);

// Sizes by matrix order, see the definition.
MultiOptions multi_options(const Plan &P);

// Consecutive groups (of one launch) and pack records whose values, packed
// from element a0 on, fit a buffer of bounded size.
struct MultiWindow {
  int64_t a0;
  int32_t launch, group0, ngroups, pack0, npack;
};

// Cuts the schedule (built with wave_cols = 0: a workgroup's values are then
// consecutive) into windows of at most `cap` elements and puts each launch's
// groups into window order, their dispatch order kept within a window.  "" or
// an error message (a group larger than cap).
std::string window_multi_plan(int storage, int64_t cap, MultiPlan *M, std::vector<MultiWindow> *out);

}  // namespace hmvm
