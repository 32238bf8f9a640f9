// Host rules that choose how a convolution is run: the tile and K split of the implicit-GEMM
// kernels (conv_igemm.hip), the box, chunk and grid of the patch kernel (conv_direct.hip).  Plain
// C++ on OgleConvArgs, so that the rules can be compiled and checked without a GPU.
#ifndef OGLE_CSRC_CONV_PLAN_H_
#define OGLE_CSRC_CONV_PLAN_H_

#include <algorithm>
#include <cstddef>
#include <cstdint>

#include "ogle_hip.h"

namespace ogle {

// Tile configurations (BM, BN, waves along M, waves along N).
enum TileCfg {
  CFG_128x128 = 0, CFG_64x64 = 1, CFG_128x32 = 2, CFG_WAVE32 = 3, CFG_WAVE16 = 4,
  CFG_128x96 = 5, CFG_128x160 = 6,  // all output channels of a narrow, long-K problem in one tile
  CFG_128x256 = 7,                   // fp16 storage: 64x128 per wave, 64-byte K slabs
  CFG_128x16 = 8                     // at most 16 output channels: 16x16 MFMA blocks
};
constexpr int kCfgBM[] = {128, 64, 128, 32, 16, 128, 128, 128, 128};
constexpr int kCfgBN[] = {128, 64, 32, 32, 16, 96, 160, 256, 16};
constexpr int kRowBytesF16Wide = 64;  // K bytes per tile row per slab of CFG_128x256

// Workgroups that contract fp32 as bf16 pieces: rows x columns, four waves one above the other
// unless named otherwise.  All but the K2 forms add an output's products in the same order.
enum PiecesForm {
  FORM_NONE = 0, FORM_64x64, FORM_128x32, FORM_128x128, FORM_128x64,
  FORM_128x64_W8,       // eight waves of 16 rows
  FORM_64x64_K2,        // two groups of four waves take K stages in turn
  FORM_64x32_K2,
  FORM_32x32_K2,        // two groups of two waves: the K2 forms in a grouped launch
  FORM_128x16,
  FORM_64x32, FORM_64x16   // in a grouped launch for the two of 128 rows, which need more registers
};
constexpr int kFormBM[] = {0, 64, 128, 128, 128, 128, 64, 64, 32, 128, 64, 64};
constexpr int kFormBN[] = {0, 64, 32, 128, 64, 64, 64, 32, 32, 16, 32, 16};

struct IgemmPlan {
  int cfg;
  int splits;
  bool rows_on_xcd;  // split-K work layout: tile rows, not K ranges, pinned to an XCD
  int slabs_per_split;
  int ktiles;
  int cchunks;
  size_t workspace_bytes;  // splits * M * N floats when splits > 1
  int form;                // the workgroup that contracts fp32 as bf16 pieces in place of cfg's (PiecesForm)
};

constexpr long kComputeUnits = 256;
constexpr int kRowBytesF32 = 64;   // bytes of K per tile row per slab, fp32
constexpr int kPiecesSlabs = 3;    // least slabs of a contraction as bf16 pieces
constexpr int kMaxSplits = 64;     // most K ranges

inline bool is_pointwise(const OgleConvArgs& a) {
  return a.kernel_size == 1 && a.stride == 1 && a.padding == 0;
}

inline bool is_wave(int cfg) { return cfg == CFG_WAVE32 || cfg == CFG_WAVE16; }
inline int tile_bm(int cfg) { return kCfgBM[cfg]; }
inline int tile_bn(int cfg) { return kCfgBN[cfg]; }

// Whether whole tile rows spread evenly (within a tenth) over the eight XCDs.
constexpr bool rows_even(long tiles_m) { return ((tiles_m + 7) / 8) * 8 * 10 <= tiles_m * 11; }

// The same for the workgroups that contract bf16 pieces, `per_row` to a tile row, of which a unit runs two at
// a time: the fullest XCD must not need another round of its 32 units for them, nor be the only one to double up.
// 100 rows of 5 leave one XCD 65 workgroups and a nearly empty second round (us by rows / in equal shares, 128x64
// of eight waves: M = 12760, K = 288 -> 320 25.0 / 18.9; 128x128: 1x1 M = 10506, 392 -> 768 61.1 / 41.3).
constexpr bool pieces_rows_even(long tiles_m, long per_row) {
  const long most = (tiles_m + 7) / 8 * per_row, least = (tiles_m * per_row + 7) / 8, slots = 64;
  return rows_even(tiles_m) && (most > slots / 2) == (least > slots / 2) &&
         (most > 8 * slots || (most + slots - 1) / slots == (least + slots - 1) / slots);
}

// 128x64 workgroups on the XCD that gets most of them.
constexpr long most_on_xcd(long m, long out_c) {
  const long rows = (m + 127) / 128, per_row = (out_c + 63) / 64;
  return pieces_rows_even(rows, per_row) ? (rows + 7) / 8 * per_row : (rows * per_row + 7) / 8;
}

// The form for `m` output rows: `large` a plan of 128x128 tiles, `pieces` whether 64x64 tiles would be
// pieces.  What counts is how evenly the workgroups spread over 256 units, and that a unit has waves
// enough to cover what each waits for.  Us of the form taken / of another one, 3x3 unless 1x1:
//   64x32 K2, at most 256 of them: M = 6272, K = 576 -> 64 11.4 / 15.8 with 64x64 (13.4 as fp32), 1x1 M = 400,
//     768 -> 200 11.6 / 18.0 (14.5); where the last 64 columns are mostly padding: M = 8664, K = 432 -> 88 13.4 / 16.0
//   64x64 K2: M = 3136, K = 1152 -> 256 21.9 / 26.1 with 64x64 (30.0), 1x1 M = 1444, 512 -> 512 11.1 / 14.1 (15.0),
//     M = 22500, 1024 -> 40 30.4 / 36.3; K = 288 with at most 256 tiles 11.0 / 10.7 (11.2): the 64x64 ones
//   128x128, pointwise: where they give a unit no more to do than 128x64 ones, in pairs (two run at a time) unless
//     long or many: 1x1 M = 92416, 512 -> 512 183.6 / 209.9, M = 360000, 128 -> 128 111.6 / 120.0, M = 6400, 1024 ->
//     1024 79.7 / 89.8, but M = 12544, 512 -> 768 71.7 / 62.2, M = 23104, 256 -> 512 46.3 / 44.1 (three a unit), M =
//     73600, 40 -> 512 58.0 / 51.6, 96 channels of 128 M = 177480, 260 -> 96 86.8 / 81.3
//   128x64, eight waves, against 64x64, mean ratio over 2000 shapes by number of workgroups: 257 to 383 1.06,
//     384 to 512 0.93, 513 to 640 1.03, more 0.95; those many pointwise ones of up to 7 slabs 1.03 (3 slabs 1.06)
//   128x64, four waves, against eight, pointwise from 8 slabs on, where a unit has more than two and a half: 641 to 1024
//     1.05 over 90 shapes, 1025 to 1536 1.00, to 2560 0.99, more 0.95.  Three fit a unit at once; where no XCD has more,
//     as 11552 x 256 -> 512, they are taken too: 28.1 / 28.0 alone (inputs half zeros 26.0 / 26.7), 21.5 / 22.4 behind its
//     depthwise convolution, in the mean of 17 shapes alone 1.01
inline int pieces_form(const OgleConvArgs& a, long m, int ktiles, bool large, bool pieces) {
  auto tiles = [&](int form) {
    return ((m + kFormBM[form] - 1) / kFormBM[form]) * ((a.out_c + kFormBN[form] - 1) / kFormBN[form]);
  };
  const bool pw = is_pointwise(a);
  const long n64 = tiles(FORM_64x64), n128 = tiles(FORM_128x64_W8);
  if (large) {
    auto per_unit = [&](int form) { return (tiles(form) + kComputeUnits - 1) / kComputeUnits; };
    const long n = per_unit(FORM_128x128);
    if (pw && ktiles >= 8 && (a.out_c + 127) / 128 * 128 * 10 <= a.out_c * 11 &&
        2 * n <= per_unit(FORM_128x64_W8) && (ktiles >= 32 || n >= 8 || n % 2 == 0))
      return FORM_128x128;
  } else if (ktiles >= 12) {
    const long n32 = tiles(FORM_64x32_K2);
    if (n32 <= kComputeUnits || (2 * n32 <= 3 * n64 && n32 <= 2 * kComputeUnits)) return FORM_64x32_K2;
    if (n64 <= kComputeUnits) return ktiles >= 24 ? FORM_64x64_K2 : ktiles >= 16 ? FORM_64x64 : FORM_NONE;
    if (n128 <= kComputeUnits) return pw && ktiles >= 64 ? FORM_64x64_K2 : FORM_128x64_W8;
  }
  if (!large && !pieces) return FORM_NONE;
  if (2 * n128 <= 5 * kComputeUnits)
    return 2 * n128 >= 3 * kComputeUnits && n128 <= 2 * kComputeUnits ? FORM_128x64_W8 : FORM_64x64;
  if (!pw) return FORM_128x64_W8;
  if (ktiles < 8) return FORM_64x64;
  return n128 > 4 * kComputeUnits || most_on_xcd(m, a.out_c) <= 3 * kComputeUnits / 8 ? FORM_128x64 : FORM_128x64_W8;
}

// Picks the output tile and the K split.  Problems with few output
// tiles but a long contraction (the SSD heads, the small feature maps) are split
// along K until the grid fills the chip, provided a workspace was supplied.
inline IgemmPlan plan_igemm(const OgleConvArgs& a, long m, bool allow_split) {
  IgemmPlan p{};
  const int esz = a.dtype == OGLE_F16 ? 2 : 4;
  const int rowb = a.dtype == OGLE_F16 ? 128 : kRowBytesF32;
  const int epr = rowb / esz;
  p.cchunks = (a.in_c + epr - 1) / epr;
  p.ktiles = a.kernel_size * a.kernel_size * p.cchunks;
  auto tiles = [&](int cfg) {
    return ((m + kCfgBM[cfg] - 1) / kCfgBM[cfg]) * ((a.out_c + kCfgBN[cfg] - 1) / kCfgBN[cfg]);
  };
  // fp32 as bf16 pieces: a 128x128 tile splits and reads its operands from LDS half as often per
  // product, a 64x64 tile quantises better over 256 units.  Measured on MI355X, us with 64x64 /
  // 128x128 tiles: M = 11552, K = 512, N = 1024 (728 large tiles) 87 / 74, 6400 x 1024 x 1024
  // (400) 103 / 85, 11552 x 256 x 512 (364) 26.6 / 26.4, 5776 x 512 x 512 (184) 26.5 / 28.2;
  // with K = 128 even 704 large tiles are behind (28.8 / 30.3), 2813 are not (K = 64: 76 / 72).
  // fp16 storage: an MFMA does sixteen times the work per operand byte, so the
  // 64x64 tile is bound by LDS traffic and instruction issue; 128x128 pays off as soon
  // as its tiles cover the compute units.
  const long k_all = (long)a.kernel_size * a.kernel_size * a.in_c;
  const long big_tiles_wanted = a.dtype == OGLE_F16 ? kComputeUnits
                                : k_all >= 256      ? 3 * kComputeUnits / 2
                                                    : 8 * kComputeUnits;
  // A last tile column that is mostly padding costs more than that, in fp16 while K is short
  // (12 x 57 x 57, 88 -> 168: 128x128 tiles 16.3 us, 64x64 11.2; 256 -> 168 19.0 / 14.1; 8 x 40 x 40,
  // 88 -> 300 17.2 / 8.8; K = 792 17.2 / 17.4).
  const bool big_columns_full = (a.dtype == OGLE_F16 && k_all > 512) ||
                                ((a.out_c + 127) / 128) * 128 * 10 <= ((a.out_c + 63) / 64) * 64 * 11;
  // A contraction of 128 slabs or more is cut along K below 2048 tiles (further down), which takes
  // scratch memory.  Large tiles neither bring that on nor avoid it where the scratch a caller
  // has to bring would differ: from 1024 of them on they are cut as well, with fewer they are taken
  // only where the small tiles would not be cut.
  const bool long_f32 = a.dtype == OGLE_F32 && p.ktiles >= 128;
  // (fp32 128x128 tiles exist as pieces only: not for two slabs, see there)
  const bool big_tiles = long_f32 ? tiles(CFG_128x128) >= 4 * kComputeUnits ||
                                        (big_columns_full && tiles(CFG_128x128) >= big_tiles_wanted &&
                                         tiles(CFG_64x64) >= 8 * kComputeUnits)
                                  : big_columns_full && tiles(CFG_128x128) >= big_tiles_wanted &&
                                        (a.dtype == OGLE_F16 || p.ktiles >= kPiecesSlabs);
  // Narrow outputs with a long contraction (the SSD heads, box and class head of a feature
  // map fused: 75 or 150 channels, K = 2304 ... 9216): one tile column holds every output
  // channel, so the input is gathered once instead of once per 64-channel tile column, and
  // 96 / 160 columns waste far less of the MFMA work than two or three 64-wide tiles.
  const bool narrow_long = a.dtype == OGLE_F32 && p.ktiles >= 32 &&
                           ((a.out_c > 64 && a.out_c <= 96) || (a.out_c > 128 && a.out_c <= 160));
  if (narrow_long) {
    p.cfg = a.out_c <= 96 ? CFG_128x96 : CFG_128x160;
  } else if (a.dtype == OGLE_F16 && a.out_c >= 256 && tiles(CFG_128x256) >= 2 * kComputeUnits) {
    // fp16 storage: one MFMA does sixteen times the work per operand byte, and a wave that
    // owns 64x64 outputs reads its operands from LDS as fast as the MFMA pipe consumes them.
    // A wave with 64x128 outputs reads a third less per MFMA and the tile pulls a quarter
    // less from L2; 64-byte slabs keep two such workgroups per compute unit.  Measured on
    // MI355X: M = 46208, K = N = 1024 gains 8 % (610 -> 662 TFLOP/s), but with fewer than two
    // tiles per compute unit (M = 11552, N = 1024: 364 tiles) the second round is mostly
    // empty and the 128x128 tile stays ahead (480 against 448 TFLOP/s).
    p.cfg = CFG_128x256;
    const int epr2 = kRowBytesF16Wide / esz;
    p.cchunks = (a.in_c + epr2 - 1) / epr2;
    p.ktiles = a.kernel_size * a.kernel_size * p.cchunks;
  } else if (a.out_c <= 16) {
    p.cfg = CFG_128x16;
  } else if (a.out_c <= 32) {
    p.cfg = CFG_128x32;
  } else if (a.out_c > 64 && big_tiles) {
    p.cfg = CFG_128x128;
  } else {
    p.cfg = CFG_64x64;
  }
  p.splits = 1;
  const long t = tiles(p.cfg);
  long sp = 1;
  bool exact_split = false;  // sp was chosen by the search below: any count is fine
  if (allow_split && narrow_long && t < 2 * kComputeUnits) {
    // One tile column, few tile rows, a long K: the K split decides how evenly the chip is
    // filled.  Workgroups are (tile, K range) pairs dealt to 256 compute units, each doing
    // ceil(ktiles / s) slabs plus a fixed cost (first loads, epilogue: about `fixed` slabs);
    // take the s with the shortest estimated time, partial-sum traffic as the tie break.
    const double fixed = p.cfg == CFG_128x96 ? 6.0 : 4.0;
    double best = 1e30;
    for (long s = 1; s <= kMaxSplits && p.ktiles / s >= 8; ++s) {
      const long rounds = (t * s + kComputeUnits - 1) / kComputeUnits;
      const double cost = (double)rounds * ((double)((p.ktiles + s - 1) / s) + fixed) + 0.25 * (double)s;
      if (cost < best - 1e-9) {
        best = cost;
        sp = s;
      }
    }
    exact_split = true;
  } else if (allow_split && 2 * t <= kComputeUnits && p.ktiles >= 8) {
    // too few tiles to occupy every compute unit: about three workgroups per unit,
    // at least four slabs per split
    const long want = (3 * kComputeUnits + t - 1) / t;
    const long most = p.ktiles / 4;
    sp = want < most ? want : most;
  } else if (allow_split && t < 8 * kComputeUnits && p.ktiles >= 128 &&
             !(long_f32 && p.cfg == CFG_128x128 && t < 4 * kComputeUnits)) {
    // a few long workgroups per unit quantise badly (one unit gets two, its
    // neighbour one) and leave one wave per SIMD: cut the long contraction so that
    // about eight shorter workgroups land on every unit, 32 slabs or more each
    const long want = (8 * kComputeUnits + t - 1) / t;
    const long most = p.ktiles / 32;
    sp = want < most ? want : most;
  }
  if (sp > kMaxSplits) sp = kMaxSplits;
  // the kernel's XCD-aware work layout wants a divisor or a multiple of 8
  if (exact_split) {}
  else if (sp >= 8) sp -= sp % 8;
  else if (sp >= 4) sp = 4;
  else if (sp >= 2) sp = 2;
  if (sp >= 2) p.splits = (int)sp;
  // A small contraction that would be split across workgroups goes to the wave-split
  // kernel instead (the split stays inside the workgroup: no workspace, no second
  // launch), whether or not a workspace was offered.  Measured on MI355X against
  // split-K + reduce: the 32x32 form wins once its tiles cover half the chip, for
  // K <= 1024 pointwise and K <= 512 otherwise; the 16x16 form wins for pointwise
  // K <= 1024 while its tiles stay under two per compute unit, and for K <= 1536 while they
  // stay under one per unit (3x3x256 <- 5x5x128 at batch 16: 7.0 against 9.5 us); a longer K
  // per wave is a serial chain of MFMAs and loses to the split across workgroups.
  {
    const long k_total = (long)a.kernel_size * a.kernel_size * a.in_c;
    const bool pw = is_pointwise(a);
    const bool would_split = (2 * t <= kComputeUnits && p.ktiles >= 8) ||
                             (t < 8 * kComputeUnits && p.ktiles >= 128);
    const long t32 = tiles(CFG_WAVE32), t16 = tiles(CFG_WAVE16);
    const bool small16 = (pw && k_total <= 1024 && t16 <= 2 * kComputeUnits) ||
                         (k_total <= 1536 && t16 <= kComputeUnits);
    // other than pointwise: K <= 512, or up to 2304 while every 32x32 tile has a compute unit
    // to itself (5x5x512 <- 10x10x256, 3x3 stride 2, at batch 16: 19.8 against 21.6 us)
    const long k32cap = t32 <= kComputeUnits ? 2304 : 512;
    if (narrow_long) {
      // stays on the wide tile
    } else if (would_split && !small16 && k_total <= (pw ? 1024 : k32cap) && t32 >= kComputeUnits / 2 &&
        t32 <= 4 * kComputeUnits) {
      p.cfg = CFG_WAVE32;
      p.splits = 1;
    } else if (would_split && small16) {
      p.cfg = CFG_WAVE16;
      p.splits = 1;
    }
  }
  p.slabs_per_split = (p.ktiles + p.splits - 1) / p.splits;
  if (p.splits > 1) {
    p.slabs_per_split += p.slabs_per_split & 1;  // the K loop runs slab pairs
    p.splits = (p.ktiles + p.slabs_per_split - 1) / p.slabs_per_split;  // no empty ranges
  }
  // (a split past the end of K would only add zeros; rounding splits down keeps the
  // divisor-or-multiple-of-8 shape, so empty splits are simply avoided by the cap above)
  // partial sums are kept in rows of the channel count rounded up to four
  p.workspace_bytes =
      p.splits > 1 ? (size_t)p.splits * (size_t)m * ((a.out_c + 3) & ~3) * sizeof(float) : 0;
  // fp32 tiles of 32x32 MFMA blocks are contracted as bf16 pieces (the 96 and 160 columns wide ones
  // are not built as such) where a compute unit has more than one workgroup and more than 16 slabs:
  // a lone workgroup has little to cover the splitting with, and a short sum is over before the faster
  // unit has made up for it.  Not for two slabs at all, nor for pointwise convolutions to at most 32
  // channels: both are bound by their bytes.  Time with pieces in the form of pieces_form over time with fp32 MFMAs,
  // plans of 64x64 tiles, means of 950 shapes:
  //   slabs  workgroups to 384   512   768  1024  1536  2560  5000
  //     2         1.06        0.96  0.91  1.09  1.11  1.13
  //     3         0.91  0.94  0.92  0.97  0.95  0.95  0.93
  //     4         0.98  0.99  0.90  0.96  0.96  0.94  0.93
  //     6         0.94  0.92  0.85  0.89  0.90  0.90  0.87
  //     9         0.91  0.88  0.85  0.87  0.85  0.84  0.83
  //    16         0.77  0.80  0.76  0.80  0.77  0.75  0.75
  //    36         0.73  0.77  0.76  0.77  0.74  0.73  0.70
  //    72         0.71  0.75  0.70  0.77  0.69
  // The line was drawn for kernels 5 to 15 % behind these; below it the full products stay although pieces would be up
  // to a tenth faster by now.  128x32 tiles 0.83 to 0.98 from 9 slabs on with 3x3, 0.97 to 1.04 pointwise.
  const long workgroups = tiles(p.cfg) * p.splits;
  const bool pieces = a.dtype == OGLE_F32 && (p.cfg == CFG_128x128 || p.cfg == CFG_64x64 || p.cfg == CFG_128x32) &&
             workgroups > kComputeUnits && p.slabs_per_split >= kPiecesSlabs &&
             workgroups * p.slabs_per_split > 16 * kComputeUnits &&
             !(p.cfg == CFG_128x32 && is_pointwise(a));
  if (a.dtype == OGLE_F32 && p.cfg == CFG_128x16 && p.splits == 1 && p.ktiles >= 12 && t <= kComputeUnits) {
    // (75x75x64 -> 16 3x3 at batch 4 18.4 / 14.7, 19x19x512 -> 16 at batch 64 14.0 / 13.3; not with K ranges,
    // which wait for the input, 19x19x512 -> 12 3x3 53 / 59, nor with more tiles, which do as well,
    // 38x38x1024 -> 16 at batch 24 43.6 / 51.3)
    p.form = FORM_128x16;
  } else if (a.dtype != OGLE_F32 || p.splits > 1) {
    p.form = !pieces ? FORM_NONE
             : p.cfg == CFG_64x64 ? FORM_64x64
             : p.cfg == CFG_128x32 ? FORM_128x32
             : is_pointwise(a) ? FORM_128x128 : FORM_128x64_W8;
  } else if (p.cfg == CFG_64x64 || p.cfg == CFG_128x128) {
    p.form = pieces_form(a, m, p.ktiles, p.cfg == CFG_128x128, pieces);
  } else if (p.cfg == CFG_128x32) {
    p.form = pieces ? FORM_128x32 : FORM_NONE;
  } else if (p.cfg == CFG_WAVE32 && is_pointwise(a) && p.ktiles >= 12) {
    // two K groups against the wave-split kernel, where that one's 32x32 tiles need a second round of the units
    // and 64x32 tiles do not: 1x1 M = 1600, 1024 -> 256 14.9 / 16.4, M = 1444, 256 -> 256 6.1 / 6.8, M = 392, 208 ->
    // 768 5.8 / 6.4, M = 961, 312 -> 96 6.4 / 9.6, but M = 1624, 256 -> 154, 255 tiles of 32x32, 6.7 / 5.3
    const long n32 = ((m + 63) / 64) * ((a.out_c + 31) / 32);
    if (n32 <= kComputeUnits && tiles(CFG_WAVE32) > kComputeUnits) p.form = FORM_64x32_K2;
  }
  // Which operand an XCD's L2 should keep to itself: with K ranges pinned to XCDs the input is
  // fetched by all eight L2s and the filter by one, with tile rows pinned it is the other way
  // round (the rocprofv3 FETCH_SIZE of the 19x19x512 class head fell from 8.5x its input to
  // about the input plus eight filters).
  {
    const long x_bytes = (long)a.n * a.in_h * a.in_w * a.in_c * esz;
    const long w_bytes = (long)a.out_c * a.kernel_size * a.kernel_size * a.in_c * esz;
    p.rows_on_xcd = p.splits > 1 && !is_wave(p.cfg) && x_bytes > w_bytes;
  }
  return p;
}

inline bool igemm_eligible(const OgleConvArgs& a, long* m_out) {
  if (a.group != 1) return false;
  const int ve = a.dtype == OGLE_F16 ? 8 : 4;
  if (a.in_c % ve != 0) return false;
  if ((long)a.kernel_size * a.kernel_size * a.in_c < 32) return false;
  const long m = (long)a.n * a.out_h * a.out_w;
  if (m <= 0 || m > 0x7fffffffL) return false;
  // operands are addressed with 32-bit byte offsets through buffer loads
  const long esz = a.dtype == OGLE_F16 ? 2 : 4;
  const long lim = 0x7fffffffL;
  if ((long)a.n * a.in_h * a.in_w * a.in_c * esz > lim) return false;
  if ((long)a.out_c * a.kernel_size * a.kernel_size * a.in_c * esz > lim) return false;
  *m_out = m;
  return true;
}

// Ungrouped fp32 convolutions whose channels fill no vector, contracted as bf16 pieces out of the runs of
// values that their filter rows are (pieces_tile).
inline bool plan_runs(const OgleConvArgs& a, IgemmPlan* out) {
  const int k = a.kernel_size;
  if (a.dtype != OGLE_F32 || a.group != 1 || (a.dilation != 1 && k > 1)) return false;
  const long m = (long)a.n * a.out_h * a.out_w, run = (long)k * a.in_c, lim = 0x7fffffffL;
  if (m <= 0 || m > lim || run > lim / 64) return false;
  if ((long)a.n * a.in_h * a.in_w * a.in_c * 4 > lim || (long)a.out_c * k * run * 4 > lim) return false;
  // a pixel's first value, in the padding or not, is counted in 32 bits too
  if (((long)a.in_w + 2L * a.padding + k) * a.in_c > lim / 4 || (long)a.padding * a.in_w * a.in_c * 4 > lim / 4) return false;
  IgemmPlan p{};
  p.cfg = CFG_64x64;
  p.splits = 1;
  p.cchunks = (int)((run + 15) / 16);
  p.ktiles = p.slabs_per_split = k * p.cchunks;
  // Against the direct kernels: a fit of 700 shapes (1x1, 3x3, 5x5, 5 to 181 channels); a chain of products
  // takes them 0.08 us each, many products their rate.  Narrow outputs leave little of the work that gathering a
  // pixel's values is worth.  Us with the direct kernels / like this, 3x3 unless noted: 4 x 56 x 56, 99 -> 99
  // 95 / 45; 16 x 40 x 40, 1x1 131 -> 77 45 / 18; 16 x 224 x 224, 7x7 stride 2 3 -> 64 99 / 58; 4 x 4 x 4, 21 ->
  // 16 16.5 / 9.5, but 22 x 49 x 47, 149 -> 5 71 / 103, 8 x 7 x 7, 1x1 39 -> 37 5.5 / 7.1.  (The faster each time
  // would be 0.711 of the direct kernels' time in the mean, the rule 0.753.)
  const double products = (double)m * a.out_c * k * run;
  const double chain = (double)a.in_c * std::min(k, a.in_h) * std::min(k, a.in_w);
  if (k * run < 24 || 0.07 * chain + 0.2e-6 * products <= 3 + 0.15 * p.ktiles) return false;
  if (a.out_c <= 32 && k > 1 && (a.out_c <= 16 || products < 3e7)) return false;
  // (two K groups where a unit has one workgroup or none: 3 x 3 x 2, 11 -> 256 3x3 stride 2 7.0 / 9.0 as 64x64, 1 x
  // 86 x 119, 1x1 34 -> 32 5.1 / 7.0 as 128x32, 2 x 64 x 64, 9x9 1 -> 64 7.5 / 9.5, 14 x 4 x 5, 1x1 139 -> 9 7.0 /
  // 8.3 as 128x16)
  if (((m + 63) / 64) * ((a.out_c + 31) / 32) <= kComputeUnits) p.form = FORM_64x32_K2;
  else if (a.out_c <= 32) p.form = a.out_c <= 16 ? FORM_128x16 : FORM_128x32;
  else p.form = pieces_form(a, m, p.ktiles, false, true);
  if (p.form == FORM_NONE || p.form == FORM_128x64) p.form = FORM_64x64;
  // with many tiles the filter, gathered value by value, counts: half as often per pixel, pointwise too (4 x 100 x
  // 140, 98 -> 127 28.2 / 27.0; the 7x7 stem 55.3 / 51.4)
  if (p.form == FORM_64x64 && m * a.out_c > 64L * 64 * 5 * kComputeUnits) p.form = FORM_128x64_W8;
  *out = p;
  return true;
}

// Byte offset of a pixel's first tap, which may lie in the padding: modulo 2^32, so that a tap inside the image comes
// out exact whatever the padding and however near to 2 GiB the tensor.
constexpr unsigned first_tap_offset(int h, int w, int pixel, int image, int iy, int ix) {
  return (((unsigned)image * (unsigned)h + (unsigned)iy) * (unsigned)w + (unsigned)ix) * (unsigned)pixel * 4u;
}

// How far behind a pixel's first tap another lies, modulo 2^32 as well: a first tap high up in the padding is farther
// from the image's last rows than a signed offset reaches.
constexpr unsigned tap_offset(int w, int pixel, int dy, int dx) {
  return ((unsigned)dy * (unsigned)w + (unsigned)dx) * (unsigned)pixel * 4u;
}

// Whether a 16-byte load with a value of a pixel's runs begins before the tensor or ends behind it: such a load
// returns zeros for all four.  `iy`: the row of the first filter row, `start`: the runs' first value, counted from
// their rows' first; both may lie in the padding.  (The first row counts wherever it lies: a row of one or two
// values that is not the tensor's first can still share its first vector with what is before the tensor.)
constexpr bool runs_leave_tensor(int images, int h, int row_values, int k, int run, int image, int iy, int start) {
  const long first = (long)image * h + (iy < 0 ? 0 : iy);
  const long last = (long)image * h + (iy + k - 1 < h - 1 ? iy + k - 1 : h - 1);
  return first * row_values + start < 0 ||
         last * row_values + start + ((run + 3) & ~3) > (long)images * h * row_values;
}

// The plan the launch will use: split-K only with a workspace that is large enough.
inline IgemmPlan final_plan(const OgleConvArgs& a, long m) {
  IgemmPlan p = plan_igemm(a, m, a.workspace_dev != nullptr);
  if (p.workspace_bytes > a.workspace_bytes) p = plan_igemm(a, m, false);
  return p;
}

// ---------------------------------------------------------------------------
// Patch kernel (conv_direct.hip).
struct FastDiv {   // n / d for n, d < 2^16: with mul = ceil(2^32 / d) the error n * (mul * d - 2^32) stays below 2^32
  unsigned mul;
  int d;
};
constexpr FastDiv fast_div(int d) {
  return FastDiv{0xffffffffu / (unsigned)d + 1u, d};   // ceil(2^32 / d); d == 1 is not looked up
}

struct PatchPlan {
  int th_log, tw_log;             // box of output pixels of a workgroup (128 >> both images)
  int tiles_b, tiles_y, tiles_x;  // boxes along images, rows, columns
  int ph, pw, pitch;              // patch rows, columns, floats per patch pixel
  int in_step, box_step;          // input pixels per patch pixel, patch pixels per output pixel
  int cc;                         // input channels per group staged at once
  int gp, gblocks;                // groups per workgroup; ceil(groups / gp)
  int cols, col_blocks;           // output channels per workgroup and group
  int runs_x;                     // K runs per filter row: one per tap, or one in all
  int tile_blocks;                // workgroups along the boxes (each walks several when channels fit at once)
  int vec_x, vec_w;               // patch / filter read four values at a time
  int patch_floats, lds_floats;
  FastDiv d_cs, d_pw, d_ph, d_runk, d_col;
};

constexpr int kPatchPixels = 128;
constexpr int kPatchStaticLds = 16;   // bytes of LDS the kernel has beside the plan's lds_floats

// The patch kernel's box, chunk and grid for a convolution; false if it does not take it.
inline bool plan_patch(const OgleConvArgs& a, PatchPlan* out) {
  const int cpg = a.in_c / a.group, opg = a.out_c / a.group, k = a.kernel_size;
  const long lim = 0x7fffffffL;
  if ((long)a.n * a.in_h * a.in_w * a.in_c > lim || (long)a.n * a.out_h * a.out_w * a.out_c > lim) return false;
  if ((long)a.n + kPatchPixels > lim || (long)a.in_h + a.padding > lim / 2 || (long)a.in_w + a.padding > lim / 2)
    return false;
  // Under 64 products per pixel and group most of an MFMA block is padding and one thread per
  // output is faster.  Measured at 4 x 48 x 48, us with one thread per output / with this kernel,
  // groups x (channels in -> out): 64 x (2 -> 2) 3x3 25 / 44, 32 x (4 -> 8) 1x1 15.3 / 17.9;
  // from 64 on 32 x (8 -> 8) 1x1 38 / 19, 16 x (4 -> 4) 3x3 27 / 17, 32 x (32 -> 32) 3x3 9905 / 122
  if ((long)k * k * cpg * opg < 64) return false;
  // A few thousand short sums are over before the patch is staged (one image 14 x 14, 32 x
  // (8 -> 8) 1x1: 6.3 / 7.6; 9 x 9, 35 -> 75 1x1: 6.3 / 12.1; 4 x 28 x 28, 181 -> 9 1x1, whose
  // patch is staged in three chunks: 20.8 / 31; but 3x3 with K = 72: 11.6 / 8.6, K = 891: 104 / 50).
  if ((long)a.n * a.out_h * a.out_w * a.out_c <= 65536 && k * k * cpg <= (k == 1 ? 192 : 48)) return false;
  const long span = (long)(k - 1) * a.dilation + 1;
  if (span > 1024 || a.stride > 64) return false;   // no such patch fits LDS
  PatchPlan p{};
  // one tap: the pixels that a stride skips are not staged
  p.in_step = k == 1 ? a.stride : 1;
  p.box_step = k == 1 ? 1 : a.stride;
  p.cols = opg <= 16 ? 16 : (opg <= 32 || (((opg + 31) / 32) % 2 == 1 && opg < 160)) ? 32 : 64;
  // the box: fewest boxes, then the smallest patch
  double best = 0;
  for (int tw = 0; tw <= 7; ++tw) {
    for (int th = 0; tw + th <= 7; ++th) {
      const int box_b = kPatchPixels >> (tw + th);
      if ((1 << tw) >= 2 * a.out_w || (1 << th) >= 2 * a.out_h) continue;
      const long ph = ((1L << th) - 1) * p.box_step + span, pw = ((1L << tw) - 1) * p.box_step + span;
      const double boxes = (double)((a.n + box_b - 1) / box_b) * ((a.out_h + (1 << th) - 1) >> th) *
                           ((a.out_w + (1 << tw) - 1) >> tw);
      const double cost = boxes * ((double)(ph * pw * box_b) + 2.0 * kPatchPixels);
      if (best != 0 && cost >= best) continue;
      best = cost;
      p.tw_log = tw;
      p.th_log = th;
      p.ph = (int)ph;
      p.pw = (int)pw;
    }
  }
  const int box_b = kPatchPixels >> (p.tw_log + p.th_log);
  p.tiles_b = (a.n + box_b - 1) / box_b;
  p.tiles_y = (a.out_h + (1 << p.th_log) - 1) >> p.th_log;
  p.tiles_x = (a.out_w + (1 << p.tw_log) - 1) >> p.tw_log;
  const long tiles = (long)p.tiles_b * p.tiles_y * p.tiles_x;
  // a grid that leaves compute units empty is cut finer along the channels instead: the time of
  // such a launch is one workgroup's staging and serial contraction
  while (p.cols > 16 && tiles * a.group * ((opg + p.cols - 1) / p.cols) < 256) p.cols /= 2;
  p.col_blocks = (opg + p.cols - 1) / p.cols;
  const long pixels = (long)box_b * p.ph * p.pw;
  const long wp = p.cols + 1;
  if (pixels > 0xffff) return false;
  // channels staged at once: all of them, or the most that leave three workgroups per unit
  // (48 KB of LDS each); 64 KB, what a launch may ask for, static part included, where the grid
  // gives a unit no third one anyway (fewer, longer chunks: each costs a round trip to memory) or
  // nothing less will do
  const bool roomy = tiles * a.group * p.col_blocks <= 512;
  auto floats = [&](long cc, long gp) { return pixels * ((cc * gp) | 1) + gp * k * k * cc * wp; };
  const long most = (64L * 1024 - kPatchStaticLds) / 4;
  long cc = 0;
  for (const long budget : {roomy ? most : 12288L, most}) {
    if (floats(cpg, 1) <= budget) cc = cpg;
    else
      for (long t : {64L, 32L, 16L, 8L, 4L, 2L})
        if (cc == 0 && t < cpg && floats(t, 1) <= budget) cc = t;
    if (cc != 0) break;
  }
  if (cc == 0) return false;
  p.cc = (int)cc;
  // several groups per workgroup share a patch's cache lines, as long as the grid still has
  // about two workgroups per compute unit
  p.gp = 1;
  if (cc == cpg && p.col_blocks == 1)
    while (p.gp < a.group && floats(cpg, p.gp + 1) <= 8192 &&
           tiles * ((a.group + p.gp) / (p.gp + 1)) >= 512)
      ++p.gp;
  p.gblocks = (a.group + p.gp - 1) / p.gp;
  const bool merge = a.dilation == 1 && cc == cpg && p.gp == 1 && cpg % 2 == 1 && k > 1;
  p.runs_x = merge ? 1 : k;
  p.pitch = (int)(cc * p.gp) | 1;
  p.patch_floats = (int)(pixels * p.pitch);
  p.lds_floats = (int)floats(cc, p.gp);
  const long per_tile = (long)p.gblocks * p.col_blocks;
  // with all channels staged at once the filter stays in LDS while a workgroup walks boxes
  // (no more workgroups than their LDS lets be resident, each with as many boxes as any other)
  const long resident = 256 * (160L * 1024 / (4 * p.lds_floats + kPatchStaticLds));
  const long turns = cc == cpg ? (tiles * per_tile + resident - 1) / resident : 1;
  p.tile_blocks = (int)((tiles + turns - 1) / turns);
  // (a launch holds fewer than 2^32 threads: a one-channel output of 8 GB in 128-pixel boxes does not fit)
  if (per_tile * p.tile_blocks * 256 > 0xffffffffL || pixels * cc * p.gp > 0xffff ||
      (long)p.gp * p.cols * k * k * cc > 0xffff)
    return false;
  const uintptr_t vec = 4 * (a.dtype == OGLE_F16 ? 2 : 4);
  p.vec_x = a.in_c % 4 == 0 && cpg % 4 == 0 && cc % 4 == 0 && reinterpret_cast<uintptr_t>(a.input_dev) % vec == 0;
  p.vec_w = cc == cpg && (k * k * cpg) % 4 == 0 && reinterpret_cast<uintptr_t>(a.filter_dev) % vec == 0;
  p.d_cs = fast_div((int)(cc * p.gp));
  p.d_pw = fast_div(p.pw);
  p.d_ph = fast_div(p.ph);
  p.d_runk = fast_div((int)(k * k * cc));
  p.d_col = fast_div(std::min(p.cols, opg % p.cols == 0 ? p.cols : opg % p.cols));
  *out = p;
  return true;
}

// Products of an output that follow each other, without taps that can only lie in the padding of a
// small map.
inline double direct_chain(const OgleConvArgs& a) {
  const int k = a.kernel_size;
  return (double)(a.in_c / a.group) * std::min(k, (a.in_h - 1) / a.dilation + 1) *
         std::min(k, (a.in_w - 1) / a.dilation + 1);
}
// Values a workgroup of the patch kernel stages, all chunks of channels.
inline double patch_staged(const OgleConvArgs& a, const PatchPlan& p) {
  const int cpg = a.in_c / a.group;
  return (double)p.lds_floats * ((cpg + p.cc - 1) / p.cc);
}

// Whether a planned patch is worth it.  One thread per output is bound by its chain of products
// while threads are few and by their number when they are many; the patch kernel by staging patch
// and filter.  Both lines are fits of 1523 shapes (1 to 32 groups, 1x1 and 3x3, up to 100,000
// pixels; the faster of the two each time would be 0.7 % faster on average).  Us with one thread per
// output / with the patch kernel, 3x3 except as noted: 1 x 1, 17 -> 33 3.9 / 29.7; 4 x 4, 12 groups
// of 16 -> 16 19.7 / 8.8; 14 x 14, 7 -> 33 8.7 / 9.4, 17 -> 33 18.7 / 13.0, 33 -> 33 35 / 18, with
// stride 2 35 / 35; 56 x 56, 1x1 35 -> 33 7.4 / 11.4, 35 -> 75 12.1 / 11.6, 131 -> 33 23.8 / 26,
// 131 -> 75 43 / 26; 4 x 56 x 56, 1x1, 4 groups of 8 -> 12 11.9 / 8.0.
inline bool patch_pays(const OgleConvArgs& a, const PatchPlan& p) {
  const double staging = p.vec_x ? 1000 + patch_staged(a, p) / 2 : 9000 + patch_staged(a, p);
  const double outputs = (double)a.n * a.out_h * a.out_w * a.out_c;
  return direct_chain(a) >= 0.006 * staging || outputs * direct_chain(a) > (p.vec_x ? 4.5e6 : 6e6);
}

// The kernel with the filter in LDS, one thread per four channels of a pixel, or per sixteen (wide)
// where that still leaves enough threads to fill the chip.
inline bool small_k_fits(const OgleConvArgs& a) {
  return a.group == 1 && a.out_c % 4 == 0 && 4L * a.kernel_size * a.kernel_size * a.in_c * a.out_c <= 48 * 1024;
}
inline bool small_k_is_wide(const OgleConvArgs& a) {
  return a.out_c % 16 == 0 && (long)a.n * a.out_h * a.out_w * (a.out_c / 16) >= 256L * 256 * 4;
}

// The patch kernel against that one: the chain of products against staging again; many products,
// times the channels, since every workgroup stages the whole filter (a wide thread's cost a quarter);
// inputs beyond the L2s, of which a wave reads a cache line per pixel and value.  Fits of 1426
// shapes (the faster each time would be 0.9 % faster on average).  Us with that kernel / with the
// patch kernel, 3x3 except as noted: 1 x 1, 33 -> 16 6.3 / 51; 14 x 14, 7 -> 16 7.5 / 9.3, 17 -> 16
// 13.6 / 12.9, stride 2 14.0 / 16.7, 33 -> 16 24 / 18, stride 2 25 / 35; 56 x 56, 1x1 35 -> 64
// 5.7 / 11.4, 131 -> 64 15.6 / 26; 4 x 56 x 56, 5 -> 128 23 / 15, 1x1 35 -> 256 50 / 23;
// 8 x 112 x 112, 1x1 35 -> 32 17 / 28, 131 -> 16 68 / 44, 7x7 stride 2 3 -> 64 56 / 23.
inline bool patch_beats_small_k(const OgleConvArgs& a, const PatchPlan& p) {
  const double staging = p.vec_x ? 6000 + patch_staged(a, p) / 2 : 10000 + patch_staged(a, p);
  const double products = (double)a.n * a.out_h * a.out_w * a.out_c * a.kernel_size * a.kernel_size * a.in_c;
  const double x_bytes = (double)a.n * a.in_h * a.in_w * a.in_c * (a.dtype == OGLE_F16 ? 2 : 4);
  const bool wide = small_k_is_wide(a);
  return direct_chain(a) >= 0.007 * staging || products * (wide ? 0.25 : 1) * a.out_c > 4e9 ||
         (x_bytes > 24e6 && !wide);
}

// Short sums of a small output, where one thread per output is as good or better (256 channels of
// 14 x 14, K = 28: 7.1 us with the filter in LDS, 5.7 with one thread per output), but for the
// pointwise ones that share many input values (28 x 28, 131 -> 64 15.3 / 16.4, 16 -> 16 3.6 / 4.3).
inline bool general_beats_small_k(const OgleConvArgs& a) {
  const int k = a.kernel_size, ktot = k * k * a.in_c;
  if ((long)a.n * a.out_h * a.out_w * a.out_c > 65536 || ktot > (k == 1 ? 192 : 48)) return false;
  return !(k == 1 && (long)a.n * a.out_h * a.out_w >= 16 &&
           ((ktot > 96 && a.out_c >= 32) || (a.in_c % 4 == 0 && a.out_c >= 16 && a.out_c <= 64)));
}

// The kernel for a convolution that neither the implicit GEMM nor the stem kernels take.
enum DirectKernel { DIRECT_GENERAL, DIRECT_PATCH, DIRECT_SMALL_K };
inline DirectKernel plan_direct(const OgleConvArgs& a, PatchPlan* plan) {
  const bool patch = plan_patch(a, plan);
  if (small_k_fits(a)) {
    if (patch && patch_beats_small_k(a, *plan)) return DIRECT_PATCH;
    return general_beats_small_k(a) ? DIRECT_GENERAL : DIRECT_SMALL_K;
  }
  return patch && patch_pays(a, *plan) ? DIRECT_PATCH : DIRECT_GENERAL;
}

}  // namespace ogle

#endif  // OGLE_CSRC_CONV_PLAN_H_
