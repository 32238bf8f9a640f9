// Dense convolution (group 1) as an implicit GEMM on the MFMA units.
//
//   Y[m, o] = act( bias[o] + sum_{tap, c} X[row(m) + tap, c] * W[o, tap, c] )
//
// with m = (image, oy, ox) flattened, K = taps * C.  Both operands are
// K-contiguous in memory: X is NHWC (a pixel's channels are contiguous) and W is
// packed OHWI (an output channel's taps*channels are contiguous), so both tiles
// are fetched as 16-byte vectors along K and the pointwise 1x1 convolution is the
// special case with one tap and no gather (conv2d_pw.glsl:35-91); the KxK form
// follows conv2d.glsl:29-92 (taps outside the image contribute zero).
//
// Tiling.  A workgroup of 4 waves (256 threads) owns a BM x BN output tile and
// walks K in slabs of ROWB bytes per row.  Slabs are staged global -> registers
// -> LDS (double buffered, one barrier per slab) with the next slab's global
// loads in flight while the current one is multiplied.  The 16-byte K groups of an
// LDS row are permuted by a function of the row, so that staging writes and operand
// reads are bank-conflict free.
//
// MFMA mapping (64-wide waves).  Most fp32 problems are contracted as bf16 pieces by kernels of
// their own (pieces_tile below).  The others use v_mfma_f32_32x32x2_f32: lane l
// supplies A[l%32][l/32] and B[l/32][l%32].  Since the contraction sums over k
// in any order, a lane reads four consecutive k of its row with one 16-byte LDS
// read (lanes 0-31 take k 0..3 of an 8-wide group, lanes 32-63 take k 4..7) and
// issues four MFMAs, one per element.  fp16 storage uses
// v_mfma_f32_32x32x16_f16: a lane's 16 bytes are the 8 halves the instruction
// wants (k = 8*(l/32)..+7).  Accumulation is fp32 in all cases.
//
// Result layout of a 32x32 block: register r of lane l holds
// row 8*(r/4) + 4*(l/32) + r%4, column l%32, so a store instruction writes two
// 128-byte runs of one output pixel's channels.
//
// A tile that is 16 columns wide (at most 16 output channels) is built from 16x16
// blocks instead: v_mfma_f32_16x16x4_f32 (lane l supplies A[l%16][l/16], four lane
// groups take k 0..3, 4..7, 8..11, 12..15 of a 16-wide group and issue four MFMAs)
// or v_mfma_f32_16x16x32_f16; register r of lane l is row 4*(l/16) + r, column l%16.
#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "common.h"
#include "conv_plan.h"

namespace ogle {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));

struct ConvGeom {
  int n, h, w, c;
  int oh, ow, o;
  int k, stride, pad, dil;
  int m_total;   // n*oh*ow
  int cchunks;   // K slabs per tap
  int ktiles;    // taps * cchunks
  unsigned x_bytes;  // size of the input tensor (buffer-load range)
  unsigned w_bytes;  // size of the packed filter
  long oimg;         // elements between the outputs of consecutive images; 0: dense
  int pixel;         // runs (pieces_tile): channels of a pixel, c being a run's values; else c
};

// Element offset of output row `row` (= (image, oy, ox) flattened) whose channels are
// `pitch` apart per row: dense, or with a gap after every image's oh * ow rows.
__device__ __forceinline__ long out_row_offset(const ConvGeom& g, int row, int pitch) {
  if (g.oimg == 0) return (long)row * pitch;
  const int hw = g.oh * g.ow;
  const int b = row / hw;
  return (long)b * g.oimg + (long)(row - b * hw) * pitch;
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Offset that is out of range for every operand (operands are kept below 2 GiB), so
// a buffer load at it returns zeros: this is how padding taps, rows past the end of
// the problem and the K tail are zero filled without a branch.
constexpr unsigned kOutOfRange = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

typedef float floatx4v __attribute__((ext_vector_type(4)));

// MFMA step on a TS x TS block of outputs (the wave-split kernel's tile; the LDS-tiled
// kernel's block when its tile is 16 columns wide).  `a` / `b` are the 16 bytes
// the lane loaded; lanes are grouped by q = lane / TS.
//   TS 32: q in {0,1};   fp32 4 x 32x32x2 (k = 4q + s), fp16 1 x 32x32x16 (k = 8q..)
//   TS 16: q in {0..3};  fp32 4 x 16x16x4 (k = 4q + s), fp16 1 x 16x16x32 (k = 8q..)
template <typename T, int TS>
struct WaveMma;
template <>
struct WaveMma<float, 32> {
  typedef floatx16 Acc;
  static constexpr int REGS = 16;
  __device__ static __forceinline__ void run(const u32x4& a, const u32x4& b, Acc& acc) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(a[s]), __uint_as_float(b[s]), acc, 0, 0, 0);
  }
};
template <>
struct WaveMma<__half, 32> {
  typedef floatx16 Acc;
  static constexpr int REGS = 16;
  __device__ static __forceinline__ void run(const u32x4& a, const u32x4& b, Acc& acc) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, a),
                                                 __builtin_bit_cast(halfx8, b), acc, 0, 0, 0);
  }
};
template <>
struct WaveMma<float, 16> {
  typedef floatx4v Acc;
  static constexpr int REGS = 4;
  __device__ static __forceinline__ void run(const u32x4& a, const u32x4& b, Acc& acc) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[s]), __uint_as_float(b[s]), acc, 0, 0, 0);
  }
};
template <>
struct WaveMma<__half, 16> {
  typedef floatx4v Acc;
  static constexpr int REGS = 4;
  __device__ static __forceinline__ void run(const u32x4& a, const u32x4& b, Acc& acc) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a),
                                                 __builtin_bit_cast(halfx8, b), acc, 0, 0, 0);
  }
};

// Work assignment.  Workgroups are dealt to the 8 XCDs by linear id modulo 8 and
// every XCD has a private L2, so the (tile, split) pairs are laid out such that
// tiles sharing a band of A rows run on one XCD and, when K is split, an XCD owns
// a fixed subset of the K ranges: the filter and input slabs of one K range are
// then fetched into one L2 only instead of all eight.
// When K is split and the input is the larger operand (a 3x3 head on a big map), the
// other layout is used instead (splits < 0 marks it): tile rows are dealt to the XCDs and
// all K ranges of a tile row run on the same XCD, so each band of input rows (with the
// halo its taps share) is fetched into one L2 only, and the filter into all eight.
// `splits` says which layout (work_layout below).  Returns false for a workgroup beyond the last tile.
__device__ __forceinline__ bool assign_work(int bid, int tiles_n, int tiles, int splits, int& pid, int& split) {
  const int xcd = bid & 7, j = bid >> 3;
  if (splits < 0) {
    if (splits >= -kMaxSplits) {
      splits = -splits;
      const int per_row = tiles_n * splits;
      const int r = (j / per_row) * 8 + xcd;
      const int rem = j % per_row;
      pid = r * tiles_n + rem / splits;
      split = rem % splits;
    } else {
      splits = -splits - kMaxSplits;
      const int per = (tiles * splits + 7) >> 3;
      const int q = j < per ? xcd * per + j : tiles * splits;
      pid = q / splits;
      split = q - pid * splits;
    }
    if (pid >= tiles) return false;
  } else {
    if (splits == 1) {
      // tile row r (the tiles_n tiles that share one band of A rows) goes to XCD
      // r % 8, so all XCDs advance through memory together
      const int r = (j / tiles_n) * 8 + xcd;
      pid = r * tiles_n + j % tiles_n;
      split = 0;
    } else if (splits == 0) {
      const int per = (tiles + 7) >> 3;
      pid = j < per ? xcd * per + j : tiles;
      split = 0;
    } else if (splits >= 8 && (splits & 7) == 0) {
      const int zs = splits >> 3;
      pid = j / zs;
      split = xcd + 8 * (j - pid * zs);
    } else if (splits == 2 || splits == 4) {
      const int xpz = 8 / splits;
      split = xcd % splits;
      pid = j * xpz + xcd / splits;
    } else {                       // any other count: the splits of a tile are neighbours
      pid = bid / splits;
      split = bid - pid * splits;
    }
    if (pid >= tiles) return false;
  }
  return true;
}

// One workgroup's share of one convolution: output tile / K range number `bid` of
// the problem.  Shared by the single-problem kernel and the grouped kernel.
// LDS bytes of one workgroup: two K-slab buffers of BM + BN padded rows.
template <int BM, int BN, int ROWB>
constexpr int igemm_lds_bytes() {
  return 2 * (BM + BN) * (ROWB + 16);
}

template <typename T, int BM, int BN, int WM, int WN, int ROWB, bool PW>
__device__ __forceinline__ void igemm_tile(
    unsigned char* __restrict__ lds, const ConvGeom& g, const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ bias, T* __restrict__ y, T* __restrict__ y2, int o1,
    const Epilogue& ep, int tiles_n, int tiles, float* __restrict__ partial,
    int slabs_per_split, int splits, int bid) {
  static_assert(WM * WN == 4, "four waves per workgroup");
  constexpr int WTM = BM / WM, WTN = BN / WN;
  // MFMA block: 32x32 outputs, or 16x16 (v_mfma_f32_16x16x4_f32 / 16x16x32_f16) for a tile
  // that is only 16 columns wide (a convolution with at most 16 output channels: in a
  // 32-wide block more than half of the MFMA work would be padding)
  constexpr int MB = WTN % 32 == 0 ? 32 : 16;
  constexpr int TM = WTM / MB, TN = WTN / MB;
  static_assert(TM >= 1 && TN >= 1 && WTM % MB == 0 && WTN % MB == 0, "wave tile in whole MFMA blocks");
  typedef typename WaveMma<T, MB>::Acc Acc;
  constexpr int REGS = WaveMma<T, MB>::REGS;
  constexpr int VPR = ROWB / 16;       // 16-byte vectors per row per slab
  constexpr int RPP = 256 / VPR;       // rows one pass of the workgroup loads
  constexpr int AP = (BM + RPP - 1) / RPP, BP = (BN + RPP - 1) / RPP;
  constexpr bool A_PART = BM % RPP != 0, B_PART = BN % RPP != 0;  // last pass partly idle
  // LDS rows.  A row is exactly its slab bytes and its 16-byte K groups are permuted by a
  // function of the row: (row >> 1) & 7 for 128-byte rows; for 64-byte rows (row >> 2) & 3
  // under 32x32 MFMA blocks and 2 * ((row >> 2) & 1) under 16x16 blocks.  That keeps both the
  // operand reads and the staging writes free of bank conflicts (a 16-byte LDS access is
  // served 16 lanes per cycle: those with the same lane / 32 and the same parity of
  // (lane >> 2) & 7; they must fall into 16 different 16-byte columns of a 256-byte window;
  // found by exhaustive search over XOR functions of the row bits against that model,
  // confirmed by SQ_LDS_BANK_CONFLICT: 1.58 M -> 0.05 M cycles per launch of a
  // 19x19x512 -> 512 pointwise layer at batch 16; rows padded by 16 bytes, as before, cost the
  // writes three times and the 16x16 reads twice the conflict-free cycles).  Other slab
  // widths: rows padded by 16 bytes.
  constexpr bool SWZ = ROWB == 64 || ROWB == 128;
  constexpr int LROW = SWZ ? ROWB : ROWB + 16;   // LDS row pitch, bytes
  auto row_perm = [](int row) {
    return ROWB == 128 ? (row >> 1) & 7 : MB == 32 ? (row >> 2) & 3 : ((row >> 2) & 1) << 1;
  };
  constexpr int ESZ = (int)sizeof(T);
  constexpr int CHUNKB = (64 / MB) * 16;  // bytes of a row one MFMA step consumes (64 / MB lane groups x 16)
  constexpr int CHUNKS = ROWB / CHUNKB;
  static_assert(CHUNKS >= 1, "a K slab holds at least one MFMA step");
  constexpr int STAGE = igemm_lds_bytes<BM, BN, ROWB>() / 2;  // one buffer: A rows then B rows

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wave_m = wave / WN, wave_n = wave % WN;

  int pid, split;
  if (!assign_work(bid, tiles_n, tiles, splits, pid, split)) return;
  const int tile_n = pid % tiles_n;
  const int tile_m = pid / tiles_n;
  const int m0 = tile_m * BM;
  const int n0 = tile_n * BN;

  const int vcol = tid % VPR;   // which 16-byte vector of the slab row
  const int vrow = tid / VPR;   // row within a pass

  const __amdgpu_buffer_rsrc_t rx = make_rsrc(x, g.x_bytes);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(w, g.w_bytes);

  // Per-pass source rows of this thread, as byte offsets into the operands.
  unsigned a_base[AP];  // PW: row offset; KxK: offset of the image the row lies in
  int a_iy[AP], a_ix[AP];
#pragma unroll
  for (int p = 0; p < AP; ++p) {
    const int m = m0 + p * RPP + vrow;
    const bool ok = m < g.m_total && (!A_PART || p * RPP + vrow < BM);
    if (PW) {
      a_base[p] = ok ? (unsigned)m * (unsigned)(g.c * ESZ) : kOutOfRange;
      a_iy[p] = 0;
      a_ix[p] = 0;
    } else {
      const int ox = m % g.ow;
      const int t = m / g.ow;
      const int oy = t % g.oh;
      const int b = t / g.oh;
      a_base[p] = (unsigned)b * (unsigned)(g.h * g.w * g.c * ESZ);
      // a row that does not exist fails every in-image test below
      a_iy[p] = ok ? oy * g.stride - g.pad : -0x40000000;
      a_ix[p] = ox * g.stride - g.pad;
    }
  }
  const unsigned krow_bytes = (unsigned)(g.k * g.k * g.c * ESZ);
  unsigned b_base[BP];
#pragma unroll
  for (int p = 0; p < BP; ++p) {
    const int o = n0 + p * RPP + vrow;
    const bool ok = o < g.o && (!B_PART || p * RPP + vrow < BN);
    b_base[p] = ok ? (unsigned)o * krow_bytes : kOutOfRange;
  }

  // Two register sets: slab kt+1 is already in flight in one while slab kt+2 is
  // being requested into the other, so a load has two slabs of MFMA work to land.
  u32x4 ra[2][AP], rb[2][BP];

  // Issues the global loads of the next K slab into ra / rb (no waiting) and moves
  // the load cursor on.  The cursor (slab number, its tap, channel chunk and tap
  // offsets) advances by increments: slabs are requested strictly in order, so the
  // two integer divisions that locate a slab are paid once, not per slab.
#define OGLE_LOAD_SLAB(SET)                                                                  \
  {                                                                                          \
    const int cbyte_ = l_cc * ROWB + vcol * 16;                                              \
    const bool c_ok_ = cbyte_ < g.c * ESZ && l_kt < kt_end; /* past the end: zeros */        \
    _Pragma("unroll") for (int p = 0; p < AP; ++p) {                                         \
      unsigned off_;                                                                         \
      if (PW) {                                                                              \
        off_ = c_ok_ ? a_base[p] + (unsigned)cbyte_ : kOutOfRange;                           \
      } else {                                                                               \
        const int iy_ = a_iy[p] + l_dy, ix_ = a_ix[p] + l_dx;                                \
        const bool in_ = c_ok_ && iy_ >= 0 && iy_ < g.h && ix_ >= 0 && ix_ < g.w;            \
        off_ = in_ ? a_base[p] + (unsigned)((iy_ * g.w + ix_) * g.c * ESZ + cbyte_)          \
                   : kOutOfRange;                                                            \
      }                                                                                      \
      ra[SET][p] = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)off_, 0, 0);               \
    }                                                                                        \
    _Pragma("unroll") for (int p = 0; p < BP; ++p) {                                         \
      const unsigned off_ = c_ok_ ? b_base[p] + l_tapbyte + (unsigned)cbyte_ : kOutOfRange;  \
      rb[SET][p] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)off_, 0, 0);               \
    }                                                                                        \
    ++l_kt;                                                                                  \
    if (++l_cc == g.cchunks) {                                                               \
      l_cc = 0;                                                                              \
      l_tapbyte += (unsigned)(g.c * ESZ);                                                    \
      l_dx += g.dil;                                                                         \
      if (++l_kx == g.k) {                                                                   \
        l_kx = 0;                                                                            \
        l_dx = 0;                                                                            \
        l_dy += g.dil;                                                                       \
      }                                                                                      \
    }                                                                                        \
  }

  // Writes ra / rb into LDS buffer `buf`.
#define OGLE_STORE_SLAB(buf, SET)                                                            \
  {                                                                                          \
      unsigned char* base_ = lds + (buf) * STAGE + vrow * LROW +                             \
                             (SWZ ? (vcol ^ row_perm(vrow)) : vcol) * 16;                    \
      _Pragma("unroll") for (int p = 0; p < AP; ++p)                                         \
        if (!A_PART || p * RPP + vrow < BM)                                                  \
          *reinterpret_cast<u32x4*>(base_ + p * RPP * LROW) = ra[SET][p];                    \
      _Pragma("unroll") for (int p = 0; p < BP; ++p)                                         \
        if (!B_PART || p * RPP + vrow < BN)                                                  \
          *reinterpret_cast<u32x4*>(base_ + (BM + p * RPP) * LROW) = rb[SET][p];             \
  }

  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < REGS; ++r) acc[i][j][r] = 0.f;

  const int l32 = lane & 31;
  const int lh = lane >> 5;
  const int lrow = lane % MB;  // operand row of this lane inside an MFMA block
  const int lq = lane / MB;    // its 16-byte group along K

  // Split-K: workgroup z of the grid contracts K slabs [kt_begin, kt_end) only and
  // leaves its partial sums in `partial`; a second kernel adds the splits in order.
  const int kt_begin = split * slabs_per_split;
  const int kt_end = min(g.ktiles, kt_begin + slabs_per_split);

  // One K slab from LDS buffer `buf` into the accumulators.
#define OGLE_COMPUTE_SLAB(buf)                                                               \
  {                                                                                          \
    const unsigned char* pa = lds + (buf) * STAGE + (wave_m * WTM + lrow) * LROW;            \
    const unsigned char* pb = lds + (buf) * STAGE + (BM + wave_n * WTN + lrow) * LROW;       \
    _Pragma("unroll") for (int ch = 0; ch < CHUNKS; ++ch) {                                  \
      /* this lane's 16-byte K group of the step (rows 32 apart share the permutation) */    \
      const int kof = SWZ ? (((ch * (CHUNKB / 16) + lq) ^ row_perm(lrow)) * 16)              \
                          : lq * 16 + ch * CHUNKB;                                           \
      u32x4 av[TM], bv[TN];                                                                  \
      _Pragma("unroll") for (int i = 0; i < TM; ++i)                                         \
        av[i] = *reinterpret_cast<const u32x4*>(pa + i * MB * LROW + kof);                   \
      _Pragma("unroll") for (int j = 0; j < TN; ++j)                                         \
        bv[j] = *reinterpret_cast<const u32x4*>(pb + j * MB * LROW + kof);                   \
      _Pragma("unroll") for (int i = 0; i < TM; ++i)                                         \
        _Pragma("unroll") for (int j = 0; j < TN; ++j)                                       \
          WaveMma<T, MB>::run(av[i], bv[j], acc[i][j]);                                      \
    }                                                                                        \
  }

  // The load cursor starts at slab kt_begin.
  int l_kt = kt_begin, l_cc = kt_begin, l_kx = 0, l_dy = 0, l_dx = 0;
  unsigned l_tapbyte = 0;
  if (!PW) {
    const int tap = kt_begin / g.cchunks;
    const int ky = tap / g.k;
    l_cc = kt_begin - tap * g.cchunks;
    l_kx = tap - ky * g.k;
    l_dy = ky * g.dil;
    l_dx = l_kx * g.dil;
    l_tapbyte = (unsigned)(tap * g.c * ESZ);
  }

  // Software pipeline, unrolled by two so that the register sets and LDS buffers
  // are compile-time: while slab kt is multiplied out of one LDS buffer, slab kt+1
  // (requested one step earlier) is moved from its registers into the other buffer
  // and slab kt+2 is requested.  Requests past kt_end return zeros and are dropped.
  OGLE_LOAD_SLAB(0);
  OGLE_LOAD_SLAB(1);
  OGLE_STORE_SLAB(0, 0);
  __syncthreads();
  for (int kt = kt_begin; kt < kt_end; kt += 2) {
    // An odd slab count runs one extra all-zero slab through the second half: a
    // loop without early exits keeps the accumulators in one set of registers.
    OGLE_LOAD_SLAB(0);
    OGLE_COMPUTE_SLAB(0);
    OGLE_STORE_SLAB(1, 1);
    __syncthreads();
    OGLE_LOAD_SLAB(1);
    OGLE_COMPUTE_SLAB(1);
    OGLE_STORE_SLAB(0, 0);
    __syncthreads();
  }
#undef OGLE_COMPUTE_SLAB
#undef OGLE_LOAD_SLAB
#undef OGLE_STORE_SLAB

  // Epilogue.  Destinations: split-K partial sums go to `partial` (rows of opitch floats,
  // the channel count rounded up to 4 so that rows stay 16-byte aligned); finished outputs
  // go to y, or, with a second destination, channels [0, o1) to y (o1 per pixel) and
  // channels [o1, o) to y2 (o - o1 per pixel).  When the row pitches allow 16-byte stores
  // the accumulators go through a wave-private LDS region to be transposed from the MFMA
  // layout (a lane holds one column) into rows, so that a wave writes whole contiguous row
  // segments with 16-byte stores; bias and activation are applied on the way out.
  // Otherwise each lane stores its elements one by one (32 lanes cover 128 contiguous
  // bytes of a row).
  const int opitch = (g.o + 3) & ~3;
  const int o2 = g.o - o1;
  float* const pdst = partial != nullptr ? partial + (long)split * g.m_total * opitch : nullptr;
  if constexpr (MB == 16) {
    // 16x16 blocks: register r of lane l is row 4 * (l / 16) + r, column l % 16, so the 16
    // lanes of a group store one 64-byte run of an output row.  Partial rows are written
    // up to their padded width (the columns past the last channel hold zeros).
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wave_n * WTN + j * 16 + lrow;
      const float bv = (pdst == nullptr && bias != nullptr && col < g.o) ? bias[col] : 0.f;
      const bool second = col >= o1;
      T* const dst = second ? y2 + (col - o1) : y + col;
      const int dpitch = second ? o2 : o1;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int r = 0; r < REGS; ++r) {
          const int row = m0 + wave_m * WTM + i * 16 + lq * 4 + r;
          if (row >= g.m_total) continue;
          if (pdst != nullptr) {
            if (col < opitch) pdst[(long)row * opitch + col] = acc[i][j][r];
          } else if (col < g.o) {
            dst[out_row_offset(g, row, dpitch)] = from_f32<T>(apply_epilogue(acc[i][j][r] + bv, ep));
          }
        }
      }
    }
    return;
  } else {
  // The staging region (reused K-loop LDS) takes JC 32-column blocks of a wave's tile at a
  // time: as many as fit, so that a row segment a wave stores is as long as possible.
  constexpr auto stage_fits = [](int jc) { return 4 * 32 * (jc * 32 + 4) * 4 <= 2 * STAGE; };
  constexpr int JC = (TN % 4 == 0 && stage_fits(4)) ? 4 : (TN % 2 == 0 && stage_fits(2)) ? 2 : 1;
  static_assert(stage_fits(JC), "epilogue staging exceeds the K-loop LDS");
  constexpr int CW = JC * 32;              // columns staged at once
  constexpr int SROW = CW + 4;             // floats per staged row (padded)
  float* const smw = reinterpret_cast<float*>(lds) + wave * 32 * SROW;
  if (pdst != nullptr || (sizeof(T) == 4 && (o1 & 3) == 0 && (o2 & 3) == 0 && (g.oimg & 3) == 0)) {
    constexpr int LPR = CW / 4;              // lanes covering one staged row
    constexpr int RPI = 64 / LPR;            // rows one store instruction covers
    const int cv = lane % LPR;
    const int rsub = lane / LPR;
#pragma unroll
    for (int j0 = 0; j0 < TN; j0 += JC) {
      const int col = n0 + wave_n * WTN + j0 * 32 + cv * 4;
      float4 bias4 = make_float4(0.f, 0.f, 0.f, 0.f);
      if (pdst == nullptr && bias != nullptr && col < g.o)
        bias4 = *reinterpret_cast<const float4*>(bias + col);
      // row pitch and first column of the destination this lane's four channels lie in
      const bool second = pdst == nullptr && col >= o1;
      const int dpitch = pdst != nullptr ? opitch : (second ? o2 : o1);
      const int dcol = second ? col - o1 : col;
      float* const dbase = pdst != nullptr ? pdst : reinterpret_cast<float*>(second ? y2 : y);
#pragma unroll
      for (int i = 0; i < TM; ++i) {
#pragma unroll
        for (int j = 0; j < JC; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            smw[((r >> 2) * 8 + lh * 4 + (r & 3)) * SROW + j * 32 + l32] = acc[i][j0 + j][r];
#pragma unroll
        for (int it = 0; it < 32 / RPI; ++it) {
          const int row = it * RPI + rsub;
          float4 v = *reinterpret_cast<const float4*>(smw + row * SROW + cv * 4);
          const int grow = m0 + wave_m * WTM + i * 32 + row;
          if (grow < g.m_total && col < g.o) {
            if (pdst == nullptr) {
              v.x = apply_epilogue(v.x + bias4.x, ep);
              v.y = apply_epilogue(v.y + bias4.y, ep);
              v.z = apply_epilogue(v.z + bias4.z, ep);
              v.w = apply_epilogue(v.w + bias4.w, ep);
            }
            const long at = pdst != nullptr ? (long)grow * dpitch : out_row_offset(g, grow, dpitch);
            store_result16(dbase + at + dcol, v);
          }
        }
      }
    }
    return;
  }
  if constexpr (sizeof(T) == 2) {
    if ((g.o & 7) == 0 && y2 == nullptr && (g.oimg & 7) == 0) {
      // fp16 output: the same staging, a lane then takes eight consecutive channels
      // of a row and stores them as one 16-byte vector of halves
      constexpr int LPR = CW / 8;
      constexpr int RPI = 64 / LPR;
      const int cv = lane % LPR;
      const int rsub = lane / LPR;
#pragma unroll
      for (int j0 = 0; j0 < TN; j0 += JC) {
        const int col = n0 + wave_n * WTN + j0 * 32 + cv * 8;
        float bias8[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) bias8[q] = 0.f;
        if (bias != nullptr && col < g.o) {
          const float4 b0 = *reinterpret_cast<const float4*>(bias + col);
          const float4 b1 = *reinterpret_cast<const float4*>(bias + col + 4);
          bias8[0] = b0.x; bias8[1] = b0.y; bias8[2] = b0.z; bias8[3] = b0.w;
          bias8[4] = b1.x; bias8[5] = b1.y; bias8[6] = b1.z; bias8[7] = b1.w;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
          for (int j = 0; j < JC; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
              smw[((r >> 2) * 8 + lh * 4 + (r & 3)) * SROW + j * 32 + l32] = acc[i][j0 + j][r];
#pragma unroll
          for (int it = 0; it < 32 / RPI; ++it) {
            const int row = it * RPI + rsub;
            const float4 v0 = *reinterpret_cast<const float4*>(smw + row * SROW + cv * 8);
            const float4 v1 = *reinterpret_cast<const float4*>(smw + row * SROW + cv * 8 + 4);
            const int grow = m0 + wave_m * WTM + i * 32 + row;
            if (grow < g.m_total && col < g.o) {
              const float f[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
              uint4 packed;
              __half2* h = reinterpret_cast<__half2*>(&packed);
#pragma unroll
              for (int q = 0; q < 4; ++q)
                h[q] = __floats2half2_rn(apply_epilogue(f[2 * q] + bias8[2 * q], ep),
                                         apply_epilogue(f[2 * q + 1] + bias8[2 * q + 1], ep));
              store_result16(reinterpret_cast<__half*>(y) + out_row_offset(g, grow, g.o) + col, packed);
            }
          }
        }
      }
      return;
    }
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = n0 + wave_n * WTN + j * 32 + l32;
    if (col >= g.o) continue;
    const float bv = (pdst == nullptr && bias != nullptr) ? bias[col] : 0.f;
    const bool second = col >= o1;
    T* const dst = second ? y2 + (col - o1) : y + col;
    const int dpitch = second ? o2 : o1;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int rbase = m0 + wave_m * WTM + i * 32 + lh * 4;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = rbase + (r >> 2) * 8 + (r & 3);
        if (row >= g.m_total) continue;
        if (pdst != nullptr) {
          pdst[(long)row * opitch + col] = acc[i][j][r];
        } else {
          dst[out_row_offset(g, row, dpitch)] = from_f32<T>(apply_epilogue(acc[i][j][r] + bv, ep));
        }
      }
    }
  }
  }  // MB == 32
}

// Everything one convolution's workgroups need, as plain data (a kernel argument).
struct IgemmProblem {
  ConvGeom g;
  const void* x;
  const void* w;
  const float* bias;
  void* y;
  void* y2;  // second destination for channels [o1, o), or nullptr
  int o1;    // channels that go to y (== g.o without a second destination)
  Epilogue ep;
  int tiles_n, tiles;
  float* partial;
  int slabs_per_split, splits;
  // mixed-group kernel only, + 1 if pointwise: tiles of 64x64 0, 128x32 2, 128x16 8, wave-split 32x32 4, 16x16 6; as
  // bf16 pieces 64x64 16, 64x32 18 (never pointwise), 32x32 in two K groups 20, 64x16 22
  int variant;
};

// fp32 operands as three bf16 pieces each: x = h + m + l (24 significand bits in three times 8;
// each piece is the rounded rest of the one before, every rest is exact in fp32), so
// x * w = hh + hm + mh + hl + lh + mm plus terms below 2^-26 of the product: six bf16 MFMAs of 16
// cycles per 16x16x32 step where fp32 takes eight of 32.
// The three terms left out cost a product at most 0.43 ulp beside its rounding of half an ulp: a
// sum that one product dominates may be 0.93 ulp off (fp32 MFMAs: 0.5), longer ones are nearer than
// fp32 MFMAs bring them (figures below).
// The pieces are exact for |x| from 2^-110 up to where h overflows.  Below, bf16's smallest
// subnormal cuts them off at 2^-134, which shows in a sum only if its products are tiny too.  So a
// tile with a sum that is not finite, or neither zero nor at least 2^-60, or (whole sums: a range of
// K can lie in the padding) with none but zeros, is contracted by fp32 MFMAs.  What is left are
// operands below 2^-110 that meet others above 2^50 in one sum, and sums of operands below 2^-134
// in a tile with larger sums or in a range of K: these are zero.  (Splitting operands scaled by 2^24
// would be exact for those as well and cost 4 % of every tile, 7 % with 3x3.)
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float floatx2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void split_bf16(const u32x4& v, uint2 (&piece)[3]) {
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    floatx2_t x = {__uint_as_float(v[2 * e]), __uint_as_float(v[2 * e + 1])};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const bf16x2_t h = __builtin_convertvector(x, bf16x2_t);
      (e == 0 ? piece[q].x : piece[q].y) = __builtin_bit_cast(unsigned, h);
      if (q < 2) {
        const unsigned b = __builtin_bit_cast(unsigned, h);
        x[0] -= __uint_as_float(b << 16);
        x[1] -= __uint_as_float(b & 0xffff0000u);
      }
    }
  }
}

// LDS of one workgroup of a pieces tile with NB blocks of 16 output channels: per K group two
// stages of three planes of 64-byte rows.
template <int NB, int KG>
constexpr int pieces_lds_bytes() { return KG * 2 * 3 * NB * 1024; }

// One workgroup's share of an fp32 convolution contracted as bf16 pieces.
//
// WM waves, each with its own 16 * WR output pixels and all 16 * NB channels of the tile.  An input
// value is used by one wave only and goes from memory straight into that wave's registers, where it
// is split; the filter, which all waves share, is split once per workgroup on its way to LDS.  So a
// stage writes only the filter's planes to LDS (72 bytes per cycle and unit measured, against 228 for
// reads) and no input value is split or gathered twice.  KG groups of WM waves take stages in turn and
// add their sums at the end.
//
// A stage is two slabs of 16 channels (each of one tap); v_mfma_f32_16x16x32_bf16 takes it in one
// step.  Lane l holds, of row l % 16 (a pixel, or a channel's filter), channels 4q .. 4q+3 of both
// slabs, q = l / 16: its two 16-byte loads and its neighbours' in q are one 64-byte run.  The filter is
// the first operand: register r of lane l of a result block is pixel l % 16, channel 4 * (l / 16) + r,
// so four channels of a pixel are stored as 16 bytes without a trip through LDS.
//
// The five products below h * h have sums of their own, a few hundredths of the main ones: their
// roundings vanish and the main sums are rounded once per 32 products.
//
// Measured on MI355X against both operands split on their way to LDS (32x32x16 MFMAs, 64 rows of each
// operand per 64x64 tile and 16 channels), us: 19x19x512 -> 512 at batch 16 25.4 -> 23.8, 3x3 56x56x64 ->
// 64 35.6 -> 28.7, 28x28x128 -> 128 38.1 -> 31.3, M = 11552, K = 512, N = 1024 73.1 -> 68.0 (178 TFLOP/s);
// error against 64-bit sums at K = 512 1.24e-7 -> 1.20e-7 (fp32 MFMAs 4.1e-7).  Large problems are bound by
// power: the library's bf16 GEMM of 8192 cubed reaches 1145 / 6 = 191.  Smaller ones share it among LDS
// writes, splitting and MFMAs; loads further ahead, and splitting interleaved with MFMAs by hand, gained nothing.
//
// MODE: KxK, whose slabs are channels of a tap; pointwise; or runs.  With no dilation the taps of a filter row
// are one run of k * c values, in memory as in the filter, whatever the channel count: kRuns cuts that
// run into slabs (g.c is its length, g.pixel the channels), so channel counts that fill no vector cost
// one slab's rest per filter row.  Its 16-byte loads start on any value; waves with pixels whose run
// reaches over the end of an image row clear what lies there, those at the tensor's ends load value by
// value, and so does the filter, where the run's length is no multiple of four.
enum PiecesMode { kKxK = 0, kPointwise = 1, kRuns = 2 };
template <int WR, int NB, int WM, int KG, int MODE>
__device__ __forceinline__ void pieces_tile(unsigned char* __restrict__ lds, const IgemmProblem& p, int bid) {
  constexpr bool PW = MODE == kPointwise, RUNS = MODE == kRuns;
  constexpr int BM = WM * WR * 16, BN = NB * 16;
  constexpr int TG = WM * 64;                          // threads of a K group
  constexpr int BP = (BN * 8 + TG - 1) / TG;           // 16-byte filter vectors a thread loads per stage
  constexpr bool B_PART = BN * 8 % TG != 0;
  constexpr int PLANE = BN * 64, STAGE = 3 * PLANE;
  const ConvGeom& g = p.g;

  int pid, split;
  if (!assign_work(bid, p.tiles_n, p.tiles, p.splits, pid, split)) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int kgroup = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid / TG);
  const int tg = KG == 1 ? tid : tid % TG, wave = __builtin_amdgcn_readfirstlane(tg >> 6);
  const int tile_n = pid % p.tiles_n, tile_m = pid / p.tiles_n;
  const int m0 = tile_m * BM + wave * (WR * 16), n0 = tile_n * BN;
  const int lr = lane & 15, kq = lane >> 4;
  unsigned char* const planes = lds + kgroup * (2 * STAGE);

  const __amdgpu_buffer_rsrc_t rx = make_rsrc(p.x, g.x_bytes);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w, g.w_bytes);

  // this lane's pixels: their offset (PW), or that of their first tap, and its place
  unsigned a_base[WR], a_tap[WR];
  int a_iy[WR], a_ix[WR];   // (runs: a_ix counts values, from the row's first)
  bool edge = false, at_end = false;
#pragma unroll
  for (int i = 0; i < WR; ++i) {
    const int m = m0 + i * 16 + lr;
    const bool ok = m < g.m_total;
    if (PW) {
      a_tap[i] = ok ? (unsigned)m * (unsigned)(g.c * 4) + kq * 16 : kOutOfRange;
    } else {
      const int ox = m % g.ow;
      const int t = m / g.ow;
      const int oy = t % g.oh;
      const int b = t / g.oh;
      a_iy[i] = ok ? oy * g.stride - g.pad : -0x40000000;   // fails every in-image test
      a_ix[i] = ox * g.stride - g.pad;
      a_base[i] = first_tap_offset(g.h, g.w, g.pixel, b, oy * g.stride - g.pad, a_ix[i]) + kq * 16;
      if (RUNS) {
        a_ix[i] *= g.pixel;
        edge = edge || (ok && (a_ix[i] < 0 || a_ix[i] + g.c > g.w * g.pixel));
        at_end = at_end || (ok && runs_leave_tensor(g.n, g.h, g.w * g.pixel, g.k, g.c, b, a_iy[i], a_ix[i]));
        a_ix[i] += kq * 4;
      }
    }
  }
  // this thread's filter rows and its place in the stage: vector bc of eight in a 128-byte row
  const int bc = tg & 7, br = tg >> 3;
  const unsigned krow_bytes = (unsigned)((RUNS ? g.k : g.k * g.k) * g.c * 4);
  const int row_values = g.w * g.pixel;
  const bool over_end = RUNS && __any(edge), by_value = RUNS && __any(at_end), b_by_value = RUNS && (g.c & 3) != 0;
  unsigned b_row[BP];
#pragma unroll
  for (int i = 0; i < BP; ++i) {
    const int row = i * (TG / 8) + br, o = n0 + row;
    b_row[i] = o < g.o && (!B_PART || row < BN) ? (unsigned)o * krow_bytes + (bc & 3) * 16 : kOutOfRange;
  }

  const int kt_begin = split * p.slabs_per_split;
  const int kt_end = min(g.ktiles, kt_begin + p.slabs_per_split);
  const int stages = (kt_end - kt_begin + 1) >> 1;
  __shared__ float bias[BN];
  if (tid < BN) bias[tid] = p.bias != nullptr && n0 + tid < g.o ? p.bias[n0 + tid] : 0.f;

  // Cursor over slabs: the tap's offsets, the slab within the tap.
  int l_kt, l_cc, l_kx, l_dy, l_dx;
  unsigned l_tapbyte;
  auto enter_tap = [&]() {
    const unsigned from = tap_offset(g.w, g.pixel, l_dy, RUNS ? 0 : l_dx);
#pragma unroll
    for (int i = 0; i < WR; ++i) {
      const bool in = (unsigned)(a_iy[i] + l_dy) < (unsigned)g.h &&
                      (RUNS || (unsigned)(a_ix[i] + l_dx) < (unsigned)g.w);
      a_tap[i] = in ? a_base[i] + from : kOutOfRange;
    }
  };
  auto seek = [&](int kt) {
    l_kt = kt;
    if (PW) {
      l_cc = kt;
      l_tapbyte = 0;
    } else {
      const int tap = kt / g.cchunks, ky = RUNS ? tap : tap / g.k;
      l_cc = kt - tap * g.cchunks;
      l_kx = RUNS ? 0 : tap - ky * g.k;
      l_dy = ky * g.dil;
      l_dx = l_kx * g.dil;
      l_tapbyte = (unsigned)(tap * g.c * 4);
      enter_tap();
    }
  };
  auto step = [&]() {
    ++l_kt;
    ++l_cc;
    if (!PW && l_cc == g.cchunks) {
      l_cc = 0;
      l_tapbyte += (unsigned)(g.c * 4);
      l_dx += g.dil;
      if (RUNS || ++l_kx == g.k) {
        l_kx = 0;
        l_dx = 0;
        l_dy += g.dil;
      }
      enter_tap();
    }
  };
  // Requests the loads of the cursor's next stage.  Slabs past the end are zeros, and so are the filter's
  // channels past the last; the input values that these meet are whatever comes next in memory (should
  // that be infinite or NaN, the sums are found not finite and contracted again).
  auto load = [&](u32x4 (&xa)[WR][2], u32x4 (&wb)[BP]) {
    unsigned b_at[2];
    int b_c[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned off = l_kt < kt_end ? 0u : kOutOfRange;
      b_at[h] = l_tapbyte + (unsigned)l_cc * 64u;
      b_c[h] = l_kt < kt_end ? g.c - l_cc * 16 : 0;   // channels left
      if (by_value) {
#pragma unroll
        for (int i = 0; i < WR; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // (below zero before the tensor; as part of an instruction's offset it would not wrap around)
            const int at = (int)((a_tap[i] | off) + (unsigned)l_cc * 64u + e * 4u);
            xa[i][h][e] = __builtin_amdgcn_raw_buffer_load_b32(rx, at < 0 ? (int)kOutOfRange : at, 0, 0);
          }
      } else {
#pragma unroll
        for (int i = 0; i < WR; ++i)
          xa[i][h] = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)((a_tap[i] | off) + (unsigned)l_cc * 64u), 0, 0);
      }
      step();
    }
    const unsigned at = bc & 4 ? b_at[1] : b_at[0];
    const int left = (bc & 4 ? b_c[1] : b_c[0]) - (bc & 3) * 4;
    const unsigned off = left > 0 ? 0u : kOutOfRange;
    if (b_by_value) {
#pragma unroll
      for (int i = 0; i < BP; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          wb[i][e] = __builtin_amdgcn_raw_buffer_load_b32(rw, (int)(left > e ? b_row[i] + at + e * 4u : kOutOfRange), 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < BP; ++i)
        wb[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)((b_row[i] | off) + at), 0, 0);
    }
    if (KG > 1) {
#pragma unroll
      for (int i = 0; i < 2 * (KG - 1); ++i) step();
    }
  };
  // Splits filter values into the planes of buffer `buf`.  Row of 64 bytes: the 16 bytes of q = 0 .. 3; in
  // rows 8 .. 15 of a block q and q ^ 2 change places, so that the 16 lanes an LDS cycle serves (same
  // lane / 32, same parity of (lane >> 2) & 7) read 16 different columns of a 256-byte window.
  auto store_b = [&](int buf, const u32x4 (&wb)[BP]) {
#pragma unroll
    for (int i = 0; i < BP; ++i) {
      const int row = i * (TG / 8) + br;
      if (B_PART && row >= BN) continue;
      uint2 piece[3];
      split_bf16(wb[i], piece);
      unsigned char* at = planes + buf * STAGE + row * 64 + (((bc & 3) ^ ((row >> 2) & 2)) * 16) + (bc >> 2) * 8;
#pragma unroll
      for (int q = 0; q < 3; ++q) *reinterpret_cast<uint2*>(at + q * PLANE) = piece[q];
    }
  };

  typedef floatx4v Acc;
  Acc acc[WR][NB], rest[WR][NB];
#pragma unroll
  for (int i = 0; i < WR; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = rest[i][j] = Acc{0.f, 0.f, 0.f, 0.f};

  // Splits a stage's input values and multiplies them with buffer `buf`.
  auto multiply = [&](int buf, const bf16x8_t (&xp)[WR][3]) {
    // blocks of channels whose operands are held at once (as registers allow)
    constexpr int JB = NB % 2 == 0 && (PW || WR * NB < 16) ? 2 : 1;
    const unsigned char* at = planes + buf * STAGE + lr * 64 + ((kq ^ ((lr >> 2) & 2)) * 16);
#pragma unroll
    for (int j0 = 0; j0 < NB; j0 += JB) {
      bf16x8_t wp[JB][3];
#pragma unroll
      for (int j = 0; j < JB; ++j)
#pragma unroll
        for (int q = 0; q < 3; ++q) wp[j][q] = *reinterpret_cast<const bf16x8_t*>(at + q * PLANE + (j0 + j) * 1024);
      auto product = [&](Acc (&sum)[WR][NB], int qw, int qx) {
#pragma unroll
        for (int j = 0; j < JB; ++j)
#pragma unroll
          for (int i = 0; i < WR; ++i)
            sum[i][j0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wp[j][qw], xp[i][qx], sum[i][j0 + j], 0, 0, 0);
      };
      product(rest, 1, 1);
      product(acc, 0, 0);
      product(rest, 0, 2);
      product(rest, 2, 0);
      product(rest, 0, 1);
      product(rest, 1, 0);
    }
  };
  int c_cc = 0;   // runs: the slab within the run that is split next
  auto split_a = [&](u32x4 (&xa)[WR][2], bf16x8_t (&xp)[WR][3]) {
    if (RUNS) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (over_end) {
#pragma unroll
          for (int i = 0; i < WR; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if ((unsigned)(a_ix[i] + c_cc * 16 + e) >= (unsigned)row_values) xa[i][h][e] = 0u;
        }
        if (++c_cc == g.cchunks) c_cc = 0;
      }
#pragma unroll
      for (int q = 0; q < 2 * (KG - 1); ++q)
        if (++c_cc == g.cchunks) c_cc = 0;
    }
#pragma unroll
    for (int i = 0; i < WR; ++i) {
      uint2 lo[3], hi[3];
      split_bf16(xa[i][0], lo);
      split_bf16(xa[i][1], hi);
#pragma unroll
      for (int q = 0; q < 3; ++q) xp[i][q] = __builtin_bit_cast(bf16x8_t, u32x4{lo[q].x, lo[q].y, hi[q].x, hi[q].y});
    }
  };

  // Two register sets: the loads of stage s + 2 are requested when stage s has been split.  One barrier
  // per stage: the planes of stage s + 1 are written while those of stage s are read.  Large tiles
  // split the filter before they multiply, which frees its registers for the next loads (the other
  // order spills: a quarter slower), small ones behind (19x19x512 -> 512, batch
  // 16, 24.3 instead of 24.9; 3x3 56x56x64 -> 64 33.7 / 34.3).
  {
    constexpr bool SPLIT_FIRST = WR * NB >= 16;
    u32x4 xa[2][WR][2], wb[2][BP];
    bf16x8_t xp[WR][3];
    // Pointwise ones, short as they can be, leave out what the last turns would do for nothing (75x75x64 ->
    // 128 at batch 16 20.3 -> 18.7 us; the others lose by the branches, 3x3 28x28x128 -> 128 31.0 -> 34.7).
    constexpr bool CUT = PW && KG == 1 && WM == 4 && WR == 1;
    auto turn = [&](auto cur, int left) {
      constexpr int C = decltype(cur)::value;
      split_a(xa[C], xp);
      if (SPLIT_FIRST) store_b(C ^ 1, wb[C ^ 1]);
      if (!CUT || left > 2) load(xa[C], wb[C]);
      if (SPLIT_FIRST) __builtin_amdgcn_sched_barrier(0);
      multiply(C, xp);
      if (!SPLIT_FIRST && (!CUT || left > 1)) store_b(C ^ 1, wb[C ^ 1]);
      __syncthreads();
    };
    seek(kt_begin + 2 * kgroup);
    c_cc = l_cc;
    load(xa[0], wb[0]);
    load(xa[1], wb[1]);
    store_b(0, wb[0]);
    __syncthreads();
    const int turns = (stages + KG - 1) / KG;
    for (int t = 0; t + 1 < turns; t += 2) {
      turn(std::integral_constant<int, 0>(), turns - t);
      turn(std::integral_constant<int, 1>(), turns - t - 1);
    }
    if (turns & 1) turn(std::integral_constant<int, 0>(), 1);
  }
#pragma unroll
  for (int i = 0; i < WR; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      asm volatile("" : "+v"(rest[i][j]));   // (the addition would be done in every turn of the loop)
      acc[i][j] += rest[i][j];
    }

  // the K groups' sums, in order
  auto add_groups = [&]() {
    if constexpr (KG > 1) {
      float4* const mine = reinterpret_cast<float4*>(lds) + tg;
      for (int k = 1; k < KG; ++k) {
        if (kgroup == k) {
#pragma unroll
          for (int i = 0; i < WR; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
              mine[(i * NB + j) * TG] = make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]);
        }
        __syncthreads();
        if (kgroup == 0) {
#pragma unroll
          for (int i = 0; i < WR; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
              const float4 t = mine[(i * NB + j) * TG];
              acc[i][j] += Acc{t.x, t.y, t.z, t.w};
            }
        }
        __syncthreads();
      }
    }
  };
  add_groups();
  if ((KG > 1 && kgroup != 0) || m0 >= g.m_total) return;

  // Sums that are not finite (an operand was infinite, NaN or so large that a piece overflowed) or so small
  // that pieces may have been cut off are contracted again, in fp32: 16 pixels x 32 channels at a time, so
  // that an output does not depend on the form that computed it.  What that costs (us with finite operands / a
  // quarter of the rows zero above and below / all zeros / one NaN an image / all NaN): 16 x 224 x 224, 7x7 stem
  // 54 / 59 / 64 / 63 / 195, 4 x 56 x 56, 3x3 99 -> 99 40 / 53 / 53 / 110 / 186, 16 x 56 x 56, 3x3 64 -> 64
  // 32 / 37 / 40 / 58 / 103, 32 x 19 x 19, 1x1 512 -> 1024 79 / 92 / 87 / 111 / 176, 4 x 19 x 19, 512 -> 512 12 / 16 / 16 / 27 / 30.
  {
    constexpr int UJ = NB % 2 == 0 ? 2 : 1;
    constexpr unsigned kLeast = (127u - 60u) << 24;   // 2^-60
    // `low`: least magnitude of the sums that are not zero, as bits
    auto look = [&](int i, int j0, float& probe, unsigned& low) {
#pragma unroll
      for (int j = j0; j < j0 + UJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          probe = fmaf(acc[i][j][r], 0.f, probe);
          low = min(low, (__float_as_uint(acc[i][j][r]) << 1) - 1u);
        }
    };
    float probe_all = 0.f;
    // `low` over all units, and of the unit of this problem where it is largest (those past the last row or
    // channel are zeros)
    unsigned low_all = 0xffffffffu, low_most = 0;
#pragma unroll
    for (int i = 0; i < WR; ++i)
#pragma unroll
      for (int j0 = 0; j0 < NB; j0 += UJ) {
        unsigned low = 0xffffffffu;
        look(i, j0, probe_all, low);
        low_all = min(low_all, low);
        low_most = max(low_most, m0 + i * 16 < g.m_total && n0 + j0 * 16 < g.o ? low : 0u);
      }
    // (no unit is all zeros if some lane has a sum that is not in each)
    const bool seems_right = !__any(probe_all != 0.f || probe_all != probe_all || low_all < kLeast - 1u) &&
                             (p.partial != nullptr || __any(low_most != 0xffffffffu));
    if (!seems_right) {
      unsigned redo = 0;         // units to replace, bit i * NB + j
      bool again = false;
#pragma unroll
      for (int i = 0; i < WR; ++i)
#pragma unroll
        for (int j0 = 0; j0 < NB; j0 += UJ) {
          float probe = 0.f;
          unsigned low = 0xffffffffu;
          look(i, j0, probe, low);
          const bool wrong = __any(probe != 0.f || probe != probe || low < kLeast - 1u);
          const bool zeros = p.partial == nullptr && !__any(low != 0xffffffffu);
          if ((wrong || zeros) && m0 + i * 16 < g.m_total && n0 + j0 * 16 < g.o) {
            redo |= 1u << (i * NB + j0);
            again = again || wrong;
          }
        }
#pragma unroll
      for (int i = 0; i < WR; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) rest[i][j] = Acc{0.f, 0.f, 0.f, 0.f};
      auto wanted = [&](int i, int j) { return (redo >> (i * NB + j / UJ * UJ) & 1) != 0; };
      // input values of the cursor's slab, zeros where they are not the run's or the image's
      auto input = [&](int i) {
        const bool off = l_kt >= kt_end || (redo >> (i * NB) & ((1u << NB) - 1)) == 0 || l_cc * 16 + kq * 4 >= g.c;
        const unsigned at = a_tap[i] + (unsigned)l_cc * 64u;
        u32x4 v;
        if (RUNS && by_value) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[e] = __builtin_amdgcn_raw_buffer_load_b32(rx, off || (int)(at + e * 4u) < 0 ? (int)kOutOfRange : (int)(at + e * 4u), 0, 0);
        } else {
          v = __builtin_amdgcn_raw_buffer_load_b128(rx, off ? (int)kOutOfRange : (int)at, 0, 0);
        }
        if (RUNS) {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if ((unsigned)(a_ix[i] + l_cc * 16 + e) >= (unsigned)row_values || l_cc * 16 + kq * 4 + e >= g.c) v[e] = 0u;
        }
        return v;
      };
      if (redo != 0 && !again) {
        // sums of nothing but zeros: most likely the input is zero here.  Four slabs' loads at a time
        seek(kt_begin);
        bool zeros = true;
#pragma unroll 1
        while (zeros && l_kt < kt_end) {
          u32x4 v[4][WR];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int i = 0; i < WR; ++i) v[u][i] = input(i);
            step();
          }
          unsigned bits = 0;
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < WR; ++i) bits |= (v[u][i][0] | v[u][i][1] | v[u][i][2] | v[u][i][3]) & 0x7fffffffu;
          zeros = !__any(bits != 0);
        }
        if (zeros) redo = 0;   // as they are
      }
      bool w_no_number = false;
      if (redo != 0) {
        // v_mfma_f32_16x16x4_f32 four times per slab, both operands straight from memory
        seek(kt_begin);
#pragma unroll 1
        while (l_kt < kt_end) {
          u32x4 xv[WR];
#pragma unroll
          for (int i = 0; i < WR; ++i) xv[i] = input(i);
          u32x4 wv[NB];
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            bool none = true;
#pragma unroll
            for (int i = 0; i < WR; ++i) none = none && !wanted(i, j);
            const int o = n0 + j * 16 + lr;
            const unsigned at = (unsigned)o * krow_bytes + l_tapbyte + (unsigned)l_cc * 64u + kq * 16u;
            const bool off = none || o >= g.o || l_cc * 16 + kq * 4 >= g.c;
            if (b_by_value) {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                wv[j][e] = __builtin_amdgcn_raw_buffer_load_b32(
                    rw, off || l_cc * 16 + kq * 4 + e >= g.c ? (int)kOutOfRange : (int)(at + e * 4u), 0, 0);
            } else {
              wv[j] = __builtin_amdgcn_raw_buffer_load_b128(rw, off ? (int)kOutOfRange : (int)at, 0, 0);
            }
          }
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            if (RUNS) {
#pragma unroll
              for (int e = 0; e < 4; ++e) w_no_number = w_no_number || (wv[j][e] & 0x7f800000u) == 0x7f800000u;
            }
#pragma unroll
            for (int i = 0; i < WR; ++i)
              if (wanted(i, j)) WaveMma<float, 16>::run(wv[j], xv[i], rest[i][j]);
          }
          step();
        }
      }
      if (RUNS && __any(w_no_number)) {
        // taps outside the image contribute nothing, also where a filter value is infinite: value by value
#pragma unroll
        for (int i = 0; i < WR; ++i) {
#pragma unroll
          for (int j = 0; j < NB; ++j) rest[i][j] = Acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
          for (int ky = 0; ky < g.k; ++ky) {
            if ((unsigned)(a_iy[i] + ky) >= (unsigned)g.h) continue;
            const unsigned x_row = a_base[i] - kq * 16u + (unsigned)(ky * row_values * 4);
#pragma unroll 1
            for (int q = 0; q < g.c; ++q) {
              if ((unsigned)(a_ix[i] - kq * 4 + q) >= (unsigned)row_values) continue;
              const float xv = *reinterpret_cast<const float*>(static_cast<const char*>(p.x) + (x_row + q * 4u));
#pragma unroll
              for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                  const int o = n0 + j * 16 + kq * 4 + r;
                  if (o < g.o) rest[i][j][r] += xv * static_cast<const float*>(p.w)[((long)o * g.k + ky) * g.c + q];
                }
            }
          }
        }
      }
#pragma unroll
      for (int i = 0; i < WR; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (redo >> (i * NB + j / UJ * UJ) & 1) acc[i][j] = rest[i][j];
    }
  }

  // Results.  Split-K partial sums go to `partial` (rows of opitch floats, the channel count rounded up
  // to 4); finished outputs to y or, with a second destination, channels [0, o1) to y and [o1, o) to y2.
  // JC blocks of a wave's 16 pixels change places in LDS of its own, so that a store instruction writes
  // whole runs of a pixel's channels (64 bytes of 16 pixels each, straight from the accumulators: 75x75x128
  // -> 128 at batch 16 33.6 us instead of 31.9).
  constexpr auto fits = [](int jc) { return NB % jc == 0 && WM * 16 * (jc * 16 + 4) * 4 <= pieces_lds_bytes<NB, KG>(); };
  constexpr int JC = fits(4) ? 4 : fits(2) ? 2 : 1;
  static_assert(fits(JC), "result staging exceeds the planes");
  constexpr int PITCH = JC * 16 + 4, LPR = JC * 4, RPI = 64 / LPR;   // floats and lanes per row, rows per instruction
  float* const mine = reinterpret_cast<float*>(lds) + wave * (16 * PITCH);
  const int cv = lane % LPR, rsub = lane / LPR;
  const int opitch = (g.o + 3) & ~3, o1 = p.o1, o2 = g.o - o1;
  const bool whole = p.partial == nullptr;
  // Rows that are no multiple of 16 bytes apart share their cache lines with other stores: written through, every
  // part of a line would go to memory by itself (us written through / left to the L2s, 1x1 M = 293550, 52 -> 33
  // 44.7 / 30.3, M = 120120, 192 -> 35 37.2 / 30.9, M = 22080, 108 -> 138 17.5 / 15.9)
  const bool through = ((o1 | o2 | (int)g.oimg) & 3) == 0;
  typedef float floatx4u __attribute__((ext_vector_type(4), aligned(4)));
  auto put = [&](float* at, const float4& v) {
    if (through) store_result16(at, v);
    else *reinterpret_cast<floatx4u*>(at) = floatx4u{v.x, v.y, v.z, v.w};
  };
  // ONE: finished outputs to dense rows of whole vectors in one destination: nothing else is asked per store (M = 11552,
  // K = 512, N = 1024 73.8 -> 68.0 us, 112 x 112 x 32, 3x3 -> 64 10.2 -> 9.8)
  auto store_all = [&](auto one) {
    constexpr bool ONE = decltype(one)::value;
#pragma unroll
    for (int i = 0; i < WR; ++i) {
#pragma unroll
      for (int j0 = 0; j0 < NB; j0 += JC) {
#pragma unroll
        for (int j = 0; j < JC; ++j) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] = acc[i][j0 + j][r];
            if (ONE || whole) v[r] = apply_epilogue(v[r] + bias[(j0 + j) * 16 + kq * 4 + r], p.ep);
          }
          *reinterpret_cast<float4*>(mine + lr * PITCH + j * 16 + kq * 4) = make_float4(v[0], v[1], v[2], v[3]);
        }
        const int col = n0 + j0 * 16 + cv * 4;
#pragma unroll
        for (int it = 0; it < 16 / RPI; ++it) {
          const float4 v = *reinterpret_cast<const float4*>(mine + (it * RPI + rsub) * PITCH + cv * 4);
          const int row = m0 + i * 16 + it * RPI + rsub;
          if (ONE) {
            if (row < g.m_total && col < g.o) store_result16(static_cast<float*>(p.y) + (long)row * g.o + col, v);
            continue;
          }
          if (row >= g.m_total) continue;
          if (!whole) {
            if (col < opitch) store_result16(p.partial + ((long)split * g.m_total + row) * opitch + col, v);
            continue;
          }
          // (a 16-byte store needs no more than 4-byte alignment)
          float* const dst = static_cast<float*>(p.y) + out_row_offset(g, row, o1) + col;
          float* const dst2 = static_cast<float*>(p.y2) + (long)row * o2 + (col - o1);
          if (col + 4 <= o1) {
            put(dst, v);
          } else if (col >= o1 && col + 4 <= g.o) {
            put(dst2, v);
          } else {
            const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (col + r < g.o) (col + r < o1 ? dst : dst2)[r] = e[r];
          }
        }
      }
    }
  };
  if (whole && through && o2 == 0 && g.oimg == 0) store_all(std::true_type());
  else store_all(std::false_type());
}

template <int WR, int NB, int WM, int KG, int MODE>
__global__ __launch_bounds__(WM * KG * 64, 2) void conv_pieces_kernel(IgemmProblem p) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[pieces_lds_bytes<NB, KG>()];
  pieces_tile<WR, NB, WM, KG, MODE>(lds, p, (int)blockIdx.x);
}

template <typename T, int BM, int BN, int WM, int WN, int ROWB, bool PW>
__global__ __launch_bounds__(256) void conv_igemm_kernel(IgemmProblem p) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[igemm_lds_bytes<BM, BN, ROWB>()];
  igemm_tile<T, BM, BN, WM, WN, ROWB, PW>(lds, p.g, static_cast<const T*>(p.x),
                                          static_cast<const T*>(p.w), p.bias,
                                          static_cast<T*>(p.y), static_cast<T*>(p.y2), p.o1, p.ep,
                                          p.tiles_n, p.tiles, p.partial, p.slabs_per_split, p.splits,
                                          (int)blockIdx.x);
}

// The fp16 128x256 tile: 128 accumulator registers per lane, so the remaining registers
// are capped to keep two waves per SIMD (one workgroup's barrier and LDS waits are then
// covered by the other's MFMAs).
template <bool PW>
__global__ __launch_bounds__(256, 2) void conv_igemm_wide_f16_kernel(IgemmProblem p) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[igemm_lds_bytes<128, 256, 64>()];
  igemm_tile<__half, 128, 256, 2, 2, 64, PW>(lds, p.g, static_cast<const __half*>(p.x),
                                             static_cast<const __half*>(p.w), p.bias,
                                             static_cast<__half*>(p.y), static_cast<__half*>(p.y2), p.o1,
                                             p.ep, p.tiles_n, p.tiles, p.partial, p.slabs_per_split,
                                             p.splits, (int)blockIdx.x);
}

// Several independent convolutions in one grid: blocks [first[i], first[i+1]) work
// on problem i.  Small problems (the SSD heads) then run side by side instead of
// one launch after another, each too small to fill the chip.
constexpr int kMaxGroup = 16;
struct IgemmGroup {
  int count;
  int first[kMaxGroup + 1];
  IgemmProblem p[kMaxGroup];
};

template <int WR, int NB, int WM, int KG, bool PW>
__global__ __launch_bounds__(WM * KG * 64, 2) void conv_pieces_group_kernel(IgemmGroup grp) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[pieces_lds_bytes<NB, KG>()];
  int i = 0;
  while (i + 1 < grp.count && (int)blockIdx.x >= grp.first[i + 1]) ++i;
  pieces_tile<WR, NB, WM, KG, PW>(lds, grp.p[i], (int)blockIdx.x - grp.first[i]);
}

template <typename T, int BM, int BN, int WM, int WN, int ROWB, bool PW>
__global__ __launch_bounds__(256) void conv_igemm_group_kernel(IgemmGroup grp) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[igemm_lds_bytes<BM, BN, ROWB>()];
  int i = 0;
  while (i + 1 < grp.count && (int)blockIdx.x >= grp.first[i + 1]) ++i;
  const IgemmProblem& p = grp.p[i];
  igemm_tile<T, BM, BN, WM, WN, ROWB, PW>(lds, p.g, static_cast<const T*>(p.x),
                                          static_cast<const T*>(p.w), p.bias,
                                          static_cast<T*>(p.y), static_cast<T*>(p.y2), p.o1, p.ep,
                                          p.tiles_n, p.tiles, p.partial, p.slabs_per_split, p.splits,
                                          (int)blockIdx.x - grp.first[i]);
}

template <typename T, bool PW, int TS, int U>
__device__ __forceinline__ void igemm_wave_tile(
    float* __restrict__ red, const ConvGeom& g, const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ bias, T* __restrict__ y, T* __restrict__ y2, int o1, const Epilogue& ep,
    int tiles_n, int bid);

// A group whose members differ in tile shape or in being pointwise: each workgroup
// takes the code path of its own problem.  The branch is uniform over the workgroup;
// the paths without pieces keep up to 16 accumulator registers per lane, those with
// them two sets of 16, so the register budget is that of the largest one.
// SPLIT: some problem of the group is contracted as bf16 pieces.  Its tiles need more registers, LDS
// and code than the others': a group without (the heads of one image) does without them as well.  Forms of
// 128 rows and of two times four waves are replaced (grouped_form) so that four workgroups fit a unit: the heads
// of 64 images 320 -> 311 us, of 16 97 -> 91 (before, 160 registers and 48 KB: three).
template <typename T, int ROWB, bool SPLIT>
__global__ __launch_bounds__(256, SPLIT ? 4 : 1) void conv_igemm_mixed_kernel(IgemmGroup grp) {
  constexpr int kLds = SPLIT ? std::max(igemm_lds_bytes<128, 32, ROWB>(), std::max(pieces_lds_bytes<4, 1>(), pieces_lds_bytes<2, 2>()))
                             : igemm_lds_bytes<128, 32, ROWB>();  // the largest of the tiles below
  static_assert(kLds >= igemm_lds_bytes<128, 16, ROWB>() && kLds >= igemm_lds_bytes<64, 64, ROWB>(), "LDS size");
  __shared__ __attribute__((aligned(16))) unsigned char lds[kLds];
  int i = 0;
  while (i + 1 < grp.count && (int)blockIdx.x >= grp.first[i + 1]) ++i;
  // a copy: with a use of the argument per path, the compiler keeps the whole group in scratch
  typename std::conditional<SPLIT, const IgemmProblem, const IgemmProblem&>::type p = grp.p[i];
  const int bid = (int)blockIdx.x - grp.first[i];
#define OGLE_MIXED_CASE(V, BM, BN, WM, WN, PW)                                                  \
  case V:                                                                                       \
    igemm_tile<T, BM, BN, WM, WN, ROWB, PW>(                                                    \
        lds, p.g, static_cast<const T*>(p.x), static_cast<const T*>(p.w), p.bias,               \
        static_cast<T*>(p.y), static_cast<T*>(p.y2), p.o1, p.ep, p.tiles_n, p.tiles,            \
        p.partial, p.slabs_per_split, p.splits, bid);                                           \
    break;
  if constexpr (SPLIT) {
    switch (p.variant) {
      case 16: pieces_tile<1, 4, 4, 1, false>(lds, p, bid); return;
      case 17: pieces_tile<1, 4, 4, 1, true>(lds, p, bid); return;
      case 18: pieces_tile<1, 2, 4, 1, false>(lds, p, bid); return;
      case 20: pieces_tile<1, 2, 2, 2, false>(lds, p, bid); return;
      case 21: pieces_tile<1, 2, 2, 2, true>(lds, p, bid); return;
      case 22: pieces_tile<1, 1, 4, 1, false>(lds, p, bid); return;
      case 23: pieces_tile<1, 1, 4, 1, true>(lds, p, bid); return;
    }
  }
  switch (p.variant) {
    OGLE_MIXED_CASE(0, 64, 64, 2, 2, false)
    OGLE_MIXED_CASE(1, 64, 64, 2, 2, true)
    OGLE_MIXED_CASE(2, 128, 32, 4, 1, false)
    OGLE_MIXED_CASE(3, 128, 32, 4, 1, true)
    OGLE_MIXED_CASE(8, 128, 16, 4, 1, false)
    OGLE_MIXED_CASE(9, 128, 16, 4, 1, true)
#define OGLE_MIXED_WAVE(V, PW, TS)                                                               \
  case V:                                                                                       \
    /* two steps in flight only: the group kernel's register budget is the 64x64 tile's */      \
    igemm_wave_tile<T, PW, TS, 2>(reinterpret_cast<float*>(lds), p.g, static_cast<const T*>(p.x), \
                               static_cast<const T*>(p.w), p.bias, static_cast<T*>(p.y),         \
                               static_cast<T*>(p.y2), p.o1, p.ep, p.tiles_n, bid);               \
    break;
    OGLE_MIXED_WAVE(4, false, 32)
    OGLE_MIXED_WAVE(5, true, 32)
    OGLE_MIXED_WAVE(6, false, 16)
    default:
      OGLE_MIXED_WAVE(7, true, 16)
#undef OGLE_MIXED_WAVE
  }
#undef OGLE_MIXED_CASE
}

// ---------------------------------------------------------------------------
// Small problems: few output tiles, long contraction (the 1x1 ... 19x19 feature
// maps at batch 1, the extras chain, the SSD heads).  Splitting K across workgroups
// needs a second launch to add the parts, and a dependent launch costs more than
// these convolutions themselves.  Here the split stays inside the workgroup: a
// workgroup owns one 32x32 (or 16x16) output tile, its four waves each contract a quarter of K,
// and the four partial tiles are added through LDS in wave order (a fixed order, so
// the result does not depend on timing).  A wave feeds its MFMAs straight from
// global memory: both operands are K-contiguous, so the 16 bytes a lane loads are
// exactly its share of an MFMA operand (fp32: four k of an 8-wide group, fp16: eight
// k of a 16-wide one); no LDS and no barrier in the K loop, and one wave per SIMD
// can keep its MFMA pipe busy because consecutive MFMAs into one accumulator issue
// back to back.  Operands are re-read by every tile that shares them, which the L2
// absorbs at these sizes.
constexpr int kWaveRedBytes = 4 * 32 * 36 * 4;  // four staged 32x32 partial tiles, padded rows

// U: steps of loads in flight per register set (two sets).
template <typename T, bool PW, int TS, int U>
__device__ __forceinline__ void igemm_wave_tile(
    float* __restrict__ red, const ConvGeom& g, const T* __restrict__ x, const T* __restrict__ w,
    const float* __restrict__ bias, T* __restrict__ y, T* __restrict__ y2, int o1, const Epilogue& ep,
    int tiles_n, int bid) {
  typedef WaveMma<T, TS> M;
  constexpr int ESZ = (int)sizeof(T);
  constexpr int VE = 16 / ESZ;          // elements per 16-byte load
  constexpr int QN = 64 / TS;           // lane groups along k
  constexpr int KSTEP = QN * VE;        // k covered by one step
  constexpr int PITCH = TS + 4;         // floats per row of a staged partial tile
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  // MFMA operand order: lane = q * TS + row.  Loads use the other order, lane =
  // row * QN + q, so that the QN lanes of a row read one contiguous run (the vector
  // cache takes one access per contiguous run, and one per lane otherwise, which is
  // what bounds these problems); a lane permute puts the data into MFMA order.  The
  // 16x16 form of a non-pointwise problem is only chosen for tiny maps that wait on
  // latency, not on the cache, and the permutes only lengthen their chain: those load
  // in MFMA order.
  const int mt = lane % TS, mq = lane / TS;        // MFMA order (also the result layout)
  constexpr bool PERM = PW || TS == 32;
  const int lt = PERM ? lane / QN : mt, lq = PERM ? lane % QN : mq;        // load order
  const int permute_from = (mt * QN + mq) * 4;     // byte address for ds_bpermute
  const int tile_n = bid % tiles_n, tile_m = bid / tiles_n;
  const int m = tile_m * TS + lt;       // the A row this lane loads
  const int col = tile_n * TS + lt;     // the B row (output channel) this lane loads
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(x, g.x_bytes);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(w, g.w_bytes);

  const int csteps = (g.c + KSTEP - 1) / KSTEP;   // steps per tap
  const int steps = g.k * g.k * csteps;
  const int s_begin = (int)(((long)steps * wave) / 4), s_end = (int)(((long)steps * (wave + 1)) / 4);

  // row geometry of this lane
  int iy0 = 0, ix0 = 0;
  unsigned img = 0;
  const bool row_ok = m < g.m_total;
  if (PW) {
    img = (unsigned)m * (unsigned)(g.c * ESZ);
  } else {
    const int ox = m % g.ow;
    const int t = m / g.ow;
    const int oy = t % g.oh;
    const int b = t / g.oh;
    img = (unsigned)b * (unsigned)(g.h * g.w * g.c * ESZ);
    iy0 = oy * g.stride - g.pad;
    ix0 = ox * g.stride - g.pad;
  }
  const unsigned wrow = (unsigned)col * (unsigned)(g.k * g.k * g.c * ESZ);
  const bool col_ok = col < g.o;

  // load cursor: (tap, channel step) of the next step to request
  int l_tap = s_begin / csteps, l_cs = s_begin - l_tap * csteps;
  unsigned a_tap = kOutOfRange, b_tap = kOutOfRange;
  auto enter_tap = [&](int tap) {
    if (PW) {
      a_tap = row_ok ? img : kOutOfRange;
    } else {
      const int ky = tap / g.k, kx = tap - ky * g.k;
      const int iy = iy0 + ky * g.dil, ix = ix0 + kx * g.dil;
      const bool in = row_ok && iy >= 0 && iy < g.h && ix >= 0 && ix < g.w;
      a_tap = in ? img + (unsigned)((iy * g.w + ix) * g.c * ESZ) : kOutOfRange;
    }
    b_tap = col_ok ? wrow + (unsigned)(tap * g.c * ESZ) : kOutOfRange;
  };
  enter_tap(l_tap);

  u32x4 ra[2][U], rb[2][U];
  int requested = s_begin;
#define OGLE_WAVE_LOAD(SET)                                                                      \
  _Pragma("unroll") for (int u = 0; u < U; ++u) {                                                \
    const int cel = l_cs * KSTEP + lq * VE;                                                      \
    const bool ok = requested < s_end && cel < g.c;                                              \
    const unsigned ao = ok && a_tap != kOutOfRange ? a_tap + (unsigned)(cel * ESZ) : kOutOfRange; \
    const unsigned bo = ok && b_tap != kOutOfRange ? b_tap + (unsigned)(cel * ESZ) : kOutOfRange; \
    ra[SET][u] = __builtin_amdgcn_raw_buffer_load_b128(rx, (int)ao, 0, 0);                       \
    rb[SET][u] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)bo, 0, 0);                       \
    ++requested;                                                                                 \
    if (++l_cs == csteps) {                                                                      \
      l_cs = 0;                                                                                  \
      ++l_tap;                                                                                   \
      enter_tap(l_tap);                                                                          \
    }                                                                                            \
  }
#define OGLE_WAVE_MMA(SET)                                                                       \
  _Pragma("unroll") for (int u = 0; u < U; ++u) {                                                \
    u32x4 av, bv;                                                                                \
    _Pragma("unroll") for (int e = 0; e < 4; ++e) {                                              \
      av[e] = PERM ? (unsigned)__builtin_amdgcn_ds_bpermute(permute_from, (int)ra[SET][u][e]) : ra[SET][u][e]; \
      bv[e] = PERM ? (unsigned)__builtin_amdgcn_ds_bpermute(permute_from, (int)rb[SET][u][e]) : rb[SET][u][e]; \
    }                                                                                            \
    M::run(av, bv, acc);                                                                         \
  }

  typename M::Acc acc;
#pragma unroll
  for (int r = 0; r < M::REGS; ++r) acc[r] = 0.f;

  // chunks of U steps, two register sets: the next chunk is in flight while the
  // current one is multiplied; steps past s_end load zeros
  // (the scheduling barriers keep a whole chunk of loads ahead of the MFMAs that
  // consume the previous one; left alone the compiler sinks the loads next to their
  // uses and the wave then waits for memory once per step)
  OGLE_WAVE_LOAD(0);
  for (int s = s_begin; s < s_end; s += 2 * U) {
    OGLE_WAVE_LOAD(1);
    __builtin_amdgcn_sched_barrier(0);
    OGLE_WAVE_MMA(0);
    __builtin_amdgcn_sched_barrier(0);
    OGLE_WAVE_LOAD(0);
    __builtin_amdgcn_sched_barrier(0);
    OGLE_WAVE_MMA(1);
    __builtin_amdgcn_sched_barrier(0);
  }
#undef OGLE_WAVE_LOAD
#undef OGLE_WAVE_MMA

  // the four partial tiles, then their sum in wave order.  Result layout: register r
  // of lane l is row 8*(r/4) + 4*(l/32) + r%4 (32x32) or 4*(l/16) + r (16x16), column l % TS.
  float* mine = red + wave * (TS * PITCH);
#pragma unroll
  for (int r = 0; r < M::REGS; ++r) {
    const int row = TS == 32 ? (r >> 2) * 8 + mq * 4 + (r & 3) : mq * 4 + r;
    mine[row * PITCH + mt] = acc[r];
  }
  __syncthreads();
  constexpr int VPR = TS / 4;             // 4-element groups per row
  if (tid >= TS * VPR) return;            // TS 16: 64 threads finish the tile
  const int orow = tid / VPR, ocol = (tid % VPR) * 4;
  const float* p0 = red + orow * PITCH + ocol;
  float4 sum = *reinterpret_cast<const float4*>(p0);
#pragma unroll
  for (int wv = 1; wv < 4; ++wv) {
    const float4 t = *reinterpret_cast<const float4*>(p0 + wv * (TS * PITCH));
    sum.x += t.x; sum.y += t.y; sum.z += t.z; sum.w += t.w;
  }
  const int grow = tile_m * TS + orow;
  const int gcol = tile_n * TS + ocol;
  if (grow >= g.m_total || gcol >= g.o) return;
  float v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (gcol + q < g.o) v[q] = apply_epilogue(v[q] + (bias != nullptr ? bias[gcol + q] : 0.f), ep);
  }
  if (y2 != nullptr) {
    // two destinations: element by element, each channel to its own tensor
    const int o2 = g.o - o1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = gcol + q;
      if (c >= g.o) continue;
      if (c < o1) y[(long)grow * o1 + c] = from_f32<T>(v[q]);
      else y2[(long)grow * o2 + (c - o1)] = from_f32<T>(v[q]);
    }
    return;
  }
  T* dst = y + out_row_offset(g, grow, g.o) + gcol;
  if ((g.o & 3) == 0 && (g.oimg & 3) == 0) {
    if constexpr (sizeof(T) == 4) {
      store_result16(dst, make_float4(v[0], v[1], v[2], v[3]));
    } else {
      const __half2 lo = __floats2half2_rn(v[0], v[1]), hi = __floats2half2_rn(v[2], v[3]);
      uint2 packed;
      packed.x = *reinterpret_cast<const unsigned*>(&lo);
      packed.y = *reinterpret_cast<const unsigned*>(&hi);
      store_result8(dst, packed);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (gcol + q < g.o) dst[q] = from_f32<T>(v[q]);
  }
}

template <typename T, bool PW, int TS>
__global__ __launch_bounds__(256) void conv_igemm_wave_kernel(IgemmProblem p) {
  __shared__ __attribute__((aligned(16))) float red[kWaveRedBytes / 4];
  igemm_wave_tile<T, PW, TS, 4>(red, p.g, static_cast<const T*>(p.x), static_cast<const T*>(p.w),
                             p.bias, static_cast<T*>(p.y), static_cast<T*>(p.y2), p.o1, p.ep, p.tiles_n,
                             (int)blockIdx.x);
}

struct ReduceProblem {
  const float* partial;  // [splits][m][opitch]
  const float* bias;
  void* y;
  void* y2;   // second destination for channels [o1, o), or nullptr
  long mn;    // m * o output elements
  int o, o1, opitch, splits;
  Epilogue ep;
  int lanes;  // lanes per output element (1, 2, 4 or 8)
  long oimg;  // elements between the outputs of consecutive images in y; 0: dense
  int hw;     // output rows per image
};
struct ReduceGroup {
  int count;
  int first[kMaxGroup + 1];
  ReduceProblem p[kMaxGroup];
};

// Sums the split-K partials, then bias and activation.  A work item is four consecutive
// channels of one output row (the partial rows are padded to a multiple of four floats,
// so it is one 16-byte load per split), shared by LANES consecutive lanes: lane q adds
// splits q, q+LANES, ... in ascending order and the LANES partial sums are then combined
// in a fixed butterfly order, so the result depends on neither timing nor grid shape.
// Spreading the splits over lanes keeps many loads in flight when there are few outputs
// but many splits.
template <typename T, int LANES>
__device__ __forceinline__ void splitk_reduce_block(const ReduceProblem& r, int bid) {
  const int q = threadIdx.x % LANES;
  const int gpr = r.opitch >> 2;       // four-channel groups per row
  const long rows = r.mn / r.o;
  const long idx = (long)bid * (blockDim.x / LANES) + threadIdx.x / LANES;
  const bool live = idx < rows * gpr;  // dead lanes still take part in the shuffles
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  const long row = idx / gpr;
  const int col = (int)(idx - row * gpr) * 4;
  if (live) {
    const float* src = r.partial + row * r.opitch + col;
    const long zstride = rows * r.opitch;
#pragma unroll 4
    for (int z = q; z < r.splits; z += LANES) {
      const float4 t = *reinterpret_cast<const float4*>(src + (long)z * zstride);
      acc.x += t.x; acc.y += t.y; acc.z += t.z; acc.w += t.w;
    }
  }
#pragma unroll
  for (int d = 1; d < LANES; d <<= 1) {
    acc.x += __shfl_xor(acc.x, d, 64);
    acc.y += __shfl_xor(acc.y, d, 64);
    acc.z += __shfl_xor(acc.z, d, 64);
    acc.w += __shfl_xor(acc.w, d, 64);
  }
  if (!live || q != 0) return;
  float v[4] = {acc.x, acc.y, acc.z, acc.w};
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (col + e < r.o) v[e] = apply_epilogue(v[e] + (r.bias != nullptr ? r.bias[col + e] : 0.f), r.ep);
  // where this row's channels start in y
  long at = row * r.o1;
  if (r.oimg != 0) {
    const long b = row / r.hw;
    at = b * r.oimg + (row - b * r.hw) * r.o;
  }
  if (sizeof(T) == 4 && r.y2 == nullptr && (r.o & 3) == 0 && (r.oimg & 3) == 0) {
    store_result16(static_cast<float*>(r.y) + at + col, make_float4(v[0], v[1], v[2], v[3]));
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int c = col + e;
    if (c >= r.o) continue;
    if (c < r.o1) static_cast<T*>(r.y)[at + c] = from_f32<T>(v[e]);
    else static_cast<T*>(r.y2)[row * (r.o - r.o1) + (c - r.o1)] = from_f32<T>(v[e]);
  }
}

template <typename T, int LANES>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(ReduceProblem r) {
  splitk_reduce_block<T, LANES>(r, (int)blockIdx.x);
}

// The reductions of a whole group in one grid; each workgroup uses the lane count
// its own problem was planned with.
template <typename T>
__global__ __launch_bounds__(256) void splitk_reduce_group_kernel(ReduceGroup grp) {
  int i = 0;
  while (i + 1 < grp.count && (int)blockIdx.x >= grp.first[i + 1]) ++i;
  const ReduceProblem& r = grp.p[i];
  const int bid = (int)blockIdx.x - grp.first[i];
  switch (r.lanes) {
    case 8: splitk_reduce_block<T, 8>(r, bid); break;
    case 4: splitk_reduce_block<T, 4>(r, bid); break;
    case 2: splitk_reduce_block<T, 2>(r, bid); break;
    default: splitk_reduce_block<T, 1>(r, bid); break;
  }
}

// Few tile rows spread unevenly over the XCDs: then each gets an eighth of the tiles, or of the (tile, K range)
// pairs, in order.  17 rows of 12 128x64 tiles by rows give one XCD 36 for its 32 units (M = 2116, K = 864 ->
// 768 channels 38.2 us, like this 26.5); 10x10x1024 -> 24, 3x3 at batch 64, with K ranges on XCDs 48.1 us, so 43.5.
// `form` in place of the plan's, as for prepare below.
bool rows_dealt(const IgemmPlan& p, int form, int tiles_m, int tiles_n) {
  return form == FORM_NONE ? rows_even(tiles_m) : pieces_rows_even(tiles_m, (long)tiles_n * p.splits);
}
int work_layout(const IgemmPlan& p, int form, int tiles_m, int tiles_n) {
  const bool rows = rows_dealt(p, form, tiles_m, tiles_n);
  if (p.splits == 1) return rows ? 1 : 0;
  if (p.rows_on_xcd) return rows ? -p.splits : -p.splits - kMaxSplits;
  return p.splits;
}

// Grid size of one problem under that layout.
unsigned grid_blocks(const IgemmPlan& p, int form, int tiles_m, int tiles_n) {
  const int tiles = tiles_m * tiles_n;
  if (p.splits == 1 || p.rows_on_xcd) {
    if (rows_dealt(p, form, tiles_m, tiles_n))
      return 8u * (unsigned)((tiles_m + 7) / 8) * (unsigned)tiles_n * (unsigned)p.splits;
    return 8u * (unsigned)(((long)tiles * p.splits + 7) / 8);
  }
  if (p.splits != 2 && p.splits != 4) return (unsigned)tiles * (unsigned)p.splits;
  const int xpz = 8 / p.splits;
  return 8u * (unsigned)((tiles + xpz - 1) / xpz);
}

struct Prepared {
  IgemmProblem prob;
  ReduceProblem red;
  unsigned grid;
  unsigned reduce_grid;
  int reduce_lanes;
};

// `form` in place of the plan's: what a problem runs as in a grouped launch.
Prepared prepare(const OgleConvArgs& a, long m, const IgemmPlan& p, int form) {
  Prepared out{};
  ConvGeom& g = out.prob.g;
  g.n = a.n; g.h = a.in_h; g.w = a.in_w; g.c = a.in_c;
  g.oh = a.out_h; g.ow = a.out_w; g.o = a.out_c;
  g.k = a.kernel_size; g.stride = a.stride; g.pad = a.padding; g.dil = a.dilation;
  g.pixel = g.c;
  g.m_total = (int)m;
  g.cchunks = p.cchunks;
  g.ktiles = p.ktiles;
  const long esz = a.dtype == OGLE_F16 ? 2 : 4;
  g.x_bytes = (unsigned)((long)a.n * a.in_h * a.in_w * a.in_c * esz);
  g.w_bytes = (unsigned)((long)a.out_c * a.kernel_size * a.kernel_size * a.in_c * esz);
  g.oimg = a.out_image_stride == (long)a.out_h * a.out_w * a.out_c ? 0 : a.out_image_stride;
  const int bm = form != FORM_NONE ? kFormBM[form] : tile_bm(p.cfg);
  const int bn = form != FORM_NONE ? kFormBN[form] : tile_bn(p.cfg);
  const int tiles_m = (g.m_total + bm - 1) / bm;
  const int tiles_n = (g.o + bn - 1) / bn;
  out.prob.x = a.input_dev;
  out.prob.w = a.filter_dev;
  out.prob.bias = a.bias_dev;
  out.prob.y = a.output_dev;
  out.prob.y2 = a.output2_dev;
  out.prob.o1 = a.output2_dev != nullptr ? a.out_c_split : a.out_c;
  out.prob.ep = make_epilogue(a.act, a.min_value, a.max_value, a.act_variant);
  out.prob.tiles_n = tiles_n;
  out.prob.tiles = tiles_m * tiles_n;
  out.prob.partial = p.splits > 1 ? static_cast<float*>(a.workspace_dev) : nullptr;
  out.prob.slabs_per_split = p.slabs_per_split;
  out.prob.splits = work_layout(p, form, tiles_m, tiles_n);
  out.prob.variant = (form == FORM_64x64 ? 16 : form == FORM_64x32 ? 18 : form == FORM_32x32_K2 ? 20 :
                      form == FORM_64x16 ? 22 :
                      p.cfg == CFG_WAVE32 ? 4 : p.cfg == CFG_WAVE16 ? 6 : p.cfg == CFG_128x32 ? 2 :
                      p.cfg == CFG_128x16 ? 8 : 0) +
                     (is_pointwise(a) ? 1 : 0);
  if (is_wave(p.cfg) && form == FORM_NONE) {
    out.grid = (unsigned)(tiles_m * tiles_n);
    return out;
  }
  out.grid = grid_blocks(p, form, tiles_m, tiles_n);
  if (p.splits > 1) {
    const long mn = (long)g.m_total * g.o;
    // enough lanes per output that the grid still has about a thousand waves
    const long items = (long)g.m_total * (((g.o + 3) & ~3) / 4);  // four channels each
    int lanes = 1;
    while (lanes < 8 && lanes * 2 <= p.splits && items * lanes < 64L * 1024) lanes *= 2;
    out.red = ReduceProblem{out.prob.partial, a.bias_dev, a.output_dev, a.output2_dev, mn, g.o,
                            out.prob.o1, (g.o + 3) & ~3, p.splits, out.prob.ep, lanes, g.oimg,
                            g.oh * g.ow};
    out.reduce_lanes = lanes;
    out.reduce_grid = (unsigned)((items * lanes + 255) / 256);
  }
  return out;
}

// The form a problem takes next to others in one launch: with 256 threads, adding in the same order.
int grouped_form(int form) {
  switch (form) {
    case FORM_128x64:
    case FORM_128x64_W8: return FORM_64x64;
    case FORM_64x64_K2:
    case FORM_64x32_K2: return FORM_32x32_K2;
    case FORM_128x32: return FORM_64x32;
    case FORM_128x16: return FORM_64x16;
    default: return form;
  }
}

// Launches pieces kernel `K<WR, NB, WM, KG, PW>`.
#define OGLE_PIECES_CASE(K, FORM, WR, NB, WM, KG)                                            \
  case FORM:                                                                                 \
    if (pw) launch((K<WR, NB, WM, KG, true>), dim3(grid), dim3(WM * KG * 64), 0, s, arg);    \
    else launch((K<WR, NB, WM, KG, false>), dim3(grid), dim3(WM * KG * 64), 0, s, arg);      \
    break;

void launch_pieces(int form, bool pw, unsigned grid, hipStream_t s, const IgemmProblem& arg) {
  switch (form) {
    OGLE_PIECES_CASE(conv_pieces_kernel, FORM_64x64, 1, 4, 4, 1)
    case FORM_128x32:    // no pointwise one is (plan_igemm)
      launch((conv_pieces_kernel<2, 2, 4, 1, false>), dim3(grid), dim3(256), 0, s, arg);
      break;
    OGLE_PIECES_CASE(conv_pieces_kernel, FORM_128x16, 2, 1, 4, 1)
    case FORM_128x128:   // pointwise only; the others have too many registers to keep
      launch((conv_pieces_kernel<2, 8, 4, 1, true>), dim3(grid), dim3(256), 0, s, arg);
      break;
    case FORM_128x64:    // the same
      launch((conv_pieces_kernel<2, 4, 4, 1, true>), dim3(grid), dim3(256), 0, s, arg);
      break;
    OGLE_PIECES_CASE(conv_pieces_kernel, FORM_128x64_W8, 1, 4, 8, 1)
    OGLE_PIECES_CASE(conv_pieces_kernel, FORM_64x64_K2, 1, 4, 4, 2)
    OGLE_PIECES_CASE(conv_pieces_kernel, FORM_64x32_K2, 1, 2, 4, 2)
  }
}

// Launches the convolutions of plan_runs.
void launch_runs(int form, unsigned grid, hipStream_t s, const IgemmProblem& arg) {
#define OGLE_RUNS_CASE(FORM, WR, NB, WM, KG)                                                          \
  case FORM:                                                                                          \
    launch((conv_pieces_kernel<WR, NB, WM, KG, kRuns>), dim3(grid), dim3(WM * KG * 64), 0, s, arg);   \
    break;
  switch (form) {
    OGLE_RUNS_CASE(FORM_64x64, 1, 4, 4, 1)
    OGLE_RUNS_CASE(FORM_128x32, 2, 2, 4, 1)
    OGLE_RUNS_CASE(FORM_128x16, 2, 1, 4, 1)
    OGLE_RUNS_CASE(FORM_128x64_W8, 1, 4, 8, 1)
    OGLE_RUNS_CASE(FORM_64x64_K2, 1, 4, 4, 2)
    OGLE_RUNS_CASE(FORM_64x32_K2, 1, 2, 4, 2)
  }
#undef OGLE_RUNS_CASE
}

// Several problems of one grouped form (and all pointwise or none).
void launch_pieces_group(int form, bool pw, unsigned grid, hipStream_t s, const IgemmGroup& arg) {
  switch (form) {
    OGLE_PIECES_CASE(conv_pieces_group_kernel, FORM_64x64, 1, 4, 4, 1)
    case FORM_64x32:
      launch((conv_pieces_group_kernel<1, 2, 4, 1, false>), dim3(grid), dim3(256), 0, s, arg);
      break;
    OGLE_PIECES_CASE(conv_pieces_group_kernel, FORM_64x16, 1, 1, 4, 1)
    case FORM_128x128:
      launch((conv_pieces_group_kernel<2, 8, 4, 1, true>), dim3(grid), dim3(256), 0, s, arg);
      break;
    OGLE_PIECES_CASE(conv_pieces_group_kernel, FORM_32x32_K2, 1, 2, 2, 2)
  }
}
#undef OGLE_PIECES_CASE

// Instantiates kernel `K<T, BM, BN, WM, WN, ROWB, PW>` for a runtime (dtype, cfg, pw).
#define OGLE_IGEMM_DISPATCH(K, dtype, cfg, pw, grid, s, arg)                                 \
  do {                                                                                       \
    if ((dtype) == OGLE_F16) {                                                               \
      if (pw) {                                                                              \
        OGLE_IGEMM_DISPATCH_F16(K, true, cfg, grid, s, arg)                                  \
      } else {                                                                               \
        OGLE_IGEMM_DISPATCH_F16(K, false, cfg, grid, s, arg)                                 \
      }                                                                                      \
    } else {                                                                                 \
      if (pw) {                                                                              \
        OGLE_IGEMM_DISPATCH_C(K, float, kRowBytesF32, true, cfg, grid, s, arg)               \
      } else {                                                                               \
        OGLE_IGEMM_DISPATCH_C(K, float, kRowBytesF32, false, cfg, grid, s, arg)              \
      }                                                                                      \
    }                                                                                        \
  } while (0)
#define OGLE_IGEMM_CASE(K, T, BM, BN, WM, WN, ROWB, PW, grid, s, arg)                        \
  launch((K<T, BM, BN, WM, WN, ROWB, PW>), dim3(grid), dim3(256), 0, s, arg);                \
  break;
#define OGLE_IGEMM_DISPATCH_C(K, T, ROWB, PW, cfg, grid, s, arg)                             \
  switch (cfg) {                                                                             \
    case CFG_128x96: OGLE_IGEMM_CASE(K, T, 128, 96, 4, 1, ROWB, PW, grid, s, arg)            \
    case CFG_128x160: OGLE_IGEMM_CASE(K, T, 128, 160, 4, 1, ROWB, PW, grid, s, arg)          \
    case CFG_64x64: OGLE_IGEMM_CASE(K, T, 64, 64, 2, 2, ROWB, PW, grid, s, arg)              \
    case CFG_128x32: OGLE_IGEMM_CASE(K, T, 128, 32, 4, 1, ROWB, PW, grid, s, arg)            \
    default: OGLE_IGEMM_CASE(K, T, 128, 16, 4, 1, ROWB, PW, grid, s, arg)                    \
  }
#define OGLE_IGEMM_DISPATCH_F16(K, PW, cfg, grid, s, arg)                                    \
  switch (cfg) {                                                                             \
    case CFG_128x128: OGLE_IGEMM_CASE(K, __half, 128, 128, 2, 2, 128, PW, grid, s, arg)      \
    case CFG_64x64: OGLE_IGEMM_CASE(K, __half, 64, 64, 2, 2, 128, PW, grid, s, arg)          \
    case CFG_128x32: OGLE_IGEMM_CASE(K, __half, 128, 32, 4, 1, 128, PW, grid, s, arg)        \
    default: OGLE_IGEMM_CASE(K, __half, 128, 16, 4, 1, 128, PW, grid, s, arg)                \
  }

// One problem, one grid of the LDS-tiled kernel.
void launch_single(int dtype, int cfg, bool pw, unsigned grid, hipStream_t s, const IgemmProblem& prob) {
  if (cfg == CFG_128x256) {  // fp16 storage only (plan_igemm)
    if (pw) launch(conv_igemm_wide_f16_kernel<true>, dim3(grid), dim3(256), 0, s, prob);
    else launch(conv_igemm_wide_f16_kernel<false>, dim3(grid), dim3(256), 0, s, prob);
    return;
  }
  OGLE_IGEMM_DISPATCH(conv_igemm_kernel, dtype, cfg, pw, grid, s, prob);
}

void launch_wave(int dtype, bool pw, int cfg, const Prepared& pr, hipStream_t s) {
  const dim3 grid(pr.grid), block(256);
#define OGLE_WAVE_LAUNCH(T, PW, TS) \
  launch((conv_igemm_wave_kernel<T, PW, TS>), grid, block, 0, s, pr.prob)
#define OGLE_WAVE_PICK(T)                                                 \
  if (cfg == CFG_WAVE32) {                                                \
    if (pw) OGLE_WAVE_LAUNCH(T, true, 32); else OGLE_WAVE_LAUNCH(T, false, 32); \
  } else {                                                                \
    if (pw) OGLE_WAVE_LAUNCH(T, true, 16); else OGLE_WAVE_LAUNCH(T, false, 16); \
  }
  if (dtype == OGLE_F16) {
    OGLE_WAVE_PICK(__half)
  } else {
    OGLE_WAVE_PICK(float)
  }
#undef OGLE_WAVE_PICK
#undef OGLE_WAVE_LAUNCH
}

template <typename T>
void launch_reduce_single(const Prepared& pr, hipStream_t s) {
  const dim3 grid(pr.reduce_grid), block(256);
  switch (pr.reduce_lanes) {
    case 8: launch((splitk_reduce_kernel<T, 8>), grid, block, 0, s, pr.red); break;
    case 4: launch((splitk_reduce_kernel<T, 4>), grid, block, 0, s, pr.red); break;
    case 2: launch((splitk_reduce_kernel<T, 2>), grid, block, 0, s, pr.red); break;
    default: launch((splitk_reduce_kernel<T, 1>), grid, block, 0, s, pr.red); break;
  }
}

}  // namespace

bool conv_igemm_takes(const OgleConvArgs& a) {
  long m = 0;
  return igemm_eligible(a, &m);
}

size_t conv_igemm_workspace_bytes(const OgleConvArgs& a) {
  long m = 0;
  if (!igemm_eligible(a, &m)) return 0;
  if (f16_async_config(a) >= 0) return 0;
  return plan_igemm(a, m, true).workspace_bytes;
}

int32_t launch_conv_igemm(const OgleConvArgs& a, hipStream_t s) {
  long m = 0;
  if (!igemm_eligible(a, &m)) return OGLE_ERR_UNSUPPORTED;
  if (f16_async_config(a) >= 0) return launch_pw_gemm_f16_async(a, s);
  const IgemmPlan p = final_plan(a, m);
  const Prepared pr = prepare(a, m, p, p.form);
  const bool pw = is_pointwise(a);
  if (p.form != FORM_NONE) {
    launch_pieces(p.form, pw, pr.grid, s, pr.prob);
  } else if (is_wave(p.cfg)) {
    launch_wave(a.dtype, pw, p.cfg, pr, s);
    return check_launch("conv_igemm_wave");
  } else {
    launch_single(a.dtype, p.cfg, pw, pr.grid, s, pr.prob);
  }
  int32_t st = check_launch("conv_igemm");
  if (st != OGLE_OK || p.splits == 1) return st;
  if (a.dtype == OGLE_F16) launch_reduce_single<__half>(pr, s);
  else launch_reduce_single<float>(pr, s);
  return check_launch("splitk_reduce");
}

int32_t launch_conv_runs(const OgleConvArgs& a, hipStream_t s) {
  IgemmPlan p{};
  if (!plan_runs(a, &p)) return OGLE_ERR_UNSUPPORTED;
  Prepared pr = prepare(a, (long)a.n * a.out_h * a.out_w, p, p.form);
  ConvGeom& g = pr.prob.g;
  g.c = a.in_c * a.kernel_size;
  launch_runs(p.form, pr.grid, s, pr.prob);
  return check_launch("conv_pieces_runs");
}

// Launches `count` mutually independent convolutions.  Those the implicit-GEMM
// kernel takes go out as ONE grid (plus one grid for all of their split-K
// reductions) per storage type: a group whose members share the kernel
// instantiation uses that instantiation, a mixed group of 64x64 and 128x32 tiles the
// kernel that branches per workgroup; 128x128-tile problems fill the chip on their
// own and are launched singly.  The others are launched one by one through `fallback`.
int32_t launch_conv_batch(const OgleConvArgs* args, int count, hipStream_t s,
                          int32_t (*fallback)(const OgleConvArgs&, hipStream_t),
                          int32_t* reduce_pending) {
  struct Item {
    int dtype, cfg;
    int own, form;        // alone, and next to others
    bool pw;
    Prepared alone, pr;
    bool wave() const { return form == FORM_NONE && is_wave(cfg); }
  };
  std::vector<Item> items;
  for (int i = 0; i < count; ++i) {
    if (reduce_pending != nullptr) reduce_pending[i] = 0;
    long m = 0;
    if (!igemm_eligible(args[i], &m)) {
      const int32_t st = fallback(args[i], s);
      if (st != OGLE_OK) return st;
      continue;
    }
    if (f16_async_config(args[i]) >= 0) {  // fills the chip on its own: its own launch
      const int32_t st = launch_pw_gemm_f16_async(args[i], s);
      if (st != OGLE_OK) return st;
      continue;
    }
    const IgemmPlan p = final_plan(args[i], m);
    const int form = grouped_form(p.form);
    items.push_back(Item{args[i].dtype, p.cfg, p.form, form, is_pointwise(args[i]), prepare(args[i], m, p, p.form),
                         prepare(args[i], m, p, form)});
    if (reduce_pending != nullptr && p.splits > 1) reduce_pending[i] = 1;
  }
  auto mixable = [](const Item& it) {
    if (it.form != FORM_NONE) return it.form != FORM_128x128;
    return it.cfg == CFG_64x64 || it.cfg == CFG_128x32 || it.cfg == CFG_128x16 || is_wave(it.cfg);
  };
  std::vector<bool> done(items.size(), false);
  for (size_t a0 = 0; a0 < items.size(); ++a0) {
    if (done[a0]) continue;
    IgemmGroup grp{};
    ReduceGroup red{};
    const Item& head = items[a0];
    bool uniform = true, pieces = false;
    for (size_t b0 = a0; b0 < items.size() && grp.count < kMaxGroup; ++b0) {
      const Item& it = items[b0];
      if (done[b0] || it.dtype != head.dtype) continue;
      const bool same = it.form == head.form && (it.form != FORM_NONE || it.cfg == head.cfg) && it.pw == head.pw &&
                        it.cfg != CFG_128x256;
      if (b0 != a0 && (it.cfg == CFG_128x256 || head.cfg == CFG_128x256)) continue;  // fills the chip alone
      if (!same && !(mixable(head) && mixable(it))) continue;
      uniform = uniform && same;
      pieces = pieces || it.form != FORM_NONE;
      done[b0] = true;
      const Prepared& pr = it.pr;
      grp.first[grp.count + 1] = grp.first[grp.count] + (int)pr.grid;
      grp.p[grp.count++] = pr.prob;
      if (pr.prob.splits > 1 || pr.prob.splits < -1) {
        red.first[red.count + 1] = red.first[red.count] + (int)pr.reduce_grid;
        red.p[red.count++] = pr.red;
      }
    }
    const unsigned grid = (unsigned)grp.first[grp.count];
    if (grp.count == 1 && head.own != FORM_NONE) {
      launch_pieces(head.own, head.pw, head.alone.grid, s, head.alone.prob);
    } else if (grp.count == 1 && head.wave()) {
      launch_wave(head.dtype, head.pw, head.cfg, head.pr, s);
    } else if (grp.count == 1) {
      launch_single(head.dtype, head.cfg, head.pw, grid, s, grp.p[0]);
    } else if (uniform && head.form != FORM_NONE) {
      launch_pieces_group(head.form, head.pw, grid, s, grp);
    } else if (uniform && !head.wave()) {
      OGLE_IGEMM_DISPATCH(conv_igemm_group_kernel, head.dtype, head.cfg, head.pw, grid, s, grp);
    } else if (pieces) {
      launch((conv_igemm_mixed_kernel<float, kRowBytesF32, true>), dim3(grid), dim3(256), 0, s, grp);
    } else if (head.dtype == OGLE_F16) {
      launch((conv_igemm_mixed_kernel<__half, 128, false>), dim3(grid), dim3(256), 0, s, grp);
    } else {
      launch((conv_igemm_mixed_kernel<float, kRowBytesF32, false>), dim3(grid), dim3(256), 0, s, grp);
    }
    int32_t st = check_launch("conv_igemm_group");
    if (st != OGLE_OK) return st;
    if (red.count == 0 || reduce_pending != nullptr) continue;  // the caller finishes them later
    const dim3 rgrid((unsigned)red.first[red.count]), block(256);
    if (red.count == 1) {
      Prepared one{};
      one.red = red.p[0];
      one.reduce_grid = rgrid.x;
      one.reduce_lanes = red.p[0].lanes;
      if (head.dtype == OGLE_F16) launch_reduce_single<__half>(one, s);
      else launch_reduce_single<float>(one, s);
    } else if (head.dtype == OGLE_F16) {
      launch((splitk_reduce_group_kernel<__half>), rgrid, block, 0, s, red);
    } else {
      launch((splitk_reduce_group_kernel<float>), rgrid, block, 0, s, red);
    }
    st = check_launch("splitk_reduce_group");
    if (st != OGLE_OK) return st;
  }
  return OGLE_OK;
}

// Finishes convolutions whose contraction was launched with the reduction left pending:
// the plan is a function of the arguments alone, so it is recomputed here and names the
// same partial-sum layout.  All reductions go out in one grid (16 problems per grid).
int32_t launch_conv_reduce(const OgleConvArgs* args, int count, hipStream_t s) {
  int at = 0;
  while (at < count) {
    ReduceGroup red{};
    int dtype = -1;
    for (; at < count && red.count < kMaxGroup; ++at) {
      long m = 0;
      if (!igemm_eligible(args[at], &m) || f16_async_config(args[at]) >= 0) continue;
      const IgemmPlan p = final_plan(args[at], m);
      if (p.splits <= 1) continue;
      if (dtype >= 0 && args[at].dtype != dtype) break;  // one storage type per grid
      dtype = args[at].dtype;
      const Prepared pr = prepare(args[at], m, p, p.form);
      red.first[red.count + 1] = red.first[red.count] + (int)pr.reduce_grid;
      red.p[red.count++] = pr.red;
    }
    if (red.count == 0) continue;
    const dim3 rgrid((unsigned)red.first[red.count]), block(256);
    if (dtype == OGLE_F16) {
      launch((splitk_reduce_group_kernel<__half>), rgrid, block, 0, s, red);
    } else {
      launch((splitk_reduce_group_kernel<float>), rgrid, block, 0, s, red);
    }
    const int32_t st = check_launch("splitk_reduce_group");
    if (st != OGLE_OK) return st;
  }
  return OGLE_OK;
}

// ---------------------------------------------------------------------------
// Split-K scratch that lives in the library's device image, for callers that may
// not allocate.  Every GPU the library runs on holds its own copy of the array
// until the process ends.  In host code the array's name is only a stand-in for the
// symbol, not a device address: the address on the current device comes from
// hipGetSymbolAddress, once per device, and only that pointer is handed to kernels.
static __device__ __align__(256) unsigned char scratch[OGLE_CONV_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// Address of `scratch` on the current device (resolved at the first call on it).
int32_t static_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error("conv2d_noalloc: hipGetDevice: %s", hipGetErrorString(e));
    return OGLE_ERR_NO_DEVICE;
  }
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("conv2d_noalloc: device ordinal %d outside 0..%d", dev, kMaxDevices - 1);
    return OGLE_ERR_UNSUPPORTED;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error("conv2d_noalloc: hipGetSymbolAddress(scratch) on device %d: %s", dev,
                hipGetErrorString(e));
      return OGLE_ERR_NO_DEVICE;
    }
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return OGLE_OK;
}
}  // namespace

// launch_conv_igemm with the split-K partial sums in the static array.  The split-K
// kernels write every partial they later read, so nothing has to start at zero.
int32_t launch_conv_igemm_static_scratch(const OgleConvArgs& a, hipStream_t s) {
  long m = 0;
  if (!igemm_eligible(a, &m)) return OGLE_ERR_UNSUPPORTED;  // the other kernels use no scratch
  const size_t need = f16_async_config(a) >= 0 ? 0 : plan_igemm(a, m, true).workspace_bytes;
  if (need > (size_t)OGLE_CONV_NOALLOC_SCRATCH_BYTES) {
    set_error("conv2d_noalloc: this convolution's split-K plan needs %zu bytes of scratch, the "
              "built-in buffer holds %zu; use ogle_hip_conv2d with a caller workspace",
              need, (size_t)OGLE_CONV_NOALLOC_SCRATCH_BYTES);
    return OGLE_ERR_INVALID_ARG;
  }
  OgleConvArgs q = a;
  q.workspace_dev = nullptr;
  q.workspace_bytes = 0;
  if (need > 0) {
    void* ptr = nullptr;
    const int32_t st = static_scratch(&ptr);
    if (st != OGLE_OK) return st;
    q.workspace_dev = ptr;
    q.workspace_bytes = (size_t)OGLE_CONV_NOALLOC_SCRATCH_BYTES;
  }
  return launch_conv_igemm(q, s);
}

}  // namespace ogle
