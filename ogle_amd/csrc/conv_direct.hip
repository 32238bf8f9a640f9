// Direct convolution over NHWC: everything the MFMA implicit-GEMM kernels do not take (channel
// counts that fill no 16-byte vector, grouped convolutions, the RGB stem).  Four kernels:
// conv_stem_* (K = k*k*C <= 32, group 1), conv_patch_mfma (input patch and filter staged in
// LDS, contracted on the MFMA units), conv_direct_small_k (group 1, the filter in LDS, one thread
// per 4 or 16 channels of a pixel) and conv_direct_general (one thread per output).  plan_direct
// chooses among the last three, for what plan_runs leaves: ungrouped fp32 convolutions without dilation run
// as bf16 pieces (conv_igemm.hip), unless their sums are short, their outputs small, with more than one tap at
// most 16 channels, or an operand reaches 2 GiB.
//
// Semantics follow conv2d.glsl:29-92 / conv2d_grp.glsl:30-123: bias, taps outside the image
// contribute nothing, then the fused activation.
#include <algorithm>
#include <type_traits>
#include "common.h"
#include "conv_plan.h"

namespace ogle {
namespace {

// Small-K kernel: one thread produces OPT consecutive output channels of one pixel.  Filter taps
// [O][K] (K = k*k*C, OHWI order) are staged through LDS transposed to [K][O]; a wave then reads
// the OPT weights of one (tap, channel) as 16-byte broadcasts, and each input value is loaded once
// per thread.  O must be a multiple of OPT.  Bound by its chain of K products (about 0.08 us each)
// while threads are few; plan_direct says which shapes it is for, and what they measured.
template <typename T, int OPT>
__global__ __launch_bounds__(256) void conv_direct_small_k(
    const T* __restrict__ x, const T* __restrict__ w, const float* __restrict__ bias,
    T* __restrict__ y, int n, int h, int wd, int c, int oh, int ow, int o, int k, int stride,
    int pad, int dil, Epilogue ep, int ktot) {
  extern __shared__ __attribute__((aligned(16))) float lds_w[];  // [ktot][o]
  for (int i = threadIdx.x; i < ktot * o; i += blockDim.x) {
    int oc = i / ktot, kk = i - oc * ktot;
    lds_w[kk * o + oc] = to_f32(w[i]);
  }
  __syncthreads();
  const int groups_per_pixel = o / OPT;
  const long total = (long)n * oh * ow * groups_per_pixel;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const int og = (int)(idx % groups_per_pixel);
    long pix = idx / groups_per_pixel;
    const int ox = (int)(pix % ow);
    pix /= ow;
    const int oy = (int)(pix % oh);
    const int b = (int)(pix / oh);
    const int oc0 = og * OPT;
    float acc[OPT];
#pragma unroll
    for (int j = 0; j < OPT; ++j) acc[j] = bias != nullptr ? bias[oc0 + j] : 0.f;
    for (int r = 0; r < k; ++r) {
      const int iy = oy * stride - pad + r * dil;
      if (iy < 0 || iy >= h) continue;
      for (int s = 0; s < k; ++s) {
        const int ix = ox * stride - pad + s * dil;
        if (ix < 0 || ix >= wd) continue;
        const T* xp = x + (((long)b * h + iy) * wd + ix) * c;
        const float* wp = lds_w + (long)((r * k + s) * c) * o + oc0;
        for (int ci = 0; ci < c; ++ci) {
          const float xv = to_f32(xp[ci]);
          const float4* w4 = reinterpret_cast<const float4*>(wp + ci * o);
#pragma unroll
          for (int j = 0; j < OPT / 4; ++j) {
            const float4 wv = w4[j];
            acc[4 * j + 0] += xv * wv.x;
            acc[4 * j + 1] += xv * wv.y;
            acc[4 * j + 2] += xv * wv.z;
            acc[4 * j + 3] += xv * wv.w;
          }
        }
      }
    }
    T* yp = y + (((long)b * oh + oy) * ow + ox) * o + oc0;
    if constexpr (sizeof(T) == 4) {
#pragma unroll
      for (int j = 0; j < OPT / 4; ++j)
        reinterpret_cast<float4*>(yp)[j] =
            make_float4(apply_epilogue(acc[4 * j], ep), apply_epilogue(acc[4 * j + 1], ep),
                        apply_epilogue(acc[4 * j + 2], ep), apply_epilogue(acc[4 * j + 3], ep));
    } else {
#pragma unroll
      for (int j = 0; j < OPT; ++j) yp[j] = from_f32<T>(apply_epilogue(acc[j], ep));
    }
  }
}

// Stem kernel: few input channels, K = k*k*C <= 32 (the RGB stem has K = 27), on
// the MFMA units.  A wave owns 32 output pixels x 32 output channels at a time and
// contracts K with KS = ceil(K/2) v_mfma_f32_32x32x2_f32: lane l supplies
// A[pixel l%32][k = 2s + l/32] and B[k][channel l%32].  The filter values a lane
// needs (KS of them) are loaded once and stay in registers while the wave walks
// over pixel tiles; the lane's KS input taps are gathered straight from global
// memory (the whole receptive field of a tile is a few KB and is served by the
// vector cache), all loads of a tile in flight before the first MFMA.  Rows past
// the end, taps outside the image and the odd K tail contribute zeros.
typedef float stem_acc_t __attribute__((ext_vector_type(16)));
typedef unsigned int stem_u32x2 __attribute__((ext_vector_type(2)));

// 32-bit element offset that no operand reaches (they are kept below 2^31 bytes):
// a buffer access at it reads zero / is dropped.
constexpr unsigned kStemOutOfRange = 0x80000000u;

template <typename T>
__device__ __forceinline__ float stem_load(__amdgpu_buffer_rsrc_t r, unsigned byte_off) {
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)byte_off, 0, 0));
  } else {
    const unsigned short v = __builtin_amdgcn_raw_buffer_load_b16(r, (int)byte_off, 0, 0);
    return __half2float(__builtin_bit_cast(__half, v));
  }
}
template <typename T>
__device__ __forceinline__ void stem_store(__amdgpu_buffer_rsrc_t r, unsigned byte_off, float v) {
  if constexpr (sizeof(T) == 4) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, (int)byte_off, 0, kResultStoreAux);
  } else {
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, __float2half_rn(v)), r,
                                          (int)byte_off, 0, kResultStoreAux);
  }
}

// What K index kidx means, worked out on the host: the tap's (dy, dx) relative to
// the pixel's top-left input position and its element offset from there.
struct StemTaps {
  int dy[32], dx[32], off[32];
};

template <typename T, int KS>
__global__ __launch_bounds__(256) void conv_stem_mfma(
    const T* __restrict__ x, const T* __restrict__ w, const float* __restrict__ bias,
    T* __restrict__ y, int h, int wd, int c, int oh, int ow, int o, int stride, Epilogue ep,
    int ktot, int m_total, int tiles_m, unsigned x_bytes, unsigned y_bytes, StemTaps taps) {
  constexpr unsigned ESZ = sizeof(T);
  const int lane = threadIdx.x & 63;
  const int l32 = lane & 31, lh = lane >> 5;
  const int wave = (int)(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int waves = (int)(gridDim.x * 4);
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(x), 0, (int)x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y, 0, (int)y_bytes, 0x00020000);
  // this lane's K indices: kidx = 2s + lane/32 (entries past K never fall inside the image)
  int tap_dy[KS], tap_dx[KS], tap_off[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    tap_dy[s] = lh ? taps.dy[2 * s + 1] : taps.dy[2 * s];
    tap_dx[s] = lh ? taps.dx[2 * s + 1] : taps.dx[2 * s];
    tap_off[s] = lh ? taps.off[2 * s + 1] : taps.off[2 * s];
  }
  for (int n0 = 0; n0 < o; n0 += 32) {
    const int col = n0 + l32;
    float bval[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int kidx = 2 * s + lh;
      bval[s] = (col < o && kidx < ktot) ? to_f32(w[(long)col * ktot + kidx]) : 0.f;
    }
    const float bias_v = (bias != nullptr && col < o) ? bias[col] : 0.f;
    // the taps of a tile, all issued at once; a tile past the end reads zeros without touching memory
    auto gather = [&](int tile, float (&dst)[KS]) {
      const int m = tile * 32 + l32;
      const int ox = m % ow;
      const int t = m / ow;
      const int oy = t % oh;
      const int b = t / oh;
      const int iy0 = oy * stride, ix0 = ox * stride;
      const int base = (tile < tiles_m && m < m_total) ? ((b * h + iy0) * wd + ix0) * c : -0x40000000;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const bool in = (unsigned)(iy0 + tap_dy[s]) < (unsigned)h &&
                        (unsigned)(ix0 + tap_dx[s]) < (unsigned)wd && base >= 0;
        dst[s] = stem_load<T>(rx, in ? (unsigned)(base + tap_off[s]) * ESZ : kStemOutOfRange);
      }
    };
    float a[KS], a_next[KS];
    gather(wave, a);
    for (int tile = wave; tile < tiles_m; tile += waves) {
      // the next tile's taps are in flight while this tile is multiplied and stored
      gather(tile + waves, a_next);
      stem_acc_t acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], bval[s], acc, 0, 0, 0);
#pragma unroll
      for (int s = 0; s < KS; ++s) a[s] = a_next[s];
      // register r of lane l: pixel 8*(r/4) + 4*(l/32) + r%4 of the tile, channel l%32
      const int row0 = tile * 32 + lh * 4;
      const unsigned off0 = (unsigned)(row0 * o + col);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = (r >> 2) * 8 + (r & 3);
        const bool ok = row0 + dr < m_total && col < o;
        stem_store<T>(ry, ok ? (off0 + (unsigned)(dr * o)) * ESZ : kStemOutOfRange,
                      apply_epilogue(acc[r] + bias_v, ep));
      }
    }
  }
}

// The RGB stem (3x3 taps on 3 channels, fp32, even stride, padding 1, even width, output
// channels a multiple of 32): the nine values one filter row needs for a pixel are nine
// consecutive floats of an input row, so instead of 27 scalar gathers (a counter run showed 32
// vector-cache accesses per such load instruction and the kernel bound by them) a lane fetches
// its share of K as runs of 8-byte pairs.  With an even stride and padding 1 a pixel's run starts
// at an odd float of its row, so the pair that starts one float earlier is 8-byte aligned.  The
// lower half of the wave takes filter row 0 and the first five values of row 1, the upper half
// the last four values of row 1 (plus one zero) and row 2: five pairs for the 9-run and three
// for the rest, eight load instructions instead of fourteen, each twice as wide.  The
// contraction order is permuted to match (the filter values a lane keeps are picked
// accordingly).  Values that fall into padding columns are cleared with a per-lane test, and
// so are padding rows, rows past the end and pairs outside the tensor.
template <int UNUSED = 0>
__global__ __launch_bounds__(256) void conv_stem_rgb_mfma(
    const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias,
    float* __restrict__ y, int h, int wd, int oh, int ow, int o, int stride, Epilogue ep,
    int m_total, int tiles_m, unsigned x_bytes, unsigned y_bytes) {
  constexpr int KS = 14;
  const int lane = threadIdx.x & 63;
  const int l32 = lane & 31, lh = lane >> 5;
  const int wave = (int)(blockIdx.x * 4 + (threadIdx.x >> 6));
  const int waves = (int)(gridDim.x * 4);
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), 0, (int)x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc(y, 0, (int)y_bytes, 0x00020000);
  const int row_floats = wd * 3;
  const unsigned total_floats = x_bytes / 4u;
  const int run0_ky = lh ? 2 : 0;
  const int run1_count = lh ? 4 : 5;
  for (int n0 = 0; n0 < o; n0 += 32) {
    const int col = n0 + l32;
    float bval[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int k = s < 9 ? run0_ky * 9 + s : 9 + (lh ? 5 : 0) + (s - 9);
      bval[s] = (s < 9 || s - 9 < run1_count) ? w[(long)col * 27 + k] : 0.f;
    }
    const float bias_v = bias != nullptr ? bias[col] : 0.f;
    for (int tile = wave; tile < tiles_m; tile += waves) {
      const int m = tile * 32 + l32;
      const int ox = m % ow;
      const int t = m / ow;
      const int oy = t % oh;
      const int b = t / oh;
      const int iy0 = oy * stride - 1;
      const int f0 = (ox * stride - 1) * 3;  // first float of a pixel's 9-run within an input row (odd)
      // PAIRS 8-byte pairs of input row iy from float f (even) on.  Plain 8-byte loads (the
      // 8-byte buffer load builtin compiles to a one-dword load with this toolchain); a pair
      // outside the tensor, or of a row that does not exist, is read from the tensor's start
      // instead and its values are cleared.
      auto fetch = [&](int iy, int f, float* v, auto pairs) {
        const bool row_ok = m < m_total && (unsigned)iy < (unsigned)h;
        const int first = (b * h + iy) * row_floats + f;  // may be negative in the first row
#pragma unroll
        for (int i = 0; i < decltype(pairs)::value; ++i) {
          const int at = first + 2 * i;
          const bool ok = row_ok && (unsigned)at + 1u < total_floats;
          const unsigned byte_off = ok ? (unsigned)at * 4u : 0u;
          const float2 q = *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(x) + byte_off);
          v[2 * i] = ok ? q.x : 0.f;
          v[2 * i + 1] = ok ? q.y : 0.f;
        }
      };
      float v0[10], v1[6];
      fetch(iy0 + run0_ky, f0 - 1, v0, std::integral_constant<int, 5>());
      // filter row 1: floats [f0, f0 + 5) for the lower half, [f0 + 5, f0 + 9) for the upper
      const int f1 = lh ? f0 + 5 : f0 - 1;
      fetch(iy0 + 1, f1, v1, std::integral_constant<int, 3>());
      float a[KS];
#pragma unroll
      for (int j = 0; j < 9; ++j)
        a[j] = (unsigned)(f0 + j) < (unsigned)row_floats ? v0[j + 1] : 0.f;
#pragma unroll
      for (int j = 0; j < 5; ++j) {
        const int f = lh ? f0 + 5 + j : f0 + j;
        const float val = lh ? v1[j] : v1[j + 1];
        a[9 + j] = ((unsigned)f < (unsigned)row_floats && j < run1_count) ? val : 0.f;
      }
      stem_acc_t acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s], bval[s], acc, 0, 0, 0);
      // register r of lane l: pixel 8*(r/4) + 4*(l/32) + r%4 of the tile, channel l%32; rows
      // past the end lie past the end of the buffer and are dropped by the range check
      const unsigned off0 = (unsigned)((tile * 32 + lh * 4) * o + col) * 4u;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = (r >> 2) * 8 + (r & 3);
        __builtin_amdgcn_raw_buffer_store_b32(
            __builtin_bit_cast(unsigned, apply_epilogue(acc[r] + bias_v, ep)), ry,
            (int)(off0 + (unsigned)(dr * o) * 4u), 0, kResultStoreAux);
      }
    }
  }
}

struct DirectGeom {
  int n, h, w, c, oh, ow, o, k, stride, pad, dil, groups;
};

DirectGeom direct_geom(const OgleConvArgs& a) {
  return DirectGeom{a.n,      a.in_h,        a.in_w,   a.in_c,    a.out_h,    a.out_w,
                    a.out_c,  a.kernel_size, a.stride, a.padding, a.dilation, a.group};
}

// One output element: bias first, then ky, kx, input channel ascending; taps outside the image
// are skipped.  Filter OHWI with I = c/groups.
template <typename T>
__device__ __forceinline__ float direct_output(const T* __restrict__ x, const T* __restrict__ w,
                                               const float* __restrict__ bias, const DirectGeom& q, int b,
                                               int oy, int ox, int oc) {
  const int cpg = q.c / q.groups;
  const int g = oc / (q.o / q.groups);
  float acc = bias != nullptr ? bias[oc] : 0.f;
  const T* wf = w + (long)oc * q.k * q.k * cpg;
  for (int r = 0; r < q.k; ++r) {
    const int iy = oy * q.stride - q.pad + r * q.dil;
    if (iy < 0 || iy >= q.h) continue;
    for (int s = 0; s < q.k; ++s) {
      const int ix = ox * q.stride - q.pad + s * q.dil;
      if (ix < 0 || ix >= q.w) continue;
      const T* xp = x + (((long)b * q.h + iy) * q.w + ix) * q.c + g * cpg;
      const T* wp = wf + (r * q.k + s) * cpg;
      for (int ci = 0; ci < cpg; ++ci) acc += to_f32(xp[ci]) * to_f32(wp[ci]);
    }
  }
  return acc;
}

// Fully general kernel: one thread per output element, output channel fastest.
template <typename T>
__global__ __launch_bounds__(256) void conv_direct_general(
    const T* __restrict__ x, const T* __restrict__ w, const float* __restrict__ bias,
    T* __restrict__ y, DirectGeom q, Epilogue ep) {
  const long total = (long)q.n * q.oh * q.ow * q.o;
  for (long idx = (long)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (long)gridDim.x * blockDim.x) {
    const int oc = (int)(idx % q.o);
    long pix = idx / q.o;
    const int ox = (int)(pix % q.ow);
    pix /= q.ow;
    const int oy = (int)(pix % q.oh);
    const int b = (int)(pix / q.oh);
    y[idx] = from_f32<T>(apply_epilogue(direct_output(x, w, bias, q, b, oy, ox, oc), ep));
  }
}

// ---------------------------------------------------------------------------
// Patch kernel: any kernel size, stride, dilation, group count and channel count, on the MFMA
// units.  A workgroup owns 128 output pixels (a box of tb images x th rows x tw columns, powers
// of two) and `gp` groups x COLS output channels.  It stages the input patch those pixels read
// and the filter values of the channels in LDS as fp32 and contracts out of LDS: both are read
// from memory once per workgroup, whatever their alignment, and the gather is an LDS address
// (pixel base + tap offset).  A wave owns 32 of the pixels.  Bound by the fp32 MFMA rate with
// its padding (COLS 16 / 32 / 64 against the channels a group has, K steps of 2 or 4), and for
// small groups by staging and launch latency.
//
// K is walked in runs: consecutive values both in the patch and in a filter row.  A run is one
// tap's channels; with an odd channel count, dilation 1 and all channels staged it is a whole
// filter row of taps (7x7x3: seven runs of 21 instead of 49 of 3).  LDS pitches are odd, so
// lanes on neighbouring pixels hit different banks.  Channels that do not fit LDS at once are
// staged `cc` at a time.
//
// Measured on MI355X, us before (one thread per output; for the 7x7 stem a vector kernel with the
// filter broadcast from LDS) / with this kernel: 4 x 57 x 43, 12 groups of 8 -> 12 183 / 16;
// 4 x 48 x 48, 32 groups of 32 -> 32 9909 / 117; 4 x 56 x 56, 99 -> 99 3x3 2995 / 96; 16 x 224 x 224,
// 3 -> 64 7x7 stride 2 168 / 99 (the products alone: 24 at the fp32 MFMA rate).  Waits for staging
// are what is left, so residency counts: registers are capped for three workgroups per unit (64
// columns: 103 -> 99, 32 groups of 32: 142 -> 117).  Staging by whole rows, without index
// arithmetic, was 15 % slower on the stem and its extra code cost the other shapes 8 %.
//
// Taps outside the image are staged as zeros.  0 * w is 0 only for a finite w, so a workgroup
// that meets an infinite or NaN filter value computes its outputs one by one instead, skipping taps.

__device__ __forceinline__ int div_fast(int n, const FastDiv& f) {
  return f.d == 1 ? n : (int)__umulhi((unsigned)n, f.mul);
}

// Scalar loads a thread has in flight while it stages.  More make longer code that is fetched
// cold by every launch, and 16 spilled registers (12 groups of 8 -> 12 channels, 3x3: 33 us).
constexpr int kPatchBatch = 8;

// V consecutive values (V 4: from a 4-element boundary) as fp32; zeros unless `on`, when `src`
// is some readable address all the same.
template <typename T, int V>
__device__ __forceinline__ void load_some(const T* src, bool on, float (&v)[V]) {
  struct __attribute__((aligned(sizeof(T) * V))) Pack { T e[V]; };
  const Pack q = *reinterpret_cast<const Pack*>(src);
#pragma unroll
  for (int e = 0; e < V; ++e) v[e] = on ? to_f32(q.e[e]) : 0.f;
}

template <typename T, int COLS>
__global__ __launch_bounds__(256, COLS == 16 ? 4 : 3) void conv_patch_mfma(const T* __restrict__ x, const T* __restrict__ w,
                                                       const float* __restrict__ bias, T* __restrict__ y,
                                                       DirectGeom q, PatchPlan p, Epilogue ep) {
  extern __shared__ __attribute__((aligned(16))) float patch_lds[];
  __shared__ int filter_not_finite;
  static_assert(sizeof(filter_not_finite) <= kPatchStaticLds, "the plan leaves room for it");
  constexpr int MB = COLS == 16 ? 16 : 32;            // MFMA block
  constexpr int FR = 32 / MB;                         // blocks along a wave's 32 pixels
  constexpr int NB = COLS / MB;                       // blocks along the columns
  constexpr int KQ = 64 / MB;                         // k values of one MFMA
  constexpr int WP = COLS + 1;                        // filter row pitch in LDS
  constexpr int REGS = MB == 32 ? 16 : 4;
  typedef float acc32_t __attribute__((ext_vector_type(16)));
  typedef float acc16_t __attribute__((ext_vector_type(4)));
  typedef typename std::conditional<MB == 32, acc32_t, acc16_t>::type Acc;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int lrow = lane % MB, lq = lane / MB;
  float* const patch = patch_lds;
  float* const wl = patch_lds + p.patch_floats;
  const int cpg = q.c / q.groups, opg = q.o / q.groups;
  const int ktot = q.k * q.k * cpg;

  // column blocks fastest, then groups: the workgroups that read one patch are neighbours, on
  // one XCD's L2
  int id = xcd_swizzle((int)blockIdx.x, (int)gridDim.x);
  const int cb = id % p.col_blocks;
  id /= p.col_blocks;
  const int g0 = (id % p.gblocks) * p.gp;
  const int tblock = id / p.gblocks;
  const int groups_here = min(p.gp, q.groups - g0);
  const int col0 = cb * COLS;
  const int cols_here = min(COLS, opg - col0);
  const int tiles = p.tiles_b * p.tiles_y * p.tiles_x;
  const int box_w = 1 << p.tw_log, box_h = 1 << p.th_log;
  const int row_pitch = p.pw * p.pitch, img_pitch = p.ph * row_pitch;

  // patch offset of this lane's pixel in each of its MFMA blocks
  int pix_off[FR];
#pragma unroll
  for (int f = 0; f < FR; ++f) {
    const int pix = wave * 32 + f * MB + lrow;
    const int tx = pix & (box_w - 1), ty = (pix >> p.tw_log) & (box_h - 1), tb = pix >> (p.tw_log + p.th_log);
    pix_off[f] = tb * img_pitch + (ty * row_pitch + tx * p.pitch) * p.box_step;
  }

  // `bad`: this thread has staged an infinite or NaN filter value; `repair`: some thread of the
  // workgroup has
  bool bad = false, repair = false;
  if (tid == 0) filter_not_finite = 0;
  for (int tile = tblock; tile < tiles; tile += p.tile_blocks) {
    const int bx = tile % p.tiles_x;
    const int rest = tile / p.tiles_x;
    const int by = rest % p.tiles_y, bb = rest / p.tiles_y;
    const int ox0 = bx << p.tw_log, oy0 = by << p.th_log, b0 = bb * (kPatchPixels >> (p.tw_log + p.th_log));
    const int iy0 = oy0 * q.stride - q.pad, ix0 = ox0 * q.stride - q.pad;

    // with gp > 1 all channels are staged at once: only one of the two loops below has more
    // than one turn, and one set of accumulators serves both
    Acc acc[FR][NB];
    for (int c0 = 0; c0 < cpg; c0 += p.cc) {
      const int cc = min(p.cc, cpg - c0);
      const int cs = p.gp > 1 ? groups_here * cpg : cc;   // channels per patch pixel this time
      // the last chunk and the last group block are narrower than the divisors the host prepared
      const bool full = cc == p.cc && groups_here == p.gp;
      const FastDiv d_cs = full ? p.d_cs : fast_div(cs), d_runk = full ? p.d_runk : fast_div(q.k * q.k * cc);
      __syncthreads();   // the previous contraction has read its operands
      // input patch: [image][row][column][channel], zeros outside the image
      {
        const T* src = x + g0 * cpg + c0;
        const int total = (kPatchPixels >> (p.tw_log + p.th_log)) * p.ph * p.pw * cs;
        auto stage = [&](auto vec) {
          constexpr int V = decltype(vec)::value, U = V == 1 ? kPatchBatch : 2;
          for (int i0 = tid * V; i0 < total; i0 += 256 * V * U) {
            float v[U][V];
            int at[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {   // every load of the batch before the first LDS write
              const int i = i0 + u * 256 * V;
              const int px_all = div_fast(i, d_cs);
              const int ch = i - px_all * cs;
              const int prow = div_fast(px_all, p.d_pw);
              const int px = px_all - prow * p.pw;
              const int b = div_fast(prow, p.d_ph);
              const int iy = iy0 + (prow - b * p.ph) * p.in_step, ix = ix0 + px * p.in_step;
              const bool in = i < total && b0 + b < q.n && (unsigned)iy < (unsigned)q.h && (unsigned)ix < (unsigned)q.w;
              at[u] = i < total ? px_all * p.pitch + ch : -1;
              load_some<T, V>(src + (in ? (unsigned)((((b0 + b) * q.h + iy) * q.w + ix) * q.c + ch) : 0u), in, v[u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (at[u] >= 0)
#pragma unroll
                for (int e = 0; e < V; ++e) patch[at[u] + e] = v[u][e];
          }
        };
        // four channels at a time where every pixel's share starts on a vector boundary
        if (p.vec_x && (cs & 3) == 0) stage(std::integral_constant<int, 4>());
        else stage(std::integral_constant<int, 1>());
      }
      // filter values: [group][run][k in run][column]; they stay when all channels fit at once
      if (tile == tblock || p.cc < cpg) {
        const int kk_total = q.k * q.k * cc;
        const int total = groups_here * cols_here * kk_total;
        auto stage = [&](auto vec) {
          constexpr int V = decltype(vec)::value, U = V == 1 ? kPatchBatch : 2;
          for (int i0 = tid * V; i0 < total; i0 += 256 * V * U) {
            float v[U][V];
            int at[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              // kk fastest: a filter row is read contiguously (all channels staged) or run by run
              const int i = i0 + u * 256 * V;
              const int row = div_fast(i, d_runk);
              const int kk = i - row * kk_total;
              const int gi = cols_here == COLS ? row / COLS : div_fast(row, p.d_col);
              const int col = row - gi * cols_here;
              long from = ((long)(g0 + gi) * opg + col0 + col) * ktot;
              if (cc == cpg) {
                from += kk;
              } else {
                const int tap = div_fast(kk, d_cs);   // gp == 1: cs is cc
                from += tap * cpg + c0 + (kk - tap * cc);
              }
              at[u] = i < total ? (gi * kk_total + kk) * WP + col : -1;
              load_some<T, V>(w + (i < total ? from : 0), i < total, v[u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
              if (at[u] >= 0)
#pragma unroll
                for (int e = 0; e < V; ++e) {
                  bad = bad || !(fabsf(v[u][e]) <= 3.402823466e38f);
                  wl[at[u] + e * WP] = v[u][e];
                }
          }
        };
        if (p.vec_w) stage(std::integral_constant<int, 4>());
        else stage(std::integral_constant<int, 1>());
        if (bad) filter_not_finite = 1;
      }
      __syncthreads();

      const int len = p.runs_x == 1 ? q.k * cc : cc;    // values per run
      for (int gi = 0; gi < groups_here; ++gi) {
        if (c0 == 0) {
#pragma unroll
          for (int f = 0; f < FR; ++f)
#pragma unroll
            for (int n = 0; n < NB; ++n)
#pragma unroll
              for (int r = 0; r < REGS; ++r) acc[f][n][r] = 0.f;
        }
        int wrow = gi * q.k * q.k * cc;
        for (int ky = 0; ky < q.k; ++ky) {
          for (int kx = 0; kx < p.runs_x; ++kx, wrow += len) {
            const float* pa = patch + ky * q.dil * row_pitch + kx * q.dil * p.pitch + gi * cpg + lq;
            const float* pb = wl + (wrow + lq) * WP + lrow;
            auto multiply = [&](const float (&av)[FR], const float (&bv)[NB]) {
#pragma unroll
              for (int f = 0; f < FR; ++f)
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                  if constexpr (MB == 32)
                    acc[f][n] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[f], bv[n], acc[f][n], 0, 0, 0);
                  else
                    acc[f][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[f], bv[n], acc[f][n], 0, 0, 0);
                }
            };
            int j = 0;
            for (; j + 4 * KQ <= len; j += 4 * KQ) {   // four steps of operands read ahead
              float av[4][FR], bv[4][NB];
#pragma unroll
              for (int u = 0; u < 4; ++u) {
#pragma unroll
                for (int f = 0; f < FR; ++f) av[u][f] = pa[pix_off[f] + j + u * KQ];
#pragma unroll
                for (int n = 0; n < NB; ++n) bv[u][n] = pb[(j + u * KQ) * WP + n * MB];
              }
#pragma unroll
              for (int u = 0; u < 4; ++u) multiply(av[u], bv[u]);
            }
            for (; j + KQ <= len; j += KQ) {
              float av[FR], bv[NB];
#pragma unroll
              for (int f = 0; f < FR; ++f) av[f] = pa[pix_off[f] + j];
#pragma unroll
              for (int n = 0; n < NB; ++n) bv[n] = pb[j * WP + n * MB];
              multiply(av, bv);
            }
            if (j < len) {   // the run's last values: lanes past its end contribute 0 * 0
              const bool on = lq < len - j;
              const int back = on ? 0 : lq;
              float av[FR], bv[NB];
#pragma unroll
              for (int f = 0; f < FR; ++f) av[f] = on ? pa[pix_off[f] + j - back] : 0.f;
#pragma unroll
              for (int n = 0; n < NB; ++n) bv[n] = on ? pb[(j - back) * WP + n * MB] : 0.f;
              multiply(av, bv);
            }
          }
        }
        if (c0 + p.cc < cpg) continue;   // more channels of this group to come (gp == 1)
        // where this lane's results go: register r is pixel 8*(r/4) + 4*(lane/32) + r%4 (32x32)
        // or 4*(lane/16) + r (16x16) of the block, column lane % MB
        constexpr unsigned kNoPixel = 0xffffffffu;
        unsigned y_off[FR][REGS];
#pragma unroll
        for (int f = 0; f < FR; ++f)
#pragma unroll
          for (int r = 0; r < REGS; ++r) {
            const int pix = wave * 32 + f * MB + (MB == 32 ? (r >> 2) * 8 + lq * 4 + (r & 3) : lq * 4 + r);
            const int ox = ox0 + (pix & (box_w - 1)), oy = oy0 + ((pix >> p.tw_log) & (box_h - 1));
            const int b = b0 + (pix >> (p.tw_log + p.th_log));
            y_off[f][r] = ox < q.ow && oy < q.oh && b < q.n ? (unsigned)(((b * q.oh + oy) * q.ow + ox) * q.o) : kNoPixel;
          }
        const int obase = (g0 + gi) * opg + col0;
#pragma unroll
        for (int n = 0; n < NB; ++n) {
          const int col = n * MB + lrow;
          if (col >= cols_here) continue;
          const float bv = bias != nullptr ? bias[obase + col] : 0.f;
#pragma unroll
          for (int f = 0; f < FR; ++f)
#pragma unroll
            for (int r = 0; r < REGS; ++r)
              if (y_off[f][r] != kNoPixel)
                y[y_off[f][r] + (unsigned)(obase + col)] = from_f32<T>(apply_epilogue(acc[f][n][r] + bv, ep));
        }
      }
    }

    if (tile == tblock) repair = filter_not_finite != 0;   // (in chunks: one box per workgroup)
    if (repair) {
      // outputs go by thread index: every wave's contracted ones have been stored before
      __threadfence();
      __syncthreads();
      const int per_pixel = groups_here * cols_here;
      for (int i = tid; i < kPatchPixels * per_pixel; i += 256) {
        const int pix = i / per_pixel, rest2 = i - pix * per_pixel;
        const int gi = rest2 / cols_here, col = rest2 - gi * cols_here;
        const int ox = ox0 + (pix & (box_w - 1)), oy = oy0 + ((pix >> p.tw_log) & (box_h - 1));
        const int b = b0 + (pix >> (p.tw_log + p.th_log));
        const int oc = (g0 + gi) * opg + col0 + col;
        if (ox < q.ow && oy < q.oh && b < q.n)
          y[(unsigned)(((b * q.oh + oy) * q.ow + ox) * q.o + oc)] =
              from_f32<T>(apply_epilogue(direct_output(x, w, bias, q, b, oy, ox, oc), ep));
      }
    }
  }
}

template <typename T>
int32_t launch_patch(const OgleConvArgs& a, const PatchPlan& p, const Epilogue& ep, hipStream_t s) {
  const T* x = static_cast<const T*>(a.input_dev);
  const T* w = static_cast<const T*>(a.filter_dev);
  T* y = static_cast<T*>(a.output_dev);
  const dim3 grid((unsigned)(p.tile_blocks * p.gblocks * p.col_blocks)), block(256);
  const size_t lds = sizeof(float) * (size_t)p.lds_floats;
  const DirectGeom q = direct_geom(a);
  if (p.cols == 16) launch((conv_patch_mfma<T, 16>), grid, block, lds, s, x, w, a.bias_dev, y, q, p, ep);
  else if (p.cols == 32) launch((conv_patch_mfma<T, 32>), grid, block, lds, s, x, w, a.bias_dev, y, q, p, ep);
  else launch((conv_patch_mfma<T, 64>), grid, block, lds, s, x, w, a.bias_dev, y, q, p, ep);
  return check_launch("conv_patch_mfma");
}

template <typename T>
int32_t run_direct(const OgleConvArgs& a, hipStream_t s) {
  const Epilogue ep = make_epilogue(a.act, a.min_value, a.max_value, a.act_variant);
  const T* x = static_cast<const T*>(a.input_dev);
  const T* w = static_cast<const T*>(a.filter_dev);
  T* y = static_cast<T*>(a.output_dev);
  const int ktot = a.kernel_size * a.kernel_size * a.in_c;
  const long pixels_all = (long)a.n * a.out_h * a.out_w;
  const long esz = (long)sizeof(T);
  const long x_bytes = (long)a.n * a.in_h * a.in_w * a.in_c * esz;
  const long y_bytes = pixels_all * a.out_c * esz;
  if (a.group == 1 && ktot <= 32 && pixels_all >= 4096 && x_bytes < 0x7fffffffL &&
      y_bytes < 0x7fffffffL) {
    const int tiles_m = (int)((pixels_all + 31) / 32);
    // a wave keeps its filter values while it walks over tiles: one wave per tile
    // until every compute unit has three workgroups (measured best), then more tiles
    // per wave
    int blocks = (tiles_m + 3) / 4;
    if (blocks > 256 * 3) blocks = 256 * 3;
    const int ks = (ktot + 1) / 2;
    StemTaps taps;
    for (int kidx = 0; kidx < 32; ++kidx) {
      const int tap = kidx / a.in_c, ci = kidx % a.in_c;
      taps.dy[kidx] = (tap / a.kernel_size) * a.dilation - a.padding;
      taps.dx[kidx] = (tap % a.kernel_size) * a.dilation - a.padding;
      taps.off[kidx] = (taps.dy[kidx] * a.in_w + taps.dx[kidx]) * a.in_c + ci;
      if (kidx >= ktot) taps.dy[kidx] = -0x40000000;
    }
    if (sizeof(T) == 4 && a.kernel_size == 3 && a.in_c == 3 && a.dilation == 1 && a.padding == 1 &&
        a.stride % 2 == 0 && a.in_w % 2 == 0 && a.out_c % 32 == 0 &&
        reinterpret_cast<uintptr_t>(x) % 8 == 0) {
      // four workgroups per compute unit measured best for this one (17.3 against 18.3 us at batch 16)
      const int rgb_blocks = std::min((tiles_m + 3) / 4, 256 * 4);
      launch((conv_stem_rgb_mfma<0>), dim3(rgb_blocks), dim3(256), 0, s,
             reinterpret_cast<const float*>(x), reinterpret_cast<const float*>(w), a.bias_dev,
             reinterpret_cast<float*>(y), a.in_h, a.in_w, a.out_h, a.out_w, a.out_c, a.stride, ep,
             (int)pixels_all, tiles_m, (unsigned)x_bytes, (unsigned)y_bytes);
      return check_launch("conv_stem_rgb_mfma");
    }
#define OGLE_STEM_CASE(KS)                                                                        \
  launch((conv_stem_mfma<T, KS>), dim3(blocks), dim3(256), 0, s, x, w, a.bias_dev, y,  \
                     a.in_h, a.in_w, a.in_c, a.out_h, a.out_w, a.out_c, a.stride, ep, ktot,       \
                     (int)pixels_all, tiles_m, (unsigned)x_bytes, (unsigned)y_bytes, taps)
    if (ks <= 5) OGLE_STEM_CASE(5);
    else if (ks <= 9) OGLE_STEM_CASE(9);
    else if (ks <= 14) OGLE_STEM_CASE(14);
    else OGLE_STEM_CASE(16);
#undef OGLE_STEM_CASE
    return check_launch("conv_stem_mfma");
  }
  if constexpr (sizeof(T) == 4) {
    const int32_t st = launch_conv_runs(a, s);
    if (st != OGLE_ERR_UNSUPPORTED) return st;
  }
  PatchPlan plan;
  const DirectKernel kernel = plan_direct(a, &plan);
  if (kernel == DIRECT_PATCH) return launch_patch<T>(a, plan, ep, s);
  if (kernel == DIRECT_SMALL_K) {
    const bool wide = small_k_is_wide(a);
    const size_t lds = sizeof(float) * (size_t)ktot * a.out_c;
    const long total = pixels_all * (a.out_c / (wide ? 16 : 4));
    int blocks = ceil_div(total, 256);
    if (blocks > 256 * 32) blocks = 256 * 32;
    if (blocks < 1) blocks = 1;
    if (wide) {
      launch((conv_direct_small_k<T, 16>), dim3(blocks), dim3(256), lds, s, x, w, a.bias_dev, y,
             a.n, a.in_h, a.in_w, a.in_c, a.out_h, a.out_w, a.out_c, a.kernel_size, a.stride,
             a.padding, a.dilation, ep, ktot);
    } else {
      launch((conv_direct_small_k<T, 4>), dim3(blocks), dim3(256), lds, s, x, w, a.bias_dev, y,
             a.n, a.in_h, a.in_w, a.in_c, a.out_h, a.out_w, a.out_c, a.kernel_size, a.stride,
             a.padding, a.dilation, ep, ktot);
    }
    return check_launch("conv_direct_small_k");
  }
  const long total = (long)a.n * a.out_h * a.out_w * a.out_c;
  int blocks = ceil_div(total, 256);
  if (blocks > 256 * 64) blocks = 256 * 64;
  if (blocks < 1) blocks = 1;
  launch((conv_direct_general<T>), dim3(blocks), dim3(256), 0, s, x, w, a.bias_dev, y,
         direct_geom(a), ep);
  return check_launch("conv_direct_general");
}

}  // namespace

int32_t launch_conv_direct(const OgleConvArgs& a, hipStream_t s) {
  if (a.dtype == OGLE_F16) return run_direct<__half>(a, s);
  return run_direct<float>(a, s);
}

}  // namespace ogle
