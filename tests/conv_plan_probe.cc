// The convolution dispatch rules, for test_conv_plan_cpu.py: compiled on the spot by the host
// compiler, loaded with ctypes.
#include "conv_plan.h"

using namespace ogle;

// First taps of pixels near the end of a tensor of almost 2 GiB and in a wide padding above it: no signed
// arithmetic that overflows (which a constant expression may not), the 64-bit offset modulo 2^32.
constexpr unsigned offset64(long h, long w, long pixel, long image, long iy, long ix) {
  return (unsigned)((((image * h + iy) * w + ix) * pixel * 4) & 0xffffffffL);
}
static_assert(first_tap_offset(11000, 12000, 4, 0, 11003, 12001) == offset64(11000, 12000, 4, 0, 11003, 12001), "");
static_assert(first_tap_offset(8000, 1000, 4, 16, 7999, 1200) == offset64(8000, 1000, 4, 16, 7999, 1200), "");
static_assert(first_tap_offset(100, 2000, 1000, 1, -40000, -40000) == offset64(100, 2000, 1000, 1, -40000, -40000), "");
// A dilation as large as the map: the last tap, inside the image, from a first one above it.
static_assert(tap_offset(100, 4, 2000000, 50) == offset64(1, 100, 4, 0, 2000000, 50), "");
static_assert(first_tap_offset(1200000, 100, 4, 0, -1100000, 0) + tap_offset(100, 4, 2200000, 0) ==
                  offset64(1200000, 100, 4, 0, 1100000, 0), "");

extern "C" {

// 1 if the patch kernel takes the convolution (once the implicit GEMM, the stem kernels and runs have
// not), then out = columns, groups and channels staged at once, K runs per filter row, boxes,
// workgroups along the boxes, workgroups in all, vector staging of patch and filter, LDS floats.
int probe_patch(const OgleConvArgs* a, int64_t* out) {
  PatchPlan p;
  IgemmPlan runs;
  long m = 0;
  if (igemm_eligible(*a, &m) || plan_runs(*a, &runs) || plan_direct(*a, &p) != DIRECT_PATCH) return 0;
  const int64_t boxes = (int64_t)p.tiles_b * p.tiles_y * p.tiles_x;
  const int64_t v[] = {p.cols, p.gp, p.cc, p.runs_x, boxes, p.tile_blocks,
                       (int64_t)p.tile_blocks * p.gblocks * p.col_blocks, p.vec_x, p.vec_w, p.lds_floats};
  for (int i = 0; i < 10; ++i) out[i] = v[i];
  return 1;
}

// Which of the direct kernels takes the convolution (DirectKernel); -1 if the implicit GEMM does, -2 if it
// is contracted as runs.
int probe_direct(const OgleConvArgs* a) {
  PatchPlan p;
  IgemmPlan runs;
  long m = 0;
  return igemm_eligible(*a, &m) ? -1 : plan_runs(*a, &runs) ? -2 : (int)plan_direct(*a, &p);
}

// 1 if the implicit GEMM takes the convolution, then out = rows and columns of the planned tile, tiles,
// K ranges, workspace bytes, whether fp32 is contracted as bf16 pieces and the rows and columns that a
// workgroup then has.
int probe_igemm(const OgleConvArgs* a, int scratch, int64_t* out) {
  long m = 0;
  if (!igemm_eligible(*a, &m)) return 0;
  const IgemmPlan p = plan_igemm(*a, m, scratch != 0);
  const int bm = tile_bm(p.cfg), bn = tile_bn(p.cfg);
  const int64_t v[] = {bm, bn, (int64_t)((m + bm - 1) / bm) * ((a->out_c + bn - 1) / bn),
                       p.splits, (int64_t)p.workspace_bytes, p.form != FORM_NONE, kFormBM[p.form], kFormBN[p.form]};
  for (int i = 0; i < 8; ++i) out[i] = v[i];
  return 1;
}

// How an fp32 convolution is contracted as bf16 pieces (PiecesForm); -1 if the implicit GEMM does not take it.
int probe_form(const OgleConvArgs* a, int scratch) {
  long m = 0;
  return igemm_eligible(*a, &m) ? plan_igemm(*a, m, scratch != 0).form : -1;
}

// The form that contracts the runs of an ungrouped fp32 convolution of the direct kernels; -1: one of those does.
int probe_runs(const OgleConvArgs* a) {
  long m = 0;
  IgemmPlan p;
  return !igemm_eligible(*a, &m) && plan_runs(*a, &p) ? p.form : -1;
}

// Loads of four values as pieces_tile requests them for runs: the pixels of which some vector holds a value of
// the image, does not lie inside the tensor and is not foretold by runs_leave_tensor.
int probe_runs_lost(const OgleConvArgs* a) {
  const int row_values = a->in_w * a->in_c, run = a->kernel_size * a->in_c;
  const long values = (long)a->n * a->in_h * row_values;
  int lost = 0;
  for (int b = 0; b < a->n; ++b)
    for (int oy = 0; oy < a->out_h; ++oy)
      for (int ox = 0; ox < a->out_w; ++ox) {
        const int iy = oy * a->stride - a->padding, start = (ox * a->stride - a->padding) * a->in_c;
        bool loses = false;
        for (int y = std::max(iy, 0); y < std::min(iy + a->kernel_size, a->in_h); ++y)
          for (int q = 0; q < run; ++q) {   // the vector of each value of the image
            if (start + q < 0 || start + q >= row_values) continue;
            const long at = ((long)b * a->in_h + y) * row_values + start + q / 4 * 4;
            loses = loses || at < 0 || at + 4 > values;
          }
        lost += loses && !runs_leave_tensor(a->n, a->in_h, row_values, a->kernel_size, run, b, iy, start);
      }
  return lost;
}

int probe_rows_even(int tiles_m, int per_row) { return pieces_rows_even(tiles_m, per_row); }
}
