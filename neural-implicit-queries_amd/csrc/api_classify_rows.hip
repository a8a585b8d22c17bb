// Growing-row classification launches (affine_all, affine_truncate,
// affine_append).
#include "niq_internal.h"
#include "niq_rows.h"

namespace {

// affine_all / affine_truncate / affine_append: one box per workgroup, error
// terms streamed through a private HBM scratch.
template <int W, int MODE, int OCC = RowsOcc<W>::value, int CH = RowsCfg<W>::CH>
niq_status launch_rows_w(const niq_model* m, const niq_eval_cfg* cfg, const ClassifyArgs& a, long long max_n,
                         hipStream_t s) {
  constexpr int NW = RowsCfg<W>::NW;
  auto k = k_classify_rows<W, MODE, OCC, CH>;
  const long long d0 = std::max(a.d, a.lower ? 0 : a.vin);
  const int n_keep = cfg ? cfg->truncate_count : 0;
  const int n_append = cfg ? cfg->n_append : 0;
  long long max_rows = d0;
  int n_act = 0;
  for (int i = 0; i + 1 < m->n_layers; ++i)
    if (m->acts[i] != NIQ_ACT_NONE) { max_rows += m->host.L[i].out_pad; ++n_act; }
  if (MODE == ROWS_APPEND) max_rows = d0 + (long long)n_act * n_append;
  if (MODE == ROWS_TRUNCATE) max_rows = d0 + n_keep + 2LL * W;
  max_rows = std::max<long long>(max_rows, 1);
  const size_t per_wg = sizeof(float) * 2 * (size_t)max_rows * W;
  if (max_n == 0) return NIQ_OK;
  long long g = std::min<long long>(max_n, persistent_blocks(k, NW * 64));
  g = std::max<long long>(1, std::min<long long>(g, (long long)((16ull << 30) / per_wg)));
  // Boxes that their corners decide (k_rows_signs): in a tree's levels, which give
  // room for a list of the others.  Not with Sin layers, whose affine rule (the
  // reference's) may carry a negative error term into err and then is no bound (and
  // whose rounding is not known).
  const bool signs = a.list && a.lower && a.d == 3 && !a.bounds && m->bounded &&
                     std::isfinite(m->round_rel) && max_n >= kRowsSignsMin;
  // A tree's top levels in passes, where a box costs far more than a pass's latency and
  // the heap is many rounds of the resident workgroups: depth-18 affine_all tree of
  // the 128x8 TanH net 24.0 -> 17.9 ms (3 passes 21.0, 8 passes 19.6), depth 11 (4,095
  // nodes) of 256x4 TanH 7.7 -> 4.6, of 512x3 33 -> 14.7, of 256x6 ReLU, whose boxes are
  // hardly ever certified, 13.7 -> 18.5 (22.3 without k_rows_signs).  With fewer nodes the
  // passes' latency is the larger: depth 9 of 256x4 TanH 2.5 -> 4.4, of 256x6 ReLU
  // 3.2 -> 9.5.  Nor at widths below 128 (affine_all tree of a 32x4 net 0.99 -> 1.04) or
  // in the other modes (affine_truncate tree of the 32x8 fox net 8.1 -> 8.9).
  const bool heap = signs && a.heap && MODE == ROWS_ALL && W >= 128 && max_n >= kRowsHeapMin;
  void* scratch = nullptr;
  HIPCHK(hipMallocAsync(&scratch, per_wg * g, s));
  RowsArgs ra{};
  ra.c = a;
  if (signs) {
    ra.c.noise = kNoiseRoom * m->round_out;
    constexpr int NW_S = W <= 64 ? 4 : 8;
    auto ks = k_rows_signs<16, NW_S, W>;
    hipLaunchKernelGGL(ks, dim3(tile_grid((max_n + 15) / 16, persistent_blocks(ks, NW_S * 64))), dim3(NW_S * 64), 0, s,
                       m->dev, ra.c, heap);
  } else {
    ra.c.list = nullptr;
  }
  ra.scratch = static_cast<float*>(scratch);
  ra.max_rows = max_rows;
  ra.n_keep = n_keep;
  ra.n_append = n_append;
  for (int pass = 0; pass < (heap ? kRowsHeapPasses : 1); ++pass) {
    if (heap) {
      hipLaunchKernelGGL(k_rows_heap_list, dim3(1), dim3(1024), 0, s, a.codes, (int)max_n,
                         pass == kRowsHeapPasses - 1, a.list, a.list_n);
    }
    hipLaunchKernelGGL(k, dim3((unsigned)g), dim3(NW * 64), 0, s, m->dev, ra);
  }
  const hipError_t e = hipGetLastError();
  HIPCHK(hipFreeAsync(scratch, s));
  if (e != hipSuccess) return fail(NIQ_ERR_HIP, std::string("k_classify_rows: ") + hipGetErrorString(e));
  return NIQ_OK;
}

// Variants (niq_eval_cfg.variant): 0 and 1 the default (RowsCfg chunk, the
// RowsOcc register budget); 2 half the rows per chunk (fewer registers, more
// barriers); 3 at widths up to 128 a two-waves-per-SIMD budget (no spills,
// half the resident workgroups; the wider templates already run at one or
// two).  Every variant sums in the same order: identical results.
template <int MODE>
niq_status launch_rows(const niq_model* m, const niq_eval_cfg* cfg, const ClassifyArgs& a, long long max_n,
                       hipStream_t s) {
  const int variant = cfg ? cfg->variant : 0;
  if (variant == 2) {
    switch (m->wt) {
      case 32: case 64: return launch_rows_w<64, MODE, RowsOcc<64>::value, RowsCfg<64>::CH / 2>(m, cfg, a, max_n, s);
      case 128: return launch_rows_w<128, MODE, RowsOcc<128>::value, RowsCfg<128>::CH / 2>(m, cfg, a, max_n, s);
      case 256: return launch_rows_w<256, MODE, RowsOcc<256>::value, RowsCfg<256>::CH / 2>(m, cfg, a, max_n, s);
      case 512: return launch_rows_w<512, MODE, RowsOcc<512>::value, RowsCfg<512>::CH / 2>(m, cfg, a, max_n, s);
    }
    return fail(NIQ_ERR_UNSUPPORTED, "width");
  }
  if (variant == 3) {
    switch (m->wt) {
      case 32: case 64: return launch_rows_w<64, MODE, 2>(m, cfg, a, max_n, s);
      case 128: return launch_rows_w<128, MODE, 2>(m, cfg, a, max_n, s);
    }
  }
  switch (m->wt) {
    case 32: case 64: return launch_rows_w<64, MODE>(m, cfg, a, max_n, s);
    case 128: return launch_rows_w<128, MODE>(m, cfg, a, max_n, s);
    case 256: return launch_rows_w<256, MODE>(m, cfg, a, max_n, s);
    case 512: return launch_rows_w<512, MODE>(m, cfg, a, max_n, s);
  }
  return fail(NIQ_ERR_UNSUPPORTED, "width");
}

}  // namespace

niq_status niqi::classify_rows(const niq_model* m, const niq_eval_cfg* cfg, const ClassifyArgs& a,
                               long long max_n, hipStream_t s) {
  const int mode = cfg ? cfg->mode : NIQ_MODE_AFFINE_FIXED;
  if (mode == NIQ_MODE_AFFINE_ALL) return launch_rows<ROWS_ALL>(m, cfg, a, max_n, s);
  if (mode == NIQ_MODE_AFFINE_TRUNCATE) {
    if (!cfg || cfg->truncate_count < 1 || cfg->truncate_count > 64)
      return fail(NIQ_ERR_INVALID, "affine_truncate needs 1 <= truncate_count <= 64");
    return launch_rows<ROWS_TRUNCATE>(m, cfg, a, max_n, s);
  }
  if (!cfg || cfg->n_append < 0 || cfg->n_append > 512)
    return fail(NIQ_ERR_INVALID, "affine_append needs 0 <= n_append <= 512");
  return launch_rows<ROWS_APPEND>(m, cfg, a, max_n, s);
}

namespace niqi {
template <int W>
static void rows_shape_w(int variant, int* ch, int* nw, int* occ) {
  *ch = variant == 2 ? RowsCfg<W>::CH / 2 : RowsCfg<W>::CH;
  *nw = RowsCfg<W>::NW;
  *occ = (variant == 3 && W <= 128) ? 2 : RowsOcc<W>::value;
}

niq_status rows_tile_shape(int variant, int wt, int* ch, int* nw, int* occ) {
  if (variant < 0 || variant > 4) return fail(NIQ_ERR_INVALID, "unknown variant");   // 4 runs the default
  switch (wt) {
    case 32: case 64: rows_shape_w<64>(variant, ch, nw, occ); return NIQ_OK;
    case 128: rows_shape_w<128>(variant, ch, nw, occ); return NIQ_OK;
    case 256: rows_shape_w<256>(variant, ch, nw, occ); return NIQ_OK;
    case 512: rows_shape_w<512>(variant, ch, nw, occ); return NIQ_OK;
  }
  return fail(NIQ_ERR_UNSUPPORTED, "width");
}
}  // namespace niqi
