// Sign codes of wide ReLU nets by the split contraction (niq_split.h).
#include "niq_internal.h"
#include "niq_split.h"

namespace {

template <int W>
niq_status launch_split_w(const niq_model* m, const ClassifyArgs& a, long long max_n, hipStream_t s) {
  constexpr int NB = SplitTile<W>::NB, NW = SplitTile<W>::NW;
  auto k = k_classify_split<3, NB, NW, W, ACTS_RELU>;
  const long long tiles = (max_n + NB - 1) / NB;
  if (tiles == 0) return NIQ_OK;
  hipLaunchKernelGGL(k, dim3(tile_grid(tiles, persistent_blocks(k, NW * 64))), dim3(NW * 64), 0, s, m->dev16, a);
  HIPCHK(hipGetLastError());
  // the listed boxes (few: one resident round of workgroups strides over them)
  constexpr int NBL = BoxTile<W>::NB, NWL = BoxTile<W>::NW;
  auto kl = k_classify<0, 3, NBL, NWL, W, false, 0, ACTS_RELU, 1, true>;
  const long long ltiles = (max_n + NBL - 1) / NBL;
  hipLaunchKernelGGL(kl, dim3(grid_for(ltiles, persistent_blocks(kl, NWL * 64))), dim3(NWL * 64), 0, s, m->dev, a);
  HIPCHK(hipGetLastError());
  return NIQ_OK;
}

// 64 points a workgroup: 4 point tiles share a wave's weight fragments.
template <int W, int AS>
niq_status launch_points_split_w(const niq_model* m, const float* x, int d, long long n, float* out, hipStream_t s) {
  constexpr int NB = 64, NW = SplitTile<W>::NW;
  auto k = k_points_split<NB, NW, W, AS>;
  const long long tiles = (n + NB - 1) / NB;
  if (tiles == 0) return NIQ_OK;
  hipLaunchKernelGGL(k, dim3(grid_for(tiles, persistent_blocks(k, NW * 64))), dim3(NW * 64), 0, s, m->dev16, m->dev,
                     x, d, n, out);
  HIPCHK(hipGetLastError());
  return NIQ_OK;
}

template <int W>
niq_status launch_points_split(const niq_model* m, const float* x, int d, long long n, float* out, hipStream_t s) {
  if (m->relu_only) return launch_points_split_w<W, ACTS_RELU>(m, x, d, n, out, s);
  return launch_points_split_w<W, ACTS_ALL>(m, x, d, n, out, s);
}

// Every hidden layer fills the template width, the widths where the contraction
// is the cost.
bool split_shape(const niq_model* m) {
  for (int i = 1; i < m->n_layers; ++i)
    if (round32(m->dims[i]) != m->wt) return false;
  return m->n_layers > 1 && m->bf16_ok && m->bounded && m->wt >= 256 && m->wt16 == m->wt;
}

}  // namespace

bool niqi::points_split_eligible(const niq_model* m) { return split_shape(m); }

niq_status niqi::points_split(const niq_model* m, const float* x, int d, long long n, float* out, hipStream_t s) {
  switch (m->wt) {
    case 256: return launch_points_split<256>(m, x, d, n, out, s);
    case 512: return launch_points_split<512>(m, x, d, n, out, s);
  }
  return fail(NIQ_ERR_UNSUPPORTED, "width");
}

// Widths 256 and 512, where the contraction is the cost (131,072 boxes of the
// 256x6 net 3.46 ms by FP32 matrix instructions, 2.07 split; of the 512x8 net
// 18.5 and 10.9 ms; narrower nets are bound by their rules).  ReLU alone: the
// TanH rule amplifies rounding too far for a band (4 % of the bound at
// half-width 1/1000).
bool niqi::split_eligible(const niq_model* m, const niq_eval_cfg* cfg) {
  if (cfg && (cfg->mode != NIQ_MODE_AFFINE_FIXED || cfg->precision != NIQ_PREC_FP32 || cfg->recheck_tol > 0.f ||
              cfg->variant > 1))
    return false;
  return split_shape(m) && m->relu_only && m->in_dim == 3 && std::isfinite(m->round_rel);
}

float niqi::split_min_half(const niq_model* m) { return m->round_rel / kSplitRound; }

niq_status niqi::classify_split(const niq_model* m, ClassifyArgs a, long long max_n, hipStream_t s) {
  a.min_half = split_min_half(m);
  a.noise = kNoiseRoom * m->round_out;
  switch (m->wt) {
    case 256: return launch_split_w<256>(m, a, max_n, s);
    case 512: return launch_split_w<512>(m, a, max_n, s);
  }
  return fail(NIQ_ERR_UNSUPPORTED, "width");
}
