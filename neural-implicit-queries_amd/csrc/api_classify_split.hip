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

}  // namespace

// Widths 256 and 512, where the contraction is the cost (131,072 boxes of the
// 256x6 net 3.46 ms by FP32 matrix instructions, 2.07 split; of the 512x8 net
// 18.5 and 10.9 ms; narrower nets are bound by their rules).  ReLU alone: the
// TanH rule amplifies rounding too far for a band (4 % of the bound at
// half-width 1/1000).
bool niqi::split_eligible(const niq_model* m, const niq_eval_cfg* cfg) {
  if (cfg && (cfg->mode != NIQ_MODE_AFFINE_FIXED || cfg->precision != NIQ_PREC_FP32 || cfg->recheck_tol > 0.f ||
              cfg->variant > 1))
    return false;
  for (int i = 1; i < m->n_layers; ++i)
    if (round32(m->dims[i]) != m->wt) return false;   // every feature tile in use
  return m->n_layers > 1 && m->relu_only && m->bias_small && m->bf16_ok && m->in_dim == 3 && m->wt >= 256 && m->wt16 == m->wt;
}

niq_status niqi::classify_split(const niq_model* m, const ClassifyArgs& a, long long max_n, hipStream_t s) {
  switch (m->wt) {
    case 256: return launch_split_w<256>(m, a, max_n, s);
    case 512: return launch_split_w<512>(m, a, max_n, s);
  }
  return fail(NIQ_ERR_UNSUPPORTED, "width");
}
