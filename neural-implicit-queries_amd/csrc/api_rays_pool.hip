// Casts of one function each by the pooled ray caster (niq_rays.h).
#include "niq_internal.h"
#include "niq_rays.h"

namespace {

template <int KIND, int V, int W, int VAR, int AS>
niq_status launch_pool_w(const DevModel* models, const RayArgs& a, long long n_rays, bool loose,
                         bool* launched, hipStream_t s) {
  constexpr int NB = RayTile<W, VAR>::NB, NW = RayTile<W, VAR>::NW;
  constexpr int R = Planes<KIND, V, 1>::R;
  constexpr int LDSOCC = LdsOcc<R, NB, NW, W>::value;
  constexpr int OCC = RayTile<W, VAR>::OCC ? std::min(RayTile<W, VAR>::OCC, LDSOCC) : LDSOCC;
  static_assert(R * NB * W * 4 + sizeof(RayPool) + 4 * (3 * NB + 1) <= kLdsLimit, "LDS");
  auto k = k_cast_rays_pool<KIND, V, NB, NW, W, OCC, AS>;
  // Few rays are spread over as many workgroups as there are, down to the NB/2
  // whose tests fit into the pass of their bounds.  Where work and not latency is the
  // bound (widths >= 64), one workgroup a compute unit (two at width 64) takes them
  // until all resident ones would have their columns full: 5,000 rays of a 256x6 ReLU
  // net take 0.78 of k_cast_rays' time, 1.43 on twice the workgroups, half filled;
  // 14,000 of a 64x8 ELU net 0.93 against 1.25.
  const long long tiles = (n_rays + NB / 2 - 1) / (NB / 2), units = num_cus();
  const long long persist = persistent_blocks(k, NW * 64);
  long long g = grid_for(tiles, persist);
  if (W >= 64 && n_rays <= persist * NB) g = std::min(g, W >= 128 ? units : 2 * units);
  const long long per = (n_rays + g - 1) / g;
  // Width 512, every column taken by one ray: a second pass for the tests costs more than
  // the fifth plane (4,096 rays of a 512x8 net: 307 ms on k_cast_rays, 319 here).
  // Nets that need most tests: only while those fit beside the bounds on one workgroup
  // a unit (width 32: 8,192 rays 0.8 to 0.9 of k_cast_rays' time, 14,000 1.05 to 1.2).
  if (W == 512) *launched = !(per > NB * 3 / 4 && per <= NB);
  if (loose) *launched = n_rays <= units * (W == 32 ? 2 * NB : NB / 2);
  if (!*launched) return NIQ_OK;
  // Rays held at once.  Wide nets (a compute unit's few workgroups are bound by
  // the matrix cores): all a pool takes, so that no ray starts late (25,600 rays of
  // a 256x6 net: 241 ms with 50 rays held, 280 with 25).  Narrow nets (many
  // workgroups, bound by latency): half as many again as columns, so that those
  // whose rays end early take more (160,000 rays of a 32x8 net: 13.9 ms with 24
  // rays held, 16.5 with 48), in equal rounds.
  constexpr long long unit = NB + NB / 2;
  const long long rounds = W >= 256 ? 1 : std::max<long long>(1, (per + unit / 2) / unit);
  const int cap = (int)std::min<long long>(std::max<long long>((per + rounds - 1) / rounds, NB / 2), kRayPool);
  hipLaunchKernelGGL(k, dim3((unsigned)g), dim3(NW * 64), 0, s, models, a, cap);
  HIPCHK(hipGetLastError());
  return NIQ_OK;
}

template <int KIND, int V, int VAR, int AS = ACTS_ALL>
niq_status launch_pool_v(int wt, const DevModel* models, const RayArgs& a, long long n_rays, bool loose,
                         bool* launched, hipStream_t s) {
  switch (wt) {
    case 32: return launch_pool_w<KIND, V, 32, VAR, AS>(models, a, n_rays, loose, launched, s);
    case 64: return launch_pool_w<KIND, V, 64, VAR, AS>(models, a, n_rays, loose, launched, s);
    case 128: return launch_pool_w<KIND, V, 128, VAR, AS>(models, a, n_rays, loose, launched, s);
    case 256: return launch_pool_w<KIND, V, 256, VAR, AS>(models, a, n_rays, loose, launched, s);
    case 512: return launch_pool_w<KIND, V, 512, VAR, AS>(models, a, n_rays, loose, launched, s);
  }
  return fail(NIQ_ERR_UNSUPPORTED, "width");
}

// acts: the one activation of every model of the cast, or ACTS_ALL; the default
// affine_fixed tile then runs the kernel compiled for it alone (bit-identical,
// fewer registers).
template <int KIND, int V>
niq_status launch_pool(int wt, int variant, int acts, const DevModel* models, const RayArgs& a, long long n_rays,
                       bool loose, bool* launched, hipStream_t s) {
  if constexpr (KIND == 0 && V == 1) {
    if (variant == 0) {
      switch (acts) {
        case ACTS_RELU: return launch_pool_v<KIND, V, 0, ACTS_RELU>(wt, models, a, n_rays, loose, launched, s);
        case ACTS_TANH: return launch_pool_v<KIND, V, 0, ACTS_TANH>(wt, models, a, n_rays, loose, launched, s);
        case ACTS_ELU: return launch_pool_v<KIND, V, 0, ACTS_ELU>(wt, models, a, n_rays, loose, launched, s);
      }
    }
  }
  switch (variant) {
    case 0: return launch_pool_v<KIND, V, 0>(wt, models, a, n_rays, loose, launched, s);
    case 1: return launch_pool_v<KIND, V, 1>(wt, models, a, n_rays, loose, launched, s);
    case 2: return launch_pool_v<KIND, V, 2>(wt, models, a, n_rays, loose, launched, s);
  }
  return fail(NIQ_ERR_INVALID, "ray_variant must be 0, 1 or 2");
}

}  // namespace

namespace niqi {

niq_status cast_pool(int mode, int wt, int variant, int acts, const DevModel* models, const RayArgs& a,
                     long long n_rays, bool loose, bool* launched, hipStream_t s) {
  switch (mode) {
    case NIQ_MODE_AFFINE_FIXED: return launch_pool<0, 1>(wt, variant, acts, models, a, n_rays, loose, launched, s);
    case NIQ_MODE_INTERVAL: return launch_pool<0, 0>(wt, variant, acts, models, a, n_rays, loose, launched, s);
    case NIQ_MODE_SLOPE_INTERVAL: return launch_pool<1, 1>(wt, variant, acts, models, a, n_rays, loose, launched, s);
  }
  return fail(NIQ_ERR_INVALID, "no range form in this mode");
}

}  // namespace niqi
