// Frustum ray casting entry point (src/queries.py:454-587).
#include "niq_internal.h"
#include "niq_frustum.h"

namespace {

long long next_bucket_size(long long s) {
  for (int e = 7; e <= 30; ++e)
    if (s <= (1LL << e)) return 1LL << e;
  return -1;
}

// est: the frusta to size the launch for (it strides over the live count).
template <int V, int AS>
niq_status launch_frust_forward(const niq_model* m, const ClassifyArgs& a, const float* pts, float* vals, long long est,
                                hipStream_t s) {
  auto k = k_frust_forward<V, AS>;
  const long long cap = persistent_blocks(k, 128) * kTileGridMult;
  const int g_box = (int)std::max<long long>(1, std::min((est + 15) / 16, cap));
  const int g_pts = (int)std::max<long long>(1, std::min((2 * est + 31) / 32, cap));
  hipLaunchKernelGGL(k, dim3(g_box + g_pts), dim3(128), 0, s, m->dev, a, pts, vals, g_box);
  HIPCHK(hipGetLastError());
  return NIQ_OK;
}

}  // namespace

extern "C" niq_status niq_cast_rays_frustum(const niq_model* const* models, int n_models, const niq_eval_cfg* cfg,
                                            const niq_frustum_cam* cam, const niq_frustum_opts* fo, float* out_t,
                                            int32_t* out_hit_id, int32_t* out_count, int64_t* n_evals,
                                            void* stream) {
  if (!models || n_models < 1 || n_models > 8) return fail(NIQ_ERR_INVALID, "need 1..8 models");
  if (!cam || !fo) return fail(NIQ_ERR_INVALID, "null camera or options");
  const niq_cast_opts& o = fo->cast;
  if (o.n_substeps < 1 || o.n_max_step < 1) return fail(NIQ_ERR_INVALID, "n_substeps and n_max_step must be >= 1");
  const int rx = cam->res_x, ry = cam->res_y, ns = fo->n_side_init;
  if (rx < 1 || ry < 1 || (long long)rx * ry > (1LL << 28)) return fail(NIQ_ERR_INVALID, "resolution out of range");
  if (ns < 1 || ns > rx || ns > ry) return fail(NIQ_ERR_INVALID, "n_side_init must be in [1, min(res_x, res_y)]");
  if (!out_t || !out_hit_id || !out_count) return fail(NIQ_ERR_INVALID, "bad buffers");
  for (int i = 0; i < n_models; ++i)
    if (niq_status st = check_model(models[i], 3)) return st;
  const int mode = cfg ? cfg->mode : NIQ_MODE_AFFINE_FIXED;
  if (cfg && cfg->precision == NIQ_PREC_BF16 &&
      (mode == NIQ_MODE_AFFINE_ALL || mode == NIQ_MODE_AFFINE_TRUNCATE || mode == NIQ_MODE_AFFINE_APPEND))
    return fail(NIQ_ERR_UNSUPPORTED, "the precision mode runs interval and affine_fixed");
  hipStream_t s = (hipStream_t)stream;
  const long long cap = (long long)rx * ry;   // frusta partition the image

  FrustCam c{};
  for (int k = 0; k < 3; ++k) {
    c.root[k] = cam->root[k]; c.look[k] = cam->look[k]; c.up[k] = cam->up[k]; c.left[k] = cam->left[k];
  }
  // tan(deg2rad(fov) / 2) and deg2rad(fov) / 2 in float32, as the reference forms them
  const float d2r = (float)(3.14159265358979323846 / 180.0);
  const float hx = (cam->fov_x * d2r) / 2.f;
  const float hy = (cam->fov_y * d2r) / 2.f;
  c.half_fov_x = hx; c.half_fov_y = hy;
  c.tan_x = std::tan(hx); c.tan_y = std::tan(hy);
  c.res_x = rx; c.res_y = ry;
  FrustParams P{};
  P.hit_eps = o.hit_eps; P.max_dist = o.max_dist; P.safety = o.safety_factor;
  P.grow = o.interval_grow_fac; P.shrink = o.interval_shrink_fac; P.refine = fo->refine_width_fac;
  P.n_models = n_models;

  // device scratch (stream ordered)
  std::vector<void*> allocs;
  niq_status st = NIQ_OK;
  auto al = [&](size_t bytes) -> void* {
    void* p = nullptr;
    if (st == NIQ_OK && hipMallocAsync(&p, (bytes + 255) / 256 * 256, s) != hipSuccess)
      st = fail(NIQ_ERR_HIP, "frustum scratch allocation failed");
    if (p) allocs.push_back(p);
    return p;
  };
  auto mk_list = [&](FrustList& L) {
    L.rng = static_cast<int4*>(al(sizeof(int4) * cap));
    L.t = static_cast<float*>(al(sizeof(float) * cap));
    L.step = static_cast<float*>(al(sizeof(float) * cap));
    L.cnt = static_cast<float*>(al(sizeof(float) * cap));
  };
  FrustList Ls[2], F;
  mk_list(Ls[0]); mk_list(Ls[1]); mk_list(F);
  int* fin_hit = static_cast<int*>(al(sizeof(int) * cap));
  FrustWork Ws[2];   // each iteration writes the next one's (in another order)
  int* codes = static_cast<int*>(al(sizeof(int) * cap * n_models));
  float* vals = static_cast<float*>(al(sizeof(float) * 2 * cap * n_models));
  int4* state = o.n_substeps > 1 ? static_cast<int4*>(al(sizeof(int4) * cap)) : nullptr;
  for (FrustWork& W : Ws) {
    W = FrustWork{};
    W.geo = static_cast<float*>(al(sizeof(float) * 14 * cap));
    W.center = static_cast<float*>(al(sizeof(float) * 3 * cap));
    W.vecs = static_cast<float*>(al(sizeof(float) * 9 * cap));
    W.pts = static_cast<float*>(al(sizeof(float) * 6 * cap));
    W.codes = codes; W.vals = vals; W.state = state;
  }
  // counts[j]: the live frusta of iteration j of a group, then the finished
  constexpr int kGroup = 8;
  FrustCount* counts = static_cast<FrustCount*>(al(sizeof(FrustCount) * (kGroup + 2)));
  int* n_fin = reinterpret_cast<int*>(counts + kGroup + 1);
  int* ticks = static_cast<int*>(al(sizeof(int) * 2 * (ns + 1)));

  // initial tiles: linspace(0, res, n_side + 1) truncated (src/queries.py:497-505)
  std::vector<int> ht(2 * (ns + 1));
  for (int i = 0; i <= ns; ++i) {
    ht[i] = (int)((double)rx * i / ns);
    ht[ns + 1 + i] = (int)((double)ry * i / ns);
  }
  const int n0 = ns * ns;
  long long n = n0, bucket = n0, empty = n0, evals = 0;
  int it = 0, cur = 0;
  if (st == NIQ_OK && (hipMemcpyAsync(ticks, ht.data(), sizeof(int) * ht.size(), hipMemcpyHostToDevice, s) != hipSuccess ||
                       hipMemsetAsync(n_fin, 0, sizeof(int), s) != hipSuccess))
    st = fail(NIQ_ERR_HIP, "frustum set-up failed");
  if (st == NIQ_OK)
    hipLaunchKernelGGL(k_frust_init, dim3((n0 + 255) / 256), dim3(256), 0, s, c, P, Ls[0], Ws[0], ns, ticks,
                       ticks + ns + 1, o.init_step);
  // Iterations run in groups without a host read between them: the live count
  // stays on the device, and the host reads a group's counts at its end (an
  // iteration past the last finds none live).  A group is short while the
  // count grows, so that launches are not sized for a count long outgrown
  // (sizes only choose tiles and grids: every kernel strides over the device
  // count).  The layer-by-layer precision mode sizes its scratch by max_n and
  // gets a true bound.
  const bool strict = cfg && cfg->precision == NIQ_PREC_BF16 && cfg->variant == 3;
  // 32-wide nets evaluate boxes and points in one launch, unless the caller chose
  // another classify tile
  const bool fused = (!cfg || (cfg->precision == NIQ_PREC_FP32 && cfg->variant == 0)) &&
                     (mode == NIQ_MODE_INTERVAL || mode == NIQ_MODE_AFFINE_FIXED);
  FrustCount h[kGroup + 2];
  int hfin = 0;
  bool done = st != NIQ_OK, growing = true;
  long long start = n;
  int from = 0;
  while (!done) {
    const int K = growing ? 2 : kGroup;
    hipLaunchKernelGGL(k_frust_counts, dim3(1), dim3(64), 0, s, counts, from, start, K + 1);
    start = -1;
    from = K;
    for (int j = 0; j < K && st == NIQ_OK; ++j) {
      const FrustList& L = Ls[cur];
      const FrustWork& W = Ws[cur];
      const long long bound = std::min(cap, n << j);
      const long long est = growing || strict ? bound : std::min(cap, n + n / 4);
      const int* n_live = reinterpret_cast<const int*>(counts + j);   // the low word
      const unsigned g = (unsigned)std::min<long long>((est + 255) / 256, 8192);
      for (int sub = 0; sub < o.n_substeps && st == NIQ_OK; ++sub) {
        for (int f = 0; f < n_models && st == NIQ_OK; ++f) {
          ClassifyArgs a{};
          a.center = W.center; a.vecs = W.vecs; a.vin = 3; a.d = 3; a.n_dev = n_live; a.offset = 0.f;
          a.codes = W.codes + (size_t)f * cap;
          float* fvals = W.vals + (size_t)f * 2 * cap;
          if (fused && models[f]->wt == 32) {
            const niq_model* m = models[f];
            if (mode == NIQ_MODE_INTERVAL)
              st = m->relu_only ? launch_frust_forward<0, ACTS_RELU>(m, a, W.pts, fvals, est, s)
                                : launch_frust_forward<0, ACTS_ALL>(m, a, W.pts, fvals, est, s);
            else
              st = m->relu_only ? launch_frust_forward<3, ACTS_RELU>(m, a, W.pts, fvals, est, s)
                                : launch_frust_forward<3, ACTS_ALL>(m, a, W.pts, fvals, est, s);
            if (st) break;
            continue;
          }
          if ((st = classify_dispatch(models[f], cfg, mode == NIQ_MODE_INTERVAL ? 0 : 3, a, est, s))) break;
          st = points_dev(models[f], W.pts, n_live, 2, 2 * est, fvals, s);
        }
        if (st) break;
        const int first = sub == 0 ? 1 : 0;
        if (sub + 1 < o.n_substeps) {
          hipLaunchKernelGGL(k_frust_sub, dim3(g), dim3(256), 0, s, c, P, L, W, counts + j, (int)cap, first);
        } else {
          hipLaunchKernelGGL(k_frust_step, dim3(g), dim3(kFrustBlock), 0, s, c, P, L, W, counts + j, (int)cap,
                             first, it + j * o.n_substeps >= o.n_max_step ? 1 : 0, Ls[cur ^ 1], Ws[cur ^ 1], F, fin_hit,
                             n_fin);
        }
      }
      cur ^= 1;
    }
    if (st) break;
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(h, counts, sizeof(h), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess) {
      st = fail(NIQ_ERR_HIP, "frustum iteration failed");
      break;
    }
    std::memcpy(&hfin, &h[kGroup + 1], sizeof(int));
    const long long n_before = n;
    for (int j = 1; j <= K && !done; ++j) {
      const long long n_next = (long long)(h[j].next & 0xffffffffull), n_refine = (long long)(h[j].next >> 32);
      const long long n_valid = n_next - n_refine;   // a split adds one entry
      evals += bucket;
      it += o.n_substeps;
      if (n_valid == 0) { done = true; break; }
      // the reference's padded-array bookkeeping, for N_evals (src/queries.py:557-569)
      const long long nb = next_bucket_size(n_valid + n_refine);
      if (empty + n_refine > bucket || nb < bucket) { bucket = nb; empty = n_valid; }
      empty += n_refine;
      n = n_next;
    }
    growing = n > n_before + n_before / 16;
  }
  if (st == NIQ_OK && hfin > 0) {
    hipLaunchKernelGGL(k_frust_write, dim3((unsigned)std::min<long long>(hfin, 65536)), dim3(256), 0, s, F,
                       fin_hit, hfin, ry, out_t, out_hit_id, out_count);
    if (hipGetLastError() != hipSuccess) st = fail(NIQ_ERR_HIP, "frustum output write failed");
  }
  for (void* p : allocs) (void)hipFreeAsync(p, s);
  if (hipStreamSynchronize(s) != hipSuccess && st == NIQ_OK) st = fail(NIQ_ERR_HIP, "frustum stream failed");
  if (st == NIQ_OK && n_evals) *n_evals = evals;
  return st;
}
