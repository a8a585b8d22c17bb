#pragma once
// Frustum ray casting (src/queries.py:178-587): image tiles march forward as
// general boxes (the frustum's step segment: its centre ray and two side
// vectors), split in two along the wider index axis when they grow too wide
// for their step or demand it, and stop when a single-pixel frustum hits, the
// frustum passes max_dist or the iteration budget runs out.  Each frustum
// evolves from its own state only, so the live frusta are kept in a compact
// list (any order); the classify and point passes are the fused kernels.
#include "niq_kernels.h"

struct FrustCam {
  float root[3], look[3], up[3], left[3];
  float tan_x, tan_y;         // tan(deg2rad(fov) / 2), float32
  float half_fov_x, half_fov_y;  // deg2rad(fov) / 2, float32
  int res_x, res_y;
};

struct FrustParams {
  float hit_eps, max_dist, safety, grow, shrink, refine;
  int n_models;
};

// A list of frusta: pixel ranges [x0, y0, x1, y1) and their march state.
struct FrustList {
  int4* rng;
  float* t;
  float* step;
  float* cnt;
};

// Counts of one iteration: `next` holds the entries written to the next list
// (survivors and B halves) in its low word and the survivors that split in its
// high word, so that one atomic claims both.
struct FrustCount {
  unsigned long long next;
};

// Per-frustum geometry of one iteration (src/queries.py:275-308), the boxes and
// points of a substep and the state between substeps; all arrays have one entry
// per live frustum.
struct FrustWork {
  float* geo;     // 14 floats: r_uu, r_lu, r_ul (9), mid (3), expand, single
  float* center;  // (n, 3) general-box centres
  float* vecs;    // (n, 3, 3) general-box vectors
  float* pts;     // (2n, 3) hit-test points
  int* codes;     // (n_models, cap) sign codes
  float* vals;    // (n_models, 2 cap) point values
  int4* state;    // hit, hit id, demands a split, substeps counted
};

__device__ __forceinline__ void frust_cam_ray(const FrustCam& c, float tx, float ty, float* r) {
  float p[3];
#pragma unroll
  for (int k = 0; k < 3; ++k) p[k] = c.look[k] + c.left[k] * (tx * c.tan_x) + c.up[k] * (ty * c.tan_y);
  const float nrm = sqrtf(p[0] * p[0] + p[1] * p[1] + p[2] * p[2]);
#pragma unroll
  for (int k = 0; k < 3; ++k) r[k] = p[k] / nrm;
}

// Geometry of an iteration (src/queries.py:275-308) and the first substep's
// segment as a general box with its two points, for list entry i.
__device__ __forceinline__ void frust_prep(const FrustCam& c, const FrustParams& P, const FrustWork& W,
                                           const float* g, float t, float step, size_t i) {
  const float t_adj = (t + step) * g[12];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float mid = g[9 + k];
    W.center[3 * i + k] = c.root[k] + 0.5f * (t + t_adj) * mid;
    W.vecs[9 * i + k] = 0.5f * (t_adj - t) * mid;
    W.vecs[9 * i + 3 + k] = (g[k] - g[3 + k]) * t_adj / 2.f;
    W.vecs[9 * i + 6 + k] = (g[k] - g[6 + k]) * t_adj / 2.f;
    W.pts[6 * i + k] = c.root[k] + t * mid;
    W.pts[6 * i + 3 + k] = c.root[k] + (t + P.hit_eps) * mid;
  }
}

__device__ __forceinline__ void frust_begin(const FrustCam& c, const FrustParams& P, const FrustWork& W,
                                            const int4& r, float t, float step, size_t i) {
  const float rx1 = (float)c.res_x + 1.f, ry1 = (float)c.res_y + 1.f;
  const float xlo = 2.f * (float)r.x / rx1 - 1.f, xhi = 2.f * (float)(r.z - 1) / rx1 - 1.f;
  const float ylo = 2.f * (float)r.y / ry1 - 1.f, yhi = 2.f * (float)(r.w - 1) / ry1 - 1.f;
  float uu[3], lu[3], ul[3], ll[3];
  frust_cam_ray(c, xhi, yhi, uu);
  frust_cam_ray(c, xlo, yhi, lu);
  frust_cam_ray(c, xhi, ylo, ul);
  frust_cam_ray(c, xlo, ylo, ll);
  float mid[3], g[14];
#pragma unroll
  for (int k = 0; k < 3; ++k) mid[k] = 0.5f * (uu[k] + ll[k]);
  const float len = sqrtf(mid[0] * mid[0] + mid[1] * mid[1] + mid[2] * mid[2]);
#pragma unroll
  for (int k = 0; k < 3; ++k) { g[k] = uu[k]; g[3 + k] = lu[k]; g[6 + k] = ul[k]; g[9 + k] = mid[k] / len; }
  g[12] = 1.f / len;
  g[13] = (r.x + 1 == r.z && r.y + 1 == r.w) ? 1.f : 0.f;
#pragma unroll
  for (int k = 0; k < 14; ++k) W.geo[14 * i + k] = g[k];
  frust_prep(c, P, W, g, t, step, i);
}

static __global__ void k_frust_init(FrustCam c, FrustParams P, FrustList L, FrustWork W, int n_side, const int* xt,
                                    const int* yt, float init_step) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_side * n_side) return;
  const int a = i % n_side, b = i / n_side;   // tile(x ticks), repeat(y ticks)
  const int4 r = make_int4(xt[a], yt[b], xt[a + 1], yt[b + 1]);
  L.rng[i] = r;
  L.t[i] = 0.f;
  L.step[i] = init_step;
  L.cnt[i] = 0.f;
  frust_begin(c, P, W, r, 0.f, init_step, i);
}

// Before a group of iterations: the live count moves to the first entry, the
// others are cleared.
static __global__ void k_frust_counts(FrustCount* counts, int from, long long n0, int n_entries) {
  const unsigned long long live = n0 >= 0 ? (unsigned long long)n0 : (counts[from].next & 0xffffffffull);
  __syncthreads();
  if (threadIdx.x == 0) counts[0].next = live;
  for (int i = 1 + threadIdx.x; i < n_entries; i += blockDim.x) counts[i].next = 0ull;
}

// End of a substep (src/queries.py:214-269) after every function's passes, for
// list entry i: advances t and step, updates the state {hit, hit id, demands,
// substeps}.
__device__ __forceinline__ void frust_sub(const FrustParams& P, const FrustWork& W, float single, size_t i, int cap,
                                          float& t, float& step, int4& st) {
  int can = !st.x;
  st.w += st.x ? 0 : 1;
  int hit = st.x, hid = st.y;
  for (int f = 0; f < P.n_models; ++f) {
    const int code = W.codes[(size_t)f * cap + i];
    can = can && (code == CODE_POSITIVE || code == CODE_NEGATIVE);
    const float v0 = W.vals[(size_t)f * 2 * cap + 2 * i];
    const float v1 = W.vals[(size_t)f * 2 * cap + 2 * i + 1];
    const bool this_hit = sign_f(v0) != sign_f(v1);
    if (this_hit) hid = f + 1;
    hit = hit || this_hit;
  }
  const float this_step = can ? step : P.hit_eps * single;
  if (!hit) t = t + this_step * P.safety;
  step = can ? step * P.grow : step * P.shrink;
  st.z = st.z || (step < P.hit_eps) || hit;
  step = fmaxf(step, P.hit_eps);
  st.x = hit; st.y = hid;
}

// Between two substeps of one iteration.
static __global__ void k_frust_sub(FrustCam c, FrustParams P, FrustList L, FrustWork W, const FrustCount* live,
                                   int cap, int first) {
  const int n = (int)(live->next & 0xffffffffull);
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float* g = W.geo + 14 * (size_t)i;
    float t = L.t[i], step = L.step[i];
    int4 st = first ? make_int4(0, 0, 0, 0) : W.state[i];
    frust_sub(P, W, g[13], i, cap, t, step, st);
    L.t[i] = t; L.step[i] = step;
    W.state[i] = st;
    frust_prep(c, P, W, g, t, step, i);
  }
}

// End of an iteration (src/queries.py:321-362, 384-425): the last substep, then
// counts, termination, refinement and the split; survivors and B halves go to
// the next list with the geometry of their next iteration.  One kernel in place
// of four; places are claimed per workgroup (one atomic for the next list, one
// for the finished), where one per thread took 22 us of a 768 x 768 image's
// iteration.
constexpr int kFrustBlock = 256;
static __global__ void __launch_bounds__(kFrustBlock)
k_frust_step(FrustCam c, FrustParams P, FrustList L, FrustWork W, FrustCount* counts, int cap, int first,
             int count_term, FrustList N, FrustWork WN, FrustList F, int* fin_hit, int* n_fin) {
  constexpr int NWV = kFrustBlock / 64;
  __shared__ int s_cnt[3][NWV];
  __shared__ int s_base[2];
  const int n = (int)(counts[0].next & 0xffffffffull);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  for (long long i0 = (long long)blockIdx.x * kFrustBlock; i0 < n; i0 += (long long)gridDim.x * kFrustBlock) {
    const size_t i = (size_t)i0 + threadIdx.x;
    const bool in = i < (size_t)n;
    int4 r = make_int4(0, 0, 1, 1), st = make_int4(0, 0, 0, 0);
    float t = 0.f, step = 0.f, cnt = 0.f;
    bool term = false, needs = false;
    if (in) {
      r = L.rng[i];
      t = L.t[i]; step = L.step[i];
      if (!first) st = W.state[i];
      frust_sub(P, W, W.geo[14 * i + 13], i, cap, t, step, st);
      const int area = (r.z - r.x) * (r.w - r.y);
      cnt = L.cnt[i] + (float)st.w * (1.f / (float)area);
      const bool hit = st.x && area == 1;
      term = hit || (t > P.max_dist) || count_term;
      if (!term) {
        const float wx = 2.f * sinf(c.half_fov_x * (float)(r.z - r.x) / (float)c.res_x) * t;
        const float wy = 2.f * sinf(c.half_fov_y * (float)(r.w - r.y) / (float)c.res_y) * t;
        const bool can_subd = (r.z > r.x + 1) || (r.w > r.y + 1);
        needs = ((wx > P.refine * step) || (wy > P.refine * step) || st.z) && can_subd;
      }
    }
    const bool live = in && !term;
    const unsigned long long mf = __ballot(in && term), ml = __ballot(live), mr = __ballot(needs);
    if (lane == 0) { s_cnt[0][wave] = __popcll(mf); s_cnt[1][wave] = __popcll(ml); s_cnt[2][wave] = __popcll(mr); }
    __syncthreads();
    if (threadIdx.x == 0) {
      int nf = 0, nl = 0, nr = 0;
#pragma unroll
      for (int w = 0; w < NWV; ++w) { nf += s_cnt[0][w]; nl += s_cnt[1][w]; nr += s_cnt[2][w]; }
      s_base[0] = nf ? atomicAdd(n_fin, nf) : 0;
      s_base[1] = nl ? (int)(atomicAdd(&counts[1].next, ((unsigned long long)nr << 32) | (unsigned)(nl + nr)) &
                             0xffffffffull)
                     : 0;
    }
    __syncthreads();
    int kf = s_base[0] + __popcll(mf & below), kn = s_base[1] + __popcll(ml & below) + __popcll(mr & below);
#pragma unroll
    for (int w = 0; w < NWV; ++w)
      if (w < wave) { kf += s_cnt[0][w]; kn += s_cnt[1][w] + s_cnt[2][w]; }
    if (in && term) {
      F.rng[kf] = r; F.t[kf] = t; F.cnt[kf] = cnt;
      fin_hit[kf] = st.y;
    } else if (live) {
      const bool sx = (r.z - r.x) >= (r.w - r.y);
      const int xm = (r.x + r.z) / 2, ym = (r.y + r.w) / 2;
      const int4 A = make_int4(r.x, r.y, sx ? xm : r.z, sx ? r.w : ym);
      const int4 B = make_int4(sx ? xm : r.x, sx ? r.y : ym, r.z, r.w);
      for (int h = 0; h <= (needs ? 1 : 0); ++h) {
        const int4 q = needs ? (h ? B : A) : r;
        const size_t k = (size_t)kn + h;
        N.rng[k] = q; N.t[k] = t; N.step[k] = step; N.cnt[k] = cnt;
        frust_begin(c, P, WN, q, t, step, k);
      }
    }
    __syncthreads();   // s_cnt and s_base are rewritten by the next chunk
  }
}

// Every finished frustum covers its pixels (src/queries.py:571-585); outputs
// are indexed [x, y].
static __global__ void k_frust_write(FrustList F, const int* fin_hit, int n_fin, int res_y, float* out_t,
                                     int* out_hit, int* out_count) {
  for (int i = blockIdx.x; i < n_fin; i += gridDim.x) {
    const int4 r = F.rng[i];
    const int w = r.w - r.y;
    const int np = (r.z - r.x) * w;
    const float t = F.t[i];
    const int h = fin_hit[i];
    const int cn = (int)F.cnt[i];
    for (int p = threadIdx.x; p < np; p += blockDim.x) {
      const size_t o = (size_t)(r.x + p / w) * res_y + (r.y + p % w);
      out_t[o] = t; out_hit[o] = h; out_count[o] = cn;
    }
  }
}

// One iteration's evaluations of one function in one launch, for 32-wide nets:
// workgroups [0, g_box) stride over the live frusta's segments, 16 a tile of two
// waves (one a feature tile), as k_classify; the others over their 2n hit-test points,
// 16 a tile of one wave, as k_points_dev.  Every (box, feature) and (point, feature)
// sums in the order of those kernels.  An iteration has one or two tiles a SIMD,
// so it is bound by a tile's latency: the points run beside the boxes instead of
// after them, and a box tile's work is halved per wave.  Fox at 768^2, an
// iteration's evaluations: 55 + 20 -> 51 us and a launch less, the image 27.1 -> 23.6
// ms; at 200^2 12.0 -> 9.1 ms.
template <int V, int AS>
__global__ void __launch_bounds__(128, (LdsOcc<Planes<0, V, 0>::R, 16, 2, 32>::value))
k_frust_forward(const DevModel* __restrict__ Mp, ClassifyArgs a, const float* __restrict__ pts,
                float* __restrict__ vals, int g_box) {
  using PB = Planes<0, V, 0>;
  using PP = Planes<2, 0, 1>;
  constexpr int NB = 16, W = 32;
  static_assert(PB::R >= 2, "two point tiles fit beside each other in X");
  __shared__ float X[PB::R * NB * W];
  const long long n = *a.n_dev;
  if ((int)blockIdx.x < g_box) {
    const long long ntiles = (n + NB - 1) / NB;
    for (long long tile = blockIdx.x; tile < ntiles; tile += g_box) {
      const long long i0 = tile * NB;
      fill_box_inputs<0, V, NB, 128, W>(X, a, i0, n);
      mlp_forward<PB, 0, V, NB, 2, W, AS>(*Mp, X, [&](const float* v, int b) {
        const long long i = i0 + b;
        if (i >= n) return;
        float lo, hi, scale;
        final_bounds<0, V>(v, lo, hi, scale);
        a.codes[i] = sign_code(lo, hi, a.offset);
      });
    }
  } else {
    const int sub = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    float* Xp = X + sub * (NB * W);
    const long long np = 2 * n, ntiles = (np + NB - 1) / NB;
    for (long long tile = (long long)(blockIdx.x - g_box) * 2 + sub; tile < ntiles; tile += 2LL * (gridDim.x - g_box)) {
      const long long p0 = tile * NB;
#pragma unroll
      for (int e = lane; e < NB * 16; e += 64) {
        const int b = e >> 4, k = e & 15;
        Xp[xoff<NB, W>(0, b, k)] = (p0 + b < np && k < 3) ? pts[(p0 + b) * 3 + k] : 0.f;
      }
      mlp_forward<PP, 2, 0, NB, 1, W, AS>(*Mp, Xp, [&](const float* v, int b) {
        if (p0 + b < np) vals[p0 + b] = v[0];
      });
    }
  }
}
