// The pooled ray caster: one function per cast, forms with a range bound.
#pragma once
#include "niq_kernels.h"

// Rays a workgroup holds (one per lane of its first wave).
constexpr int kRayPool = 64;

// State of the rays a workgroup holds, one column per slot.  In LDS, since only
// the first wave reads it, once a pass: in registers it would be live, in every
// wave, through the network's layers.
struct RayPool {
  float t[kRayPool], step[kRayPool], cov[kRayPool];
  float o[3][kRayPool], d[3][kRayPool];
  int rid[kRayPool], cnt[kRayPool], iters[kRayPool], sub[kRayPool];
  int phase[kRayPool];   // kRayBounds, or the segment's code, its points not yet tested
};
enum { kRayBounds = -1 };
constexpr int kRaySure = 4;   // beside a code: the segment's bound excludes a hit in it

// Slots chosen for a pass, in turn: the rank of lane's bit in `want`, counted from
// lane `rot` round the wave, or -1.
__device__ __forceinline__ int turn_rank(unsigned long long want, int rot, int lane) {
  if (!((want >> lane) & 1ull)) return -1;
  const unsigned long long below = (1ull << lane) - 1ull, before = (1ull << rot) - 1ull;
  return lane >= rot ? __popcll(want & below & ~before) : __popcll(want & ~before) + __popcll(want & below);
}

// Persistent certified-step ray caster (src/queries.py:39-175) for one function.
// A ray's step bounds the segment ahead of it and compares the signs of f at its
// start and hit_eps further on.  Where the bound certifies the segment with room
// (its nearer end 2 % of its scale and the rounding of this net from zero, see
// kNoiseRoom, a segment long beside its distance), both points have the certified sign,
// so the test cannot report a hit and is not evaluated; nor is it where both
// points lie in an earlier segment certified so.  About 60 % of the steps of a
// 256x6 random net, 85 % of a trained 32x8 net's.
//
// A workgroup holds up to kRayPool rays and passes the network NB columns wide
// each time: the segments of NB rays that need a bound, and in one point plane the
// two points of NB/2 rays that need the test (those whose bound did not exclude
// it, then, in the room left, rays bounded in the same pass, which then need no
// second pass).  Four planes a pass, where a test for every step takes five.  The
// rays take turns, so that a workgroup's rays end together instead of each slot's
// one after another and passes stay full until the last steps.
//
// Bound by the FP32 matrix cores at widths >= 128, by the layers' latency below.
// Against the caster with a fixed ray a column (k_cast_rays, still the one
// for several functions): 25,600 rays of a 256x6 ReLU net, 424 steps on average,
// 357 -> 241 ms; 160,000 of the 32x8 fox net, 91 steps, 17.0 -> 13.8 ms; 40,000 of
// the 64x8 ELU bunny net 25.5 -> 21.1 ms.
template <int KIND, int V, int NB, int NW, int WMAX, int OCC, int AS = ACTS_ALL>
__global__ void __launch_bounds__(NW * 64, OCC)
k_cast_rays_pool(const DevModel* __restrict__ models, RayArgs a, int cap) {
  using PL = Planes<KIND, V, 1>;
  static_assert(PL::RB > 0 && NB <= kRayPool, "needs a range bound");
  constexpr int R = PL::R, PT = PL::RB, NT = NW * 64, NP = NB / 2;
  __shared__ float X[R * NB * WMAX];
  __shared__ RayPool S;
  __shared__ int s_code[NB];
  __shared__ float s_val[NB], s_near[NB];
  __shared__ int s_model;
  const int lane = threadIdx.x & 63;
  const bool first_wave = NW == 1 || __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0;

  int gi = blockIdx.x % a.n_groups, seen = 0, rot = 0;
  RayGroup G = a.groups[gi];
  bool exhausted = false;   // this group's rays are all claimed
  int pa = -1, pb = -1;     // this slot's column in the last pass: its segment, its points
  if (first_wave) S.rid[lane] = -1;

  while (true) {
    // the padding of the first layer's input (nobody reads X here)
    for (int e = threadIdx.x; e < R * NB * 16; e += NT) {
      const int k = e & 15;
      if (k >= 3) X[xoff<NB, WMAX>(e / (NB * 16), (e / 16) % NB, k)] = 0.f;
    }
    if (first_wave) {
      int rid = S.rid[lane], phase = S.phase[lane];
      float t = S.t[lane], step = S.step[lane], cov = S.cov[lane];
      float ro[3], di[3];
      for (int k = 0; k < 3; ++k) { ro[k] = S.o[k][lane]; di[k] = S.d[k][lane]; }

      // ---- the last pass's results
      if (pa >= 0) {
        phase = s_code[pa];
        if (phase & kRaySure) {
          float p2 = 0.f, d2 = 0.f;
          for (int k = 0; k < 3; ++k) {
            const float p = ro[k] + t * di[k];
            p2 = p2 + p * p;
            d2 = d2 + di[k] * di[k];
          }
          // the segment is no shorter than 2^-12 of its start's distance from the
          // origin, holds both points, lies where the network cannot overflow, and its
          // bound ends further from zero than bound and points round ((|p| + l)^2 is at
          // most 2 (p2 + l2))
          const float l2 = step * step * d2, near = s_near[pa];
          if (!(l2 >= 0x1p-24f * p2 && l2 <= 1e11f && p2 <= 1e11f && G.hit_eps >= 0.f && G.hit_eps <= step &&
                near * near >= G.noise2 * fmaxf(1.f, 2.f * (p2 + l2))))
            phase &= ~kRaySure;
        }
      }
      const bool covered = t + G.hit_eps <= cov;
      if (rid >= 0 && phase != kRayBounds && (pb >= 0 || covered || (phase & kRaySure))) {
        const bool is_hit = pb >= 0 && sign_f(s_val[2 * pb]) != sign_f(s_val[2 * pb + 1]);
        const int code = phase & ~kRaySure;
        const bool can_step = code == CODE_POSITIVE || code == CODE_NEGATIVE;
        if (phase & kRaySure) cov = t + step;
        const float this_step = can_step ? step : G.hit_eps;
        if (!is_hit) t = t + this_step * G.safety;
        step = can_step ? step * G.grow : step * G.shrink;
        step = fmaxf(step, G.hit_eps);
        phase = kRayBounds;
        const int cnt = S.cnt[lane] + 1;
        S.cnt[lane] = cnt;
        // an iteration is n_substeps of these; a hit ends it (src/queries.py:94-129)
        int sub = S.sub[lane] + 1;
        if (is_hit || sub >= G.n_substeps) {
          sub = 0;
          const int iters = S.iters[lane] + 1;
          S.iters[lane] = iters;
          if (is_hit || (t > G.max_dist) || (cnt >= G.n_max_step)) {
            G.out_t[rid] = t;
            G.out_hit[rid] = is_hit ? 1 : 0;
            G.out_count[rid] = cnt;
            if (G.iter_hist) atomicAdd(&G.iter_hist[min(iters, G.n_max_step + 1)], 1);
            rid = -1;
          }
        }
        S.sub[lane] = sub;
      }

      // ---- new rays for free slots; the next group once this one has drained
      int model = -1;
      while (true) {
        const unsigned long long dead = __ballot(lane < cap && rid < 0);
        const int n_dead = __popcll(dead);
        if (n_dead && !exhausted) {
          long long base = 0;
          if (lane == 0) base = (long long)atomicAdd(G.next_ray, (unsigned long long)n_dead);
          base = ((long long)__builtin_amdgcn_readfirstlane((int)(base >> 32)) << 32) |
                 (unsigned)__builtin_amdgcn_readfirstlane((int)base);
          exhausted = base + n_dead >= G.n;
          const long long claim = base + __popcll(dead & ((1ull << lane) - 1ull));
          if (lane < cap && rid < 0 && claim < G.n) {
            const long long r = claim * G.stride % G.n;
            rid = (int)r;
            t = 0.f; step = G.init_size; cov = -3.4028234663852886e38f; phase = kRayBounds;
            S.cnt[lane] = 0; S.iters[lane] = 0; S.sub[lane] = 0;
            for (int k = 0; k < 3; ++k) {
              ro[k] = G.roots[3 * r + k]; di[k] = G.dirs[3 * r + k];
              S.o[k][lane] = ro[k]; S.d[k][lane] = di[k];
            }
          }
        }
        if (__ballot(rid >= 0)) { model = G.model0; break; }
        if (++seen >= a.n_groups) break;
        gi = gi + 1 == a.n_groups ? 0 : gi + 1;
        G = a.groups[gi];
        exhausted = false;
      }
      S.rid[lane] = rid; S.phase[lane] = phase;
      S.t[lane] = t; S.step[lane] = step; S.cov[lane] = cov;

      // ---- the pass's columns
      const unsigned long long want = __ballot(rid >= 0 && phase == kRayBounds);
      const unsigned long long wantp = __ballot(rid >= 0 && phase != kRayBounds);
      pa = turn_rank(want, rot, lane);
      if (pa >= NB) pa = -1;
      pb = turn_rank(wantp, rot, lane);
      const int na = min(__popcll(want), NB), np = __popcll(wantp);
      if (pa >= 0 && !(t + G.hit_eps <= cov)) pb = np + pa;
      if (pb >= NP) pb = -1;
      const unsigned long long last = __ballot(pa >= 0 && pa == na - 1);
      if (last) rot = __ffsll((long long)last) & 63;   // the lane after the last one chosen
      for (int k = 0; k < 3; ++k) {
        const float ps = ro[k] + t * di[k];
        const float hv = 0.5f * step * di[k];
        if (pa >= 0) {
          for (int p = 0; p < PT; ++p) X[xoff<NB, WMAX>(p, pa, k)] = 0.f;
          X[xoff<NB, WMAX>(0, pa, k)] = ps + hv;
          X[xoff<NB, WMAX>(1, pa, k)] = KIND == 0 && V == 0 ? fabsf(hv) : hv;
        }
        if (pb >= 0) {
          X[xoff<NB, WMAX>(PT, 2 * pb, k)] = ps;
          X[xoff<NB, WMAX>(PT, 2 * pb + 1, k)] = ro[k] + (t + G.hit_eps) * di[k];
        }
      }
      if (lane == 0) s_model = model;
    }
    __syncthreads();
    const int model = __builtin_amdgcn_readfirstlane(s_model);
    if (model < 0) break;

    // columns without a ray hold what the last pass left: their results are not read
    mlp_forward<PL, KIND, V, NB, NW, WMAX, AS>(models[model], X, [&](const float* v, int b) {
      float lo, hi, scale;
      final_bounds<KIND, V>(v, lo, hi, scale);
      const int code = sign_code(lo, hi, 0.f);
      const bool sure = code != CODE_UNKNOWN && scale <= 3.4028234663852886e38f &&
                        fminf(fabsf(lo), fabsf(hi)) >= 0.02f * scale;
      s_code[b] = code | (sure ? kRaySure : 0);
      s_near[b] = fminf(fabsf(lo), fabsf(hi));
      s_val[b] = v[PT];
    });
    __syncthreads();
  }
}
