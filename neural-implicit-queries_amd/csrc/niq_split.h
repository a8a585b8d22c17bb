// Classification with the FP32 contraction carried by bf16 matrix
// instructions, for launches that ask for sign codes only.
//
// Every activation and weight is split into three bf16 terms that add up to it
// exactly (x = x1 + x2 + x3: 8 bits of significand each, 24 in all; above 1e-33, below
// which the third term leaves the range of normal numbers), and a
// dense layer sums the six products down to 2^-18 of the largest,
//     x3 w1 + x2 w2 + x1 w3 + x2 w1 + x1 w2 + x1 w1
// (the three dropped ones are below 2^-26 |x w|, a quarter of half an ulp),
// each exact, with v_mfma_f32_16x16x32_bf16 into one FP32 accumulator.  30 such
// instructions of 16 cycles do the work of 40 FP32 ones of 32 over 5 planes and
// 32 inputs: 480 against 1,280 matrix cycles.  Inputs, accumulator and the
// layer rules stay FP32; there are fewer roundings than in the FP32 chain (6
// accumulations per 32 inputs instead of 32).
//
// The sums round differently from k_classify's, so a box whose bound lies near
// the threshold is listed and classified again by k_classify's own forward:
// the codes are the plain kernel's where the difference stays within that band, whose
// width and limits are measured (kSplitNear).
#pragma once
#include "niq_bf16.h"

// Tiles: 16 boxes, each wave 4 feature tiles (a fragment of X split once in a
// wave's registers serves them all).
template <int WMAX> struct SplitTile;
template <> struct SplitTile<256> { static constexpr int NB = 16, NW = 4; };
template <> struct SplitTile<512> { static constexpr int NB = 16, NW = 8; };

// 8 FP32 values to their three bf16 terms.
__device__ __forceinline__ void split_x8(const floatx4 lo, const floatx4 hi, bf16x8& b1, bf16x8& b2, bf16x8& b3) {
  uintx4_t u1, u2, u3;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float a = q < 2 ? lo[2 * q] : hi[2 * q - 4];
    const float b = q < 2 ? lo[2 * q + 1] : hi[2 * q - 3];
    unsigned h1, h2, h3;
    split3_pair(a, b, h1, h2, h3);
    u1[q] = h1; u2[q] = h2; u3[q] = h3;
  }
  b1 = __builtin_bit_cast(bf16x8, u1);
  b2 = __builtin_bit_cast(bf16x8, u2);
  b3 = __builtin_bit_cast(bf16x8, u3);
}

// The terms of |W| from those of W: w2 and w3 change sign with w1.
__device__ __forceinline__ void abs_terms(bf16x8& w1, bf16x8& w2, bf16x8& w3) {
  const uintx4_t u1 = __builtin_bit_cast(uintx4_t, w1);
  const uintx4_t s = u1 & 0x80008000u;
  w1 = __builtin_bit_cast(bf16x8, u1 ^ s);
  w2 = __builtin_bit_cast(bf16x8, __builtin_bit_cast(uintx4_t, w2) ^ s);
  w3 = __builtin_bit_cast(bf16x8, __builtin_bit_cast(uintx4_t, w3) ^ s);
}

__device__ __forceinline__ floatx4 mfma_bf16(bf16x8 a, bf16x8 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// mlp_forward (affine planes) with the split contraction, for nets whose hidden
// layers are all WMAX wide (padded).  On entry the input planes hold features
// 0..31, zero padded.
template <class PL, int KIND, int V, int NB, int NW, int WMAX, int AS, class Fin>
__device__ __forceinline__ void mlp_forward_split(const DevModelBf16& M, float* __restrict__ X, Fin&& fin) {
  constexpr int R = PL::R;
  constexpr int BT = NB / 16;
  constexpr int FTMAX = (WMAX / 16 + NW - 1) / NW;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 15, lg = lane >> 4;

  for (int l = 0; l < M.n_layers; ++l) {
    const DevLayerBf16& Ly = M.L[l];
    const int nkb = Ly.in_pad >> 5;
    const int nft = Ly.out_pad >> 4;
    const bool last = (l == M.n_layers - 1);
    const auto* W1 = as_global(Ly.W1);
    const auto* W2 = as_global(Ly.W2);
    const auto* W3 = as_global(Ly.W3);
    floatx4 acc[FTMAX][R][BT];
#pragma unroll
    for (int f = 0; f < FTMAX; ++f)
#pragma unroll
      for (int p = 0; p < R; ++p)
#pragma unroll
        for (int t = 0; t < BT; ++t) acc[f][p][t] = floatx4{0.f, 0.f, 0.f, 0.f};

    __syncthreads();   // layer input complete in X

    auto step = [&](auto nf_tag, int kb, const bf16x8* w1, const bf16x8* w2, const bf16x8* w3)
        __attribute__((always_inline)) {
      constexpr int NF = decltype(nf_tag)::value;
#pragma unroll
      for (int pt = 0; pt < R * BT; ++pt) {
        const int p = pt / BT, t = pt % BT;
        const floatx4 lo = *reinterpret_cast<const floatx4*>(&X[xoff<NB, WMAX>(p, t * 16 + ln, kb * 32 + lg * 8)]);
        const floatx4 hi =
            *reinterpret_cast<const floatx4*>(&X[xoff<NB, WMAX>(p, t * 16 + ln, kb * 32 + lg * 8 + 4)]);
        bf16x8 b1, b2, b3;
        split_x8(lo, hi, b1, b2, b3);
        bf16x8 a1[NF], a2[NF], a3[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          a1[f] = w1[f]; a2[f] = w2[f]; a3[f] = w3[f];
          if (PL::absw(p)) abs_terms(a1[f], a2[f], a3[f]);
        }
        // Smallest products first, the feature tiles' independent chains
        // interleaved.  The matrix unit does not round a sum to nearest, which
        // shows where all terms have one sign (the error plane) and in the
        // base: there a chunk sums from zero and is added by the vector ALU.
        const bool fresh = PL::absw(p) || PL::bias(p);
        floatx4 c[NF];
#pragma unroll
        for (int f = 0; f < NF; ++f) c[f] = mfma_bf16(a1[f], b3, fresh ? floatx4{0.f, 0.f, 0.f, 0.f} : acc[f][p][t]);
#pragma unroll
        for (int f = 0; f < NF; ++f) c[f] = mfma_bf16(a2[f], b2, c[f]);
#pragma unroll
        for (int f = 0; f < NF; ++f) c[f] = mfma_bf16(a3[f], b1, c[f]);
#pragma unroll
        for (int f = 0; f < NF; ++f) c[f] = mfma_bf16(a1[f], b2, c[f]);
#pragma unroll
        for (int f = 0; f < NF; ++f) c[f] = mfma_bf16(a2[f], b1, c[f]);
#pragma unroll
        for (int f = 0; f < NF; ++f) c[f] = mfma_bf16(a1[f], b1, c[f]);
#pragma unroll
        for (int f = 0; f < NF; ++f) acc[f][p][t] = fresh ? acc[f][p][t] + c[f] : c[f];
      }
    };
    // one chunk of 32 inputs ahead
    bf16x8 n1[FTMAX], n2[FTMAX], n3[FTMAX];
    auto fetch = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
      for (int f = 0; f < FTMAX; ++f) {
        const size_t o = (size_t)((wave + f * NW) * nkb + kb) * 64 + lane;
        n1[f] = W1[o]; n2[f] = W2[o]; n3[f] = W3[o];
      }
    };
    if (!last) {   // a hidden layer: every feature tile of the wave exists
      fetch(0);
      for (int kb = 0; kb < nkb; ++kb) {
        bf16x8 w1[FTMAX], w2[FTMAX], w3[FTMAX];
#pragma unroll
        for (int f = 0; f < FTMAX; ++f) { w1[f] = n1[f]; w2[f] = n2[f]; w3[f] = n3[f]; }
        fetch(kb + 1 < nkb ? kb + 1 : kb);
        step(std::integral_constant<int, FTMAX>{}, kb, w1, w2, w3);
      }
    } else {
      // the last layer's one tile: its chunks shared out over the waves, the
      // partial sums added below
      for (int kb = wave; kb < nkb; kb += NW) {
        const size_t o = (size_t)kb * 64 + lane;
        const bf16x8 w1[1] = {W1[o]}, w2[1] = {W2[o]}, w3[1] = {W3[o]};
        step(std::integral_constant<int, 1>{}, kb, w1, w2, w3);
      }
    }

    floatx4 bias4[FTMAX];
#pragma unroll
    for (int f = 0; f < FTMAX; ++f) {
      const int ft = wave + f * NW;
      if (ft < nft) bias4[f] = *reinterpret_cast<const __attribute__((address_space(1))) floatx4*>(
                        as_global(Ly.bias) + ft * 16 + lg * 4);
    }
    __syncthreads();   // every wave has consumed X

    if (last) {
      floatx4* Pp = reinterpret_cast<floatx4*>(X);
      if (wave > 0) {
#pragma unroll
        for (int p = 0; p < R; ++p)
#pragma unroll
          for (int t = 0; t < BT; ++t) Pp[(((wave - 1) * R + p) * BT + t) * 64 + lane] = acc[0][p][t];
      }
      __syncthreads();
      if (wave == 0) {
#pragma unroll
        for (int w = 1; w < NW; ++w)
#pragma unroll
          for (int p = 0; p < R; ++p)
#pragma unroll
            for (int t = 0; t < BT; ++t) acc[0][p][t] += Pp[(((w - 1) * R + p) * BT + t) * 64 + lane];
      }
      __syncthreads();   // partials read before the caller reuses X
      if (wave == 0 && lg == 0) {
#pragma unroll
        for (int t = 0; t < BT; ++t) {
          float v[R];
#pragma unroll
          for (int p = 0; p < R; ++p) v[p] = acc[0][p][t][0] + (PL::bias(p) ? bias4[0][0] : 0.f);
          fin(v, t * 16 + ln);
        }
      }
    } else {
      layer_epilogue<PL, KIND, V, NB, NW, WMAX, AS>(Ly.act, nft, wave, lane, acc, bias4, X);
    }
  }
}

// Classify axis-aligned boxes by the split contraction.  A box goes to the list
// that k_classify then classifies when its bound lies within kSplitNear * (|base|
// + radius) of the threshold or within the rounding of f (a.noise), is not a number
// or is too small to judge by, or when the box is smaller than 1/200 of its
// distance from the origin or than a.min_half = round_rel / kSplitRound.
//
// The band: the two forms' bounds differ by their rounding alone.  The rounding D of
// a pre-activation moves its ReLU's chord, so the difference of two bounds relative to
// |base| + radius is some D / r, r the pre-activation's radius over the box, and
// round_rel / (half-width) estimates the largest D / r of the net's layers.
// Measured with emulated float32 sums, 2,500 boxes each of 20 nets (He and Xavier,
// 256x1 to 512x8, hidden biases up to 1e3 among them) at half-widths 1/16 to 1/200: the
// largest difference is at most 5.6 times that estimate, and kSplitRound = 5e-4 keeps
// it below 2.8e-3, a seventh of the band.  (On the card, 131,072 boxes each of He and
// Xavier nets: 1.3e-4 at half-width 1/64, 5e-4 at 1/128.)  Nets without large biases have
// round_rel below 2e-6 and reach the 1/200 first.  The band holds 1 % of the boxes of a
// shallow net at half-width 1/128, none of a deep one's, whose bounds all span the
// threshold widely.
constexpr float kSplitNear = 2e-2f;
constexpr float kSplitRound = 5e-4f;

// The tile of boxes i0 .. i0 + NB - 1 of n.
template <int V, int NB, int NW, int WMAX, int AS>
__device__ __forceinline__ void classify_split_tile(const DevModelBf16& M, const ClassifyArgs& a, float* X,
                                                    long long i0, long long n) {
  using PL = Planes<0, V, 0>;
  constexpr int NT = NW * 64, R = PL::R;
  fill_box_inputs<0, V, NB, NT, WMAX>(X, a, i0, n);
  for (int e = threadIdx.x; e < R * NB * 16; e += NT)   // the chunk's upper half
    X[xoff<NB, WMAX>(e / (NB * 16), (e / 16) % NB, 16 + (e & 15))] = 0.f;
  mlp_forward_split<PL, 0, V, NB, NW, WMAX, AS>(M, X, [&](const float* v, int b) {
    const long long i = i0 + b;
    if (i >= n) return;
    float hmin = INFINITY, cmax = 0.f;
    for (int k = 0; k < a.d; ++k) {
      const float l = a.lower[i * a.d + k], u = a.upper[i * a.d + k];
      hmin = fminf(hmin, 0.5f * (u - l));
      cmax = fmaxf(cmax, fmaxf(fabsf(l), fabsf(u)));
    }
    float lo, hi, scale;
    final_bounds<0, V>(v, lo, hi, scale);
    a.codes[i] = sign_code(lo, hi, a.offset);
    const float far = fmaxf(1.f, cmax);
    const float tol = fmaxf(kSplitNear * scale, a.noise * far);
    const bool clear = fabsf(lo - a.offset) > tol && fabsf(hi + a.offset) > tol && scale > 1e-20f && scale < 1e30f &&
                       hmin >= kSplitMinSize * cmax && hmin >= a.min_half * far;
    if (!clear) {
      const int slot = atomicAdd(a.list_n, 1);
      if (slot < a.list_cap) a.list[slot] = (int)i;
    }
  });
}

template <int V, int NB, int NW, int WMAX, int AS>
__global__ void __launch_bounds__(NW * 64, 2)
k_classify_split(const DevModelBf16* __restrict__ Mp, ClassifyArgs a) {
  __shared__ float X[Planes<0, V, 0>::R * NB * WMAX];
  const long long n = a.n_dev ? (long long)(*a.n_dev) : a.n;
  const long long ntiles = (n + NB - 1) / NB;
  for (long long tile = blockIdx.x; tile < ntiles; tile += gridDim.x)
    classify_split_tile<V, NB, NW, WMAX, AS>(*Mp, a, X, tile * NB, n);
}

// Point values by the split contraction, for nets whose activations stay far
// below the bf16 range on inputs up to kSplitMaxInput (the host checks).  A
// point with a larger, infinite or NaN coordinate is evaluated by the FP32
// contraction instead, to the bits of k_points.
// 1,000,003 points of the 256x6 ReLU net: 3.14 ms, against 5.43 by FP32 matrix
// instructions.  Error against float64 (256x6, 100,003 points of the unit cube):
// 5.2e-7 against 1.4e-6; 0.3 to 0.85 of the FP32 chain's over ReLU, TanH, ELU and
// sin nets of 2 to 8 layers and inputs up to 0.01, 1 and 100.
//
// A tile that holds such points is set aside, its points in one list for each
// contraction, and a list is worked off in full tiles (what is left at the end, in a
// last one): a batch costs what its two kinds of points cost, however they are mixed.
constexpr float kSplitMaxInput = 1e6f;

template <int NB, int NW, int WMAX, int AS>
__global__ void __launch_bounds__(NW * 64, 2)
k_points_split(const DevModelBf16* __restrict__ Mp, const DevModel* __restrict__ M32, const float* __restrict__ x,
               int d, long long n, float* __restrict__ out) {
  using PL = Planes<2, 0, 1>;
  constexpr int NT = NW * 64;
  static_assert(NB == 64, "one wave sorts a tile's points");
  __shared__ float X[NB * WMAX];
  __shared__ int bad[NB + 1];            // points outside the split's range, and whether any
  __shared__ long long aside[2][2 * NB]; // points inside the range, and outside it
  const long long ntiles = (n + NB - 1) / NB;
  int n_aside[2] = {0, 0};
  long long tile = blockIdx.x;
  while (true) {
    const bool end = tile >= ntiles;
    int from = -1;   // the list that this tile is taken from
    if (n_aside[0] >= NB || (end && n_aside[0] > 0)) from = 0;
    else if (n_aside[1] >= NB || (end && n_aside[1] > 0)) from = 1;
    else if (end) break;
    const long long i0 = tile * NB;
    const int cnt = from >= 0 ? min(n_aside[from], NB) : (int)min((long long)NB, n - i0);
    auto point = [&](int b) { return from >= 0 ? aside[from][b] : i0 + b; };
    if (from < 0) {
      tile += gridDim.x;
      for (int b = threadIdx.x; b <= NB; b += NT) bad[b] = 0;
      __syncthreads();
    }
    for (int e = threadIdx.x; e < NB * 32; e += NT) {
      const int b = e >> 5, k = e & 31;
      const float v = (b < cnt && k < d) ? x[point(b) * d + k] : 0.f;
      if (from < 0 && !(fabsf(v) <= kSplitMaxInput)) { bad[b] = 1; bad[NB] = 1; }
      X[xoff<NB, WMAX>(0, b, k)] = v;
    }
    if (from < 0) {
      __syncthreads();
      if (bad[NB]) {   // uniform
        const bool in = (int)threadIdx.x < cnt, out_of = in && bad[threadIdx.x & (NB - 1)];
        const unsigned long long mo = __ballot(out_of), mi = __ballot(in && !out_of);   // of the first wave
        if (in) {
          const unsigned long long below = (1ull << threadIdx.x) - 1ull;
          if (out_of) aside[1][n_aside[1] + __popcll(mo & below)] = i0 + threadIdx.x;
          else aside[0][n_aside[0] + __popcll(mi & below)] = i0 + threadIdx.x;
        }
        int n_out = 0;
        for (int b = 0; b < NB; ++b) n_out += bad[b];
        n_aside[0] += cnt - n_out;
        n_aside[1] += n_out;
        __syncthreads();   // the lists are complete, the flags read
        continue;
      }
    }
    auto fin = [&](const float* v, int b) {
      if (b < cnt) out[point(b)] = v[0];
    };
    if (from == 1) mlp_forward<PL, 2, 0, NB, NW, WMAX, AS>(*M32, X, fin);
    else mlp_forward_split<PL, 2, 0, NB, NW, WMAX, AS>(*Mp, X, fin);
    __syncthreads();   // X is free, the list read
    if (from >= 0) {
      const int left = n_aside[from] - cnt;
      if ((int)threadIdx.x < left) {   // less than a tile: the first wave moves it in one step
        const long long p = aside[from][cnt + threadIdx.x];
        aside[from][threadIdx.x] = p;
      }
      n_aside[from] = left;
      __syncthreads();
    }
  }
}
