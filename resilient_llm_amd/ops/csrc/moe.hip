// Mixture of experts, two kinds.  Gated: the routing weight (a sigmoid)
// multiplies the expert's INPUT, y = sum over the chosen experts of
// expert(w * h), clamped swish-like gate.  Squared relu: y = sum of
// w expert(h), weights a softmax over all routes, scaled to sum to one over
// the chosen; a correction may shift the choice, routes may be chosen by
// groups, and the last routes may be identity experts (w h), which run
// nothing here: whoever sums a token's outputs adds them.
//
//   moe_route     router logits (f32 accumulation over the activation's
//                 own values), scores, top-k
//   moe_plan      (token, choice) pairs in expert order + row tiles, from the
//                 router's counts; no host round trip, so it is capturable
//   moe_experts   two grouped GEMMs.  Up: w * (W h) is scaled in the
//                 accumulator, gated in registers (gate and up rows are
//                 packed in alternating blocks of 16) and leaves as one
//                 [pairs, ff] tensor; or w relu(W h)^2, which the down
//                 product carries through.  Down: scatters every pair's row to
//                 [token, choice]; the sum over choices happens in the
//                 residual kernel that reads it anyway.
// Small row counts stream the weights straight into MFMA fragments, K
// split over the waves; large ones run tiles of 128 or 256 rows by 256
// columns through LDS (tile_product.h).

#include "mix.h"
#include "tile_product.h"

#include <algorithm>

namespace rlli {
namespace {

// ------------------------------------------------------------- router
// Reductions over either half of a wave on the VALU, the result in all of its
// lanes: rows of 16, then across the two, then out of the half's last lane.
template <int CTRL>
DEV_INLINE float dpp_or_own(float v) {
  const int b = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, false));
}
// of each half, what it has in its lane at0 or at1
DEV_INLINE float of_lane(float v, int at0, int at1) {
  const int b = __builtin_bit_cast(int, v);
  const int x = __builtin_amdgcn_readlane(b, at0);
  const int y = __builtin_amdgcn_readlane(b, 32 + at1);
  return __builtin_bit_cast(float, threadIdx.x & 32 ? y : x);
}
DEV_INLINE float half_sum_dpp(float v) {
  v = group_sum_dpp<16>(v);
  // rows 0 + 1 | 2 + 3
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
           0, __builtin_bit_cast(int, v), 0x142, 0xa, 0xf, false));
  return of_lane(v, 31, 31);
}
DEV_INLINE float half_max_dpp(float v) {
  v = fmaxf(v, dpp_or_own<0x111>(v));     // row_shr 1, 2, 4, 8
  v = fmaxf(v, dpp_or_own<0x112>(v));
  v = fmaxf(v, dpp_or_own<0x114>(v));
  v = fmaxf(v, dpp_or_own<0x118>(v));
  v = fmaxf(v, dpp_or_own<0x142>(v));     // row_bcast 15
  return of_lane(v, 31, 31);
}

// 16 rows per workgroup, K split over eight waves, whose halves then rank a row
// each.  What bounds it is latency: a round of loads where they fit the
// registers (32 routes of 2048: all of them), sums through LDS, and a choice
// after the other.  Loaded as the products take them, neighbouring lanes have rows
// of their own and the cache looks up 16 bytes at a time; turned in LDS they come
// by 64 (32 routes of 2048, us: 1 row 8.5 and 7.5, 64 9.7 and 8.1, 6001 17.8 and
// 16.1).  It leaves how often its rows chose each expert behind, so
// that the plan needs no pass of its own over the choices.
template <typename T, int ET>
__global__ __launch_bounds__(512)
void moe_route_kernel(MoeArgs a) {
  constexpr int E16 = ET * 16, NW = 8;
  // (32-bit activations and many routes are too much for LDS)
  constexpr bool LINES = sizeof(T) == 2 && ET <= 4;
  __shared__ union {
    s16x8_t turns[LINES ? NW * 64 * (ET + 1) : 1];
    float part[NW][16][E16 + 1];          // behind them
  } lds;
  auto& part = lds.part;
  __shared__ int chosen[E16];
  auto wave_fence = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.x * 16;
  if (threadIdx.x < E16) chosen[threadIdx.x] = 0;
  const T* h = reinterpret_cast<const T*>(a.h) +
               int64_t(min(row0 + lr, a.rows - 1)) * a.width;
  const T* wr = reinterpret_cast<const T*>(a.router);
  const T* wp[ET];
  f32x4_t acc[ET];
#pragma unroll
  for (int e = 0; e < ET; ++e) {
    // columns past the last route repeat it; nobody reads them
    wp[e] = wr + int64_t(min(e * 16 + lr, a.routes - 1)) * a.width;
    acc[e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  constexpr int U = ET <= 4 ? 4 : 1;      // k steps with loads in flight
  int k0 = w * 32;
  if constexpr (LINES) {
    // four lanes to 64 bytes of a row, and to the lanes that multiply them
    // through LDS, turned by the row so that reads meet no bank twice
    s16x8_t* turn = lds.turns + w * 64 * (ET + 1);
    const int rr = lane >> 2, piece = (lane & 3) ^ (rr >> 2);
    const T* hp = reinterpret_cast<const T*>(a.h) +
                  int64_t(min(row0 + rr, a.rows - 1)) * a.width + piece * 8;
    const T* rp[ET];
#pragma unroll
    for (int e = 0; e < ET; ++e)
      rp[e] = wr + int64_t(min(e * 16 + rr, a.routes - 1)) * a.width +
              piece * 8;
    const int mine = lr * 4 + (g ^ (lr >> 2));
    for (; k0 + (U - 1) * NW * 32 + 32 <= a.width; k0 += U * NW * 32) {
      s16x8_t raw[U][ET + 1];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = k0 + u * NW * 32;
        raw[u][ET] = *reinterpret_cast<const s16x8_t*>(hp + k);
#pragma unroll
        for (int e = 0; e < ET; ++e)
          raw[u][e] = *reinterpret_cast<const s16x8_t*>(rp[e] + k);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int i = 0; i <= ET; ++i) turn[i * 64 + lane] = raw[u][i];
        wave_fence();
        Frag8<T> fa, fb[ET];
        fa.v = turn[ET * 64 + mine];
#pragma unroll
        for (int e = 0; e < ET; ++e)
          fb[e].v = turn[e * 64 + mine];
        wave_fence();
#pragma unroll
        for (int e = 0; e < ET; ++e)
          acc[e] = Frag8<T>::mma(fa, fb[e], acc[e]);
      }
    }
  }
  for (; k0 + (U - 1) * NW * 32 + 32 <= a.width; k0 += U * NW * 32) {
    Frag8<T> fa[U], fb[U][ET];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * NW * 32 + g * 8;
      fa[u].load(h + k);
#pragma unroll
      for (int e = 0; e < ET; ++e) fb[u][e].load(wp[e] + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < ET; ++e)
        acc[e] = Frag8<T>::mma(fa[u], fb[u][e], acc[e]);
  }
  for (; k0 < a.width; k0 += NW * 32) {
    const int k = k0 + g * 8;
    Frag8<T> fa;
    fa.zero();
    if (k < a.width) fa.load(h + k);
#pragma unroll
    for (int e = 0; e < ET; ++e) {
      Frag8<T> fb;
      fb.zero();
      if (k < a.width) fb.load(wp[e] + k);
      acc[e] = Frag8<T>::mma(fa, fb, acc[e]);
    }
  }
  if constexpr (LINES) __syncthreads();
#pragma unroll
  for (int e = 0; e < ET; ++e)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      part[w][g * 4 + r][e * 16 + lr] = acc[e][r];
  __syncthreads();
  // a half ranks a row, its lane l holding routes l, l + 32, ...
  constexpr int EL = (E16 + 31) / 32;
  constexpr float kNone = -INFINITY;      // cannot be chosen
  const int hl = lane & 31;
  const int t = w * 2 + (lane >> 5);
  const int row = row0 + t;               // (past the last: nobody's)
  float s[EL], choice[EL];
#pragma unroll
  for (int i = 0; i < EL; ++i) {
    const int e = i * 32 + hl;
    s[i] = kNone;
    if (e < a.routes) {
      s[i] = 0.f;
#pragma unroll
      for (int p = 0; p < NW; ++p) s[i] += part[p][t][e];
    }
  }
  if (a.softmax) {
    float mx = kNone, sum = 0.f;
#pragma unroll
    for (int i = 0; i < EL; ++i) mx = fmaxf(mx, s[i]);
    mx = half_max_dpp(mx);
#pragma unroll
    for (int i = 0; i < EL; ++i) {
      s[i] = expf(s[i] - mx);             // 0 past the last route
      sum += s[i];
    }
    sum = half_sum_dpp(sum);
#pragma unroll
    for (int i = 0; i < EL; ++i) s[i] /= sum;
  } else {
#pragma unroll
    for (int i = 0; i < EL; ++i) s[i] = 1.f / (1.f + expf(-s[i]));
  }
#pragma unroll
  for (int i = 0; i < EL; ++i) {
    const int e = i * 32 + hl;
    choice[i] = kNone;
    if (e < a.routes)
      choice[i] = s[i] + (a.correction ? a.correction[e] : 0.f);
  }
  if (a.keep < a.groups) {
    // this row's part sums are read; their place holds the choice scores,
    // the groups' best ones, and which groups stay
    float *cs = part[0][t], *best = part[1][t], *stays = part[2][t];
    const int size = a.routes / a.groups;
    wave_fence();
#pragma unroll
    for (int i = 0; i < EL; ++i)
      if (i * 32 + hl < a.routes) cs[i * 32 + hl] = choice[i];
    wave_fence();
    for (int g = hl; g < a.groups; g += 32) {
      float b = kNone;
      for (int e = g * size; e < (g + 1) * size; ++e) b = fmaxf(b, cs[e]);
      best[g] = b;
    }
    wave_fence();
    for (int g = hl; g < a.groups; g += 32) {
      int ahead = 0;
      for (int o = 0; o < a.groups; ++o)
        ahead += best[o] > best[g] || (best[o] == best[g] && o < g);
      stays[g] = ahead < a.keep ? 1.f : 0.f;
    }
    wave_fence();
#pragma unroll
    for (int i = 0; i < EL; ++i) {
      const int e = i * 32 + hl;
      if (e < a.routes && stays[e / size] == 0.f) choice[i] = kNone;
    }
  }
  float won[EL], total = 0.f;             // lane c & 31 keeps weight c
  for (int c = 0; c < a.top; ++c) {
    // the best score left, and the first route that has it, of either half
    float bv = choice[0];
#pragma unroll
    for (int i = 1; i < EL; ++i) bv = fmaxf(bv, choice[i]);
    bv = half_max_dpp(bv);
    int b0 = 0x7fffffff, b1 = b0;
#pragma unroll
    for (int i = EL - 1; i >= 0; --i) {
      const uint64_t has = __ballot(choice[i] == bv);
      if (uint32_t(has)) b0 = i * 32 + __builtin_ctz(uint32_t(has));
      if (has >> 32) b1 = i * 32 + __builtin_ctz(uint32_t(has >> 32));
    }
    int bi = lane & 32 ? b1 : b0;
#pragma unroll
    for (int i = 0; i < EL; ++i)
      if (i * 32 + hl == bi) choice[i] = kNone;
    bi = min(bi, a.routes - 1);           // a NaN row still names a route
    b0 = min(b0, a.routes - 1);
    b1 = min(b1, a.routes - 1);
    float mine = s[0];
#pragma unroll
    for (int i = 1; i < EL; ++i)
      if (bi >> 5 == i) mine = s[i];
    mine = of_lane(mine, b0 & 31, b1 & 31);
    total += mine;
#pragma unroll
    for (int i = 0; i < EL; ++i)
      if (c == i * 32 + hl) won[i] = mine;
    if (hl == 0 && row < a.rows) {
      a.ids[int64_t(row) * a.top + c] = bi;
      atomicAdd(&chosen[bi], 1);
    }
  }
  const float scale = a.softmax ? 1.f / (total + 1e-20f) : 1.f;
#pragma unroll
  for (int i = 0; i < EL; ++i)
    if (i * 32 + hl < a.top && row < a.rows)
      a.weights[int64_t(row) * a.top + i * 32 + hl] = won[i] * scale;
  if (!a.chosen) return;
  __syncthreads();
  // (a row of NaN may choose one route ``top`` times: 4096 at most)
  if (threadIdx.x < chosen_stride(a.experts))
    a.chosen[int64_t(blockIdx.x) * chosen_stride(a.experts) + threadIdx.x] =
        threadIdx.x < a.experts ? uint16_t(chosen[threadIdx.x]) : 0;
}

// --------------------------------------------------------------- plan
constexpr int MAXE = 256;

// Pairs to places in expert order, from how often each workgroup of the router
// chose each expert: a workgroup sums all of that and what belongs to rows ahead
// of its own, PLAN_ROWS or more, and places its pairs.  What bounds it is latency:
// 8.4 us for 6001 rows and 32 experts, four each, 4.8 for 64 rows.  (Two passes
// over the choices with counts by atomics between them 14.8 and a gap, one
// workgroup for 64 rows 6.0.)
constexpr int PLAN_ROWS = 512, PLAN_MOST = 64;    // rows, workgroups

__global__ __launch_bounds__(256)
void moe_plan_kernel(MoeArgs a, int rows_each) {
  __shared__ int part[2][4 * 256];        // by four experts: threads' sums
  __shared__ int cursor[MAXE], wave_total[4][3];
  const int tid = threadIdx.x, lane = tid & 63;
  const int blocks = (a.rows + 15) / 16, own = blockIdx.x * rows_each / 16;
  const int cols = chosen_stride(a.experts) / 4;
  const int sums = min(256 / cols, min(blocks, 32));
  // its pairs' choices, the first eight of a thread asked for at once
  const int p0 = blockIdx.x * rows_each * a.top;
  const int p1 = min(a.rows * a.top, p0 + rows_each * a.top);
  constexpr int EARLY = 8;
  int early[EARLY];
#pragma unroll
  for (int i = 0; i < EARLY; ++i)
    early[i] = a.ids[min(p0 + i * 256 + tid, p1 - 1)];
  {
    // four experts' counts at a time: all, and of the router's workgroups
    // ahead of this one's rows
    const int c = tid % cols, p = tid / cols;
    int all[4] = {0, 0, 0, 0}, ahead[4] = {0, 0, 0, 0};
    if (p < sums) {
      const uint2* from = reinterpret_cast<const uint2*>(a.chosen) + c;
#pragma unroll 8
      for (int b = p; b < blocks; b += sums) {
        const uint2 v = from[int64_t(b) * cols];
        const int n[4] = {int(v.x & 0xffff), int(v.x >> 16),
                          int(v.y & 0xffff), int(v.y >> 16)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          all[i] += n[i];
          ahead[i] += b < own ? n[i] : 0;
        }
      }
      // [p][4 c + i], as wide as the experts' columns
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        part[0][p * cols * 4 + c * 4 + i] = all[i];
        part[1][p * cols * 4 + c * 4 + i] = ahead[i];
      }
    }
  }
  __syncthreads();
  int n = 0, before = 0;
  if (tid < a.experts)
    for (int p = 0; p < sums; ++p) {
      n += part[0][p * cols * 4 + tid];
      before += part[1][p * cols * 4 + tid];
    }
  const int half = a.tile_m > 16 ? a.tile_m / 2 : 0;
  const int tiles = (n + a.tile_m - 1) / a.tile_m;
  const int full = a.together ? tiles
                              : n / a.tile_m + (n % a.tile_m > half ? 1 : 0);
  // pairs, full tiles and others of the experts up to each: sums over lanes,
  // then over waves
  int upto[3] = {n, full, tiles - full};
#pragma unroll
  for (int d = 1; d < 64; d <<= 1)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int v = __shfl_up(upto[i], d, kWave);
      if (lane >= d) upto[i] += v;
    }
  if (lane == 63)
#pragma unroll
    for (int i = 0; i < 3; ++i) wave_total[tid >> 6][i] = upto[i];
  __syncthreads();
  for (int w = 0; w < tid >> 6; ++w)
#pragma unroll
    for (int i = 0; i < 3; ++i) upto[i] += wave_total[w][i];
  const int start = upto[0] - n;
  if (tid < a.experts) cursor[tid] = start + before;
  __syncthreads();
  auto place = [&](int p, int e) {
    if (p < p1 && e < a.experts) a.perm[atomicAdd(&cursor[e], 1)] = p;
  };
#pragma unroll
  for (int i = 0; i < EARLY; ++i) place(p0 + i * 256 + tid, early[i]);
  for (int p = p0 + EARLY * 256 + tid; p < p1; p += 256) place(p, a.ids[p]);
  if (blockIdx.x != 0) return;

  // The tile list: tiles more than half full in expert order, then the other
  // ones, so that the cheap tiles run where the last full ones leave compute
  // units idle; or all in expert order (a.together), where an expert's weights
  // would be read twice for its two tiles.
  int all_full = 0, others = 0;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    all_full += wave_total[w][1];
    others += wave_total[w][2];
  }
  for (int i = 0; i < tiles; ++i) {
    const int t = i < full ? upto[1] - full + i
                           : all_full + upto[2] - (tiles - full);
    a.tile_expert[t] = tid;
    a.tile_row0[t] = start + i * a.tile_m;
    a.tile_rows[t] = min(a.tile_m, n - i * a.tile_m);
  }
  for (int t = all_full + others + tid; t < a.max_tiles; t += 256)
    a.tile_rows[t] = 0;
  if (tid == 0) {
    a.counters[0] = all_full;
    a.counters[1] = others;
  }
}

template <typename T>
DEV_INLINE float expert_gate(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  // the result is rounded to bf16: hardware exponential and reciprocal do
  if constexpr (sizeof(T) == 2)
    return g * __builtin_amdgcn_rcpf(1.f + __expf(-1.702f * g)) * (u + 1.f);
  return g / (1.f + expf(-1.702f * g)) * (u + 1.f);
}

DEV_INLINE float relu_squared(float x) {
  x = fmaxf(x, 0.f);
  return x * x;
}

// --------------------------------------- small row counts: stream weights
// One workgroup per (16-row tile, 32 weight rows); its waves split K.
template <typename T, bool UP, bool GATED>
__global__ __launch_bounds__(256)
void moe_small_kernel(MoeArgs a) {
  __shared__ float part[4][2][16][17];
  const int tile = blockIdx.y;
  const int rows = a.tile_rows[tile];
  if (rows == 0) return;
  const int e = a.tile_expert[tile];
  const int p0 = a.tile_row0[tile];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, g = lane >> 4;
  const int K = UP ? a.width : a.ffp;
  const int N = UP ? (GATED ? 2 : 1) * a.ffp : a.width;
  const int n0 = blockIdx.x * 32;

  const int pr = p0 + min(lr, rows - 1);
  const T* arow;
  if constexpr (UP)
    arow = reinterpret_cast<const T*>(a.h) +
           int64_t(a.perm[pr] / a.top) * a.width;
  else
    arow = reinterpret_cast<const T*>(a.act) + int64_t(pr) * a.ffp;
  const T* wb = reinterpret_cast<const T*>(UP ? a.w_up : a.w_down) +
                int64_t(e) * N * K;
  const T* b0 = wb + int64_t(min(n0 + lr, N - 1)) * K;
  const T* b1 = wb + int64_t(min(n0 + 16 + lr, N - 1)) * K;
  f32x4_t acc0 = f32x4_t{0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
  // a wave takes 128 consecutive k (whole lines of every weight row),
  // all loads before the MFMAs
  for (int k0 = w * 128; k0 < K; k0 += 512) {
    Frag8<T> fa[4], f0[4], f1[4];
    if (k0 + 128 <= K) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k0 + u * 32 + g * 8;
        f0[u].load(b0 + k);
        f1[u].load(b1 + k);
        fa[u].load(arow + k);
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = k0 + u * 32 + g * 8;
        fa[u].zero();
        f0[u].zero();
        f1[u].zero();
        if (k < K) {
          fa[u].load(arow + k);
          f0[u].load(b0 + k);
          f1[u].load(b1 + k);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      acc0 = Frag8<T>::mma(fa[u], f0[u], acc0);
      acc1 = Frag8<T>::mma(fa[u], f1[u], acc1);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    part[w][0][g * 4 + r][lr] = acc0[r];
    part[w][1][g * 4 + r][lr] = acc1[r];
  }
  __syncthreads();
  const int row = threadIdx.x >> 4, col = threadIdx.x & 15;
  if (row >= rows) return;
  float s0 = 0.f, s1 = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    s0 += part[i][0][row][col];
    s1 += part[i][1][row][col];
  }
  const int pair = a.perm[p0 + row];
  if constexpr (UP) {
    const float wt = a.weights[pair];
    T* o = reinterpret_cast<T*>(a.act) + int64_t(p0 + row) * a.ffp;
    if constexpr (GATED) {
      act_store(o + blockIdx.x * 16 + col,
                expert_gate<T>(s0 * wt, s1 * wt, a.limit));
    } else {
      act_store(o + n0 + col, relu_squared(s0) * wt);
      act_store(o + n0 + 16 + col, relu_squared(s1) * wt);
    }
  } else {
    T* y = reinterpret_cast<T*>(a.y) + int64_t(pair) * a.width;
    if (n0 + col < N) act_store(y + n0 + col, s0);
    if (n0 + 16 + col < N) act_store(y + n0 + 16 + col, s1);
  }
}

// ------------------------------------------- large row counts: LDS tiles
// A workgroup has a tile of 256 x 256, or 128 rows by 256 for experts with
// fewer rows (tile_product.h).
// Consecutive workgroups go to different XCDs.  Each XCD gets an equal run of
// the full tiles' blocks, then an equal run of the others', counted on the
// device: the tiles there could be are up to one per expert more, and runs of
// those left whole XCDs idle.  A run goes over four tiles' column blocks at a
// time, so that what an XCD works on at once, about 32 blocks, shares eight
// column blocks' weights and four tiles' rows in its L2 (hits at width 4096: 49
// -> 77 % up, 62 -> 77 % down).  Whole calls, before -> now, us, three runs
// each: 8192 rows of 4096, 16 experts of 3584, two each: 1658-1669 ->
// 1389-1398; 2048 rows of them 753-783 -> 604-635; 6001 rows of 2048, 32
// experts of 1024, four each: 397-407 -> 375-381 (on another card 404 -> 396).
enum TileKind { FULL, LOW, NARROW };

template <int MH>
DEV_INLINE bool tile_of(const MoeArgs& a, int block, int n_blocks, int& tile,
                        int& nb, TileKind& kind) {
  const int x = block & 7;
  int s = block >> 3, n = a.counters[0], first = 0;
  // of 128 rows, which are as high as low ones, all where CUs are left for them
  const bool all = MH == 2 && (n + a.counters[1]) * n_blocks <= 128;
  if (all) n_blocks *= 2;
  int per = (n * n_blocks + 7) / 8;
  kind = all ? NARROW : FULL;
  if (s >= per) {
    s -= per;
    // CUs that the full tiles' last round leaves idle
    const int idle = 255 - (n * n_blocks + 255) % 256;
    first = n;
    n = a.counters[1];
    if (!all) {
      kind = n * n_blocks > 2 * idle && n * n_blocks <= 128 ? NARROW : LOW;
      if (kind == NARROW) n_blocks *= 2;
    }
    per = (n * n_blocks + 7) / 8;
    if (s >= per) return false;
  }
  const int i = x * per + s;
  if (i >= n * n_blocks) return false;
  const int group = i / (4 * n_blocks), j = i - group * 4 * n_blocks;
  const int high = min(4, n - group * 4);
  nb = j / high;
  tile = first + group * 4 + j % high;
  return true;
}

template <bool UP, int MH, int NH, bool GATED>
DEV_INLINE void moe_tile(const MoeArgs& a, int rows, int e, int p0, int nb) {
  using P = tile::Product<MH, NH>;
  constexpr int TM = P::TM, TN = P::TN;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int K = UP ? a.width : a.ffp;
  const int N = UP ? (GATED ? 2 : 1) * a.ffp : a.width;
  // gate rows in one half of the tile, the same channels' up rows in the other
  constexpr bool PAIRS = UP && GATED;
  constexpr int CHANNELS = PAIRS ? TN / 2 : TN;
  const int n0 = nb * CHANNELS, n1 = UP ? a.ffp : a.width;
  const int panels = (n1 + CHANNELS - 1) / CHANNELS, nk = K / tile::KS;

  // the rows' pairs and weights, for the gather and the epilogue
  __shared__ int s_pair[TM];
  __shared__ float s_weight[TM];
  for (int r = threadIdx.x; r < TM; r += 512) {
    const int pair = a.perm[p0 + min(r, rows - 1)];
    s_pair[r] = pair;
    if constexpr (UP) s_weight[r] = a.weights[pair];
  }
  __syncthreads();

  // Where reading weights is what takes the time, column blocks start K at steps
  // of their own, so that what is asked for at a time is spread over the memory
  // channels (see rows_gemm.hip; the same block of an expert's other tiles starts
  // where this one does and meets it in L2).  Of shorter rows it is slower.  (us
  // without and with, for all of it: 32 experts of 1024 by 2048, four each, 400
  // rows 116 and 97, 1000 127 and 113, 2000 167 and 154; 16 of 3584 by 4096, two
  // each, 400 rows 287 and 270, 2000 468 and 440; but 64 of 1024 by 1024 102 and
  // 108; some more tiles than experts, 32 of 1024 by 2048, 2115 rows 191 and 179, but
  // three times as many, 6001 rows, 320 and 324.)
  P p;
  p.rows(
      [&](int r) {
        return uint32_t(UP ? s_pair[r] / a.top : p0 + min(r, rows - 1)) * K *
               2;
      },
      [&](int r) {
        const int c = min(n0 + r % CHANNELS, n1 - 1);
        return uint32_t(PAIRS ? c / 16 * 32 + c % 16 + r / CHANNELS * 16 : c) *
               K * 2;
      });
  p.run(static_cast<const char*>(UP ? a.h : a.act),
        static_cast<const char*>(UP ? a.w_up : a.w_down) +
            int64_t(e) * N * K * 2,
        nk, a.spread && nk >= 32 ? (e * panels + nb) % nk : 0, lds);

#pragma unroll
  for (int i = 0; i < MH; ++i) {
    float wt[2];
#pragma unroll
    for (int half = 0; half < 2; ++half)
      wt[half] = UP ? s_weight[half * TM / 2 + P::row_of(i)] : 0.f;
    const int tr = P::half_of() * TM / 2 + P::row_of(i);
    uint16_t* to = UP ? static_cast<uint16_t*>(a.act) + int64_t(p0 + tr) * a.ffp
                      : static_cast<uint16_t*>(a.y) +
                            int64_t(s_pair[tr]) * a.width;
#pragma unroll
    for (int b = 0; b < (PAIRS ? 1 : 2); ++b)
#pragma unroll
      for (int j = 0; j < NH; ++j) {
        uint2 v[2];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          f32x4_t f = p.acc[half][b][i][j];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if constexpr (PAIRS)
              f[r] = expert_gate<uint16_t>(f[r] * wt[half],
                                           p.acc[half][1][i][j][r] * wt[half],
                                           a.limit);
            else if constexpr (UP)
              f[r] = relu_squared(f[r]) * wt[half];
          }
          act_store4(reinterpret_cast<uint16_t*>(&v[half]), f);
        }
        const uint4 eight = P::eight(v[0], v[1]);
        const int col = n0 + P::eight_of(b, j);
        if (tr < rows && col < n1) *reinterpret_cast<uint4*>(to + col) = eight;
      }
  }
}

// Tiles that are up to half full take half the height.  They come last; where
// they are few and the CUs that full ones leave idle are not for most of them,
// they are half as wide as well, shared out over the chip.  (6001 rows of 2048 in
// 32 experts of 1024, four each, us for all of it: full ones only 345, half the
// height 336, and half the width 326.  8192 rows, 116 full tiles and 12 others,
// with half the width 434 and without 417: they run beside the last full ones.)
// Of 128 rows, all are half as wide where that many blocks are no more than CUs (8
// experts of 1024 by 2048, two each, 80 rows an expert 50 and 38; 4 of 512 by 1024 34
// and 27).
template <bool UP, int MH, int NH, bool GATED>
__global__ __launch_bounds__(512, 2)
void moe_tile_kernel(MoeArgs a, int n_blocks) {
  int tile, nb;
  TileKind kind;
  if (!tile_of<MH>(a, blockIdx.x, n_blocks, tile, nb, kind)) return;
  const int rows = a.tile_rows[tile];
  const int e = a.tile_expert[tile];
  const int p0 = a.tile_row0[tile];
  if (MH == 4 && kind == FULL && rows <= 128) kind = LOW;     // a.together
  if (kind == NARROW) moe_tile<UP, 2, NH / 2, GATED>(a, rows, e, p0, nb);
  else if (kind == LOW) moe_tile<UP, 2, NH, GATED>(a, rows, e, p0, nb);
  else moe_tile<UP, MH, NH, GATED>(a, rows, e, p0, nb);
}

template <typename T>
void route(const MoeArgs& a, hipStream_t st) {
  const dim3 grid((a.rows + 15) / 16), blk(512);
  if (a.routes <= 16)
    hipLaunchKernelGGL((moe_route_kernel<T, 1>), grid, blk, 0, st, a);
  else if (a.routes <= 32)
    hipLaunchKernelGGL((moe_route_kernel<T, 2>), grid, blk, 0, st, a);
  else if (a.routes <= 48)
    hipLaunchKernelGGL((moe_route_kernel<T, 3>), grid, blk, 0, st, a);
  else if (a.routes <= 64)
    hipLaunchKernelGGL((moe_route_kernel<T, 4>), grid, blk, 0, st, a);
  else if (a.routes <= 128)
    hipLaunchKernelGGL((moe_route_kernel<T, 8>), grid, blk, 0, st, a);
  else
    hipLaunchKernelGGL((moe_route_kernel<T, 16>), grid, blk, 0, st, a);
}

template <typename T>
void small(const MoeArgs& a, hipStream_t st) {
  if (a.gated)
    hipLaunchKernelGGL((moe_small_kernel<T, true, true>),
                       dim3(2 * a.ffp / 32, a.max_tiles), dim3(256), 0, st,
                       a);
  else
    hipLaunchKernelGGL((moe_small_kernel<T, true, false>),
                       dim3(a.ffp / 32, a.max_tiles), dim3(256), 0, st, a);
  hipLaunchKernelGGL((moe_small_kernel<T, false, false>),
                     dim3((a.width + 31) / 32, a.max_tiles), dim3(256), 0, st,
                     a);
}

template <bool UP, int MH, int NH, bool GATED>
void tiled_one(const MoeArgs& a, hipStream_t st) {
  using P = tile::Product<MH, NH>;
  const int nb =
      ((UP ? (GATED ? 2 : 1) * a.ffp : a.width) + P::TN - 1) / P::TN;
  // Two runs per XCD, each up to one block longer than its part, and of narrow
  // blocks two for one.
  const int blocks =
      (nb * a.max_tiles + 128 + 7) / 8 * 8 + 8;
  auto* k = moe_tile_kernel<UP, MH, NH, GATED>;
  if (P::LDS > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              int(P::LDS));
  hipLaunchKernelGGL(k, dim3(blocks), dim3(512), P::LDS, st, a, nb);
}

template <int MH>
void tiled(const MoeArgs& a, hipStream_t st) {
  if (a.gated) tiled_one<true, MH, 2, true>(a, st);
  else tiled_one<true, MH, 2, false>(a, st);
  tiled_one<false, MH, 2, false>(a, st);
}

}  // namespace

void launch_moe_route(const MoeArgs& a, hipStream_t st) {
  if (a.rows == 0) return;
  if (a.f32) route<float>(a, st);
  else route<uint16_t>(a, st);
}

void launch_moe_plan(const MoeArgs& a, hipStream_t st) {
  if (a.rows == 0) return;
  // whole workgroups of the router's
  const int each = std::max(PLAN_ROWS,
                            ((a.rows + PLAN_MOST - 1) / PLAN_MOST + 15) / 16 * 16);
  hipLaunchKernelGGL(moe_plan_kernel, dim3((a.rows + each - 1) / each),
                     dim3(256), 0, st, a, each);
}

void launch_moe_experts(const MoeArgs& a, hipStream_t st) {
  if (a.rows == 0) return;
  if (a.f32) {
    small<float>(a, st);
  } else if (a.tile_m == 16) {
    small<uint16_t>(a, st);
  } else {
    if (a.tile_m == 256) tiled<4>(a, st);
    else tiled<2>(a, st);
  }
}

}  // namespace rlli
