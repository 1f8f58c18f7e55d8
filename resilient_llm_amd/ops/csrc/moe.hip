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
//   moe_plan      (token, choice) pairs in expert order + row tiles; one
//                 workgroup for decode-sized batches, three small grids
//                 for prompts; no host round trip, so it is capturable
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

namespace rlli {
namespace {

// ------------------------------------------------------------- router
// Wave-wide reductions on the VALU, the result in every lane: rows of 16,
// then across rows, then out of the last lane.
template <int CTRL>
DEV_INLINE float dpp_or_own(float v) {
  const int b = __builtin_bit_cast(int, v);
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, false));
}
DEV_INLINE float last_lane(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
DEV_INLINE float wave_sum_dpp(float v) {
  v = group_sum_dpp<16>(v);
  // rows 0 + 1 | 2 + 3, then all four, in the last lane
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
           0, __builtin_bit_cast(int, v), 0x142, 0xa, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(
           0, __builtin_bit_cast(int, v), 0x143, 0xc, 0xf, false));
  return last_lane(v);
}
DEV_INLINE float wave_max_dpp(float v) {
  v = fmaxf(v, dpp_or_own<0x111>(v));     // row_shr 1, 2, 4, 8
  v = fmaxf(v, dpp_or_own<0x112>(v));
  v = fmaxf(v, dpp_or_own<0x114>(v));
  v = fmaxf(v, dpp_or_own<0x118>(v));
  v = fmaxf(v, dpp_or_own<0x142>(v));     // row_bcast 15, 31
  v = fmaxf(v, dpp_or_own<0x143>(v));
  return last_lane(v);
}

// 16 rows per workgroup, K split over eight waves
template <typename T, int ET>
__global__ __launch_bounds__(512)
void moe_route_kernel(MoeArgs a) {
  constexpr int E16 = ET * 16, NW = 8;
  __shared__ float part[NW][16][E16 + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane & 15, g = lane >> 4;
  const int row0 = blockIdx.x * 16;
  // the plan's counters, for the kernels after this one
  if (blockIdx.x == 0 && a.counters)
    for (int e = threadIdx.x; e < 2 * a.experts; e += 512) a.counters[e] = 0;
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
#pragma unroll
  for (int e = 0; e < ET; ++e)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      part[w][g * 4 + r][e * 16 + lr] = acc[e][r];
  __syncthreads();
  // each wave ranks two rows, lane l holding routes l, l + 64, ...
  constexpr int EL = (E16 + 63) / 64;
  constexpr float kNone = -INFINITY;      // cannot be chosen
  auto wave_fence = [] {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  for (int t = w * 2; t < w * 2 + 2; ++t) {
    const int row = row0 + t;
    if (row >= a.rows) break;
    float s[EL], choice[EL];
#pragma unroll
    for (int i = 0; i < EL; ++i) {
      const int e = i * 64 + lane;
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
      mx = wave_max_dpp(mx);
#pragma unroll
      for (int i = 0; i < EL; ++i) {
        s[i] = expf(s[i] - mx);           // 0 past the last route
        sum += s[i];
      }
      sum = wave_sum_dpp(sum);
#pragma unroll
      for (int i = 0; i < EL; ++i) s[i] /= sum;
    } else {
#pragma unroll
      for (int i = 0; i < EL; ++i) s[i] = 1.f / (1.f + expf(-s[i]));
    }
#pragma unroll
    for (int i = 0; i < EL; ++i) {
      const int e = i * 64 + lane;
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
        if (i * 64 + lane < a.routes) cs[i * 64 + lane] = choice[i];
      wave_fence();
      for (int g = lane; g < a.groups; g += 64) {
        float b = kNone;
        for (int e = g * size; e < (g + 1) * size; ++e) b = fmaxf(b, cs[e]);
        best[g] = b;
      }
      wave_fence();
      for (int g = lane; g < a.groups; g += 64) {
        int ahead = 0;
        for (int o = 0; o < a.groups; ++o)
          ahead += best[o] > best[g] || (best[o] == best[g] && o < g);
        stays[g] = ahead < a.keep ? 1.f : 0.f;
      }
      wave_fence();
#pragma unroll
      for (int i = 0; i < EL; ++i) {
        const int e = i * 64 + lane;
        if (e < a.routes && stays[e / size] == 0.f) choice[i] = kNone;
      }
    }
    float won[EL], total = 0.f;           // lane c & 63 keeps weight c
    for (int c = 0; c < a.top; ++c) {
      // the best score left, and the first route that has it
      float bv = choice[0];
#pragma unroll
      for (int i = 1; i < EL; ++i) bv = fmaxf(bv, choice[i]);
      bv = wave_max_dpp(bv);
      int bi = 0x7fffffff;
#pragma unroll
      for (int i = EL - 1; i >= 0; --i) {
        const uint64_t has = __ballot(choice[i] == bv);
        if (has) bi = i * 64 + __builtin_ctzll(has);
      }
#pragma unroll
      for (int i = 0; i < EL; ++i)
        if (i * 64 + lane == bi) choice[i] = kNone;
      bi = min(bi, a.routes - 1);       // a NaN row still names a route
      float mine = s[0];
#pragma unroll
      for (int i = 1; i < EL; ++i)
        if (bi >> 6 == i) mine = s[i];
      mine = __builtin_bit_cast(
          float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine),
                                           bi & 63));
      total += mine;
#pragma unroll
      for (int i = 0; i < EL; ++i)
        if (c == i * 64 + lane) won[i] = mine;
      if (lane == 0) a.ids[int64_t(row) * a.top + c] = bi;
    }
    const float scale = a.softmax ? 1.f / (total + 1e-20f) : 1.f;
#pragma unroll
    for (int i = 0; i < EL; ++i)
      if (i * 64 + lane < a.top)
        a.weights[int64_t(row) * a.top + i * 64 + lane] = won[i] * scale;
  }
}

// --------------------------------------------------------------- plan
constexpr int MAXE = 256;

// The tile list: tiles more than half full in expert order, then the other
// ones, so that the cheap tiles run where the last full ones leave compute
// units idle.  The counts of both follow the counters of the plan.
DEV_INLINE void write_tiles(const MoeArgs& a, const int* count,
                            const int* start, int tid, int nthr) {
  // index of expert e's first full tile, of its last one if that is not
  __shared__ int tfull[MAXE + 1], tpart[MAXE + 1];
  const int half = a.tile_m > 16 ? a.tile_m / 2 : 0;
  auto full = [&](int n) {
    return n / a.tile_m + (n % a.tile_m > half ? 1 : 0);
  };
  auto all = [&](int n) { return (n + a.tile_m - 1) / a.tile_m; };
  if (tid == 0) {
    int f = 0, p = 0;
    for (int e = 0; e < a.experts; ++e) {
      tfull[e] = f;
      tpart[e] = p;
      f += full(count[e]);
      p += all(count[e]) - full(count[e]);
    }
    tfull[a.experts] = f;
    tpart[a.experts] = p;
    a.counters[2 * a.experts] = f;
    a.counters[2 * a.experts + 1] = p;
  }
  __syncthreads();
  const int nfull = tfull[a.experts];
  for (int e = tid; e < a.experts; e += nthr)
    for (int i = 0; i < all(count[e]); ++i) {
      const int r = i * a.tile_m;
      const int t = i < full(count[e]) ? tfull[e] + i : nfull + tpart[e];
      a.tile_expert[t] = e;
      a.tile_row0[t] = start[e] + r;
      a.tile_rows[t] = min(a.tile_m, count[e] - r);
    }
  for (int t = nfull + tpart[a.experts] + tid; t < a.max_tiles; t += nthr)
    a.tile_rows[t] = 0;
}

__global__ __launch_bounds__(256)
void moe_plan_one_kernel(MoeArgs a) {
  __shared__ int count[MAXE], start[MAXE], cursor[MAXE];
  const int tid = threadIdx.x;
  const int P = a.rows * a.top;
  for (int e = tid; e < a.experts; e += 256) count[e] = 0;
  __syncthreads();
  for (int p = tid; p < P; p += 256)
    if (a.ids[p] < a.experts) atomicAdd(&count[a.ids[p]], 1);
  __syncthreads();
  if (tid == 0) {
    int s = 0;
    for (int e = 0; e < a.experts; ++e) {
      start[e] = s;
      cursor[e] = s;
      s += count[e];
    }
  }
  __syncthreads();
  for (int p = tid; p < P; p += 256)
    if (a.ids[p] < a.experts) a.perm[atomicAdd(&cursor[a.ids[p]], 1)] = p;
  write_tiles(a, count, start, tid, 256);
}

constexpr int PLAN_PAIRS = 2048;          // pairs per workgroup

__global__ __launch_bounds__(256)
void moe_count_kernel(MoeArgs a) {
  __shared__ int count[MAXE];
  const int tid = threadIdx.x;
  const int P = a.rows * a.top;
  const int p0 = blockIdx.x * PLAN_PAIRS;
  for (int e = tid; e < a.experts; e += 256) count[e] = 0;
  __syncthreads();
  for (int p = p0 + tid; p < min(P, p0 + PLAN_PAIRS); p += 256)
    if (a.ids[p] < a.experts) atomicAdd(&count[a.ids[p]], 1);
  __syncthreads();
  for (int e = tid; e < a.experts; e += 256)
    if (count[e]) atomicAdd(&a.counters[e], count[e]);
}

__global__ __launch_bounds__(256)
void moe_scatter_kernel(MoeArgs a) {
  __shared__ int count[MAXE], start[MAXE], total[MAXE], base[MAXE];
  const int tid = threadIdx.x;
  const int P = a.rows * a.top;
  const int p0 = blockIdx.x * PLAN_PAIRS;
  for (int e = tid; e < a.experts; e += 256) {
    total[e] = a.counters[e];
    count[e] = 0;
  }
  __syncthreads();
  if (tid == 0) {
    int s = 0;
    for (int e = 0; e < a.experts; ++e) {
      start[e] = s;
      s += total[e];
    }
  }
  for (int p = p0 + tid; p < min(P, p0 + PLAN_PAIRS); p += 256)
    if (a.ids[p] < a.experts) atomicAdd(&count[a.ids[p]], 1);
  __syncthreads();
  for (int e = tid; e < a.experts; e += 256)
    base[e] = start[e] +
              (count[e] ? atomicAdd(&a.counters[a.experts + e], count[e]) : 0);
  __syncthreads();
  for (int p = p0 + tid; p < min(P, p0 + PLAN_PAIRS); p += 256)
    if (a.ids[p] < a.experts) a.perm[atomicAdd(&base[a.ids[p]], 1)] = p;
  if (blockIdx.x == 0) write_tiles(a, total, start, tid, 256);
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
DEV_INLINE bool tile_of(const MoeArgs& a, int block, int n_blocks, int& tile,
                        int& nb) {
  const int x = block & 7;
  int s = block >> 3, n = a.counters[2 * a.experts], first = 0;
  int per = (n * n_blocks + 7) / 8;
  if (s >= per) {
    s -= per;
    first = n;
    n = a.counters[2 * a.experts + 1];
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
  static_assert(!GATED || NH % 2 == 0);
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int K = UP ? a.width : a.ffp;
  const int N = UP ? (GATED ? 2 : 1) * a.ffp : a.width;
  const int n0 = nb * TN;

  // the rows' pairs and weights, for the gather and the epilogue
  __shared__ int s_pair[TM];
  __shared__ float s_weight[TM];
  for (int r = threadIdx.x; r < TM; r += 512) {
    const int pair = a.perm[p0 + min(r, rows - 1)];
    s_pair[r] = pair;
    if constexpr (UP) s_weight[r] = a.weights[pair];
  }
  __syncthreads();

  P p;
  p.rows(
      [&](int r) {
        return uint32_t(UP ? s_pair[r] / a.top : p0 + min(r, rows - 1)) * K *
               2;
      },
      [&](int r) { return uint32_t(min(n0 + r, N - 1)) * K * 2; });
  p.run(static_cast<const char*>(UP ? a.h : a.act),
        static_cast<const char*>(UP ? a.w_up : a.w_down) +
            int64_t(e) * N * K * 2,
        K / tile::KS, lds);

  constexpr bool PAIRS = UP && GATED;
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
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int j = 0; j < NH; j += PAIRS ? 2 : 1) {
        uint2 v[2];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          f32x4_t f = p.acc[half][b][i][j];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            // blocks of 16 gate rows and their 16 up rows by turns
            if constexpr (PAIRS)
              f[r] = expert_gate<uint16_t>(
                  f[r] * wt[half], p.acc[half][b][i][j + 1][r] * wt[half],
                  a.limit);
            else if constexpr (UP)
              f[r] = relu_squared(f[r]) * wt[half];
          }
          act_store4(reinterpret_cast<uint16_t*>(&v[half]), f);
        }
        const uint4 eight = P::eight(v[0], v[1]);
        const int c = n0 + P::eight_of(b, j);
        const int col = PAIRS ? c / 32 * 16 + c % 16 : c;
        if (tr < rows && col < (UP ? a.ffp : a.width))
          *reinterpret_cast<uint4*>(to + col) = eight;
      }
  }
}

// Tiles that are up to half full take half the height (6001 rows of 2048 in 32
// experts of 1024, four each: 1.075 -> 1.130 times as fast as before both).
template <bool UP, int MH, int NH, bool GATED>
__global__ __launch_bounds__(512, 2)
void moe_tile_kernel(MoeArgs a, int n_blocks) {
  int tile, nb;
  if (!tile_of(a, blockIdx.x, n_blocks, tile, nb)) return;
  const int rows = a.tile_rows[tile];
  const int e = a.tile_expert[tile];
  const int p0 = a.tile_row0[tile];
  if (MH == 4 && rows <= 128) moe_tile<UP, 2, NH, GATED>(a, rows, e, p0, nb);
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
  // two runs per XCD, each up to one block longer than its part
  const int blocks = (nb * a.max_tiles + 7) / 8 * 8 + 8;
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
  const int P = a.rows * a.top;
  if (P == 0) return;
  if (P <= 2 * PLAN_PAIRS) {
    hipLaunchKernelGGL(moe_plan_one_kernel, dim3(1), dim3(256), 0, st, a);
    return;
  }
  const dim3 grid((P + PLAN_PAIRS - 1) / PLAN_PAIRS);
  hipLaunchKernelGGL(moe_count_kernel, grid, dim3(256), 0, st, a);
  hipLaunchKernelGGL(moe_scatter_kernel, grid, dim3(256), 0, st, a);
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
