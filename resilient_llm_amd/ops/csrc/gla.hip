// Gated linear recurrences: S_t = diag(alpha_t) S_{t-1} + k_t v_t^T,
// o_t = S_t^T q_t per head, alpha a decay per key channel, then RMS norm
// over the value width.  Three ways to make q, k and alpha from the
// projections:
//   GLA     q | k | v | gate | A1 h:  alpha = sigmoid(z)^(1/tau) with
//           z = A2 (A1 h) + b, q scaled by dim^-1/2, silu output gate
//   HGRN2   q | z | v:  alpha = l + (1 - l) sigmoid(z + b) with a lower
//           bound l per channel, k = 1 - alpha, q = silu(q), no gate
//   RWKV    alpha = e^(-e^z) with z = A2 tanh(A1 h) + b, silu output gate,
//           and o_t = S_{t-1}^T q_t + (q_t . u k_t) v_t: the past, and the
//           present through a bonus u per channel
//
// Projections arrive as GEMM output rows; everything from z on is
// 32-bit, matrix products included (f32 MFMA, or three 16-bit parts of each
// number in the scan), and so are the states.
//
// Decode is one fused kernel per layer: decay, state update, readout,
// norm and gate; a state is read and written exactly once.
//
// Prompts run in chunks of 64 tokens whose four 16-token sub-chunks bound
// every exponent: with L the running log-decay inside a sub-chunk, tot its
// last row and B_I the running log-decay at the start of sub-chunk I,
//     A[t,s] = sum_d (q_t e^{L_t} e^{B_I - B_{J+1}}) * (k_s e^{tot_J - L_s})
// for J < I has only exponents <= 0, whatever the decay.  Inside a
// sub-chunk the factors are e^{L_t - m} and e^{m - L_s} with m the middle
// row's log-decay, as long as either half decays by less than e^40; beyond
// that four-row blocks do the same once more.  RWKV's queries take the
// log-decay of the row before theirs, its diagonal is the bonus.
//   gla_intra   per (chunk, head): A, q e^{b_t}, k e^{b_C - b_s}, e^{b_C}
// then the scan and the gate of rec_scan.hip.

#include "rec_math.h"

#include <algorithm>
#include <type_traits>

namespace rlli {
namespace {

constexpr int C = kRecChunk;
constexpr float kSafeLog = 40.f;

// HGRN2: alpha = low + (1 - low) sigmoid(z), k = 1 - alpha without the
// cancellation
template <typename T>
DEV_INLINE float forget_key(float z, float low, float* alpha) {
  const float e = gexp<T>(-fabsf(z));
  const float r = grcp<T>(1.f + e), er = e * r;
  *alpha = low + (1.f - low) * (z >= 0.f ? r : er);
  return (1.f - low) * (z >= 0.f ? er : r);
}

// log alpha; e^-80 and less is nothing beside a key of order one
template <typename T>
DEV_INLINE float log_forget(float alpha, float k) {
  if constexpr (sizeof(T) == 2) return fmaxf(__logf(alpha), -80.f);
  return alpha > 0.5f ? log1pf(-k) : fmaxf(logf(alpha), -80.f);
}

// RWKV: log alpha; e^-80 is nothing
template <typename T>
DEV_INLINE float log_rwkv(float z) {
  return -fminf(gexp<T>(z), 80.f);
}

// ------------------------------------------------------------- decode
// One workgroup per sequence and head; what there is to do is to read and
// write the state, of which NT threads have U rows each in flight.  Few
// sequences leave a chain of round trips, so everything is asked for at once,
// what the decays are made from first and the state behind it, and nothing
// that was loaded decides what to load but the state's slot.  16 sequences of
// 8 heads of 128 x 256 with states in HBM: 13.9 us when the state was asked for
// after the decays, which one thread a channel made, now 11.7; 1 sequence 7.7
// and 6.8, 64 of them 34.3 and 31.3.
template <typename T, int KIND, int NT, int U>
__global__ __launch_bounds__(NT)
void gla_decode_kernel(GlaArgs a, bool vec_a2) {
  constexpr bool FG = KIND == kHgrn2, BONUS = KIND == kRwkv;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int seq = blockIdx.x, h = blockIdx.y;
  const int tid = threadIdx.x;
  // [dim] decay, key, query and (RWKV) bonus times key
  f32x4_t* chan = reinterpret_cast<f32x4_t*>(sm);
  float* red = sm + 4 * a.dpad;         // [rows][vpad] then sums
  const T* row = reinterpret_cast<const T*>(a.proj) + int64_t(seq) * a.stride;
  const int v4n = a.vpad / 4;
  const int n_rows = NT / v4n;
  const int vr = tid / v4n, vc = tid % v4n;
  const bool live = vr < n_rows;
  const bool fresh = a.positions[seq] == 0;
  float* S =
      a.state + (int64_t(a.slots[seq]) * a.heads + h) * a.dim * a.vpad;
  const auto at = [&](int d) {            // (1 MB at most)
    return reinterpret_cast<f32x4_t*>(S) + unsigned(d * v4n + vc);
  };
  const T* low = reinterpret_cast<const T*>(a.a1) + int64_t(seq) * a.a1_stride;
  const float qscale = BONUS ? 1.f : 1.f / sqrtf(float(a.dim));
  // 2^lg lanes a channel, as many as there are threads for, that take four
  // neighbouring elements of the rank at a time
  int lg = 0;
  if constexpr (!FG)
    while (lg < 4 && (a.dim << (lg + 1)) <= NT) ++lg;
  const int part = tid & ((1 << lg) - 1);
  struct Item {
    float q, k, b, x;
    f32x4_t w, l;
  };
  const auto load = [&](int i) {
    const int d = i >> lg, hc = h * a.dim + d;
    Item t;
    t.q = act_load(row + hc);
    t.k = act_load(row + a.off_k + hc);
    t.b = a.a2_bias[hc];
    if constexpr (FG) t.x = a.lower[hc];
    if constexpr (BONUS) t.x = a.bonus[hc];
    if constexpr (!FG) {
      if (vec_a2) {
        const int r = min(part * 4, a.rank - 4);
        t.w = act_load4(reinterpret_cast<const T*>(a.a2) +
                        int64_t(hc) * a.rank + r);
        t.l = act_load4(low + r);
      }
    }
    return t;
  };
  const auto finish = [&](int i, const Item& t) {
    const int d = i >> lg, hc = h * a.dim + d;
    if constexpr (FG) {
      float alpha;
      const float key = forget_key<T>(t.k + t.b, t.x, &alpha);
      chan[d] = f32x4_t{alpha, key, silu<T>(t.q), 0.f};
    } else {
      const T* w = reinterpret_cast<const T*>(a.a2) + int64_t(hc) * a.rank;
      const auto times = [](f32x4_t w4, f32x4_t l4) {
        float z = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          z += w4[j] * (BONUS ? gtanh<T>(l4[j]) : l4[j]);
        return z;
      };
      float z = 0.f;
      int r = part * 4;
      if (vec_a2) {
        if (r < a.rank) z = times(t.w, t.l);
        for (r += 4 << lg; r < a.rank; r += 4 << lg)
          z += times(act_load4(w + r), act_load4(low + r));
      } else {
        for (; r < a.rank; r += 4 << lg)
          for (int j = r; j < min(r + 4, a.rank); ++j)
            z += act_load(w + j) *
                 (BONUS ? gtanh<T>(act_load(low + j)) : act_load(low + j));
      }
      if (lg > 0) z += dpp_mov_f32<0xB1>(z);
      if (lg > 1) z += dpp_mov_f32<0x4E>(z);
      if (lg > 2) z += dpp_mov_f32<0x141>(z);
      if (lg > 3) z += dpp_mov_f32<0x140>(z);
      if (part == 0) {
        z += t.b;
        chan[d] = f32x4_t{
            BONUS ? expf(log_rwkv<T>(z)) : expf(log_sigmoid<T>(z) / a.tau),
            t.k, t.q * qscale, BONUS ? t.x * t.k : 0.f};
      }
    }
  };
  const Item first = load(min(tid, (a.dim << lg) - 1));
  f32x4_t v;
  const T* vp = row + a.off_v + h * a.vdim;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = act_load(vp + min(vc * 4 + j, a.vdim - 1));
  // the norm and the gate of the first columns
  const int e0 = min(tid, a.vdim - 1);
  float nw = a.norm[h * a.norm_stride + e0], gate = 0.f;
  if constexpr (!FG) gate = act_load(row + a.off_g + h * a.vdim + e0);
  f32x4_t s[U];
  // (without a condition, so that none of the waits above is for these)
  const auto ask = [&](int d0) {
#pragma unroll
    for (int u = 0; u < U; ++u)
      s[u] = *at(min(d0 + u * n_rows, a.dim - 1));
  };
  ask(vr);
  if (tid < a.dim << lg) finish(tid, first);
  for (int i = tid + NT; i < a.dim << lg; i += NT) finish(i, load(i));
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (vc * 4 + j >= a.vdim) v[j] = 0.f;
  __syncthreads();
  f32x4_t o = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // ALL: none of the rows is behind the last one
  const auto step = [&](int d0, auto all) {
    constexpr bool ALL = decltype(all)::value;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool mine = ALL || d0 + u * n_rows < a.dim;
      const int d = ALL ? d0 + u * n_rows : min(d0 + u * n_rows, a.dim - 1);
      const f32x4_t c = chan[d];
      if (fresh) s[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float before = s[u][j];
        s[u][j] = c[0] * before + c[1] * v[j];
        if (mine) o[j] += c[2] * (BONUS ? before + c[3] * v[j] : s[u][j]);
      }
      if (mine) *at(d) = s[u];
    }
  };
  if (live) {
    for (int d0 = vr; d0 < a.dim;) {
      if (d0 - vr + U * n_rows <= a.dim) step(d0, std::true_type{});
      else step(d0, std::false_type{});
      d0 += U * n_rows;
      if (d0 < a.dim) ask(d0);
    }
    *reinterpret_cast<f32x4_t*>(red + vr * a.vpad + vc * 4) = o;
  }
  __syncthreads();
  float ss = 0.f;
  for (int e = tid; e < a.vdim; e += NT) {
    float t = 0.f;
    for (int r = 0; r < n_rows; ++r) t += red[r * a.vpad + e];
    red[e] = t;                         // column e is this thread's alone
    ss += t * t;
  }
  __shared__ float ws[NT / 64];
  ss = wave_sum(ss);
  if ((tid & 63) == 0) ws[tid >> 6] = ss;
  __syncthreads();
  ss = 0.f;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) ss += ws[i];
  const float inv = 1.f / sqrtf(ss / a.vdim + a.eps);
  T* out = reinterpret_cast<T*>(a.out) + int64_t(seq) * a.out_stride +
           h * a.vdim;
  for (int e = tid; e < a.vdim; e += NT) {
    if (e != tid) {
      nw = a.norm[h * a.norm_stride + e];
      if constexpr (!FG) gate = act_load(row + a.off_g + h * a.vdim + e);
    }
    float o2 = red[e] * inv * nw;
    if constexpr (!FG) o2 *= silu<T>(gate);
    act_store(out + e, o2);
  }
}

// -------------------------------------------------------------- intra
// the running log-decay that a query sees: its own row's or, before the
// present row counts, the last one's (rows are lanes)
template <bool BEFORE>
DEV_INLINE float seen_log(float L) {
  if constexpr (BEFORE) return dpp_mov_f32<0x111>(L);
  return L;
}

// Waves w, w + 4, ... own sub-chunk w, NT 16-wide tiles of key columns each, lane
// l its row l & 15 and four neighbouring columns of a tile; MD bounds the tiles
// (dpad <= 64 * MD).  FULL: dim is 64 MD, the rank a multiple of 16 and rows are
// aligned, so that no load is conditional (rows behind the last one are loaded
// from it).  What bounds a workgroup is its waves' instructions, one after another
// as no other waves are there to run between them: 128 columns in one wave are
// some 10000 of them.
template <typename T, int KIND, int MD, int NT, bool FULL, bool PARTS>
__global__ __launch_bounds__(1024 * MD / NT)
void gla_intra_kernel(GlaArgs a, bool vec, bool vec_a) {
  constexpr bool FG = KIND == kHgrn2, BONUS = KIND == kRwkv;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  constexpr int Q = 4 * MD / NT;
  const int tile = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int w = wave & 3, part = wave >> 2, dt0 = part * NT;
  const int lr = lane & 15, g = lane >> 4;
  const int DP = FULL ? 64 * MD : a.dpad, LR = DP + 4, ndt = DP / 16;
  float* kl = sm;                        // [64][LR] keys, then decayed keys
  float* tot = kl + C * LR;              // [4][DP] log-decays of sub-chunks
  float* EB = tot + 4 * DP;              // [3][DP] e^{B_w}, w = 1 .. 3
  float* ED = EB + 3 * DP;               // [3][DP] e^{B_4 - B_{w+1}}, w < 3
  float* EJ = ED + 3 * DP;               // [3][DP] sub-chunks in between
  const int row0 = a.tiles[tile];
  const int n = a.tiles[2 * a.n_tiles + tile];
  const int trow = w * 16 + lr;          // this lane's row
  const bool row_ok = trow < n;
  const int64_t at = row0 + (FULL ? min(trow, n - 1) : trow);
  const T* qrow = reinterpret_cast<const T*>(a.proj) + at * a.stride +
                  h * a.dim;
  auto row4 = [&](const T* p, int d, int width, bool v) {
    if constexpr (FULL) return act_load4(p + d);
    else return load4_guard(p, d, width, row_ok, v);
  };
  auto vec4 = [&](const float* p, int d) {
    if constexpr (FULL) return *reinterpret_cast<const f32x4_t*>(p + d);
    else return load4_guard(p, d, a.dim, true, a.dim % 4 == 0);
  };
  const T* krow = qrow + a.off_k;
  const float* bias = a.a2_bias + h * a.dim;
  const float* low = FG ? a.lower + h * a.dim : nullptr;
  const float qscale = 1.f / sqrtf(float(a.dim));

  // queries and the running log-decay stay in registers, keys in LDS
  f32x4_t q[NT], L[NT];
  float wmin = 0.f;
  // (raw keys wait in the registers of the log-decays)
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    if (!FULL && dt0 + i >= ndt) continue;
    const int d = (dt0 + i) * 16 + g * 4;
    q[i] = row4(qrow, d, a.dim, vec);
    L[i] = row4(krow, d, a.dim, vec);
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int dt = dt0 + i;
    if (!FULL && dt >= ndt) continue;
    const int d = dt * 16 + g * 4;
    f32x4_t k = L[i];
    if constexpr (FULL && !FG)
      if (!row_ok) k = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const f32x4_t bv = vec4(bias, d);
    if constexpr (FG) {
      const f32x4_t lv = vec4(low, d);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool ok = row_ok && d + j < a.dim;
        float alpha;
        const float kk = forget_key<T>(k[j] + bv[j], lv[j], &alpha);
        k[j] = ok ? kk : 0.f;
        L[i][j] = ok ? log_forget<T>(alpha, kk) : 0.f;
        q[i][j] = silu<T>(q[i][j]);
      }
    } else {
      // z transposed: columns down, rows across the lanes
      f32x4_t z = f32x4_t{0.f, 0.f, 0.f, 0.f};
      const T* a1 = reinterpret_cast<const T*>(a.a1) + at * a.a1_stride;
      const T* a2 = reinterpret_cast<const T*>(a.a2) +
                    int64_t(h * a.dim + dt * 16 + lr) * a.rank;
      for (int k0 = 0; k0 < a.rank; k0 += 16) {
        f32x4_t av = row4(a1, k0 + g * 4, a.rank, vec_a);
        if constexpr (BONUS)
#pragma unroll
          for (int j = 0; j < 4; ++j) av[j] = gtanh<T>(av[j]);
        f32x4_t wv;
        if constexpr (FULL) wv = act_load4(a2 + k0 + g * 4);
        else wv = load4_guard(a2, k0 + g * 4, a.rank, dt * 16 + lr < a.dim,
                              vec_a);
#pragma unroll
        for (int j = 0; j < 4; ++j) z = mma4(wv[j], av[j], z);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool ok = row_ok && d + j < a.dim;
        const float lw = BONUS ? log_rwkv<T>(z[j] + bv[j])
                               : log_sigmoid<T>(z[j] + bv[j]) / a.tau;
        L[i][j] = ok ? lw : 0.f;
        if constexpr (!BONUS) q[i][j] *= qscale;
      }
    }
    *reinterpret_cast<f32x4_t*>(kl + trow * LR + d) = k;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      L[i][j] = row_prefix(L[i][j]);
      const float mid = __shfl(L[i][j], g * 16 + 7, kWave);
      if (lr == 15) {
        tot[w * DP + d + j] = L[i][j];
        wmin = fminf(wmin, fminf(mid, L[i][j] - mid));
      }
    }
  }
  const bool safe = __all(wmin > -kSafeLog);
  auto seen = [&](float Lt) { return seen_log<BONUS>(Lt); };
  float own = 0.f;                       // this row's diagonal
  if constexpr (BONUS) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      if (!FULL && dt0 + i >= ndt) continue;
      const int d = (dt0 + i) * 16 + g * 4;
      const f32x4_t kv = *reinterpret_cast<const f32x4_t*>(kl + trow * LR + d);
      const f32x4_t uv = vec4(a.bonus + h * a.dim, d);
#pragma unroll
      for (int j = 0; j < 4; ++j) own += q[i][j] * uv[j] * kv[j];
    }
    own += __shfl_xor(own, 16, kWave);
    own += __shfl_xor(own, 32, kWave);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < DP; d += blockDim.x) {
    float t[4], b = 0.f;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      t[s] = tot[s * DP + d];
      if (s > 0) EB[(s - 1) * DP + d] = gexp<T>(b);
      b += t[s];
    }
    a.dec[(int64_t(tile) * a.heads + h) * DP + d] = expf(b);
    float after = 0.f;
#pragma unroll
    for (int s = 3; s >= 0; --s) {
      if (s < 3) ED[s * DP + d] = gexp<T>(after);
      after += t[s];
    }
    EJ[d] = gexp<T>(t[1]);                // from 0 to 2
    EJ[DP + d] = gexp<T>(t[1] + t[2]);    // from 0 to 3
    EJ[2 * DP + d] = gexp<T>(t[2]);       // from 1 to 3
  }
  f32x4_t acc[4];
#pragma unroll
  for (int J = 0; J < 4; ++J) acc[J] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if (!safe) {
    // steep decay: four-row blocks.  Block pairs a > b factor around the
    // row before a, so every exponent is <= 0; inside a block the three
    // distances are summed lane by lane.
    float near[4] = {0.f, 0.f, 0.f, 0.f};  // row lr and the row so far back
    f32x4_t far = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      if (!FULL && dt0 + i >= ndt) continue;
      const f32x4_t k = *reinterpret_cast<const f32x4_t*>(
          kl + trow * LR + (dt0 + i) * 16 + g * 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float Lt = L[i][j], Lq = seen(Lt), qv = q[i][j], kv = k[j];
        float ref[4];
#pragma unroll
        for (int b = 1; b < 4; ++b)
          ref[b] = __shfl(Lt, g * 16 + 4 * b - 1, kWave);
        const int blk = lr >> 2;
        const float mine = blk == 3 ? ref[3] : blk == 2 ? ref[2] : ref[1];
        const float qa = blk > 0 ? qv * gexp<T>(Lq - mine) : 0.f;
#pragma unroll
        for (int b = 1; b < 4; ++b)
          far = mma4(blk == b ? qa : 0.f,
                     lr < 4 * b ? kv * gexp<T>(ref[b] - Lt) : 0.f, far);
        if constexpr (!BONUS) near[0] += qv * kv;
        near[1] += qv * dpp_mov_f32<0x111>(kv) *
                   gexp<T>(fminf(Lq - dpp_mov_f32<0x111>(Lt), 0.f));
        near[2] += qv * dpp_mov_f32<0x112>(kv) *
                   gexp<T>(fminf(Lq - dpp_mov_f32<0x112>(Lt), 0.f));
        near[3] += qv * dpp_mov_f32<0x113>(kv) *
                   gexp<T>(fminf(Lq - dpp_mov_f32<0x113>(Lt), 0.f));
      }
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      near[x] += __shfl_xor(near[x], 16, kWave);
      near[x] += __shfl_xor(near[x], 32, kWave);
    }
    if constexpr (BONUS) near[0] = own;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const float v = __shfl(near[x], g * 4 + r, kWave);
        if (lr >> 2 == g && g * 4 + r - lr == x) far[r] = v;
      }
#pragma unroll
    for (int J = 0; J < 4; ++J)
      if (J == w) acc[J] = far;
  }
  __syncthreads();

  // this wave's own rows: q e^{L}, k e^{tot - L} and the diagonal block
  const int64_t ch = int64_t(tile) * a.heads + h;
  const int nks = (ndt + 1) / 2;
  float* qd = static_cast<float*>(a.qd) + ch * C * DP;
  float* kd = static_cast<float*>(a.kd) + ch * DP * C;
  uint16_t* qp = static_cast<uint16_t*>(a.qd) + ch * nks * 6144;
  uint16_t* kp = static_cast<uint16_t*>(a.kd) + ch * ndt * 3072;
  uint2 qh[2][3];
  auto put_q = [&](int ks) {
#pragma unroll
    for (int p = 0; p < 3; ++p)
      *reinterpret_cast<uint4*>(qp + (((ks * 4 + w) * 3 + p) * 64 + lane) * 8) =
          uint4{qh[0][p].x, qh[0][p].y, qh[1][p].x, qh[1][p].y};
  };
  // the lane whose operand this lane has once it is transposed
  const int turned = (lr >> 2) * 16 + g * 4 + (lr & 3);
  f32x4_t diag = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int dt = dt0 + i;
    if (!FULL && dt >= ndt) continue;
    const int d = dt * 16 + g * 4;
    const f32x4_t tw = *reinterpret_cast<const f32x4_t*>(tot + w * DP + d);
    f32x4_t eb = f32x4_t{1.f, 1.f, 1.f, 1.f}, ed = eb;
    if (w > 0) eb = *reinterpret_cast<const f32x4_t*>(EB + (w - 1) * DP + d);
    if (w < 3) ed = *reinterpret_cast<const f32x4_t*>(ED + w * DP + d);
    f32x4_t kt = *reinterpret_cast<const f32x4_t*>(kl + trow * LR + d), qo, ko;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float Lt = L[i][j];
      if (safe) {
        const float Lm = __shfl(Lt, g * 16 + 7, kWave);
        diag = mma4(q[i][j] * gexp<T>(seen(Lt) - Lm),
                    kt[j] * gexp<T>(Lm - Lt), diag);
      }
      q[i][j] *= gexp<T>(seen(Lt));
      qo[j] = q[i][j] * eb[j];
      kt[j] *= gexp<T>(tw[j] - Lt);
      ko[j] = kt[j] * ed[j];
    }
    ko = quad_transposed(ko);
    if constexpr (PARTS) {
      three_parts(qo, qh[i & 1]);
      if (i & 1) put_q(dt / 2);
      uint2 kh[3];
      three_parts(ko, kh);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<uint2*>(
            kp + (((dt * 2 + w / 2) * 3 + p) * 64 + turned) * 8 + w % 2 * 4) =
            kh[p];
    } else {
      *reinterpret_cast<f32x4_t*>(qd + ((dt * 4 + w) * 64 + lane) * 4) = qo;
      *reinterpret_cast<f32x4_t*>(kd + ((dt * 4 + w) * 64 + turned) * 4) = ko;
    }
    *reinterpret_cast<f32x4_t*>(kl + trow * LR + d) = kt;
  }
  if (PARTS && !FULL && ndt % 2 && (ndt - 1) / NT == part) {
#pragma unroll
    for (int p = 0; p < 3; ++p) qh[1][p] = uint2{0, 0};
    put_q(ndt / 2);
  }
  if (safe) {
    if constexpr (BONUS)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = __shfl(own, g * 4 + r, kWave);
        if (g * 4 + r == lr) diag[r] = v;
      }
#pragma unroll
    for (int J = 0; J < 4; ++J)
      if (J == w) acc[J] = diag;
  }
  __syncthreads();
  // rows of the sub-chunks before
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    const int dt = dt0 + i;
    if (!FULL && dt >= ndt) continue;
    const int d = dt * 16 + g * 4;
#pragma unroll
    for (int J = 0; J < 3; ++J) {
      if (J >= w) break;
      f32x4_t qe = q[i];
      if (J + 1 < w) {
        const f32x4_t e = *reinterpret_cast<const f32x4_t*>(
            EJ + (J == 1 ? 2 : w - 2) * DP + d);
#pragma unroll
        for (int j = 0; j < 4; ++j) qe[j] *= e[j];
      }
      const f32x4_t kt =
          *reinterpret_cast<const f32x4_t*>(kl + (J * 16 + lr) * LR + d);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[J] = mma4(qe[j], kt[j], acc[J]);
    }
  }
  // the waves' sums meet, in order; a wave finishes every Q-th tile
  f32x4_t* sums = reinterpret_cast<f32x4_t*>(sm) + lane;
  if constexpr (Q > 1) {
    __syncthreads();
#pragma unroll
    for (int J = 0; J < 4; ++J)
      if (J <= w) sums[(part * 10 + w * (w + 1) / 2 + J) * 64] = acc[J];
    __syncthreads();
  }
  float* sc = static_cast<float*>(a.sc) + ch * C * C;
  uint16_t* sp = static_cast<uint16_t*>(a.sc) + ch * 12288;
#pragma unroll
  for (int J = 0; J < 4; ++J) {
    if (J > (PARTS ? w | 1 : w)) break;    // (a pair's second tile: zeros)
    if (J % Q != part) continue;
    f32x4_t v = acc[J];
    if constexpr (Q > 1) {
      v = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (J <= w)
#pragma unroll
        for (int i = 0; i < Q; ++i)
          v += sums[(i * 10 + w * (w + 1) / 2 + J) * 64];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (J > w || (J == w && lr > g * 4 + r)) v[r] = 0.f;
    v = quad_transposed(v);
    if constexpr (PARTS) {
      uint2 h[3];
      three_parts(v, h);
#pragma unroll
      for (int p = 0; p < 3; ++p)
        *reinterpret_cast<uint2*>(
            sp + (((w * 2 + J / 2) * 3 + p) * 64 + turned) * 8 + J % 2 * 4) =
            h[p];
    } else {
      *reinterpret_cast<f32x4_t*>(sc + ((w * 4 + J) * 64 + turned) * 4) = v;
    }
  }
}

template <typename T, int KIND>
void prefill(const GlaArgs& a, hipStream_t st) {
  const bool vec = a.dim % 4 == 0 && a.stride % 4 == 0 && a.off_k % 4 == 0 &&
                   reinterpret_cast<uintptr_t>(a.proj) % (4 * sizeof(T)) == 0;
  const bool vec_a = a.rank % 4 == 0 && a.a1_stride % 4 == 0 &&
                     reinterpret_cast<uintptr_t>(a.a1) % (4 * sizeof(T)) == 0;
  auto intra = [&](auto* k, int waves) {
    // keys and decays, then the waves' sums
    const size_t smem =
        std::max(size_t(C * (a.dpad + 4) + 13 * a.dpad) * sizeof(float),
                 size_t(waves / 4) * 10 * 64 * sizeof(f32x4_t));
    if (smem > 65536)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(smem));
    hipLaunchKernelGGL(k, dim3(a.n_tiles, a.heads), dim3(64 * waves), smem, st,
                       a, vec, vec_a);
  };
  const bool parts = gla_parts(a);
  auto by_parts = [&](auto md, auto full) {
    constexpr int MD = decltype(md)::value;
    constexpr bool FULL = decltype(full)::value;
    auto by_tiles = [&](auto nt) {
      constexpr int NT = decltype(nt)::value;
      if constexpr (sizeof(T) == 4)
        intra(gla_intra_kernel<T, KIND, MD, NT, FULL, false>, 16 * MD / NT);
      else if (parts)
        intra(gla_intra_kernel<T, KIND, MD, NT, FULL, true>, 16 * MD / NT);
      else
        intra(gla_intra_kernel<T, KIND, MD, NT, FULL, false>, 16 * MD / NT);
    };
    // Columns of a wave: 32 of heads of up to 128, 64 of wider ones, but of 128
    // twice as many where workgroups are more than CUs.  (us by columns of a wave,
    // all of them last, and workgroups: heads of 128, 32, 64 and 128 columns, 16:
    // 14.4, 17.1 and 24.8, 256: 19.1, 20.7 and 27.4, 328: 31.0, 28.9 and 33.5, 960:
    // 65.3, 59.8 and 63.5; of 64, 32: 11.2 and 15.0, 1920: 44.5 and 49.3; of 256,
    // 64 columns, 16: 28 and 65, 960: 127 and 159.)
    if constexpr (MD == 4)
      by_tiles(std::integral_constant<int, 4>{});
    else if (MD == 1 || a.n_tiles * a.heads <= 256)
      by_tiles(std::integral_constant<int, 2>{});
    else
      by_tiles(std::integral_constant<int, 2 * MD>{});
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I4 = std::integral_constant<int, 4>;
  // without a conditional load where sizes allow (GLA, 4 sequences of 1.9k, 8 heads
  // of 128 x 256: 57 and 50 us)
  bool done = false;
  if constexpr (sizeof(T) == 2 && KIND != kHgrn2) {
    done = vec && vec_a && a.rank % 16 == 0 && (a.dim == 64 || a.dim == 128) &&
           reinterpret_cast<uintptr_t>(a.a2) % 8 == 0;
    if (done && a.dim == 64) by_parts(I1{}, std::true_type{});
    else if (done) by_parts(I2{}, std::true_type{});
  }
  if (done) {
  } else if (a.dpad <= 64) {
    by_parts(I1{}, std::false_type{});
  } else if (a.dpad <= 128) {
    by_parts(I2{}, std::false_type{});
  } else {
    by_parts(I4{}, std::false_type{});
  }
  ScanArgs sa{};
  sa.v = reinterpret_cast<const T*>(a.proj) + a.off_v;
  sa.v_stride = a.stride;
  sa.qd = a.qd;
  sa.kt = a.kd;
  sa.sc = a.sc;
  sa.dec = a.dec;
  sa.state = a.state;
  sa.o = a.o;
  sa.tiles = a.tiles;
  sa.seqs = a.seqs;
  sa.n_rows = a.rows;
  sa.n_tiles = a.n_tiles;
  sa.n_seqs = a.n_seqs;
  sa.heads = a.heads;
  sa.group = 1;
  sa.dim = a.dim;
  sa.dpad = a.dpad;
  sa.vdim = sa.cols = sa.opad = a.vdim;
  sa.vpad = a.vpad;
  sa.mode = kScanPlain;
  sa.f32 = a.f32;
  sa.parts = parts;
  launch_rec_scan(sa, st);
  RecGateArgs ga{};
  ga.o = a.o;
  ga.gate = reinterpret_cast<const T*>(a.proj) + a.off_g;
  ga.gate_stride = a.stride;
  ga.norm = a.norm;
  ga.norm_stride = a.norm_stride;
  ga.out = a.out;
  ga.out_stride = a.out_stride;
  ga.rows = a.rows;
  ga.heads = a.heads;
  ga.vdim = ga.opad = a.vdim;
  ga.kind = KIND == kHgrn2 ? kGateNone : kGateSilu;
  ga.eps = a.eps;
  ga.f32 = a.f32;
  launch_rec_gate(ga, st);
}

template <typename F>
void by_kind(const GlaArgs& a, F f) {
  auto go = [&](auto t) {
    if (a.kind == kHgrn2) f(t, std::integral_constant<int, kHgrn2>{});
    else if (a.kind == kRwkv) f(t, std::integral_constant<int, kRwkv>{});
    else f(t, std::integral_constant<int, kGla>{});
  };
  if (a.f32) go(float{});
  else go(uint16_t{});
}

}  // namespace

// The scan's operands in parts where the activations are 16-bit ones: fewer steps
// of each chunk's chain, and half as many bytes more, which cost more than they
// give where the chip is full (`many` heads) or few narrow blocks stream `much`.
// Whole prompts, time in f32 over time in parts (heads of all sequences and rows of
// each; two MI355X differ by up to 0.08):
//   64 x 64     512 heads 0.89; 64, 2000 rows 0.90; 32, 4000 rows 1.01; 16, 4000
//               rows 1.37, 8000 rows 1.04 to 1.14, left to f32; 256, 250 rows 1.11
//   64 x 128    16, 8000 rows 1.15; 64, 2000 rows 1.00; 256, 500 rows 0.98
//   64 x 256    32, 3200 rows 1.23; 64, 2000 rows 1.25; 256, 500 rows 0.97
//   128 x 64    32, 500 rows 1.15; 64, 256 rows 1.09, 512 rows 0.91 to 0.99, 1000 rows
//               0.99, 1600 rows 0.91; 128, 250 rows 1.06, 500 rows 0.99, 1000 rows
//               0.93
//   128 x 128   16, 2048 rows 1.11, 8000 rows 1.17; 64, 1600 rows 1.10; 128, 1000
//               rows 1.16; 256, 512 rows 1.01; 480, 500 rows 0.98; 512 0.91
//   128 x 256   8, 12500 rows 1.27; 16, 7000 rows 1.18; 32, 3500 rows 1.32; 256, 400
//               rows 1.12; 512, 250 rows 1.14, 400 rows 1.04
//   256 x 256   16, 8000 rows 1.23; 64 1.62; 128 1.07; 256 0.74
//   256 x 128   16, 8000 rows 1.24; 64 1.40; 128 1.14; 256 0.77
//   256 x 64    32, 4000 rows 1.12; 64, 1600 rows 1.00; 256 heads 1.03; 512 0.80 to
//               0.86
// Parts are the closer ones on both sides of these lines: of 29 such prompts of GLA,
// 10 of RWKV and 12 of HGRN2, of up to 12500 rows, the state's error against 64 bits
// was 0.54 to 0.79, 0.59 to 0.63 and 0.98 to 1.00 of that of f32 products; of outputs
// it was the same to five places, and 0.5 to 1.02 as many were not the nearest
// 16-bit number.
bool gla_parts(const GlaArgs& a) {
  if (a.f32) return false;
  const int64_t sh = int64_t(a.n_seqs) * a.heads;
  const int64_t blocks = sh * ((a.vdim + 63) / 64);
  if (a.dpad <= 64 && blocks >= 512) return false;
  const bool many = sh > 128 && blocks >= 512;
  const bool much = int64_t(a.rows) * a.heads >= (sh < 512 ? 3 << 15 : 3 << 14);
  if (a.dpad > 128) return !many;
  if (a.vdim <= 64) return !(much && (many || blocks <= 128));
  return !(much && many && a.vdim <= 128);
}

void launch_gla_decode(const GlaArgs& a, hipStream_t st) {
  if (a.rows == 0) return;
  // 512 threads for states of 64 KB and more where each can have a CU of its
  // own (us with 256, 512 and 1024 threads, states in HBM; heads of 128 x 256:
  // 8 of them 8.3, 6.8 and 7.0, 128 of them 13.6, 11.7 and 11.6, 512 of them
  // 31.3, 30.5 and 33.1; of 128 x 128: 5.9, 5.3 and 6.9, 8.8, 7.9 and 9.3, 19.5,
  // 19.4 and 23.0; of 64 x 128: 128 of them 5.7, 6.5 and 8.0).  The readout sums
  // rows in another order with them, so that its last bits depend on the batch.
  const bool wide = int64_t(a.dim) * a.vpad >= 128 * 128 &&
                    int64_t(a.rows) * a.heads <= 256;
  const int n_rows = (wide ? 512 : 256) / (a.vpad / 4);
  const size_t smem =
      size_t(4 * a.dpad + n_rows * a.vpad) * sizeof(float);
  by_kind(a, [&](auto t, auto kind) {
    using T = decltype(t);
    constexpr int KIND = decltype(kind)::value;
    // four elements of the rank at a time where all rows of both factors lie
    // for it, otherwise one
    const size_t four = 4 * sizeof(T);
    const bool vec = a.rank >= 4 && a.rank % 4 == 0 && a.a1_stride % 4 == 0 &&
                     reinterpret_cast<uintptr_t>(a.a1) % four == 0 &&
                     reinterpret_cast<uintptr_t>(a.a2) % four == 0;
    const dim3 grid(a.rows, a.heads);
    const auto run = [&](auto nt, auto u) {
      constexpr int NT = decltype(nt)::value, U = decltype(u)::value;
      hipLaunchKernelGGL((gla_decode_kernel<T, KIND, NT, U>), grid, dim3(NT),
                         smem, st, a, vec);
    };
    using std::integral_constant;
    // four rows a thread where that is all of them, so that none is asked for
    // twice (1536 heads of 64 x 64: 18.3 us with eight, 15.6 with four)
    if (wide) run(integral_constant<int, 512>{}, integral_constant<int, 8>{});
    else if (a.dim <= 4 * n_rows)
      run(integral_constant<int, 256>{}, integral_constant<int, 4>{});
    else run(integral_constant<int, 256>{}, integral_constant<int, 8>{});
  });
}

void launch_gla_prefill(const GlaArgs& a, hipStream_t st) {
  if (a.rows == 0 || a.n_seqs == 0) return;
  by_kind(a, [&](auto t, auto kind) {
    prefill<decltype(t), decltype(kind)::value>(a, st);
  });
}

}  // namespace rlli
