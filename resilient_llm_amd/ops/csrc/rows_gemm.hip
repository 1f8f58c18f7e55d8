// Products of few rows with a weight matrix, as decoding has them:
// y[M, N] = x[M, K] w[N, K]^T, M <= 128, bf16 with f32 sums.
//
// What there is to do is to read w once; everything else has to stay out of
// its way.  A workgroup has 64 (or 128) rows of w over a range of K, four
// waves with 16 (32) of them each, and walks 64-wide steps of K through a
// ring in LDS that direct global -> LDS loads fill R - 1 steps ahead: 32 to
// 64 KB of w are under way per CU whatever the waves do, which is what the
// latency of memory at its full rate asks for.  Rows of w arrive in whole
// 128-byte lines; the 16-byte pieces of a line are swizzled by the row, so
// that the matrix operand's reads (one piece of sixteen rows) are free of
// bank conflicts.  x comes along in the same ring and is shared by the waves.
// Rows are a power of two apart more often than not, so the lines of one step
// lie on few memory channels: each workgroup starts its walk at a step of its
// own, which spreads what is asked for at a time over all of them (28672 rows
// of 4096: 43.7 -> 36 us).
//
// Where 64-row panels are fewer than the CUs, K is divided as well, and the
// parts are written in f32, [splits, M, N], for whoever reads the product to
// sum; in order, so a result does not depend on when workgroups run.  Nor
// does it depend on M, up to 64 rows and from there on: the order of sums
// follows from N and K alone.

#include "common.h"
#include "decode_parts.h"
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace rlli {

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// streams and gains may start at any float
typedef f32x4 f32x4_any __attribute__((aligned(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));

constexpr int KS = 64;            // a step of K: one 128-byte line of a row
constexpr int LINE = KS;          // elements

enum { OUT_PARTS = 0, OUT_BF16 = 1, OUT_SILU = 2 };

DEV_INLINE uint32_t pack2(float a, float b) {
  const b16x2 v = __builtin_convertvector((f32x2{a, b}), b16x2);
  return __builtin_bit_cast(uint32_t, v);
}

template <int AUX>
DEV_INLINE void lds_load16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)g,
      (__attribute__((address_space(3))) void*)l, 16, 0, AUX);
}

template <int N>
DEV_INLINE void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// all but the newest L * left loads have landed
template <int L, int MOST>
DEV_INLINE void wait_steps(int left) {
  if constexpr (MOST == 0) {
    wait_vm<0>();
  } else {
    if (left >= MOST) wait_vm<L * MOST>();
    else wait_steps<L, MOST - 1>(left);
  }
}

// ---- the norm ahead of a product ----------------------------------------
// Of a single row, what a norm reads is so little that every workgroup of the
// product behind it can make x for itself: the residual plus the sum of an
// earlier product's f32 parts, normed, in LDS, by four more waves while the
// others' first steps of w are under way.  What bounds it is the time to that
// read's data.  us, norm and product apart and in one, gaps between launches
// included, with weights that no cache holds and as many parts as a step has:
// 6144 x 4096 parts 15.5 and 13.2, 28672 x 4096 with silu 42.3 and 40.0, 3072 x
// 2048 7.4 and 5.3, 16384 x 2048 with silu 15.9 and 13.8.  (A thread asks for
// eight pieces of the parts at a time, four of K beyond 4096 in each: 6144 x 5120
// with two parts 16.7 and 14.6, with eight 17.3 and 18.3; products of as many
// columns come in three at most.  Two rows read twice as much: 2 us slower than
// apart.  Rows made once and handed to the other workgroups through memory: 2 us
// slower as well, five trips to memory while it is busy with weights.)
struct NormArgs {
  const float* parts;          // [n, K]
  const uint16_t* residual;    // [K]
  uint16_t* residual_out;      // residual + sum of the parts
  const uint16_t* gain;        // [K]
  int n;
  float eps;
};

// loads into LDS stay under way
DEV_INLINE void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The row by 256 threads, NCH pieces of 8 elements each.  All of the
// workgroup's waves pass two barriers: behind the first, what is read here has
// been asked for, ahead of the weights, behind which it would wait for 1 to 3
// us more.
template <int NCH>
DEV_INLINE void norm_row(const NormArgs& a, int K, int t, float* sums,
                         uint16_t* xs) {
  constexpr int B = 8 / NCH;              // parts whose loads are one batch
  uint4 r[NCH], gain[NCH];
  float4 first[B][NCH][2];
  float v[NCH][8];
  int at[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) at[c] = min((c * 256 + t) * 8, K - 8);
#pragma unroll
  for (int s = 0; s < B; ++s)
    if (s < a.n)
#pragma unroll
      for (int c = 0; c < NCH; ++c)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          first[s][c][i] = *reinterpret_cast<const float4*>(
              a.parts + int64_t(s) * K + at[c] + i * 4);
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    r[c] = *reinterpret_cast<const uint4*>(a.residual + at[c]);
    gain[c] = *reinterpret_cast<const uint4*>(a.gain + at[c]);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[c][i] = 0.f;
  }
  lds_barrier();
  auto add = [&](int c, const float4& x, const float4& y) {
    v[c][0] += x.x; v[c][1] += x.y; v[c][2] += x.z; v[c][3] += x.w;
    v[c][4] += y.x; v[c][5] += y.y; v[c][6] += y.z; v[c][7] += y.w;
  };
#pragma unroll
  for (int s = 0; s < B; ++s)
    if (s < a.n)
#pragma unroll
      for (int c = 0; c < NCH; ++c) add(c, first[s][c][0], first[s][c][1]);
#pragma unroll(B)
  for (int s = B; s < a.n; ++s)
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const float* q = a.parts + int64_t(s) * K + at[c];
      add(c, *reinterpret_cast<const float4*>(q),
          *reinterpret_cast<const float4*>(q + 4));
    }
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    bf16x8 o;
    o.u = r[c];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      o.s[i] = f32_to_bf16(v[c][i] + bf16_to_f32(o.s[i]));
      const float f = bf16_to_f32(o.s[i]);    // x is of the stored residual
      if ((c * 256 + t) * 8 < K) ss += f * f;
    }
    r[c] = o.u;
  }
  ss = wave_sum(ss);
  if ((t & 63) == 0) sums[t >> 6] = ss;
  lds_barrier();
  ss = sums[0] + sums[1] + sums[2] + sums[3];
  const float inv = rsqrtf(ss / K + a.eps);
#pragma unroll
  for (int c = 0; c < NCH; ++c) {
    const int d = (c * 256 + t) * 8;
    if (d >= K) continue;
    if (blockIdx.x == 0)
      *reinterpret_cast<uint4*>(a.residual_out + d) = r[c];
    bf16x8 o, g;
    o.u = r[c];
    g.u = gain[c];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      o.s[i] = f32_to_bf16(bf16_to_f32(o.s[i]) * inv * bf16_to_f32(g.s[i]));
    *reinterpret_cast<uint4*>(xs + d) = o.u;
  }
}

// The same for a decoded row's attention that comes in parts (decode_attn.hip):
// channels from c0 to c1 of it, put together by whom they are multiplied by
// anyway.  What bounds it is a round of loads for eight parts of 1024 channels.
// Attention and a product of 4096 x 4096, us, apart and in one: behind 1000
// tokens, eight parts, 19.5 and 16.9, 4000, 32 parts, 21.1 and 20.9.
DEV_INLINE void combine_row(const RowsCombine& a, int c0, int c1, int t,
                            uint16_t* xs) {
  using namespace decode;
  constexpr int B = 8;                    // parts whose loads are one batch
  const int D = a.head_dim, G = a.group;
  int c = c0 + t * 4;
  // (parts that there are not are somebody's scratch: read, not used)
  auto head_of = [&](int ch) { return ch / D; };
  auto slot = [&](int ch, int p) {
    const int h = head_of(ch);
    return (int64_t(h / G) * (a.shares + 1) + p) * G + h % G;
  };
  f32x4 v[B];
  f32x2 ml[B];
  auto ask = [&](int ch, int p0, int top) {
#pragma unroll
    for (int i = 0; i < B; ++i) {
      const int64_t at = slot(ch, min(p0 + i, top));
      v[i] = *reinterpret_cast<const f32x4*>(a.o + at * D + ch % D);
      ml[i] = *reinterpret_cast<const f32x2*>(a.ml + at * 2);
    }
  };
  const int len = *a.len;
  uint2 raw{0, 0};
  if (c < c1) {
    ask(c, 0, a.shares);
    raw = *reinterpret_cast<const uint2*>(a.whole + c);
  }
  lds_barrier();
  const int n = parts_of(len, part_size_of(units_of(len), a.shares, 1));
  for (; c < c1; c += 1024) {
    if (c >= c0 + 1024) {
      ask(c, 0, a.shares);
      raw = *reinterpret_cast<const uint2*>(a.whole + c);
    }
    if (n != 1) {
      float M = kNegInf, den = 0.f;
      f32x4 num = {0.f, 0.f, 0.f, 0.f};
      for (int p0 = 0; p0 < n; p0 += B) {
        if (p0 > 0) ask(c, p0, n - 1);
        float top = M;
#pragma unroll
        for (int i = 0; i < B; ++i)
          if (p0 + i < n) top = fmaxf(top, ml[i][0]);
        const float corr = __builtin_amdgcn_exp2f(M - top);
        num *= corr;
        den *= corr;
        M = top;
#pragma unroll
        for (int i = 0; i < B; ++i)
          if (p0 + i < n) {
            const float w = __builtin_amdgcn_exp2f(ml[i][0] - top);
            num += w * v[i];
            den += w * ml[i][1];
          }
      }
      float x[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = den > 0.f ? num[i] / den : 0.f;
      raw = uint2{uint32_t(f32_to_bf16(x[0])) |
                      uint32_t(f32_to_bf16(x[1])) << 16,
                  uint32_t(f32_to_bf16(x[2])) |
                      uint32_t(f32_to_bf16(x[3])) << 16};
    }
    *reinterpret_cast<uint2*>(xs + c) = raw;
  }
  lds_barrier();
}

enum { NO_PRE = 0, PRE_NORM = 1, PRE_COMBINE = 2 };

// ---- a norm shared between two products ---------------------------------
// The product ahead of a norm, where it is whole, adds its result to the
// streams and leaves rows times gains and, by sixteen columns, their sums of
// squares behind (ADDS of rows_short_kernel); the product behind it multiplies
// its sums by what the norm would have multiplied the rows by.  The norm's launch
// is gone; rows are rounded to 16 bits once, as before.  us, apart and so, two
// streams of 2048 behind 2048 x 2048 and ahead of 6144 x 2048 with the squared
// positive part: 1 row 12.9 and 11.5, 16 14.9 and 12.7, 32 17.2 and 14.8.  (Not
// where the first product is faster in parts: 2048 x 6144, 16 rows 16.7 and 17.8.
// With one 16-bit residual, 4096 x 4096 and 28672 x 4096 with silu: 16 rows 46.1
// and 44.9, 32 47.7 and 47.6, which is not worth another order of roundings.)
template <int MT>
struct Scale {
  static constexpr int Q = MT * 4;        // four rows each
  f32x4 v[Q];
  // ``part``: [4][16 MT], for a workgroup of 256
  DEV_INLINE void ask(const RowsScale& a) {
    const int q = threadIdx.x % Q, p0 = threadIdx.x / Q;
#pragma unroll
    for (int i = 0; i < Q; ++i)
      v[i] = *reinterpret_cast<const f32x4*>(
          a.ss + (min(p0 + i * (256 / Q), a.panels - 1) * Q + q) * 4);
  }
  DEV_INLINE void land(const RowsScale& a, float* part) {
    const int q = threadIdx.x % Q, p0 = threadIdx.x / Q;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < Q; ++i)
      if (p0 + i * (256 / Q) < a.panels) sum += v[i];
#pragma unroll
    for (int d = Q; d < 64; d <<= 1)
#pragma unroll
      for (int r = 0; r < 4; ++r) sum[r] += __shfl_xor(sum[r], d, kWave);
    if ((threadIdx.x & 63) < Q)
      *reinterpret_cast<f32x4*>(part + (threadIdx.x >> 6) * 16 * MT + q * 4) =
          sum;
  }
  static DEV_INLINE float of(const RowsScale& a, const float* part, int row) {
    float ss = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) ss += part[w * 16 * MT + row];
    return rsqrtf(ss / a.width + a.eps);
  }
};

// CT: 16-row tiles of w per wave; XR: rows of x that are staged; MT: 16-row
// tiles of x; R: steps in the ring.  OUT_SILU: a wave's first tile is of the
// gate's rows, the second the same rows of the upper half of w.
// PRE: of one row x, made here (XR 0); it stays in LDS, behind the ring.
template <int CT, int XR, int MT, int R, int OUT, int PRE = NO_PRE>
__global__ __launch_bounds__(PRE ? 512 : 256)
void rows_gemm_kernel(const uint16_t* __restrict__ x,
                      const uint16_t* __restrict__ w, void* __restrict__ out,
                      int M, int N, int K, int splits, NormArgs norm,
                      RowsCombine attn) {
  constexpr int WPART = 4 * CT * 16 * LINE;          // elements of a step
  constexpr int STEP = WPART + XR * LINE;
  constexpr int L = CT * 2 + XR / 32;                // loads of a wave
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];

  const int panel = blockIdx.x / splits, split = blockIdx.x % splits;
  const int steps = K / KS;
  const int s0 = int(int64_t(steps) * split / splits);
  const int n = int(int64_t(steps) * (split + 1) / splits) - s0;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = N / 2;
  uint16_t* xs = lds + R * STEP;
  if constexpr (PRE == PRE_COMBINE) {
    if (wv >= 4) {
      combine_row(attn, s0 * KS, (s0 + n) * KS, threadIdx.x - 256, xs);
      lds_barrier();
      return;
    }
  }
  if constexpr (PRE == PRE_NORM) {
    if (wv >= 4) {
      // (the ring's last step is not asked for before the second barrier)
      float* sums = reinterpret_cast<float*>(lds + (R - 1) * STEP);
      const int t = threadIdx.x - 256;
      if (K <= 2048) norm_row<1>(norm, K, t, sums, xs);
      else if (K <= 4096) norm_row<2>(norm, K, t, sums, xs);
      else norm_row<4>(norm, K, t, sums, xs);
      lds_barrier();
      return;
    }
  }
  // where this workgroup starts within its steps
  const int rot = int(blockIdx.x / 8 % unsigned(n));

  // first row of w of this wave's tile t
  auto tile_row = [&](int t) {
    if constexpr (OUT != OUT_SILU) return panel * 64 * CT + (wv * CT + t) * 16;
    else if constexpr (CT == 2) return t * half + panel * 64 + wv * 16;
    else return (wv >> 1) * half + panel * 32 + (wv & 1) * 16;
  };
  const int last = OUT == OUT_SILU ? half : N;       // rows end here
  // a load takes 8 rows, a lane the piece of row lane / 8 that belongs in
  // slot lane % 8
  const int lr = lane >> 3;
  const uint16_t *wp[CT * 2], *xp[XR / 32 + 1];
#pragma unroll
  for (int j = 0; j < CT * 2; ++j) {
    const int r = (j & 1) * 8 + lr;
    int row = tile_row(j >> 1) + r;
    // rows past the end repeat the last one; nobody stores them
    if constexpr (OUT == OUT_SILU)
      row = min(row, (CT == 2 ? j >> 1 : wv >> 1) * half + half - 1);
    else
      row = min(row, N - 1);
    wp[j] = w + int64_t(row) * K + int64_t(s0) * KS +
            ((lane & 7) ^ ((r >> 1) & 7)) * 8;
  }
#pragma unroll
  for (int j = 0; j < XR / 32; ++j) {
    const int r = (j * 4 + wv) * 8 + lr;
    xp[j] = x + int64_t(min(r, M - 1)) * K + int64_t(s0) * KS +
            ((lane & 7) ^ ((r >> 1) & 7)) * 8;
  }
  auto issue = [&](int s, int slot) {
    uint16_t* at = lds + slot * STEP;
    s += rot;
    if (s >= n) s -= n;
#pragma unroll
    for (int j = 0; j < CT * 2; ++j)
      lds_load16<2>(wp[j] + s * KS, at + (wv * CT * 2 + j) * 8 * LINE);
#pragma unroll
    for (int j = 0; j < XR / 32; ++j)
      lds_load16<0>(xp[j] + s * KS, at + WPART + (j * 4 + wv) * 8 * LINE);
  };

  f32x4 acc[CT][MT];
#pragma unroll
  for (int t = 0; t < CT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int tr = lane & 15, oct = lane >> 4;
  const int sw = tr >> 1;
  if constexpr (PRE) lds_barrier();
#pragma unroll
  for (int s = 0; s < R - 1; ++s)
    if (s < n) issue(s, s);
  if constexpr (PRE) {
    lds_barrier();
    lds_barrier();
  }
  const uint16_t* own = xs + int64_t(s0) * KS + oct * 8;
  int slot = 0;
  for (int s = 0; s < n; ++s) {
    // this wave's loads of the step have landed, then everybody's; nobody
    // reads the step before any more
    wait_steps<L, R - 2>(n - 1 - s);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + R - 1 < n) issue(s + R - 1, slot == 0 ? R - 1 : slot - 1);
    const uint16_t* at = lds + slot * STEP;
    slot = slot == R - 1 ? 0 : slot + 1;
    const uint16_t* wt = at + wv * CT * 16 * LINE + tr * LINE;
    const uint16_t* xt = at + WPART + tr * LINE;
    const uint16_t* xo = own + (s + rot < n ? s + rot : s + rot - n) * KS;
    s16x8 a[2][CT], b[2][MT];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int piece = ((k * 4 + oct) ^ sw) * 8;
#pragma unroll
      for (int t = 0; t < CT; ++t)
        a[k][t] = *reinterpret_cast<const s16x8*>(wt + t * 16 * LINE + piece);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        b[k][m] = *reinterpret_cast<const s16x8*>(
            PRE ? xo + k * 32 : xt + m * 16 * LINE + piece);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int t = 0; t < CT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a[k][t], b[k][m], acc[t][m], 0, 0, 0);
    constexpr int MFMA = 0x8, DS_READ = 0x100;
    __builtin_amdgcn_sched_group_barrier(DS_READ, 2 * (CT + MT), 0);
    __builtin_amdgcn_sched_group_barrier(MFMA, 2 * CT * MT, 0);
  }

  if constexpr (OUT == OUT_SILU && CT == 1) {
    // the upper waves' sums to the lower ones
    __syncthreads();
    f32x4* side = reinterpret_cast<f32x4*>(lds) + (wv & 1) * MT * 64 + lane;
    if (wv >= 2)
#pragma unroll
      for (int m = 0; m < MT; ++m) side[m * 64] = acc[0][m];
    __syncthreads();
    if (wv >= 2) return;
  }
  // a lane has four columns of y of one row
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = m * 16 + tr;
    if (row >= M) continue;
    if constexpr (OUT == OUT_SILU) {
      const int c = tile_row(0) + oct * 4;
      if (c >= last) continue;
      f32x4 up;
      if constexpr (CT == 2) up = acc[1][m];
      else up = reinterpret_cast<const f32x4*>(lds)[((wv & 1) * MT + m) * 64 +
                                                    lane];
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float g = acc[0][m][r];
        v[r] = g / (1.f + __expf(-g)) * up[r];
      }
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) +
                                int64_t(row) * half + c) =
          uint2{pack2(v[0], v[1]), pack2(v[2], v[3])};
    } else {
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        const int c = tile_row(t) + oct * 4;
        if (c >= last) continue;
        const f32x4 v = acc[t][m];
        if constexpr (OUT == OUT_PARTS)
          *reinterpret_cast<f32x4*>(static_cast<float*>(out) +
                                    (int64_t(split) * M + row) * N + c) = v;
        else
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) +
                                    int64_t(row) * N + c) =
              uint2{pack2(v[0], v[1]), pack2(v[2], v[3])};
      }
    }
  }
}

// The same product by workgroups that divide K among their four waves, for
// shapes whose 64-row panels leave CUs idle: 8 HR rows of w per workgroup, no
// parts in memory and no launch to sum them.  A wave has a ring of its own for
// the steps it takes (every fourth, so that the four together read 512 bytes of
// a row at a time): its loads, waits and reads concern nobody else, and there
// is no barrier before the sums meet at the end.  What bounds it is the time
// from the launch to the first data and, past 4096 in K, that it reads x once
// per 8 to 32 rows of w.
// More rows than 64 are tiles of 48 or 64 (TALL), as many as run at once.  What
// bounds those is what a CU can ask for: it takes 58 bytes a ns while any of it
// comes from HBM, whatever is under way, so that a workgroup's rows of x and w
// together are what counts, and a tile that is nearly square is the best.  (us,
// the other way first, 65, 128 and 256 rows: 2048 x 2048 8.7 and 6.1, 8.6 and
// 7.3, 9.6 and 8.2; 6144 x 2048 14.0 and 10.8, 15.3 and 11.7; 4096 x 4096 14.9
// and 14.8, 18.3 and 14.8, 22.6 and 20.7; 3072 x 1024 8.6 and 5.2, 9.4 and 6.1,
// 8.9 and 7.4.)
// END: the result, its squared positive part, or (ADDS; HR 2) S streams with it.
// TALL: ``tiles`` of XR rows, which read the same rows of w on one XCD.
enum End { WHOLE, RELU2, ADDS };

template <int HR, int XR, int MT, int R, End END, int S = 0,
          bool SCALED = false, bool TALL = false>
__global__ __launch_bounds__(256)
void rows_short_kernel(const uint16_t* __restrict__ x,
                       const uint16_t* __restrict__ w,
                       uint16_t* __restrict__ out, int M, int N, int K,
                       RowsScale scale, RowsAdds adds, int tiles) {
  constexpr int PT = (HR + 1) / 2;                   // tiles of w
  constexpr int WPART = HR * 8 * LINE;               // elements of a step
  constexpr int STEP = WPART + XR * LINE;
  constexpr int LX = XR / 8, L = HR + LX;            // loads of a wave
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot0 = blockIdx.x >> 3;
  const int panel =
      TALL ? slot0 / tiles * 8 + int(blockIdx.x & 7) : int(blockIdx.x);
  const int m0 = TALL ? slot0 % tiles * XR : 0;
  const int n0 = panel * HR * 8;
  if (TALL && n0 >= N) return;
  // this wave's steps: wv, wv + 4, ...
  const int n = (K / KS - wv + 3) / 4;
  const int rot = n > 0 ? int(unsigned(panel) / 8 % unsigned(n)) : 0;
  uint16_t* ring = lds + wv * R * STEP;

  const int lr = lane >> 3;
  const uint16_t *wp[HR], *xp[LX];
#pragma unroll
  for (int j = 0; j < HR; ++j) {
    const int r = (j & 1) * 8 + lr;
    // rows past the end repeat the last one; nobody stores them
    const int row = min(n0 + (j >> 1) * 16 + r, N - 1);
    wp[j] = w + int64_t(row) * K + wv * KS + ((lane & 7) ^ ((r >> 1) & 7)) * 8;
  }
#pragma unroll
  for (int j = 0; j < LX; ++j) {
    const int r = j * 8 + lr;
    xp[j] = x + int64_t(min(m0 + r, M - 1)) * K + wv * KS +
            ((lane & 7) ^ ((r >> 1) & 7)) * 8;
  }
  auto issue = [&](int s, int slot) {
    uint16_t* at = ring + slot * STEP;
    s += rot;
    if (s >= n) s -= n;
#pragma unroll
    for (int j = 0; j < HR; ++j)
      lds_load16<2>(wp[j] + s * 4 * KS, at + j * 8 * LINE);
#pragma unroll
    for (int j = 0; j < LX; ++j)
      lds_load16<0>(xp[j] + s * 4 * KS, at + WPART + j * 8 * LINE);
  };

  f32x4 acc[PT][MT];
#pragma unroll
  for (int t = 0; t < PT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int tr = lane & 15, oct = lane >> 4;
  const int sw = tr >> 1;
  __shared__ __attribute__((aligned(16))) float part[SCALED ? 64 * MT : 4];
  Scale<SCALED ? MT : 1> sc;
  if constexpr (SCALED) sc.ask(scale);
  // what a lane of wave m < MT adds to: four columns of row 16 m + tr
  const int arow = min(wv * 16 + tr, M - 1), acol = n0 + oct * 4;
  f32x4 had[S > 0 ? S : 1], gain;
  float mix[S > 0 ? S : 1][S > 0 ? S : 1], outw[S > 0 ? S : 1],
      inw[S > 0 ? S : 1];
  if constexpr (END == ADDS) {
    static_assert(HR == 2 && MT <= 4, "");
#pragma unroll
    for (int s = 0; s < S; ++s) {
      had[s] = *reinterpret_cast<const f32x4_any*>(
          adds.streams + (int64_t(arow) * S + s) * N + acol);
      outw[s] = adds.out_w[s];
      inw[s] = adds.in_w[s];
#pragma unroll
      for (int t = 0; t < S; ++t) mix[s][t] = adds.mix[s * S + t];
    }
    gain = *reinterpret_cast<const f32x4_any*>(adds.gain + acol);
  }
#pragma unroll
  for (int s = 0; s < R - 1; ++s)
    if (s < n) issue(s, s);
  if constexpr (SCALED) sc.land(scale, part);
  int slot = 0;
  for (int s = 0; s < n; ++s) {
    wait_steps<L, R - 2>(n - 1 - s);
    const uint16_t* at = ring + slot * STEP;
    const uint16_t* wt = at + tr * LINE;
    const uint16_t* xt = at + WPART + tr * LINE;
    s16x8 a[2][PT], b[2][MT];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int piece = ((k * 4 + oct) ^ sw) * 8;
#pragma unroll
      for (int t = 0; t < PT; ++t)
        a[k][t] = *reinterpret_cast<const s16x8*>(wt + t * 16 * LINE + piece);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        b[k][m] = *reinterpret_cast<const s16x8*>(xt + m * 16 * LINE + piece);
    }
    // the slot before this one was read a step ago
    if (s + R - 1 < n) issue(s + R - 1, slot == 0 ? R - 1 : slot - 1);
    slot = slot == R - 1 ? 0 : slot + 1;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int t = 0; t < PT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a[k][t], b[k][m], acc[t][m], 0, 0, 0);
  }

  // the waves' sums meet, in order
  __syncthreads();
  f32x4* side = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int t = 0; t < PT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      side[(wv * PT * MT + t * MT + m) * 64 + lane] = acc[t][m];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (PT * MT + 3) / 4; ++i) {
    const int e = i * 4 + wv;
    if (e >= PT * MT) break;
    f32x4 v = side[e * 64 + lane];
#pragma unroll
    for (int o = 1; o < 4; ++o) v += side[(o * PT * MT + e) * 64 + lane];
    const int row = m0 + e % MT * 16 + tr;
    const int c = n0 + e / MT * 16 + oct * 4;
    if constexpr (SCALED) v *= Scale<SCALED ? MT : 1>::of(scale, part, row);
    if constexpr (END == RELU2) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // (of more rows of the 16-bit product, as by tiles)
        if constexpr (TALL) v[r] = bf16_to_f32(f32_to_bf16(v[r]));
        v[r] = fmaxf(v[r], 0.f);
        v[r] *= v[r];
      }
    }
    if constexpr (END == ADDS) {
      // (of one tile a wave, e is wv)
      f32x4 u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < S; ++t) {
        f32x4 to;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float sum = outw[t] * v[r];
#pragma unroll
          for (int s = 0; s < S; ++s) sum += mix[s][t] * had[s][r];
          to[r] = sum;
          u[r] += inw[t] * sum;
        }
        if (row < M)
          *reinterpret_cast<f32x4_any*>(adds.streams +
                                        (int64_t(row) * S + t) * N + c) = to;
      }
      float ss = 0.f;
#pragma unroll
      for (int r = 0; r < 4; ++r) ss += u[r] * u[r];
      ss += __shfl_xor(ss, 16, kWave);
      ss += __shfl_xor(ss, 32, kWave);
      if (oct == 0) adds.ss[int64_t(blockIdx.x) * 16 * MT + row] = ss;
      v = u * gain;
    }
    // (an odd last tile has only eight rows of w)
    if (row < M && c < min(N, n0 + HR * 8))
      *reinterpret_cast<uint2*>(out + int64_t(row) * N + c) =
          uint2{pack2(v[0], v[1]), pack2(v[2], v[3])};
  }
}

__global__ __launch_bounds__(256)
void sum_parts_kernel(const float* __restrict__ parts,
                      uint16_t* __restrict__ out, int splits, int64_t n) {
  const int64_t i = (int64_t(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  f32x4 v = *reinterpret_cast<const f32x4*>(parts + i);
  for (int s = 1; s < splits; ++s)
    v += *reinterpret_cast<const f32x4*>(parts + s * n + i);
  *reinterpret_cast<uint2*>(out + i) =
      uint2{pack2(v[0], v[1]), pack2(v[2], v[3])};
}

// R32, R64, R128: steps in the ring with as many rows of x
template <int CT, int R32, int R64, int R128, int OUT>
void go(const uint16_t* x, const uint16_t* w, void* out, int M, int N, int K,
        int panels, int splits, hipStream_t st) {
  auto run = [&](auto xr, auto mt) {
    constexpr int XR = decltype(xr)::value, MT = decltype(mt)::value;
    constexpr int R = XR == 32 ? R32 : XR == 64 ? R64 : R128;
    constexpr size_t smem = size_t(R) * (4 * CT * 16 + XR) * LINE * 2;
    auto* k = rows_gemm_kernel<CT, XR, MT, R, OUT>;
    if (smem > 65536)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(smem));
    hipLaunchKernelGGL(k, dim3(panels * splits), dim3(256), smem, st, x, w,
                       out, M, N, K, splits, NormArgs{}, RowsCombine{});
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  using I4 = std::integral_constant<int, 4>;
  using X32 = std::integral_constant<int, 32>;
  using I6 = std::integral_constant<int, 6>;
  using I8 = std::integral_constant<int, 8>;
  using X64 = std::integral_constant<int, 64>;
  using X128 = std::integral_constant<int, 128>;
  if (M <= 16) run(X32{}, I1{});
  else if (M <= 32) run(X32{}, I2{});
  else if (M <= 48) run(X64{}, I3{});
  else if (M <= 64) run(X64{}, I4{});
  else if (M <= 96) run(X128{}, I6{});
  else run(X128{}, I8{});
}

template <int CT, int R, int OUT>
void go_norm(const RowsNorm& norm, const uint16_t* w, void* out, int N, int K,
             int panels, int splits, hipStream_t st) {
  const size_t smem = (size_t(R) * 4 * CT * 16 * LINE + size_t(K)) * 2;
  auto* k = rows_gemm_kernel<CT, 0, 1, R, OUT, PRE_NORM>;
  if (smem > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              int(smem));
  hipLaunchKernelGGL(k, dim3(panels * splits), dim3(512), smem, st, nullptr, w,
                     out, 1, N, K, splits,
                     NormArgs{norm.parts, norm.residual, norm.residual_out,
                              norm.gain, norm.n, norm.eps},
                     RowsCombine{});
}

template <int HR, int R16, int R32, int R64, End END>
void go_short(const uint16_t* x, const uint16_t* w, uint16_t* out, int M,
              int N, int K, hipStream_t st) {
  auto run = [&](auto xr) {
    constexpr int XR = decltype(xr)::value, MT = XR / 16;
    constexpr int R = XR == 16 ? R16 : XR == 32 ? R32 : R64;
    constexpr size_t smem = size_t(4) * R * (HR * 8 + XR) * LINE * 2;
    auto* k = rows_short_kernel<HR, XR, MT, R, END>;
    if (smem > 65536)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(smem));
    hipLaunchKernelGGL(k, dim3((N + HR * 8 - 1) / (HR * 8)), dim3(256), smem,
                       st, x, w, out, M, N, K, RowsScale{}, RowsAdds{}, 1);
  };
  if (M <= 16) run(std::integral_constant<int, 16>{});
  else if (M <= 32) run(std::integral_constant<int, 32>{});
  else run(std::integral_constant<int, 64>{});
}

// with a norm that is shared, up to 32 rows
template <int HR, int R16, int R32, End END, int S, bool SCALED>
void go_shared(const uint16_t* x, const uint16_t* w, uint16_t* out, int M,
               int N, int K, const RowsScale& scale, const RowsAdds& adds,
               hipStream_t st) {
  auto run = [&](auto xr) {
    constexpr int XR = decltype(xr)::value, MT = XR / 16;
    constexpr int R = XR == 16 ? R16 : R32;
    constexpr size_t smem = size_t(4) * R * (HR * 8 + XR) * LINE * 2;
    auto* k = rows_short_kernel<HR, XR, MT, R, END, S, SCALED>;
    if (smem > 65536)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(smem));
    hipLaunchKernelGGL(k, dim3((N + HR * 8 - 1) / (HR * 8)), dim3(256), smem,
                       st, x, w, out, M, N, K, scale, adds, 1);
  };
  if (M <= 16) run(std::integral_constant<int, 16>{});
  else run(std::integral_constant<int, 32>{});
}

// of more rows than a tile has
template <int HR, int XR, int R, End END>
void go_tall(const uint16_t* x, const uint16_t* w, uint16_t* out, int M, int N,
             int K, hipStream_t st) {
  constexpr int MT = XR / 16;
  constexpr size_t smem = size_t(4) * R * (HR * 8 + XR) * LINE * 2;
  auto* k = rows_short_kernel<HR, XR, MT, R, END, 0, false, true>;
  if (smem > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              int(smem));
  const int tiles = (M + XR - 1) / XR, panels = (N + HR * 8 - 1) / (HR * 8);
  hipLaunchKernelGGL(k, dim3((panels + 7) / 8 * 8 * tiles), dim3(256), smem, st,
                     x, w, out, M, N, K, RowsScale{}, RowsAdds{}, tiles);
}

}  // namespace

// As many parts as 64-row panels leave CUs for: with more workgroups than
// CUs some CUs have twice the work (N 4096, K 14336: 256 workgroups 19.1 us,
// 320 24.2, 512 19.5), with half of them latency shows (128: 24.4).
int rows_gemm_splits(int N, int K) {
  const int panels = (N + 63) / 64;
  int n = std::max(1, 256 / panels);
  // far from a whole round, two rounds waste less
  if (panels * n < 180 && panels < 256) n = 512 / panels;
  return std::min(n, K / KS);
}

// Rings with up to 32, 64 and 128 rows of x: parts 72, 80 and 120 KB, whole
// panels of 64 (and 32 pairs with silu) 72, 80 and 72, of 128 60, 72 and 128, of
// 64 pairs 100, 120 and 128.  One workgroup per CU keeps enough under way; two
// share its 160 KB where rings are of 80 or less.  Panels of 128
// halve what x costs and are taken where they still cover the CUs (128256
// rows of 4096: 155 us against 158 for one row, 177 against 207 for 64).
void launch_rows_gemm(const uint16_t* x, const uint16_t* w, float* parts,
                      uint16_t* out, int M, int N, int K, int splits,
                      hipStream_t st) {
  const int panels = (N + 63) / 64;
  if (parts)
    go<1, 6, 5, 5, OUT_PARTS>(x, w, parts, M, N, K, panels, splits, st);
  else if (panels < 400)
    go<1, 6, 5, 3, OUT_BF16>(x, w, out, M, N, K, panels, 1, st);
  else
    go<2, 3, 3, 4, OUT_BF16>(x, w, out, M, N, K, (N + 127) / 128, 1, st);
}

// Panels of 64 pairs where they cover the CUs, of 32 otherwise (14336 pairs
// of 4096: 35.3 us against 39.3; 8192 of 2048: 14.5 against 12.1).
bool rows_gemm_silu_ok(int inter) { return (inter + 31) / 32 >= 160; }

void launch_rows_gemm_silu(const uint16_t* x, const uint16_t* w,
                           uint16_t* out, int M, int inter, int K,
                           hipStream_t st) {
  if ((inter + 63) / 64 >= 200)
    go<2, 5, 5, 4, OUT_SILU>(x, w, out, M, 2 * inter, K, (inter + 63) / 64, 1,
                          st);
  else
    go<1, 6, 5, 3, OUT_SILU>(x, w, out, M, 2 * inter, K, (inter + 31) / 32, 1,
                          st);
}

// Whether a product of one row makes it from a residual by itself: with no more
// workgroups than CUs, as each makes all of it.
bool rows_norm_ok(int N, int K, bool silu) {
  if (K > 8192) return false;
  if (silu) return rows_gemm_silu_ok(N / 2) && (N / 2 + 63) / 64 <= 256;
  return (N + 63) / 64 <= 256 && rows_gemm_splits(N, K) > 1;
}

// Rings of 48 KB (80 for panels of 64 pairs) and up to 16 KB of x; 6144 x 4096,
// us with 24, 32, 40, 48, 64 and 80 KB: 15.6 13.2 12.8 12.7 13.0 13.3.
void launch_rows_norm(const RowsNorm& norm, const uint16_t* w, float* parts,
                      int N, int K, int splits, hipStream_t st) {
  go_norm<1, 6, OUT_PARTS>(norm, w, parts, N, K, (N + 63) / 64, splits, st);
}

// For up to 1024 channels of a workgroup (8192 x 8192, 4096 of them: four parts
// 42.5 and 43.4 us, 16 parts 46.2 and 50.5) and 32 parts (more are of sequences
// beyond 8192 tokens; 63 of 4096 channels in all: 25.9 and 27.4).
bool rows_combine_ok(int N, int K, int max_tokens) {
  using namespace decode;
  const int splits = rows_gemm_splits(N, K);
  return rows_norm_ok(N, K, false) && (K / KS + splits - 1) / splits <= 16 &&
         max_tokens <= MOST_ONE * MIN_UNITS * UNIT;
}

void launch_rows_combine(const RowsCombine& attn, const uint16_t* w,
                         float* parts, int N, int K, int splits,
                         hipStream_t st) {
  constexpr int R = 6;
  const size_t smem = (size_t(R) * 64 * LINE + size_t(K)) * 2;
  auto* k = rows_gemm_kernel<1, 0, 1, R, OUT_PARTS, PRE_COMBINE>;
  if (smem > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              int(smem));
  hipLaunchKernelGGL(k, dim3((N + 63) / 64 * splits), dim3(512), smem, st,
                     nullptr, w, parts, 1, N, K, splits, NormArgs{}, attn);
}

void launch_rows_norm_silu(const RowsNorm& norm, const uint16_t* w,
                           uint16_t* out, int inter, int K, hipStream_t st) {
  if ((inter + 63) / 64 >= 200)
    go_norm<2, 5, OUT_SILU>(norm, w, out, 2 * inter, K, (inter + 63) / 64, 1,
                            st);
  else
    go_norm<1, 6, OUT_SILU>(norm, w, out, 2 * inter, K, (inter + 31) / 32, 1,
                             st);
}

// Whether rows_short_kernel takes a product; by N and K alone, like all orders of
// sums here.  (1, 16, 64 rows of x, us, parts and their sum first: 2048 x 2048 6.5
// and 3.9, 7.7 and 4.4, 9.3 and 7.0; 8192 x 2048 10.7 and 7.0, 11.5 and 7.2, 13.7
// and 10.2; 6144 x 4096 13.6 and 9.3, 14.5 and 9.7, 18.3 and 14.7; 256 x 8192 18.7
// and 7.0, 22.3 and 8.5, 20.7 and 17.3; but 4096 x 4096 9.7 and 7.8, 10.3 and 8.9,
// 13.1 and 13.4; 2048 x 8192 10.5 and 9.8, 11.6 and 12.4, 13.7 and 20.4; 5120 x
// 5120 12.5 and 11.8, 13.4 and 15.9, 18.3 and 21.9.)
bool rows_short_ok(int N, int K) {
  return N <= 8192 && K <= (N > 4096 ? 4096 : N > 512 ? 3072 : 8192);
}

namespace {

// Rows of w of one of its workgroups, in eights: as few as make no more
// workgroups than CUs, whose rings leave no room for a second one.  The order of
// sums follows it, as a workgroup begins its steps by its index: of one N it is
// one order here, another in the products that share a norm, which take 16 rows
// of w up to N of 4096.  (1, 16, 64 rows of x, us, 8, 16, 24 and 32 rows of w:
// 2048 x 2048 3.9 4.1 4.3 4.7, 4.4 4.8 5.1 5.6, 7.0 7.1 7.9 8.4; 4096 x 2048 6.8
// 4.9 4.7 5.1, 7.7 5.1 5.6 6.0, 12.6 7.7 8.5 8.9; 6144 x 2048 9.6 7.8 5.7 5.8,
// 11.0 8.6 6.0 6.4, 18.2 13.2 9.0 9.5; 6160 x 2048 11.5 7.7 8.1 5.8, 13.1 8.6 8.5
// 6.4, 22.2 13.0 13.7 9.5.)
int short_eights(int N) { return std::clamp((N + 2047) / 2048, 1, 4); }

}  // namespace

void launch_rows_short(const uint16_t* x, const uint16_t* w, uint16_t* out,
                       int M, int N, int K, bool relu2, hipStream_t st) {
  auto run = [&](auto end) {
    constexpr End END = decltype(end)::value;
    switch (short_eights(N)) {
      case 1: return go_short<1, 12, 7, 4, END>(x, w, out, M, N, K, st);
      case 2: return go_short<2, 9, 6, 3, END>(x, w, out, M, N, K, st);
      case 3: return go_short<3, 7, 5, 3, END>(x, w, out, M, N, K, st);
      default: return go_short<4, 6, 4, 3, END>(x, w, out, M, N, K, st);
    }
  };
  if (relu2) run(std::integral_constant<End, RELU2>{});
  else run(std::integral_constant<End, WHOLE>{});
}

// The least rows of x and w a workgroup, where all workgroups of an XCD run at
// once on its 32 CUs; none: rows 0.
TallPlan rows_tall_plan(int M, int N) {
  TallPlan best{0, 0};
  for (int rows : {64, 48})
    for (int eights : {2, 3, 4, 6, 8}) {
      const int64_t tiles = (int64_t(M) + rows - 1) / rows;
      const int64_t panels = (int64_t(N) + eights * 8 - 1) / (eights * 8);
      if (tiles * ((panels + 7) / 8) <= 32 &&
          (best.rows == 0 ||
           rows + 8 * eights < best.rows + 8 * best.eights))
        best = TallPlan{rows, eights};
    }
  return best;
}

void launch_rows_tall(const uint16_t* x, const uint16_t* w, uint16_t* out,
                      int M, int N, int K, bool relu2, const TallPlan& plan,
                      hipStream_t st) {
  auto run = [&](auto end) {
    constexpr End END = decltype(end)::value;
    switch (plan.rows * 16 + plan.eights) {
      case 48 * 16 + 2: return go_tall<2, 48, 4, END>(x, w, out, M, N, K, st);
      case 48 * 16 + 3: return go_tall<3, 48, 4, END>(x, w, out, M, N, K, st);
      case 48 * 16 + 4: return go_tall<4, 48, 3, END>(x, w, out, M, N, K, st);
      case 48 * 16 + 6: return go_tall<6, 48, 3, END>(x, w, out, M, N, K, st);
      case 48 * 16 + 8: return go_tall<8, 48, 2, END>(x, w, out, M, N, K, st);
      case 64 * 16 + 2: return go_tall<2, 64, 3, END>(x, w, out, M, N, K, st);
      case 64 * 16 + 3: return go_tall<3, 64, 3, END>(x, w, out, M, N, K, st);
      case 64 * 16 + 4: return go_tall<4, 64, 3, END>(x, w, out, M, N, K, st);
      case 64 * 16 + 6: return go_tall<6, 64, 2, END>(x, w, out, M, N, K, st);
      default: return go_tall<8, 64, 2, END>(x, w, out, M, N, K, st);
    }
  };
  if (relu2) run(std::integral_constant<End, RELU2>{});
  else run(std::integral_constant<End, WHOLE>{});
}

bool rows_adds_ok(int M, int N, int K, int streams) {
  return M >= 1 && M <= 32 && N % 16 == 0 && N <= 4096 && K % 64 == 0 &&
         rows_short_ok(N, K) && streams >= 1 && streams <= 4;
}

void launch_rows_adds(const uint16_t* x, const uint16_t* w, uint16_t* out,
                      int M, int N, int K, int streams, const RowsAdds& adds,
                      hipStream_t st) {
  auto run = [&](auto s) {
    go_shared<2, 9, 6, ADDS, decltype(s)::value, false>(
        x, w, out, M, N, K, RowsScale{}, adds, st);
  };
  switch (streams) {
    case 1: return run(std::integral_constant<int, 1>{});
    case 2: return run(std::integral_constant<int, 2>{});
    case 3: return run(std::integral_constant<int, 3>{});
    default: return run(std::integral_constant<int, 4>{});
  }
}

bool rows_scaled_ok(int M, int N, int K) {
  return M >= 1 && M <= 32 && N % 4 == 0 && K % 64 == 0 &&
         rows_short_ok(N, K);
}

void launch_rows_scaled_relu2(const uint16_t* x, const uint16_t* w,
                              uint16_t* out, int M, int N, int K,
                              const RowsScale& scale, hipStream_t st) {
  switch (short_eights(N)) {
    case 1:
    case 2:
      return go_shared<2, 9, 6, RELU2, 0, true>(x, w, out, M, N, K, scale,
                                                RowsAdds{}, st);
    case 3:
      return go_shared<3, 7, 5, RELU2, 0, true>(x, w, out, M, N, K, scale,
                                                RowsAdds{}, st);
    default:
      return go_shared<4, 6, 4, RELU2, 0, true>(x, w, out, M, N, K, scale,
                                                RowsAdds{}, st);
  }
}

void launch_sum_parts(const float* parts, uint16_t* out, int splits,
                      int64_t n, hipStream_t st) {
  hipLaunchKernelGGL(sum_parts_kernel, dim3(unsigned((n / 4 + 255) / 256)),
                     dim3(256), 0, st, parts, out, splits, n);
}

}  // namespace rlli
