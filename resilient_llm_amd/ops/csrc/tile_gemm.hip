// Products of some hundred rows, as chunks of prompts and short prompts beside
// decoding sequences have them: y[M, N] = x[M, K] w[N, K]^T, bf16 with f32
// sums.
//
// A workgroup has a tile of 64 MH x 128 NH, eight waves two by four, each with
// MH x NH blocks of 16 x 16 in each quarter of the tile.  A 64-wide step of K
// is four phases, one quarter each: fragments are read from LDS, then
// multiplied.  The two waves of a SIMD take turns, one half-phase apart, so
// that one's products run while the other reads and asks for what comes next;
// a barrier ends each half-phase.  Steps come through two buffers in LDS by
// direct global -> LDS loads, half a tile's rows of x or w at a time, each as
// soon as its place was read for the last time: five to seven phases ahead of
// its use, and waits count loads, so nothing drains.  Rows' 16-byte pieces are
// swizzled as in rows_gemm.hip.

#include "common.h"
#include "kernels.h"

#include <algorithm>
#include <type_traits>

namespace rlli {

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));

constexpr int KS = 64;

enum { OUT_PARTS = 0, OUT_BF16 = 1, OUT_SILU = 2 };

DEV_INLINE uint32_t pack2(float a, float b) {
  const b16x2 v = __builtin_convertvector((f32x2{a, b}), b16x2);
  return __builtin_bit_cast(uint32_t, v);
}

DEV_INLINE void lds_load16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)g,
      (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

template <int N>
DEV_INLINE void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// nothing is moved over it
DEV_INLINE void section() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

template <int MH, int NH, int OUT>
__global__ __launch_bounds__(512, 2)
void tile_gemm_kernel(const uint16_t* __restrict__ x,
                      const uint16_t* __restrict__ w, void* __restrict__ out,
                      int M, int N, int K, int rows, int splits, int units) {
  constexpr int TM = 64 * MH, TN = 128 * NH;
  constexpr int STEP = (TM + TN) * KS;          // elements of a buffer
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];

  // Units of an XCD are consecutive: row tiles first, which read the same w.
  const int per = (units + 7) / 8;
  const int unit = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || unit >= units) return;
  const int m0 = unit % rows * TM;
  const int split = unit / rows % splits;
  const int panel = unit / rows / splits;
  const int n0 = panel * TN;
  const int steps = K / KS;
  const int s0 = int(int64_t(steps) * split / splits);
  const int nk = int(int64_t(steps) * (split + 1) / splits) - s0;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave >> 2;
  const int wn = wave & 3;
  const int half = N / 2;

  // ---- loads: 8 rows each; of w NH per half and wave, of x MH / 2, or one
  // and two by turns where that is not whole
  constexpr int AL = (MH + 1) / 2;
  uint32_t ao[2][AL], bo[2][NH];                // bytes, below 2^32
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int j = 0; j < AL; ++j) {
      const int q = j * 8 + (MH == 3 && j ? wave & 3 : wave);
      const int r = h * TM / 2 + q * 8 + (lane >> 3);
      ao[h][j] = (uint32_t(min(m0 + r, M - 1)) * K +
                  ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2;
    }
#pragma unroll
    for (int j = 0; j < NH; ++j) {
      const int r = h * TN / 2 + (j * 8 + wave) * 8 + (lane >> 3);
      const int row =
          OUT == OUT_SILU
              ? h * half + min(panel * TN / 2 + r - h * TN / 2, half - 1)
              : min(n0 + r, N - 1);
      bo[h][j] =
          (uint32_t(row) * K + ((lane & 7) ^ ((r >> 1) & 7)) * 8) * 2;
    }
  }
  const char* xb = reinterpret_cast<const char*>(x + int64_t(s0) * KS);
  const char* wb = reinterpret_cast<const char*>(w + int64_t(s0) * KS);
  auto ask_x = [&](int s, int h) {
    uint16_t* to = lds + (s & 1) * STEP + h * TM / 2 * KS;
#pragma unroll
    for (int j = 0; j < AL; ++j) {
      if (MH == 3 && j && h != group) continue;
      const int q = j * 8 + (MH == 3 && j ? wave & 3 : wave);
      lds_load16(xb + int64_t(min(s, nk - 1)) * (KS * 2) + ao[h][j], to + q * 8 * KS);
    }
  };
  auto ask_w = [&](int s, int h) {
    uint16_t* to = lds + (s & 1) * STEP + (TM + h * TN / 2) * KS;
#pragma unroll
    for (int j = 0; j < NH; ++j)
      lds_load16(wb + int64_t(min(s, nk - 1)) * (KS * 2) + bo[h][j],
                 to + (j * 8 + wave) * 8 * KS);
  };
  // All of this wave's loads but the newest have landed: X0 and X1 first and
  // second halves of x, W halves of w.
  auto wait_but = [&](auto x0, auto x1, auto w_) {
    constexpr int X0 = decltype(x0)::value, X1 = decltype(x1)::value;
    constexpr int W = decltype(w_)::value * NH;
    if constexpr (MH != 3) wait_vm<(X0 + X1) * (MH / 2) + W>();
    else if (group == 0) wait_vm<X0 * 2 + X1 + W>();
    else wait_vm<X0 + X1 * 2 + W>();
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;

  f32x4 acc[2][2][MH][NH];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int i = 0; i < MH; ++i)
#pragma unroll
        for (int j = 0; j < NH; ++j) acc[a][b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int tr = lane & 15, oct = lane >> 4;
  int piece[2];
#pragma unroll
  for (int k = 0; k < 2; ++k)
    piece[k] = tr * KS + ((k * 4 + oct) ^ (tr >> 1)) * 8;
  s16x8 fa[MH][2], fb[2][NH][2];
  auto read_x = [&](int s, int h) {
    const uint16_t* at =
        lds + (s & 1) * STEP + (h * TM / 2 + group * MH * 16) * KS;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < MH; ++i)
        fa[i][k] =
            *reinterpret_cast<const s16x8*>(at + i * 16 * KS + piece[k]);
  };
  auto read_w = [&](int s, int h) {
    const uint16_t* at =
        lds + (s & 1) * STEP + (TM + h * TN / 2 + wn * NH * 16) * KS;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int j = 0; j < NH; ++j)
        fb[h][j][k] =
            *reinterpret_cast<const s16x8*>(at + j * 16 * KS + piece[k]);
  };
  auto multiply = [&](int a, int b) {
    section();
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int i = 0; i < MH; ++i)
#pragma unroll
        for (int j = 0; j < NH; ++j)
          acc[a][b][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              fb[b][j][k], fa[i][k], acc[a][b][i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    // what was read is free to be written from here on
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    section();
  };
  // A step.  The halves of w take turns in being the first (F), which was read
  // in the step before, so that a phase reads one half and needs no registers
  // beyond.  (The largest tile has none for two forms of the step: its first
  // phase reads two halves.)  Behind the last step, the last is asked for
  // again: nobody reads it.
  constexpr bool TURNS = MH + NH < 6;
  auto step = [&](int s, auto first) {
    constexpr int F = decltype(first)::value;
    read_x(s, 0);
    if constexpr (!TURNS) read_w(s, F);
    ask_x(s + 1, 1);
    wait_but(I1{}, I2{}, I2{});
    multiply(0, F);
    read_w(s, 1 - F);
    if constexpr (TURNS) ask_w(s + 2, F);
    wait_but(I1{}, I1{}, std::integral_constant<int, TURNS ? 3 : 2>{});
    multiply(0, 1 - F);
    read_x(s, 1);
    ask_x(s + 2, 0);
    if constexpr (TURNS) wait_but(I2{}, I1{}, I2{});
    else ask_w(s + 2, F);
    multiply(1, 1 - F);
    if constexpr (TURNS) read_w(s + 1, 1 - F);
    ask_w(s + 2, 1 - F);
    wait_but(I1{}, I1{}, I3{});
    multiply(1, F);
  };

  ask_w(0, 0);
  ask_x(0, 0);
  ask_w(0, 1);
  ask_x(0, 1);
  ask_w(1, TURNS);
  ask_x(1, 0);
  ask_w(1, !TURNS);
  wait_but(I1{}, I1{}, I3{});
  section();
  if constexpr (TURNS) read_w(0, 0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (group) section();
#pragma unroll 1
  for (int s = 0; s < nk; s += 2) {
    step(s, I0{});
    if (s + 1 < nk) step(s + 1, std::integral_constant<int, TURNS>{});
  }
  if (!group) section();
  wait_vm<0>();

  // a lane has four columns of y of one row
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int i = 0; i < MH; ++i) {
      const int row = m0 + a * TM / 2 + (group * MH + i) * 16 + tr;
      if (row >= M) continue;
#pragma unroll
      for (int j = 0; j < NH; ++j) {
        const int c = (wn * NH + j) * 16 + oct * 4;
        if constexpr (OUT == OUT_SILU) {
          const int col = panel * TN / 2 + c;
          if (col >= half) continue;
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float g = acc[a][0][i][j][r];
            v[r] = g / (1.f + __expf(-g)) * acc[a][1][i][j][r];
          }
          *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) +
                                    int64_t(row) * half + col) =
              uint2{pack2(v[0], v[1]), pack2(v[2], v[3])};
        } else {
#pragma unroll
          for (int b = 0; b < 2; ++b) {
            const int col = n0 + b * TN / 2 + c;
            if (col >= N) continue;
            const f32x4 v = acc[a][b][i][j];
            if constexpr (OUT == OUT_PARTS)
              *reinterpret_cast<f32x4*>(static_cast<float*>(out) +
                                        (int64_t(split) * M + row) * N + col) =
                  v;
            else
              *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) +
                                        int64_t(row) * N + col) =
                  uint2{pack2(v[0], v[1]), pack2(v[2], v[3])};
          }
        }
      }
    }
}

template <int MH, int NH, int OUT>
void go(const uint16_t* x, const uint16_t* w, void* out, int M, int N, int K,
        int splits, hipStream_t st) {
  constexpr int TM = 64 * MH, TN = 128 * NH;
  constexpr size_t smem = size_t(2) * (TM + TN) * KS * 2;
  auto* k = tile_gemm_kernel<MH, NH, OUT>;
  if (smem > 65536)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                              hipFuncAttributeMaxDynamicSharedMemorySize,
                              int(smem));
  const int rows = (M + TM - 1) / TM, panels = (N + TN - 1) / TN;
  const int units = rows * panels * splits;
  hipLaunchKernelGGL(k, dim3((units + 7) / 8 * 8), dim3(512), smem, st, x, w,
                     out, M, N, K, rows, splits, units);
}

// Tiles, us for a workgroup's start and end and for a step of K, as measured
// with up to one workgroup per CU.
struct Tile {
  int mh, nh;
  float fixed, step;
};
constexpr Tile TILES[] = {{2, 1, 4.8f, 0.52f}, {2, 2, 5.8f, 0.81f},
                          {2, 3, 7.9f, 1.05f}, {3, 1, 4.5f, 0.84f},
                          {3, 2, 6.7f, 0.95f}, {3, 3, 10.5f, 1.45f},
                          {4, 1, 5.5f, 0.81f}, {4, 2, 5.9f, 1.24f}};
constexpr int MOST_SPLITS = 8;

}  // namespace

// The tile and the division of K that should take least: rounds of 256
// workgroups, each with its steps, and 0.6 us for each megabyte of parts that
// is written and read again.  (Over seven shapes at 14 numbers of rows from 132
// to 2048 what it chose took 2 % more than the best did.)
TilePlan tile_gemm_plan(int M, int N, int K, bool silu) {
  TilePlan best{};
  float least = 0.f;
  const int steps = K / KS;
  for (const Tile& t : TILES) {
    const int rows = (M + 64 * t.mh - 1) / (64 * t.mh);
    const int tiles = rows * ((N + 128 * t.nh - 1) / (128 * t.nh));
    for (int s = 1; s <= (silu ? 1 : std::min(MOST_SPLITS, steps)); ++s) {
      const int rounds = (tiles * s + 255) / 256;
      const float parts = s > 1 ? float(s) * M * N * 4e-6f : 0.f;
      const float us =
          rounds * (t.fixed + (steps + s - 1) / s * t.step) + 0.6f * parts;
      if (best.mh == 0 || us < least) {
        best = TilePlan{t.mh, t.nh, s};
        least = us;
      }
    }
  }
  return best;
}

void launch_tile_gemm(const uint16_t* x, const uint16_t* w, float* parts,
                      uint16_t* out, int M, int N, int K, bool silu,
                      const TilePlan& plan, hipStream_t st) {
  auto run = [&](auto m, auto n) {
    constexpr int MH = decltype(m)::value, NH = decltype(n)::value;
    if (silu)
      go<MH, NH, OUT_SILU>(x, w, out, M, N, K, 1, st);
    else if (parts)
      go<MH, NH, OUT_PARTS>(x, w, parts, M, N, K, plan.splits, st);
    else
      go<MH, NH, OUT_BF16>(x, w, out, M, N, K, 1, st);
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  using I4 = std::integral_constant<int, 4>;
  switch (plan.mh * 4 + plan.nh) {
    case 9: return run(I2{}, I1{});
    case 10: return run(I2{}, I2{});
    case 11: return run(I2{}, I3{});
    case 13: return run(I3{}, I1{});
    case 14: return run(I3{}, I2{});
    case 15: return run(I3{}, I3{});
    case 17: return run(I4{}, I1{});
    default: return run(I4{}, I2{});
  }
}

}  // namespace rlli
