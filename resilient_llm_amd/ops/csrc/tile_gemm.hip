// Products of some hundred rows, as chunks of prompts and short prompts beside
// decoding sequences have them: y[M, N] = x[M, K] w[N, K]^T, bf16 with f32
// sums.
//
// Tiles of 128 to 256 rows by 128 to 384 columns (tile_product.h), one per
// workgroup; where those leave CUs idle, K is divided and the parts are written
// in f32, for whoever reads the product to sum, in order.  Of gate and up rows a
// tile has half its columns each, so that silu of one meets the other in a
// lane's registers.
#include "common.h"
#include "kernels.h"
#include "tile_product.h"

#include <algorithm>
#include <iterator>
#include <type_traits>

namespace rlli {

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));

enum { OUT_PARTS = 0, OUT_BF16 = 1, OUT_SILU = 2, OUT_RELU2 = 3 };

DEV_INLINE uint32_t pack2(float a, float b) {
  const b16x2 v = __builtin_convertvector((f32x2{a, b}), b16x2);
  return __builtin_bit_cast(uint32_t, v);
}

template <int MH, int NH, int OUT>
__global__ __launch_bounds__(512, 2)
void tile_gemm_kernel(const uint16_t* __restrict__ x,
                      const uint16_t* __restrict__ w, void* __restrict__ out,
                      int M, int N, int K, int rows, int splits, int units) {
  using P = tile::Product<MH, NH>;
  constexpr int TM = P::TM, TN = P::TN;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];

  // Units of an XCD are consecutive: row tiles first, which read the same w.
  const int per = (units + 7) / 8;
  const int unit = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || unit >= units) return;
  const int m0 = unit % rows * TM;
  const int split = unit / rows % splits;
  const int panel = unit / rows / splits;
  const int n0 = panel * TN;
  const int steps = K / tile::KS;
  const int s0 = int(int64_t(steps) * split / splits);
  const int nk = int(int64_t(steps) * (split + 1) / splits) - s0;

  const int half = N / 2;
  P p;
  p.rows(
      [&](int r) { return uint32_t(min(m0 + r, M - 1)) * K * 2; },
      [&](int r) {
        if constexpr (OUT != OUT_SILU)
          return uint32_t(min(n0 + r, N - 1)) * K * 2;
        // gate rows, then the same ones of up
        const int h = r >= TN / 2, at = panel * TN / 2 + r - h * TN / 2;
        return uint32_t(h * half + min(at, half - 1)) * K * 2;
      });
  p.run(reinterpret_cast<const char*>(x + int64_t(s0) * tile::KS),
        reinterpret_cast<const char*>(w + int64_t(s0) * tile::KS), nk, 0,
        lds);

  if constexpr (OUT == OUT_PARTS) {
    float* y = static_cast<float*>(out) + int64_t(split) * M * N;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int i = 0; i < MH; ++i) {
        const int row = m0 + a * TM / 2 + P::row_of(i);
        if (row >= M) continue;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int j = 0; j < NH; ++j) {
            const int col = n0 + P::col_of(b, j);
            if (col < N)
              *reinterpret_cast<tile::f32x4*>(y + int64_t(row) * N + col) =
                  p.acc[a][b][i][j];
          }
      }
  } else {
    constexpr bool SILU = OUT == OUT_SILU;
    const int wide = SILU ? half : N;
#pragma unroll
    for (int i = 0; i < MH; ++i) {
      const int row = m0 + P::half_of() * TM / 2 + P::row_of(i);
#pragma unroll
      for (int b = 0; b < (SILU ? 1 : 2); ++b)
#pragma unroll
        for (int j = 0; j < NH; ++j) {
          uint2 v[2];
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            tile::f32x4 f = p.acc[a][b][i][j];
            if constexpr (SILU) {
#pragma unroll
              for (int r = 0; r < 4; ++r)
                f[r] = f[r] / (1.f + __expf(-f[r])) * p.acc[a][1][i][j][r];
            }
            if constexpr (OUT == OUT_RELU2) {
              // of the 16-bit product: a prompt's first tokens can turn any
              // difference to the product and relu2 apart into large ones
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                f[r] = fmaxf(bf16_to_f32(f32_to_bf16(f[r])), 0.f);
                f[r] *= f[r];
              }
            }
            v[a] = uint2{pack2(f[0], f[1]), pack2(f[2], f[3])};
          }
          const uint4 eight = P::eight(v[0], v[1]);
          const int col = panel * (SILU ? TN / 2 : TN) + P::eight_of(b, j);
          if (row < M && col < wide)
            *reinterpret_cast<uint4*>(static_cast<uint16_t*>(out) +
                                      int64_t(row) * wide + col) = eight;
        }
    }
  }
}

template <int MH, int NH, int OUT>
void go(const uint16_t* x, const uint16_t* w, void* out, int M, int N, int K,
        int splits, hipStream_t st) {
  constexpr int TM = 64 * MH, TN = 128 * NH;
  constexpr size_t smem = tile::Product<MH, NH>::LDS;
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
TilePlan tile_gemm_plan(int M, int N, int K, bool whole) {
  TilePlan best{};
  float least = 0.f;
  const int steps = K / tile::KS;
  for (const Tile& t : TILES) {
    const int rows = (M + 64 * t.mh - 1) / (64 * t.mh);
    const int tiles = rows * ((N + 128 * t.nh - 1) / (128 * t.nh));
    for (int s = 1; s <= (whole ? 1 : std::min(MOST_SPLITS, steps)); ++s) {
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

bool tile_gemm_ok(const TilePlan& plan, int K, bool whole) {
  return plan.splits >= 1 &&
         plan.splits <= (whole ? 1 : std::min(MOST_SPLITS, K / tile::KS)) &&
         std::any_of(std::begin(TILES), std::end(TILES), [&](const Tile& t) {
           return t.mh == plan.mh && t.nh == plan.nh;
         });
}

void launch_tile_gemm(const uint16_t* x, const uint16_t* w, float* parts,
                      uint16_t* out, int M, int N, int K, TileAct act,
                      const TilePlan& plan, hipStream_t st) {
  auto run = [&](auto m, auto n) {
    constexpr int MH = decltype(m)::value, NH = decltype(n)::value;
    if (act == TileAct::silu)
      go<MH, NH, OUT_SILU>(x, w, out, M, N, K, 1, st);
    else if (act == TileAct::relu2)
      go<MH, NH, OUT_RELU2>(x, w, out, M, N, K, 1, st);
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
