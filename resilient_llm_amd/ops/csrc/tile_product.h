// The tiles of products on the matrix cores, x[rows, K] w[N, K]^T in bf16 with
// f32 sums, of tile_gemm.hip and moe.hip.
//
// A workgroup has a tile of 64 MH x 128 NH, eight waves two by four, each with
// MH x NH blocks of 16 x 16 in each quarter of the tile.  A 64-wide step of K
// is four phases, one quarter each: fragments are read from LDS, then
// multiplied.  The two waves of a SIMD take turns, one half-phase apart, so
// that one's products run while the other reads and asks for what comes next;
// a barrier ends each half-phase.  Steps come through two buffers in LDS by
// direct global -> LDS loads, half a tile's rows of x or w at a time, each as
// soon as its place was read for the last time: five to six phases ahead of
// its use, and waits count loads, so nothing drains.  The 16-byte pieces of a
// row are swizzled by the row, so that reading one piece of sixteen rows is
// free of bank conflicts.
//
// What bounds it is LDS, whose 192 KB of reads and 64 of writes a step of 256 x
// 256 take as long as its products, 2048 cycles: 2470 are needed, at 1.7 GHz,
// the clock under this load.  (With as many reads in the first phase as in the
// next two and a wait before each barrier, 2840.)
#pragma once

#include "common.h"

#include <type_traits>

namespace rlli {
namespace tile {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int KS = 64;

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

// Of 512 threads.  A tile's rows are numbered as they lie in LDS: those of x in
// two halves of TM / 2, those of w of TN / 2; wave group g (of four waves) has
// rows g * 16 MH on of each half of x, its wave n columns n * 16 NH on of each
// half of w.
template <int MH, int NH>
struct Product {
  static constexpr int TM = 64 * MH, TN = 128 * NH;
  static constexpr int STEP = (TM + TN) * KS;          // elements of a buffer
  static constexpr size_t LDS = size_t(2) * STEP * 2;  // bytes
  // loads are of 8 rows each: of w NH per half and wave, of x MH / 2, or one
  // and two by turns where that is not whole
  static constexpr int AL = (MH + 1) / 2;

  // acc[a][b][i][j]: block (i, j) of half a of x and b of w; a lane has four
  // columns of a row
  f32x4 acc[2][2][MH][NH];
  uint32_t ao[2][AL], bo[2][NH];                // bytes

  static DEV_INLINE int wave() {
    return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  }
  // a lane's row of a half of x, and the tile's column that its four start at
  static DEV_INLINE int row_of(int i) {
    return ((wave() >> 2) * MH + i) * 16 + (threadIdx.x & 15);
  }
  static DEV_INLINE int col_of(int b, int j) {
    return b * TN / 2 + ((wave() & 3) * NH + j) * 16 +
           (threadIdx.x >> 4 & 3) * 4;
  }
  // Four 16-bit results of a block in either half of x to eight of one of them,
  // so that 16 bytes a lane are stored: half the stores, whose number is what
  // leaving a tile takes (17 cycles each, 8700 for 256 x 256).  They are of the
  // half half_of() and the columns from eight_of() on.
  static DEV_INLINE uint4 eight(const uint2& first, const uint2& second) {
    const auto x =
        __builtin_amdgcn_permlane16_swap(first.x, second.x, false, false);
    const auto y =
        __builtin_amdgcn_permlane16_swap(first.y, second.y, false, false);
    return uint4{x[0], y[0], x[1], y[1]};
  }
  static DEV_INLINE int half_of() { return threadIdx.x >> 4 & 1; }
  // the tile's column that a lane's eight start at
  static DEV_INLINE int eight_of(int b, int j) {
    return b * TN / 2 + ((wave() & 3) * NH + j) * 16 +
           (threadIdx.x >> 5 & 1) * 8;
  }

  // x_at(r), w_at(r): where the tile's rows start, in bytes from x and w
  template <typename X, typename W>
  DEV_INLINE void rows(X x_at, W w_at) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < AL; ++j) {
        const int r = h * TM / 2 + x_load(j) * 8 + (lane >> 3);
        ao[h][j] = x_at(r) + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
      }
#pragma unroll
      for (int j = 0; j < NH; ++j) {
        const int r = h * TN / 2 + (j * 8 + wave()) * 8 + (lane >> 3);
        bo[h][j] = w_at(r) + ((lane & 7) ^ ((r >> 1) & 7)) * 16;
      }
    }
  }
  static DEV_INLINE int x_load(int j) {
    return j * 8 + (MH == 3 && j ? wave() & 3 : wave());
  }

  // nk steps of K from x and w on, nk > 0, the first of them ``rot`` < nk
  DEV_INLINE void run(const char* xb, const char* wb, int nk, int rot,
                      uint16_t* lds) {
    const int lane = threadIdx.x & 63;
    const int wv = wave(), group = wv >> 2, wn = wv & 3;
    // Where the next step's rows and those of the one after that begin; behind
    // the last step, the last is asked for again: nobody reads it.
    const uint32_t end = uint32_t(nk) * (KS * 2);
    const uint32_t last = (rot ? uint32_t(rot) * (KS * 2) : end) - KS * 2;
    uint32_t k1 = uint32_t(rot) * (KS * 2), k2 = k1;
    auto advance = [&] {
      k1 = k2;
      if (k2 != last) k2 = k2 + KS * 2 == end ? 0 : k2 + KS * 2;
    };
    // (offsets stay 32 bits wide beside a scalar address: kept as 64, they are
    // ten registers more, which the largest tile does not have)
    auto ask_x = [&](int s, uint32_t k, int h) {
      uint16_t* to = lds + (s & 1) * STEP + h * TM / 2 * KS;
#pragma unroll
      for (int j = 0; j < AL; ++j) {
        if (MH == 3 && j && h != group) continue;
        const int q = x_load(j);
        asm volatile("" : "+v"(ao[h][j]));
        lds_load16(xb + k + ao[h][j], to + q * 8 * KS);
      }
    };
    auto ask_w = [&](int s, uint32_t k, int h) {
      uint16_t* to = lds + (s & 1) * STEP + (TM + h * TN / 2) * KS;
#pragma unroll
      for (int j = 0; j < NH; ++j) {
        asm volatile("" : "+v"(bo[h][j]));
        lds_load16(wb + k + bo[h][j], to + (j * 8 + wv) * 8 * KS);
      }
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

#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int i = 0; i < MH; ++i)
#pragma unroll
          for (int j = 0; j < NH; ++j)
            acc[a][b][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

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
    // A step.  The halves of w take turns in being the first (F), which was
    // read in the step before, so that a phase reads one half and needs no
    // registers beyond.  (The largest tile has none for two forms of the step:
    // its first phase reads two halves.)
    constexpr bool TURNS = MH + NH < 6;
    auto step = [&](int s, auto first) {
      constexpr int F = decltype(first)::value;
      read_x(s, 0);
      if constexpr (!TURNS) read_w(s, F);
      ask_x(s + 1, k1, 1);
      wait_but(I1{}, I2{}, I2{});
      multiply(0, F);
      read_w(s, 1 - F);
      if constexpr (TURNS) ask_w(s + 2, k2, F);
      wait_but(I1{}, I1{}, std::integral_constant<int, TURNS ? 3 : 2>{});
      multiply(0, 1 - F);
      read_x(s, 1);
      ask_x(s + 2, k2, 0);
      if constexpr (TURNS) wait_but(I2{}, I1{}, I2{});
      else ask_w(s + 2, k2, F);
      multiply(1, 1 - F);
      if constexpr (TURNS) read_w(s + 1, 1 - F);
      ask_w(s + 2, k2, 1 - F);
      wait_but(I1{}, I1{}, I3{});
      advance();
      multiply(1, F);
    };

    ask_w(0, k1, 0);
    ask_x(0, k1, 0);
    ask_w(0, k1, 1);
    ask_x(0, k1, 1);
    advance();
    ask_w(1, k2, TURNS);
    ask_x(1, k2, 0);
    ask_w(1, k2, !TURNS);
    advance();
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
  }
};

}  // namespace tile
}  // namespace rlli
