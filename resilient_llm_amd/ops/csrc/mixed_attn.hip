// Attention of a mixed step, prompt rows beside decoding sequences, in one
// launch: workgroups that multiply, prefill_flash.h's, and workgroups that read,
// decode_attn.h's, at the same time.
//
// A prompt tile is a chain of steps on one CU, 41 us for 512 rows behind 1500
// tokens, and 128 such tiles leave half the chip idle; divided by keys they fill
// it, for the price of parts that another launch puts together.  Decoding
// sequences need no more of the chip than their bytes ask of memory.  So tiles
// come first, in as few parts as keep the whole short (mixed_attn_plan), and
// the sequences go to the CUs that are left, and to others as they come free,
// whole where that is not the longest chain.  What is in parts, one more launch
// puts together.  A workgroup of either kind has a CU to itself (the tiles' LDS),
// and eight waves, so that one reading keeps 128 KB under way.
#include "decode_attn.h"
#include "kernels.h"
#include "prefill_flash.h"

#include <algorithm>
#include <type_traits>

namespace rlli {

namespace {

constexpr int NW = 8;             // a workgroup's waves, of either kind

template <int D, int GROUP, typename KC>
__global__ __launch_bounds__(64 * NW, 2)
void mixed_attn_kernel(Pages<KC> src, uint16_t* __restrict__ out, int n_tiles,
                       int tile_blocks, float scale, PrefillParts parts,
                       decode::DecodeArgs dec) {
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  using Lds = decode::Lds<D, GROUP, KC, NW>;
  static_assert(sizeof(Lds) <= FLASH_LDS<D, 2>, "");
  if (int(blockIdx.x) < tile_blocks)
    flash_tile<D, 4, 16, 2>(src, out, blockIdx.x, n_tiles, dec.n_kv, GROUP,
                            dec.q_stride, scale, parts, lds);
  else
    decode::attend<D, GROUP, KC, 16, false, decode::EITHER, NW>(
        dec, blockIdx.x - tile_blocks, *reinterpret_cast<Lds*>(lds));
}

template <int D, int GROUP, typename KC>
__global__ __launch_bounds__(256)
void mixed_combine_kernel(Pages<KC> src, uint16_t* __restrict__ out,
                          int tile_blocks, float scale, PrefillParts parts,
                          decode::DecodeArgs dec) {
  if (int(blockIdx.x) < tile_blocks)
    flash_combine<D>(src, out, blockIdx.x, dec.n_kv * GROUP, scale, parts);
  else
    decode::combine<D, GROUP>(dec, blockIdx.x - tile_blocks);
}

}  // namespace

// Which division should take least, from what its parts take, us: a tile's step
// of 128 keys 2.1, its start and end 6.5, 4 more with parts to write, and what
// writing and reading them takes at 5 TB/s; a round of a sequence's workgroup,
// 256 tokens, 3.2 and 5 around them, 3 around a part; the tables' room, more
// than half full, at 5 TB/s; another launch 3.  Workgroups of sequences start
// with those of tiles or, where these fill the chip, behind them.  (One after
// the other, so, and the best of 35 divisions, kernels by themselves, 32/8
// heads of 128, 24 sequences of 750 to 1500 tokens unless said otherwise: 512
// rows behind 1500 67.3, 46.7 (in the step 52) and 45.8; 64 behind 1500 56.4,
// 36.8 and 32.9; 256 behind 700 53.9, 28.6 and 28.6; 1500 behind 1500 125, 95
// and 93; 8 of 7000 beside 512 behind 7000 137, 124 and 113; 16 of 4000 beside
// 128 behind 4000 79.9, 55 and 52; 37 with an 8-bit cache beside 512 behind
// 1500 67.2, 49.3 and 47.9; 60 of 132 beside 52 behind 132, one after the other
// still, 17.0.)
//
// And whether that is less than one after the other, with the rates that tell the
// two apart at 2829 sizes: a step 2.6 (heads of 64 2.1, two workgroups a CU), 4.5
// around a sequence.  Alone, tiles are divided by prefill_splits and take several
// rounds where they are more than CUs; sequences have small workgroups that share a
// CU, so that many short ones are little, and read at 3.1 TB/s with a launch for
// their parts.  (64/8 heads of 128, 200 sequences of 16 tokens beside 512 rows 34
// and here 45; 8/1, 2048 rows of an 8-bit cache, which two parts halve, 46 and 50.
// Of those 2829, 1.17 times as fast in the mean, three below 0.95 by more than
// two runs differ: 8 of 4000 beside 200 behind 4000, 64/8 heads, 88 and 100.)
MixedPlan mixed_attn_plan(int n_tiles, int batch, int n_kv, int group,
                          int head_dim, int keys, int max_tokens, int elem,
                          int block_size) {
  MixedPlan best{0, 0, false};
  if (n_tiles == 0 || batch == 0 || block_size != 16 ||
      (group != 4 && group != 8) || !two_waves(n_tiles, n_kv, group, keys))
    return best;
  struct Rates {
    float step, seq;
    int places;                // workgroups that the chip holds
  };
  const Rates divide{2.1f, 5.f, 256};
  const Rates decide =
      head_dim == 128 ? Rates{2.6f, 4.5f, 256} : Rates{2.1f, 4.5f, 512};
  const int blocks = n_tiles * n_kv * (group / 4);
  const int steps = (keys + 2 * KT - 1) / (2 * KT);
  const float bytes = float(batch) * max_tokens * n_kv * head_dim * elem;
  const float round = 1.2f + 2.f * head_dim * elem / 256;
  const bool never_cut = decode_attn_shares(batch, n_kv, max_tokens) == 0;
  auto chain_of = [&](int n, const Rates& r) {
    return (steps + n - 1) / n * r.step + (n > 1 ? 10.5f : 6.5f);
  };
  auto parts_of = [&](int n) {
    const float of_one = 2.f * n_tiles * QR * n_kv * group * head_dim * 4;
    return n > 1 ? 3.f + n * of_one / 5e6f : 0.f;
  };
  auto together = [&](int n, int shares, const Rates& r) {
    const float chain = chain_of(n, r);
    const float late = blocks * n >= r.places ? chain : 0.f;
    const float all =
        (blocks * n * chain + n_kv * (shares ? shares * 3.f : batch * r.seq)) /
            r.places +
        1.2f * bytes / 5e6f;
    const float longest =
        shares ? 0.f : late + 5.f + (max_tokens + 255) / 256 * round;
    return std::max({chain, all, longest}) +
           (n > 1 ? parts_of(n) : shares ? 3.f : 0.f);
  };
  float least = 0.f;
  for (int n = 1; n <= std::max(1, std::min(16, 256 / blocks)); ++n) {
    if (n > 1 && (steps / n < 4 || (n_kv % 8 && n > 4 && n != 8 && n != 16)))
      continue;
    for (const bool cut : {false, true}) {
      if (cut && never_cut) continue;
      const int left = 256 - blocks * n;
      // Some more workgroups than CUs that are left (or come free): each costs
      // its start.
      const int shares =
          cut ? std::max(1, 5 * (left >= 64 ? left : 256) / (4 * n_kv)) : 0;
      const float us = together(n, shares, divide);
      if (best.splits == 0 || us < least) {
        best = MixedPlan{n, shares, false};
        least = us;
      }
    }
  }
  const int apart = prefill_splits(n_tiles, n_kv, group, keys);
  const float tiles = (chain_of(apart, decide) + parts_of(apart)) *
                      std::max(1.f, float(blocks * apart) / decide.places);
  const float walk = never_cut ? (max_tokens + 127) / 128 * 1.2f : 0.f;
  const float seqs = (never_cut ? 5.f : 9.f) +
                     std::max({5.f + walk, 4.f + bytes / 3.1e6f,
                               3.f + batch * n_kv * 0.65f / 256});
  // (fewer parts of the tiles than they have alone have to be worth it)
  best.faster = together(best.splits, best.shares, decide) *
                    (apart > best.splits ? 1.09f : 0.97f) <=
                tiles + seqs;
  return best;
}

void launch_mixed_attn(const uint16_t* qkv, void* k_cache, void* v_cache,
                       const int32_t* chunk_row0, const int32_t* chunk_pos0,
                       const int32_t* chunk_nrows, const int32_t* chunk_btrow,
                       const int32_t* tables_pre, int pre_blocks,
                       const int32_t* tables_dec, const int32_t* lens_dec,
                       int dec_blocks, uint16_t* out, int n_tiles, int batch,
                       int n_kv, int group, int head_dim, int stride,
                       float scale, bool cache_fp8, const PrefillParts& parts,
                       int shares, float* part_out, float* part_ml,
                       hipStream_t st) {
  auto go = [&](auto d, auto g, auto kc) {
    constexpr int D = decltype(d)::value, G = decltype(g)::value;
    using KC = decltype(kc);
    using elem = typename KC::elem;
    const Pages<KC> src{qkv, static_cast<const elem*>(k_cache),
                        static_cast<const elem*>(v_cache), chunk_row0,
                        chunk_pos0, chunk_nrows, chunk_btrow, tables_pre,
                        pre_blocks, 16};
    const decode::DecodeArgs dec{
        qkv, nullptr, k_cache, v_cache, nullptr, nullptr, tables_dec, lens_dec,
        nullptr, nullptr, nullptr, out, part_out, part_ml, batch, n_kv, 16,
        dec_blocks, stride, 0, shares, scale, false};
    const int tile_blocks = n_tiles * n_kv * (G / 4) * parts.splits;
    const int dec_wgs = (shares > 0 ? shares + batch : batch) * n_kv;
    auto* k = mixed_attn_kernel<D, G, KC>;
    constexpr size_t smem = FLASH_LDS<D, 2>;
    if (smem > 65536)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(smem));
    hipLaunchKernelGGL(k, dim3(tile_blocks + dec_wgs), dim3(64 * NW), smem, st,
                       src, out, n_tiles, tile_blocks, scale, parts, dec);
    const int tiles = parts.splits > 1 ? n_tiles * n_kv * G : 0;
    const int seqs = shares > 0 ? batch * n_kv * G : 0;
    if (tiles + seqs > 0)
      hipLaunchKernelGGL((mixed_combine_kernel<D, G, KC>), dim3(tiles + seqs),
                         dim3(256), 0, st, src, out, tiles, scale, parts, dec);
  };
  auto by_cache = [&](auto d, auto g) {
    if (cache_fp8) go(d, g, CacheFP8{}); else go(d, g, CacheBF16{});
  };
  auto by_group = [&](auto d) {
    if (group == 8) by_cache(d, std::integral_constant<int, 8>{});
    else by_cache(d, std::integral_constant<int, 4>{});
  };
  if (head_dim == 128) by_group(std::integral_constant<int, 128>{});
  else by_group(std::integral_constant<int, 64>{});
}

}  // namespace rlli
