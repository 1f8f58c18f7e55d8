// Paged GQA decode attention: one new query per sequence.
//
// What it costs is to read every key and value once, so the work is laid out
// by tokens: a wave takes units of 32 of them for the query heads of one
// key/value head, asks for all their keys and values at once (16 KB), and
// needs few registers beyond, so that three waves per SIMD (five with heads of
// 64) keep several times what memory's latency asks for under way.
//
// Both products run on the matrix cores, 16 tokens by 16 columns.  A query
// and a weight are 32-bit numbers: each is cut into three 16-bit ones that
// add up to it, all 24 bits, and for up to four heads the three are columns
// of one product (0-3 the heads' first parts, 4-7 the second, 12-15 the
// third), which costs nothing.  Eight heads take two products into the same
// sums: columns 0-7 have half of the first part in both, 8-15 the second part
// in one and the third in the other.  (With two parts, 16 bits, 0.36 % of the
// outputs were not the bf16 number nearest to the 64-bit result; so 0.029 %,
// with f32 products 0.028 %.  That, and infinite keys and values as they are,
// took the first three calls below from 12.1 to 12.6, from 45.1 to 45.6 and
// from 33.0 to 33.7 us.)
// Scores come out as the second product wants its weights: a lane holds four
// tokens of a column.
// The second product is transposed; row n of its tile t is channel VT n + t,
// so a lane loads VT neighbouring channels of each of its tokens, in whole
// rows, and makes the operands of all tiles from them.
//
// Who takes what, two ways:
//   whole sequences  a workgroup per (sequence, key/value head), for batches
//                    that fill the chip with contexts that are not long
//   parts            sequences are cut into parts of a size that follows
//                    from all lengths, so that about as many workgroups as
//                    the chip holds have about as much to do each, whatever
//                    the lengths are; decode_combine puts the parts of a
//                    sequence together
// Against as many parts for each sequence as the batch had of sequences, in
// lane groups with one accumulator each, 32/8 heads of 128, us: 64 sequences
// of 134-192 tokens 19.6 -> 12.8 (3.3 TB/s); 16 of 1.7k-4.1k 59 -> 46
// (4.3 TB/s, 5 but for what a launch, the lengths and the second kernel
// take); 37 of 1k-2k with an 8-bit cache 59 -> 34; one of 8000 33 -> 16.
//
// Fused form: rotation of q and k, the append to the cache and the new
// token's own term are part of it; that token's key and value come from LDS,
// so nothing waits for the append.  Without slots it rotates queries only.

#pragma once

#include "common.h"
#include "decode_parts.h"

#include <type_traits>

namespace rlli {
namespace decode {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct DecodeArgs {
  const uint16_t* q;       // rows q_stride apart: q heads (| k | v: fused)
  const float* parts;      // or n_parts f32 parts of them, to be summed
  const void *k_cache, *v_cache;     // [blocks, n_kv, block, D]
  void *k_cache_w, *v_cache_w;
  const int32_t* block_table;
  const int32_t* seq_lens;
  const int32_t* positions;
  const float* cos_sin;
  const int32_t* slot_mapping;
  uint16_t* out;
  float* part_out;         // shares: [n_kv, shares + batch, GROUP, D]
  float* part_ml;          //         [.., GROUP, 2]
  int batch, n_kv, block_size, max_blocks, q_stride, n_parts, shares;
  float scale;
  bool apart;              // whoever reads the parts puts them together
};

// Sums of the lanes up to each; all lanes at once.  (On the VALU: fourteen steps
// through LDS ahead of everything else were 0.5 us.)
DEV_INLINE int sums_upto(int v) {
  auto add = [&](auto ctrl, auto rows) {
    v += __builtin_amdgcn_update_dpp(0, v, decltype(ctrl)::value,
                                     decltype(rows)::value, 0xf, false);
  };
  using All = std::integral_constant<int, 0xf>;
  add(std::integral_constant<int, 0x111>{}, All{});     // row_shr 1, 2, 4, 8
  add(std::integral_constant<int, 0x112>{}, All{});
  add(std::integral_constant<int, 0x114>{}, All{});
  add(std::integral_constant<int, 0x118>{}, All{});
  // the row before's last to rows 1 and 3, the lower half's to the upper
  add(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});
  add(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});
  return v;
}

// How many units a part may have, so that ``shares`` parts cover all
// sequences (each ends in one that is not full).
// (``own``: the length of the lane's sequence, of the first 64; or 0.)
DEV_INLINE int part_size(const DecodeArgs& a, int own) {
  int t = units_of(own);
  for (int s = (threadIdx.x & 63) + 64; s < a.batch; s += 64)
    t += units_of(a.seq_lens[s]);
  return part_size_of(__builtin_amdgcn_readlane(sums_upto(t), 63), a.shares,
                      a.batch);
}

// Parts of the sequences ahead of ``seq``.
DEV_INLINE int parts_before(const DecodeArgs& a, int size, int seq) {
  int t = 0;
  for (int s = threadIdx.x & 63; s < seq; s += 64)
    t += parts_of(a.seq_lens[s], size);
  return __builtin_amdgcn_readlane(sums_upto(t), 63);
}

// The sequence that part number ``part`` belongs to (a.batch: none), its length
// and which of its parts it is.
DEV_INLINE int find_part(const DecodeArgs& a, int own, int size, int part,
                         int& len, int& rel) {
  const int lane = threadIdx.x & 63;
  int before = 0;
  for (int s0 = 0; s0 < a.batch; s0 += 64) {
    if (s0 > 0) own = s0 + lane < a.batch ? a.seq_lens[s0 + lane] : 0;
    const int mine = parts_of(own, size);
    const int upto = sums_upto(mine);
    const int at = part - before;
    const uint64_t hit = __ballot(at < upto && at >= upto - mine);
    if (hit) {
      const int src = __builtin_amdgcn_readfirstlane(__builtin_ctzll(hit));
      rel = at - __builtin_amdgcn_readlane(upto - mine, src);
      len = __builtin_amdgcn_readlane(own, src);
      return s0 + src;
    }
    before += __builtin_amdgcn_readlane(upto, 63);
  }
  len = rel = 0;
  return a.batch;
}

// for what goes through LDS; loads from memory stay under way
DEV_INLINE void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// the sum of the parts in a head's columns, HS apart; the same bits in each.
// (Of up to four heads, second and third part first: they are eight columns
// apart, and so are the first and the idle column, where a query's part is the
// least number.)
template <int HS>
DEV_INLINE float sum_parts(float v) {
  v += dpp_mov_f32<0x128>(v);
  if constexpr (HS == 4) v += dpp_mov_f32<0x124>(v);
  return v;
}

// N bytes of cache elements, in registers
template <int N>
struct Words {
  typedef uint32_t type __attribute__((ext_vector_type(N / 4)));
};
template <>
struct Words<4> {
  using type = uint32_t;
};

DEV_INLINE uint32_t word(uint32_t w, int) { return w; }
template <typename V>
DEV_INLINE uint32_t word(const V& w, int i) { return w[i]; }

// The upper half of a 32-bit float is a bf16 number, its first eight bits; what
// is left has sixteen, of which its upper half has eight, and the rest fits a
// bf16 number.
constexpr uint32_t kUpper = 0xffff0000u;
constexpr float kLeast = 0x1p-120f;

DEV_INLINE float masked(float v, uint32_t mask) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & mask);
}
DEV_INLINE uint16_t upper_half(float v) {
  return uint16_t(__builtin_bit_cast(uint32_t, v) >> 16);
}
DEV_INLINE uint32_t upper_halves(float a, float b) {
  return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b),
                               __builtin_bit_cast(uint32_t, a), 0x07060302u);
}

// cache elements as bf16 (8-bit ones are exact in it), two per dword; by one
// conversion a pair (through 32-bit floats, and with keys loaded 8 bytes a
// lane, 37 sequences of 1k-2k took 40 us)
template <typename KC, int N, typename R>
DEV_INLINE void widen(const R& raw, uint32_t (&out)[N]) {
  if constexpr (std::is_same<KC, CacheBF16>::value) {
#pragma unroll
    for (int i = 0; i < N; ++i) out[i] = word(raw, i);
  } else {
#pragma unroll
    for (int i = 0; i < N; i += 2) {
      const uint32_t w = word(raw, i / 2);
      out[i] = __builtin_bit_cast(
          uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, false));
      out[i + 1] = __builtin_bit_cast(
          uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, true));
    }
  }
}

// What a workgroup of NW waves keeps in LDS.
template <int D, int GROUP, typename KC, int NW>
struct Lds {
  static constexpr int QROW = D + 8;
  // queries by part and head: of up to four heads as the columns have them,
  // of eight first (halved), second, third part
  static constexpr int QROWS = GROUP <= 4 ? 16 : 24;
  alignas(16) float raw[(GROUP + 2) * D];
  alignas(16) uint16_t qs[QROWS * QROW];
  alignas(16) typename KC::elem self[2 * D];       // k | v
  alignas(16) float accs[NW * GROUP * D];
  float ml[NW * GROUP * 2];
};

enum Cut { WHOLE, SHARES, EITHER };      // EITHER: as a.shares says

// Workgroup ``block``, of NW waves.  BS: block size of the cache where it is
// known (0: any)
template <int D, int GROUP, typename KC, int BS, bool FUSED, Cut CUT, int NW>
DEV_INLINE void attend(const DecodeArgs& a, unsigned block,
                       Lds<D, GROUP, KC, NW>& lds) {
  using elem = typename KC::elem;
  using vec8 = typename KC::vec8;
  constexpr int KSTEPS = D / 32;
  constexpr int VT = D / 16;               // channel tiles
  // A lane's 16 bytes of a key are the channels of KPL steps of the scores'
  // product: step k has of lane group ``oct`` those from k_chan(k).
  constexpr int KPL = 2 / sizeof(elem), KLOADS = KSTEPS / KPL;
  using kraw = typename Words<16>::type;
  using vraw = typename Words<sizeof(elem) * VT>::type;
  constexpr int QROW = Lds<D, GROUP, KC, NW>::QROW, NT = NW * 64;
  constexpr int HS = GROUP <= 4 ? 4 : 8;   // columns of a part
  float* raw = lds.raw;
  uint16_t* qs = lds.qs;
  elem* self = lds.self;
  float *accs = lds.accs, *ml = lds.ml;
  const bool cut = CUT == SHARES || (CUT == EITHER && a.shares > 0);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, oct = lane >> 4;
  const int cpart = col / HS;              // of its head's query or weight
  const uint32_t mask1 = cpart > 0 ? kUpper : 0, mask2 = cpart > 1 ? kUpper : 0;
  const int bs = BS ? BS : a.block_size;
  const elem* kc = static_cast<const elem*>(a.k_cache);
  const elem* vc = static_cast<const elem*>(a.v_cache);
  const int n_q = a.n_kv * GROUP;
  const float c2 = a.scale * 1.4426950408889634f;
  auto k_chan = [&](int k) {
    return k / KPL * 32 * KPL + (oct * KPL + k % KPL) * 8;
  };

  int kvh, seq, len, part = 0, u0 = 0, u1, n_parts = 1;
  kvh = block % a.n_kv;
  if (cut) {
    part = block / a.n_kv;
    const int own = lane < a.batch ? a.seq_lens[lane] : 0;
    const int size = part_size(a, own);
    int rel;
    seq = find_part(a, own, size, part, len, rel);
    if (seq >= a.batch) return;
    const int all = units_of(len);
    n_parts = parts_of(len, size);
    u0 = all * rel / n_parts;
    u1 = all * (rel + 1) / n_parts;
  } else {
    seq = block / a.n_kv;
    len = a.seq_lens[seq];
    u1 = units_of(len);
  }
  // whether this workgroup appends the new token
  const bool newest = FUSED && a.slot_mapping && u1 == units_of(len);
  // what later loads and stores go by
  const int position = FUSED ? a.positions[seq] : 0;
  const int slot_at = newest ? a.slot_mapping[seq] : 0;

  const int32_t* table = a.block_table + int64_t(seq) * a.max_blocks;
  const int last = len - 1;
  // Pages of a unit: of its two halves where a half lies in one page,
  // otherwise of this lane's key and value tokens.
  constexpr int NPG = BS == 16 ? 2 : 10;
  int page[NPG];
  auto key_tok = [&](int u, int t) {     // tokens past the last repeat it
    return min(u * UNIT + t * 16 + col, last);
  };
  auto value_tok = [&](int u, int t, int i) {
    return min(u * UNIT + t * 16 + oct * 4 + i, last);
  };
  auto look_up = [&](int u) {
    if (u >= u1) return;
    if constexpr (BS == 16) {
#pragma unroll
      for (int t = 0; t < 2; ++t) page[t] = table[min(u * 2 + t, last / 16)];
    } else {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        page[t * 5] = table[key_tok(u, t) / bs];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          page[t * 5 + 1 + i] = table[value_tok(u, t, i) / bs];
      }
    }
  };
  auto row_of = [&](int u, int t, int i, int tok) -> int64_t {
    if constexpr (BS == 16)
      return (int64_t(page[t]) * a.n_kv + kvh) * 16 + tok -
             min(u * 2 + t, last / 16) * 16;
    else
      return (int64_t(page[t * 5 + i]) * a.n_kv + kvh) * bs + tok % bs;
  };
  kraw kr[2][KLOADS];
  vraw vr[2][4];
  auto load_keys = [&](int u) {
    if (u >= u1) return;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const elem* p = kc + row_of(u, t, 0, key_tok(u, t)) * D + k_chan(0);
#pragma unroll
      for (int k = 0; k < KLOADS; ++k)
        kr[t][k] = *reinterpret_cast<const kraw*>(p + k * 32 * KPL);
    }
  };
  // Whole lines that nobody reads again pass the caches by (16 sequences of
  // 1.7k-4.1k: 49.0 -> 46.0 us); an instruction takes halves of lines of the
  // keys, which come slower so (47.2).
  auto load_values = [&](int u) {
    if (u >= u1) return;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        vr[t][i] = __builtin_nontemporal_load(reinterpret_cast<const vraw*>(
            vc + row_of(u, t, 1 + i, value_tok(u, t, i)) * D + col * VT));
  };
  look_up(u0 + wave);
  // ---- the heads' queries (and the new key and value) -----------------
  // All that a lane takes of them is asked for at once, ahead of keys and values.
  // (Part after part, then the position, the rotation and the slot are four to
  // eight waits more, one behind the other.  us, with sums over lanes through LDS
  // and now: one sequence of 101 tokens, 64-wide heads, five parts 5.7 and 4.9; of
  // 1000, 128-wide, two parts 7.4 and 6.8; 64 of 192 10.7 and 10.3; 16 of 1.7k to
  // 4.1k 30.7 and 30.1; 37 of 1k to 2k with an 8-bit cache 21.2 and 20.3.)
  constexpr int EARLY = 8;                 // parts of the product
  const int n_in = (GROUP + (newest ? 2 : 0)) * D;
  auto place = [&](int e) {
    int at = kvh * GROUP * D + e;
    if (e >= GROUP * D) {
      const int r = e - GROUP * D;
      at = r < D ? (n_q + kvh) * D + r : (n_q + a.n_kv + kvh) * D + r - D;
    }
    return int64_t(seq) * a.q_stride + at;
  };
  const int64_t part_step = int64_t(a.batch) * a.q_stride;
  f32x4 early[EARLY];
  uint2 early_q{0, 0};
  auto ask = [&](int e) {
    if (a.parts) {
      const float* p = a.parts + place(e);
#pragma unroll
      for (int s = 0; s < EARLY; ++s)
        if (s < a.n_parts)
          early[s] = *reinterpret_cast<const f32x4*>(p + s * part_step);
    } else {
      early_q = *reinterpret_cast<const uint2*>(a.q + place(e));
    }
  };
  if (tid * 4 < n_in) ask(tid * 4);
  // (a thread's channel is the same of all heads)
  float cosine = 1.f, sine = 0.f;
  if constexpr (FUSED) {
    const float* cs = a.cos_sin + int64_t(position) * D + tid % (D / 2);
    cosine = cs[0];
    sine = cs[D / 2];
  }
  load_keys(u0 + wave);
  load_values(u0 + wave);
  look_up(u0 + wave + NW);

  for (int e = tid * 4; e < n_in; e += NT * 4) {
    if (e != tid * 4) ask(e);
    f32x4 v;
    if (a.parts) {
      v = early[0];
#pragma unroll
      for (int s = 1; s < EARLY; ++s)
        if (s < a.n_parts) v += early[s];
      const float* p = a.parts + place(e);
      for (int s = EARLY; s < a.n_parts; ++s)
        v += *reinterpret_cast<const f32x4*>(p + s * part_step);
      // the product is a 16-bit one
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = bf16_to_f32(f32_to_bf16(v[i]));
    } else {
      const uint2 w = early_q;
      v = f32x4{__builtin_bit_cast(float, w.x << 16),
                __builtin_bit_cast(float, w.x & 0xffff0000u),
                __builtin_bit_cast(float, w.y << 16),
                __builtin_bit_cast(float, w.y & 0xffff0000u)};
    }
    *reinterpret_cast<f32x4*>(raw + e) = v;
  }
  lds_barrier();
  {
    constexpr int HALF = D / 2;
    static_assert(NT % HALF == 0, "");
    auto store = [&](int h, int d, float v) {
      // All parts have the sign of the first, and none is zero, so that an
      // infinite key makes all of a score's parts infinite alike and not NaN.
      const float least = copysignf(kLeast, v);
      const float r0 = v - masked(v, kUpper) + least;
      const float r1 = r0 - masked(r0, kUpper) + least;
      qs[h * QROW + d] = upper_half(HS == 4 ? v : 0.5f * v);
      qs[(HS + h) * QROW + d] = upper_half(r0);
      qs[(2 * HS + h) * QROW + d] = upper_half(HS == 4 ? least : r1);
      if (HS == 4) qs[(3 * HS + h) * QROW + d] = upper_half(r1);
    };
    for (int e = tid; e < (GROUP + (newest ? 1 : 0)) * HALF; e += NT) {
      const int h = e / HALF, j = e % HALF;
      const float u = raw[h * D + j], v = raw[h * D + HALF + j];
      float x = u, y = v;
      if constexpr (FUSED) {
        x = fmaf(u, cosine, -(v * sine));
        y = fmaf(v, cosine, u * sine);
      }
      if (h < GROUP) {
        store(h, j, x);
        store(h, HALF + j, y);
      } else {
        raw[h * D + j] = x;
        raw[h * D + HALF + j] = y;
      }
    }
  }
  lds_barrier();
  if (newest) {
    // append at cache precision; this step sees what later ones will
    if (tid < 2 * D / 8) {
      const int e = tid * 8;
      const vec8 w = KC::from_f32(raw + GROUP * D + e);
      const int slot = slot_at;
      elem* to = static_cast<elem*>(e < D ? a.k_cache_w : a.v_cache_w);
      *reinterpret_cast<vec8*>(
          to + ((int64_t(slot / bs) * a.n_kv + kvh) * bs + slot % bs) * D +
          e % D) = w;
      *reinterpret_cast<vec8*>(self + e) = w;
    }
    lds_barrier();
  }
  s16x8 qf[KSTEPS];
#pragma unroll
  for (int k = 0; k < KSTEPS; ++k) {
    uint4 w{0, 0, 0, 0};
    if (col % HS < GROUP)
      w = *reinterpret_cast<const uint4*>(qs + col * QROW + k_chan(k));
    qf[k] = __builtin_bit_cast(s16x8, w);
  }

  // ---- units; the next one's loads as soon as registers are free ------
  f32x4 o[VT];
#pragma unroll
  for (int t = 0; t < VT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNegInf, l = 0.f;
  for (int u = u0 + wave; u < u1; u += NW) {
    const int tok0 = u * UNIT;
    if (newest && tok0 + UNIT > last) {
      // the new token's key and value instead of what its slot held
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const bool own = key_tok(u, t) == last;
#pragma unroll
        for (int k = 0; k < KLOADS; ++k) {
          const kraw w =
              *reinterpret_cast<const kraw*>(self + k_chan(k * KPL));
          kr[t][k] = own ? w : kr[t][k];
        }
      }
      const vraw w = *reinterpret_cast<const vraw*>(self + D + col * VT);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          vr[t][i] = value_tok(u, t, i) == last ? w : vr[t][i];
    }
    f32x4 s[2];
    // (read again for each unit: registers are short)
    if constexpr (HS == 8) asm volatile("" ::: "memory");
    const uint16_t* third = qs + (col < 8 ? col : col + 8) * QROW;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KLOADS; ++k) {
        uint32_t w[4 * KPL];
        widen<KC>(kr[t][k], w);
#pragma unroll
        for (int j = 0; j < KPL; ++j) {
          const s16x8 kf =
              __builtin_bit_cast(s16x8, (uint4{w[j * 4], w[j * 4 + 1],
                                               w[j * 4 + 2], w[j * 4 + 3]}));
          s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              kf, qf[k * KPL + j], s[t], 0, 0, 0);
          if constexpr (HS == 8)
            s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                kf,
                *reinterpret_cast<const s16x8*>(third + k_chan(k * KPL + j)),
                s[t], 0, 0, 0);
        }
      }
    }
    load_keys(u + NW);
    float mx = kNegInf;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tok = tok0 + t * 16 + oct * 4 + r;
        const float v = sum_parts<HS>(s[t][r]) * c2;
        s[t][r] = tok <= last ? v : kNegInf;
        mx = fmaxf(mx, s[t][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, kWave));
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    const float mn = fmaxf(m, mx);
    if (!__all(mn == m)) {
      const float corr = __builtin_amdgcn_exp2f(m - mn);
      l *= corr;
#pragma unroll
      for (int t = 0; t < VT; ++t) o[t] *= corr;
      m = mn;
    }
    // this column's part of the weights: what is left of them when the parts
    // before are taken off, its upper half
    uint32_t pw[2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float x[2], y[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const float p = __builtin_amdgcn_exp2f(s[i / 2][i % 2 * 2 + r] - m);
        l += p;
        x[r] = fmaf(p, HS == 4 || cpart ? 1.f : 0.5f, -masked(p, mask1));
        y[r] = x[r] - masked(x[r], HS == 4 ? mask2 : mask1);
      }
      if constexpr (HS == 8) pw[1][i] = upper_halves(x[0], x[1]);
      pw[0][i] = upper_halves(y[0], y[1]);
    }
    s16x8 pf[2];
#pragma unroll
    for (int i = 0; i < HS / 4; ++i)
      pf[i] = __builtin_bit_cast(
          s16x8, (uint4{pw[i][0], pw[i][1], pw[i][2], pw[i][3]}));
    // what repeats the last value may be infinite, of which no weight makes zero
    if (std::is_same<KC, CacheBF16>::value && tok0 + UNIT > len)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (tok0 + t * 16 + oct * 4 + i > last) vr[t][i] = vraw{};
    uint32_t vw[2][4][VT / 2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) widen<KC>(vr[t][i], vw[t][i]);
#pragma unroll
    for (int t = 0; t < VT; ++t) {
      const uint32_t sel = t & 1 ? 0x07060302u : 0x05040100u;
      const int d = t / 2;
      const uint4 w = {
          __builtin_amdgcn_perm(vw[0][1][d], vw[0][0][d], sel),
          __builtin_amdgcn_perm(vw[0][3][d], vw[0][2][d], sel),
          __builtin_amdgcn_perm(vw[1][1][d], vw[1][0][d], sel),
          __builtin_amdgcn_perm(vw[1][3][d], vw[1][2][d], sel)};
#pragma unroll
      for (int i = 0; i < HS / 4; ++i)
        o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(s16x8, w), pf[i], o[t], 0, 0, 0);
    }
    load_values(u + NW);
    look_up(u + 2 * NW);
  }

  // ---- the waves' results, through LDS ---------------------------
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      // to the first part's column; of four heads the idle columns have the
      // third part once more
      const float v = o[t][r];
      const float sum =
          HS == 4 ? v + (dpp_mov_f32<0x12c>(v) + dpp_mov_f32<0x124>(v))
                  : sum_parts<HS>(v);
      o[t][r] = __builtin_isinf(v) ? v : sum;    // of infinite values
    }
  if (col < GROUP) {
    float* to = accs + (wave * GROUP + col) * D + oct * 4 * VT;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < VT; t += 4)
        *reinterpret_cast<f32x4*>(to + r * VT + t) =
            f32x4{o[t][r], o[t + 1][r], o[t + 2][r], o[t + 3][r]};
    if (oct == 0) {
      ml[(wave * GROUP + col) * 2] = m;
      ml[(wave * GROUP + col) * 2 + 1] = l;
    }
  }
  lds_barrier();
  const bool whole = !cut || n_parts == 1;
  const int64_t slot =
      (int64_t(kvh) * (a.shares + a.batch) + part) * GROUP;
  for (int e = tid; e < GROUP * D; e += NT) {
    const int h = e / D, d = e % D;
    float M = kNegInf;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, ml[(w * GROUP + h) * 2]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float c = __builtin_amdgcn_exp2f(ml[(w * GROUP + h) * 2] - M);
      num += c * accs[(w * GROUP + h) * D + d];
      den += c * ml[(w * GROUP + h) * 2 + 1];
    }
    if (whole) {
      a.out[(int64_t(seq) * n_q + kvh * GROUP + h) * D + d] =
          f32_to_bf16(den > 0.f ? num / den : 0.f);
    } else {
      a.part_out[(slot + h) * D + d] = num;
      if (d == 0) {
        a.part_ml[(slot + h) * 2] = M;
        a.part_ml[(slot + h) * 2 + 1] = den;
      }
    }
  }
  }

// Sequences of several parts (and those without tokens), by 256 threads.  A
// workgroup per (sequence, query head): D / 4 threads have a part's channels,
// the others other parts.
template <int D, int GROUP>
DEV_INLINE void combine(const DecodeArgs& a, unsigned block) {
  constexpr int TD = D / 4, NG = 256 / TD;
  const int n_q = a.n_kv * GROUP;
  const int seq = block / n_q, h = block % n_q;
  const int kvh = h / GROUP;
  const int lane = threadIdx.x & 63;
  const int size = part_size(a, lane < a.batch ? a.seq_lens[lane] : 0);
  const int n = parts_of(a.seq_lens[seq], size);
  if (n == 1) return;
  const int first = parts_before(a, size, seq);
  const int td = threadIdx.x % TD, tg = threadIdx.x / TD;
  const int64_t slot0 =
      (int64_t(kvh) * (a.shares + a.batch) + first) * GROUP + h % GROUP;
  const float* po = a.part_out + slot0 * D + td * 4;
  const float* pm = a.part_ml + slot0 * 2;
  float M = kNegInf, den = 0.f;
  f32x4 num = {0.f, 0.f, 0.f, 0.f};
  // four parts' loads at a time
  for (int g = tg; g < n; g += 4 * NG) {
    f32x4 v[4];
    float mm[4], ll[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool ok = g + i * NG < n;
      const int64_t at = int64_t(ok ? g + i * NG : g) * GROUP;
      v[i] = *reinterpret_cast<const f32x4*>(po + at * D);
      if (!ok) v[i] = f32x4{0.f, 0.f, 0.f, 0.f};     // not 0 * inf
      mm[i] = ok ? pm[at * 2] : kNegInf;
      ll[i] = ok ? pm[at * 2 + 1] : 0.f;
    }
    const float mn =
        fmaxf(M, fmaxf(fmaxf(mm[0], mm[1]), fmaxf(mm[2], mm[3])));
    const float corr = __builtin_amdgcn_exp2f(M - mn);
    num *= corr;
    den *= corr;
    M = mn;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float c = g + i * NG < n ? __builtin_amdgcn_exp2f(mm[i] - mn) : 0.f;
      num += c * v[i];
      den += c * ll[i];
    }
  }
  __shared__ f32x4 nums[NG][TD];
  __shared__ float ms[NG], dens[NG];
  nums[tg][td] = num;
  if (td == 0) {
    ms[tg] = M;
    dens[tg] = den;
  }
  __syncthreads();
  if (threadIdx.x >= D) return;
  M = kNegInf;
#pragma unroll
  for (int g = 0; g < NG; ++g) M = fmaxf(M, ms[g]);
  float x = 0.f, y = 0.f;
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const float c = __builtin_amdgcn_exp2f(ms[g] - M);
    x += c * nums[g][threadIdx.x / 4][threadIdx.x % 4];
    y += c * dens[g];
  }
  a.out[(int64_t(seq) * n_q + h) * D + threadIdx.x] =
      f32_to_bf16(y > 0.f ? x / y : 0.f);
}

}  // namespace decode
}  // namespace rlli
