// Causal prompt attention on the matrix cores (bf16 products, f32 softmax):
// over the rows of a batch of whole prompts, or over the pages of a cache
// that holds a sequence's earlier tokens as well.
//
// A workgroup takes 32 rows of a sequence and up to four query heads of one
// key/value head, a wave a head each, so that keys and values of a 64-key
// tile are staged once for 128 (row, head) queries.  Tiles are double-
// buffered in LDS; 16-bit ones arrive by direct global -> LDS loads that are
// in flight under the products of the tile before, 8-bit ones pass through
// registers, where they are widened.
//
// Scores are computed transposed (keys down, queries across): a lane holds
// 32 scores of one query, the maximum needs one cross-lane step, and the
// weights are the second product's operand as they are, keys in the order
// 0-3, 8-11 | 4-7, 12-15 of sixteen.  Its other operand, values by channel,
// is read from the row-major tile with the transposing LDS read in just that
// order, so nothing transposes values on the way in.  A query's accumulators
// are scaled again in the tiles where its maximum grows, few in a long prompt:
// the largest weight is then exactly one, which later growth by a factor would
// not leave so.  The sum of weights is that of the 16-bit ones, two at a time
// by dot products, so that their rounding is in both sides of the quotient
// (error against 64 bits with the sum of the 32-bit ones and growth by up to
// 2^8: 0.00205, with three times the scale 0.00212; so: 0.00198 and 0.00175).
//
// Bounds: for long prompts the products (32 MFMA of 32 cycles a tile and
// wave) beside about as many cycles of exponentials and conversions and of
// LDS reads; two workgroups share a CU so that one computes while the other
// does the rest.  Against 16x16 tiles of 32 rows with weights through LDS and
// values transposed on the way in, 32/8 heads of 128: a prompt of 7901 rows
// 3850 -> 623 us (133 -> 820 TF), 64 prompts of 128 rows 140 -> 50 us, 512
// rows behind 1500 cached tokens 236 -> 45 us.

#pragma once

#include "common.h"
#include "prefill_parts.h"

#include <type_traits>

namespace rlli {

namespace {

typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));

constexpr float kHidden = -3e38f;
constexpr int QR = 32;            // rows of a tile
constexpr int KT = 64;            // keys of a tile

DEV_INLINE uint32_t pack2(float a, float b) {
  const b16x2 v = __builtin_convertvector((f32x2{a, b}), b16x2);
  return __builtin_bit_cast(uint32_t, v);
}

// both halves of ``p`` added to ``l``
DEV_INLINE float add2(uint32_t p, float l) {
  return __builtin_amdgcn_fdot2_f32_bf16(
      __builtin_bit_cast(b16x2, p), __builtin_bit_cast(b16x2, 0x3f803f80u), l,
      false);
}

DEV_INLINE void lds_load16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds(
      (const __attribute__((address_space(1))) void*)g,
      (__attribute__((address_space(3))) void*)l, 16, 0, 0);
}

// four keys of this lane's channel; see prefill_flash_kernel for addresses
DEV_INLINE s16x4 read_tr(const uint16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s16x4*)p);
}

// Eight channels of a rotated row, of its lower or upper half, from those and
// their partners; ``cs``: the cosines, ``half`` before the sines.
DEV_INLINE void rotate8(bool lower, const uint4& own, const uint4& other,
                        const float* cs, int half, float* out) {
  bf16x8 a, b;
  a.u = lower ? own : other;
  b.u = lower ? other : own;
  float c[8], s[8];
#pragma unroll
  for (int i = 0; i < 8; i += 4) {
    *reinterpret_cast<float4*>(c + i) =
        *reinterpret_cast<const float4*>(cs + i);
    *reinterpret_cast<float4*>(s + i) =
        *reinterpret_cast<const float4*>(cs + half + i);
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float x = bf16_to_f32(a.s[i]), y = bf16_to_f32(b.s[i]);
    // rope_lower and rope_upper
    out[i] = fmaf(x, lower ? c[i] : s[i], y * (lower ? -s[i] : c[i]));
  }
}

DEV_INLINE uint4 flipped(const uint4& v, const uint4& f) {
  return uint4{v.x ^ f.x, v.y ^ f.y, v.z ^ f.z, v.w ^ f.w};
}

// A source says where a workgroup's rows and keys are.  find(): which rows
// are this tile's; false: none.  A windowed one also says which keys a row
// sees (``window`` of them and the first ``keep``) and a head's sink.  Of kRope
// the rows are as the product left them, one tile of keys a sequence at most:
// queries and keys are rotated on their way in, and a tile of rows writes their
// keys and values to the cache.

template <typename C>
struct Pages {                    // [blocks, n_kv, block, D]
  static constexpr bool kPaged = true, kWindow = false, kRope = false;
  using KC = C;
  const uint16_t* qkv;
  const typename C::elem *k, *v;
  const int32_t *row0s, *pos0s, *nrowss, *btrows, *tables;
  int max_blocks, block_size;

  DEV_INLINE bool find(int tile, int& row0, int& nrows, int& first,
                       int& pos0) const {
    row0 = row0s[tile];
    pos0 = pos0s[tile];
    nrows = nrowss[tile];
    first = btrows[tile];
    return nrows > 0;
  }
};

// How many parts a tile's steps of KS tiles of keys are divided into.
DEV_INLINE int parts_of(int steps, int splits) {
  return min(splits, max(steps / 4, 1));
}

template <int D, int KS>
constexpr size_t FLASH_LDS = size_t(2) * KS * 2 * KT * D * 2;

// D: head width; W: heads, a wave each; BS: block size of the cache where it
// is known; KS: waves per head, each with every KS-th tile of keys, for
// launches that leave CUs idle.  Their sums meet in LDS.
// ``lds`` holds two stages, FLASH_LDS bytes.  (``out`` is not __restrict__ here: of
// a function that is inlined that makes the compiler wait for all reads of the values
// ahead of the first product, 3 to 5 % of long prompts.)
template <int D, int W, int BS, int KS, typename Src>
DEV_INLINE void flash_tile(const Src& src, uint16_t* out, unsigned block,
                           int n_tiles, int n_kv, int group, int stride,
                           float scale, const PrefillParts& parts,
                           uint16_t* lds) {
  using KC = typename Src::KC;
  constexpr bool kRope = Src::kRope;
  constexpr bool kDirect = std::is_same<KC, CacheBF16>::value && !kRope;
  static_assert(KS == 1 || !Src::kWindow, "windows skip single tiles");
  constexpr int NT = 64 * W * KS;
  constexpr int CH = D / 8;                  // 16-byte pieces of a row
  constexpr int NP = KS * KT * CH / NT;      // pieces a thread stages
  constexpr int DC = D / 16;                 // steps of a score's product
  constexpr int VT = D / 32;                 // channel tiles
  constexpr int HALF = KT * D;
  constexpr int STAGE = KS * 2 * HALF;       // keys | values, of KS tiles

  // the tiles of a key/value head stay on an XCD (workgroups go to XCDs in
  // turn), those with the longest context first
  const int splits = KS > 1 ? parts.splits : 1;
  const int per_head = n_tiles * (group / W) * splits;
  int kvh, i;
  if (n_kv % 8 == 0) {
    i = block / 8;
    kvh = i / per_head * 8 + block % 8;
  } else {
    i = block;
    kvh = i / per_head;
  }
  i %= per_head;
  const int part = i % splits;
  i /= splits;
  const int tile = n_tiles - 1 - i / (group / W);
  int row0, nrows, first, pos0;
  // (of kRope, a lane's row's: asked for beside what find() reads)
  int place = 0, slot = 0;
  if constexpr (Src::kRope) {
    const int r = min(int(threadIdx.x) & 63, src.rows - 1);
    place = src.positions[r];
    slot = src.slots[r];
  }
  if (!src.find(tile, row0, nrows, first, pos0)) return;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int w = wave % W, ks = wave / W;
  const int qi = lane & 31, hi = lane >> 5;
  const int n_q = n_kv * group;
  const int head = kvh * group + i % (group / W) * W + w;
  const int qpos = pos0 + min(qi, nrows - 1), qpos_last = pos0 + nrows - 1;
  const int len = pos0 + nrows;              // keys that the last row sees
  const int steps = (len + KS * KT - 1) / (KS * KT);
  const int n_parts = parts_of(steps, splits);
  if (part >= n_parts) return;
  const int begin = steps * part / n_parts * (KS * KT);
  const int end = min(len, steps * (part + 1) / n_parts * (KS * KT));
  // tiles of keys between the kept ones and the first row's window are
  // passed over
  int window = 0, keep = 0, win0 = 0;
  if constexpr (Src::kWindow) {
    window = src.window;
    keep = min(src.keep, len);
    win0 = max(0, pos0 - window + 1) / KT * KT;
  }
  auto after = [&](int kv0) {
    const int n = kv0 + KS * KT;
    return Src::kWindow && n >= keep && n < win0 ? win0 : n;
  };

  // queries; a negative scale goes into their signs
  s16x8 qf[DC];
  {
    const uint16_t* q = src.qkv + int64_t(row0 + min(qi, nrows - 1)) * stride +
                        head * D + hi * 8;
    const uint32_t flip = scale < 0.f ? 0x80008000u : 0u;
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      uint4 raw = *reinterpret_cast<const uint4*>(q + c * 16);
      if constexpr (!kRope) {
        raw.x ^= flip; raw.y ^= flip; raw.z ^= flip; raw.w ^= flip;
      }
      qf[c] = __builtin_bit_cast(s16x8, raw);
    }
    if constexpr (kRope) {
      const int at = __shfl(place, row0 + min(qi, nrows - 1), kWave);
      const float* cs = src.cos_sin + int64_t(at) * D;
#pragma unroll
      for (int c = 0; c < DC / 2; ++c) {
        const uint4 a = __builtin_bit_cast(uint4, qf[c]);
        const uint4 b = __builtin_bit_cast(uint4, qf[c + DC / 2]);
        float x[8], y[8];
        rotate8(true, a, b, cs + c * 16 + hi * 8, D / 2, x);
        rotate8(false, b, a, cs + c * 16 + hi * 8, D / 2, y);
        const uint4 f{flip, flip, flip, flip};
        qf[c] = __builtin_bit_cast(s16x8, flipped(CacheBF16::from_f32(x), f));
        qf[c + DC / 2] =
            __builtin_bit_cast(s16x8, flipped(CacheBF16::from_f32(y), f));
      }
    }
  }
  const float c2 = fmaxf(fabsf(scale), 1e-30f) * 1.4426950408889634f;

  // ---- staging.  Piece n of this thread goes to 16-byte slot n NT + tid
  // of the tile; within a row the slots of keys are swizzled by the row so
  // that sixteen rows' pieces of one column are in sixteen banks of 16
  // bytes, those of values by 64 bytes so that four rows' 64-byte columns
  // are in four.
  auto row_of = [&](int n) { return (n * NT + tid) / CH; };
  auto slot_of = [&](int s) {                // slot of KS tiles -> elements
    return (KS == 1 ? s : s / (KT * CH) * 2 * KT * CH + s % (KT * CH)) * 8;
  };
  auto k_piece = [&](int n) {
    const int r = row_of(n);
    return (tid % CH) ^ (D == 128 ? r & 15 : (r >> 1) & 7);
  };
  auto v_piece = [&](int n) {
    const int r = row_of(n);
    return (tid % CH) ^ (D == 128 ? (r & 3) << 2 : ((r >> 1) & 1) << 2);
  };
  int page[NP];                              // of the tile to come
  auto look_up = [&](int kv0) {
    if constexpr (Src::kPaged) {
#pragma unroll
      for (int n = 0; n < NP; ++n) {
        const int p = min(kv0 + row_of(n), len - 1);
        const int bs = BS ? BS : src.block_size;
        page[n] = src.tables[int64_t(first) * src.max_blocks + p / bs];
      }
    }
  };
  // rows past the last key repeat it: they are hidden, but have to be finite
  auto k_at = [&](int n, int kv0) {
    const int p = min(kv0 + row_of(n), len - 1);
    if constexpr (Src::kPaged) {
      const int bs = BS ? BS : src.block_size;
      return src.k + ((int64_t(page[n]) * n_kv + kvh) * bs + p % bs) * D +
             k_piece(n) * 8;
    } else {
      return src.qkv + int64_t(first + p) * stride + (n_q + kvh) * D +
             k_piece(n) * 8;
    }
  };
  auto v_at = [&](int n, int kv0) {
    const int p = min(kv0 + row_of(n), len - 1);
    if constexpr (Src::kPaged) {
      const int bs = BS ? BS : src.block_size;
      return src.v + ((int64_t(page[n]) * n_kv + kvh) * bs + p % bs) * D +
             v_piece(n) * 8;
    } else {
      return src.qkv + int64_t(first + p) * stride + (n_q + n_kv + kvh) * D +
             v_piece(n) * 8;
    }
  };
  typename KC::vec8 kr[kDirect ? 1 : NP], vr[kDirect ? 1 : NP];
  typename KC::vec8 kr2[kRope ? NP : 1];     // the other halves' channels
  auto fetch = [&](uint16_t* buf, int kv0) {
#pragma unroll
    for (int n = 0; n < NP; ++n) {
      if constexpr (kRope) {
        const int other = ((k_piece(n) ^ (CH / 2)) - k_piece(n)) * 8;
        kr[n] = *reinterpret_cast<const uint4*>(k_at(n, kv0));
        kr2[n] = *reinterpret_cast<const uint4*>(k_at(n, kv0) + other);
        vr[n] = *reinterpret_cast<const uint4*>(v_at(n, kv0));
      } else if constexpr (kDirect) {
        // wave-uniform LDS base; lane l lands at base + 16 l
        uint16_t* l = buf + slot_of(n * NT + wave * 64);
        lds_load16(k_at(n, kv0), l);
        lds_load16(v_at(n, kv0), l + HALF);
      } else {
        kr[n] = *reinterpret_cast<const typename KC::vec8*>(k_at(n, kv0));
        vr[n] = *reinterpret_cast<const typename KC::vec8*>(v_at(n, kv0));
      }
    }
  };
  auto land = [&](uint16_t* buf) {           // 8-bit rows, widened
    if constexpr (kRope) {
#pragma unroll
      for (int n = 0; n < NP; ++n) {
        const int p = row_of(n), row = first + min(p, len - 1);
        const float* cs = src.cos_sin + int64_t(__shfl(place, row, kWave)) * D +
                          k_piece(n) % (CH / 2) * 8;
        float f[8], g[8];
        rotate8(k_piece(n) < CH / 2, kr[n], kr2[n], cs, D / 2, f);
        *reinterpret_cast<uint4*>(buf + slot_of(n * NT + tid)) =
            CacheBF16::from_f32(f);
        *reinterpret_cast<uint4*>(buf + HALF + slot_of(n * NT + tid)) = vr[n];
        // a row's key and value by the tile and head that have it
        const int to = __shfl(slot, row, kWave);
        if (p < pos0 || p >= len || i % (group / W) != 0) continue;
        CacheBF16::to_f32(vr[n], g);
        src.keep(to, kvh, n_kv, D, k_piece(n) * 8, f, v_piece(n) * 8, g);
      }
    } else if constexpr (!kDirect) {
#pragma unroll
      for (int n = 0; n < NP; ++n) {
        float f[8];
        uint4 o;
        KC::to_f32(kr[n], f);
        o = {pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]),
             pack2(f[6], f[7])};
        *reinterpret_cast<uint4*>(buf + slot_of(n * NT + tid)) = o;
        KC::to_f32(vr[n], f);
        o = {pack2(f[0], f[1]), pack2(f[2], f[3]), pack2(f[4], f[5]),
             pack2(f[6], f[7])};
        *reinterpret_cast<uint4*>(buf + HALF + slot_of(n * NT + tid)) = o;
      }
    }
  };

  f32x16 o[VT];
#pragma unroll
  for (int v = 0; v < VT; ++v)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[v][r] = 0.f;
  float m = kHidden, l = 0.f;                // maximum in unscaled units

  // A transposing read gives lane i of sixteen column i of a tile of four
  // rows by sixteen; lane i names row i / 4, columns 4 (i % 4) ..
  const int tr = (lane & 15) >> 2;
  const int v_row = (tr + hi * 4) * D + ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
  const int v_sw = D == 128 ? tr : tr >> 1;
  const int k_sw = D == 128 ? qi & 15 : (qi >> 1) & 7;

  auto products = [&](const uint16_t* ks, int kv0) {
    const uint16_t* vs = ks + HALF;
    f32x16 s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
      for (int r = 0; r < 16; ++r) s[kt][r] = 0.f;
#pragma unroll
      for (int c = 0; c < DC; ++c) {
        const s16x8 kf = *reinterpret_cast<const s16x8*>(
            ks + (kt * 32 + qi) * D + (((c * 2 + hi) ^ k_sw) * 8));
        s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[c], s[kt], 0,
                                                        0, 0);
      }
    }
    if (kv0 + KT - 1 > pos0) {               // some row does not see all
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kv0 + kt * 32 + (r >> 2) * 8 + hi * 4 + (r & 3);
          if (key > qpos) s[kt][r] = kHidden;
        }
    }
    if constexpr (Src::kWindow) {
      // some row's window begins behind some key of the tile
      if (qpos_last - kv0 >= window)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = kv0 + kt * 32 + (r >> 2) * 8 + hi * 4 + (r & 3);
            if (qpos - key >= window && key >= keep) s[kt][r] = kHidden;
          }
    }
    float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(fmaxf(mx, s[0][r]), s[1][r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, kWave));
    // each query by itself, so that a row's result does not depend on the
    // rows it shares a tile with (only on the waves per head, see by_group)
    const bool grown = mx > m;
    if (__any(grown)) {
      const float mn = grown ? mx : m;
      const float corr = __builtin_amdgcn_exp2f((m - mn) * c2);
      l *= corr;
#pragma unroll
      for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[v][r] *= corr;
      m = mn;
    }
    // a row that has seen nothing yet: weights of what is hidden are nothing
    const float mc =
        (Src::kWindow || KS > 1) && m == kHidden ? 0.f : m * c2;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        s[kt][r] = __builtin_amdgcn_exp2f(fmaf(s[kt][r], c2, -mc));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const f32x16& p = s[t >> 1];
      const int r = (t & 1) * 8;
      const uint4 raw = {pack2(p[r], p[r + 1]), pack2(p[r + 2], p[r + 3]),
                         pack2(p[r + 4], p[r + 5]), pack2(p[r + 6], p[r + 7])};
      const s16x8 pf = __builtin_bit_cast(s16x8, raw);
      // this half's keys; of the weights as the product takes them
      l = add2(raw.x, l);
      l = add2(raw.y, l);
      l = add2(raw.z, l);
      l = add2(raw.w, l);
#pragma unroll
      for (int v = 0; v < VT; ++v) {
        const uint16_t* at = vs + v_row + t * 16 * D + (v ^ v_sw) * 32;
        const s16x4 a = read_tr(at), b = read_tr(at + 8 * D);
        const s16x8 vf = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
        o[v] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf, o[v], 0, 0, 0);
      }
    }
  };

  int kv0 = Src::kWindow ? (keep > 0 ? 0 : win0) : begin, ahead = after(kv0);
  look_up(kv0);
  fetch(lds, kv0);
  land(lds);
  look_up(ahead);
  int cur = 0;
  while (kv0 < end) {
    // this wave's part of the tile has landed, then everybody's; and nobody
    // reads the tile before any more
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint16_t* next = lds + (cur ^ 1) * STAGE;
    const bool more = !kRope && ahead < end;
    if (more) {
      fetch(next, ahead);
      look_up(after(ahead));
    }
    if (KS == 1 || kv0 + ks * KT < len)
      products(lds + cur * STAGE + ks * 2 * HALF, kv0 + ks * KT);
    if (more) land(next);
    cur ^= 1;
    kv0 = ahead;
    ahead = after(kv0);
  }

  if constexpr (KS > 1) {
    static_assert(KS == 2, "two waves of a head meet");
    constexpr int ROW = VT * 16 + 2;
    float* side = reinterpret_cast<float*>(lds) + w * ROW * 64 + lane;
    __syncthreads();
    if (ks == 1) {
#pragma unroll
      for (int v = 0; v < VT; ++v)
#pragma unroll
        for (int r = 0; r < 16; ++r) side[(v * 16 + r) * 64] = o[v][r];
      side[VT * 16 * 64] = m;
      side[(VT * 16 + 1) * 64] = l;
    }
    __syncthreads();
    if (ks == 1) return;
    // (of a later part, either wave's tiles may be hidden from a row)
    const float m1 = side[VT * 16 * 64], top = fmaxf(m, m1);
    const float c0 = __builtin_amdgcn_exp2f((m - top) * c2);
    const float c1 = __builtin_amdgcn_exp2f((m1 - top) * c2);
    l = l * c0 + side[(VT * 16 + 1) * 64] * c1;
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        o[v][r] = o[v][r] * c0 + side[(v * 16 + r) * 64] * c1;
    m = top;
  }
  if (qi >= nrows) return;
  l += __shfl_xor(l, 32, kWave);
  if (KS > 1 && n_parts > 1) {
    const int64_t at = (int64_t(part) * parts.rows + row0 + qi) * n_q + head;
    if (hi == 0) {
      parts.ml[at * 2] = m;
      parts.ml[at * 2 + 1] = l;
    }
#pragma unroll
    for (int v = 0; v < VT; ++v)
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<float4*>(parts.o + at * D + v * 32 + (r >> 2) * 8 +
                                   hi * 4) =
            float4{o[v][r], o[v][r + 1], o[v][r + 2], o[v][r + 3]};
    return;
  }
  float inv = 1.f / l;
  if constexpr (Src::kWindow) {
    if (src.sink) {                          // it takes its share, no value
      const float snk = src.sink[head] * 1.4426950408889634f;
      const float top = fmaxf(m * c2, snk);
      const float corr = __builtin_amdgcn_exp2f(m * c2 - top);
      inv = corr / (l * corr + __builtin_amdgcn_exp2f(snk - top));
    }
  }
  uint16_t* to = out + int64_t(row0 + qi) * n_q * D + head * D;
#pragma unroll
  for (int v = 0; v < VT; ++v)
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<uint2*>(to + v * 32 + (r >> 2) * 8 + hi * 4) =
          uint2{pack2(o[v][r] * inv, o[v][r + 1] * inv),
                pack2(o[v][r + 2] * inv, o[v][r + 3] * inv)};
}

template <int D, int W, int BS, int KS, typename Src>
__global__ __launch_bounds__(64 * W * KS, W == 4 ? 2 : 1)
void prefill_flash_kernel(Src src, uint16_t* __restrict__ out, int n_tiles,
                          int n_kv, int group, int stride, float scale,
                          PrefillParts parts) {
  __shared__ __attribute__((aligned(16))) uint16_t
      lds_static[KS == 1 ? FLASH_LDS<D, KS> / 2 : 8];
  extern __shared__ __attribute__((aligned(16))) uint16_t lds_dynamic[];
  flash_tile<D, W, BS, KS>(src, out, blockIdx.x, n_tiles, n_kv, group, stride,
                           scale, parts, KS == 1 ? lds_static : lds_dynamic);
}

// The parts of a tile's rows together: a workgroup of 256 threads per (tile,
// query head).
template <int D, typename Src>
DEV_INLINE void flash_combine(const Src& src, uint16_t* out, unsigned block,
                              int n_q, float scale, PrefillParts parts) {
  const int tile = block / n_q, head = block % n_q;
  int row0, nrows, first, pos0;
  if (!src.find(tile, row0, nrows, first, pos0)) return;
  const int n =
      parts_of((pos0 + nrows + 2 * KT - 1) / (2 * KT), parts.splits);
  if (n == 1) return;
  const float c2 = fmaxf(fabsf(scale), 1e-30f) * 1.4426950408889634f;
  for (int e = threadIdx.x; e < nrows * (D / 4); e += 256) {
    const int64_t row = int64_t(row0 + e / (D / 4)) * n_q + head;
    const int d = e % (D / 4) * 4;
    const int64_t step = int64_t(parts.rows) * n_q;
    float top = kHidden;
    for (int p = 0; p < n; ++p)
      top = fmaxf(top, parts.ml[(p * step + row) * 2]);
    float4 num = {0.f, 0.f, 0.f, 0.f};
    float den = 0.f;
#pragma unroll 4
    for (int p = 0; p < n; ++p) {
      const float2 ml = *reinterpret_cast<const float2*>(
          parts.ml + (p * step + row) * 2);
      const float4 o = *reinterpret_cast<const float4*>(
          parts.o + (p * step + row) * D + d);
      const float c = __builtin_amdgcn_exp2f((ml.x - top) * c2);
      num.x += c * o.x;
      num.y += c * o.y;
      num.z += c * o.z;
      num.w += c * o.w;
      den += c * ml.y;
    }
    const float inv = 1.f / den;
    *reinterpret_cast<uint2*>(out + row * D + d) =
        uint2{pack2(num.x * inv, num.y * inv), pack2(num.z * inv, num.w * inv)};
  }
}

template <int D, typename Src>
__global__ __launch_bounds__(256)
void prefill_combine_kernel(Src src, uint16_t* __restrict__ out, int n_q,
                            float scale, PrefillParts parts) {
  flash_combine<D>(src, out, blockIdx.x, n_q, scale, parts);
}

// ``keys``: about how many a sequence has, as far as the host knows without
// waiting for the device: the mean of a batch of prompts, the width of the
// block table for pages.
template <int D, int BS, typename Src>
void by_group(const Src& src, uint16_t* out, int n_tiles, int n_kv, int group,
              int stride, float scale, int keys, hipStream_t st,
              const PrefillParts& parts = {nullptr, nullptr, 1, 0}) {
  auto go = [&](auto tag, auto waves) {
    constexpr int W = decltype(tag)::value, KS = decltype(waves)::value;
    constexpr size_t smem = KS == 1 ? 0 : FLASH_LDS<D, KS>;
    auto* k = prefill_flash_kernel<D, W, BS, KS, Src>;
    if (smem > 65536)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(smem));
    const int splits = KS > 1 ? parts.splits : 1;
    hipLaunchKernelGGL(k, dim3(n_tiles * n_kv * (group / W) * splits),
                       dim3(64 * W * KS), smem, st, src, out, n_tiles, n_kv,
                       group, stride, scale, parts);
    if constexpr (KS > 1)
      if (splits > 1)
        hipLaunchKernelGGL((prefill_combine_kernel<D, Src>),
                           dim3(n_tiles * n_kv * group), dim3(256), 0, st, src,
                           out, n_kv * group, scale, parts);
  };
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I4 = std::integral_constant<int, 4>;
  if (n_tiles == 0) return;
  if (group == 1) go(I1{}, I1{});
  else if (group == 2) go(I2{}, I1{});
  else if constexpr (Src::kWindow || Src::kRope) go(I4{}, I1{});
  // up to a workgroup and a half per CU, and more than a few tiles of keys (us
  // with one wave per head and with two, 32/8 heads of 128: 512 rows behind
  // 1500 tokens 56.5 and 45.0, 1536 behind 1500 93 and 88; a prompt of 1000
  // 31.0 and 27.6, 1536 44.7 and 36.7, 384 15.4 and 15.0, 128 9.7 and 10.7;
  // 4 of 512 28.0 and 31.1).  Neither count is that of a ragged batch's longest
  // sequence: 1000 rows and 4 of 100, mean 280, take one wave, 28.1, and would
  // 24.2 with two, but 4000 rows and 20 of 30, mean 219, 160 and 174; 128 rows
  // of pages in a table for 8192 take two, 9.1, and would 8.3 with one.  The
  // two forms sum keys in different order, so that the last bits of a row's
  // result depend on the batch.
  else if (two_waves(n_tiles, n_kv, group, keys))
    go(I4{}, I2{});
  else go(I4{}, I1{});
}

}  // namespace

}  // namespace rlli
