// Windowed decode attention on the matrix cores: keys and values as wide as each
// other, four query heads of a key/value head, no distance bias.
//
// The work of a wave is decode_attn.h's: units of 32 tokens whose keys and
// values are all asked for at once, 24 bits of every weight.  Units are those of
// the kept tokens and then the window's, whose number is bounded, so that a workgroup
// of twelve waves has all of a sequence's units or as many parts of them as make a
// round each, where that leaves CUs idle.  What bounds it is latency: from the
// launch to positions, pages and keys 3 us, 3.5 us a round.  us, in lane groups of
// 16-token steps and as here, 16/4 heads of 128, window 1024: 1 sequence 15.0 and
// 11.6, 16 21.8 and 14.7, 64 39.6 and 28.7 (4.7 TB/s); 16 of 100 tokens 9.0 and
// 6.2; 64 with an 8-bit cache 35.6 and 17.8; window 4096, 16 38.7 and 27.8.
#include "attn.h"
#include "decode_attn.h"

#include <algorithm>
#include <type_traits>

namespace rlli {

namespace {

using decode::f32x4;
using decode::s16x8;

constexpr float kLog2e = 1.4426950408889634f;
constexpr int NW = 12;            // waves of a workgroup
constexpr int UNIT = decode::UNIT, GROUP = 4;

template <int D, typename KC>
__global__ __launch_bounds__(NW * 64, NW / 4)
void window_units_kernel(WindowAttnArgs a) {
  using namespace decode;
  using elem = typename KC::elem;
  using vec8 = typename KC::vec8;
  constexpr int KSTEPS = D / 32, VT = D / 16, HS = 4, NT = NW * 64;
  constexpr int KPL = 2 / sizeof(elem), KLOADS = KSTEPS / KPL;
  using kraw = typename Words<16>::type;
  using vraw = typename Words<sizeof(elem) * VT>::type;
  constexpr int QROW = Lds<D, GROUP, KC, NW>::QROW;
  __shared__ Lds<D, GROUP, KC, NW> lds;
  float* raw = lds.raw;
  uint16_t* qs = lds.qs;
  elem* self = lds.self;

  const int split = blockIdx.x, kvh = blockIdx.y, seq = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, oct = lane >> 4;
  const int cpart = col / HS;
  const uint32_t mask1 = cpart > 0 ? kUpper : 0, mask2 = cpart > 1 ? kUpper : 0;
  const int last = a.positions[seq], bs = a.block_size;
  const elem* kc = static_cast<const elem*>(a.k_cache);
  const elem* vc = static_cast<const elem*>(a.v_cache);
  const float c2 =
      a.scale * query_temp(last, a.temp_coef, a.temp_every) * kLog2e;
  auto k_chan = [&](int k) {
    return k / KPL * 32 * KPL + (oct * KPL + k % KPL) * 8;
  };

  // units: of the kept tokens, then from the window's first on
  const int lo = max(0, last - a.window + 1);
  const int n_all = last / UNIT + 1;
  int w0 = lo / UNIT, kept = min((a.keep_first + UNIT - 1) / UNIT, n_all);
  if (kept >= w0) {
    kept = 0;
    if (a.keep_first > 0) w0 = 0;
  }
  const int n_units = kept + n_all - w0;
  const int first = split * NW + wave, stride = NW * a.n_split;
  auto unit_at = [&](int i) { return i < kept ? i : w0 + i - kept; };
  // whether this workgroup has the new token and appends it
  const bool newest =
      a.has_kv && (n_units - 1) / NW % a.n_split == split;

  const int32_t* table = a.block_tables + int64_t(seq) * a.max_blocks;
  int page[2];
  auto half_tok = [&](int u, int t) { return min(u * 2 + t, last / 16) * 16; };
  auto key_tok = [&](int u, int t) {     // tokens past the last repeat it
    return min(u * UNIT + t * 16 + col, last);
  };
  auto value_tok = [&](int u, int t, int i) {
    return min(u * UNIT + t * 16 + oct * 4 + i, last);
  };
  auto look_up = [&](int i) {
    if (i >= n_units) return;
#pragma unroll
    for (int t = 0; t < 2; ++t) page[t] = table[half_tok(unit_at(i), t) / bs];
  };
  auto row_of = [&](int u, int t, int tok) -> int64_t {
    const int half = half_tok(u, t);
    return (int64_t(page[t]) * a.n_kv + kvh) * bs + half % bs + tok - half;
  };
  kraw kr[2][KLOADS];
  vraw vr[2][4];
  auto load_keys = [&](int i) {
    if (i >= n_units) return;
    const int u = unit_at(i);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const elem* p = kc + row_of(u, t, key_tok(u, t)) * D + k_chan(0);
#pragma unroll
      for (int k = 0; k < KLOADS; ++k)
        kr[t][k] = *reinterpret_cast<const kraw*>(p + k * 32 * KPL);
    }
  };
  auto load_values = [&](int i) {
    if (i >= n_units) return;
    const int u = unit_at(i);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        vr[t][j] = __builtin_nontemporal_load(reinterpret_cast<const vraw*>(
            vc + row_of(u, t, value_tok(u, t, j)) * D + col * VT));
  };
  look_up(first);
  load_keys(first);
  load_values(first);
  look_up(first + stride);

  // ---- the heads' queries, the new key and value: rotated in pairs --------
  const uint16_t* row =
      static_cast<const uint16_t*>(a.qkv) + int64_t(seq) * a.stride;
  const int half = a.rot / 2;
  const float* cs = a.cos_sin + int64_t(last) * a.rot;
  const int n_in = (GROUP + (newest ? 2 : 0)) * (D / 2);
  for (int e = tid; e < n_in; e += NT) {
    const int h = e / (D / 2), p = e % (D / 2);
    const int head = h < GROUP ? kvh * GROUP + h
                     : a.n_q + (h > GROUP ? a.n_kv : 0) + kvh;
    const uint32_t w =
        *reinterpret_cast<const uint32_t*>(row + head * D + 2 * p);
    float u = __builtin_bit_cast(float, w << 16);
    float v = __builtin_bit_cast(float, w & 0xffff0000u);
    if (p < half && h <= GROUP) {
      const float c = cs[p], s = cs[half + p], x = u;
      u = x * c - v * s;
      v = v * c + x * s;
    }
    if (h < GROUP) {
      // Prompts round rotated queries to 16 bits for the matrix cores; so here.
      // The other parts' least numbers: see decode_attn.h.
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint16_t q = f32_to_bf16(i ? v : u);
        const uint16_t least =
            upper_half(copysignf(kLeast, bf16_to_f32(q)));
        const int d = 2 * p + i;
        qs[h * QROW + d] = q;
        qs[(HS + h) * QROW + d] = least;
        qs[(2 * HS + h) * QROW + d] = least;
        qs[(3 * HS + h) * QROW + d] = least;
      }
    } else {
      raw[h * D + 2 * p] = u;
      raw[h * D + 2 * p + 1] = v;
    }
  }
  lds_barrier();
  if (newest) {
    // append at cache precision; this step sees what later ones will
    if (tid < 2 * D / 8) {
      const int e = tid * 8;
      const vec8 w = KC::from_f32(raw + GROUP * D + e);
      const int slot = a.slots[seq];
      elem* to = static_cast<elem*>(e < D ? a.k_cache : a.v_cache);
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
    const uint4 w =
        *reinterpret_cast<const uint4*>(qs + col * QROW + k_chan(k));
    qf[k] = __builtin_bit_cast(s16x8, w);
  }

  f32x4 o[VT];
#pragma unroll
  for (int t = 0; t < VT; ++t) o[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = kNegInf, l = 0.f;
  for (int i = first; i < n_units; i += stride) {
    const int u = unit_at(i), tok0 = u * UNIT;
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
        for (int j = 0; j < 4; ++j)
          vr[t][j] = value_tok(u, t, j) == last ? w : vr[t][j];
    }
    f32x4 s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < KLOADS; ++k) {
        uint32_t w[4 * KPL];
        widen<KC>(kr[t][k], w);
#pragma unroll
        for (int j = 0; j < KPL; ++j)
          s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(s16x8, (uint4{w[j * 4], w[j * 4 + 1],
                                               w[j * 4 + 2], w[j * 4 + 3]})),
              qf[k * KPL + j], s[t], 0, 0, 0);
      }
    }
    load_keys(i + stride);
    auto seen = [&](int tok) {
      return tok <= last && (last - tok < a.window || tok < a.keep_first);
    };
    float mx = kNegInf;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float v = sum_parts<HS>(s[t][r]) * c2;
        s[t][r] = seen(tok0 + t * 16 + oct * 4 + r) ? v : kNegInf;
        mx = fmaxf(mx, s[t][r]);
      }
    // what is hidden may be anything, and what repeats the last value infinite,
    // of which no weight makes zero
    if (last - tok0 >= a.window || tok0 + UNIT - 1 > last)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (!seen(tok0 + t * 16 + oct * 4 + r)) vr[t][r] = vraw{};
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
    uint32_t pw[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float y[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const float p = __builtin_amdgcn_exp2f(s[j / 2][j % 2 * 2 + r] - m);
        l += p;
        const float x = p - masked(p, mask1);
        y[r] = x - masked(x, mask2);
      }
      pw[j] = upper_halves(y[0], y[1]);
    }
    const s16x8 pf =
        __builtin_bit_cast(s16x8, (uint4{pw[0], pw[1], pw[2], pw[3]}));
    uint32_t vw[2][4][VT / 2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) widen<KC>(vr[t][j], vw[t][j]);
#pragma unroll
    for (int t = 0; t < VT; ++t) {
      const uint32_t sel = t & 1 ? 0x07060302u : 0x05040100u;
      const int d = t / 2;
      const uint4 w = {
          __builtin_amdgcn_perm(vw[0][1][d], vw[0][0][d], sel),
          __builtin_amdgcn_perm(vw[0][3][d], vw[0][2][d], sel),
          __builtin_amdgcn_perm(vw[1][1][d], vw[1][0][d], sel),
          __builtin_amdgcn_perm(vw[1][3][d], vw[1][2][d], sel)};
      o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(s16x8, w), pf, o[t], 0, 0, 0);
    }
    load_values(i + stride);
    look_up(i + 2 * stride);
  }

  // ---- the waves' results, through LDS --------------------------------
  l += __shfl_xor(l, 16, kWave);
  l += __shfl_xor(l, 32, kWave);
#pragma unroll
  for (int t = 0; t < VT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float v = o[t][r];
      const float sum = v + (dpp_mov_f32<0x12c>(v) + dpp_mov_f32<0x124>(v));
      o[t][r] = __builtin_isinf(v) ? v : sum;    // of infinite values
    }
  if (col < GROUP) {
    float* to = lds.accs + (wave * GROUP + col) * D + oct * 4 * VT;
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < VT; t += 4)
        *reinterpret_cast<f32x4*>(to + r * VT + t) =
            f32x4{o[t][r], o[t + 1][r], o[t + 2][r], o[t + 3][r]};
    if (oct == 0) {
      lds.ml[(wave * GROUP + col) * 2] = m;
      lds.ml[(wave * GROUP + col) * 2 + 1] = l;
    }
  }
  lds_barrier();
  for (int e = tid; e < GROUP * D; e += NT) {
    const int h = e / D, d = e % D, head = kvh * GROUP + h;
    float M = kNegInf, num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, lds.ml[(w * GROUP + h) * 2]);
    const bool whole = a.n_split == 1;
    if (whole && a.sink) {
      const float snk = a.sink[head] * kLog2e;
      M = fmaxf(M, snk);
      den = __builtin_amdgcn_exp2f(snk - M);
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float c =
          __builtin_amdgcn_exp2f(lds.ml[(w * GROUP + h) * 2] - M);
      num += c * lds.accs[(w * GROUP + h) * D + d];
      den += c * lds.ml[(w * GROUP + h) * 2 + 1];
    }
    const int64_t at = int64_t(seq) * a.n_q + head;
    if (whole) {
      static_cast<uint16_t*>(a.out)[at * D + d] = f32_to_bf16(num / den);
    } else {
      a.part_acc[(at * a.n_split + split) * D + d] = num;
      if (d == 0) {
        a.part_ml[(at * a.n_split + split) * 2] = M / kLog2e;
        a.part_ml[(at * a.n_split + split) * 2 + 1] = den;
      }
    }
  }
}

}  // namespace

bool window_units_ok(const WindowAttnArgs& a) {
  return !a.f32 && a.dim == a.vdim && (a.dim == 64 || a.dim == 128) &&
         a.n_q == GROUP * a.n_kv && !a.r1 && !a.v_norm && a.rot % 2 == 0 &&
         a.block_size % 16 == 0 && a.stride % 8 == 0;
}

// Where it is the faster one whatever the sequences' lengths are, of which the host
// knows the tables' room and the window (``reach``): no more pairs of a sequence and
// a key/value head than CUs, or than those for which lane groups would go in parts as
// well.  A workgroup is large; where more of them than that have short sequences in
// wide tables, waves without work cost more than the others gain, and where one or
// two heads share a read, far more.  (us, lane groups and so, tables of 4096 tokens,
// window 1024: 16/4 heads of 128, 64 sequences of 20 tokens 13.7 and 7.0, 100 20.9 and
// 11.7, 256 19.2 and 21.6; 16/8 heads, 64 of 20 7.9 and 11.5, of 300 19.0 and 22.4, of
// 1000 51 and 45; 8/8 heads, 64 of 20 6.9 and 11.4, 8 of 300 11.9 and 13.5.)  512
// pairs that may see much go so too, for what they gain on long sequences: 32/8 heads
// of 128, 64 of 1000 60 and 46, of 20 10.7 and 11.5.
bool window_units_faster(const WindowAttnArgs& a, int64_t reach) {
  const int64_t pairs = int64_t(a.rows) * a.n_kv;
  return pairs <= 256 || (pairs < 512 && reach >= 128) ||
         (pairs == 512 && reach >= 512 && a.dim == 128);
}

// Parts of a sequence's ``units`` (as many as its window can have): rounds of
// units take 3.5 us each, a launch that puts parts together 4; no more parts than
// fill the chip.
int window_units_splits(const WindowAttnArgs& a, int units) {
  const int pairs = std::max(1, a.rows * a.n_kv);
  int best = 1;
  float least = 0.f;
  for (int n = 1; n <= std::max(1, std::min(16, 256 / pairs)); ++n) {
    const float us = (units + NW * n - 1) / (NW * n) * 3.5f + (n > 1 ? 4.f : 0.f);
    if (n == 1 || us < least) {
      best = n;
      least = us;
    }
  }
  return best;
}

void launch_window_units(const WindowAttnArgs& a, hipStream_t st) {
  if (a.rows == 0) return;
  auto go = [&](auto d, auto kc) {
    hipLaunchKernelGGL((window_units_kernel<decltype(d)::value, decltype(kc)>),
                       dim3(a.n_split, a.n_kv, a.rows), dim3(NW * 64), 0, st,
                       a);
  };
  auto by_cache = [&](auto d) {
    if (a.cache == kCacheFP8) go(d, CacheFP8{});
    else go(d, CacheBF16{});
  };
  if (a.dim == 128) by_cache(std::integral_constant<int, 128>{});
  else by_cache(std::integral_constant<int, 64>{});
  if (a.n_split > 1) launch_window_combine(a, st);
}

}  // namespace rlli
