// The sequential half of the recurrences' prompt kernels: chunk after chunk
// of a sequence with the state in MFMA accumulators, and the norm and gate
// that follow.
//
// A workgroup owns one (sequence, head, slice of value columns); a wave the
// 16 output rows of a sub-chunk and every fourth key tile of the state.
// Products are f32 MFMA (but see rec_scan_parts_kernel).  A chunk's operands
// travel in registers, loaded while the chunk before it computes.  A
// sequence's chunks follow one another and only the last is short, so no table
// is on the path of a load.
// Loads and stores are unconditional where sizes allow (what has no place
// goes to spare rows), since a branch around one makes later waits drain
// everything in flight.
//
// kScanPlain's operands come in the order in which lanes take them, 1 KB a load:
// read as rows are, neighbouring lanes have rows of their own, and the cache
// looks up each lane's 16 bytes by themselves, which was what bounded it (4
// sequences of 1.9k, 8 heads of 128 x 256: 179 us, of which 145 such lookups,
// and 133 so).
//
// kScanMax: with F the chunk's running log-decay, a = i - F and the maximum
// M_t = max(m, max_{s <= t} a_s), m what the chunk started with,
//     m_t = F_t + M_t,   O_t = e^{m - M_t} q_t S + sum_s q_t k_s e^{a_s - M_t} v_s
//     S   = e^{m - M_C} S + sum_s k_s e^{a_s - M_C} v_s^T
// A holds e^{a_s - max_{r <= t} a_r}; the rest of the exponent is a row
// factor <= 1.
// kScanDelta: U = Ub - W S takes the place of the values, two waves of
// barriers per chunk.

#include "rec_math.h"

#include <algorithm>
#include <type_traits>

namespace rlli {
namespace {

constexpr int C = kRecChunk;

// VT value tiles of 16 columns per workgroup, MD key tiles per wave.  FULL:
// dim is 64 MD, values come in whole slices and rows are aligned, so that no
// load is conditional (a branch around a load ends in a wait for it): rows
// behind the last one are loaded from the last one instead.
template <typename T, int MODE, int VT, int MD, bool FULL>
__global__ __launch_bounds__(256, FULL && VT == 1 && MD <= 2 ? 2 : 1)
void rec_scan_kernel(ScanArgs a, bool vec_q, bool vec_v) {
  constexpr bool MAX = MODE == kScanMax, DELTA = MODE == kScanDelta;
  constexpr bool RAW = MODE != kScanPlain;      // operands as they are
  using KE = std::conditional_t<RAW, T, float>;
  using QE = KE;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  constexpr int VS = VT * 16, SR = VS + 4;
  const int DP = FULL ? 64 * MD : a.dpad, ndt = DP / 16;
  float* Sl = sm;                         // [DP][SR]
  float* Vl = Sl + DP * SR;               // [64][SR]
  float* Vk = RAW ? Vl + C * SR : Vl;     // [64][SR] with the key factors
  const int seq = blockIdx.x / a.heads, h = blockIdx.x % a.heads;
  const int v0 = blockIdx.y * VS;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, g = lane >> 4;
  const int first = a.seqs[seq], count = a.seqs[a.n_seqs + seq];
  if (count <= 0) return;
  const bool fresh = a.seqs[2 * a.n_seqs + seq] == 0;
  const int64_t slot_h =
      int64_t(a.seqs[3 * a.n_seqs + seq]) * a.heads + h;
  float* state = a.state + slot_h * a.dim * a.vpad;
  float m = 0.f;
  if constexpr (MAX) m = fresh ? 0.f : a.m[slot_h];

  f32x4_t S[MD][VT];
#pragma unroll
  for (int i = 0; i < MD; ++i)
#pragma unroll
    for (int nt = 0; nt < VT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = (i * 4 + w) * 16 + g * 4 + r;
        const int c = v0 + nt * 16 + lr;
        S[i][nt][r] = (!fresh && d < a.dim && c < a.cols)
                          ? state[int64_t(d) * a.vpad + c] : 0.f;
      }

  // A chunk's operands are loaded into registers as soon as those of the
  // chunk before it are used up, and not touched before they are needed.
  constexpr int NQ = 4 * MD, NV = VT, VQ = VS / 4;
  const int trow = w * 16 + lr;
  const int last = first + count - 1;
  const int row_first = a.tiles[first];
  const int n_last = a.tiles[2 * a.n_tiles + last];
  Raw4<QE> qr[NQ];
  Raw4<KE> kr[MD][4];
  f32x4_t ar[4], wr[DELTA ? NQ : 1], ur[DELTA ? VT : 1];
  Raw4<T> vr[DELTA ? 1 : NV];             // four columns of a row
  // row factors: of four output rows, of this lane's operand row, of the
  // staged value rows, of the chunk
  f32x4_t f_row, f_key;
  float f_lane = 0.f, av[MAX ? NV : 1], F_row = 0.f, F_end = 0.f, end = 0.f;
  const T* vb = reinterpret_cast<const T*>(a.v) + h * a.vdim;
  const int hk = h / a.group, kv_heads = a.heads / a.group;
  auto row_of = [&](int t) { return row_first + (t - first) * C; };
  auto rows_of = [&](int t) { return t == last ? n_last : C; };
  auto chunk = [&](int t) { return int64_t(t) * a.heads + h; };
  auto load_q = [&](int t) {
    if constexpr (RAW) {
      const T* q = reinterpret_cast<const T*>(a.q) +
                   int64_t(row_of(t) + trow) * a.q_stride + hk * a.dim;
      const bool ok = trow < rows_of(t);
      if constexpr (FULL) q -= int64_t(ok ? 0 : trow - n_last + 1) * a.q_stride;
#pragma unroll
      for (int i = 0; i < NQ; ++i) {
        if constexpr (FULL) qr[i].load(q + i * 16 + g * 4);
        else if (i < ndt)
          qr[i] = raw_guard(q, i * 16 + g * 4, a.dim, ok, vec_q);
      }
    } else {
      const float* qd = static_cast<const float*>(a.qd) + chunk(t) * C * DP +
                        (w * 64 + lane) * 4;
#pragma unroll
      for (int i = 0; i < NQ; ++i)
        if (i < ndt) qr[i].load(qd + i * 1024);
    }
    if constexpr (DELTA) {
      const float* wp = a.w + chunk(t) * C * DP + trow * DP + g * 4;
#pragma unroll
      for (int i = 0; i < NQ; ++i)
        if (i < ndt) wr[i] = *reinterpret_cast<const f32x4_t*>(wp + i * 16);
    }
  };
  auto load_a = [&](int t) {
    const float* sc = static_cast<const float*>(a.sc) + chunk(t) * C * C +
                      (RAW ? trow * C + g * 4 : (w * 256 + lane) * 4);
#pragma unroll
    for (int J = 0; J < 4; ++J)            // (blocks behind w: not used)
      ar[J] = *reinterpret_cast<const f32x4_t*>(sc + min(J, w) *
                                                         (RAW ? 16 : 256));
  };
  auto load_v = [&](int t) {
    const float* rf = a.rows + chunk(t) * 3 * C;
    if constexpr (DELTA) {
      const float* ub =
          a.ub + (chunk(t) * C + w * 16 + g * 4) * a.ubp + v0 + lr;
#pragma unroll
      for (int nt = 0; nt < VT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          ur[nt][r] = v0 + nt * 16 < a.ubp ? ub[r * a.ubp + nt * 16] : 0.f;
    } else {
      const int row0 = row_of(t), n = rows_of(t);
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = i * 256 + threadIdx.x;
        const int r = e / VQ, c = v0 + e % VQ * 4;
        if constexpr (FULL)
          vr[i].load(vb + int64_t(row0 + min(r, n - 1)) * a.v_stride +
                     (c < a.vdim ? c : 0));
        else
          vr[i] = raw_guard(vb + int64_t(row0 + r) * a.v_stride, c, a.vdim,
                            r < n, vec_v);
        if constexpr (MAX) av[i] = rf[C + r];
      }
    }
  };
  auto load_rows = [&](int t) {
    const float* rf = a.rows + chunk(t) * 3 * C;
    if constexpr (DELTA) {
      f_row = *reinterpret_cast<const f32x4_t*>(rf + w * 16 + g * 4);
      f_key = *reinterpret_cast<const f32x4_t*>(rf + C + w * 16 + g * 4);
      end = a.dec[chunk(t)];
    }
    if constexpr (MAX) {
      f_row = *reinterpret_cast<const f32x4_t*>(rf + 2 * C + w * 16 + g * 4);
      f_lane = rf[2 * C + trow];
      F_row = rf[trow];
      F_end = rf[C - 1];
      end = rf[3 * C - 1];
    }
  };
  auto load_k = [&](int t) {
    const KE* kt = reinterpret_cast<const KE*>(a.kt) +
                   (int64_t(t) * kv_heads + hk) * DP * C;
#pragma unroll
    for (int i = 0; i < MD; ++i)
      if (FULL || i * 4 + w < ndt)
#pragma unroll
        for (int s = 0; s < 4; ++s)
          kr[i][s].load(
              kt + (RAW ? ((i * 4 + w) * 16 + lr) * C + s * 16 + g * 4
                        : (((i * 4 + w) * 4 + s) * 64 + lane) * 4));
  };
  load_v(first);
  load_rows(first);
  load_q(first);
  load_a(first);
  load_k(first);
  for (int t = first; t <= last; ++t) {
    const int next = min(t + 1, last);     // (no load is conditional)
    const int row0 = row_of(t), n = rows_of(t);
    f32x4_t dv[RAW ? 1 : MD];
    float keep = 1.f;
    if constexpr (!RAW) {
      const float* dec = a.dec + chunk(t) * DP;
#pragma unroll
      for (int i = 0; i < MD; ++i)
        if (FULL || i * 4 + w < ndt)
          dv[i] = *reinterpret_cast<const f32x4_t*>(
              dec + (i * 4 + w) * 16 + g * 4);
    }
    f32x4_t f_out = f_row, f_k = f_key;
    float f_a = 1.f, M_end = 0.f;
    if constexpr (DELTA) keep = end;
    if constexpr (MAX) {
      M_end = fmaxf(m, end);
      keep = gexp<T>(m - M_end);
      a.mrow[int64_t(trow < n ? row0 + trow : a.n_rows + trow) * a.heads + h] =
          F_row + fmaxf(m, f_lane);       // (every slice, the same value)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        f_out[r] = a.qscale * gexp<T>(m - fmaxf(m, f_row[r]));
      f_a = gexp<T>(f_lane - fmaxf(m, f_lane));
      m = F_end + M_end;
    }
#pragma unroll
    for (int i = 0; i < MD; ++i)
      if (FULL || i * 4 + w < ndt)
#pragma unroll
        for (int nt = 0; nt < VT; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            Sl[((i * 4 + w) * 16 + g * 4 + r) * SR + nt * 16 + lr] =
                S[i][nt][r];
    if constexpr (!DELTA) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const int e = i * 256 + threadIdx.x;
        const int r = e / VQ, c = e % VQ * 4;
        f32x4_t v;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          v[k] = vr[i].get(k);
          if constexpr (MAX)              // the normalizer's column of ones
            if (v0 + c + k >= a.vdim) v[k] = v0 + c + k == a.vdim ? 1.f : 0.f;
          if (r >= n) v[k] = 0.f;
        }
        *reinterpret_cast<f32x4_t*>(Vl + r * SR + c) = v;
        if constexpr (MAX)
          *reinterpret_cast<f32x4_t*>(Vk + r * SR + c) =
              v * gexp<T>(av[i] - M_end);
      }
      load_v(next);
    }
    load_rows(next);
    __syncthreads();
    f32x4_t o[VT], x[DELTA ? VT : 1];
#pragma unroll
    for (int nt = 0; nt < VT; ++nt) {
      o[nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if constexpr (DELTA) x[nt] = o[nt];
    }
    // LDS operands are asked for in batches ahead of the products
    constexpr int GI = NQ < 8 / VT ? NQ : 8 / VT;
#pragma unroll
    for (int i0 = 0; i0 < NQ; i0 += GI) {
      float s[GI][4][VT];
#pragma unroll
      for (int i = 0; i < GI; ++i)
        if (FULL || i0 + i < ndt)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int nt = 0; nt < VT; ++nt)
              s[i][j][nt] =
                  Sl[((i0 + i) * 16 + g * 4 + j) * SR + nt * 16 + lr];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < GI; ++i)
        if (FULL || i0 + i < ndt)
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int nt = 0; nt < VT; ++nt) {
              o[nt] = mma4(qr[i0 + i].get(j), s[i][j][nt], o[nt]);
              if constexpr (DELTA)
                x[nt] = mma4(wr[i0 + i][j], s[i][j][nt], x[nt]);
            }
    }
    load_q(next);
    if constexpr (RAW)
#pragma unroll
      for (int nt = 0; nt < VT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[nt][r] *= f_out[r];
    if constexpr (DELTA) {
#pragma unroll
      for (int nt = 0; nt < VT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int at = (w * 16 + g * 4 + r) * SR + nt * 16 + lr;
          const float u = ur[nt][r] - x[nt][r];
          Vl[at] = u;
          Vk[at] = u * f_k[r];
        }
      load_v(next);
      __syncthreads();
    }
    float vv[16][VT];
    auto values = [&](const float* from) {
#pragma unroll
      for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int nt = 0; nt < VT; ++nt)
          vv[k][nt] =
              from[(k / 4 * 16 + g * 4 + k % 4) * SR + nt * 16 + lr];
      __builtin_amdgcn_sched_barrier(0);
    };
    values(Vl);
#pragma unroll
    for (int k = 0; k < 16; ++k) {         // (the last wave needs all four)
      const float e = ar[k / 4][k % 4];
      const float p = k / 4 > w ? 0.f : MAX ? e * f_a : e;
#pragma unroll
      for (int nt = 0; nt < VT; ++nt) o[nt] = mma4(p, vv[k][nt], o[nt]);
    }
    load_a(next);
    if constexpr (RAW) values(Vk);
#pragma unroll
    for (int nt = 0; nt < VT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tr = w * 16 + g * 4 + r, c = v0 + nt * 16 + lr;
        const bool ok = tr < n && (!(MAX || !FULL) || c < a.cols);
        a.o[(int64_t(ok ? row0 + tr : a.n_rows + tr) * a.heads + h) * a.opad +
            (ok ? c : 0)] = o[nt][r];
      }
#pragma unroll
    for (int i = 0; i < MD; ++i) {
      if (!FULL && i * 4 + w >= ndt) continue;
#pragma unroll
      for (int nt = 0; nt < VT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[i][nt][r] *= RAW ? keep : dv[RAW ? 0 : i][r];
#pragma unroll
      for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int nt = 0; nt < VT; ++nt)
          S[i][nt] = mma4(kr[i][k / 4].get(k % 4), vv[k][nt], S[i][nt]);
    }
    load_k(next);
    // (delta: the next chunk's first barrier comes before its first write
    // to the value tiles, and Sl was last read before the second)
    if constexpr (!DELTA) __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < MD; ++i)
#pragma unroll
    for (int nt = 0; nt < VT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int d = (i * 4 + w) * 16 + g * 4 + r;
        const int c = v0 + nt * 16 + lr;
        if (d < a.dim && c < a.cols) state[int64_t(d) * a.vpad + c] = S[i][nt][r];
      }
  // other slices of this head may yet read the old maximum: it returns to
  // its slot in the launch that follows
  if constexpr (MAX)
    if (blockIdx.y == 0 && threadIdx.x == 0)
      a.m_new[int64_t(seq) * a.heads + h] = m;
}

// kScanPlain in parts, of 16-bit activations.  The values are 16-bit numbers;
// queries, keys, A and the state are 32-bit ones, each of three 16-bit parts that
// add up to it, so that products run on the 16-bit matrix cores: three for each of
// the values', six for queries and state.  The three that are left out are up to
// 2^-21 of a product, 2^-24 in the mean, always towards zero.  Four waves carry the
// state from chunk to chunk (w MD of its key tiles), four others have the
// outputs (w the rows of a sub-chunk) of the chunk that the state is carried over,
// from its parts in LDS.  LDS has two copies of parts and values, written by turns,
// so that a chunk takes one barrier.  What bounds it is that each workgroup loads
// 120 KB a chunk, which takes as long as its products and LDS: a fragment's next
// load comes right behind its last product, so that loads go out between products
// and not all at once with all waves waiting to issue them, and loads ahead of the
// loop come in the loop's order, as the waits in it are for both.  Operands that no
// cache holds any more come slower; TOUCH: each of the slices that read them asks
// for 256 of their 576 or 960 lines a chunk ahead, so that three or four ask for
// all.  (In a step's call, 8 heads of 128 x
// 256, us, loads together behind the products and now: 1 sequence of 2600 70 and
// 57, 3 of 2000 105 and 73, 4 of 2000 111 and 80, 8 of 900 77 and 63, 16 of 500 92
// and 83; asked for two chunks ahead 62, 76, 84, 64 and 93.)  4 sequences of 1.9k
// with f32 products 133 us, of which these 67; the kernel that makes the operands 49
// and 50 (with infinite numbers' parts NaN, 3 us less each).  Against 64 bits, 2048
// tokens, the state is off by 4.3e-7 and 2.6e-7, as it is rounded less often; 6e-4
// and 4e-4 of the outputs are not the nearest 16-bit number.
template <int VT, int MD, bool FULL, bool TOUCH>
__global__ __launch_bounds__(512, 2)
void rec_scan_parts_kernel(ScanArgs a, bool vec_v) {
  using T = uint16_t;
  constexpr int VS = VT * 16, NKS = 2 * MD;
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];
  const int DP = FULL ? 64 * MD : a.dpad, ndt = DP / 16;
  const int nks = FULL ? NKS : (ndt + 1) / 2;
  // a copy: [nks][3][VT][64][8] state, [2][VT][64][8] values
  const int copy = (nks * 3 + 2) * VT * 512;
  const int seq = blockIdx.x / a.heads, h = blockIdx.x % a.heads;
  const int v0 = blockIdx.y * VS;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6 & 3);
  const int lr = lane & 15, g = lane >> 4;
  const int first = a.seqs[seq], count = a.seqs[a.n_seqs + seq];
  if (count <= 0) return;
  const int last = first + count - 1;
  auto chunk = [&](int t) { return int64_t(t) * a.heads + h; };
  auto frag = [&](const uint16_t* p) {
    return *reinterpret_cast<const s16x8_t*>(p);
  };
  auto mma = [](const s16x8_t& x, const s16x8_t& y, const f32x4_t& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
  };
  auto values = [&](int t, s16x8_t (&v)[2][VT]) {
    const uint16_t* from =
        lds + (t & 1) * copy + nks * 3 * VT * 512 + lane * 8;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int nt = 0; nt < VT; ++nt)
        v[ks][nt] = frag(from + (ks * VT + nt) * 512);
  };

  if (threadIdx.x < 256) {
    const bool fresh = a.seqs[2 * a.n_seqs + seq] == 0;
    float* state = a.state + (int64_t(a.seqs[3 * a.n_seqs + seq]) * a.heads +
                              h) * a.dim * a.vpad;
    f32x4_t S[MD][VT], dv[MD];
    s16x8_t kr[MD][2][3];
#pragma unroll
    for (int i = 0; i < MD; ++i)
#pragma unroll
      for (int nt = 0; nt < VT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = (w * MD + i) * 16 + g * 4 + r;
          const int c = v0 + nt * 16 + lr;
          S[i][nt][r] = (!fresh && d < a.dim && c < a.cols)
                            ? state[int64_t(d) * a.vpad + c] : 0.f;
        }
    // (tiles behind the last one have its operands, and nobody reads them)
    auto tile_of = [&](int i) {
      return FULL ? w * MD + i : min(w * MD + i, ndt - 1);
    };
    auto load_part = [&](int t, int ks, int p) {
      const uint16_t* k = static_cast<const uint16_t*>(a.kt) +
                          chunk(t) * ndt * 3072 + lane * 8;
#pragma unroll
      for (int i = 0; i < MD; ++i)
        kr[i][ks][p] = frag(k + ((tile_of(i) * 2 + ks) * 3 + p) * 512);
    };
    auto load_dec = [&](int t) {
      const float* dec = a.dec + chunk(t) * DP;
#pragma unroll
      for (int i = 0; i < MD; ++i)
        dv[i] = *reinterpret_cast<const f32x4_t*>(dec + tile_of(i) * 16 +
                                                  g * 4);
    };
    // two tiles are a fragment's two halves, an odd last one's second half zero
    auto put = [&](int t) {
      uint16_t* to = lds + (t & 1) * copy + lane * 8;
#pragma unroll
      for (int i = 0; i < MD; i += 2) {
        const int tile = w * MD + i;
        if (!FULL && tile >= 2 * nks) break;
#pragma unroll
        for (int nt = 0; nt < VT; ++nt) {
          uint2 part[2][3];
          const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
          three_parts(FULL || tile < ndt ? S[i][nt] : zero, part[0]);
          if constexpr (MD > 1)
            three_parts(FULL || tile + 1 < ndt ? S[i + 1][nt] : zero, part[1]);
#pragma unroll
          for (int p = 0; p < 3; ++p) {
            uint16_t* at = to + ((tile / 2 * 3 + p) * VT + nt) * 512;
            if constexpr (MD > 1)
              *reinterpret_cast<uint4*>(at) =
                  uint4{part[0][p].x, part[0][p].y, part[1][p].x,
                        part[1][p].y};
            else
              *reinterpret_cast<uint2*>(at + tile % 2 * 4) = part[0][p];
          }
        }
      }
    };
    // (TOUCH) a line of each chunk's operands
    const char* line_at = nullptr;
    int64_t line_step = 0;
    uint32_t line = 0;
    if constexpr (TOUCH) {
      const int nk = ndt * 48, nq = nks * 96, all = nk + nq + 192;
      const int i = min(int(blockIdx.y + gridDim.y * threadIdx.x), all - 1);
      const void* p = i < nk ? a.kt : i < nk + nq ? a.qd : a.sc;
      const int in = i < nk ? nk : i < nk + nq ? nq : 192;
      const int at = i < nk ? i : i < nk + nq ? i - nk : i - nk - nq;
      line_at = static_cast<const char*>(p) + (int64_t(h) * in + at) * 128;
      line_step = int64_t(a.heads) * in * 128;
    }
    auto touch = [&](int t) {
      if constexpr (!TOUCH) return;
      asm volatile("" ::"v"(line));       // (it has landed)
      line = *reinterpret_cast<const uint32_t*>(line_at + t * line_step);
    };
    // (in the order that they come in in the loop, whose waits are for both)
    touch(min(first + 1, last));
    load_dec(first);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int p = 2; p >= 0; --p)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        load_part(first, ks, p);
        __builtin_amdgcn_sched_barrier(0);
      }
    for (int t = first; t <= last; ++t) {
      put(t);
      __syncthreads();
      s16x8_t v[2][VT];
      values(t, v);
      const int next = min(t + 1, last);  // (no load is conditional)
      touch(min(t + 2, last));
#pragma unroll
      for (int i = 0; i < MD; ++i)
#pragma unroll
        for (int nt = 0; nt < VT; ++nt) S[i][nt] *= dv[i];
      __builtin_amdgcn_sched_barrier(0);
      load_dec(next);
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
          for (int i = 0; i < MD; ++i)
#pragma unroll
            for (int nt = 0; nt < VT; ++nt)
              S[i][nt] = mma(kr[i][ks][p], v[ks][nt], S[i][nt]);
          __builtin_amdgcn_sched_barrier(0);
          load_part(next, ks, p);
        }
    }
#pragma unroll
    for (int i = 0; i < MD; ++i)
#pragma unroll
      for (int nt = 0; nt < VT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = (w * MD + i) * 16 + g * 4 + r;
          const int c = v0 + nt * 16 + lr;
          if (d < a.dim && c < a.cols)
            state[int64_t(d) * a.vpad + c] = S[i][nt][r];
        }
    return;
  }

  const int tid = threadIdx.x - 256;
  const int row_first = a.tiles[first];
  const int n_last = a.tiles[2 * a.n_tiles + last];
  s16x8_t qr[NKS][3], ar[2][3];
  // of the values, a lane stages four rows of VT columns
  using VRow = std::conditional_t<
      VT == 1, uint16_t, std::conditional_t<VT == 2, uint32_t, uint2>>;
  VRow vr[4];
  const int vrow = tid / 16 * 4, vcol = tid % 16 * VT;
  const T* vb = static_cast<const T*>(a.v) + h * a.vdim;
  auto row_of = [&](int t) { return row_first + (t - first) * C; };
  auto rows_of = [&](int t) { return t == last ? n_last : C; };
  auto load_q = [&](int t, int ks) {
    const uint16_t* q = static_cast<const uint16_t*>(a.qd) +
                        chunk(t) * nks * 6144 + (w * 192 + lane) * 8 +
                        (FULL ? ks : min(ks, nks - 1)) * 6144;
#pragma unroll
    for (int p = 0; p < 3; ++p) qr[ks][p] = frag(q + p * 512);
  };
  auto load_a = [&](int t, int ks) {
    const uint16_t* sc = static_cast<const uint16_t*>(a.sc) +
                         chunk(t) * 12288 + (w * 384 + lane) * 8;
#pragma unroll
    for (int p = 0; p < 3; ++p)            // (a pair behind w: not used)
      ar[ks][p] = frag(sc + (min(ks, w / 2) * 3 + p) * 512);
  };
  auto load_v = [&](int t) {
    const int row0 = row_of(t), n = rows_of(t), c = v0 + vcol;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = min(vrow + i, n - 1);
      const T* p = vb + int64_t(row0 + r) * a.v_stride + c;
      if (FULL || (vec_v && c < a.vdim)) {
        vr[i] = *reinterpret_cast<const VRow*>(p);
      } else {
        T v[VT];
#pragma unroll
        for (int k = 0; k < VT; ++k) v[k] = c + k < a.vdim ? p[k] : T(0);
        __builtin_memcpy(&vr[i], v, sizeof v);
      }
    }
  };
  load_v(first);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) {
    load_q(first, ks);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    load_a(first, ks);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int t = first; t <= last; ++t) {
    const int next = min(t + 1, last);     // (no load is conditional)
    const int row0 = row_of(t), n = rows_of(t);
    const uint16_t* Sl = lds + (t & 1) * copy + lane * 8;
    // (down a column, as the products take it)
    uint16_t* staged = lds + (t & 1) * copy + nks * 3 * VT * 512 +
                       (vrow / 32 * VT + vcol / 16) * 512 +
                       (vrow % 16 * 4 + vcol % 16) * 8 + vrow / 16 % 2 * 4;
    T v[4][VT];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const VRow row = vrow + i < n ? vr[i] : VRow{};
      __builtin_memcpy(v[i], &row, sizeof row);
    }
#pragma unroll
    for (int k = 0; k < VT; ++k)
      *reinterpret_cast<uint2*>(staged + k * 8) =
          uint2{uint32_t(v[0][k]) | uint32_t(v[1][k]) << 16,
                uint32_t(v[2][k]) | uint32_t(v[3][k]) << 16};
    load_v(next);
    __syncthreads();
    f32x4_t o[2][VT];
#pragma unroll
    for (int nt = 0; nt < VT; ++nt)
      o[0][nt] = o[1][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      if (FULL || ks < nks) {
        s16x8_t s[3][VT];
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int nt = 0; nt < VT; ++nt)
            s[p][nt] = frag(Sl + ((ks * 3 + p) * VT + nt) * 512);
        auto both = [&](int acc, int i, int j) {
#pragma unroll
          for (int nt = 0; nt < VT; ++nt)
            o[acc][nt] = mma(s[j][nt], qr[ks][i], o[acc][nt]);
        };
        both(0, 0, 2);
        both(1, 2, 0);
        both(0, 1, 1);
        both(1, 1, 0);
        both(0, 0, 0);
        both(1, 0, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      load_q(next, ks);
    }
    s16x8_t vs[2][VT];
    values(t, vs);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      if (ks <= w / 2)
#pragma unroll
        for (int p = 2; p >= 0; --p)
#pragma unroll
          for (int nt = 0; nt < VT; ++nt)
            o[p > 0][nt] = mma(vs[ks][nt], ar[ks][p], o[p > 0][nt]);
      __builtin_amdgcn_sched_barrier(0);
      load_a(next, ks);
    }
    // a lane has four columns of row lr of the sub-chunk
    const int tr = w * 16 + lr;
    auto out_row = [&](int row) {
      return a.o + (int64_t(row) * a.heads + h) * a.opad;
    };
    float* to = out_row(tr < n ? row0 + tr : a.n_rows + tr) + v0 + g * 4;
#pragma unroll
    for (int nt = 0; nt < VT; ++nt) {
      const f32x4_t v = o[0][nt] + o[1][nt];
      if constexpr (FULL)
        *reinterpret_cast<f32x4_t*>(to + nt * 16) = v;
      else
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = v0 + nt * 16 + g * 4 + r;
          *(c < a.cols ? to + nt * 16 + r : out_row(a.n_rows + tr)) = v[r];
        }
    }
  }
}

template <int VT>
void scan_parts(const ScanArgs& a, bool touch, hipStream_t st) {
  constexpr int VS = VT * 16;
  const int nks = (a.dpad / 16 + 1) / 2;
  const size_t smem = size_t(2) * (nks * 3 + 2) * VT * 1024;
  const bool vec_v = a.v_stride % 4 == 0 && a.vdim % 4 == 0 &&
                     reinterpret_cast<uintptr_t>(a.v) % 8 == 0;
  auto run = [&](auto* k) {
    if (smem > 65536)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(smem));
    hipLaunchKernelGGL(k, dim3(a.n_seqs * a.heads, (a.cols + VS - 1) / VS),
                       dim3(512), smem, st, a, vec_v);
  };
  const bool full = vec_v && a.vdim % VS == 0;
  auto go = [&](auto md) {
    constexpr int MD = decltype(md)::value;
    if (!full || a.dim != MD * 64)
      run(rec_scan_parts_kernel<VT, MD, false, false>);
    else if (touch)
      run(rec_scan_parts_kernel<VT, MD, true, true>);
    else
      run(rec_scan_parts_kernel<VT, MD, true, false>);
  };
  if (a.dpad <= 64) go(std::integral_constant<int, 1>{});
  else if (a.dpad <= 128) go(std::integral_constant<int, 2>{});
  else if constexpr (VT < 4) run(rec_scan_parts_kernel<VT, 4, false, false>);
}

template <typename T, int MODE, int VT>
void scan_md(const ScanArgs& a, hipStream_t st) {
  constexpr int VS = VT * 16;
  const size_t smem = size_t(a.dpad + (MODE == kScanPlain ? 1 : 2) * C) *
                      (VS + 4) * sizeof(float);
  auto aligned = [](const void* p, int64_t stride, int width) {
    return stride % 4 == 0 && width % 4 == 0 &&
           reinterpret_cast<uintptr_t>(p) % (4 * sizeof(T)) == 0;
  };
  const bool vec_q = aligned(a.q, a.q_stride, a.dim);
  const bool vec_v = aligned(a.v, a.v_stride, a.vdim);
  auto run = [&](auto* k) {
    if (smem > 65536)
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                int(smem));
    hipLaunchKernelGGL(k, dim3(a.n_seqs * a.heads, (a.cols + VS - 1) / VS),
                       dim3(256), smem, st, a, vec_q, vec_v);
  };
  const bool full = (a.dim == 64 || a.dim == 128) && a.vdim % VS == 0 &&
                    (MODE == kScanPlain || vec_q) &&
                    (MODE == kScanDelta || vec_v);
  if constexpr (sizeof(T) == 2) {
    if (full) {
      if (a.dim == 64) run(rec_scan_kernel<T, MODE, VT, 1, true>);
      else run(rec_scan_kernel<T, MODE, VT, 2, true>);
      return;
    }
  }
  if (a.dpad <= 64) run(rec_scan_kernel<T, MODE, VT, 1, false>);
  else if (a.dpad <= 128) run(rec_scan_kernel<T, MODE, VT, 2, false>);
  else run(rec_scan_kernel<T, MODE, VT, 4, false>);
}

template <typename T, int MODE>
void scan(const ScanArgs& a, hipStream_t st) {
  // a scan step is latency-bound: narrow value slices, several
  // workgroups per CU, until there are plenty anyway
  const int64_t sh = int64_t(a.n_seqs) * a.heads;
  if constexpr (MODE == kScanPlain && sizeof(T) == 2)
    if (a.parts) {
      const ScanSlices by = scan_slices(a);
      if (by.cols == 64) scan_parts<4>(a, by.touch, st);
      else if (by.cols == 32) scan_parts<2>(a, by.touch, st);
      else scan_parts<1>(a, by.touch, st);
      return;
    }
  if (a.vdim > 32 && sh * ((a.vdim + 63) / 64) >= 512)
    scan_md<T, MODE, 4>(a, st);
  else if (a.vdim > 16 && sh * ((a.vdim + 31) / 32) >= 1024)
    scan_md<T, MODE, 2>(a, st);
  else
    scan_md<T, MODE, 1>(a, st);
}

// GL lanes per (row, head); V4 float4 columns per lane when the width and
// its offsets allow vectors (V4 = 0: one column at a time)
template <typename T, int KIND, int V4, int GL>
__global__ __launch_bounds__(256)
void rec_gate_kernel(RecGateArgs a) {
  if (a.m_new) {                          // (a few values, any thread)
    const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i < int64_t(a.n_seqs) * a.heads)
      a.m[int64_t(a.seqs[3 * a.n_seqs + i / a.heads]) * a.heads +
          i % a.heads] = a.m_new[i];
  }
  const int lane = threadIdx.x % GL;
  const int64_t rh = int64_t(blockIdx.x) * (256 / GL) + threadIdx.x / GL;
  if (rh >= int64_t(a.rows) * a.heads) return;
  const int64_t row = rh / a.heads;
  const int h = int(rh % a.heads);
  const float* o = a.o + rh * a.opad;
  const T* gate = reinterpret_cast<const T*>(a.gate) + row * a.gate_stride +
                  h * a.vdim;
  const float* norm = a.norm + h * a.norm_stride;
  T* out = reinterpret_cast<T*>(a.out) + row * a.out_stride + h * a.vdim;
  float pre = 1.f;
  if (a.mrow)
    pre = 1.f / (fmaxf(fabsf(o[a.vdim]), gexp<T>(-a.mrow[rh])) + 1e-6f);
  auto gated = [](float r, float g) {
    return KIND == kGateSilu ? r * (g / (1.f + gexp<T>(-g)))
                             : r / (1.f + gexp<T>(-g));
  };
  float ss = 0.f;
  if constexpr (V4 > 0) {
    f32x4_t ov[V4], gv[V4];
#pragma unroll
    for (int i = 0; i < V4; ++i) {
      const int c = (i * GL + lane) * 4;
      ov[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (c < a.vdim) {
        ov[i] = *reinterpret_cast<const f32x4_t*>(o + c);
        if constexpr (KIND != kGateNone) gv[i] = act_load4(gate + c);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        ov[i][j] *= pre;
        ss += ov[i][j] * ov[i][j];
      }
    }
    const float inv = 1.f / sqrtf(group_sum<GL>(ss) / a.vdim + a.eps);
#pragma unroll
    for (int i = 0; i < V4; ++i) {
      const int c = (i * GL + lane) * 4;
      if (c >= a.vdim) break;
      const f32x4_t nv = *reinterpret_cast<const f32x4_t*>(norm + c);
      f32x4_t r;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        r[j] = ov[i][j] * inv * nv[j];
        if constexpr (KIND != kGateNone) r[j] = gated(r[j], gv[i][j]);
      }
      act_store4(out + c, r);
    }
  } else {
    for (int e = lane; e < a.vdim; e += GL) ss += o[e] * o[e] * pre * pre;
    const float inv = pre / sqrtf(group_sum<GL>(ss) / a.vdim + a.eps);
    for (int e = lane; e < a.vdim; e += GL) {
      float r = o[e] * inv * norm[e];
      if constexpr (KIND != kGateNone) r = gated(r, act_load(gate + e));
      act_store(out + e, r);
    }
  }
}

template <typename T, int KIND>
void gate(const RecGateArgs& a, hipStream_t st) {
  auto go = [&](auto* kg, int per_wg = 4) {
    const int64_t rh = int64_t(a.rows) * a.heads;
    hipLaunchKernelGGL(kg, dim3(uint32_t((rh + per_wg - 1) / per_wg)),
                       dim3(256), 0, st, a);
  };
  const bool vec_g =
      KIND == kGateNone ||
      (a.gate_stride % 4 == 0 &&
       reinterpret_cast<uintptr_t>(a.gate) % (4 * sizeof(T)) == 0);
  if (a.vdim % 4 || a.opad % 4 || !vec_g || a.out_stride % 4 ||
      reinterpret_cast<uintptr_t>(a.out) % 16)
    go(rec_gate_kernel<T, KIND, 0, 64>);
  else if (a.vdim <= 64)
    go(rec_gate_kernel<T, KIND, 1, 16>, 16);
  else if (a.vdim <= 128)
    go(rec_gate_kernel<T, KIND, 1, 32>, 8);
  else if (a.vdim <= 256)
    go(rec_gate_kernel<T, KIND, 1, 64>);
  else
    go(rec_gate_kernel<T, KIND, 4, 64>);
}

}  // namespace

// A CU has one workgroup, which takes the longer the wider its slice is.  (us,
// slices of 16, 32 and 64 columns: heads of 128 x 256, 1000 tokens, 16 of them 34 38
// 50, 24 60 42 55, 32 67 46 59, 40 98 82 62, 64 of 900 134 88 64; of 64 x 64, 64 of
// them 33 40 41, 80 61 43 44.  Two copies of 256 rows by 64 columns do not fit LDS.)
ScanSlices scan_slices(const ScanArgs& a) {
  const int64_t sh = int64_t(a.n_seqs) * a.heads;
  auto groups = [&](int cols) { return sh * ((a.vdim + cols - 1) / cols); };
  auto cost = [&](int cols, int each) {
    return (groups(cols) + 255) / 256 * each;
  };
  const int64_t one = cost(16, 6), two = cost(32, 7);
  const int cols = a.dpad <= 128 && cost(64, 9) < std::min(one, two) ? 64
                   : two < one                                       ? 32
                                                                     : 16;
  // From some 60 MB of operands on, if all workgroups run at once (in a step's call,
  // us without and with, heads of 128 x 256: 1 sequence of 2600 57 59, 2 of 2000 57
  // 57, 3 80 73, 4 102 80, 8 of 900 65 63; 16 of 500, which take turns, 83 93).
  return {cols, int64_t(a.n_tiles) * a.heads * a.dpad >= 65536 &&
                    groups(cols) <= 256 && (a.dim == 64 || a.dim == 128) &&
                    a.vdim % cols == 0};
}

void launch_rec_scan(const ScanArgs& a, hipStream_t st) {
  if (a.n_seqs == 0) return;
  auto go = [&](auto t) {
    using T = decltype(t);
    if (a.mode == kScanMax) scan<T, kScanMax>(a, st);
    else if (a.mode == kScanDelta) scan<T, kScanDelta>(a, st);
    else scan<T, kScanPlain>(a, st);
  };
  if (a.f32) go(float{});
  else go(uint16_t{});
}

void launch_rec_gate(const RecGateArgs& a, hipStream_t st) {
  if (a.rows == 0) return;
  auto go = [&](auto t) {
    using T = decltype(t);
    if (a.kind == kGateSilu) gate<T, kGateSilu>(a, st);
    else if (a.kind == kGateSigmoid) gate<T, kGateSigmoid>(a, st);
    else gate<T, kGateNone>(a, st);
  };
  if (a.f32) go(float{});
  else go(uint16_t{});
}

}  // namespace rlli
