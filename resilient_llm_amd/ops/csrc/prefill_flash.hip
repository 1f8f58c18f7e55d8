// Launches of prompt attention over batch rows and over pages; the kernel is
// in prefill_flash.h.

#include "kernels.h"
#include "prefill_flash.h"

namespace rlli {

namespace {

struct BatchRows {                // k and v are columns of the batch's rows
  static constexpr bool kPaged = false, kWindow = false, kRope = false;
  using KC = CacheBF16;
  const uint16_t* qkv;
  const int32_t* cu;              // [n_seqs + 1]
  int n_seqs;

  DEV_INLINE bool find(int tile, int& row0, int& nrows, int& first,
                       int& pos0) const {
    // tiles of the sequences before, 64 sequences at a time
    const int lane = threadIdx.x & 63;
    int before = 0;
    for (int s0 = 0; s0 < n_seqs; s0 += 64) {
      const int s = s0 + lane;
      const int beg = s < n_seqs ? cu[s] : 0;
      const int len = s < n_seqs ? cu[s + 1] - beg : 0;
      const int mine = (len + QR - 1) / QR;
      int upto = mine;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int t = __shfl_up(upto, d, kWave);
        if (lane >= d) upto += t;
      }
      const int rel = tile - before;
      const uint64_t hit =
          __ballot(rel < upto && rel >= upto - mine && mine > 0);
      if (hit) {
        const int src = __ffsll(static_cast<unsigned long long>(hit)) - 1;
        const int off = (rel - __shfl(upto - mine, src, kWave)) * QR;
        first = __shfl(beg, src, kWave);
        pos0 = off;
        row0 = first + off;
        nrows = min(QR, __shfl(len, src, kWave) - off);
        return true;
      }
      before += __shfl(upto, 63, kWave);
    }
    return false;
  }
};

// Up to 64 rows, whose queries and keys are not rotated yet, and the cache for
// what comes of them.
template <typename C>
struct RopedRows : BatchRows {
  static constexpr bool kRope = true;
  const int32_t* positions;
  const float* cos_sin;
  const int32_t* slots;
  typename C::elem *k, *v;        // [blocks, n_kv, block, D]
  int block_size, rows;

  // eight channels of a row's key, from ``kd`` on, and of its value
  DEV_INLINE void keep(int slot, int kvh, int n_kv, int D, int kd,
                       const float* k8, int vd, const float* v8) const {
    if (slot < 0) return;
    const int64_t at = ((int64_t(slot / block_size) * n_kv + kvh) * block_size +
                        slot % block_size) * D;
    *reinterpret_cast<typename C::vec8*>(k + at + kd) = C::from_f32(k8);
    *reinterpret_cast<typename C::vec8*>(v + at + vd) = C::from_f32(v8);
  }
};

}  // namespace

// Rotation and append inside, us in a layer of 45 rows, 32/8 heads of 64: launches
// of their own 3.1 and 5.7 and a gap, in one 7.5; a prompt of the 1B model 899 and
// 885.  What bounds it is latency: two rounds of loads, sixteen workgroups.
void launch_prompt_rows_attn(const uint16_t* qkv, const int32_t* cu_seqlens,
                             const int32_t* positions, const float* cos_sin,
                             void* k_cache, void* v_cache,
                             const int32_t* slot_mapping, uint16_t* out,
                             int n_seqs, int rows, int n_kv_heads, int group,
                             int head_dim, int block_size, int qkv_stride,
                             float scale, bool cache_fp8, hipStream_t st) {
  if (rows == 0) return;
  auto go = [&](auto kc, auto d) {
    using C = decltype(kc);
    const RopedRows<C> src{{qkv, cu_seqlens, n_seqs}, positions, cos_sin,
                           slot_mapping,
                           static_cast<typename C::elem*>(k_cache),
                           static_cast<typename C::elem*>(v_cache),
                           block_size, rows};
    // (of so few keys always by one wave a head)
    by_group<decltype(d)::value, 0>(src, out, rows / QR + n_seqs, n_kv_heads,
                                    group, qkv_stride, scale, rows / n_seqs,
                                    st);
  };
  using D128 = std::integral_constant<int, 128>;
  using D64 = std::integral_constant<int, 64>;
  if (cache_fp8) {
    if (head_dim == 128) go(CacheFP8{}, D128{}); else go(CacheFP8{}, D64{});
  } else {
    if (head_dim == 128) go(CacheBF16{}, D128{}); else go(CacheBF16{}, D64{});
  }
}

void launch_prefill_rows(const uint16_t* qkv, const int32_t* cu_seqlens,
                         uint16_t* out, int n_seqs, int rows, int n_kv_heads,
                         int group, int head_dim, int qkv_stride, float scale,
                         hipStream_t st) {
  const BatchRows src{qkv, cu_seqlens, n_seqs};
  // every sequence ends in at most one tile that is not full
  const int n_tiles = rows / QR + n_seqs;
  if (rows == 0) return;
  if (head_dim == 128)
    by_group<128, 0>(src, out, n_tiles, n_kv_heads, group, qkv_stride, scale,
                     rows / n_seqs, st);
  else
    by_group<64, 0>(src, out, n_tiles, n_kv_heads, group, qkv_stride, scale,
                    rows / n_seqs, st);
}

void launch_prefill_paged(const uint16_t* qkv, const void* k_cache,
                          const void* v_cache, const int32_t* chunk_row0,
                          const int32_t* chunk_pos0,
                          const int32_t* chunk_nrows,
                          const int32_t* chunk_btrow,
                          const int32_t* block_tables, uint16_t* out,
                          int n_chunks, int n_kv_heads, int group,
                          int head_dim, int qkv_stride, int max_blocks,
                          int block_size, float scale, bool cache_fp8,
                          const PrefillParts& parts, hipStream_t st) {
  auto go = [&](auto kc, auto d, auto bs) {
    using KC = decltype(kc);
    const Pages<KC> src{qkv,
                        static_cast<const typename KC::elem*>(k_cache),
                        static_cast<const typename KC::elem*>(v_cache),
                        chunk_row0, chunk_pos0, chunk_nrows, chunk_btrow,
                        block_tables, max_blocks, block_size};
    by_group<decltype(d)::value, decltype(bs)::value>(
        src, out, n_chunks, n_kv_heads, group, qkv_stride, scale,
        max_blocks * block_size, st, parts);
  };
  auto by_dim = [&](auto kc) {
    using I16 = std::integral_constant<int, 16>;
    using I0 = std::integral_constant<int, 0>;
    using D128 = std::integral_constant<int, 128>;
    using D64 = std::integral_constant<int, 64>;
    if (head_dim == 128) {
      if (block_size == 16) go(kc, D128{}, I16{}); else go(kc, D128{}, I0{});
    } else {
      if (block_size == 16) go(kc, D64{}, I16{}); else go(kc, D64{}, I0{});
    }
  };
  if (cache_fp8) by_dim(CacheFP8{}); else by_dim(CacheBF16{});
}

}  // namespace rlli
