// Launches of decode attention by itself; the kernel is in decode_attn.h.

#include "decode_attn.h"
#include "kernels.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace rlli {

namespace {

using namespace decode;

// A workgroup per row of a mixed step: the row's table and length, from the
// decoding sequences or from the tile of prompt rows that has it.  Rows of no
// tile see nothing.  (One launch instead of the ten or so that tensor ops
// take, which small models' steps, waiting for the host, would feel.)
__global__ __launch_bounds__(256)
void row_tables_kernel(RowTables a, int32_t* __restrict__ tables,
                       int32_t* __restrict__ lens, int wide) {
  __shared__ int tile;
  const int row = blockIdx.x;
  const bool decoding = row < a.n_decode;
  if (threadIdx.x == 0) tile = -1;
  __syncthreads();
  if (!decoding)
    for (int t = threadIdx.x; t < a.n_tiles; t += 256) {
      const int at = row - a.row0[t];
      if (at >= 0 && at < min(a.nrows[t], 32)) atomicMax(&tile, t);
    }
  __syncthreads();
  const int t = tile;
  const int32_t* src = nullptr;
  int width = 0, len = 0;
  if (decoding) {
    src = a.tables_dec + int64_t(row) * a.dec_width;
    width = a.dec_width;
    len = a.lens_dec[row];
  } else if (t >= 0) {
    src = a.tables_pre + int64_t(a.btrow[t]) * a.pre_width;
    width = a.pre_width;
    len = a.pos0[t] + row - a.row0[t] + 1;
  }
  for (int c = threadIdx.x; c < wide; c += 256)
    tables[int64_t(row) * wide + c] = c < width ? src[c] : 0;
  if (threadIdx.x == 0) lens[row] = len;
}

template <int D, int GROUP, typename KC, int BS, bool FUSED, Cut CUT>
__global__ __launch_bounds__(256, 3)
void decode_attn_kernel(DecodeArgs a) {
  __shared__ Lds<D, GROUP, KC, 4> lds;
  attend<D, GROUP, KC, BS, FUSED, CUT>(a, blockIdx.x, lds);
}

template <int D, int GROUP>
__global__ __launch_bounds__(256)
void decode_combine_kernel(DecodeArgs a) {
  combine<D, GROUP>(a, blockIdx.x);
}

template <int D, int GROUP, typename KC, bool FUSED>
void run(const DecodeArgs& a, hipStream_t st) {
  auto go = [&](auto bs) {
    constexpr int BS = decltype(bs)::value;
    if (a.shares > 0) {
      hipLaunchKernelGGL((decode_attn_kernel<D, GROUP, KC, BS, FUSED, SHARES>),
                         dim3((a.shares + a.batch) * a.n_kv), dim3(256), 0, st,
                         a);
      if (a.apart) return;
      hipLaunchKernelGGL((decode_combine_kernel<D, GROUP>),
                         dim3(a.batch * a.n_kv * GROUP), dim3(256), 0, st, a);
    } else {
      hipLaunchKernelGGL((decode_attn_kernel<D, GROUP, KC, BS, FUSED, WHOLE>),
                         dim3(a.batch * a.n_kv), dim3(256), 0, st, a);
    }
  };
  if (a.block_size == 16) go(std::integral_constant<int, 16>{});
  else go(std::integral_constant<int, 0>{});
}

template <bool FUSED>
void dispatch(const DecodeArgs& a, int group, int head_dim, bool fp8,
              hipStream_t st) {
  if (a.batch == 0) return;
  auto by_cache = [&](auto d, auto g) {
    constexpr int D = decltype(d)::value, G = decltype(g)::value;
    if (fp8) run<D, G, CacheFP8, FUSED>(a, st);
    else run<D, G, CacheBF16, FUSED>(a, st);
  };
  auto by_group = [&](auto d) {
    if (group == 1) by_cache(d, std::integral_constant<int, 1>{});
    else if (group == 2) by_cache(d, std::integral_constant<int, 2>{});
    else if (group == 4) by_cache(d, std::integral_constant<int, 4>{});
    else if (group == 8) by_cache(d, std::integral_constant<int, 8>{});
  };
  if (head_dim == 128) by_group(std::integral_constant<int, 128>{});
  else if (head_dim == 64) by_group(std::integral_constant<int, 64>{});
}

}  // namespace

int decode_attn_shares(int batch, int n_kv_heads, int max_tokens) {
  static const bool off = std::getenv("RLLI_NO_SPLITK") != nullptr;
  if (off) return 0;
  if (batch * n_kv_heads >= 384 && max_tokens <= 1024) return 0;
  // never cut (whether the table is wider or not, so that one sequence's sums
  // are the same in a step of its own and in a captured one)
  if (max_tokens <= least_units(batch, 1) * UNIT) return 0;
  return std::max(1, 512 / n_kv_heads);
}

void launch_row_tables(const RowTables& a, int32_t* tables, int32_t* lens,
                       int rows, int wide, hipStream_t stream) {
  if (rows == 0) return;
  hipLaunchKernelGGL(row_tables_kernel, dim3(rows), dim3(256), 0, stream, a,
                     tables, lens, wide);
}

void launch_decode_attn(
    const uint16_t* q, const float* parts, int n_parts, void* k_cache,
    void* v_cache, const int32_t* block_table, const int32_t* seq_lens,
    const int32_t* positions, const float* cos_sin,
    const int32_t* slot_mapping, uint16_t* out, int batch, int n_q_heads,
    int n_kv_heads, int head_dim, int block_size, int max_blocks, float scale,
    int q_stride, int shares, float* part_out, float* part_ml, bool cache_fp8,
    bool apart, hipStream_t stream) {
  const DecodeArgs a{q, parts, k_cache, v_cache, k_cache, v_cache,
                     block_table, seq_lens, positions, cos_sin, slot_mapping,
                     out, part_out, part_ml, batch, n_kv_heads, block_size,
                     max_blocks, q_stride, n_parts, shares, scale, apart};
  const int group = n_q_heads / n_kv_heads;
  if (positions) dispatch<true>(a, group, head_dim, cache_fp8, stream);
  else dispatch<false>(a, group, head_dim, cache_fp8, stream);
}

}  // namespace rlli
