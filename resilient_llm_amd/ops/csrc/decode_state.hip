// What a captured decode step does around the model: a new batch into the
// step's buffers, where each row's key and value go, the state one token on.
//
// All of it is some hundred bytes a row; what bounds it is launches, 2 to 4 us
// each with the gap behind it, so each of the three is one.  As tensor ops they
// are 5 to 12, 8 and 3: a step of one sequence, these and two more launches of
// the embedding apart, took 712 us and takes 685 through 16 layers of 2048, 2951
// and 2923 through 32 of 4096, of 16 sequences 704 and 689 through 12 mixed
// layers.  The table's row is by 256 threads, one load each.

#include "common.h"
#include "kernels.h"

namespace rlli {

namespace {

// A workgroup per row of the bucket; those behind the batch neither read nor
// write anything of a live sequence: they own the scratch block and slot.
__global__ __launch_bounds__(256)
void decode_load_kernel(DecodeState to, DecodeState from, int batch, int wide,
                        int scratch_block, int scratch_slot) {
  const int row = blockIdx.x;
  const bool live = row < batch;
  const int32_t* src = from.tables + int64_t(row) * wide;
  int32_t* dst = to.tables + int64_t(row) * to.width;
  const int n = live ? wide : 0;
  for (int i = threadIdx.x; i < to.width; i += 256)
    dst[i] = i < n ? src[i] : scratch_block;
  if (threadIdx.x) return;
  to.ids[row] = live ? from.ids[row] : 0;
  to.positions[row] = live ? from.positions[row] : 0;
  to.temps[row] = live ? from.temps[row] : 0.f;
  to.seeds[row] = live ? from.seeds[row] : 0;
  if (!live) to.slots[row] = scratch_slot;
  else if (from.slots) to.slots[row] = from.slots[row];
}

__global__ __launch_bounds__(64)
void decode_begin_kernel(const int32_t* __restrict__ positions,
                         const int32_t* __restrict__ tables,
                         int32_t* __restrict__ slots,
                         int32_t* __restrict__ lens, int batch, int width,
                         int block_size) {
  const int row = blockIdx.x * 64 + threadIdx.x;
  if (row >= batch) return;
  const int pos = positions[row];
  const int block = min(pos / block_size, width - 1);
  slots[row] =
      tables[int64_t(row) * width + block] * block_size + pos % block_size;
  lens[row] = pos + 1;
}

__global__ __launch_bounds__(64)
void decode_advance_kernel(int32_t* __restrict__ ids,
                           int32_t* __restrict__ positions,
                           uint64_t* __restrict__ seeds,
                           const int32_t* __restrict__ tokens, int batch,
                           uint64_t seed_step) {
  const int row = blockIdx.x * 64 + threadIdx.x;
  if (row >= batch) return;
  ids[row] = tokens[row];
  positions[row] += 1;
  seeds[row] += seed_step;
}

}  // namespace

void launch_decode_load(const DecodeState& to, const DecodeState& from,
                        int bucket, int batch, int wide, int scratch_block,
                        int scratch_slot, hipStream_t st) {
  hipLaunchKernelGGL(decode_load_kernel, dim3(bucket), dim3(256), 0, st, to,
                     from, batch, wide, scratch_block, scratch_slot);
}

void launch_decode_begin(const int32_t* positions, const int32_t* tables,
                         int32_t* slots, int32_t* lens, int batch, int width,
                         int block_size, hipStream_t st) {
  hipLaunchKernelGGL(decode_begin_kernel, dim3((batch + 63) / 64), dim3(64), 0,
                     st, positions, tables, slots, lens, batch, width,
                     block_size);
}

void launch_decode_advance(int32_t* ids, int32_t* positions, int64_t* seeds,
                           const int32_t* tokens, int batch, int64_t seed_step,
                           hipStream_t st) {
  hipLaunchKernelGGL(decode_advance_kernel, dim3((batch + 63) / 64), dim3(64),
                     0, st, ids, positions, reinterpret_cast<uint64_t*>(seeds),
                     tokens, batch, uint64_t(seed_step));
}

}  // namespace rlli
