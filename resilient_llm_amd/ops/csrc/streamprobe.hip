// Microbench kernel: pure nontemporal streaming read of an [N, K] bf16
// weight matrix (64-row panels x splitk, 4 waves, each lane in the rows
// that a matrix operand takes) — what a product that reads its operands
// straight into registers could reach per shape if compute were free.
// Diagnostic only; not part of the serving path.
#include "common.h"

namespace rlli {
namespace {
using u32x4 = __attribute__((ext_vector_type(4))) unsigned int;

__global__ __launch_bounds__(256)
void stream_probe_kernel(const uint16_t* __restrict__ w, float* __restrict__ sink,
                         int N, int K, int chunks_per_slice, int depth) {
  const int n_panels = N / 64;
  const int panel = blockIdx.x % n_panels;
  const int slice = blockIdx.x / n_panels;
  const int total_chunks = K / 256;
  const int c0 = slice * chunks_per_slice;
  const int c1 = min(c0 + chunks_per_slice, total_chunks);
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const uint16_t* wrow = w + int64_t(panel * 64 + wave * 16 + (lane & 15)) * K
                         + (lane >> 4) * 8;
  unsigned acc = 0;
  for (int c = c0; c < c1; ++c) {
#pragma unroll 8
    for (int ks = 0; ks < 8; ++ks) {
      u32x4 v = __builtin_nontemporal_load(
          reinterpret_cast<const u32x4*>(wrow + c * 256 + ks * 32));
      acc ^= v[0] ^ v[1] ^ v[2] ^ v[3];
    }
  }
  if (acc == 0xdeadbeefu) sink[threadIdx.x] = 1.f;  // keep loads live
}
}  // namespace

void launch_stream_probe(const uint16_t* w, float* sink, int N, int K,
                         int splitk, hipStream_t stream) {
  const int total_chunks = K / 256;
  const int cps = (total_chunks + splitk - 1) / splitk;
  hipLaunchKernelGGL(stream_probe_kernel, dim3((N / 64) * splitk), dim3(256),
                     0, stream, w, sink, N, K, cps, splitk);
}
}  // namespace rlli
