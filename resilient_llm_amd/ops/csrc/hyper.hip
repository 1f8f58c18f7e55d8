// Residual streams (hyper-connections) fused with the norms around them.
//
// A model with s residual streams reads u = sum_s in[s] x_s, norms u,
// runs a sublayer on it and writes x_t <- sum_s mix[s,t] x_s + out[t] y.
// Done op by op that is five passes over [rows, s, width] 32-bit floats
// per sublayer; here the write of one sublayer and the read + norm of
// the next are ONE pass: each row is loaded once, mixed in registers,
// stored once, and its norm leaves as the next GEMM's input.  Streams,
// mixing and norms are 32-bit; only y and h have the activation type.
// y may come in several parts per row (the chosen experts of a mixture),
// or as the f32 parts of a product that was divided over K (PARTS, one matrix
// per part); both are summed on the way in.  The latter spares a launch that
// sums them (3.9 us for 8 parts of 16 x 2048) and y's rounding.

#include "mix.h"

#include <type_traits>

namespace rlli {
namespace {

template <int WAVES>
DEV_INLINE float wg_sum(float v, float* lds) {
  v = wave_sum(v);
  if constexpr (WAVES == 1) return v;
  __syncthreads();                       // earlier readers are done
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) t += lds[w];
  return t;
}

// IT float4s of a row per thread
template <typename T, int S, int WAVES, int IT, bool EMBED, bool PARTS>
__global__ __launch_bounds__(WAVES * 64)
void hyper_kernel(HyperArgs a) {
  __shared__ float lds[WAVES];
  const int n = blockIdx.x;
  const int64_t row = a.rows ? a.rows[n] : n;
  const int W = a.width;
  float* xr = a.x + row * S * int64_t(W);
  T* hr = reinterpret_cast<T*>(a.h) + int64_t(n) * W;

  float mix[S][S], outw[S], inw[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    inw[s] = a.in_w ? a.in_w[s] : 1.f;
    if constexpr (!EMBED) {
      outw[s] = a.out_w[s];
#pragma unroll
      for (int t = 0; t < S; ++t) mix[s][t] = a.mix[s * S + t];
    }
  }

  f32x4_t u[IT];
  float ss = 0.f;
  if constexpr (EMBED) {
    const T* er = reinterpret_cast<const T*>(a.table) +
                  int64_t(a.ids[n]) * W;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = (i * WAVES * 64 + threadIdx.x) * 4;
      u[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (c < W) u[i] = act_load4(er + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) ss += u[i][j] * u[i][j];
    }
    ss = wg_sum<WAVES>(ss, lds);
    const float inv = 1.f / sqrtf(ss / W + a.eps);
    float insum = 0.f;
#pragma unroll
    for (int s = 0; s < S; ++s) insum += inw[s];
    ss = 0.f;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = (i * WAVES * 64 + threadIdx.x) * 4;
      if (c < W) {
        const f32x4_t g = *reinterpret_cast<const f32x4_t*>(a.w_embed + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) u[i][j] = u[i][j] * inv * g[j];
#pragma unroll
        for (int s = 0; s < S; ++s)
          *reinterpret_cast<f32x4_t*>(xr + int64_t(s) * W + c) = u[i];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        u[i][j] *= insum;
        ss += u[i][j] * u[i][j];
      }
    }
  } else {
    using Y = std::conditional_t<PARTS, float, T>;
    const Y* yr = reinterpret_cast<const Y*>(a.y) +
                  row * (PARTS ? 1 : a.parts) * int64_t(W);
    const int64_t next = PARTS ? int64_t(a.y_rows) * W : W;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = (i * WAVES * 64 + threadIdx.x) * 4;
      u[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (c < W) {
        f32x4_t xs[S];
#pragma unroll
        for (int s = 0; s < S; ++s)
          xs[s] = *reinterpret_cast<const f32x4_t*>(xr + int64_t(s) * W + c);
        f32x4_t y = act_load4(yr + c);
        int p = 1;
        if constexpr (PARTS) {              // seven parts under way at a time
          for (; p + 7 <= a.parts; p += 7) {
            f32x4_t yp[7];
#pragma unroll
            for (int k = 0; k < 7; ++k)
              yp[k] = act_load4(yr + (p + k) * next + c);
#pragma unroll
            for (int k = 0; k < 7; ++k) y += yp[k];
          }
        }
        for (; p < a.parts; ++p) {
          const f32x4_t yp = act_load4(yr + p * next + c);
#pragma unroll
          for (int j = 0; j < 4; ++j) y[j] += yp[j];
        }
#pragma unroll
        for (int t = 0; t < S; ++t) {
          f32x4_t v;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            float acc = outw[t] * y[j];
#pragma unroll
            for (int s = 0; s < S; ++s) acc += mix[s][t] * xs[s][j];
            v[j] = acc;
            u[i][j] += inw[t] * acc;
          }
          if (a.keep)
            *reinterpret_cast<f32x4_t*>(xr + int64_t(t) * W + c) = v;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) ss += u[i][j] * u[i][j];
    }
  }

  ss = wg_sum<WAVES>(ss, lds);
  const float inv = 1.f / sqrtf(ss / W + a.eps);
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int c = (i * WAVES * 64 + threadIdx.x) * 4;
    if (c < W) {
      const f32x4_t g = *reinterpret_cast<const f32x4_t*>(a.gain + c);
      f32x4_t v;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = u[i][j] * inv * g[j];
      act_store4(hr + c, v);
    }
  }
}

template <typename T, int S, bool EMBED, bool PARTS>
void go_width(const HyperArgs& a, hipStream_t st) {
  auto run = [&](auto k, int threads) {
    hipLaunchKernelGGL(k, dim3(a.n), dim3(threads), 0, st, a);
  };
  if (a.width <= 256) run(hyper_kernel<T, S, 1, 1, EMBED, PARTS>, 64);
  else if (a.width <= 1024) run(hyper_kernel<T, S, 4, 1, EMBED, PARTS>, 256);
  // few rows, whose loads are all to be under way at once (8 parts of 16 x
  // 2048: 4.2 us against 6.5 with four waves)
  else if (PARTS && a.width <= 2048)
    run(hyper_kernel<T, S, 8, 1, EMBED, PARTS>, 512);
  else if (PARTS && a.width <= 4096)
    run(hyper_kernel<T, S, 16, 1, EMBED, PARTS>, 1024);
  else if (a.width <= 2048) run(hyper_kernel<T, S, 4, 2, EMBED, PARTS>, 256);
  else if (a.width <= 4096) run(hyper_kernel<T, S, 8, 2, EMBED, PARTS>, 512);
  else run(hyper_kernel<T, S, 8, 4, EMBED, PARTS>, 512);
}

template <typename T, bool EMBED, bool PARTS>
void go_streams(const HyperArgs& a, hipStream_t st) {
  switch (a.streams) {
    case 1: go_width<T, 1, EMBED, PARTS>(a, st); break;
    case 2: go_width<T, 2, EMBED, PARTS>(a, st); break;
    case 3: go_width<T, 3, EMBED, PARTS>(a, st); break;
    case 4: go_width<T, 4, EMBED, PARTS>(a, st); break;
    case 5: go_width<T, 5, EMBED, PARTS>(a, st); break;
    case 6: go_width<T, 6, EMBED, PARTS>(a, st); break;
    case 7: go_width<T, 7, EMBED, PARTS>(a, st); break;
    default: go_width<T, 8, EMBED, PARTS>(a, st); break;
  }
}

template <typename T>
__global__ void relu2_kernel(const T* __restrict__ x, T* __restrict__ out,
                             int64_t n4, int64_t n) {
  const int64_t stride = int64_t(gridDim.x) * blockDim.x;
  int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  for (; i < n4; i += stride) {
    f32x4_t v = act_load4(x + i * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float r = fmaxf(v[j], 0.f);
      v[j] = r * r;
    }
    act_store4(out + i * 4, v);
  }
  i = n4 * 4 + int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  for (; i < n; i += stride) {
    const float r = fmaxf(act_load(x + i), 0.f);
    act_store(out + i, r * r);
  }
}

}  // namespace

void launch_hyper_embed(const HyperArgs& a, hipStream_t st) {
  if (a.n == 0) return;
  if (a.f32) go_streams<float, true, false>(a, st);
  else go_streams<uint16_t, true, false>(a, st);
}

void launch_hyper_step(const HyperArgs& a, hipStream_t st) {
  if (a.n == 0) return;
  if (a.y_rows) go_streams<uint16_t, false, true>(a, st);
  else if (a.f32) go_streams<float, false, false>(a, st);
  else go_streams<uint16_t, false, false>(a, st);
}

void launch_relu2(const void* x, void* out, int64_t n, bool f32,
                  hipStream_t st) {
  if (n == 0) return;
  const int64_t n4 = n / 4;
  int64_t blocks = (n4 + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) blocks = 1;
  if (f32)
    hipLaunchKernelGGL(relu2_kernel<float>, dim3(blocks), dim3(256), 0, st,
                       static_cast<const float*>(x), static_cast<float*>(out),
                       n4, n);
  else
    hipLaunchKernelGGL(relu2_kernel<uint16_t>, dim3(blocks), dim3(256), 0, st,
                       static_cast<const uint16_t*>(x),
                       static_cast<uint16_t*>(out), n4, n);
}

}  // namespace rlli
