// Direct hipBLASLt linear with explicit algorithm selection.
//
// torch's F.linear lets hipBLASLt's (torch-side) heuristic pick the
// kernel; probing the library's full heuristic candidate list
// (scripts/probe_hipblaslt.cpp) showed the best candidate beats that
// pick by 13-40% on the skinny decode projections of Llama-8B at batch
// 64 (o-proj: 19.5 -> 11.7 us) while losing on others (gate/up) — so
// selection must be MEASURED per shape.  ops/autotune.py races each
// candidate against F.linear at first sight of a shape and calls back
// into lt_linear with the winning index (or falls back to torch).
//
// Layout: y[M,N] = x[M,K] @ W[N,K]^T is expressed column-major as
// C[N,M] = A^T(K,N-view of W) * B(K,M-view of x), all leading dims
// packed.  bf16 in/out, f32 accumulate — identical numerics contract
// to the serving GEMM path.
//
// The 128 MiB workspace is one static per-process device allocation;
// ops on the same stream serialize, and under hipGraph capture the
// enqueued matmul is captured like any other kernel.

#include <torch/library.h>
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/HIPContextLight.h>
#include <ATen/hip/tunable/Tunable.h>
#include <hipblaslt/hipblaslt-ext.hpp>
#include <hipblaslt/hipblaslt.h>

#include "ext_common.h"
#include "kernels.h"

#include <algorithm>
#include <array>
#include <cstdlib>
#include <list>
#include <map>
#include <memory>
#include <mutex>
#include <vector>

namespace {

using at::Tensor;

hipblasLtHandle_t lt_handle() {
  static hipblasLtHandle_t handle = [] {
    hipblasLtHandle_t h;
    TORCH_CHECK(hipblasLtCreate(&h) == HIPBLAS_STATUS_SUCCESS,
                "hipblasLtCreate failed");
    return h;
  }();
  return handle;
}

constexpr size_t kWorkspaceBytes = size_t(128) << 20;

void* lt_workspace() {
  static void* ws = [] {
    void* p = nullptr;
    TORCH_CHECK(hipMalloc(&p, kWorkspaceBytes) == hipSuccess,
                "hipblaslt workspace alloc failed");
    return p;
  }();
  return ws;
}

hipblaslt_ext::Gemm make_gemm(const Tensor& x, const Tensor& w, Tensor& y,
                              const float* alpha, const float* beta) {
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  hipblaslt_ext::Gemm gemm(lt_handle(), HIPBLAS_OP_T, HIPBLAS_OP_N,
                           HIP_R_16BF, HIP_R_16BF, HIP_R_16BF, HIP_R_16BF,
                           HIPBLAS_COMPUTE_32F);
  hipblaslt_ext::GemmEpilogue ep;
  hipblaslt_ext::GemmInputs in;
  in.setA(w.data_ptr());
  in.setB(x.data_ptr());
  in.setC(y.data_ptr());
  in.setD(y.data_ptr());
  in.setAlpha(alpha);
  in.setBeta(beta);
  TORCH_CHECK(gemm.setProblem(N, M, K, 1, ep, in) == HIPBLAS_STATUS_SUCCESS,
              "hipblaslt setProblem failed for M=", M, " N=", N, " K=", K);
  return gemm;
}

void check_linear_args(const Tensor& x, const Tensor& w) {
  TORCH_CHECK(x.scalar_type() == at::kBFloat16 && x.is_contiguous() &&
                  x.dim() == 2, "lt_linear: x must be 2-D contiguous bf16");
  TORCH_CHECK(w.scalar_type() == at::kBFloat16 && w.is_contiguous() &&
                  w.dim() == 2, "lt_linear: w must be 2-D contiguous bf16");
  TORCH_CHECK(x.size(1) == w.size(1), "lt_linear: K mismatch");
}

// y = x @ w^T with an explicit hipBLASLt algorithm index.
Tensor lt_linear(const Tensor& x, const Tensor& w, int64_t algo_index) {
  check_linear_args(x, w);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor y = at::empty({x.size(0), w.size(0)}, x.options());
  static const float alpha = 1.f, beta = 0.f;
  auto gemm = make_gemm(x, w, y, &alpha, &beta);

  std::vector<int> want{int(algo_index)};
  std::vector<hipblasLtMatmulHeuristicResult_t> algos;
  TORCH_CHECK(hipblaslt_ext::getAlgosFromIndex(lt_handle(), want, algos) ==
                      HIPBLAS_STATUS_SUCCESS && !algos.empty(),
              "lt_linear: unknown algo index ", algo_index);
  size_t need = 0;
  TORCH_CHECK(gemm.isAlgoSupported(algos[0].algo, need) ==
                      HIPBLAS_STATUS_SUCCESS && need <= kWorkspaceBytes,
              "lt_linear: algo ", algo_index, " unsupported for shape");
  TORCH_CHECK(gemm.initialize(algos[0].algo, lt_workspace()) ==
              HIPBLAS_STATUS_SUCCESS);
  auto stream = at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
  TORCH_CHECK(gemm.run(stream) == HIPBLAS_STATUS_SUCCESS, "lt_linear run");
  return y;
}

// Heuristic candidate algo indices for this problem, best-first per the
// library's own ranking (the autotuner times them).
Tensor lt_heuristics(const Tensor& x, const Tensor& w, int64_t max_n) {
  check_linear_args(x, w);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  Tensor y = at::empty({x.size(0), w.size(0)}, x.options());
  static const float alpha = 1.f, beta = 0.f;
  auto gemm = make_gemm(x, w, y, &alpha, &beta);
  hipblaslt_ext::GemmPreference pref;
  pref.setMaxWorkspaceBytes(kWorkspaceBytes);
  std::vector<hipblasLtMatmulHeuristicResult_t> algos;
  if (gemm.algoGetHeuristic(int(max_n), pref, algos) !=
      HIPBLAS_STATUS_SUCCESS)
    algos.clear();
  std::vector<int64_t> out;
  for (auto& a : algos) {
    size_t need = 0;
    if (gemm.isAlgoSupported(a.algo, need) == HIPBLAS_STATUS_SUCCESS &&
        need <= kWorkspaceBytes)
      out.push_back(hipblaslt_ext::getIndexFromAlgo(a.algo));
  }
  return at::tensor(out, at::TensorOptions().dtype(at::kLong));
}

// ---- the library's own choice, without looking for it at every call ------
// at::linear asks the library for its pick at each call: 18 us of the host,
// of which 8 are spared by keeping what was found for a shape (a prompt of 165
// rows through 16 layers of 2048 has 31 such products).  The pick may have the
// workspace that at::linear's may, and a process that sets that itself has no plans.
// (One in which plans had up to 128 MiB and at::linear 64 KiB faulted the GPU at its
// first product of either; the cause was not found.)
struct LibraryPlan {
  hipblasLtMatmulDesc_t product = nullptr;
  hipblasLtMatrixLayout_t w = nullptr, x = nullptr, y = nullptr;
  hipblasLtMatmulAlgo_t algo{};
  size_t workspace = 0;
  bool found = false;

  LibraryPlan(int64_t M, int64_t N, int64_t K) {
    const hipblasOperation_t t = HIPBLAS_OP_T, n = HIPBLAS_OP_N;
    hipblasLtMatmulPreference_t pref = nullptr;
    const size_t most = at::cuda::getCUDABlasLtWorkspaceSize();
    hipblasLtMatmulHeuristicResult_t result{};
    int count = 0;
    auto ok = [](hipblasStatus_t s) { return s == HIPBLAS_STATUS_SUCCESS; };
    found =
        ok(hipblasLtMatmulDescCreate(&product, HIPBLAS_COMPUTE_32F,
                                     HIP_R_32F)) &&
        ok(hipblasLtMatmulDescSetAttribute(
            product, HIPBLASLT_MATMUL_DESC_TRANSA, &t, sizeof t)) &&
        ok(hipblasLtMatmulDescSetAttribute(
            product, HIPBLASLT_MATMUL_DESC_TRANSB, &n, sizeof n)) &&
        ok(hipblasLtMatrixLayoutCreate(&w, HIP_R_16BF, K, N, K)) &&
        ok(hipblasLtMatrixLayoutCreate(&x, HIP_R_16BF, K, M, K)) &&
        ok(hipblasLtMatrixLayoutCreate(&y, HIP_R_16BF, N, M, N)) &&
        ok(hipblasLtMatmulPreferenceCreate(&pref)) &&
        ok(hipblasLtMatmulPreferenceSetAttribute(
            pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &most,
            sizeof most)) &&
        ok(hipblasLtMatmulAlgoGetHeuristic(
            at::cuda::getCurrentCUDABlasLtHandle(), product, w, x, y, y, pref,
            1, &result, &count)) &&
        count == 1;
    if (pref) hipblasLtMatmulPreferenceDestroy(pref);
    algo = result.algo;
    workspace = result.workspaceSize;
  }
  LibraryPlan(const LibraryPlan&) = delete;
  ~LibraryPlan() {
    for (auto layout : {w, x, y})
      if (layout) hipblasLtMatrixLayoutDestroy(layout);
    if (product) hipblasLtMatmulDescDestroy(product);
  }
};

// Whether the process leaves the library's workspace as it is
bool library_plans_on() {
  static const bool on = !std::getenv("HIPBLASLT_WORKSPACE_SIZE") &&
                         !std::getenv("CUBLASLT_WORKSPACE_SIZE");
  return on;
}

// Plans by device and sizes, of any thread: the 1024 that were asked for last.  A
// call keeps the plan that it uses.
class LibraryPlans {
 public:
  using Plan = std::shared_ptr<const LibraryPlan>;

  Plan of(int device, int64_t M, int64_t N, int64_t K) {
    const std::lock_guard<std::mutex> lock(mutex_);
    const Key key{device, M, N, K};
    const auto at = places_.find(key);
    if (at != places_.end()) {
      plans_.splice(plans_.begin(), plans_, at->second);
      return plans_.front().second;
    }
    plans_.emplace_front(key, std::make_shared<const LibraryPlan>(M, N, K));
    places_[key] = plans_.begin();
    if (plans_.size() > MOST) {
      places_.erase(plans_.back().first);
      plans_.pop_back();
    }
    return plans_.front().second;
  }

  int64_t kept() {
    const std::lock_guard<std::mutex> lock(mutex_);
    return int64_t(plans_.size());
  }

 private:
  using Key = std::array<int64_t, 4>;
  static constexpr size_t MOST = 1024;
  std::mutex mutex_;
  std::list<std::pair<Key, Plan>> plans_;     // the last one first
  std::map<Key, std::list<std::pair<Key, Plan>>::iterator> places_;
};

LibraryPlans& library_plans() {
  static LibraryPlans all;
  return all;
}

int64_t library_plans_kept() { return library_plans().kept(); }

// The tiles of library_linear: K is divided where that takes less and the parts
// have room in what the library may have.
rlli::TilePlan tiles_for_library(int64_t M, int64_t N, int64_t K) {
  const auto plan = rlli::tile_gemm_plan(int(M), int(N), int(K), false);
  if (plan.splits == 1 ||
      plan.splits * M * N * 4 <=
          int64_t(at::cuda::getCUDABlasLtWorkspaceSize()))
    return plan;
  return rlli::tile_gemm_plan(int(M), int(N), int(K), true);
}

// its 64 rows and 128 columns of a tile, and parts
std::vector<int64_t> tile_numbers(int64_t M, int64_t N, int64_t K) {
  const rlli::TilePlan plan = tiles_for_library(M, N, K);
  return {plan.mh, plan.nh, plan.splits};
}

// x w^T as at::linear has it.  Of many rows, where the library's pick divides K
// and sums in a workspace (beside tiles that do not come out even), tiles of our
// own are faster, which divide K themselves where they are few.  (us, the library,
// tiles of all of K and these: 4096 x 14336, 4300 rows 735, 369 and 369, 7613 979,
// 665 and 665; 6160 x 2048, 7259 rows 188 and 160; 8192 x 28672, 2100 rows 1470 and
// 729; 1024 x 28672, 1900 rows 195, 250 and 99; 2048 x 28672, 3000 rows 283, 349 and
// 273; 64 x 28672, 1100 rows 74, 227 and 38.  Of 410 such products the library was
// faster by 5 % and more at 7, where its pick for one size is far better than for
// those beside it: 576 x 28672, 8000 rows 246, 386 and 267, but 7900 403 and 256;
// 3072 x 28672, 2048 rows 280, 360 and 297, but 1900 454 and 258; 14336 x 7168, 7000
// rows 1005 and 1105, but 6500 1073 and 970.)
Tensor library_linear(const Tensor& x, const Tensor& w) {
  check_linear_args(x, w);
  TORCH_CHECK(x.device() == w.device(), "x and W on one GPU");
  const int64_t M = x.size(0), N = w.size(0), K = x.size(1);
  const auto start = reinterpret_cast<uintptr_t>(x.data_ptr()) |
                     reinterpret_cast<uintptr_t>(w.data_ptr());
  if (M == 0 || N == 0 || K == 0 || start % 16 != 0 || !library_plans_on() ||
      at::globalContext().blasPreferredBackend() != at::BlasBackend::Cublaslt ||
      at::cuda::tunable::getTuningContext()->IsTunableOpEnabled())
    return at::linear(x, w);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
  const auto plan = library_plans().of(x.device().index(), M, N, K);
  if (!plan->found) return at::linear(x, w);
  Tensor y = at::empty({M, N}, x.options()), workspace;
  const auto stream = at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
  if (plan->workspace && M > 1024 && K % 64 == 0 && N % 8 == 0 &&
      std::max({x.numel(), w.numel(), y.numel()}) < int64_t(1) << 31) {
    const rlli::TilePlan tiles = tiles_for_library(M, N, K);
    auto* out = static_cast<uint16_t*>(y.data_ptr());
    const bool divided = tiles.splits > 1;
    if (divided)
      workspace = at::empty({tiles.splits, M, N}, x.options().dtype(at::kFloat));
    float* parts = divided ? workspace.data_ptr<float>() : nullptr;
    rlli::launch_tile_gemm(static_cast<const uint16_t*>(x.data_ptr()),
                           static_cast<const uint16_t*>(w.data_ptr()), parts,
                           divided ? nullptr : out, int(M), int(N), int(K),
                           rlli::TileAct::none, tiles, stream);
    rlli_ext::check_launch("library_linear");
    if (divided) {
      rlli::launch_sum_parts(parts, out, tiles.splits, y.numel(), stream);
      rlli_ext::check_launch("sum_parts");
    }
    return y;
  }
  if (plan->workspace)
    workspace = at::empty({int64_t(plan->workspace)},
                          x.options().dtype(at::kByte));
  const float one = 1.f, zero = 0.f;
  const hipblasStatus_t status = hipblasLtMatmul(
      at::cuda::getCurrentCUDABlasLtHandle(), plan->product, &one,
      w.data_ptr(), plan->w, x.data_ptr(), plan->x, &zero, y.data_ptr(),
      plan->y, y.data_ptr(), plan->y, &plan->algo,
      workspace.defined() ? workspace.data_ptr() : nullptr, plan->workspace,
      stream);
  TORCH_CHECK(status == HIPBLAS_STATUS_SUCCESS, "library_linear: status ",
              int(status), " for M=", M, " N=", N, " K=", K);
  return y;
}

TORCH_LIBRARY_FRAGMENT(rlli, m) {
  m.def("library_linear(Tensor x, Tensor w) -> Tensor");
  m.def("library_plans_on() -> bool", &library_plans_on);
  m.def("library_plans_kept() -> int", &library_plans_kept);
  m.def("tiles_for_library(int m, int n, int k) -> int[]", &tile_numbers);
  m.def("lt_linear(Tensor x, Tensor w, int algo_index) -> Tensor");
  m.def("lt_heuristics(Tensor x, Tensor w, int max_n) -> Tensor");
}

TORCH_LIBRARY_IMPL(rlli, CUDA, m) {
  m.impl("library_linear", library_linear);
  m.impl("lt_linear", lt_linear);
  m.impl("lt_heuristics", lt_heuristics);
}

}  // namespace
