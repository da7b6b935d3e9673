// Tuned hipBLASLt GEMM for the linear layers (bf16/fp16, TN, row-major)
// whose rows are not few enough for stream_linear.hip or tile_linear.hip.
//
// torch's F.linear on ROCm picks heuristics that leave ~1.5-2x on the
// table for both skinny decode shapes (weight-streaming bound) and big
// prefill shapes (hipBLASLt standalone reaches ~2.0 PF bf16 @8k^3 vs
// ~1.3 PF through torch; see profiles/). This op asks hipBLASLt for a
// list of candidate algorithms per (M, N, K, dtype) and picks the
// fastest by measuring each once on first use; the choice is cached for
// the process lifetime. Role of the reference's tuned-GEMM dispatch
// (vllm/model_executor/layers/utils.py apply_w8a8_* and rocm skinny
// gemms csrc/rocm/skinny_gemms.cu) — re-designed around hipBLASLt's own
// search instead of hand-picked kernels.

#include <torch/all.h>
#include <c10/hip/HIPStream.h>

#include <hipblaslt/hipblaslt.h>
#include <hipblaslt/hipblaslt-ext.hpp>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

#include "common.h"
#include "fault_note.h"
#include "tile_linear.h"

namespace vllm_amd {

// stream_linear.hip
bool stream_linear_takes(const torch::Tensor& x, const torch::Tensor& w,
                         int64_t n);
torch::Tensor stream_linear(const torch::Tensor& x, const torch::Tensor& w,
                            const c10::optional<torch::Tensor>& bias);
// tile_linear.hip
bool tile_linear(torch::Tensor& out, const torch::Tensor& x,
                 const torch::Tensor& w, bool silu);

namespace {

#define HIP_CHECK(expr)                                              \
  do {                                                               \
    hipError_t _e = (expr);                                          \
    TORCH_CHECK(_e == hipSuccess, "HIP error: ",                     \
                hipGetErrorString(_e), " at ", __FILE__, ":",        \
                __LINE__);                                           \
  } while (0)

#define HIPBLASLT_CHECK(expr)                                        \
  do {                                                               \
    hipblasStatus_t _st = (expr);                                    \
    TORCH_CHECK(_st == HIPBLAS_STATUS_SUCCESS, "hipBLASLt error ",   \
                (int)_st, " at ", __FILE__, ":", __LINE__);          \
  } while (0)

constexpr size_t kWorkspaceBytes = 128ull * 1024 * 1024;

// What an algorithm is chosen for, in full: products of other types are other
// products, whatever their sizes.
struct ProductKey {
  int64_t m, n, k;
  hipDataType in, out;
  bool bias;
  bool operator<(const ProductKey& o) const {
    return std::tie(m, n, k, in, out, bias) <
           std::tie(o.m, o.n, o.k, o.in, o.out, o.bias);
  }
};

struct LtContext {
  hipblasLtHandle_t handle{nullptr};
  void* workspace{nullptr};
  std::map<ProductKey, hipblasLtMatmulAlgo_t> algo_cache;
  std::mutex mu;
};

LtContext& ctx() {
  static LtContext c;
  static std::once_flag once;
  std::call_once(once, [] {
    HIPBLASLT_CHECK(hipblasLtCreate(&c.handle));
    HIP_CHECK(hipMalloc(&c.workspace, kWorkspaceBytes));
  });
  return c;
}

// Cache lookup, or race hipBLASLt's candidate algorithms for this
// (desc, layouts) once — `call` runs the matmul with a given algo — and
// cache the winner.
//
// Candidate pool: the heuristic's 48 and, where it gains anything, the
// library's full algorithm list (hipblaslt_ext::getAllAlgos, shape-filtered by
// matmulIsAlgoSupported). Two-phase race: one timed rep over every supported
// candidate, then a longer rerace of the top finishers.
// VLLM_AMD_GEMM_TUNE=quick restores heuristic-only.
//
// The full list holds algorithms that say they support a shape and compute
// something else, and they are fast: at K = 64 they won the race of 64 to 2048
// rows x 65536 columns with sums of what the workspace held before. So the
// winner is the fastest whose result is that of the heuristic's first choice,
// out of memory that nothing has been left in.
//
// Nothing vouches for them but that, and a process has ended in a segmentation
// fault of the host within a race of 65 x 4096 x 4096, for a cause that is not
// known. So they stay out where they gain nothing: products of 65 to 128 rows
// with 16 MB of weights and more in 16 bits. us by the heuristic's alone and by
// all, each the better of two races: 72 rows 4096 x 4096 14.8 and 14.9, 6144 x
// 4096 19.5 and 19.5, 37888 x 3584 56.3 and 56.5, 5120 x 4096 17.0 and 16.6, 128
// rows 20.4 and 20.6, 112 rows 4608 x 3584 18.2 and 17.8, 2048 x 4096 10.7 and
// 10.8 (and a first call of 60 ms takes 10).
// Smaller weights gain (96 rows, 3072 x 1024 8.6 and 6.6, 1024 x 2048 8.5 and
// 6.5), and so do some products of more rows (250 x 24576 x 1536 31.4 and 29.5,
// 1024 x 37888 x 3584 254 and 230). Whatever is called next is noted, so that
// a process that does not come back says what it was.
template <typename Call>
hipblasLtMatmulAlgo_t pick_algo(const ProductKey& key,
                                hipblasLtMatmulDesc_t op_desc,
                                hipblasLtMatrixLayout_t lw,
                                hipblasLtMatrixLayout_t la,
                                hipblasLtMatrixLayout_t lc,
                                hipStream_t stream, const torch::Tensor& out,
                                Call call) {
  auto& c = ctx();
  {
    std::lock_guard<std::mutex> g(c.mu);
    auto it = c.algo_cache.find(key);
    if (it != c.algo_cache.end()) return it->second;
  }
  hipblasLtMatmulPreference_t pref;
  HIPBLASLT_CHECK(hipblasLtMatmulPreferenceCreate(&pref));
  HIPBLASLT_CHECK(hipblasLtMatmulPreferenceSetAttribute(
      pref, HIPBLASLT_MATMUL_PREF_MAX_WORKSPACE_BYTES, &kWorkspaceBytes,
      sizeof(kWorkspaceBytes)));
  constexpr int kMaxAlgos = 48;
  std::vector<hipblasLtMatmulHeuristicResult_t> results(kMaxAlgos);
  int found = 0;
  HIPBLASLT_CHECK(hipblasLtMatmulAlgoGetHeuristic(
      c.handle, op_desc, lw, la, lc, lc, pref, kMaxAlgos, results.data(),
      &found));
  HIPBLASLT_CHECK(hipblasLtMatmulPreferenceDestroy(pref));
  results.resize(found);
  // (Of one that did not succeed nothing else holds.)
  const auto failed = [](const hipblasLtMatmulHeuristicResult_t& r) {
    return r.state != HIPBLAS_STATUS_SUCCESS;
  };
  results.erase(std::remove_if(results.begin(), results.end(), failed),
                results.end());
  found = (int)results.size();
  TORCH_CHECK(found > 0, "hipBLASLt: no algorithms for this GEMM");

  FaultNote note;
  auto say = [&](const char* what, int i, int n) {
    note.say("algorithms of a library product, %lld x %lld x %lld (rows, "
             "columns, K; types %d to %d%s): %s, %d of %d (%d by its "
             "heuristic)", (long long)key.m, (long long)key.n,
             (long long)key.k, (int)key.in, (int)key.out,
             key.bias ? ", bias" : "", what, i, n, found);
  };
  const char* tune = getenv("VLLM_AMD_GEMM_TUNE");
  const bool gains = key.m <= 64 || key.m > 128 ||
                     key.n * key.k < (1 << 23) || key.in == HIP_R_32F ||
                     key.in == HIP_R_8F_E4M3;
  if (gains && (tune == nullptr || strcmp(tune, "quick") != 0)) {
    say("listing", 0, 0);
    std::vector<hipblasLtMatmulHeuristicResult_t> all;
    if (hipblaslt_ext::getAllAlgos(
            c.handle, hipblaslt_ext::GemmType::HIPBLASLT_GEMM,
            HIPBLAS_OP_T, HIPBLAS_OP_N, key.in, key.in, key.out, key.out,
            HIPBLAS_COMPUTE_32F, all) == HIPBLAS_STATUS_SUCCESS) {
      const float alpha = 1.f, beta = 0.f;
      for (size_t i = 0; i < all.size(); ++i) {
        auto& r = all[i];
        if (failed(r)) continue;
        say("asked whether supported", (int)i, (int)all.size());
        size_t ws = 0;
        if (hipblaslt_ext::matmulIsAlgoSupported(c.handle, op_desc, &alpha,
                                                 lw, la, &beta, lc, lc,
                                                 r.algo, ws) ==
                HIPBLAS_STATUS_SUCCESS &&
            ws <= kWorkspaceBytes)
          results.push_back(r);
      }
    }
  }

  hipEvent_t ev0, ev1;
  HIP_CHECK(hipEventCreate(&ev0));
  HIP_CHECK(hipEventCreate(&ev1));
  auto time_algo = [&](const hipblasLtMatmulAlgo_t& algo,
                       int reps) -> float {
    if (call(algo, out, c.workspace) != HIPBLAS_STATUS_SUCCESS)
      return 1e30f;  // warm + probe
    HIP_CHECK(hipEventRecord(ev0, stream));
    for (int r = 0; r < reps; ++r) (void)call(algo, out, c.workspace);
    HIP_CHECK(hipEventRecord(ev1, stream));
    HIP_CHECK(hipEventSynchronize(ev1));
    float ms = 1e30f;
    HIP_CHECK(hipEventElapsedTime(&ms, ev0, ev1));
    return ms;
  };
  // Phase A: one rep each over the whole pool.
  std::vector<std::pair<float, int>> ranked;
  ranked.reserve(results.size());
  for (int i = 0; i < (int)results.size(); ++i) {
    say("timed", i, (int)results.size());
    ranked.emplace_back(time_algo(results[i].algo, 1), i);
  }
  std::sort(ranked.begin(), ranked.end(),
            [](auto& x, auto& y) { return x.first < y.first; });
  // Phase B: rerace the 12 fastest with more reps.
  for (int j = 0; j < std::min<int>(12, (int)ranked.size()); ++j)
    if (ranked[j].first < 1e30f) {
      say("timed again", ranked[j].second, (int)results.size());
      ranked[j].first = time_algo(results[ranked[j].second].algo, 8);
    }
  std::sort(ranked.begin(),
            ranked.begin() + std::min<int>(12, (int)ranked.size()),
            [](auto& x, auto& y) { return x.first < y.first; });
  HIP_CHECK(hipEventDestroy(ev0));
  HIP_CHECK(hipEventDestroy(ev1));
  // (The workspace that all products share may be in use on another stream.)
  const auto space = torch::empty({(int64_t)(kWorkspaceBytes / 4)},
                                  out.options().dtype(torch::kFloat));
  auto run_clean = [&](int i, const torch::Tensor& to) {
    say("compared", i, (int)results.size());
    space.fill_(NAN);
    to.fill_(NAN);
    return call(results[i].algo, to, space.data_ptr()) ==
           HIPBLAS_STATUS_SUCCESS;
  };
  const auto expect = torch::empty_like(out);
  int first = 0;
  while (first < found && !run_clean(first, expect)) ++first;
  const double rms = at::norm(expect, 2, torch::kFloat).item<double>() /
                     std::sqrt((double)expect.numel());
  auto agrees = [&](int i) {
    // (Of operands that are not finite nothing can be told.)
    if (first == found || !std::isfinite(rms)) return i < found;
    if (i == first) return true;
    if (!run_clean(i, out)) return false;
    const int64_t M = out.size(0);
    const int64_t rows = std::max<int64_t>(1, (1 << 24) / out.size(1));
    for (int64_t r = 0; r < M; r += rows) {
      const auto e = expect.narrow(0, r, std::min(rows, M - r));
      const auto d = out.narrow(0, r, std::min(rows, M - r)) - e;
      if (!d.abs().le((e.abs() + rms) * (1. / 64)).all().item<bool>())
        return false;
    }
    return true;
  };
  int best_i = first < found ? first : ranked[0].second;
  for (const auto& [time, i] : ranked)
    if (time < 1e30f && agrees(i)) {
      best_i = i;
      break;
    }
  std::lock_guard<std::mutex> g(c.mu);
  c.algo_cache.emplace(key, results[best_i].algo);
  return results[best_i].algo;
}

// C[M,N] row-major = A[M,K] row-major * W[N,K]^T row-major (+bias[N]).
// In hipBLASLt's column-major view: C'[N,M] = op_T(W'[K,N]) * op_N(A'[K,M]).
void run_matmul(torch::Tensor& out, const torch::Tensor& a,
                const torch::Tensor& w, const c10::optional<torch::Tensor>& bias) {
  const int64_t M = a.size(0);
  const int64_t K = a.size(1);
  const int64_t N = w.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(0) == M && out.size(1) == N);
  TORCH_CHECK(a.is_contiguous() && w.is_contiguous() && out.is_contiguous());
  const bool is_bf16 = a.scalar_type() == torch::kBFloat16;
  const bool is_f32 = a.scalar_type() == torch::kFloat32;
  TORCH_CHECK(is_bf16 || is_f32 || a.scalar_type() == torch::kHalf,
              "lt_linear: bf16, fp16 or fp32 operands");
  TORCH_CHECK(w.scalar_type() == a.scalar_type() &&
              out.scalar_type() == a.scalar_type());
  // fp32 operands run true fp32 (COMPUTE_32F, no reduced-precision
  // matrix mode).
  hipDataType dt = is_f32 ? HIP_R_32F : (is_bf16 ? HIP_R_16BF : HIP_R_16F);

  auto& c = ctx();
  auto stream = c10::hip::getCurrentHIPStream().stream();

  hipblasLtMatmulDesc_t op_desc;
  HIPBLASLT_CHECK(hipblasLtMatmulDescCreate(&op_desc, HIPBLAS_COMPUTE_32F,
                                            HIP_R_32F));
  hipblasOperation_t opA = HIPBLAS_OP_T;
  hipblasOperation_t opB = HIPBLAS_OP_N;
  HIPBLASLT_CHECK(hipblasLtMatmulDescSetAttribute(
      op_desc, HIPBLASLT_MATMUL_DESC_TRANSA, &opA, sizeof(opA)));
  HIPBLASLT_CHECK(hipblasLtMatmulDescSetAttribute(
      op_desc, HIPBLASLT_MATMUL_DESC_TRANSB, &opB, sizeof(opB)));
  const bool has_bias = bias.has_value();
  if (has_bias) {
    hipblasLtEpilogue_t epi = HIPBLASLT_EPILOGUE_BIAS;
    HIPBLASLT_CHECK(hipblasLtMatmulDescSetAttribute(
        op_desc, HIPBLASLT_MATMUL_DESC_EPILOGUE, &epi, sizeof(epi)));
    const void* bptr = bias->data_ptr();
    HIPBLASLT_CHECK(hipblasLtMatmulDescSetAttribute(
        op_desc, HIPBLASLT_MATMUL_DESC_BIAS_POINTER, &bptr, sizeof(bptr)));
  }

  // Column-major descriptors: A-slot = W (K x N viewed, opT), ld = K.
  hipblasLtMatrixLayout_t lw, la, lc;
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&lw, dt, K, N, K));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&la, dt, K, M, K));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&lc, dt, N, M, N));

  const float alpha = 1.f, beta = 0.f;

  auto call = [&](const hipblasLtMatmulAlgo_t& cand,
                  const torch::Tensor& to, void* space) {
    return hipblasLtMatmul(
        c.handle, op_desc, &alpha, w.data_ptr(), lw, a.data_ptr(), la,
        &beta, to.data_ptr(), lc, to.data_ptr(), lc, &cand, space,
        kWorkspaceBytes, stream);
  };
  hipblasLtMatmulAlgo_t algo =
      pick_algo({M, N, K, dt, dt, has_bias}, op_desc, lw, la, lc, stream, out,
                call);

  HIPBLASLT_CHECK(hipblasLtMatmul(
      c.handle, op_desc, &alpha, w.data_ptr(), lw, a.data_ptr(), la, &beta,
      out.data_ptr(), lc, out.data_ptr(), lc, &algo, c.workspace,
      kWorkspaceBytes, stream));

  HIPBLASLT_CHECK(hipblasLtMatrixLayoutDestroy(lw));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutDestroy(la));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutDestroy(lc));
  HIPBLASLT_CHECK(hipblasLtMatmulDescDestroy(op_desc));
}

// fp8 e4m3 x fp8 e4m3 -> bf16 raw GEMM (no scaling — the caller rescales
// rows/cols in one fused pass; see quant_fp8.hip). Same tuned-algo cache
// as the 16-bit and fp32 products.
// gfx950 fp8 MFMA peak is ~2x bf16, so big prefill GEMMs roughly double.
void run_matmul_fp8(torch::Tensor& out, const torch::Tensor& a,
                    const torch::Tensor& w) {
  const int64_t M = a.size(0);
  const int64_t K = a.size(1);
  const int64_t N = w.size(0);
  TORCH_CHECK(w.size(1) == K && out.size(0) == M && out.size(1) == N);
  TORCH_CHECK(a.is_contiguous() && w.is_contiguous() && out.is_contiguous());
  TORCH_CHECK(a.scalar_type() == torch::kFloat8_e4m3fn &&
              w.scalar_type() == torch::kFloat8_e4m3fn);
  TORCH_CHECK(out.scalar_type() == torch::kBFloat16);

  auto& c = ctx();
  auto stream = c10::hip::getCurrentHIPStream().stream();

  hipblasLtMatmulDesc_t op_desc;
  HIPBLASLT_CHECK(hipblasLtMatmulDescCreate(&op_desc, HIPBLAS_COMPUTE_32F,
                                            HIP_R_32F));
  hipblasOperation_t opA = HIPBLAS_OP_T;
  hipblasOperation_t opB = HIPBLAS_OP_N;
  HIPBLASLT_CHECK(hipblasLtMatmulDescSetAttribute(
      op_desc, HIPBLASLT_MATMUL_DESC_TRANSA, &opA, sizeof(opA)));
  HIPBLASLT_CHECK(hipblasLtMatmulDescSetAttribute(
      op_desc, HIPBLASLT_MATMUL_DESC_TRANSB, &opB, sizeof(opB)));

  hipblasLtMatrixLayout_t lw, la, lc;
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&lw, HIP_R_8F_E4M3, K, N, K));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&la, HIP_R_8F_E4M3, K, M, K));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutCreate(&lc, HIP_R_16BF, N, M, N));

  const float alpha = 1.f, beta = 0.f;

  auto call = [&](const hipblasLtMatmulAlgo_t& cand,
                  const torch::Tensor& to, void* space) {
    return hipblasLtMatmul(
        c.handle, op_desc, &alpha, w.data_ptr(), lw, a.data_ptr(), la,
        &beta, to.data_ptr(), lc, to.data_ptr(), lc, &cand, space,
        kWorkspaceBytes, stream);
  };
  hipblasLtMatmulAlgo_t algo =
      pick_algo({M, N, K, HIP_R_8F_E4M3, HIP_R_16BF, false}, op_desc, lw, la,
                lc, stream, out, call);

  HIPBLASLT_CHECK(hipblasLtMatmul(
      c.handle, op_desc, &alpha, w.data_ptr(), lw, a.data_ptr(), la, &beta,
      out.data_ptr(), lc, out.data_ptr(), lc, &algo, c.workspace,
      kWorkspaceBytes, stream));

  HIPBLASLT_CHECK(hipblasLtMatrixLayoutDestroy(lw));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutDestroy(la));
  HIPBLASLT_CHECK(hipblasLtMatrixLayoutDestroy(lc));
  HIPBLASLT_CHECK(hipblasLtMatmulDescDestroy(op_desc));
}

}  // namespace

torch::Tensor lt_linear_fp8(torch::Tensor a, torch::Tensor w) {
  TORCH_CHECK(w.device() == a.device(), "operands on ", w.device(), " and ",
              a.device());
  auto out = torch::empty({a.size(0), w.size(0)},
                          a.options().dtype(torch::kBFloat16));
  run_matmul_fp8(out, a, w);
  return out;
}

torch::Tensor lt_linear(torch::Tensor a, torch::Tensor w,
                        c10::optional<torch::Tensor> bias) {
  // (An operand elsewhere would be read by its address there.)
  TORCH_CHECK(w.device() == a.device() &&
                  (!bias.has_value() || bias->device() == a.device()),
              "operands on ", w.device(), " and ", a.device());
  auto sizes = a.sizes().vec();
  const int64_t K = sizes.back();
  auto a2 = a.reshape({-1, K}).contiguous();
  sizes.back() = w.size(0);
  // Few rows stream the weights through a kernel of our own, and some more
  // meet them in tiles (which side is faster at which size: stream_linear.hip
  // and tile_linear.hip).
  const bool ours =
      w.dim() == 2 && a2.size(0) > 0 &&
      (!bias.has_value() ||
       (bias->scalar_type() == a2.scalar_type() && bias->is_contiguous() &&
        bias->numel() == w.size(0)));
  if (ours &&
      (bias.has_value() ||
       !tile_linear_first(a2.size(0), w.size(0), K, false)) &&
      stream_linear_takes(a2, w, w.size(0)))
    return stream_linear(a2, w, bias).reshape(sizes);
  auto out = torch::empty({a2.size(0), w.size(0)}, a.options());
  if (ours && !bias.has_value() && tile_linear(out, a2, w, false))
    return out.reshape(sizes);
  run_matmul(out, a2, w, bias);
  return out.reshape(sizes);
}

}  // namespace vllm_amd
