// Counters for kernels whose last workgroup to arrive merges the parts of
// the others (arrivals.h).

#include <torch/all.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>

namespace vllm_amd {

// One set per stream, whose launches follow each other; 32 sets of 64 KB at
// most. Three kinds of call clear counters of their own: those that want
// more; those of a graph, which may run beside the stream that it was
// captured on; and those of streams that are not torch's (their ids are even
// handles), which may end and come back as another stream while work is
// under way.
at::Tensor arrival_counters(const at::Tensor& like, int64_t n) {
  constexpr size_t SETS = 32;
  constexpr int64_t COUNTERS = 16384;
  auto opt = like.options().dtype(torch::kInt);
  const auto stream = c10::hip::getCurrentHIPStream();
  const int64_t id = stream.id();
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (n > COUNTERS || (id != 0 && id % 2 == 0) ||
      hipStreamIsCapturing(stream.stream(), &capturing) != hipSuccess ||
      capturing != hipStreamCaptureStatusNone)
    return torch::zeros({n}, opt);
  // (Never destroyed: the runtime may be gone by then.)
  static auto* sets = new std::map<std::pair<int, int64_t>, at::Tensor>();
  static std::mutex mu;
  std::lock_guard<std::mutex> guard(mu);
  const auto key = std::make_pair((int)like.get_device(), id);
  auto it = sets->find(key);
  if (it != sets->end()) return it->second;
  auto t = torch::zeros({COUNTERS}, opt);
  if (sets->size() < SETS) sets->emplace(key, t);
  return t;
}

}  // namespace vllm_amd
