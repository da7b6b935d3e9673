// Counters for kernels whose last workgroup to arrive merges the parts of
// the others (arrivals.h).

#include <torch/all.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>

#include "arrivals.h"

namespace vllm_amd {

namespace {

// Whether a stream takes part in a capture, and in which.
struct Capture {
  bool known, active;
  unsigned long long id;
  bool operator==(const Capture& o) const {
    return known && o.known && active == o.active && id == o.id;
  }
};
Capture capture_of(hipStream_t stream) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  const bool known =
      hipStreamGetCaptureInfo(stream, &status, &id) == hipSuccess &&
      status != hipStreamCaptureStatusInvalidated;
  const bool active = status == hipStreamCaptureStatusActive;
  return {known, active, active ? id : 0};
}

struct Captured {
  hipStream_t stream;
  Capture capture;
  at::Tensor counters;
};

}  // namespace

// One set per stream, whose launches follow each other; 32 sets of 64 KB at
// most. A graph may run beside the stream that it was captured on, so its
// launches have a set of their own, from the graph's memory, for each stream
// of the capture: the first of them clears it and all leave it zero. (With a
// fill a launch, us in a graph: attention of 8 rows of 33..160 keys 9.0, now 7.4;
// 64 rows x 1024 x 4096 10.8, now 9.4.) It is held until the capture has ended,
// as long as the graph might give its place to others.
// Two kinds of call clear counters of their own: those that want more, and
// those of streams that are not torch's (their ids are even handles), which
// may end and come back as another stream while work is under way.
at::Tensor arrival_counters(const at::Tensor& like, int64_t n) {
  constexpr size_t SETS = 32;
  auto opt = like.options().dtype(torch::kInt);
  const auto stream = c10::hip::getCurrentHIPStream();
  const int64_t id = stream.id();
  const auto capture = capture_of(stream.stream());
  const int64_t blocks = (n + ARRIVAL_BLOCK - 1) / ARRIVAL_BLOCK;
  if (blocks > 1 || (id != 0 && id % 2 == 0) || !capture.known)
    return torch::zeros({blocks * ARRIVAL_BLOCK}, opt);
  // (Never destroyed: the runtime may be gone by then.)
  using Key = std::pair<int, int64_t>;
  static auto* sets = new std::map<Key, at::Tensor>();
  static auto* captured = new std::map<Key, Captured>();
  static std::mutex mu;
  std::lock_guard<std::mutex> guard(mu);
  for (auto it = captured->begin(); it != captured->end();)
    it = capture_of(it->second.stream) == it->second.capture
             ? std::next(it)
             : captured->erase(it);
  const auto key = std::make_pair((int)like.get_device(), id);
  if (capture.active) {
    auto it = captured->find(key);
    if (it != captured->end()) return it->second.counters;
    auto t = torch::zeros({ARRIVAL_BLOCK}, opt);
    if (captured->size() < SETS)
      captured->emplace(key, Captured{stream.stream(), capture, t});
    return t;
  }
  auto it = sets->find(key);
  if (it != sets->end()) return it->second;
  auto t = torch::zeros({ARRIVAL_BLOCK}, opt);
  if (sets->size() < SETS) sets->emplace(key, t);
  return t;
}

}  // namespace vllm_amd
