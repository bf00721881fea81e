// Which of the library's counters an attention launch meets on: the host's part of the choice (no device code).
#pragma once

#include <cstdint>
#include <mutex>

namespace mlakv {

// A name for the memory of a workspace of `bytes` bytes, such that workspaces that do not overlap have different names. From two
// pages on it is the first page that lies in the workspace as a whole, so that a program that carves its workspaces
// anew again and again comes by few names; below that the address. (Odd and even: the two kinds never meet, and no name is 0.)
constexpr uint64_t kWorkspacePage = uint64_t{8} << 20;
inline uint64_t WorkspaceName(const void* workspace, uint64_t bytes) {
  const uint64_t address = reinterpret_cast<uintptr_t>(workspace);
  if (bytes < 2 * kWorkspacePage) return address & ~uint64_t{1};
  return 2 * ((address + kWorkspacePage - 1) / kWorkspacePage) + 1;
}

// Hands every name a region of its own, the same one each time. Launches that share a workspace are ordered by their
// caller, whose partials they would overwrite otherwise, so launches that share a region are ordered too, however
// many are in flight, and also when they are replayed from a recording, which holds its region for good. For that
// reason a region is never taken back either: when all are handed out, a new name gets none (-1).
template <int kRegions>
class SyncRegions {
 public:
  int Of(uint64_t name) {
    std::lock_guard<std::mutex> lock(guard_);
    uint64_t at = (name * 0x9e3779b97f4a7c15ull) >> 32;
    for (int i = 0; i < kRegions; ++i, ++at) {
      uint64_t& held = names_[at % kRegions];
      if (held == 0) held = name;
      if (held == name) return static_cast<int>(at % kRegions);
    }
    return -1;
  }

 private:
  std::mutex guard_;
  uint64_t names_[kRegions] = {};
};

// Workgroups per unit of 16 heads where there are no counters for the `parts` that were chosen: one, or the 64-head kernel (0) for
// more tokens than one stages.
constexpr int PartsWithoutCounters(int parts) { return parts > 4 ? 0 : (parts > 1 ? 1 : parts); }

}  // namespace mlakv
