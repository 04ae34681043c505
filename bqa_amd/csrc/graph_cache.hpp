// The captured graphs a job keeps, least recently used first.  Host code without HIP, so its rule is tested on the CPU.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <utility>
#include <vector>

namespace bqa {

// At most CAP graphs by key; a hit becomes the most recent, and a graph beyond CAP replaces the least recent.  So the
// last CAP - 1 graphs found or added outlive the next addition: a BP run takes its two graphs before its first
// replay and may launch both until it ends.
template <typename Exec, size_t CAP>
class GraphCache {
  static_assert(CAP >= 2, "a run's two graphs are kept together");

 public:
  using Key = std::vector<intptr_t>;

  // The graph of `key`, or nullptr.
  Exec* find(const Key& key) {
    for (auto it = kept_.begin(); it != kept_.end(); ++it)
      if (it->first == key) {
        std::rotate(it, it + 1, kept_.end());
        return &kept_.back().second;
      }
    return nullptr;
  }
  // Adds the graph of a key that find() did not have; `destroy` takes the one it replaces.
  template <typename F>
  void add(Key key, Exec exec, F&& destroy) {
    if (kept_.size() >= CAP) {
      destroy(kept_.front().second);
      kept_.erase(kept_.begin());
    }
    kept_.emplace_back(std::move(key), exec);
  }
  template <typename F>
  void clear(F&& destroy) {
    for (auto& g : kept_) destroy(g.second);
    kept_.clear();
  }

 private:
  std::vector<std::pair<Key, Exec>> kept_;
};

}  // namespace bqa
