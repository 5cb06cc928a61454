// Executable graphs of decode steps, one per shape, at most `most` of them: beyond that the one that has not been asked for the longest goes.  Nothing may
// be in flight when one is added or they are dropped.
#pragma once

#include <cstddef>
#include <utility>
#include <vector>

namespace pst {

template <typename Key, typename Exec>
class GraphCache {
 public:
  explicit GraphCache(size_t most) : most_(most) {}
  // the shape's graph, which is now the last to go; nullptr: there is none
  Exec find(const Key& key) {
    for (size_t i = 0; i < held_.size(); ++i)
      if (held_[i].first == key) {
        held_.push_back(held_[i]);
        held_.erase(held_.begin() + (std::ptrdiff_t)i);
        return held_.back().second;
      }
    return nullptr;
  }
  template <typename Destroy>
  void add(const Key& key, Exec exec, Destroy&& destroy) {
    for (; held_.size() >= most_; held_.erase(held_.begin())) destroy(held_.front().second);
    held_.emplace_back(key, exec);
  }
  template <typename Destroy>
  void drop(Destroy&& destroy) {
    for (auto& h : held_) destroy(h.second);
    held_.clear();
  }

 private:
  size_t most_;
  std::vector<std::pair<Key, Exec>> held_;      // the last one asked for at the end
};

}  // namespace pst
