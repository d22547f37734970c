// A few tables kept by key: what a handle has built for its calls. Host code
// without HIP types, so that the CPU tests compile it alone.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <vector>

namespace tt {

// At most `most` values, the least recently used goes first; and which keys
// could not be built, so that a call whose table does not fit the memory does
// not try again, waiting for its stream each time. The caller serialises calls.
// Key: comparable with ==.
template <class Key, class Value>
class Kept {
 public:
  explicit Kept(size_t most) : most_(most) {}

  // The value of k or null. build: a missing one is made, make(&value) saying
  // whether it could be; again: also where it could not before. drop(value)
  // frees the one that has to go.
  template <class Make, class Drop>
  Value* get(const Key& k, bool build, bool again, Make&& make, Drop&& drop) {
    for (Entry& e : made_)
      if (e.key == k) {
        e.turn = ++turn_;
        return &e.value;
      }
    const auto f = std::find(failed_.begin(), failed_.end(), k);
    if (!build || (f != failed_.end() && !again)) return nullptr;
    Entry e;
    e.key = k;
    if (!make(&e.value)) {
      if (f == failed_.end()) {
        if (failed_.size() >= kFailures) failed_.erase(failed_.begin());
        failed_.push_back(k);
      }
      return nullptr;
    }
    if (f != failed_.end()) failed_.erase(f);
    while (made_.size() >= most_ + beyond_) {
      const auto old = std::min_element(made_.begin(), made_.end(),
                                        [](const Entry& a, const Entry& b) { return a.turn < b.turn; });
      drop(old->value);
      made_.erase(old);
    }
    e.turn = ++turn_;
    made_.push_back(e);
    return &made_.back().value;
  }

  // What is kept now; back_to() drops what came since (and forgets its
  // failures). Between them one more than `most` may be kept, so that nothing
  // of before has to go.
  struct Mark {
    std::vector<Key> made, failed;
  };
  Mark mark() {
    ++beyond_;
    Mark m;
    for (const Entry& e : made_) m.made.push_back(e.key);
    m.failed = failed_;
    return m;
  }
  template <class Drop>
  void back_to(const Mark& m, Drop&& drop) {
    --beyond_;
    auto has = [](const std::vector<Key>& v, const Key& k) { return std::find(v.begin(), v.end(), k) != v.end(); };
    for (size_t i = made_.size(); i-- > 0;)
      if (!has(m.made, made_[i].key)) {
        drop(made_[i].value);
        made_.erase(made_.begin() + ptrdiff_t(i));
      }
    failed_ = m.failed;
  }

  template <class Drop>
  void clear(Drop&& drop) {
    for (Entry& e : made_) drop(e.value);
    made_.clear();
    failed_.clear();
  }

  size_t size() const { return made_.size(); }

 private:
  static constexpr size_t kFailures = 64;
  struct Entry {
    Key key{};
    Value value{};
    uint64_t turn = 0;
  };
  size_t most_, beyond_ = 0;
  uint64_t turn_ = 0;
  std::vector<Entry> made_;
  std::vector<Key> failed_;
};

}  // namespace tt
