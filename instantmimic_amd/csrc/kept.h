// Answers of the runtime that a process asks for once (a kernel's occupancy, a device's compute units):
// kept under a key that holds everything the answer depends on, the device among it, and safe with
// several threads.  What belongs to one object (a plan's loaded kernels) is kept in that object and goes
// with it: the address of an unloaded kernel may be given out again.
#pragma once

#include <cstddef>
#include <map>
#include <mutex>

namespace im {

template <class Key, class Value>
class Kept {
 public:
  // The answer for `key`, from `ask(Value &)` the first time.  A status other than 0 is returned and not kept.
  template <class Ask>
  int get(const Key &key, Ask &&ask, Value *value) {
    const std::lock_guard<std::mutex> hold(lock_);
    auto it = known_.find(key);
    if (it == known_.end()) {
      Value answer{};
      if (const int status = ask(answer)) return status;
      if (known_.size() >= kMost) known_.clear();
      it = known_.emplace(key, answer).first;
    }
    *value = it->second;
    return 0;
  }
  static constexpr std::size_t kMost = 512;

 private:
  std::mutex lock_;
  std::map<Key, Value> known_;
};

}  // namespace im
