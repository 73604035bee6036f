// The arrival-counter blocks of the per-op calls: which one a stream's calls count in, and
// whether its split-K exchange may stay in one XCD's L2. Plain host code.
#pragma once
#include <atomic>
#include <cstdint>
#include <map>
#include <mutex>

namespace drt {

constexpr int OP_COUNTER_BLOCKS = 32, OP_COUNTERS = 4096;

// One per device. A block belongs to one stream, whose launches follow one another; two
// streams on one block would count each other's slices.
class CounterBlocks {
 public:
  enum { UNKNOWN = 0, IN_L2 = 1, FENCED = 2 };
  struct Block {
    int index = 0;
    std::atomic<int> form{UNKNOWN};
    std::mutex mu;
  };

  // The block of a stream handle; null when every block is taken, or for the handle that
  // stands for another stream in each thread (two of them would count in one block at the
  // same time): the caller then takes a path without counters.
  Block* of(uintptr_t stream) {
    if (stream == PER_THREAD) return nullptr;
    std::lock_guard<std::mutex> lock(mu_);
    auto it = blocks_.find(stream);
    if (it == blocks_.end()) {
      if ((int)blocks_.size() >= OP_COUNTER_BLOCKS) return nullptr;
      it = blocks_.try_emplace(stream).first;
      it->second.index = (int)blocks_.size() - 1;
    }
    return &it->second;
  }

  // Whether the exchange runs through device-scope fences on this block's stream: probed
  // there once, since the placement is the stream's (one with a CU mask need not be
  // round-robin where another is). probe() gives the rotation, or a negative number without
  // one; while capturing() it is left for a later call, and the fenced form is the safe one
  // (the same bits). Only calls on the same stream wait for its probe.
  template <class Capturing, class Probe>
  static bool fenced(Block& b, Capturing&& capturing, Probe&& probe) {
    int form = b.form.load(std::memory_order_relaxed);
    if (form == UNKNOWN) {
      std::lock_guard<std::mutex> lock(b.mu);
      form = b.form;
      if (form == UNKNOWN) {
        if (capturing()) return true;
        b.form = form = probe() < 0 ? FENCED : IN_L2;
      }
    }
    return form == FENCED;
  }

  static constexpr uintptr_t PER_THREAD = 2;  // hipStreamPerThread

 private:
  std::mutex mu_;
  std::map<uintptr_t, Block> blocks_;
};

}  // namespace drt
