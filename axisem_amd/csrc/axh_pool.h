// axh_pool.h -- equal blocks of memory kept for reuse.
//
// A run needs a block of pinned host memory, and pinning one costs 50 to 250 us, more
// than a short run.  A block given back is kept for the next taker (at most `keep` of
// them) while another block is in use, so that a program which makes a batch per set
// of requests pins memory once; with the last block in use all of them are released.
// Any thread may take and give.
#pragma once
#include <cstddef>
#include <mutex>
#include <vector>

namespace axh {

class BlockPool {
 public:
  // make returns a new block or throws; drop releases one and does not throw
  BlockPool(void *(*make)(), void (*drop)(void *), size_t keep)
      : make_(make), drop_(drop), keep_(keep) {
    free_.reserve(keep + 1);
  }
  void *take() {
    std::lock_guard<std::mutex> lock(mu_);
    void *p = nullptr;
    if (free_.empty()) {
      p = make_();
    } else {
      p = free_.back();
      free_.pop_back();
    }
    used_++;
    return p;
  }
  void give(void *p) {
    std::lock_guard<std::mutex> lock(mu_);
    used_--;
    free_.push_back(p);
    while (free_.size() > (used_ > 0 ? keep_ : 0)) {
      drop_(free_.back());
      free_.pop_back();
    }
  }

 private:
  std::mutex mu_;
  void *(*make_)();
  void (*drop_)(void *);
  size_t keep_, used_ = 0;
  std::vector<void *> free_;
};

}  // namespace axh
