// Memory for the partial sums of split reductions (split-K GEMM, split GEMV,
// the one-pass GER adjoint); host only, no HIP dependency, so that a CPU test
// can drive it.
//
// No two pieces of work that may run at the same time share a block, and no
// block is freed while something may still write to it:
//   - outside capture each queue (stream) of the handle has a block of its own,
//     so moving the handle from stream to stream needs no wait in between. A
//     block that has to grow is replaced by one of at least twice its size and
//     kept until the end (all replaced blocks together are no larger than the
//     one in use): growing neither waits nor frees;
//   - a call under graph capture takes a block that belongs to that capture, one
//     for each queue in it, and is kept until the end: eager calls never use
//     it, other graphs neither, and no warm-up is needed.
// Where there is no block, get() returns nullptr and the caller runs its form
// that needs none.
#pragma once

#include <cstddef>
#include <new>
#include <vector>

namespace hcb {

class PartialBlocks {
 public:
  // Queues served side by side; of more, the one used longest ago gives its
  // block back.
  static constexpr size_t kQueues = 128;
  // All blocks of captures together.
  static constexpr size_t kCaptureBytes = (size_t)1 << 30;

  // alloc: nullptr if there is no memory. free: may be called while work on the
  // block is under way, and waits for it.
  PartialBlocks(void *(*alloc)(size_t), void (*free)(void *))
      : alloc_(alloc), free_(free) {}
  PartialBlocks(const PartialBlocks &) = delete;
  PartialBlocks &operator=(const PartialBlocks &) = delete;
  ~PartialBlocks() {
    for (const Block &b : eager_) free_(b.ptr);
    for (const Block &b : captured_) free_(b.ptr);
    for (const Block &b : replaced_) free_(b.ptr);
  }

  // `bytes` for a call on `queue`, under the capture `capture` if `capturing`.
  void *get(const void *queue, bool capturing, unsigned long long capture,
            size_t bytes) {
    try {
      return capturing ? captured(queue, capture, bytes) : eager(queue, bytes);
    } catch (const std::bad_alloc &) {
      return nullptr;
    }
  }

 private:
  struct Block {
    const void *queue;
    unsigned long long capture;
    void *ptr;
    size_t bytes;
  };

  void *eager(const void *queue, size_t bytes) {
    size_t i = 0;
    while (i < eager_.size() && eager_[i].queue != queue) ++i;
    const bool known = i < eager_.size();
    if (!known || eager_[i].bytes < bytes) {
      // (room for the bookkeeping first: what is allocated cannot get lost)
      replaced_.reserve(replaced_.size() + 1);
      eager_.reserve(kQueues);
      Block b{queue, 0, nullptr, rounded(bytes)};
      if (known && b.bytes < 2 * eager_[i].bytes) b.bytes = 2 * eager_[i].bytes;
      if ((b.ptr = alloc_(b.bytes)) == nullptr) return nullptr;
      if (known) {
        replaced_.push_back(eager_[i]);
        eager_[i] = b;
      } else {
        if (eager_.size() == kQueues) give_back();
        eager_.push_back(b);
        i = eager_.size() - 1;
      }
    }
    // latest first
    const Block b = eager_[i];
    for (; i > 0; --i) eager_[i] = eager_[i - 1];
    eager_[0] = b;
    return b.ptr;
  }

  void *captured(const void *queue, unsigned long long capture, size_t bytes) {
    for (size_t i = captured_.size(); i-- > 0;) {
      const Block &b = captured_[i];
      if (b.queue == queue && b.capture == capture && b.bytes >= bytes)
        return b.ptr;
    }
    Block b{queue, capture, nullptr, rounded(bytes)};
    if (b.bytes > kCaptureBytes - captured_bytes_) return nullptr;
    captured_.reserve(captured_.size() + 1);
    if ((b.ptr = alloc_(b.bytes)) == nullptr) return nullptr;
    captured_.push_back(b);
    captured_bytes_ += b.bytes;
    return b.ptr;
  }

  // The block of the queue used longest ago, and those that it replaced.
  void give_back() {
    const void *queue = eager_.back().queue;
    free_(eager_.back().ptr);
    eager_.pop_back();
    size_t n = 0;
    for (const Block &b : replaced_) {
      if (b.queue == queue)
        free_(b.ptr);
      else
        replaced_[n++] = b;
    }
    replaced_.resize(n);
  }

  static size_t rounded(size_t bytes) { return (bytes + 255) / 256 * 256; }

  void *(*alloc_)(size_t);
  void (*free_)(void *);
  std::vector<Block> eager_, captured_, replaced_;
  size_t captured_bytes_ = 0;
};

}  // namespace hcb
