/*
 * gp_arena.h -- the device memory of a handle or of a gradient as one allocation.
 */
#pragma once

#include <hip/hip_runtime_api.h>

#include <stddef.h>

#include <utility>
#include <vector>

/* Device memory cut into pieces of 256-byte alignment: take() the sizes, allocate once, then read the pieces. (One
 * hipMalloc and hipFree per buffer made up a quarter of a short gradient: 45 calls of 35 and 116 us.) An allocation that
 * fails leaves the arena as it was made, so that the caller may take() again. */
class Arena {
 public:
  Arena() = default;
  Arena(const Arena &) = delete;
  Arena &operator=(const Arena &) = delete;
  ~Arena() { reset(); }
  /* reserve room for a buffer whose address goes to *p when the arena is allocated */
  template <typename T>
  void take(T **p, size_t bytes) {
    *p = nullptr;
    pieces_.push_back({(void **)p, size_});
    size_ += (bytes + 255) & ~(size_t)255;
  }
  bool allocate() {
    if (size_ && hipMalloc(&base_, size_) != hipSuccess) {
      (void)hipGetLastError(); /* reported here: the next launch's check must not find it */
      base_ = nullptr;
      reset();
      return false;
    }
    for (auto &q : pieces_) *q.first = (char *)base_ + q.second;
    pieces_.clear();
    return true;
  }
  /* give the memory back; the addresses of the pieces are void */
  void reset() {
    if (base_) (void)hipFree(base_);
    base_ = nullptr;
    size_ = 0;
    pieces_.clear();
  }
  void *base() const { return base_; }
  size_t size() const { return size_; }

 private:
  std::vector<std::pair<void **, size_t>> pieces_;
  void *base_ = nullptr;
  size_t size_ = 0;
};
