// Copies between the caller's (pageable) matrices and the device.
#pragma once
#include <cstddef>

#include "common.h"

namespace mhip {

// The runtime's 2D copy takes a pageable array row by row, with gaps between
// the rows or without: the eigenvectors of 282 orbitals (636 KB) took 2.5 ms
// each way.  Rows without gaps on either side, or a single row, are a plain
// copy; others pass through two pinned slots, packed or unpacked by the host
// beside the other slot's DMA, which takes rows with gaps from pinned memory at
// its full rate: 60 us.  Memory that the runtime knows (pinned, managed,
// device) is left to it.
//
// One owner, one thread at a time; pins at most kSlots * kMaxSlot bytes.
class PitchedCopy {
 public:
  PitchedCopy() = default;
  PitchedCopy(const PitchedCopy&) = delete;
  PitchedCopy& operator=(const PitchedCopy&) = delete;
  // `rows` rows of `width` bytes to the device, queued on s.  A pageable src
  // may be reused on return.
  void up(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t rows, hipStream_t s);
  // From the device, after what is queued on s; dst is filled on return.
  void down(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t rows, hipStream_t s);
  // Give the pinned memory back, after its copies have ended.
  void release();

 private:
  static constexpr int kSlots = 2;
  static constexpr size_t kMinSlot = size_t(256) << 10, kMaxSlot = size_t(4) << 20;
  bool direct(const void* host, size_t width) const;
  void ensure(size_t width, size_t rows, hipStream_t s);
  void wait(int i);
  char* pin_ = nullptr;
  size_t slot_ = 0;
  hipEvent_t ev_[kSlots] = {};
  bool busy_[kSlots] = {};
};

}  // namespace mhip
