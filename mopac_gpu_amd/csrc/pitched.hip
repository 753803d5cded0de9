#include "pitched.h"

#include <algorithm>
#include <cstring>

namespace mhip {
namespace {

void host_rows(char* dst, size_t dpitch, const char* src, size_t spitch, size_t width, size_t rows) {
  for (size_t i = 0; i < rows; ++i) std::memcpy(dst + i * dpitch, src + i * spitch, width);
}

}  // namespace

bool PitchedCopy::direct(const void* host, size_t width) const {
  if (width > kMaxSlot) return true;
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, host) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

void PitchedCopy::wait(int i) {
  if (!busy_[i]) return;
  MHIP_CHECK(hipEventSynchronize(ev_[i]));
  busy_[i] = false;
}

// Slots of a third to two thirds of the matrix (within kMinSlot and kMaxSlot),
// which then passes in a few pieces, the host's part of one beside the DMA of
// another; and of one row at least, which `direct` keeps below kMaxSlot.
void PitchedCopy::ensure(size_t width, size_t rows, hipStream_t s) {
  size_t want = kMinSlot;
  while (want < kMaxSlot && (want < width || 3 * want < width * rows)) want *= 2;
  MHIP_REQUIRE(want >= width, "copy through pinned slots: row longer than a slot");
  if (want <= slot_) return;
  release();
  MHIP_CHECK(hipHostMalloc((void**)&pin_, want * kSlots, hipHostMallocDefault));
  slot_ = want;
  // an event belongs to the device that is current, a stream to its own
  int device = 0, of_stream = 0;
  MHIP_CHECK(hipGetDevice(&device));
  MHIP_CHECK(hipStreamGetDevice(s, &of_stream));
  if (device != of_stream) MHIP_CHECK(hipSetDevice(of_stream));
  hipError_t r = hipSuccess;
  for (auto& e : ev_)
    if (r == hipSuccess) r = hipEventCreateWithFlags(&e, hipEventDisableTiming);
  if (device != of_stream) (void)hipSetDevice(device);
  if (r != hipSuccess) release();
  MHIP_CHECK(r);
}

void PitchedCopy::up(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t rows,
                     hipStream_t s) {
  if (width == 0 || rows == 0) return;
  MHIP_REQUIRE(dst && src && dpitch >= width && spitch >= width, "copy to the device: invalid argument");
  if (rows == 1 || (dpitch == width && spitch == width)) {
    MHIP_CHECK(hipMemcpyAsync(dst, src, width * rows, hipMemcpyHostToDevice, s));
    return;
  }
  if (direct(src, width)) {
    MHIP_CHECK(hipMemcpy2DAsync(dst, dpitch, src, spitch, width, rows, hipMemcpyHostToDevice, s));
    return;
  }
  ensure(width, rows, s);
  wait(0);
  wait(1);
  const size_t per = slot_ / width;
  int i = 0;
  for (size_t r = 0; r < rows; r += per, i ^= 1) {
    const size_t n = std::min(per, rows - r);
    char* p = pin_ + i * slot_;
    wait(i);
    host_rows(p, width, static_cast<const char*>(src) + r * spitch, spitch, width, n);
    MHIP_CHECK(hipMemcpy2DAsync(static_cast<char*>(dst) + r * dpitch, dpitch, p, width, width, n,
                                hipMemcpyHostToDevice, s));
    MHIP_CHECK(hipEventRecord(ev_[i], s));
    busy_[i] = true;
  }
}

void PitchedCopy::down(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t rows,
                       hipStream_t s) {
  if (width == 0 || rows == 0) return;
  MHIP_REQUIRE(dst && src && dpitch >= width && spitch >= width, "copy from the device: invalid argument");
  if (rows == 1 || (dpitch == width && spitch == width)) {
    MHIP_CHECK(hipMemcpyAsync(dst, src, width * rows, hipMemcpyDeviceToHost, s));
    MHIP_CHECK(hipStreamSynchronize(s));
    return;
  }
  if (direct(dst, width)) {
    MHIP_CHECK(hipMemcpy2DAsync(dst, dpitch, src, spitch, width, rows, hipMemcpyDeviceToHost, s));
    MHIP_CHECK(hipStreamSynchronize(s));
    return;
  }
  ensure(width, rows, s);
  wait(0);
  wait(1);
  const size_t per = slot_ / width;
  auto issue = [&](size_t r, int i) {
    MHIP_CHECK(hipMemcpy2DAsync(pin_ + i * slot_, width, static_cast<const char*>(src) + r * spitch, spitch, width,
                                std::min(per, rows - r), hipMemcpyDeviceToHost, s));
    MHIP_CHECK(hipEventRecord(ev_[i], s));
    busy_[i] = true;
  };
  issue(0, 0);
  int i = 0;
  for (size_t r = 0; r < rows; r += per, i ^= 1) {
    if (r + per < rows) issue(r + per, i ^ 1);
    wait(i);
    host_rows(static_cast<char*>(dst) + r * dpitch, dpitch, pin_ + i * slot_, width, width, std::min(per, rows - r));
  }
}

void PitchedCopy::release() {
  for (int i = 0; i < kSlots; ++i) {
    if (busy_[i]) (void)hipEventSynchronize(ev_[i]);
    busy_[i] = false;
    if (ev_[i]) (void)hipEventDestroy(ev_[i]);
    ev_[i] = nullptr;
  }
  if (pin_) (void)hipHostFree(pin_);
  pin_ = nullptr;
  slot_ = 0;
}

}  // namespace mhip
