// PitchedCopy on host memory (hip/hip_runtime.h beside this file): matrices
// around the sizes of a slot, each through slots of its own.  Prints the
// shapes that went wrong.
#include <cstdio>
#include <cstring>
#include <deque>
#include <functional>

#include "../../mopac_gpu_amd/csrc/pitched.hip"

struct FakeEvent {
  size_t at = 0;
};

namespace {

constexpr size_t kGuard = size_t(8) << 20;  // more than the widest row that passes through a slot
constexpr unsigned char kMark = 0xA5;

std::deque<std::function<void()>> queued;
size_t done = 0;  // operations run so far
unsigned char* pin = nullptr;
size_t pin_bytes = 0;
int outside = 0;

void run_to(size_t at) {
  while (done < at) {
    queued.front()();
    queued.pop_front();
    ++done;
  }
}
size_t issued() { return done + queued.size(); }

bool in_guarded(const void* p) {
  const auto* q = static_cast<const unsigned char*>(p);
  return pin && q >= pin && q < pin + pin_bytes + 2 * kGuard;
}
void check_access(const void* p, size_t bytes) {
  const auto* q = static_cast<const unsigned char*>(p);
  if (in_guarded(p) && (q < pin + kGuard || q + bytes > pin + kGuard + pin_bytes)) ++outside;
}
void check_guards() {
  for (size_t i = 0; pin && i < kGuard; ++i)
    if (pin[i] != kMark || pin[kGuard + pin_bytes + i] != kMark) {
      ++outside;
      return;
    }
}

}  // namespace

const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void**, size_t) { return hipErrorInvalidValue; }
hipError_t hipFree(void*) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) {
  if (pin) return hipErrorInvalidValue;
  pin_bytes = bytes;
  pin = new unsigned char[bytes + 2 * kGuard];
  std::memset(pin, kMark, bytes + 2 * kGuard);
  *p = pin + kGuard;
  return hipSuccess;
}
hipError_t hipHostFree(void*) {
  run_to(issued());
  check_guards();
  delete[] pin;
  pin = nullptr;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  a->type = in_guarded(p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, int* d) { return *d = 0, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = new FakeEvent, hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return e->at = issued(), hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { return run_to(e->at), hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return run_to(issued()), hipSuccess; }
hipError_t hipMemcpy2DAsync(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t rows,
                            hipMemcpyKind, hipStream_t) {
  if (width > dpitch || width > spitch) return hipErrorInvalidValue;
  queued.push_back([=] {
    for (size_t r = 0; r < rows; ++r) {
      char* d = static_cast<char*>(dst) + r * dpitch;
      const char* s = static_cast<const char*>(src) + r * spitch;
      check_access(d, width);
      check_access(s, width);
      std::memcpy(d, s, width);
    }
  });
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind k, hipStream_t s) {
  if (k != hipMemcpyHostToDevice || in_guarded(src)) return hipMemcpy2DAsync(dst, bytes, src, bytes, bytes, 1, k, s);
  // pageable memory has been read on return
  const auto* from = static_cast<const char*>(src);
  queued.push_back([dst, staged = std::vector<char>(from, from + bytes)] {
    std::memcpy(dst, staged.data(), staged.size());
  });
  return hipSuccess;
}

namespace {

// `rows` columns of m doubles, pad doubles between them in the caller's array
bool round_trip(size_t m, size_t rows, size_t pad) {
  const size_t w = sizeof(double) * m, host = m + pad, dev = m + 1;
  std::vector<double> a(host * rows), d(dev * rows + 1, -1.0), back(host * rows, -2.0);
  for (size_t i = 0; i < a.size(); ++i) a[i] = (double)i;
  outside = 0;
  mhip::PitchedCopy c;
  c.up(d.data(), sizeof(double) * dev, a.data(), sizeof(double) * host, w, rows, nullptr);
  const std::vector<double> kept = a;
  std::fill(a.begin(), a.end(), -3.0);  // the caller may reuse it
  hipStreamSynchronize(nullptr);
  c.down(back.data(), sizeof(double) * host, d.data(), sizeof(double) * dev, w, rows, nullptr);
  c.release();
  bool good = outside == 0 && d[dev * rows] == -1.0;
  for (size_t r = 0; r < rows; ++r) {
    for (size_t i = 0; i < m; ++i)
      good = good && d[r * dev + i] == kept[r * host + i] && back[r * host + i] == kept[r * host + i];
    good = good && d[r * dev + m] == -1.0;
    for (size_t i = m; i < host; ++i) good = good && back[r * host + i] == -2.0;
  }
  return good;
}

}  // namespace

int main() {
  int bad = 0, all = 0;
  for (size_t m : {1, 77, 300, 8191, 8192, 8193, 9000, 10000, 12000, 16384, 16385, 20000, 24000, 32768, 32769, 40000, 131072, 262145,
                   524287, 524288})
    for (size_t rows : {1, 2, 3, 5, 40}) {
      if (m * rows > 6000000) continue;
      ++all;
      if (!round_trip(m, rows, 3)) {
        ++bad;
        std::printf("wrong: %zu x %zu\n", m, rows);
      }
    }
  std::printf("%d of %d shapes wrong\n", bad, all);
  return bad ? 1 : 0;
}
