// rcg_pool.hip -- device memory and streams kept between the calls of the
// host-memory entry points, and their large copies.
//
// The MS4 gridder and degridder calls hold some 30 device buffers each, which
// they used to allocate and free on every call: hipMalloc and hipFree take
// 10 us to 1 ms apiece by size, and hipFree waits for the device.  A block
// comes back to the pool only when its call has waited for its stream, so it
// is idle and may go to any thread and stream next.  At most POOL_BYTES are
// kept per process; a block that does not fit is freed, and so is all that is
// kept when an allocation of the library fails and in rcg_shutdown.  The state is never
// destroyed, so nothing calls HIP when the process ends.  Nothing here throws
// (callers are C entry points, destructors and threads): without host memory
// for its lists the pool allocates nothing, or keeps nothing.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <unordered_map>
#include <utility>
#include <vector>

#include "rcg_internal.h"

namespace rcg {
namespace {

constexpr size_t POOL_BYTES = (size_t)4 << 30;
constexpr size_t POOL_STREAMS = 16;
constexpr size_t POOL_PINS = 16;               // kept
// Copies through staging buffers, by up to COPY_THREADS threads.  Pageable
// memory moves at 30 GB/s to the device and 17 GB/s back, one thread copying
// inside the runtime; four threads that copy between the caller's memory and
// pinned buffers of their own, each behind its own stream, reach 48 GB/s both
// ways at 40 to 67 MB (six and eight no more).  Starting them costs 0.1 ms: 4
// MB take 0.17 ms either way, against 0.08 ms to the device and 0.25 ms back
// without them; 15 MB to the device 0.38 against 0.52 ms.
constexpr size_t COPY_MIN_TO = (size_t)8 << 20, COPY_MIN_BACK = (size_t)3 << 20;
constexpr int COPY_THREADS = 4;

struct Pool {
  std::mutex mu;
  size_t kept = 0;
  std::map<std::pair<int, size_t>, std::vector<void *>> free;   // by device and size
  std::unordered_map<void *, std::pair<int, size_t>> out;      // handed out
  std::map<int, std::vector<hipStream_t>> streams;
  std::vector<void *> pins;
};

Pool &pool()
{
  static Pool *p = new Pool;
  return *p;
}

// Sizes in steps of an eighth of their power of two, at least 4 KiB, so that
// calls of nearly equal sizes share blocks.
size_t rounded(size_t bytes)
{
  size_t step = 4096;
  while (step * 8 < bytes) step *= 2;
  return (bytes + step - 1) / step * step;
}

void drop_all(Pool &p)
{
  for (auto &f : p.free)
    for (void *b : f.second) (void)hipFree(b);
  p.free.clear();
  p.kept = 0;
}

bool note_out(Pool &p, void *b, std::pair<int, size_t> key) noexcept
{
  try {
    p.out[b] = key;
    return true;
  } catch (...) {
    return false;
  }
}

// p.mu is held.
hipError_t malloc_or_drop(Pool &p, void **out, size_t bytes)
{
  hipError_t e = hipMalloc(out, bytes);
  if (e != hipSuccess && p.kept) {
    (void)hipGetLastError();
    drop_all(p);
    e = hipMalloc(out, bytes);
  }
  if (e != hipSuccess) {
    *out = nullptr;
    (void)hipGetLastError();
  }
  return e;
}

}  // namespace

hipError_t dev_malloc(void **out, size_t bytes)
{
  Pool &p = pool();
  std::lock_guard<std::mutex> lk(p.mu);
  return malloc_or_drop(p, out, bytes);
}

hipError_t pool_get(void **out, size_t bytes)
{
  Pool &p = pool();
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const size_t size = rounded(bytes ? bytes : 1);
  std::lock_guard<std::mutex> lk(p.mu);
  auto f = p.free.lower_bound({dev, size});
  if (f != p.free.end() && f->first.first == dev && f->first.second <= size + size / 4) {
    void *b = f->second.back();
    if (!note_out(p, b, f->first)) return hipErrorOutOfMemory;
    *out = b;
    f->second.pop_back();
    p.kept -= f->first.second;
    if (f->second.empty()) p.free.erase(f);
    return hipSuccess;
  }
  e = malloc_or_drop(p, out, size);
  if (e == hipSuccess && !note_out(p, *out, {dev, size})) {
    (void)hipFree(*out);
    *out = nullptr;
    e = hipErrorOutOfMemory;
  }
  return e;
}

void pool_put(void *b)
{
  if (!b) return;
  Pool &p = pool();
  std::lock_guard<std::mutex> lk(p.mu);
  const auto o = p.out.find(b);
  const auto key = o->second;
  p.out.erase(o);
  if (p.kept + key.second <= POOL_BYTES) {
    auto f = p.free.end();
    try {
      f = p.free.try_emplace(key).first;
      f->second.push_back(b);
      p.kept += key.second;
      return;
    } catch (...) {
      if (f != p.free.end() && f->second.empty()) p.free.erase(f);
    }
  }
  (void)hipFree(b);
}

hipError_t pool_stream(hipStream_t *st)
{
  Pool &p = pool();
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  {
    std::lock_guard<std::mutex> lk(p.mu);
    const auto s = p.streams.find(dev);
    if (s != p.streams.end() && !s->second.empty()) {
      *st = s->second.back();
      s->second.pop_back();
      return hipSuccess;
    }
  }
  return hipStreamCreateWithFlags(st, hipStreamNonBlocking);
}

void pool_stream_put(hipStream_t st)
{
  Pool &p = pool();
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess) {
    std::lock_guard<std::mutex> lk(p.mu);
    try {
      auto &s = p.streams[dev];
      if (s.size() < POOL_STREAMS) {
        s.push_back(st);
        return;
      }
    } catch (...) {
    }
  }
  (void)hipStreamDestroy(st);
}

void pool_trim()
{
  Pool &p = pool();
  std::lock_guard<std::mutex> lk(p.mu);
  drop_all(p);
  for (auto &d : p.streams)
    for (hipStream_t s : d.second) (void)hipStreamDestroy(s);
  p.streams.clear();
  for (void *b : p.pins) (void)hipHostFree(b);
  p.pins.clear();
}

hipError_t pool_pin(void **out)
{
  Pool &p = pool();
  {
    std::lock_guard<std::mutex> lk(p.mu);
    if (!p.pins.empty()) {
      *out = p.pins.back();
      p.pins.pop_back();
      return hipSuccess;
    }
  }
  return hipHostMalloc(out, PIN_BYTES, hipHostMallocDefault);
}

void pool_pin_put(void *b)
{
  Pool &p = pool();
  {
    std::lock_guard<std::mutex> lk(p.mu);
    try {
      if (p.pins.size() < POOL_PINS) {
        p.pins.push_back(b);
        return;
      }
    } catch (...) {
    }
  }
  (void)hipHostFree(b);
}

namespace {

// One thread's share: every chunk it draws, through its own buffer and stream.
hipError_t copy_chunks(char *dst, const char *src, size_t bytes, size_t chunk, bool to_device,
                       std::atomic<size_t> &next)
{
  void *pin = nullptr;
  hipStream_t st = nullptr;
  hipError_t e = pool_pin(&pin);
  if (e != hipSuccess) return e;
  e = pool_stream(&st);
  while (e == hipSuccess) {
    const size_t at = next.fetch_add(chunk);
    if (at >= bytes) break;
    const size_t n = std::min(chunk, bytes - at);
    if (to_device) {
      memcpy(pin, src + at, n);
      e = hipMemcpyAsync(dst + at, pin, n, hipMemcpyHostToDevice, st);
    } else {
      e = hipMemcpyAsync(pin, src + at, n, hipMemcpyDeviceToHost, st);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e == hipSuccess && !to_device) memcpy(dst + at, pin, n);
  }
  if (st) pool_stream_put(st);
  pool_pin_put(pin);
  return e;
}

}  // namespace

hipError_t pool_copy(void *dst, const void *src, size_t bytes, bool to_device, hipStream_t st)
{
  const hipMemcpyKind kind = to_device ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
  if (bytes < (to_device ? COPY_MIN_TO : COPY_MIN_BACK)) {
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, st);
    return e != hipSuccess || to_device ? e : hipStreamSynchronize(st);
  }
  // the copies run on streams of their own: after what st holds
  hipError_t e = hipStreamSynchronize(st);
  int dev = 0;
  if (e == hipSuccess) e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const size_t chunk = std::min(PIN_BYTES, std::max((size_t)256 << 10, bytes / (4 * COPY_THREADS)));
  std::atomic<size_t> next{0};
  hipError_t err[COPY_THREADS] = {};
  std::thread help[COPY_THREADS];
  int n = 1;
  try {
    for (; n < COPY_THREADS; n++)
      help[n] = std::thread([&, n] {
        err[n] = hipSetDevice(dev);
        if (err[n] == hipSuccess)
          err[n] = copy_chunks(static_cast<char *>(dst), static_cast<const char *>(src), bytes,
                               chunk, to_device, next);
      });
  } catch (...) {
    // fewer helpers: this thread takes what is left
  }
  err[0] = copy_chunks(static_cast<char *>(dst), static_cast<const char *>(src), bytes, chunk,
                       to_device, next);
  for (int k = 1; k < n; k++) help[k].join();
  for (int k = 0; k < n; k++)
    if (err[k] != hipSuccess) {
      // a thread that could not get its buffer or stream: once more, plainly
      (void)hipGetLastError();
      e = hipMemcpyAsync(dst, src, bytes, kind, st);
      return e != hipSuccess ? e : hipStreamSynchronize(st);
    }
  return hipSuccess;
}

}  // namespace rcg
