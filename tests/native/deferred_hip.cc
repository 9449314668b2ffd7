// A HIP runtime for the CPU whose copies happen as late as the interface
// allows: memory is host memory, kernels do nothing, and an asynchronous copy
// is carried out by the wait that covers it (hipStreamSynchronize,
// hipEventSynchronize). Loaded with RTLD_GLOBAL before libpikgpu.so, it takes
// the calls that tests/test_copies.py makes through the library.
//
// Every copy remembers what its source held when it was queued; a source that
// holds something else, or is no longer mapped, when the copy is carried out
// is counted by deferred_hip_changed(). A copy that reaches into or out of a
// range known to the runtime (hipHostMalloc, or declared by
// deferred_hip_range) is refused.
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <sys/uio.h>
#include <unistd.h>

#include <map>
#include <vector>

#define API extern "C" __attribute__((visibility("default")))

namespace {

constexpr int kSuccess = 0, kInvalidValue = 1, kHostToDevice = 1;
// HIP_POINTER_ATTRIBUTE_RANGE_START_ADDR and _RANGE_SIZE
constexpr int kRangeStart = 11, kRangeSize = 12;

struct Copy {
  uint8_t* dst;
  const uint8_t* src;
  size_t dpitch, spitch, row, rows;
  std::vector<uint8_t> was;  // the source when queued (host to device)
};
std::vector<Copy> queue;   // waiting
std::vector<size_t> sizes; // bytes of every copy queued so far
size_t done = 0;           // copies carried out
int changed = 0, refused = 0;
std::map<uintptr_t, size_t> ranges;

bool Read(const void* from, void* to, size_t n) {
  iovec a = {to, n}, b = {const_cast<void*>(from), n};
  return n == 0 || process_vm_readv(getpid(), &a, 1, &b, 1, 0) == ssize_t(n);
}

// The known range p starts in, if any.
bool RangeOf(const void* p, uintptr_t* base, size_t* size) {
  auto it = ranges.upper_bound(reinterpret_cast<uintptr_t>(p));
  if (it == ranges.begin()) return false;
  --it;
  *base = it->first;
  *size = it->second;
  return reinterpret_cast<uintptr_t>(p) < *base + *size;
}
bool Fits(const void* p, size_t n) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  uintptr_t base;
  size_t size;
  if (RangeOf(p, &base, &size)) return a + n <= base + size;
  const auto next = ranges.upper_bound(a);
  return next == ranges.end() || a + n <= next->first;
}

int Queue(void* dst, size_t dpitch, const void* src, size_t spitch, size_t row,
          size_t rows, int kind) {
  const size_t reach_s = rows ? (rows - 1) * spitch + row : 0;
  const size_t reach_d = rows ? (rows - 1) * dpitch + row : 0;
  if (!Fits(src, reach_s) || !Fits(dst, reach_d)) {
    refused += 1;
    return kInvalidValue;
  }
  Copy c = {static_cast<uint8_t*>(dst), static_cast<const uint8_t*>(src),
            dpitch, spitch, row, rows, {}};
  if (kind == kHostToDevice) {
    c.was.resize(row * rows);
    for (size_t y = 0; y < rows; ++y) {
      memcpy(&c.was[y * row], c.src + y * spitch, row);
    }
  }
  queue.push_back(c);
  sizes.push_back(row * rows);
  return kSuccess;
}

void CarryOut(size_t upto) {
  size_t n = 0;
  for (; n < queue.size() && done < upto; ++n, ++done) {
    const Copy& c = queue[n];
    std::vector<uint8_t> now(c.row * c.rows);
    bool ok = true;
    for (size_t y = 0; y < c.rows; ++y) {
      ok &= Read(c.src + y * c.spitch, now.data() + y * c.row, c.row);
    }
    if (!ok || (!c.was.empty() && now != c.was)) changed += 1;
    if (!ok) continue;
    for (size_t y = 0; y < c.rows; ++y) {
      memcpy(c.dst + y * c.dpitch, now.data() + y * c.row, c.row);
    }
  }
  queue.erase(queue.begin(), queue.begin() + n);
}

int Alloc(void** p, size_t n) {
  *p = calloc(1, n ? n : 1);
  return kSuccess;
}

}  // namespace

API int deferred_hip_changed() { return changed; }
API int deferred_hip_refused() { return refused; }
API int deferred_hip_waiting() { return int(queue.size()); }
API int deferred_hip_copies() { return int(sizes.size()); }
API size_t deferred_hip_bytes(int i) { return sizes[i]; }
API void deferred_hip_range(void* p, size_t n) {
  ranges[reinterpret_cast<uintptr_t>(p)] = n;
}
API void deferred_hip_forget(void* p) {
  ranges.erase(reinterpret_cast<uintptr_t>(p));
}

API int hipSetDevice(int) { return kSuccess; }
API int hipDeviceGetAttribute(int* v, int, int) {
  *v = 100000;
  return kSuccess;
}
API int hipGetLastError() { return kSuccess; }
API const char* hipGetErrorString(int) { return "deferred_hip error"; }
API int hipStreamCreateWithFlags(void** s, unsigned) { return Alloc(s, 1); }
API int hipStreamDestroy(void* s) {
  free(s);
  return kSuccess;
}
API int hipStreamSynchronize(void*) {
  CarryOut(~size_t(0));
  return kSuccess;
}
API int hipEventCreateWithFlags(void** e, unsigned) {
  return Alloc(e, sizeof(size_t));
}
API int hipEventDestroy(void* e) {
  free(e);
  return kSuccess;
}
API int hipEventRecord(void* e, void*) {
  *static_cast<size_t*>(e) = done + queue.size();
  return kSuccess;
}
API int hipEventSynchronize(void* e) {
  CarryOut(*static_cast<size_t*>(e));
  return kSuccess;
}
API int hipMalloc(void** p, size_t n) { return Alloc(p, n); }
API int hipFree(void* p) {
  CarryOut(~size_t(0));  // hipFree waits for the device
  free(p);
  return kSuccess;
}
API int hipHostMalloc(void** p, size_t n, unsigned) {
  Alloc(p, n);
  deferred_hip_range(*p, n);
  return kSuccess;
}
API int hipHostFree(void* p) {
  CarryOut(~size_t(0));
  deferred_hip_forget(p);
  free(p);
  return kSuccess;
}
API int hipMemcpy(void* dst, const void* src, size_t n, int) {
  CarryOut(~size_t(0));
  memcpy(dst, src, n);
  return kSuccess;
}
API int hipMemcpyAsync(void* dst, const void* src, size_t n, int kind, void*) {
  return Queue(dst, n, src, n, n, 1, kind);
}
API int hipMemcpy2DAsync(void* dst, size_t dpitch, const void* src,
                         size_t spitch, size_t row, size_t rows, int kind,
                         void*) {
  return Queue(dst, dpitch, src, spitch, row, rows, kind);
}
API int hipPointerGetAttribute(void* out, int what, void* p) {
  uintptr_t base;
  size_t size;
  if (!RangeOf(p, &base, &size)) return kInvalidValue;
  if (what == kRangeStart) {
    memcpy(out, &base, sizeof base);
  } else if (what == kRangeSize) {
    memcpy(out, &size, sizeof size);
  } else {
    return kInvalidValue;
  }
  return kSuccess;
}
API int hipLaunchKernel(const void*, uint64_t, uint32_t, uint64_t, uint32_t,
                        void**, size_t, void*) {
  return kSuccess;
}
