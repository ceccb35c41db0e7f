// Stands before the HIP runtime's allocation calls in a process that loads
// it first (global scope): passes them on, counts them, keeps the flags of
// pinned allocations, and refuses sizes above a limit when told to, as a
// runtime that is out of memory does: the call goes on with a size that no
// machine has, so that the runtime keeps the error as its last one.
#include <dlfcn.h>

#include <atomic>
#include <cstddef>
#include <cstdint>

namespace {
template <class F> F runtime(const char *name) {
  static void *lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_LOCAL);
  return lib ? reinterpret_cast<F>(dlsym(lib, name)) : nullptr;
}
constexpr size_t kTooMuch = (size_t)1 << 60;
}  // namespace

extern "C" {
std::atomic<uint64_t> stub_max_pinned{~0ull}, stub_max_device{~0ull};  // largest size granted
std::atomic<uint64_t> stub_pinned{0}, stub_pinned_bytes{0}, stub_frees{0}, stub_refused{0};
std::atomic<uint32_t> stub_pinned_flags_all{~0u};  // the flags every pinned allocation had

int hipHostMalloc(void **p, size_t n, unsigned flags) {
  stub_pinned_flags_all &= flags;
  static const auto f = runtime<int (*)(void **, size_t, unsigned)>("hipHostMalloc");
  if (n > stub_max_pinned) {
    ++stub_refused;
    return f(p, kTooMuch, flags);
  }
  ++stub_pinned;
  stub_pinned_bytes += n;
  return f(p, n, flags);
}
int hipMalloc(void **p, size_t n) {
  static const auto f = runtime<int (*)(void **, size_t)>("hipMalloc");
  if (n > stub_max_device) {
    ++stub_refused;
    return f(p, kTooMuch);
  }
  return f(p, n);
}
int hipFree(void *p) {
  ++stub_frees;
  static const auto f = runtime<int (*)(void *)>("hipFree");
  return f(p);
}
}
