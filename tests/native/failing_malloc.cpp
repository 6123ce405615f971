// A hipMalloc and a hipHostMalloc for tests: they count, forward to the runtime's, and fail once when told to.
// Loaded with its symbols global before the library under test, whose calls then come here.
#include <cstddef>

namespace {
int (*real)(void**, size_t) = nullptr;
int countdown = -1;  // calls until the one that fails; negative: none
int calls = 0;
int (*real_host)(void**, size_t, unsigned) = nullptr;
int host_countdown = -1, host_calls = 0;
}  // namespace

extern "C" {
void failing_malloc_real(void* f) { real = reinterpret_cast<int (*)(void**, size_t)>(f); }
void failing_malloc_in(int n) { countdown = n; }
int failing_malloc_calls() { return calls; }
void failing_host_malloc_real(void* f) { real_host = reinterpret_cast<int (*)(void**, size_t, unsigned)>(f); }
void failing_host_malloc_in(int n) { host_countdown = n; }
int failing_host_malloc_calls() { return host_calls; }
int hipHostMalloc(void** p, size_t n, unsigned flags) {
  ++host_calls;
  if (host_countdown >= 0 && host_countdown-- == 0) {
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  return real_host(p, n, flags);
}
int hipMalloc(void** p, size_t n) {
  ++calls;
  if (countdown >= 0 && countdown-- == 0) {
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, n);
}
}
