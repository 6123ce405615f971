// A hipMalloc for tests: forwards to the runtime's, and fails once when told to.  Loaded with its symbols
// global before the library under test, whose calls then come here.
#include <cstddef>

namespace {
int (*real)(void**, size_t) = nullptr;
int countdown = -1;  // calls until the one that fails; negative: none
int calls = 0;
}  // namespace

extern "C" {
void failing_malloc_real(void* f) { real = reinterpret_cast<int (*)(void**, size_t)>(f); }
void failing_malloc_in(int n) { countdown = n; }
int failing_malloc_calls() { return calls; }
int hipMalloc(void** p, size_t n) {
  ++calls;
  if (countdown >= 0 && countdown-- == 0) {
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, n);
}
}
