// Stands in front of hipMalloc when loaded (RTLD_GLOBAL) before the product
// library: once armed, the count-th allocation from then on fails as it does
// when memory has run out.
#include <dlfcn.h>
#include <stddef.h>

static int left = -1;

extern "C" void oom_arm(int count) { left = count; }

extern "C" int hipMalloc(void** p, size_t n) {
  typedef int (*fn)(void**, size_t);
  static fn real = (fn)dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY), "hipMalloc");
  if (left > 0 && --left == 0) {
    left = -1;
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, n);
}
