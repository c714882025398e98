// hipMalloc with failures on demand, for tests/test_gpu_no_memory.py: loaded
// with its symbols global before libacc_cn.so, it stands before the runtime's
// hipMalloc in that process and passes on every request but those of the chosen sizes.
#include <stddef.h>

static int (*real)(void **, size_t);
static size_t lo = 1, hi = 0;
static long failed = 0;

extern "C" {
void fail_alloc_real(void *f) { real = reinterpret_cast<int (*)(void **, size_t)>(f); }
void fail_alloc_between(size_t least, size_t most) {
  lo = least;
  hi = most;
  failed = 0;
}
long fail_alloc_failed() { return failed; }
int hipMalloc(void **p, size_t bytes) {
  if (bytes >= lo && bytes <= hi) {
    failed++;
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, bytes);
}
}
