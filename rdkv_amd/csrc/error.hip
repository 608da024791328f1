// Thread-local last-error string and version of librdkv_hip.so.
#include "rdkv_common.h"

#include <chrono>

#include <stdarg.h>

static thread_local char g_err[512] = "";

void rdkv_set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

RDKV_API int rdkv_version(void) { return 100; }

RDKV_API const char *rdkv_last_error(void) { return g_err; }

RDKV_API int rdkv_host_words_wait(const uint64_t *words, int64_t n, uint32_t tag, int32_t *values, int64_t wait_us) {
  RDKV_REQUIRE(n >= 0 && (n == 0 || (words && values)), "rdkv_host_words_wait: bad arguments");
  const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(wait_us);
  for (int64_t i = 0; i < n; ++i) {
    for (int spins = 0;; ++spins) {
      const uint64_t w = __atomic_load_n(words + i, __ATOMIC_ACQUIRE);
      if ((uint32_t)(w >> 32) == tag) {
        values[i] = (int32_t)(uint32_t)w;
        break;
      }
      if ((spins & 255) == 255 && std::chrono::steady_clock::now() > until) {
        rdkv_set_error("rdkv_host_words_wait: not there after %lld us", (long long)wait_us);
        return RDKV_EWAIT;
      }
#if defined(__x86_64__)
      __builtin_ia32_pause();
#endif
    }
  }
  return RDKV_OK;
}
