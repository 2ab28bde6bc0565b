// The pool of host threads where the system grants fewer threads than it asks
// for: argv[1] of them, then EAGAIN. Every range must be covered exactly once,
// in every one of many calls.
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>

#include "gcs_host_pool.hpp"

static int granted = 0;

extern "C" int pthread_create(pthread_t *t, const pthread_attr_t *a, void *(*f)(void *),
                              void *arg) {
  using Create = int (*)(pthread_t *, const pthread_attr_t *, void *(*)(void *), void *);
  static const Create create = (Create)dlsym(RTLD_NEXT, "pthread_create");
  if (granted == 0) return EAGAIN;
  --granted;
  return create(t, a, f, arg);
}

int main(int argc, char **argv) {
  granted = argc > 1 ? std::atoi(argv[1]) : 0;
  for (long n : {0L, 1L, 2L, 15L, 16L, 17L, 1000L})
    for (int repeat = 0; repeat < 200; ++repeat) {
      std::vector<std::atomic<int>> seen(n);
      for (auto &s : seen) s = 0;
      gcs::HostPool::get().run(n, [&](long b, long e) {
        for (long i = b; i < e; ++i) ++seen[i];
      });
      for (long i = 0; i < n; ++i)
        if (seen[i] != 1) {
          std::printf("n %ld: element %ld seen %d times\n", n, i, (int)seen[i]);
          return 1;
        }
    }
  std::printf("ok\n");
  return 0;
}
