// Shares of a host loop where threads cannot be started (pthread_create fails after the
// first `allowed` calls) and where shares throw.  Usage: t_host_threads shares allowed thrower
#include <dlfcn.h>
#include <errno.h>
#include <pthread.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../../codeare_amd/csrc/host_threads.hpp"

static std::atomic<int> g_allowed{0};

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* x) {
  typedef int (*Create)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*);
  static const Create real = (Create)dlsym(RTLD_NEXT, "pthread_create");
  return g_allowed-- > 0 ? real(t, a, f, x) : EAGAIN;
}

int main(int argc, char** argv) {
  if (argc != 4) return 2;
  const int n = std::atoi(argv[1]), thrower = std::atoi(argv[3]);
  g_allowed = std::atoi(argv[2]);
  std::vector<int> done(n, 0);
  bool thrown = false;
  try {
    cgs::run_shares(n, [&](int t) {
      done[t]++;
      if (t == thrower) throw std::bad_alloc();
    });
  } catch (const std::bad_alloc&) {
    thrown = true;
  }
  int once = 0;
  for (int v : done) once += v == 1;
  std::printf("%d %d\n", once, thrown ? 1 : 0);
  return 0;
}
