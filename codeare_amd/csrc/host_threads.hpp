// host_threads.hpp -- host loops in shares on several threads, for code behind the C ABI:
// nothing leaves a thread as an exception, and no thread is left joinable.
#pragma once

#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace cgs {

// fn(t) for t = 0 .. n - 1, each on its own thread (t = 0 on the caller's).  Where a
// thread cannot be started the caller takes its share; what a share throws is thrown
// here once all have ended (the first of several).
template <class Fn>
void run_shares(int n, Fn&& fn) {
  std::mutex mu;
  std::exception_ptr err;
  auto share = [&](int t) noexcept {
    try {
      fn(t);
    } catch (...) {
      std::lock_guard<std::mutex> lk(mu);
      if (!err) err = std::current_exception();
    }
  };
  std::vector<std::thread> th;
  th.reserve(n > 0 ? n : 0);
  int t = 1;
  try {
    for (; t < n; ++t) th.emplace_back(share, t);
  } catch (...) {   // out of threads or memory: shares t .. n - 1 stay here
  }
  if (n > 0) share(0);
  for (; t < n; ++t) share(t);
  for (auto& x : th) x.join();
  if (err) std::rethrow_exception(err);
}

}  // namespace cgs
