// FFT passes in modes that no kernel has: an error code, not a launch left out.  Nothing
// here reaches a GPU (no kernel matches).
#include <cstdio>

#include "../../codeare_amd/csrc/cgs_internal.hpp"

int main() {
  int wrong = 0;
  const float spectrum = 0.f;
  for (int kernel = 0; kernel < 3; ++kernel)
    for (int n : {36, 81, 128, 192, 256, 384, 432, 512, 576, 648}) {
      cgs::FftArgs a{};
      a.n = n;
      a.nin = a.nout = n;
      a.inner = 16;
      a.outers = a.outer_per_frame = 1;
      a.lb = 16;
      a.lines_log2 = 4;
      a.use_pt = kernel == 1;
      a.use_reg = kernel == 2;
      auto refused = [&](int ld, int st, int sign, const float* That) {
        a.sign = sign;
        a.That = That;
        if (cgs::launch_fft(a, ld, st, nullptr) == CGS_ERR_UNSUPPORTED) return;
        std::printf("kernel %d n %d load %d store %d sign %d conv %d\n", kernel, n, ld, st, sign, That != nullptr);
        ++wrong;
      };
      refused(5, 0, -1, nullptr);
      refused(0, 3, 1, nullptr);
      refused(1, 1, -1, nullptr);
      if (kernel == 1) {
        refused(0, 1, -1, nullptr);
        refused(4, 0, 1, nullptr);
        refused(0, 0, 1, &spectrum);
      }
      if (kernel != 2) refused(1, 0, -1, &spectrum);
    }
  return wrong != 0;
}
