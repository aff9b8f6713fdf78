// kernels_fft_pt_b.hip -- k_fft_pt at n = 162, 192, 216, 243, 256, 288
// (the lengths are spread over several files, which compile in parallel)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels_fft_pt.hpp"

namespace cgs {

bool launch_fft_pt_b(const FftArgs& a, int ld_mode, int st_mode, hipStream_t s) {
  switch (a.n) {
    case 162: return launch_pt<9, 18>(a, ld_mode, st_mode, s);
    case 192: return launch_pt<12, 16>(a, ld_mode, st_mode, s);
    case 216: return launch_pt<12, 18>(a, ld_mode, st_mode, s);
    case 243: return launch_pt<9, 27>(a, ld_mode, st_mode, s);
    case 256: return launch_pt<16, 16>(a, ld_mode, st_mode, s);
    case 288: return launch_pt<16, 18>(a, ld_mode, st_mode, s);
    default: return false;
  }
}

}  // namespace cgs
