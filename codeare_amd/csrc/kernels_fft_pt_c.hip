// kernels_fft_pt_c.hip -- k_fft_pt at n = 324, 384, 432, 486
// (the lengths are spread over several files, which compile in parallel)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels_fft_pt.hpp"

namespace cgs {

bool launch_fft_pt_c(const FftArgs& a, int ld_mode, int st_mode, hipStream_t s) {
  switch (a.n) {
    case 324: return launch_pt<18, 18>(a, ld_mode, st_mode, s);
    case 384: return launch_pt<16, 24>(a, ld_mode, st_mode, s);
    case 432: return launch_pt<18, 24>(a, ld_mode, st_mode, s);
    case 486: return launch_pt<18, 27>(a, ld_mode, st_mode, s);
    default: return false;
  }
}

}  // namespace cgs
