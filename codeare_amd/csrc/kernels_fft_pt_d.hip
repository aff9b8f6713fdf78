// kernels_fft_pt_d.hip -- k_fft_pt at n = 512, 576, 648
// (the lengths are spread over several files, which compile in parallel)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels_fft_pt.hpp"

namespace cgs {

bool launch_fft_pt_d(const FftArgs& a, int ld_mode, int st_mode, hipStream_t s) {
  switch (a.n) {
    case 512: return launch_pt<16, 32>(a, ld_mode, st_mode, s);
    case 576: return launch_pt<24, 24>(a, ld_mode, st_mode, s);
    case 648: return launch_pt<24, 27>(a, ld_mode, st_mode, s);
    default: return false;
  }
}

}  // namespace cgs
