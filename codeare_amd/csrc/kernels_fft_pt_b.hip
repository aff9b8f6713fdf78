// kernels_fft_pt_b.hip -- k_fft_pt at n = 162, 192, 216, 243, 256, 288
// (the lengths are spread over several files, which compile in parallel)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels_fft_pt.hpp"

namespace cgs {

bool launch_fft_pt_b(const FftArgs& a, int ld_mode, int st_mode, hipStream_t s) {
  switch (a.n) {
    case 162: launch_pt<9, 18>(a, ld_mode, st_mode, s); return true;
    case 192: launch_pt<12, 16>(a, ld_mode, st_mode, s); return true;
    case 216: launch_pt<12, 18>(a, ld_mode, st_mode, s); return true;
    case 243: launch_pt<9, 27>(a, ld_mode, st_mode, s); return true;
    case 256: launch_pt<16, 16>(a, ld_mode, st_mode, s); return true;
    case 288: launch_pt<16, 18>(a, ld_mode, st_mode, s); return true;
    default: return false;
  }
}

}  // namespace cgs
