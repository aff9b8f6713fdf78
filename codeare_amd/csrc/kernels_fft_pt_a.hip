// kernels_fft_pt_a.hip -- k_fft_pt at n = 36, 48, 54, 64, 72, 81, 96, 108, 128, 144
// (the lengths are spread over several files, which compile in parallel)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels_fft_pt.hpp"

namespace cgs {

bool launch_fft_pt_b(const FftArgs& a, int ld_mode, int st_mode, hipStream_t s);
bool launch_fft_pt_c(const FftArgs& a, int ld_mode, int st_mode, hipStream_t s);
bool launch_fft_pt_d(const FftArgs& a, int ld_mode, int st_mode, hipStream_t s);

// the lengths below, where every offset from a block's first row fits 31 bits
bool fft_pt_supported(const FftArgs& a) {
  switch (a.n) {
    case 36: case 48: case 54: case 64: case 72: case 81: case 96: case 108:
    case 128: case 144: case 162: case 192: case 216: case 243: case 256: case 288:
    case 324: case 384: case 432: case 486: case 512: case 576: case 648:
      break;
    default: return false;
  }
  const int64_t lim = kOutOfRange - 64, R = 16 >> a.lines_log2;
  if (R * std::max(a.nin, a.nout) * a.inner * 8 >= lim) return false;
  const int64_t maps = (R == 1 ? (int64_t)a.N0 : a.Sfs ? R * a.N0 : a.Ntot) * a.C * 8;
  return maps < lim && R * a.N0 * 8 < lim;
}

bool launch_fft_pt(const FftArgs& a, int ld_mode, int st_mode, hipStream_t s) {
  switch (a.n) {
    case 36: return launch_pt<6, 6>(a, ld_mode, st_mode, s);
    case 48: return launch_pt<6, 8>(a, ld_mode, st_mode, s);
    case 54: return launch_pt<6, 9>(a, ld_mode, st_mode, s);
    case 64: return launch_pt<8, 8>(a, ld_mode, st_mode, s);
    case 72: return launch_pt<8, 9>(a, ld_mode, st_mode, s);
    case 81: return launch_pt<9, 9>(a, ld_mode, st_mode, s);
    case 96: return launch_pt<8, 12>(a, ld_mode, st_mode, s);
    case 108: return launch_pt<9, 12>(a, ld_mode, st_mode, s);
    case 128: return launch_pt<8, 16>(a, ld_mode, st_mode, s);
    case 144: return launch_pt<12, 12>(a, ld_mode, st_mode, s);
    default: break;
  }
  return launch_fft_pt_b(a, ld_mode, st_mode, s) || launch_fft_pt_c(a, ld_mode, st_mode, s) ||
         launch_fft_pt_d(a, ld_mode, st_mode, s);
}

}  // namespace cgs
