// kernels_fft_pt.hpp -- register-resident FFT passes for lines of n = P T points.
//
// Same job and arguments as k_fft (kernels_fft.hip): a pass views the array as
// [outer][n][inner] with inner contiguous and transforms the n-point lines.  A
// block takes 16 lines; T threads share a line and thread j holds its points
// j + T k, k < P <= T, in registers.  With positions p = j + T k
//   X[k1 + P k2] = sum_j W_T^(j k2) W_n^(j k1) [ sum_k x[j + T k] W_P^(k k1) ]
// so a pass is a P-point DFT in registers, a twiddle, ONE exchange through LDS
// and a T-point DFT on the first P threads of each line; the Toeplitz
// convolution multiplies the spectrum in that layout and runs the same steps
// backwards.
//
// What bounds a pass is the array's trip through memory, so the layout serves
// the loads and stores: the 16 lines are 16 consecutive inner indices (128
// contiguous bytes per access), or, where the inner extent is below 16 (the
// axis-0 passes with fewer than 16 coils), the inner indices of several
// consecutive rows, each padded to the next power of two, so that a wave's
// lanes stay busy; all P loads of a thread are in flight together; the zero pad,
// the crop and idle lanes are vector offsets past the buffer's range (no
// branch, no memory traffic).
//
// Measured against the kernels these lengths had before: 432- and 324-point
// lines of 12 coils 22.4 -> 8.8 us a pass (LDS kernel, every stage through
// LDS); the 96^3 x 8 coil Toeplitz iteration (192 points): convolution 340 ->
// 129 us (3.7 TB/s), middle axis 84 -> 64, pad 89 -> 44, crop 98 -> 46; 192-point
// lines of 16 coils in 3D 339 -> 235 us; 256-point lines of 8 coils 12 -> 7 us;
// convolutions of 20 coils against 16 threads a line: 256 points 9.4 -> 9.0, 512
// points 25.9 -> 21.2 us (16 frames 305 -> 270).  One and two coils on few rows go to
// the LDS kernel (fft_few_rows, plan.hip).
#pragma once

#include "cgs_internal.hpp"
#include "dft_reg.hpp"

namespace cgs {

namespace {

// sum over the block's 16 T threads (every thread calls it); rows of 16 lanes
// first, since the last wave may be partly filled
template <int T>
__device__ __forceinline__ double pt_block_sum(double v, double* red) {
  v += dpp_mov_d<0xB1>(v);
  v += dpp_mov_d<0x4E>(v);
  v += dpp_mov_d<0x141>(v);
  v += dpp_mov_d<0x140>(v);
  lds_barrier();
  if ((threadIdx.x & 15) == 0) red[threadIdx.x >> 4] = v;
  lds_barrier();
  double t = 0.0;
#pragma unroll
  for (int w = 0; w < T; ++w) t += red[w];
  return t;
}

template <int CTRL>
__device__ __forceinline__ float2 pt_add2(float2 v) {
  return make_float2(v.x + dpp_mov<CTRL>(v.x), v.y + dpp_mov<CTRL>(v.y));
}

// LD: 0 array; 1 x S_c dinv; 2 array dinv; 3 array dinv inside the mask; 4 x S_c
// ST: 0 array; 1 array dinv; 2 sum over the block's coils of conj(S_c) X_c
// SG: sign of the kernel's exponent; CONV: forward, times That, inverse
template <int P, int T, int LD, int ST, int CONV, int SG>
__global__ void __launch_bounds__(16 * T) k_fft_pt(FftArgs a) {
  static_assert(P <= T, "one row per thread after the exchange");
  constexpr int n = P * T, NT = 16 * T;
  constexpr int XS = 16 * T + 8;   // exchange row (float2): T columns x 16 lines + pad
  __shared__ float2 ex[P * XS];
  __shared__ float2 twT[n];        // [j][k1] = exp(SG 2 pi i j k1 / n)
  __shared__ double red[T];
  const int tid = threadIdx.x;
  const int q = tid & 15, j = tid >> 4;
  // lines: coil group g of one row, or R rows of `inner` lines each
  const int lg = a.lines_log2, R = 16 >> lg;
  const int nib = (int)((a.inner + 15) / 16);
  const int64_t o0 = (int64_t)(blockIdx.x / (unsigned)nib) * R;
  const int g = (int)(blockIdx.x % (unsigned)nib);
  const int64_t q0 = (int64_t)g * 16;
  const int dr = q >> lg, cl = q & ((1 << lg) - 1);   // row and inner index within the block
  const int64_t opf = a.outer_per_frame;
  const int64_t f0 = o0 / opf;
  int64_t f = f0;
  if (R > 1) {
    int64_t ol = o0 + R - 1;
    if (ol >= a.outers) ol = a.outers - 1;
    if (a.fdone && a.fdone[f0] && ol / opf == f0) return;   // block-uniform
    f = (o0 + dr) / opf;
  } else if (a.fdone && a.fdone[f0]) {
    return;
  }
  bool live = q0 + cl < a.inner && o0 + dr < a.outers;
  if (R > 1 && live && a.fdone && a.fdone[f]) live = false;
  const int64_t rest0 = o0 - f0 * opf, rest = o0 + dr - f * opf;

  // window factor of the other axes and the mask's row term
  float dvr = 1.f;
  int msk = 0;
  if (LD == 1 || LD == 2 || LD == 3 || ST == 1) {
    const int rr = live ? (int)rest : 0, i1 = rr % a.N1, i2 = rr / a.N1;
    dvr = a.dinv1[i1];
    if (a.d == 3) dvr *= a.dinv2[i2];
    if (LD == 3) msk = (i1 - a.mask_nh) * (i1 - a.mask_nh) + (a.d == 3 ? (i2 - a.mask_nh) * (i2 - a.mask_nh) : 0);
  }
  const Rsrc rdv = rsrc(a.dinv0, (int64_t)a.N0 * 4);

  // maps of the block's rows (image index p: + p C)
  // (frame maps lie one after the other: rows of several frames are adjacent)
  const int64_t nc = (int64_t)a.N0 * a.C;
  const int64_t sb = R > 1 ? (a.Sfs ? o0 * nc : 0) : a.Sfs * f0 + nc * rest0 + q0;
  const Rsrc rS = rsrc((LD == 1 || LD == 4 || ST == 2) ? a.S + sb : nullptr, kOutOfRange - 16);
  const int vS = (R > 1 ? (int)((a.Sfs ? dr : rest) * nc) + cl : cl) * 8;

  // ---- load positions j + T k (image index p with the zero pad) ----
  float2 v[P];
  {
    const int in8 = (int)(a.inner * 8);
    const Rsrc ri = rsrc((LD == 1 || LD == 4) ? nullptr : a.in + o0 * a.nin * a.inner + q0, kOutOfRange - 16);
    const int vb = (dr * a.nin) * in8 + cl * 8;
    const int sh = a.pad_in ? a.nin / 2 : 0;
    int pk[P];
#pragma unroll
    for (int k = 0; k < P; ++k) {
      int p = j + T * k + sh;
      if (p >= n) p -= n;
      pk[k] = (live && p < a.nin) ? p : -1;
    }
    if (LD == 1 || LD == 4) {
#pragma unroll
      for (int k = 0; k < P; ++k) v[k] = bld2(rS, pk[k] >= 0 ? vS + pk[k] * a.C * 8 : kOutOfRange, 0);
      const int vx = dr * a.N0;
      const int64_t xb = o0 * a.N0;
      if (a.pold) {   // p_new = r + beta p_old (CGLS.hpp:55-56), fused
        const Rsrc rr = rsrc(a.r + xb, kOutOfRange - 16), rp = rsrc(a.pold + xb, kOutOfRange - 16);
        const Rsrc rn = rsrc(a.pnew + xb, kOutOfRange - 16);
        const float be = live ? (float)a.cgst[f].beta : 0.f;
        const bool c0 = q0 + cl == 0;
        float2 rv[P], pv[P];
#pragma unroll
        for (int k = 0; k < P; ++k) {
          const int vo = pk[k] >= 0 ? (vx + pk[k]) * 8 : kOutOfRange;
          rv[k] = bld2(rr, vo, 0);
          pv[k] = bld2(rp, vo, 0);
        }
        float pp = 0.f;   // ||p_new||^2 over this row
#pragma unroll
        for (int k = 0; k < P; ++k) {
          const float2 x = make_float2(rv[k].x + be * pv[k].x, rv[k].y + be * pv[k].y);
          bst2(rn, x, c0 && pk[k] >= 0 ? (vx + pk[k]) * 8 : kOutOfRange, 0);
          if (c0) pp += x.x * x.x + x.y * x.y;
          v[k] = cmul(x, v[k]);
        }
        if (a.pp_part && q0 == 0) {   // block-uniform; R == 1
          const double t = pt_block_sum<T>(pp, red);
          if (tid == 0) a.pp_part[o0] = t;
        }
      } else {
        const Rsrc rx = rsrc(a.x + xb, kOutOfRange - 16);
#pragma unroll
        for (int k = 0; k < P; ++k) v[k] = cmul(bld2(rx, pk[k] >= 0 ? (vx + pk[k]) * 8 : kOutOfRange, 0), v[k]);
      }
    } else {
#pragma unroll
      for (int k = 0; k < P; ++k) v[k] = bld2(ri, pk[k] >= 0 ? vb + pk[k] * in8 : kOutOfRange, 0);
    }
    if (LD >= 1 && LD <= 3) {
#pragma unroll
      for (int k = 0; k < P; ++k) {
        float dv = dvr * bld1(rdv, pk[k] >= 0 ? pk[k] * 4 : kOutOfRange, 0);
        if (LD == 3) {
          const int e = pk[k] - a.mask_nh;
          if (e * e + msk > a.mask_nh * a.mask_nh) dv = 0.f;
        }
        v[k] = make_float2(v[k].x * dv, v[k].y * dv);
      }
    }
  }
  // the small tables are asked for after the points, the window factors of the last
  // pass with them: one round trip for all (256-point lines of 8 coils, last pass
  // 7.6 -> 6.1 us; the 96^3 x 8 coil convolution 135 -> 129 us)
  constexpr int NU = (n + NT - 1) / NT;
  float2 wt[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) {
    const int e = min(tid + u * NT, n - 1);
    wt[u] = a.tw[(e / P) * (e % P)];
  }
  float dvo[ST == 1 ? T : 1];
  if constexpr (ST == 1) {
    const int so1 = a.crop_out ? a.nout / 2 : 0;
#pragma unroll
    for (int k2 = 0; k2 < T; ++k2) {
      int p = j + P * k2 + so1;
      if (p >= n) p -= n;
      dvo[k2] = bld1(rdv, live && p < a.nout ? p * 4 : kOutOfRange, 0);
    }
  }
#pragma unroll
  for (int u = 0; u < NU; ++u)
    if (tid + u * NT < n) twT[tid + u * NT] = SG < 0 ? wt[u] : make_float2(wt[u].x, -wt[u].y);
  lds_barrier();   // twiddle table

  // ---- P-point DFT over k, twiddle, exchange, T-point DFT of row j ----
  dft<P, SG>(v);
#pragma unroll
  for (int k1 = 0; k1 < P; ++k1) {
    if (k1) v[k1] = cmul(v[k1], twT[j * P + k1]);
    ex[k1 * XS + j * 16 + q] = v[k1];
  }
  lds_barrier();
  const bool act = P == T || j < P;
  float2 X[T];
  if (act) {
#pragma unroll
    for (int jj = 0; jj < T; ++jj) X[jj] = ex[j * XS + jj * 16 + q];
    dft<T, SG>(X);   // bins j + P k2
  }
  const int in8 = (int)(a.inner * 8);
  const int so = a.crop_out ? a.nout / 2 : 0;

  if (CONV) {
    if (act) {
      const int64_t cell = live ? f * a.conv_cells + (q0 + cl) / a.C : 0;
      const float* th = a.That + cell * n + j;
      float t[T];
#pragma unroll
      for (int k2 = 0; k2 < T; ++k2) t[k2] = th[P * k2];
#pragma unroll
      for (int k2 = 0; k2 < T; ++k2) X[k2] = make_float2(X[k2].x * t[k2], X[k2].y * t[k2]);
      dft<T, -SG>(X);   // over k2 -> column
#pragma unroll
      for (int jj = 0; jj < T; ++jj) ex[j * XS + jj * 16 + q] = cmulc(X[jj], twT[jj * P + j]);   // its own row
    }
    lds_barrier();
#pragma unroll
    for (int k1 = 0; k1 < P; ++k1) v[k1] = ex[k1 * XS + j * 16 + q];
    dft<P, -SG>(v);   // position j + T k
    const Rsrc ro = rsrc(a.out + o0 * a.nout * a.inner + q0, kOutOfRange - 16);
    const int vb = (dr * a.nout) * in8 + cl * 8;
#pragma unroll
    for (int k = 0; k < P; ++k) {
      int p = j + T * k + so;
      if (p >= n) p -= n;
      bst2(ro, v[k], live && p < a.nout ? vb + p * in8 : kOutOfRange, 0);
    }
    return;
  }

  if (ST == 2) {   // G = nib partial images
    const int64_t ob = (f0 * nib + g) * a.Ntot + (int64_t)a.N0 * rest0;   // R > 1: nib == 1, rows adjacent
    const Rsrc ro = rsrc(a.out + ob, kOutOfRange - 16);
    const Rsrc rd = rsrc(a.pdot ? a.pdot + o0 * a.N0 : a.out, a.pdot ? (int64_t)a.N0 * 8 : 0);
    double pq = 0.0;
    if (act) {
      int pk[T];
      float2 sv[T];
#pragma unroll
      for (int k2 = 0; k2 < T; ++k2) {
        int p = j + P * k2 + so;
        if (p >= n) p -= n;
        pk[k2] = live && p < a.nout ? p : -1;
        sv[k2] = bld2(rS, pk[k2] >= 0 ? vS + pk[k2] * a.C * 8 : kOutOfRange, 0);
      }
#pragma unroll
      for (int k2 = 0; k2 < T; ++k2) X[k2] = cmulc(X[k2], sv[k2]);
      // over the row's coils (the map is zero on idle lanes)
      if (lg >= 1) {
#pragma unroll
        for (int k2 = 0; k2 < T; ++k2) X[k2] = pt_add2<0xB1>(X[k2]);
      }
      if (lg >= 2) {
#pragma unroll
        for (int k2 = 0; k2 < T; ++k2) X[k2] = pt_add2<0x4E>(X[k2]);
      }
      if (lg >= 3) {
#pragma unroll
        for (int k2 = 0; k2 < T; ++k2) X[k2] = pt_add2<0x141>(X[k2]);
      }
      if (lg >= 4) {
#pragma unroll
        for (int k2 = 0; k2 < T; ++k2) X[k2] = pt_add2<0x140>(X[k2]);
      }
#pragma unroll
      for (int k2 = 0; k2 < T; ++k2) {
        const bool st = cl == 0 && pk[k2] >= 0;
        bst2(ro, X[k2], st ? (dr * a.N0 + pk[k2]) * 8 : kOutOfRange, 0);
        const float2 pv = bld2(rd, st ? pk[k2] * 8 : kOutOfRange, 0);
        pq += (double)pv.x * X[k2].x + (double)pv.y * X[k2].y;
      }
    }
    if (a.pq_part) {   // block-uniform; R == 1
      const double t = pt_block_sum<T>(pq, red);
      if (tid == 0) a.pq_part[(f0 * nib + g) * opf + rest0] = t;
    }
    return;
  }

  if (act) {
    const Rsrc ro = rsrc(a.out + o0 * a.nout * a.inner + q0, kOutOfRange - 16);
    const int vb = (dr * a.nout) * in8 + cl * 8;
#pragma unroll
    for (int k2 = 0; k2 < T; ++k2) {
      int p = j + P * k2 + so;
      if (p >= n) p -= n;
      const int vo = live && p < a.nout ? vb + p * in8 : kOutOfRange;
      if (ST == 1) {
        const float dv = dvr * dvo[k2];
        X[k2] = make_float2(X[k2].x * dv, X[k2].y * dv);
      }
      bst2(ro, X[k2], vo, 0);
    }
  }
}

}  // namespace

template <int P, int T>
static bool launch_pt(const FftArgs& a, int ld, int st, hipStream_t s) {   // false: no such kernel
  const int R = 16 >> a.lines_log2;
  const dim3 grid((unsigned)((a.outers + R - 1) / R * ((a.inner + 15) / 16)));
  const int conv = a.That != nullptr;
#define CGS_PT_CASE(L, S_, CV, SG_)                                                                  \
  if (ld == L && st == S_ && conv == CV && a.sign == SG_) {                                          \
    CGS_LAUNCH((k_fft_pt<P, T, L, S_, CV, SG_>), grid, dim3(16 * T), 0, s, a);                        \
    return true;                                                                                        \
  }
  CGS_PT_CASE(0, 0, 0, -1)
  CGS_PT_CASE(0, 0, 0, 1)
  CGS_PT_CASE(1, 0, 0, -1)
  CGS_PT_CASE(2, 0, 0, -1)
  CGS_PT_CASE(3, 0, 0, -1)
  CGS_PT_CASE(4, 0, 0, -1)
  CGS_PT_CASE(0, 1, 0, 1)
  CGS_PT_CASE(0, 0, 1, -1)
  CGS_PT_CASE(0, 2, 0, 1)
#undef CGS_PT_CASE
  return false;
}

}  // namespace cgs
