// dft_reg.hpp -- what the register-resident FFT kernels share: raw buffer
// access, complex products and DFTs of compile-time length held in registers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "fft_roots.hpp"

namespace cgs {

namespace {

typedef __amdgpu_buffer_rsrc_t Rsrc;
typedef unsigned int u32x2 __attribute__((__vector_size__(2 * sizeof(unsigned int))));

// raw buffer descriptor over [base, base + bytes); word 3 = 0x00020000 selects
// the 32-bit data format of the gfx9 buffer unit
__device__ __forceinline__ Rsrc rsrc(const void* base, int64_t bytes) {
  const int nr = bytes > 0x7fffffff ? 0x7fffffff : (int)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, nr, 0x00020000);
}
__device__ __forceinline__ float2 bld2(Rsrc r, int voff, int soff) {
  return __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
}
__device__ __forceinline__ float bld1(Rsrc r, int voff, int soff) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}
__device__ __forceinline__ void bst2(Rsrc r, float2 v, int voff, int soff) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, 0);
}

__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cmulc(float2 a, float2 b) {   // a * conj(b)
  return make_float2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}

// a * exp(SG 2 pi i t / L); t is a compile-time constant after unrolling, so
// the tests fold and 1, -1, +-i cost no multiplies
template <int L, int SG>
__device__ __forceinline__ float2 rot(float2 a, int t) {
  t %= L;
  if (t == 0) return a;
  if (2 * t == L) return make_float2(-a.x, -a.y);
  if (4 * t == L) return SG > 0 ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
  if (4 * t == 3 * L) return SG > 0 ? make_float2(a.y, -a.x) : make_float2(-a.y, a.x);
  const float c = kTwL<L>.c[t];
  const float s = SG < 0 ? kTwL<L>.s[t] : -kTwL<L>.s[t];
  return make_float2(a.x * c - a.y * s, a.x * s + a.y * c);
}

// one Stockham radix-R stage (R = 2, 3 or 4), span Ns, of an N-point DFT with
// kernel exp(SG 2 pi i / N); natural order after the last stage
template <int N, int Ns, int R, int SG>
__device__ __forceinline__ void stg(const float2 (&in)[N], float2 (&out)[N]) {
#pragma unroll
  for (int jj = 0; jj < N / R; ++jj) {
    const int k = jj % Ns;
    float2 a[R];
#pragma unroll
    for (int m = 0; m < R; ++m) a[m] = in[jj + m * (N / R)];
#pragma unroll
    for (int m = 1; m < R; ++m) a[m] = rot<Ns * R, SG>(a[m], m * k);
    if constexpr (R == 2) {
      const float2 b0 = make_float2(a[0].x + a[1].x, a[0].y + a[1].y);
      const float2 b1 = make_float2(a[0].x - a[1].x, a[0].y - a[1].y);
      a[0] = b0;
      a[1] = b1;
    } else if constexpr (R == 3) {
      // w = exp(SG 2 pi i / 3) = -1/2 + SG i sqrt(3)/2
      constexpr float h = 0.86602540378443864676f * (float)SG;
      const float2 t1 = make_float2(a[1].x + a[2].x, a[1].y + a[2].y);
      const float2 t2 = make_float2(a[1].x - a[2].x, a[1].y - a[2].y);
      const float2 mm = make_float2(a[0].x - 0.5f * t1.x, a[0].y - 0.5f * t1.y);
      a[0] = make_float2(a[0].x + t1.x, a[0].y + t1.y);
      a[1] = make_float2(mm.x - h * t2.y, mm.y + h * t2.x);   // mm + (i h) t2
      a[2] = make_float2(mm.x + h * t2.y, mm.y - h * t2.x);
    } else {
      const float2 t0 = make_float2(a[0].x + a[2].x, a[0].y + a[2].y);
      const float2 t1 = make_float2(a[0].x - a[2].x, a[0].y - a[2].y);
      const float2 t2 = make_float2(a[1].x + a[3].x, a[1].y + a[3].y);
      const float2 t3 = make_float2(a[1].x - a[3].x, a[1].y - a[3].y);
      const float2 u3 = SG > 0 ? make_float2(-t3.y, t3.x) : make_float2(t3.y, -t3.x);   // (SG i) t3
      a[0] = make_float2(t0.x + t2.x, t0.y + t2.y);
      a[2] = make_float2(t0.x - t2.x, t0.y - t2.y);
      a[1] = make_float2(t1.x + u3.x, t1.y + u3.y);
      a[3] = make_float2(t1.x - u3.x, t1.y - u3.y);
    }
    const int base = (jj / Ns) * Ns * R + k;
#pragma unroll
    for (int m = 0; m < R; ++m) out[base + m * Ns] = a[m];
  }
}

// in-place N-point DFT in registers, natural order in and out
template <int N, int SG>
__device__ __forceinline__ void dft(float2 (&v)[N]) {
  float2 t[N];
  if constexpr (N == 2) {
    stg<2, 1, 2, SG>(v, t);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = t[i];
  } else if constexpr (N == 3) {
    stg<3, 1, 3, SG>(v, t);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = t[i];
  } else if constexpr (N == 6) {
    stg<6, 1, 2, SG>(v, t);
    stg<6, 2, 3, SG>(t, v);
  } else if constexpr (N == 12) {
    stg<12, 1, 4, SG>(v, t);
    stg<12, 4, 3, SG>(t, v);
  } else if constexpr (N == 4) {
    stg<4, 1, 4, SG>(v, t);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = t[i];
  } else if constexpr (N == 8) {
    stg<8, 1, 2, SG>(v, t);
    stg<8, 2, 4, SG>(t, v);
  } else if constexpr (N == 16) {
    stg<16, 1, 4, SG>(v, t);
    stg<16, 4, 4, SG>(t, v);
  } else if constexpr (N == 9) {
    stg<9, 1, 3, SG>(v, t);
    stg<9, 3, 3, SG>(t, v);
  } else if constexpr (N == 18) {
    stg<18, 1, 2, SG>(v, t);
    stg<18, 2, 3, SG>(t, v);
    stg<18, 6, 3, SG>(v, t);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = t[i];
  } else if constexpr (N == 24) {
    stg<24, 1, 4, SG>(v, t);
    stg<24, 4, 2, SG>(t, v);
    stg<24, 8, 3, SG>(v, t);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = t[i];
  } else if constexpr (N == 27) {
    stg<27, 1, 3, SG>(v, t);
    stg<27, 3, 3, SG>(t, v);
    stg<27, 9, 3, SG>(v, t);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = t[i];
  } else {
    static_assert(N == 32, "DFT length");
    stg<32, 1, 4, SG>(v, t);
    stg<32, 4, 4, SG>(t, v);
    stg<32, 16, 2, SG>(v, t);
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = t[i];
  }
}

// P-point DFT of v[0 .. P/2) (upper half zero): X[2r] = DFT_{P/2}(v)[r],
// X[2r+1] = DFT_{P/2}(v_k w^k)[r], w = exp(SG 2 pi i / P); all P bins on exit
template <int P, int SG>
__device__ __forceinline__ void dft_zero_top(float2 (&v)[P]) {
  constexpr int H = P / 2;
  float2 e[H], o[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    e[k] = v[k];
    o[k] = rot<P, SG>(v[k], k);
  }
  dft<H, SG>(e);
  dft<H, SG>(o);
#pragma unroll
  for (int r = 0; r < H; ++r) {
    v[2 * r] = e[r];
    v[2 * r + 1] = o[r];
  }
}

// the first P/2 outputs of a P-point DFT: x[k] = E[k] + w^k O[k] with E, O
// the P/2-point DFTs of the even and odd inputs; v[0 .. P/2) on exit
template <int P, int SG>
__device__ __forceinline__ void dft_low_half(float2 (&v)[P]) {
  constexpr int H = P / 2;
  float2 e[H], o[H];
#pragma unroll
  for (int r = 0; r < H; ++r) {
    e[r] = v[2 * r];
    o[r] = v[2 * r + 1];
  }
  dft<H, SG>(e);
  dft<H, SG>(o);
#pragma unroll
  for (int k = 0; k < H; ++k) {
    const float2 t = rot<P, SG>(o[k], k);
    v[k] = make_float2(e[k].x + t.x, e[k].y + t.y);
  }
}

constexpr int kOutOfRange = 0x7ffffff0;   // a vector offset past every buffer's range

}  // namespace

}  // namespace cgs
