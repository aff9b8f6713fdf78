// unet.hip -- the learned CG warm start: a 2D U-Net (3x3 convolutions, ReLU,
// 2x2 max-pool down, nearest 2x up + skip concatenation) trained and run with
// hand-written BF16 MFMA kernels (v_mfma_f32_32x32x16_bf16, FP32 accumulate).
//
// Tensors are NHWC: activation[((b*H + y)*W + x)*C + c], BF16 storage.  The
// network input and output are complex64 images, i.e. NHWC with C = 2
// (re, im).  Conv weights are kept as FP32 masters [tap][co][ci] (tap = 3*ky+kx)
// with BF16 copies in the order the matrix instructions take them (k_wprep): one of
// the weights for the forward pass, one of the flipped, transposed weights
// W'[8-tap][ci][co] for the input-gradient pass, which is then the same convolution
// kernel (none for the first layer: nothing takes its input's gradient).  Every reduction (weight and bias gradients, loss) runs in
// a fixed order, so a training step is deterministic.
//
// There is no counterpart in codeare: the network supplies x0 for the CG solve
// (NCSENSE::Adjoint -> CGLS::Solve, src/optimisation/CGLS.hpp:30-59, starts
// from zero).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/cgs_unet.h"
#include "../../include/cgsense.h"

namespace cgs {
void set_error(const std::string& m);
}

namespace {

using bf16 = uint16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float bf2f(bf16 h) { return __uint_as_float((uint32_t)h << 16); }
__host__ __device__ inline bf16 f2bf(float f) {
  uint32_t u;
#ifdef __HIP_DEVICE_COMPILE__
  u = __float_as_uint(f);
#else
  std::memcpy(&u, &f, 4);
#endif
  if ((u & 0x7f800000u) == 0x7f800000u) return (bf16)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));  // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (bf16)(u >> 16);
}

__device__ __forceinline__ bf16x8 as_bf8(uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// ----------------------------------------------------------------------------
// 3x3 convolution, stride 1, zero padding 1, as an implicit GEMM on MFMA.
// Input channels [0, Ca) come from A (H x W), channels [Ca, Ca+Cb) from B at
// half resolution read through a nearest 2x upsampling (B may be absent).
// Output channels [0, split) go to out0 (channel stride `split`), optionally
// multiplied by (mask0 > 0) with mask0 laid out like out0; channels
// [split, Cout) go to out1 (stride Cout - split).  bias/relu: forward epilogue.
struct ConvArgs {
  const bf16* A;
  const bf16* B;
  const uint4* Wt;    // operand order, see k_wprep
  const float* bias;  // [Cout] or null
  bf16* out0;
  bf16* out1;
  const bf16* mask0;
  int Ca, Cb, Cout, split;
  int H, W, batch;
  int relu;
};

// Block: 4 waves; tile 8 PW x 16 pixels x 32 CW output channels; each wave owns
// PW 32-pixel rows of products (2 image rows of 16) x CW 32-channel columns.  K
// is walked in chunks of KC input channels (32; 16 for the packed network input),
// within a chunk over the 9 taps, then over steps of 16 channels: one order of
// sums for every tile shape.  Per chunk the input halo and the weights go through
// LDS; the next chunk's loads are in flight while the current one is multiplied.
// The weights come in operand order (k_wprep), so their staging is a linear copy
// and their reads are conflict-free; a halo position takes 80 bytes, which puts
// 16 neighbours on 16 different 16-byte banks.  Products are weights x pixels,
// D[channel][pixel]: a lane holds one pixel's channels in runs of four, and one
// swap of the wave's halves makes its stores 16 bytes.
//
// What bounds it: at a batch of 16 images of 256^2 the matrix work and, in the
// 32-channel level, the activations' traffic (665 TFLOP/s forward, 602 input
// gradient over the 14 layers; 219 with blocks that loaded a chunk, waited and
// multiplied, weights staged in rows and 2-byte stores); at one image the few
// blocks' walk over the chunks (14 layers 411 -> 110 us).
constexpr int kHaloStride = 40;   // halves per halo position (32 channels + 16 bytes)
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint32_t pack_bf2(float x, float y) {   // round to nearest even
  const f32x2 v = {x, y};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}
// barrier for data passed through LDS: does not wait for global loads in flight
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <int PW, int CW, int KC>
__global__ __launch_bounds__(256) void k_conv3x3(ConvArgs a) {
  constexpr int TR = 8 * PW, HP = (TR + 2) * 18, KS = KC / 16, G = KC / 8;
  constexpr int NH = (HP * G + 255) / 256;             // halo units (16 bytes) per thread
  constexpr int WU = 9 * KS * CW * 64;                 // weight units per chunk
  constexpr int NW = (WU + 255) / 256;
  __shared__ __attribute__((aligned(16))) bf16 hal[HP * kHaloStride];
  __shared__ u32x4 wl[WU];

  const int Cin = a.Ca + a.Cb, nct = a.Cout / 32;
  const int tiles_x = a.W / 16, tiles_y = a.H / TR;
  int t = blockIdx.x;
  const int tx0 = (t % tiles_x) * 16;
  t /= tiles_x;
  const int ty0 = (t % tiles_y) * TR;
  const int b = t / tiles_y;
  const int ct0 = blockIdx.y * CW;                     // first 32-channel tile of the block
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int row = lane & 31, kh = lane >> 5;
  const int Hh = a.H >> 1, Wh = a.W >> 1;

  // this thread's halo units: pixel index at full and at half resolution (0 where
  // outside the image: loaded and dropped)
  int pixA[NH], pixB[NH];
  unsigned inside = 0;
#pragma unroll
  for (int u = 0; u < NH; ++u) {
    const int pos = (u * 256 + tid) / G;
    const int hy = pos / 18, hx = pos - hy * 18;
    const int y = ty0 + hy - 1, x = tx0 + hx - 1;
    const bool ok = pos < HP && y >= 0 && y < a.H && x >= 0 && x < a.W;
    inside |= (unsigned)ok << u;
    pixA[u] = ok ? (b * a.H + y) * a.W + x : 0;
    pixB[u] = ok && a.Cb ? (b * Hh + (y >> 1)) * Wh + (x >> 1) : 0;
  }
  const int grp8 = (tid % G) * 8;                      // (256 is a multiple of G: the same for every unit)

  u32x4 hv[NH], wv[NW];
  auto load_chunk = [&](int c0) {
    const bool inA = c0 < a.Ca;
    const bf16* src = inA ? a.A + c0 + grp8 : a.B + (c0 - a.Ca) + grp8;
    const int st = inA ? a.Ca : a.Cb;
#pragma unroll
    for (int u = 0; u < NH; ++u)
      hv[u] = *reinterpret_cast<const u32x4*>(src + (size_t)(unsigned)(inA ? pixA[u] : pixB[u]) * (unsigned)st);
    // operand order: [step][channel tile][lane], step = (chunk * 9 + tap) * KS + ks
    const u32x4* ws = reinterpret_cast<const u32x4*>(a.Wt) + ((size_t)(c0 / KC) * 9 * KS * nct + ct0) * 64;
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const int idx = min(u * 256 + tid, WU - 1);
      wv[u] = ws[(size_t)(idx / (CW * 64)) * nct * 64 + idx % (CW * 64)];
    }
  };
  auto store_chunk = [&]() {
#pragma unroll
    for (int u = 0; u < NH; ++u) {
      const int pos = (u * 256 + tid) / G;
      const bool ok = (inside >> u) & 1u;
      const u32x4 v = ok ? hv[u] : u32x4{0, 0, 0, 0};
      if (pos < HP) *reinterpret_cast<u32x4*>(&hal[pos * kHaloStride + grp8]) = v;
    }
#pragma unroll
    for (int u = 0; u < NW; ++u)
      if (u * 256 + tid < WU) wl[u * 256 + tid] = wv[u];
  };

  f32x16 acc[PW][CW];
#pragma unroll
  for (int s = 0; s < PW; ++s)
#pragma unroll
    for (int c = 0; c < CW; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[s][c][r] = 0.f;
  const bf16* hp = hal + ((w * 2 * PW + (row >> 4)) * 18 + (row & 15)) * kHaloStride + kh * 8;

  load_chunk(0);
  for (int c0 = 0; c0 < Cin; c0 += KC) {
    if (c0) lds_sync();                                // the chunk before is consumed
    store_chunk();
    if (c0 + KC < Cin) load_chunk(c0 + KC);
    lds_sync();
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        bf16x8 wf[CW];
#pragma unroll
        for (int c = 0; c < CW; ++c) wf[c] = __builtin_bit_cast(bf16x8, wl[((tap * KS + ks) * CW + c) * 64 + lane]);
#pragma unroll
        for (int s = 0; s < PW; ++s) {
          const bf16x8 pf = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(
              hp + ((2 * s + tap / 3) * 18 + tap % 3) * kHaloStride + ks * 16));
#pragma unroll
          for (int c = 0; c < CW; ++c) acc[s][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[c], pf, acc[s][c], 0, 0, 0);
        }
      }
    }
  }

  // ---- epilogue: lane holds pixel `row`, register r channel 8 (r / 4) + 4 kh + r % 4
#pragma unroll
  for (int c = 0; c < CW; ++c) {
    const int co = (ct0 + c) * 32;
    const bool first = co < a.split;                   // (split is a multiple of 32)
    bf16* out = first ? a.out0 + co : a.out1 + (co - a.split);
    const bf16* mask = first && a.mask0 ? a.mask0 + co : nullptr;
    const int st = first ? a.split : a.Cout - a.split;
    float bias[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) bias[r] = a.bias ? a.bias[co + 8 * (r >> 2) + 4 * kh + (r & 3)] : 0.f;
#pragma unroll
    for (int s = 0; s < PW; ++s) {
      const int y = ty0 + w * 2 * PW + 2 * s + (row >> 4), x = tx0 + (row & 15);
      const size_t pix = (size_t)(b * a.H + y) * a.W + x;
      uint32_t d[4][2];                                // quad q: channels 8 q + 4 kh .. + 3
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = acc[s][c][4 * q + e] + bias[4 * q + e];
          if (a.relu) v[e] = fmaxf(v[e], 0.f);
        }
        d[q][0] = pack_bf2(v[0], v[1]);
        d[q][1] = pack_bf2(v[2], v[3]);
      }
      // halves of the wave swap: lanes 0..31 end with channels 0..15 of their
      // pixel, lanes 32..63 with channels 16..31
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        uint4 v;
        const auto s0 = __builtin_amdgcn_permlane32_swap(d[q][0], d[q + 2][0], false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(d[q][1], d[q + 2][1], false, false);
        v = make_uint4(s0[0], s1[0], s0[1], s1[1]);
        const int ch = 16 * kh + 8 * q;
        if (mask) {
          const uint4 m = *reinterpret_cast<const uint4*>(mask + pix * st + ch);
          auto keep = [](uint32_t x, uint32_t g) {     // halves of x where the bf16 halves of g are > 0
            const uint32_t lo = (int16_t)(g & 0xffffu) > 0 ? 0xffffu : 0u;
            const uint32_t hi = (int32_t)g >= 0x10000 ? 0xffff0000u : 0u;
            return x & (lo | hi);
          };
          v = make_uint4(keep(v.x, m.x), keep(v.y, m.y), keep(v.z, m.z), keep(v.w, m.w));
        }
        *reinterpret_cast<uint4*>(out + pix * st + ch) = v;
      }
    }
  }
}

// ----------------------------------------------------------------------------
// Weight gradient of the 3x3 convolution: dW[tap][co][ci] = sum over pixels of
// dY[p][co] * X[p + off(tap)][ci], X = the forward input (A | up(B)), and the bias
// gradient db[co] = sum over pixels of dY[p][co].  A GEMM whose K is the pixels:
// both operands are wanted with eight pixels of one channel in a lane, while the
// tensors are channel-fastest.  Tiles of dY and of X's halo go to LDS as they are
// (16-byte copies) and ds_read_b64_tr_b16 reads them transposed: of the 16 lanes of
// a row, lane i names 4 channels 4 (i % 4) of pixel i / 4 and receives 4 pixels of
// channel i.  A tap is then an address offset into the one halo.  The bias gradient
// is one more product, with ones.  Measured, all 14 layers of a batch of 16 images of
// 256^2 with the reductions: 454 TFLOP/s, 0.77 ms (scattering 2-byte values into
// transposed LDS copies, one per horizontal shift, and adding the partials one thread
// a value: 94 TFLOP/s, 3.7 ms, and 2.8 ms more for the biases).
//
// Block: 4 waves = WCO x WCI tiles of 32 x 32 channels, all 9 taps in registers, x WK
// parts of the pixel tile (TY x 16) summed through LDS at the end.  blockIdx.z takes
// a contiguous range of pixel tiles and writes partial sums part[z][9 Cout Cin +
// Cout] (a layer's weights then biases, as the parameters lie); k_reduce_splits adds
// the ranges in a fixed order.
struct WgradArgs {
  const bf16* dY;  // [B][H][W][Cout], gradient at the pre-activation
  const bf16* A;
  const bf16* B;
  float* part;
  int Ca, Cb, Cout, H, W, batch;
  int tiles_per_split, ntiles;
};

// 8 pixels of a channel: two transposed reads of 4, `p` + 4 pixels apart
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ bf16x8 read_tr8(const bf16* p, int four_pixels) {
  typedef __attribute__((address_space(3))) s16x4* lds4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)(p + four_pixels));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

template <int WCO, int WCI, int WK, int TY>
__global__ __launch_bounds__(256, 2) void k_conv3x3_wgrad(WgradArgs a) {
  static_assert(WCO * WCI * WK == 4, "4 waves");
  constexpr int COT = 32 * WCO, CIT = 32 * WCI;
  // halves per pixel: four pixels' 32-byte runs start 8 banks apart
  constexpr int DS = COT + 16, XS = CIT + 16;
  constexpr int NPX = TY * 16, NHP = (TY + 2) * 18;
  constexpr int GD = COT / 8, GX = CIT / 8;
  constexpr int ND = NPX * GD / 256, NX = (NHP * GX + 255) / 256;
  constexpr int LDSH = NPX * DS + NHP * XS;            // halves
  static_assert(NPX * GD % 256 == 0 && LDSH * 2 >= 4 * 4096, "staging; a reduction round fits");
  __shared__ __attribute__((aligned(16))) bf16 lds[LDSH];
  bf16* dy = lds;
  bf16* xh = lds + NPX * DS;

  const int Cin = a.Ca + a.Cb;
  const int co0 = blockIdx.x * COT, ci0 = blockIdx.y * CIT;
  const int t_begin = blockIdx.z * a.tiles_per_split;
  const int t_end = min(a.ntiles, t_begin + a.tiles_per_split);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = w % WK, wci = (w / WK) % WCI, wco = w / (WK * WCI);
  const int tiles_x = a.W / 16, tiles_y = a.H / TY;
  const int Hh = a.H >> 1, Wh = a.W >> 1;
  const bool inA = ci0 < a.Ca;                         // (the input's tensors are multiples of CIT, or Cin < CIT)
  const int cs = inA ? a.Ca : a.Cb;
  const int gx8 = (tid % GX) * 8;                      // channel of this thread's halo units
  const bool chan = ci0 + gx8 < Cin;
  const bf16* xsrc = (inA ? a.A + ci0 : a.B + (ci0 - a.Ca)) + (chan ? gx8 : 0);

  u32x4 dv[ND], xv[NX];
  unsigned inside = 0;
  auto load_tile = [&](int t) {
    const int x0 = (t % tiles_x) * 16;
    const int tt = t / tiles_x;
    const int y0 = (tt % tiles_y) * TY, b = tt / tiles_y;
#pragma unroll
    for (int u = 0; u < ND; ++u) {
      const int p = (u * 256 + tid) / GD;
      const size_t pix = (size_t)(b * a.H + y0 + (p >> 4)) * a.W + x0 + (p & 15);
      dv[u] = *reinterpret_cast<const u32x4*>(a.dY + pix * a.Cout + co0 + (tid % GD) * 8);
    }
    inside = 0;
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int pos = (u * 256 + tid) / GX;
      const int hy = pos / 18, hx = pos - hy * 18;
      const int y = y0 + hy - 1, x = x0 + hx - 1;
      const bool ok = chan && pos < NHP && y >= 0 && y < a.H && x >= 0 && x < a.W;
      inside |= (unsigned)ok << u;
      const size_t pix = !ok ? 0 : inA ? (size_t)(b * a.H + y) * a.W + x : (size_t)(b * Hh + (y >> 1)) * Wh + (x >> 1);
      xv[u] = *reinterpret_cast<const u32x4*>(xsrc + pix * cs);
    }
  };
  auto store_tile = [&]() {
#pragma unroll
    for (int u = 0; u < ND; ++u)
      *reinterpret_cast<u32x4*>(&dy[(u * 256 + tid) / GD * DS + (tid % GD) * 8]) = dv[u];
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int pos = (u * 256 + tid) / GX;
      const u32x4 v = (inside >> u) & 1u ? xv[u] : u32x4{0, 0, 0, 0};
      if (pos < NHP) *reinterpret_cast<u32x4*>(&xh[pos * XS + gx8]) = v;
    }
  };

  f32x16 acc[9], accb;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    accb[r] = 0.f;
#pragma unroll
    for (int q = 0; q < 9; ++q) acc[q][r] = 0.f;
  }
  const bool bias = blockIdx.y == 0 && wci == 0;
  const s16x8 one8 = {0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80, 0x3f80};
  const bf16x8 ones = __builtin_bit_cast(bf16x8, one8);
  // a product takes 16 pixels: rows 2 k and 2 k + 1 (lanes 0..31, 32..63) of 8
  // columns; lane i of 16 names pixel i / 4, channels 4 (i % 4)
  const int kh = lane >> 5, c16 = (lane >> 4) & 1, i4 = (lane & 15) >> 2, cc = (lane & 3) * 4;
  const bf16* dp = dy + (kh * 16 + i4) * DS + wco * 32 + c16 * 16 + cc;
  const bf16* xp = xh + (kh * 18 + i4) * XS + wci * 32 + c16 * 16 + cc;

  if (t_begin < t_end) load_tile(t_begin);
  for (int t = t_begin; t < t_end; ++t) {
    if (t > t_begin) lds_sync();                       // the tile before is consumed
    store_tile();
    if (t + 1 < t_end) load_tile(t + 1);
    lds_sync();
#pragma unroll
    for (int k = 0; k < TY / WK; ++k) {                // TY products in all, interleaved over the WK waves
      const int kk = k * WK + wk;
      const int py = (kk >> 1) * 2, px = (kk & 1) * 8;
      const bf16x8 av = read_tr8(dp + (py * 16 + px) * DS, 4 * DS);
      const bf16* xk = xp + (py * 18 + px) * XS;
#pragma unroll
      for (int tap = 0; tap < 9; ++tap) {
        const bf16x8 bv = read_tr8(xk + ((tap / 3) * 18 + tap % 3) * XS, 4 * XS);
        acc[tap] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc[tap], 0, 0, 0);
      }
      if (bias) accb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, ones, accb, 0, 0, 0);
    }
  }

  // D[row = co][col = ci]: register r of a lane is co 8 (r / 4) + 4 kh + r % 4
  const size_t nw = (size_t)9 * a.Cout * Cin;
  float* out = a.part + (size_t)blockIdx.z * (nw + a.Cout);
  const int ci = ci0 + wci * 32 + (lane & 31);
  auto put = [&](int tap, int q, f32x4 v) {            // quad q of a tap (9: the bias)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int co = co0 + wco * 32 + 8 * q + 4 * kh + e;
      if (tap < 9) {
        if (ci < Cin) out[((size_t)tap * a.Cout + co) * Cin + ci] = v[e];
      } else if ((lane & 31) == 0) {
        out[nw + co] = v[e];
      }
    }
  };
  auto quad = [&](int tap, int q) {
    const f32x16& v = tap < 9 ? acc[tap] : accb;
    return f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
  };
  if constexpr (WK == 1) {
#pragma unroll
    for (int tap = 0; tap < 9; ++tap)
#pragma unroll
      for (int q = 0; q < 4; ++q) put(tap, q, quad(tap, q));
    if (bias)
#pragma unroll
      for (int q = 0; q < 4; ++q) put(9, q, quad(9, q));
  } else {
    f32x4* red = reinterpret_cast<f32x4*>(lds);        // [wave][quad][lane]
#pragma unroll
    for (int tap = 0; tap < 10; ++tap) {
      lds_sync();
#pragma unroll
      for (int q = 0; q < 4; ++q) red[(w * 4 + q) * 64 + lane] = quad(tap, q);
      lds_sync();
      if (tap == 9 && !bias) continue;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (q % WK != wk) continue;
        f32x4 v = red[((w - wk) * 4 + q) * 64 + lane];
#pragma unroll
        for (int j = 1; j < WK; ++j) v += red[((w - wk + j) * 4 + q) * 64 + lane];
        put(tap, q, v);
      }
    }
  }
}

// out[i] = sum_z part[z][i]: 64 values a block, ZG groups of threads each adding a
// contiguous range of z in order, the groups' sums added in order (a fixed order)
template <int ZG>
__global__ __launch_bounds__(64 * ZG) void k_reduce_splits(const float* __restrict__ part, int nz, size_t n,
                                                           float* __restrict__ out) {
  __shared__ float red[64 * ZG];
  const int g = threadIdx.x >> 6, l = threadIdx.x & 63;
  const size_t i = (size_t)blockIdx.x * 64 + l;
  const int per = (nz + ZG - 1) / ZG, z0 = min(nz, g * per), z1 = min(nz, z0 + per);
  float s = 0.f;
  if (i < n) {
    int z = z0;
    for (; z + 8 <= z1; z += 8) {                      // eight loads in flight
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = part[(size_t)(z + u) * n + i];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; z < z1; ++z) s += part[(size_t)z * n + i];
  }
  red[threadIdx.x] = s;
  __syncthreads();
  if (g == 0 && i < n) {
    float t = 0.f;
#pragma unroll
    for (int k = 0; k < ZG; ++k) t += red[k * 64 + l];
    out[i] = t;
  }
}

// ----------------------------------------------------------------------------
// 2x2 max pool (forward) and its gradient, which adds into dIn the pooled
// gradient at the first maximum, times (In > 0) (In is a ReLU output).
// A thread takes 8 channels (16 bytes) of one coarse pixel; C is a multiple of 8.
// (One channel a thread, 2-byte accesses: pool 16, its gradient 26, upsampling gradient
// 31 us on average over the levels of 16 images of 256^2; so: 8.7, 22 and 18 us.)
__device__ __forceinline__ void bf8_split(u32x4 v, float* f) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    f[2 * k] = __uint_as_float(v[k] << 16);
    f[2 * k + 1] = __uint_as_float(v[k] & 0xffff0000u);
  }
}
// unit i of n = batch (H / 2) (W / 2) (C / 8): offsets of the coarse unit and of the
// first of its four fine ones, in halves
__device__ __forceinline__ size_t fine_offset(size_t i, int C, int H, int W) {
  const int G = C >> 3, Wo = W >> 1;
  const size_t t = i / G;
  const int x = (int)(t % Wo);
  return ((t / Wo * 2) * W + 2 * x) * (size_t)C + (i % G) * 8;   // (t / Wo runs over batch and coarse rows)
}

__global__ void k_maxpool(const bf16* __restrict__ in, bf16* __restrict__ out, int C, int H, int W, int batch) {
  const size_t n = (size_t)batch * (H >> 1) * (W >> 1) * (C >> 3);
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const bf16* r0 = in + fine_offset(i, C, H, W);
    float v[4][8];
    bf8_split(*reinterpret_cast<const u32x4*>(r0), v[0]);
    bf8_split(*reinterpret_cast<const u32x4*>(r0 + C), v[1]);
    bf8_split(*reinterpret_cast<const u32x4*>(r0 + (size_t)W * C), v[2]);
    bf8_split(*reinterpret_cast<const u32x4*>(r0 + (size_t)W * C + C), v[3]);
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float m[2];
#pragma unroll
      for (int h = 0; h < 2; ++h)
        m[h] = fmaxf(fmaxf(v[0][2 * k + h], v[1][2 * k + h]), fmaxf(v[2][2 * k + h], v[3][2 * k + h]));
      o[k] = pack_bf2(m[0], m[1]);
    }
    *reinterpret_cast<u32x4*>(out + i * 8) = o;
  }
}

__global__ void k_maxpool_bwd(const bf16* __restrict__ in, const bf16* __restrict__ dout, bf16* __restrict__ din, int C,
                              int H, int W, int batch) {
  const size_t n = (size_t)batch * (H >> 1) * (W >> 1) * (C >> 3);
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const size_t o0 = fine_offset(i, C, H, W);
    const size_t off[4] = {o0, o0 + C, o0 + (size_t)W * C, o0 + (size_t)W * C + C};
    float v[4][8], d[4][8], g[8];
#pragma unroll
    for (int q = 0; q < 4; ++q) bf8_split(*reinterpret_cast<const u32x4*>(in + off[q]), v[q]);
#pragma unroll
    for (int q = 0; q < 4; ++q) bf8_split(*reinterpret_cast<const u32x4*>(din + off[q]), d[q]);
    bf8_split(*reinterpret_cast<const u32x4*>(dout + i * 8), g);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      int am = 0;
      float best = v[0][c];
#pragma unroll
      for (int q = 1; q < 4; ++q)
        if (v[q][c] > best) { best = v[q][c]; am = q; }
#pragma unroll
      for (int q = 0; q < 4; ++q) d[q][c] += (am == q && best > 0.f) ? g[c] : 0.f;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      u32x4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = pack_bf2(d[q][2 * k], d[q][2 * k + 1]);
      *reinterpret_cast<u32x4*>(din + off[q]) = o;
    }
  }
}

// gradient of the nearest 2x upsampling: dB[p] = (B[p] > 0) * sum of the 4
// children of dUp (B is a ReLU output)
__global__ void k_upsample_bwd(const bf16* __restrict__ dup, const bf16* __restrict__ Bv, bf16* __restrict__ dB, int C,
                               int H, int W, int batch) {
  const size_t n = (size_t)batch * (H >> 1) * (W >> 1) * (C >> 3);
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const bf16* r0 = dup + fine_offset(i, C, H, W);
    float v[4][8], m[8];
    bf8_split(*reinterpret_cast<const u32x4*>(r0), v[0]);
    bf8_split(*reinterpret_cast<const u32x4*>(r0 + C), v[1]);
    bf8_split(*reinterpret_cast<const u32x4*>(r0 + (size_t)W * C), v[2]);
    bf8_split(*reinterpret_cast<const u32x4*>(r0 + (size_t)W * C + C), v[3]);
    bf8_split(*reinterpret_cast<const u32x4*>(Bv + i * 8), m);
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      float t[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int c = 2 * k + h;
        t[h] = m[c] > 0.f ? (v[0][c] + v[1][c]) + (v[2][c] + v[3][c]) : 0.f;
      }
      o[k] = pack_bf2(t[0], t[1]);
    }
    *reinterpret_cast<u32x4*>(dB + i * 8) = o;
  }
}

// complex64 images (NHWC, C=2, FP32) -> BF16 with 16 channels (2..15 zero)
__global__ void k_pack_input(const float2* __restrict__ x, bf16* __restrict__ out, size_t npix) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < npix; i += (size_t)gridDim.x * blockDim.x) {
    const float2 v = x[i];
    uint4 q0 = make_uint4((uint32_t)f2bf(v.x) | ((uint32_t)f2bf(v.y) << 16), 0, 0, 0);
    uint4* o = reinterpret_cast<uint4*>(out + i * 16);
    o[0] = q0;
    o[1] = make_uint4(0, 0, 0, 0);
  }
}

// final 1x1 convolution (C -> 2) with the residual connection, FP32 output:
// y[p] = x[p] + bias + W f[p].  With a target, also writes dOut = 2 (y - t) / n
// and per-block partial sums of (y - t)^2.
template <int C>
__global__ __launch_bounds__(256) void k_head_fwd(const bf16* __restrict__ f, const float2* __restrict__ x,
                                                  const float* __restrict__ Wh, const float* __restrict__ bh,
                                                  float2* __restrict__ y, const float2* __restrict__ tgt,
                                                  float2* __restrict__ dout, double* __restrict__ loss_part,
                                                  size_t npix, float inv_n) {
  __shared__ float sw[2 * C + 2];
  __shared__ double red[256];
  for (int i = threadIdx.x; i < 2 * C; i += 256) sw[i] = Wh[i];
  if (threadIdx.x < 2) sw[2 * C + threadIdx.x] = bh[threadIdx.x];
  __syncthreads();
  double ls = 0.0;
  for (size_t p = blockIdx.x * (size_t)256 + threadIdx.x; p < npix; p += (size_t)gridDim.x * 256) {
    float o0 = sw[2 * C], o1 = sw[2 * C + 1];
    const uint4* fr = reinterpret_cast<const uint4*>(f + p * C);
#pragma unroll
    for (int g = 0; g < C / 8; ++g) {
      const uint4 v = fr[g];
      const bf16* h = reinterpret_cast<const bf16*>(&v);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float fv = bf2f(h[i]);
        o0 += sw[g * 8 + i] * fv;
        o1 += sw[C + g * 8 + i] * fv;
      }
    }
    const float2 xv = x[p];
    const float2 yv = make_float2(xv.x + o0, xv.y + o1);
    if (y) y[p] = yv;
    if (tgt) {
      const float2 tv = tgt[p];
      const float e0 = yv.x - tv.x, e1 = yv.y - tv.y;
      ls += (double)e0 * e0 + (double)e1 * e1;
      dout[p] = make_float2(2.f * e0 * inv_n, 2.f * e1 * inv_n);
    }
  }
  if (tgt) {
    red[threadIdx.x] = ls;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
      if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
      __syncthreads();
    }
    if (threadIdx.x == 0) loss_part[blockIdx.x] = red[0];
  }
}

// head backward: df[p][c] = (f[p][c] > 0) * sum_o dOut[p][o] W[o][c] (BF16), and
// per-block partials of dW[o][c] = sum_p dOut[p][o] f[p][c], db[o] = sum_p dOut[p][o]
// (2 C weights, then 2 biases).  C / 8 lanes a pixel, 8 channels a lane; a lane adds
// its pixels in order, then the lanes of a wave and the waves are added in a fixed
// order.
template <int C>
__global__ __launch_bounds__(256) void k_head_bwd(const bf16* __restrict__ f, const float2* __restrict__ dout,
                                                  const float* __restrict__ Wh, bf16* __restrict__ df,
                                                  float* __restrict__ part, size_t npix, int ppb) {
  constexpr int LP = C / 8, PPW = 256 / LP;            // lanes per pixel, pixels per step of the block
  static_assert(LP == 4, "the lane sums below step over 4 lanes per pixel");
  __shared__ float red[4][2 * C + 2];
  const int g = threadIdx.x % LP, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const size_t p0 = (size_t)blockIdx.x * ppb, p1 = min(npix, p0 + ppb);
  float w0[8], w1[8], s[18];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    w0[i] = Wh[g * 8 + i];
    w1[i] = Wh[C + g * 8 + i];
  }
#pragma unroll
  for (int i = 0; i < 18; ++i) s[i] = 0.f;
  for (size_t p = p0 + threadIdx.x / LP; p < p1; p += PPW) {
    const float2 d = dout[p];
    const uint4 v = *reinterpret_cast<const uint4*>(f + p * C + g * 8);
    const uint32_t vw[4] = {v.x, v.y, v.z, v.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a = __uint_as_float(vw[i] << 16), b = __uint_as_float(vw[i] & 0xffff0000u);
      s[2 * i] += d.x * a;
      s[2 * i + 1] += d.x * b;
      s[8 + 2 * i] += d.y * a;
      s[8 + 2 * i + 1] += d.y * b;
      const float x = d.x * w0[2 * i] + d.y * w1[2 * i], y = d.x * w0[2 * i + 1] + d.y * w1[2 * i + 1];
      o[i] = pack_bf2(a > 0.f ? x : 0.f, b > 0.f ? y : 0.f);
    }
    *reinterpret_cast<uint4*>(df + p * C + g * 8) = make_uint4(o[0], o[1], o[2], o[3]);
    s[16] += d.x;
    s[17] += d.y;
  }
#pragma unroll
  for (int i = 0; i < 18; ++i)
#pragma unroll
    for (int m = LP; m < 64; m *= 2) s[i] += __shfl_xor(s[i], m);
  if (lane < LP) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      red[w][g * 8 + i] = s[i];
      red[w][C + g * 8 + i] = s[8 + i];
    }
    if (g == 0) {
      red[w][2 * C] = s[16];
      red[w][2 * C + 1] = s[17];
    }
  }
  __syncthreads();
  for (int j = threadIdx.x; j < 2 * C + 2; j += 256)
    part[(size_t)blockIdx.x * (2 * C + 2) + j] = (red[0][j] + red[1][j]) + (red[2][j] + red[3][j]);
}

// Adam (Kingma & Ba 2015) on the FP32 masters, bias-corrected step size
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m, float* __restrict__ v,
                       size_t n, float lr_t, float b1, float b2, float eps) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr_t * mi / (sqrtf(vi) + eps);
  }
}

// BF16 working copies of one conv layer in the order k_conv3x3 stages them:
// [step][32-channel output tile][lane][8], step = (chunk * 9 + tap) * KS + ks with
// chunks of KC = 16 KS input channels, lane = output channel + 32 kh holding input
// channels chunk KC + 16 ks + 8 kh + 0..7.  wb: the same of the flipped, transposed
// weights W'[8 - tap][ci][co] (the input-gradient pass), null where no pass reads it.
__device__ __forceinline__ size_t operand_index(int tap, int co, int ci, int Cout, int Cin) {
  const int KS = Cin % 32 ? 1 : 2, KC = 16 * KS;
  const int chunk = ci / KC, ks = (ci % KC) / 16, kh = (ci % 16) / 8;
  const size_t step = ((size_t)chunk * 9 + tap) * KS + ks;
  return ((step * (Cout / 32) + co / 32) * 64 + (co % 32) + 32 * kh) * 8 + ci % 8;
}
__global__ void k_wprep(const float* __restrict__ wm, bf16* __restrict__ wf, bf16* __restrict__ wb, int Cout, int Cin) {
  const size_t n = (size_t)9 * Cout * Cin;
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    const int ci = i % Cin;
    const size_t t = i / Cin;
    const int co = t % Cout, tap = t / Cout;
    const bf16 h = f2bf(wm[i]);
    wf[operand_index(tap, co, ci, Cout, Cin)] = h;
    if (wb) wb[operand_index(8 - tap, ci, co, Cin, Cout)] = h;
  }
}

inline int grid_for(size_t n, int per = 256) { return (int)std::min<size_t>((n + per - 1) / per, 8192); }

}  // namespace

// ============================================================================
// host side
namespace {

struct Conv {
  int ca, cb, cout;
  int level;          // resolution level (H >> level)
  size_t w_off, b_off;
  bf16 *wf = nullptr, *wb = nullptr;
};

#define UCHK(x)                                                                          \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess) {                                                              \
      cgs::set_error(std::string(#x) + " failed: " + hipGetErrorString(e_));             \
      return CGS_ERR_HIP;                                                                \
    }                                                                                    \
  } while (0)

}  // namespace

struct cgs_unet_s {
  int H = 0, W = 0, L = 4, c0 = 32, maxb = 1;
  std::vector<Conv> convs;     // enc a/b per level, then dec a/b for levels L-2..0
  size_t nparams = 0, head_w = 0, head_b = 0;
  float *params = nullptr, *grads = nullptr, *adam_m = nullptr, *adam_v = nullptr;
  long long step = 0;
  // activations (per level): a, s (enc), u, o (dec); pooled p; grads alike
  std::vector<bf16*> act_a, act_s, act_p, act_u, act_o, g_a, g_s, g_p, g_u, g_o;
  bf16* xin = nullptr;    // packed input, 16 channels
  bf16* g_up = nullptr;   // full-resolution gradient of the upsampled branch
  float2* dout = nullptr;
  float* part = nullptr;
  size_t part_n = 0;
  double* loss_part = nullptr;
  double* h_loss = nullptr;
  float2 *io_x = nullptr, *io_y = nullptr;   // staging for host I/O
  hipStream_t stream = nullptr;
  bool profile = false;
  // profile: [0] conv fwd ms, [1] conv fwd flop, [2] dgrad ms, [3] dgrad flop,
  // [4] wgrad ms, [5] wgrad flop, [6] other ms
  double stats[8] = {0};
  std::vector<hipEvent_t> ev;
};

namespace {

int level_ch(const cgs_unet_s& n, int l) { return n.c0 << l; }

size_t alloc_bytes_total = 0;

template <class T>
int dmalloc(T** p, size_t count) {
  *p = nullptr;
  if (count == 0) return CGS_OK;
  hipError_t e = hipMalloc((void**)p, sizeof(T) * count);
  if (e != hipSuccess) {
    cgs::set_error("hipMalloc of " + std::to_string(sizeof(T) * count) + " bytes failed");
    return CGS_ERR_ALLOC;
  }
  alloc_bytes_total += sizeof(T) * count;
  return CGS_OK;
}

#define RCHK(x)                  \
  do {                           \
    int r_ = (x);                \
    if (r_ != CGS_OK) return r_; \
  } while (0)

struct Timer {
  cgs_unet_s& n;
  int slot;
  double flop;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  Timer(cgs_unet_s& n_, int slot_, double flop_) : n(n_), slot(slot_), flop(flop_) {
    if (!n.profile) return;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    (void)hipEventRecord(e0, n.stream);
  }
  ~Timer() {
    if (!n.profile) return;
    (void)hipEventRecord(e1, n.stream);
    (void)hipEventSynchronize(e1);
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    n.stats[slot] += ms;
    if (slot < 6) n.stats[slot + 1] += flop;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
  }
};

// forward or input-gradient convolution launch: the largest tile (pixels x
// channels) that still gives every CU two blocks, else the one with most blocks
// (asking for one or four blocks a CU measured the same within 3 %)
template <int PW, int CW>
void conv_go(cgs_unet_s& n, const ConvArgs& a) {
  const dim3 g((unsigned)((a.W / 16) * (a.H / (8 * PW)) * a.batch), (unsigned)(a.Cout / (32 * CW)));
  if ((a.Ca + a.Cb) % 32) hipLaunchKernelGGL((k_conv3x3<PW, CW, 16>), g, dim3(256), 0, n.stream, a);
  else hipLaunchKernelGGL((k_conv3x3<PW, CW, 32>), g, dim3(256), 0, n.stream, a);
}

int conv_launch(cgs_unet_s& n, const ConvArgs& a, int slot) {
  const int Cin = a.Ca + a.Cb;
  // (inputs: 16 channels, or chunks of 32 that lie in one of the two tensors)
  if (a.Cout % 32 || (Cin != 16 && (a.Ca % 32 || a.Cb % 32))) {
    cgs::set_error("conv channel counts must be multiples of 32 (or a 16-channel input)");
    return CGS_ERR_UNSUPPORTED;
  }
  if (a.W % 16 || a.H % 16) {
    cgs::set_error("conv tile does not divide the image");
    return CGS_ERR_UNSUPPORTED;
  }
  Timer tm(n, slot, 2.0 * 9.0 * Cin * a.Cout * (double)a.H * a.W * a.batch);
  const long long px = (long long)a.H * a.W * a.batch, ct = a.Cout / 32;
  constexpr long long need = 512;
  const bool even = ct % 2 == 0;
  if (even && px / 256 * (ct / 2) >= need) conv_go<2, 2>(n, a);
  else if (px / 256 * ct >= need) conv_go<2, 1>(n, a);
  else conv_go<1, 1>(n, a);
  UCHK(hipGetLastError());
  return CGS_OK;
}

// out[0..n) = sum of nz partial vectors in n.part
void reduce_go(cgs_unet_s& n, int nz, size_t len, float* out) {
  const dim3 g((unsigned)((len + 63) / 64));
  if (nz >= 32) hipLaunchKernelGGL((k_reduce_splits<16>), g, dim3(1024), 0, n.stream, (const float*)n.part, nz, len, out);
  else hipLaunchKernelGGL((k_reduce_splits<4>), g, dim3(256), 0, n.stream, (const float*)n.part, nz, len, out);
}

template <int WCO, int WCI, int WK, int TY>
int wgrad_go(cgs_unet_s& n, WgradArgs a, int* nsplit_out) {
  const int Cin = a.Ca + a.Cb;
  const int gx = a.Cout / (32 * WCO), gy = (Cin + 32 * WCI - 1) / (32 * WCI);
  const size_t len = (size_t)9 * a.Cout * Cin + a.Cout;
  a.ntiles = a.batch * (a.H / TY) * (a.W / 16);
  // two blocks per CU in all (one or four measured 860 and 973 against 766 us for
  // the 14 layers at a batch of 16 images of 256^2)
  int nsplit = std::max(1, std::min(512 / (gx * gy), a.ntiles));
  while (nsplit > 1 && (size_t)nsplit * len > n.part_n) --nsplit;
  a.tiles_per_split = (a.ntiles + nsplit - 1) / nsplit;
  nsplit = (a.ntiles + a.tiles_per_split - 1) / a.tiles_per_split;
  hipLaunchKernelGGL((k_conv3x3_wgrad<WCO, WCI, WK, TY>), dim3(gx, gy, nsplit), dim3(256), 0, n.stream, a);
  UCHK(hipGetLastError());
  *nsplit_out = nsplit;
  return CGS_OK;
}

// gradients of one layer's weights and biases (dW: 9 Cout Cin values, then Cout).
// Wave tiles: 64 x 64 channels where the counts allow, else the waves that are left
// split the pixels.
int wgrad_launch(cgs_unet_s& n, const bf16* dY, const bf16* A, const bf16* B, int Ca, int Cb, int Cout, int H, int W,
                 int batch, float* dW) {
  const int Cin = Ca + Cb;
  Timer tm(n, 4, 2.0 * 9.0 * Cin * Cout * (double)H * W * batch);
  const WgradArgs a{dY, A, B, n.part, Ca, Cb, Cout, H, W, batch, 0, 0};
  const bool co64 = Cout % 64 == 0, ci64 = Ca % 64 == 0 && Cb % 64 == 0;
  int nsplit = 0;
  if (co64 && ci64) RCHK((wgrad_go<2, 2, 1, 8>(n, a, &nsplit)));
  else if (co64) RCHK((wgrad_go<2, 1, 2, 8>(n, a, &nsplit)));
  else RCHK((wgrad_go<1, 1, 4, 16>(n, a, &nsplit)));
  reduce_go(n, nsplit, (size_t)9 * Cout * Cin + Cout, dW);
  UCHK(hipGetLastError());
  return CGS_OK;
}

int prep_weights(cgs_unet_s& n) {
  for (auto& c : n.convs) {
    const int Cin = c.ca + c.cb;
    const size_t nw = (size_t)9 * c.cout * Cin;
    hipLaunchKernelGGL(k_wprep, dim3(grid_for(nw)), dim3(256), 0, n.stream, (const float*)(n.params + c.w_off), c.wf,
                       c.wb, c.cout, Cin);
    UCHK(hipGetLastError());
  }
  return CGS_OK;
}

int check_batch(const cgs_unet_s& n, int batch) {
  if (batch < 1 || batch > n.maxb) {
    cgs::set_error("batch must be 1.." + std::to_string(n.maxb));
    return CGS_ERR_ARG;
  }
  return CGS_OK;
}

// forward pass; x: device complex64 (batch, H, W); y: device or null;
// tgt: device or null (then loss partials and dOut are written)
int forward(cgs_unet_s& n, const float2* x, float2* y, const float2* tgt, int batch, double* loss) {
  const int L = n.L;
  const size_t npix = (size_t)batch * n.H * n.W;
  {
    Timer tm(n, 6, 0);
    hipLaunchKernelGGL(k_pack_input, dim3(grid_for(npix)), dim3(256), 0, n.stream, x, n.xin, npix);
    UCHK(hipGetLastError());
  }
  const bf16* in = n.xin;
  int cin = 16;
  for (int l = 0; l < L; ++l) {
    const int H = n.H >> l, W = n.W >> l, C = level_ch(n, l);
    const Conv& ca = n.convs[2 * l];
    const Conv& cb = n.convs[2 * l + 1];
    RCHK(conv_launch(n, ConvArgs{in, nullptr, (const uint4*)ca.wf, n.params + ca.b_off, n.act_a[l], nullptr, nullptr, cin, 0, C, C, H, W,
                                 batch, 1}, 0));
    RCHK(conv_launch(n, ConvArgs{n.act_a[l], nullptr, (const uint4*)cb.wf, n.params + cb.b_off, n.act_s[l], nullptr, nullptr, C, 0, C, C,
                                 H, W, batch, 1}, 0));
    if (l < L - 1) {
      Timer tm(n, 6, 0);
      const size_t no = (size_t)batch * (H / 2) * (W / 2) * (C / 8);
      hipLaunchKernelGGL(k_maxpool, dim3(grid_for(no)), dim3(256), 0, n.stream, (const bf16*)n.act_s[l], n.act_p[l], C,
                         H, W, batch);
      UCHK(hipGetLastError());
      in = n.act_p[l];
      cin = C;
    }
  }
  // decoder
  for (int l = L - 2; l >= 0; --l) {
    const int H = n.H >> l, W = n.W >> l, C = level_ch(n, l);
    const Conv& da = n.convs[2 * L + 2 * (L - 2 - l)];
    const Conv& db = n.convs[2 * L + 2 * (L - 2 - l) + 1];
    const bf16* below = (l + 1 == L - 1) ? n.act_s[L - 1] : n.act_o[l + 1];
    RCHK(conv_launch(n, ConvArgs{n.act_s[l], below, (const uint4*)da.wf, n.params + da.b_off, n.act_u[l], nullptr, nullptr, C, 2 * C, C,
                                 C, H, W, batch, 1}, 0));
    RCHK(conv_launch(n, ConvArgs{n.act_u[l], nullptr, (const uint4*)db.wf, n.params + db.b_off, n.act_o[l], nullptr, nullptr, C, 0, C, C,
                                 H, W, batch, 1}, 0));
  }
  {
    Timer tm(n, 6, 0);
    const int nb = (int)std::min<size_t>((npix + 255) / 256, 2048);
    if (n.c0 != 32) {
      cgs::set_error("head kernel is built for 32 channels");
      return CGS_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL((k_head_fwd<32>), dim3(nb), dim3(256), 0, n.stream, (const bf16*)n.act_o[0], x,
                       (const float*)(n.params + n.head_w), (const float*)(n.params + n.head_b), y, tgt, n.dout,
                       n.loss_part, npix, (float)(1.0 / (2.0 * (double)npix)));
    UCHK(hipGetLastError());
    if (tgt && loss) {
      UCHK(hipMemcpyAsync(n.h_loss, n.loss_part, sizeof(double) * nb, hipMemcpyDeviceToHost, n.stream));
      UCHK(hipStreamSynchronize(n.stream));
      double s = 0.0;
      for (int i = 0; i < nb; ++i) s += n.h_loss[i];
      *loss = s / (2.0 * (double)npix);
    }
  }
  return CGS_OK;
}

// backward pass after forward(..., tgt, ...): fills n.grads
int backward(cgs_unet_s& n, int batch) {
  const int L = n.L;
  const size_t npix = (size_t)batch * n.H * n.W;
  {
    Timer tm(n, 6, 0);
    const int ppb = (int)std::max<size_t>(256, (npix + 1023) / 1024);   // at most 1024 blocks
    const int nb = (int)((npix + ppb - 1) / ppb);
    hipLaunchKernelGGL((k_head_bwd<32>), dim3(nb), dim3(256), 0, n.stream, (const bf16*)n.act_o[0],
                       (const float2*)n.dout, (const float*)(n.params + n.head_w), n.g_o[0], n.part, npix, ppb);
    UCHK(hipGetLastError());
    // head_w and head_b are adjacent (2C then 2 values)
    reduce_go(n, nb, (size_t)(2 * n.c0 + 2), n.grads + n.head_w);
    UCHK(hipGetLastError());
  }
  // decoder levels, l = 0 .. L-2
  for (int l = 0; l <= L - 2; ++l) {
    const int H = n.H >> l, W = n.W >> l, C = level_ch(n, l);
    const Conv& da = n.convs[2 * L + 2 * (L - 2 - l)];
    const Conv& db = n.convs[2 * L + 2 * (L - 2 - l) + 1];
    const bf16* below = (l + 1 == L - 1) ? n.act_s[L - 1] : n.act_o[l + 1];
    bf16* g_below = (l + 1 == L - 1) ? n.g_s[L - 1] : n.g_o[l + 1];
    // conv db: X = u_l, dY = g_o[l]
    RCHK(wgrad_launch(n, n.g_o[l], n.act_u[l], nullptr, C, 0, C, H, W, batch, n.grads + db.w_off));
    RCHK(conv_launch(n, ConvArgs{n.g_o[l], nullptr, (const uint4*)db.wb, nullptr, n.g_u[l], nullptr, n.act_u[l], C, 0, C, C, H, W, batch,
                                 0}, 2));
    // conv da: X = (s_l | up(below)), dY = g_u[l]
    RCHK(wgrad_launch(n, n.g_u[l], n.act_s[l], below, C, 2 * C, C, H, W, batch, n.grads + da.w_off));
    RCHK(conv_launch(n, ConvArgs{n.g_u[l], nullptr, (const uint4*)da.wb, nullptr, n.g_s[l], n.g_up, n.act_s[l], C, 0, 3 * C, C, H, W,
                                 batch, 0}, 2));
    {
      Timer tm(n, 6, 0);
      const size_t no = (size_t)batch * (H / 2) * (W / 2) * (2 * C / 8);
      hipLaunchKernelGGL(k_upsample_bwd, dim3(grid_for(no)), dim3(256), 0, n.stream, (const bf16*)n.g_up, below,
                         g_below, 2 * C, H, W, batch);
      UCHK(hipGetLastError());
    }
  }
  // encoder levels, l = L-1 .. 0
  for (int l = L - 1; l >= 0; --l) {
    const int H = n.H >> l, W = n.W >> l, C = level_ch(n, l);
    const Conv& ca = n.convs[2 * l];
    const Conv& cb = n.convs[2 * l + 1];
    const bf16* in = l ? n.act_p[l - 1] : n.xin;
    const int cin = l ? level_ch(n, l - 1) : 16;
    RCHK(wgrad_launch(n, n.g_s[l], n.act_a[l], nullptr, C, 0, C, H, W, batch, n.grads + cb.w_off));
    RCHK(conv_launch(n, ConvArgs{n.g_s[l], nullptr, (const uint4*)cb.wb, nullptr, n.g_a[l], nullptr, n.act_a[l], C, 0, C, C, H, W, batch,
                                 0}, 2));
    RCHK(wgrad_launch(n, n.g_a[l], in, nullptr, cin, 0, C, H, W, batch, n.grads + ca.w_off));
    if (l > 0) {
      // gradient at the pooled input (unmasked), then routed into g_s[l-1]
      RCHK(conv_launch(n, ConvArgs{n.g_a[l], nullptr, (const uint4*)ca.wb, nullptr, n.g_p[l - 1], nullptr, nullptr, C, 0, cin, cin, H, W,
                                   batch, 0}, 2));
      Timer tm(n, 6, 0);
      const size_t no = (size_t)batch * H * W * (cin / 8);
      hipLaunchKernelGGL(k_maxpool_bwd, dim3(grid_for(no)), dim3(256), 0, n.stream, (const bf16*)n.act_s[l - 1],
                         (const bf16*)n.g_p[l - 1], n.g_s[l - 1], cin, 2 * H, 2 * W, batch);
      UCHK(hipGetLastError());
    }
  }
  return CGS_OK;
}

int upload(cgs_unet_s& n, const void* x, int batch, int device_io, const float2** dx, float2* stage) {
  if (device_io) {
    *dx = (const float2*)x;
    return CGS_OK;
  }
  UCHK(hipMemcpyAsync(stage, x, sizeof(float2) * (size_t)batch * n.H * n.W, hipMemcpyHostToDevice, n.stream));
  *dx = stage;
  return CGS_OK;
}

}  // namespace

// n normal values of deviation sd.  On its own and aligned because its time (two
// million values, most of a network's creation) came out at 77 or at 133 ms from one
// link of the same objects to the next; what decides is not known
static __attribute__((noinline, aligned(64))) void normal_fill(float* w, size_t n, float sd, std::mt19937_64& rng) {
  std::normal_distribution<float> nd(0.f, sd);
  for (size_t i = 0; i < n; ++i) w[i] = nd(rng);
}

extern "C" {

int cgs_unet_create(cgs_unet* out, int H, int W, int levels, int base_channels, int max_batch, unsigned long long seed) {
  if (!out) return CGS_ERR_ARG;
  *out = nullptr;
  if (levels < 2 || levels > 6 || base_channels != 32 || max_batch < 1) {
    cgs::set_error("unet: levels 2..6, base_channels 32, max_batch >= 1");
    return CGS_ERR_UNSUPPORTED;
  }
  const int q = 16 << (levels - 1);   // every level's side must take a 16-pixel tile
  if (H < q || W < q || H % q || W % q) {
    cgs::set_error("unet: image sides must be multiples of " + std::to_string(q));
    return CGS_ERR_UNSUPPORTED;
  }
  auto* n = new cgs_unet_s();
  n->H = H;
  n->W = W;
  n->L = levels;
  n->c0 = base_channels;
  n->maxb = max_batch;
  // layer table
  size_t off = 0;
  for (int l = 0; l < levels; ++l) {
    const int C = base_channels << l, cin = l ? (base_channels << (l - 1)) : 16;
    n->convs.push_back(Conv{cin, 0, C, l, 0, 0});
    n->convs.push_back(Conv{C, 0, C, l, 0, 0});
  }
  for (int l = levels - 2; l >= 0; --l) {
    const int C = base_channels << l;
    n->convs.push_back(Conv{C, 2 * C, C, l, 0, 0});
    n->convs.push_back(Conv{C, 0, C, l, 0, 0});
  }
  for (auto& c : n->convs) {
    c.w_off = off;
    off += (size_t)9 * c.cout * (c.ca + c.cb);
    c.b_off = off;
    off += c.cout;
  }
  n->head_w = off;
  off += 2 * (size_t)base_channels;
  n->head_b = off;
  off += 2;
  n->nparams = off;

  auto fail = [&](int rc) {
    cgs_unet_destroy(n);
    return rc;
  };
  if (hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking) != hipSuccess) {
    cgs::set_error("hipStreamCreate failed");
    delete n;
    return CGS_ERR_HIP;
  }
  int rc;
  if ((rc = dmalloc(&n->params, off)) || (rc = dmalloc(&n->grads, off)) || (rc = dmalloc(&n->adam_m, off)) ||
      (rc = dmalloc(&n->adam_v, off)))
    return fail(rc);
  for (auto& c : n->convs) {
    const size_t nw = (size_t)9 * c.cout * (c.ca + c.cb);
    const bool first = (c.ca + c.cb) % 32 != 0;   // its input's gradient is not formed
    if ((rc = dmalloc(&c.wf, nw)) || (!first && (rc = dmalloc(&c.wb, nw)))) return fail(rc);
  }
  const size_t B = max_batch;
  n->act_a.assign(levels, nullptr);
  n->act_s.assign(levels, nullptr);
  n->act_p.assign(levels, nullptr);
  n->act_u.assign(levels, nullptr);
  n->act_o.assign(levels, nullptr);
  n->g_a.assign(levels, nullptr);
  n->g_s.assign(levels, nullptr);
  n->g_p.assign(levels, nullptr);
  n->g_u.assign(levels, nullptr);
  n->g_o.assign(levels, nullptr);
  for (int l = 0; l < levels; ++l) {
    const size_t px = B * (size_t)(H >> l) * (W >> l);
    const size_t C = (size_t)base_channels << l;
    if ((rc = dmalloc(&n->act_a[l], px * C)) || (rc = dmalloc(&n->act_s[l], px * C)) ||
        (rc = dmalloc(&n->g_a[l], px * C)) || (rc = dmalloc(&n->g_s[l], px * C)))
      return fail(rc);
    if (l < levels - 1) {
      if ((rc = dmalloc(&n->act_p[l], px / 4 * C)) || (rc = dmalloc(&n->g_p[l], px / 4 * C)) ||
          (rc = dmalloc(&n->act_u[l], px * C)) || (rc = dmalloc(&n->act_o[l], px * C)) ||
          (rc = dmalloc(&n->g_u[l], px * C)) || (rc = dmalloc(&n->g_o[l], px * C)))
        return fail(rc);
    }
  }
  const size_t px0 = B * (size_t)H * W;
  if ((rc = dmalloc(&n->xin, px0 * 16)) || (rc = dmalloc(&n->g_up, px0 * 2 * base_channels)) ||
      (rc = dmalloc(&n->dout, px0)) || (rc = dmalloc(&n->io_x, px0)) || (rc = dmalloc(&n->io_y, px0)) ||
      (rc = dmalloc(&n->loss_part, 4096)))
    return fail(rc);
  // split-K partials: the largest layer at 64 splits, at most 64 Mi floats
  size_t wmax = 0;
  for (auto& c : n->convs) wmax = std::max(wmax, (size_t)9 * c.cout * (c.ca + c.cb) + c.cout);
  n->part_n = std::min<size_t>(std::max<size_t>(64 * wmax, px0 * 2 / 1024 * 256 + 4096), (size_t)64 << 20);
  n->part_n = std::max(n->part_n, wmax);
  if ((rc = dmalloc(&n->part, n->part_n))) return fail(rc);
  if (hipHostMalloc((void**)&n->h_loss, sizeof(double) * 4096, 0) != hipSuccess) return fail(CGS_ERR_ALLOC);

  // He-normal initialisation (std = sqrt(2 / fan_in)), zero biases, zero head
  std::vector<float> h(off, 0.f);
  std::mt19937_64 rng(seed);
  for (auto& c : n->convs) {
    const int Cin = c.ca + c.cb;
    const int real_in = (c.level == 0 && c.ca == 16) ? 2 : Cin;   // packed input has 2 live channels
    normal_fill(h.data() + c.w_off, (size_t)9 * c.cout * Cin, std::sqrt(2.f / (9.f * real_in)), rng);
  }
  if (hipMemcpy(n->params, h.data(), sizeof(float) * off, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(n->adam_m, 0, sizeof(float) * off) != hipSuccess ||
      hipMemset(n->adam_v, 0, sizeof(float) * off) != hipSuccess ||
      hipMemset(n->grads, 0, sizeof(float) * off) != hipSuccess) {
    cgs::set_error("unet: parameter upload failed");
    return fail(CGS_ERR_HIP);
  }
  if ((rc = prep_weights(*n)) != CGS_OK) return fail(rc);
  if (hipStreamSynchronize(n->stream) != hipSuccess) return fail(CGS_ERR_HIP);
  *out = n;
  return CGS_OK;
}

int cgs_unet_destroy(cgs_unet n) {
  if (!n) return CGS_OK;
  if (n->stream) (void)hipStreamSynchronize(n->stream);
  auto fr = [](void* p) {
    if (p) (void)hipFree(p);
  };
  fr(n->params);
  fr(n->grads);
  fr(n->adam_m);
  fr(n->adam_v);
  for (auto& c : n->convs) {
    fr(c.wf);
    fr(c.wb);
  }
  for (auto* v : {&n->act_a, &n->act_s, &n->act_p, &n->act_u, &n->act_o, &n->g_a, &n->g_s, &n->g_p, &n->g_u, &n->g_o})
    for (auto* p : *v) fr(p);
  fr(n->xin);
  fr(n->g_up);
  fr(n->dout);
  fr(n->io_x);
  fr(n->io_y);
  fr(n->part);
  fr(n->loss_part);
  if (n->h_loss) (void)hipHostFree(n->h_loss);
  if (n->stream) (void)hipStreamDestroy(n->stream);
  delete n;
  return CGS_OK;
}

int cgs_unet_num_params(cgs_unet n, long long* count) {
  if (!n || !count) return CGS_ERR_ARG;
  *count = (long long)n->nparams;
  return CGS_OK;
}

int cgs_unet_get_params(cgs_unet n, float* host) {
  if (!n || !host) return CGS_ERR_ARG;
  UCHK(hipMemcpyAsync(host, n->params, sizeof(float) * n->nparams, hipMemcpyDeviceToHost, n->stream));
  UCHK(hipStreamSynchronize(n->stream));
  return CGS_OK;
}

int cgs_unet_set_params(cgs_unet n, const float* host) {
  if (!n || !host) return CGS_ERR_ARG;
  UCHK(hipMemcpyAsync(n->params, host, sizeof(float) * n->nparams, hipMemcpyHostToDevice, n->stream));
  RCHK(prep_weights(*n));
  UCHK(hipStreamSynchronize(n->stream));
  return CGS_OK;
}

int cgs_unet_get_grads(cgs_unet n, float* host) {
  if (!n || !host) return CGS_ERR_ARG;
  UCHK(hipMemcpyAsync(host, n->grads, sizeof(float) * n->nparams, hipMemcpyDeviceToHost, n->stream));
  UCHK(hipStreamSynchronize(n->stream));
  return CGS_OK;
}

int cgs_unet_reset_optimizer(cgs_unet n) {
  if (!n) return CGS_ERR_ARG;
  UCHK(hipMemsetAsync(n->adam_m, 0, sizeof(float) * n->nparams, n->stream));
  UCHK(hipMemsetAsync(n->adam_v, 0, sizeof(float) * n->nparams, n->stream));
  UCHK(hipStreamSynchronize(n->stream));
  n->step = 0;
  return CGS_OK;
}

int cgs_unet_forward(cgs_unet n, const void* x, void* y, int batch, int device_io) {
  if (!n || !x || !y) return CGS_ERR_ARG;
  RCHK(check_batch(*n, batch));
  const float2* dx;
  RCHK(upload(*n, x, batch, device_io, &dx, n->io_x));
  float2* dy = device_io ? (float2*)y : n->io_y;
  RCHK(forward(*n, dx, dy, nullptr, batch, nullptr));
  if (!device_io)
    UCHK(hipMemcpyAsync(y, dy, sizeof(float2) * (size_t)batch * n->H * n->W, hipMemcpyDeviceToHost, n->stream));
  UCHK(hipStreamSynchronize(n->stream));
  return CGS_OK;
}

int cgs_unet_gradients(cgs_unet n, const void* x, const void* target, int batch, int device_io, double* loss) {
  if (!n || !x || !target) return CGS_ERR_ARG;
  RCHK(check_batch(*n, batch));
  const float2 *dx, *dt;
  RCHK(upload(*n, x, batch, device_io, &dx, n->io_x));
  RCHK(upload(*n, target, batch, device_io, &dt, n->io_y));
  double l = 0.0;
  RCHK(forward(*n, dx, nullptr, dt, batch, &l));
  RCHK(backward(*n, batch));
  UCHK(hipStreamSynchronize(n->stream));
  if (loss) *loss = l;
  return CGS_OK;
}

int cgs_unet_train_step(cgs_unet n, const void* x, const void* target, int batch, double lr, int device_io,
                        double* loss) {
  RCHK(cgs_unet_gradients(n, x, target, batch, device_io, loss));
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  n->step += 1;
  const double lr_t = lr * std::sqrt(1.0 - std::pow((double)b2, (double)n->step)) /
                      (1.0 - std::pow((double)b1, (double)n->step));
  {
    Timer tm(*n, 6, 0);
    hipLaunchKernelGGL(k_adam, dim3(grid_for(n->nparams)), dim3(256), 0, n->stream, n->params,
                       (const float*)n->grads, n->adam_m, n->adam_v, n->nparams, (float)lr_t, b1, b2, eps);
    UCHK(hipGetLastError());
    RCHK(prep_weights(*n));
  }
  UCHK(hipStreamSynchronize(n->stream));
  return CGS_OK;
}

int cgs_unet_profile(cgs_unet n, int enable, double* stats8) {
  if (!n) return CGS_ERR_ARG;
  if (stats8)
    for (int i = 0; i < 8; ++i) stats8[i] = n->stats[i];
  if (enable >= 0) {
    n->profile = enable != 0;
    for (double& s : n->stats) s = 0.0;
  }
  return CGS_OK;
}

}  // extern "C"
