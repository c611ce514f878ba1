// conv_direct.hip -- direct convolution for the FP16 and FP32 providers when a
// window holds at most kDirectConvTaps values (C * k * k: the CNN's first conv
// has 27) and there are at most 64 output channels.
//
// One thread computes OB output channels of one output pixel, summing the taps
// serially in the reference's im2col order (ch * k + ki) * k + kj, padding taps
// (zeros) included, as fp16_gemm_fused (npu.rs:425-445) and the serial matmul
// of conv2d_forward (kernels.rs:218-265) do.  FP16: each input is round_fp16'd
// and each product of two binary16 values is exact in f32, so fma gives the
// reference's multiply-then-add; the output is act(round_fp16(sum + bias)).
// FP32: multiply, then add (no contraction); the output is sum + bias (the
// activation is a layer of its own).
//
// The work per pixel is a chain of TAPS x OB multiply-adds (864 for the CNN's
// 27 taps and 32 channels, ~2 us of the chip on 100 images), so what counts is
// what stands around it:
//  * The input rows under a workgroup's 256 pixels are loaded and converted once
//    into LDS (BAND), where each thread reads its taps; loads of each tap by
//    each pixel convert every input k * k times and compute as many addresses.
//    Images too wide for that load their TAPS inputs, all before the first is
//    used (a loop that loads and uses one tap waits for memory 27 times).  The
//    tap count is rounded up to a compiled one; the extra taps have zero weights
//    and zero inputs (an input there could be infinite, and Inf * 0 is NaN), and
//    adding +0 changes no sum that began at +0.
//  * The weights are f32, tap-major, at wave-uniform addresses: scalar loads
//    into SGPR operands.  (Broadcast LDS reads cost the CU 8 clocks per 4
//    weights and wave, twice the multiply-adds they feed.)
//  * The pool exchanges rows with one permlane swap per two channels and fills
//    the odd lanes with two more channels, so a store carries 4 channels; with
//    ReLU it pools the sums, before bias, rounding and activation.
// CNN conv 1 + pool (trace): FP16 on 100 images of 3 x 32 x 32 20.6 -> 10.7 us, on
// 200 of 3 x 46 x 46 without pool and 60 channels 60 -> 45 us against the same
// kernel without the band; FP32 on 256 images 26.0 -> 21.8 us.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>

#include "devmath.h"
#include "gemm_core.h"
#include "rgnpu_internal.h"

namespace rgnpu {

constexpr int64_t kDirectBandBytes = 32 * 1024;  // LDS band of a workgroup at most (5 fit a CU)

struct DirectShape {
  int32_t C, H, W, O, OH, OW, k, stride, pad;
  int32_t blocks;  // 256-pixel blocks per image
  int32_t total;   // of all images
  int32_t taps;
  int32_t BR, BW;         // rows per channel and row length of the LDS band
  uint32_t mBR, mBW, mOW;  // ceil(2^32 / d): exact quotients below 2^16
};

__device__ __forceinline__ uint32_t quot(uint32_t v, uint32_t m) { return m ? __umulhi(v, m) : v; }  // 0: d = 1

// The max pool's window step: NaN propagates and ties keep the earlier element
// (kernels.rs:180-191).
__device__ __forceinline__ float pool_step(float best, float v) { return (v > best || v != v) ? v : best; }

// The value of lane ^ 1.
__device__ __forceinline__ float lane_xor1(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));  // quad_perm 1,0,3,2
}

template <int ACT, int MODE>
__device__ __forceinline__ float direct_value(float acc, float bias, float p) {
  const float s = acc + bias;
  return act_fixed<ACT>(MODE == kModeF16 ? rgmath::round_fp16(s) : s, p);
}

template <int ACT, int OB, int MODE>
__device__ __forceinline__ void direct_store(const float (&acc)[OB], const float* __restrict__ bias, float* yb,
                                             int64_t L, int o_n, float act_param) {
#pragma unroll
  for (int o = 0; o < OB; o++)
    if (o < o_n) yb[(int64_t)o * L] = direct_value<ACT, MODE>(acc[o], bias[o], act_param);
}

// MaxPool2d(2, 2) (npu.rs:384-390) of a wave's 64 pixels in registers.  OW is
// 16 or 32 and OH even (host-checked), so the wave holds whole pairs of output
// rows: pixel p + 1 is in lane ^ 1 and p + OW in lane ^ OW.  Each row pair of
// values is pooled first (r), then the two rows: taking the lower row's winner
// gives what taking its elements one by one gives (the first maximum and the
// last NaN of the window, in the reference's order).  For channels o, o + 1 a
// permlane swap puts (upper, lower) of o in the lanes of the upper rows and of
// o + 1 in those of the lower rows; channels o + 2, o + 3 go to the odd lanes.
template <int ACT, int OB, int MODE>
__device__ __forceinline__ void direct_pool(const float (&acc)[OB], const float* __restrict__ bias,
                                            float* __restrict__ yb, int o_n, int OH, int OW, int pix0, int lane,
                                            int L, float act_param) {
  static_assert(OB % 4 == 0, "channels in fours");
  // relu(round(acc + bias)) never decreases in acc and has neither NaN nor -0
  // (NaN sums give +0, which no other element of the window is below), so with
  // ReLU the largest sum, NaN dropped, gives the window's result.
  constexpr bool SUMS = ACT == rgmath::ACT_RELU;
  const int lower = (lane & OW) != 0, odd = lane & 1;
  const int pix = pix0 + (lane & ~(OW | 1));  // the window's first pixel
  const int oy = pix / OW, ox = pix - oy * OW;
  const int64_t PL = (int64_t)(OH >> 1) * (OW >> 1);
  const int mine = lower + 2 * odd;  // which of the four channels this lane stores
  float* const yl = yb + (int64_t)mine * PL + (int64_t)(oy >> 1) * (OW >> 1) + (ox >> 1);
  const bool live = pix < L;
#pragma unroll
  for (int o = 0; o < OB; o += 4) {
    float r[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
      if constexpr (SUMS) {
        r[e] = __builtin_fmaxf(acc[o + e], lane_xor1(acc[o + e]));
        continue;
      }
      const float v = direct_value<ACT, MODE>(acc[o + e], bias[o + e], act_param);
      const float n = lane_xor1(v);
      // both lanes of a pair compute the even lane's result
      const float first = odd ? n : v, second = odd ? v : n;
      r[e] = pool_step(pool_step(-__builtin_inff(), first), second);
    }
    float w[2];
#pragma unroll
    for (int e = 0; e < 2; e++) {
      const uint32_t a = __float_as_uint(r[2 * e]), c = __float_as_uint(r[2 * e + 1]);
      const auto s = OW == 32 ? __builtin_amdgcn_permlane32_swap(a, c, false, false)
                              : __builtin_amdgcn_permlane16_swap(a, c, false, false);
      const float up = __uint_as_float(s[0]), low = __uint_as_float(s[1]);
      w[e] = SUMS ? __builtin_fmaxf(up, low) : pool_step(up, low);
    }
    float best = odd ? w[1] : w[0];
    if constexpr (SUMS) best = direct_value<ACT, MODE>(best, bias[o + mine], act_param);
    if (live && o + mine < o_n) yl[(int64_t)o * PL] = best;
  }
}

template <int MODE, int TAPS, int OB, bool BAND>
__global__ __launch_bounds__(256) void conv_direct_kernel(const float* __restrict__ x, const float* __restrict__ wt,
                                                          const float* __restrict__ bias, float* __restrict__ y,
                                                          DirectShape s, int act, float act_param, int pool2) {
  const int wg = (int)(blockIdx.z * gridDim.x + blockIdx.x);
  if (wg >= s.total) return;
  const int b = wg / s.blocks, blk = wg - b * s.blocks;
  const int o0 = (int)blockIdx.y * OB, o_n = s.O - o0;
  const int L = s.OH * s.OW, lane = (int)threadIdx.x & 63;
  const int pix_raw = blk * 256 + (int)threadIdx.x;
  const bool live = pix_raw < L;
  const int pix = live ? pix_raw : L - 1;  // every lane joins the pool's exchanges
  const float* const xb = x + (int64_t)b * s.C * s.H * s.W;
  constexpr int MIN_TAPS = TAPS == 32 ? 28 : TAPS - 8;  // fewer take a smaller TAPS
  float v[TAPS];
  if constexpr (BAND) {
    extern __shared__ __attribute__((aligned(16))) float band[];
    // pixels of the block from the start of its first row on (< 2^16)
    const int row0 = blk * 256 / s.OW, rel = pix - row0 * s.OW;
    const int by = (int)quot((uint32_t)rel, s.mOW), ox = rel - by * s.OW;
    const int iyb = row0 * s.stride - s.pad;
    const uint32_t n = (uint32_t)(s.C * s.BR * s.BW);
    for (uint32_t i0 = threadIdx.x; i0 < n; i0 += 4 * 256) {
      float l[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const uint32_t i = i0 + u * 256;
        const uint32_t r = quot(i, s.mBW), c = i - r * (uint32_t)s.BW;
        const uint32_t ch = quot(r, s.mBR);
        const int iy = iyb + (int)(r - ch * (uint32_t)s.BR), ix = (int)c - s.pad;
        const bool ok = i < n && (uint32_t)iy < (uint32_t)s.H && (uint32_t)ix < (uint32_t)s.W;
        // a place outside the image loads the image's first value and drops it
        const float g = xb[ok ? ((int64_t)ch * s.H + iy) * s.W + ix : 0];
        l[u] = ok ? (MODE == kModeF16 ? rgmath::round_fp16(g) : g) : 0.0f;
      }
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (i0 + u * 256 < n) band[i0 + u * 256] = l[u];
    }
    __syncthreads();
    const int base = by * s.stride * s.BW + ox * s.stride;
    int ch = 0, ki = 0, kj = 0;
#pragma unroll
    for (int kk = 0; kk < TAPS; kk++) {
      const float g = band[base + (ch * s.BR + ki) * s.BW + kj];  // past the last tap: that tap's input
      v[kk] = kk < MIN_TAPS || kk < s.taps ? g : 0.0f;
      if (kk + 1 < s.taps && ++kj == s.k) {
        kj = 0;
        if (++ki == s.k) {
          ki = 0;
          ch++;
        }
      }
    }
  } else {
    const int oy = pix / s.OW, ox = pix - oy * s.OW;
    const int iy0 = oy * s.stride - s.pad, ix0 = ox * s.stride - s.pad;
    int ch = 0, ki = 0, kj = 0;
#pragma unroll
    for (int kk = 0; kk < TAPS; kk++) {
      const int iy = iy0 + ki, ix = ix0 + kj;
      const bool ok = kk < s.taps && (uint32_t)iy < (uint32_t)s.H && (uint32_t)ix < (uint32_t)s.W;
      // a tap outside the image loads the plane's first value and drops it
      const float* const plane = xb + (int64_t)(kk < s.taps ? ch : 0) * s.H * s.W;
      const float g = plane[ok ? (uint32_t)(iy * s.W + ix) : 0u];
      v[kk] = ok ? (MODE == kModeF16 ? rgmath::round_fp16(g) : g) : 0.0f;
      if (++kj == s.k) {
        kj = 0;
        if (++ki == s.k) {
          ki = 0;
          ch++;
        }
      }
    }
  }
  float acc[OB];
#pragma unroll
  for (int o = 0; o < OB; o++) acc[o] = 0.0f;
  const float* const w0 = wt + o0;
#pragma unroll
  for (int kk = 0; kk < TAPS; kk++) {
    const float* const w = w0 + kk * 64;
    if constexpr (MODE == kModeF16) {
#pragma unroll
      for (int o = 0; o < OB; o++) acc[o] = __builtin_fmaf(v[kk], w[o], acc[o]);
    } else {
#pragma unroll
      for (int o = 0; o < OB; o++) {
        const float p = v[kk] * w[o];
        acc[o] = acc[o] + p;
      }
    }
  }
  const float* const bb = bias + o0;
  if (pool2) {
    float* const yb = y + ((int64_t)b * s.O + o0) * ((int64_t)(s.OH >> 1) * (s.OW >> 1));
    const int pix0 = blk * 256 + ((int)threadIdx.x & ~63);
    if (act == rgmath::ACT_RELU)
      direct_pool<rgmath::ACT_RELU, OB, MODE>(acc, bb, yb, o_n, s.OH, s.OW, pix0, lane, L, act_param);
    else
      direct_pool<rgmath::ACT_NONE, OB, MODE>(acc, bb, yb, o_n, s.OH, s.OW, pix0, lane, L, act_param);
    return;
  }
  if (!live) return;
  float* const yb = y + ((int64_t)b * s.O + o0) * L + pix;
  // one activation per unrolled store loop: with the activation switch inside
  // the loop, the accumulators ended up on the stack
#define RG_CDS(ACTV) direct_store<ACTV, OB, MODE>(acc, bb, yb, L, o_n, act_param)
  switch (act) {
    case rgmath::ACT_RELU: RG_CDS(rgmath::ACT_RELU); break;
    case rgmath::ACT_SIGMOID: RG_CDS(rgmath::ACT_SIGMOID); break;
    case rgmath::ACT_TANH: RG_CDS(rgmath::ACT_TANH); break;
    case rgmath::ACT_GELU: RG_CDS(rgmath::ACT_GELU); break;
    case rgmath::ACT_LEAKY_RELU: RG_CDS(rgmath::ACT_LEAKY_RELU); break;
    case rgmath::ACT_SILU: RG_CDS(rgmath::ACT_SILU); break;
    default: RG_CDS(rgmath::ACT_NONE); break;
  }
#undef RG_CDS
}

bool conv_direct_supported(const ConvShape& cs) {
  // 32-bit pixel, plane and workgroup indexes
  return cs.C * cs.k * cs.k <= kDirectConvTaps && cs.O <= 64 && cs.H * cs.W < (int64_t(1) << 29) &&
         cs.OH * cs.OW < (int64_t(1) << 29) && cs.n * ((cs.OH * cs.OW + 255) / 256) < (int64_t(1) << 31);
}

template <int MODE>
static void launch_conv_direct_t(const float* x, const float* w, const float* bias, float* y, const ConvShape& cs,
                                 int act, float act_param, int pool2, hipStream_t s) {
  if (!conv_direct_supported(cs) || cs.O <= 0) throw std::logic_error("direct conv: unsupported shape");
  if (pool2 && ((pool2 != 16 && pool2 != 32) || cs.OW != pool2 || cs.OH % 2 != 0 ||
                (act != rgmath::ACT_RELU && act != rgmath::ACT_NONE)))
    throw std::logic_error("direct conv: the fused pool needs ReLU or none, even height, width 16 or 32");
  const int64_t L = cs.OH * cs.OW;
  if (L <= 0 || cs.n <= 0) return;
  DirectShape d{(int32_t)cs.C,      (int32_t)cs.H,   (int32_t)cs.W,              (int32_t)cs.O,
                      (int32_t)cs.OH,     (int32_t)cs.OW,  (int32_t)cs.k,              (int32_t)cs.stride,
                      (int32_t)cs.pad,    (int32_t)((L + 255) / 256), 0,
                      (int32_t)(cs.C * cs.k * cs.k)};
  // The band of a block: its output rows (one more where blocks start inside a
  // row) over the padded width.
  const int64_t rows = 256 % cs.OW == 0 ? 256 / cs.OW : (255 + cs.OW - 1) / cs.OW + 1;
  const int64_t BR = (rows - 1) * cs.stride + cs.k, BW = (cs.OW - 1) * cs.stride + cs.k;
  const bool band = cs.C * BR * BW * 4 <= kDirectBandBytes && rows * cs.OW < 65536;
  auto magic = [](int64_t v) { return (uint32_t)(((uint64_t(1) << 32) + (uint64_t)v - 1) / (uint64_t)v); };
  d.BR = (int32_t)BR;
  d.BW = (int32_t)BW;
  d.mBR = band ? magic(BR) : 0;
  d.mBW = band ? magic(BW) : 0;
  d.mOW = band ? magic(cs.OW) : 0;
  // 32 channels per thread share the loads and conversions of the inputs; 16
  // where that leaves fewer than 3 waves per SIMD.
  const int64_t wgs = cs.n * d.blocks;
  const int OB = band && cs.O > 16 && wgs * ((cs.O + 31) / 32) >= 768 ? 32 : 16;
  d.total = (int32_t)wgs;
  // a grid dimension holds fewer than 2^32 threads: the rest goes into z
  constexpr int64_t kMaxX = int64_t(1) << 22;
  const dim3 grid((unsigned)std::min(wgs, kMaxX), (unsigned)((cs.O + OB - 1) / OB), (unsigned)((wgs + kMaxX - 1) / kMaxX));
#define RG_CD(T, B, BD)                                                                                            \
  RG_LAUNCH((conv_direct_kernel<MODE, T, B, BD>), grid, dim3(256), BD ? (unsigned)(cs.C * BR * BW * 4) : 0u, s, x, \
            w, bias, y, d, act, act_param, pool2)
#define RG_CDB(T)                            \
  do {                                       \
    if (band && OB == 32) RG_CD(T, 32, true); \
    else if (band) RG_CD(T, 16, true);       \
    else RG_CD(T, 16, false);                \
  } while (0)
  if (d.taps <= 9) RG_CDB(9);
  else if (d.taps <= 18) RG_CDB(18);
  else if (d.taps <= 27) RG_CDB(27);
  else RG_CDB(32);
#undef RG_CDB
#undef RG_CD
}

void launch_conv_direct_f16(const float* x, const float* w, const float* bias, float* y, const ConvShape& cs, int act,
                            float act_param, int pool_ow, hipStream_t s) {
  launch_conv_direct_t<kModeF16>(x, w, bias, y, cs, act, act_param, pool_ow, s);
}

void launch_conv_direct_f32(const float* x, const float* w, const float* bias, float* y, const ConvShape& cs,
                            int pool_act, int pool_ow, hipStream_t s) {
  launch_conv_direct_t<kModeF32>(x, w, bias, y, cs, pool_ow ? pool_act : rgmath::ACT_NONE, 0.0f, pool_ow, s);
}

// This translation unit's code object, loaded at program creation.
__global__ void conv_direct_load_probe_kernel() {}

void load_conv_direct_code_object(hipStream_t s) {
  hipLaunchKernelGGL(conv_direct_load_probe_kernel, dim3(1), dim3(64), 0, s);
}

}  // namespace rgnpu
