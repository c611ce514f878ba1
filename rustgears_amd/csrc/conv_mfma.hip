// conv_mfma.hip -- FP16 and FP32 convolutions (C k k > 32 taps or more than 64
// output channels; the others run in conv_direct_kernel) as one implicit GEMM
// kernel, with the MaxPool2d(2, 2) and the next Linear's operand where they
// follow: D[channel, pixel] = W[channel, (tap, c)] . X[(tap, c), pixel].
//
// These layers have few pixels per image (the CNN's second conv: 16 x 16) and
// little work per byte on the matrix cores, so the time goes to launches and
// round trips: as im2col + GEMM + transpose + pool they took 43 us for 100
// images (17.3 + 12.2 + 9.8 + 3.7), the im2col matrix alone 9 times the input.
//  * A workgroup of 4 waves owns RB x XB output pixels of one image and 16, 32
//    or 64 channels.  The input rows under its pixels are staged in LDS
//    channel-last, 64 bytes of channels (32 binary16 or 16 f32) at a time, zeros
//    around the image; a K step of 64 bytes is then one tap of one channel
//    block, and every fragment is one 16-byte LDS read.
//  * The weights lie in memory as [channel block][tap][output channel][64
//    bytes], so a tap of a workgroup is one contiguous run that global_load_lds
//    copies beside the band.
//  * Both are stored with their 16-byte pieces at piece ^ ((row >> 1) & 3), the
//    bank-conflict-free order of the large GEMM.
//  * Pooled outputs go through LDS, so any width and height pools here.
// Now 8.8 us for those 100 images (15.0 before the branch-free half_bits, with a
// wave per channel in the pool), FP32 on 256 images 27.5 us.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "devmath.h"
#include "gemm_core.h"
#include "rgnpu_internal.h"

namespace rgnpu {

namespace cmf {
constexpr int kWaves = 4, kThreads = kWaves * 64;
constexpr int kGroupBytes = 36 * 1024;  // weights staged at a time: 9 taps of 64 channels
constexpr int kMaxLds = 156 * 1024;
}  // namespace cmf

struct ConvMfmaShape {
  int32_t C, H, W, O, OH, OW, k, stride, pad;
  int32_t blocks_c;            // 64-byte channel blocks
  int32_t Opad;                // output channels of the weight layout
  int32_t RB, XB, tiles_y, tiles_x, tiles_o;
  int32_t BR, BC;              // band rows and columns
  int32_t TG;                  // taps staged at a time
  uint32_t mBC, mBR, mXB, mPW, mPer;  // magic_of the divisors of the indexes divided here
  int32_t wbase;               // LDS byte offset of the weights
  int32_t pool, PH, PW, pbw, pbh;  // pooled output, and the pooled pixels of a full tile
};

// v / d for v, d < 2^16 and m = magic_of(d) (0 stands for d = 1).
__device__ __forceinline__ uint32_t div_by(uint32_t v, uint32_t m) { return m ? __umulhi(v, m) : v; }

// The max pool's window step: NaN propagates and ties keep the earlier element
// (kernels.rs:180-191).
__device__ __forceinline__ float window_take(float best, float v) { return (v > best || v != v) ? v : best; }

template <int MODE, int ACT, int OCF, int PN>
__device__ __forceinline__ void conv_mfma_out(int8_t* smem, const v4f (&sum)[OCF][PN], const ConvMfmaShape& s,
                                              const Epilogue& ep, int b, int oy0, int ox0, int o0, int wave,
                                              int lane) {
  constexpr int P = 64 * PN, PS = P + 4;  // PS: the 4 lane quads' rows in different banks
  float* const stage = reinterpret_cast<float*>(smem);
  const int64_t L = (int64_t)s.OH * s.OW;
#pragma unroll
  for (int n = 0; n < PN; n++) {
    const int p = (wave * PN + n) * 16 + (lane & 15);
    const int ry = (int)div_by((uint32_t)p, s.mXB), rx = p - ry * s.XB;
    const bool live = ry < s.RB && oy0 + ry < s.OH && ox0 + rx < s.OW;
    float* const yp = ep.y + (int64_t)b * s.O * L + (int64_t)(oy0 + ry) * s.OW + ox0 + rx;
#pragma unroll
    for (int o = 0; o < OCF; o++) {
      const int ch = o * 16 + 4 * (lane >> 4);
      const v4f bias = *reinterpret_cast<const v4f*>(ep.bias + o0 + ch);  // padded past O
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const float v = epi_word<ACT, MODE>(__float_as_int(sum[o][n][e]), 1.0f, bias[e], ep.act_param);
        if (s.pool)
          stage[(ch + e) * PS + p] = v;
        else if (live && o0 + ch + e < s.O)
          yp[(int64_t)(o0 + ch + e) * L] = v;
      }
    }
  }
  if (!s.pool) return;
  __syncthreads();
  // the tile's pooled outputs, columns fastest, then rows, then channels
  const int py0 = oy0 >> 1, px0 = ox0 >> 1;
  const uint32_t per = (uint32_t)(s.pbh * s.pbw), n = per * 16u * OCF;
  const int64_t PL = (int64_t)s.PH * s.PW;
  for (uint32_t it = threadIdx.x; it < n; it += cmf::kThreads) {
    const uint32_t ch = div_by(it, s.mPer), i = it - ch * per;
    const int ry = (int)div_by(i, s.mPW), rx = (int)i - ry * s.pbw;
    const int py = py0 + ry, px = px0 + rx;
    const float* const w = stage + ch * PS + 2 * ry * s.XB + 2 * rx;
    float best = -__builtin_inff();
    best = window_take(best, w[0]);
    best = window_take(best, w[1]);
    best = window_take(best, w[s.XB]);
    best = window_take(best, w[s.XB + 1]);
    if (py >= s.PH || px >= s.PW || o0 + (int)ch >= s.O) continue;
    const int64_t at = (int64_t)(o0 + (int)ch) * PL + (int64_t)py * s.PW + px;
    if (MODE == kModeF16 && ep.h_out)
      ep.h_out[(int64_t)b * ep.ldh + at] = (uint16_t)rgmath::half_bits(best);
    else
      ep.y[(int64_t)b * s.O * PL + at] = best;
  }
}

template <int MODE, int OCF, int PN>
__global__ __launch_bounds__(cmf::kThreads, 2) void conv_mfma_kernel(const float* __restrict__ x,
                                                                  const int8_t* __restrict__ wt, ConvMfmaShape s,
                                                                  Epilogue ep) {
  using namespace cmf;
  constexpr int E = MODE == kModeF16 ? 8 : 4;  // channels per 16-byte piece
  extern __shared__ __attribute__((aligned(1024))) int8_t cm_smem[];
  int8_t* const smem = cm_smem;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // tiles of one image are neighbours on one XCD (dealt round-robin)
  const int total = (int)gridDim.x, q8 = total >> 3, rem = total & 7, xcd = (int)blockIdx.x & 7;
  int t = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + ((int)blockIdx.x >> 3);
  const int to = t % s.tiles_o;
  t /= s.tiles_o;
  const int tx = t % s.tiles_x;
  t /= s.tiles_x;
  const int ty = t % s.tiles_y, b = t / s.tiles_y;
  const int oy0 = ty * s.RB, ox0 = tx * s.XB, o0 = to * 16 * OCF;
  const int iy0 = oy0 * s.stride - s.pad, ix0 = ox0 * s.stride - s.pad;
  const uint32_t HW4 = (uint32_t)(s.H * s.W) * 4u;
  const __amdgpu_buffer_rsrc_t rx = bounded_rsrc(x + (int64_t)b * s.C * s.H * s.W);
  const int taps = s.k * s.k;
  // A chain over all of K rounds at every step, so runs of taps are summed from
  // zero and then join a total: FP32 three taps (48 products), FP16 nine, the
  // even and odd ones apart (its MFMA adds 32 products with fewer roundings).
  // Against 64 bits, one chain (in FP32 per channel block) and now, in 2^-24 of
  // the sum: FP32 32 channels 3 x 3 3.9 and 2.2 (im2col + split K 3.0), 16 channels
  // 7 x 7 7.9 and 2.6 (2.9); FP16 60 channels 3 x 3 2.6
  // and 1.4 (1.5).
  constexpr int NA = MODE == kModeF16 ? 2 : 1;
  v4f tot[OCF][PN] = {};
  uint32_t pb[PN];  // band pixel under each of the lane's output pixels (0 past the tile)
#pragma unroll
  for (int n = 0; n < PN; n++) {
    const int p = (wave * PN + n) * 16 + (lane & 15);
    const int ry = (int)div_by((uint32_t)p, s.mXB), rx_ = p - ry * s.XB;
    pb[n] = ry < s.RB ? (uint32_t)((ry * s.BC + rx_) * s.stride) : 0u;
  }
  const uint32_t rd = (uint32_t)((lane & 15) * 64 + (((lane >> 4) ^ lds_swz(lane & 15)) << 4));
  const int lr = lane >> 2, lp = (lane & 3) ^ lds_swz(lane >> 2);
  const uint32_t items = (uint32_t)(4 * s.BR * s.BC);
  for (int cb = 0; cb < s.blocks_c; cb++) {
    for (int t0 = 0; t0 < taps; t0 += s.TG) {
      const int nt = min(s.TG, taps - t0);
      // weights of taps t0 .. t0 + nt: OCF instructions of 1 KiB per tap
      for (int j = wave; j < nt * OCF; j += kWaves) {
        const int tt = j / OCF, o = j % OCF;
        const int8_t* const src = wt + (((int64_t)cb * taps + t0 + tt) * s.Opad + o0 + o * 16) * 64;
        dma16(src + (uint32_t)(lr * 64 + lp * 16), smem + s.wbase + j * 1024);
      }
      if (t0 == 0) {
        // the band: 16-byte pieces of E channels of one pixel, columns fastest
        for (uint32_t i0 = (uint32_t)tid; i0 < items; i0 += 2 * kThreads) {
          float v[2][E];
          uint32_t dst[2];
#pragma unroll
          for (int u = 0; u < 2; u++) {
            const uint32_t i = i0 + u * kThreads < items ? i0 + u * kThreads : i0;
            const uint32_t r = div_by(i, s.mBC), bx = i - r * (uint32_t)s.BC;
            const uint32_t pc = div_by(r, s.mBR), by = r - pc * (uint32_t)s.BR;
            const int iy = iy0 + (int)by, ix = ix0 + (int)bx, c = cb * 4 * E + (int)pc * E;
            const bool in = (uint32_t)iy < (uint32_t)s.H && (uint32_t)ix < (uint32_t)s.W;
            const uint32_t off = (uint32_t)c * HW4 + (uint32_t)(iy * s.W + ix) * 4u;
#pragma unroll
            for (int e = 0; e < E; e++)
              v[u][e] = __builtin_bit_cast(
                  float, __builtin_amdgcn_raw_buffer_load_b32(
                             rx, (int)(in && c + e < s.C ? off + (uint32_t)e * HW4 : kDropOffset), 0, 0));
            const uint32_t pix = by * (uint32_t)s.BC + bx;
            dst[u] = pix * 64u + ((pc ^ ((pix >> 1) & 3u)) << 4);
          }
#pragma unroll
          for (int u = 0; u < 2; u++) {
            v4i w;
            if constexpr (MODE == kModeF16) {
#pragma unroll
              for (int g = 0; g < 4; g++)
                w[g] = (int)(rgmath::half_bits(v[u][2 * g]) | (rgmath::half_bits(v[u][2 * g + 1]) << 16));
            } else {
#pragma unroll
              for (int g = 0; g < 4; g++) w[g] = __float_as_int(v[u][g]);
            }
            *reinterpret_cast<v4i*>(smem + dst[u]) = w;
          }
        }
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's weight copies
      __syncthreads();
      int ki = t0 / s.k, kj = t0 - ki * s.k;
      v4f acc[NA][OCF][PN];
      // Tap tt's products onto a sum, or from zero with `first`.
      auto tap = [&](int tt, v4f (&to)[OCF][PN], auto first) {
        const uint32_t shift = (uint32_t)(ki * s.BC + kj);
        v4i a[OCF], f[PN];
#pragma unroll
        for (int n = 0; n < PN; n++) {
          const uint32_t pix = pb[n] + shift;
          f[n] = *reinterpret_cast<const v4i*>(smem + pix * 64u + ((((uint32_t)lane >> 4) ^ ((pix >> 1) & 3u)) << 4));
        }
#pragma unroll
        for (int o = 0; o < OCF; o++)
          a[o] = *reinterpret_cast<const v4i*>(smem + s.wbase + (tt * OCF + o) * 1024 + rd);
#pragma unroll
        for (int c = 0; c < (MODE == kModeF32 ? 4 : 1); c++)
#pragma unroll
          for (int o = 0; o < OCF; o++)
#pragma unroll
            for (int n = 0; n < PN; n++) {
              const v4f from = first.value && c == 0 ? v4f{0.0f, 0.0f, 0.0f, 0.0f} : to[o][n];
              if constexpr (MODE == kModeF16)
                to[o][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a[o]),
                                                                   __builtin_bit_cast(v8h, f[n]), from, 0, 0, 0);
              else
                to[o][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(v4f, a[o])[c],
                                                                 __builtin_bit_cast(v4f, f[n])[c], from, 0, 0, 0);
            }
        if (++kj == s.k) {
          kj = 0;
          ki++;
        }
      };
      auto add_run = [&] {
#pragma unroll
        for (int o = 0; o < OCF; o++)
#pragma unroll
          for (int n = 0; n < PN; n++) tot[o][n] += acc[0][o][n];
      };
      constexpr std::true_type first{};
      constexpr std::false_type next{};
      int tt = 0;
      if constexpr (MODE == kModeF16) {
        while (tt < nt) {
          const int end = min(tt + 9, nt);
          tap(tt++, acc[0], first);
          if (tt < end) {
            tap(tt++, acc[1], first);
            if (end - tt == 7) {  // without branches, the reads run ahead of the MFMAs
#pragma unroll
              for (int u = 0; u < 7; u++) tap(tt + u, acc[u & 1], next);
              tt = end;
            }
            for (; tt + 2 <= end; tt += 2) {
              tap(tt, acc[0], next);
              tap(tt + 1, acc[1], next);
            }
            if (tt < end) tap(tt++, acc[0], next);
#pragma unroll
            for (int o = 0; o < OCF; o++)
#pragma unroll
              for (int n = 0; n < PN; n++) acc[0][o][n] += acc[1][o][n];
          }
          add_run();
        }
      } else {
        for (; tt + 3 <= nt; tt += 3) {
          tap(tt, acc[0], first);
          tap(tt + 1, acc[0], next);
          tap(tt + 2, acc[0], next);
          add_run();
        }
        if (tt < nt) {
          tap(tt, acc[0], first);
          if (tt + 1 < nt) tap(tt + 1, acc[0], next);
          add_run();
        }
      }
      __syncthreads();  // the reads are done before the next copies, or the pool's stage, overwrite them
    }
  }
#define RG_CMF(ACTV) conv_mfma_out<MODE, ACTV, OCF, PN>(smem, tot, s, ep, b, oy0, ox0, o0, wave, lane)
  switch (ep.act) {
    case rgmath::ACT_RELU: RG_CMF(rgmath::ACT_RELU); break;
    case rgmath::ACT_SIGMOID: RG_CMF(rgmath::ACT_SIGMOID); break;
    case rgmath::ACT_TANH: RG_CMF(rgmath::ACT_TANH); break;
    case rgmath::ACT_GELU: RG_CMF(rgmath::ACT_GELU); break;
    case rgmath::ACT_LEAKY_RELU: RG_CMF(rgmath::ACT_LEAKY_RELU); break;
    case rgmath::ACT_SILU: RG_CMF(rgmath::ACT_SILU); break;
    default: RG_CMF(rgmath::ACT_NONE); break;
  }
#undef RG_CMF
}

// The tile of a convolution: whole output rows where they are at most 64
// pixels wide, as many of them as 64, 128 or 256 pixels hold.  The largest of
// those that still gives 1.5 workgroups per CU, else the smallest that fits (the
// CNN's second conv on 100 images: 400 workgroups of 4 rows); none that a smaller
// one holds as well, whose pixels past the image would be multiplied for nothing
// (256 images of 7 x 7, 256 -> 256: FP32 610 -> 194 us, FP16 117 -> 76 us), and not
// 256 where 128 take far fewer rounds of the workgroups that a CU holds (100 images
// of 23 x 23, 60 -> 120: FP32 132 -> 109 us, FP16 47 -> 35; 256 of 28 x 28, 128 -> 256,
// 1 x 1: 276 -> 196 and 277 -> 154; but 256 of 14 x 14, 128 -> 128, one round of 256:
// FP16 42 against 59; a window of 1 is mostly band, which more workgroups load
// sooner).  Then fewer output channels while that gives at most two
// workgroups per CU and the band is small: a workgroup walks all of K, and a short
// walk is worth reading the band again (4 images of 14 x 14, 128 -> 128 channels: 64,
// 32 and 16 of them FP32 33, 22 and 17 us, FP16 16, 14 and 10; but 7 x 7 at stride 2
// on 1 x 3 x 224 x 224 FP16 25 and 37 us).
struct ConvMfmaTile {
  int ocf = 0, pn = 0;
  ConvMfmaShape s{};
  int64_t grid = 0;
  size_t lds = 0;
};

// ceil(2^32 / d): m d exceeds 2^32 by less than d, so v m / 2^32 has the
// quotient's integer part while v d < 2^32.  d = 1 wraps to 0.
static uint32_t magic_of(int64_t d) { return (uint32_t)(((uint64_t(1) << 32) + (uint64_t)d - 1) / (uint64_t)d); }

static bool conv_mfma_tile(const ConvShape& cs, bool f16, bool pool, ConvMfmaTile* out) {
  const int64_t cpb = f16 ? 32 : 16;  // channels per 64 bytes
  if (cs.n <= 0 || cs.OH <= 0 || cs.OW <= 0 || (pool && (cs.OH < 2 || cs.OW < 2)) ||
      cs.C * cs.H * cs.W * 4 >= (int64_t(1) << 31) || cs.k > 64)
    return false;
  int ocf = cs.O <= 16 ? 1 : cs.O <= 32 ? 2 : 4;
  const int64_t XB = std::min<int64_t>(cs.OW, 64);
  const int64_t used = pool ? cs.OH & ~int64_t(1) : cs.OH;  // the pool drops an odd last row
  auto rows = [&](int pn) {
    const int64_t r = std::min<int64_t>(used, 64 * pn / XB);
    return pool ? r & ~int64_t(1) : r;
  };
  auto tiles = [&](int pn) { return cs.n * ((used + rows(pn) - 1) / rows(pn)) * ((cs.OW + XB - 1) / XB); };
  // 256 pixels leave a CU two workgroups, 128 three
  const int64_t to = (cs.O + 63) / 64;
  const bool half = rows(2) > 0 && rows(2) < rows(4) &&
                    5 * ((tiles(2) * to + 767) / 768) < (cs.k == 1 ? 8 : 7) * ((tiles(4) * to + 511) / 512);
  for (int pn = half ? 2 : 4; pn >= 1;) {
    const int64_t RB = rows(pn), ob = 16 * ocf;
    const int smaller = pn > 1 && rows(pn / 2) > 0 ? pn / 2 : 0;
    if (RB <= 0 || (smaller >= 1 && rows(smaller) == RB)) {
      pn = smaller;
      continue;
    }
    const int64_t TG = std::max<int64_t>(1, std::min<int64_t>(cs.k * cs.k, cmf::kGroupBytes / (ob * 64)));
    const int64_t BR = (RB - 1) * cs.stride + cs.k, BC = (XB - 1) * cs.stride + cs.k;
    const int64_t band = (BR * BC * 64 + 1023) / 1024 * 1024;
    const int64_t lds = std::max(band + TG * ob * 64, pool ? ob * (64 * pn + 4) * 4 : int64_t(0));
    const int64_t ty = (used + RB - 1) / RB, tx = (cs.OW + XB - 1) / XB, to = (cs.O + ob - 1) / ob;
    const int64_t grid = cs.n * ty * tx * to;
    // quotients by multiplication are exact while dividend * divisor < 2^32; a grid
    // holds fewer than 2^32 threads
    if (4 * BR * BC >= 65536 || BC >= 65536 || BR >= 65536 || lds > cmf::kMaxLds ||
        grid * cmf::kThreads >= (int64_t(1) << 32)) {
      pn = smaller;
      continue;
    }
    ConvMfmaTile g;
    g.ocf = ocf;
    g.pn = pn;
    g.grid = grid;
    g.lds = (size_t)lds;
    ConvMfmaShape& s = g.s;
    s.C = (int32_t)cs.C; s.H = (int32_t)cs.H; s.W = (int32_t)cs.W; s.O = (int32_t)cs.O;
    s.OH = (int32_t)cs.OH; s.OW = (int32_t)cs.OW; s.k = (int32_t)cs.k;
    s.stride = (int32_t)cs.stride; s.pad = (int32_t)cs.pad;
    s.blocks_c = (int32_t)((cs.C + cpb - 1) / cpb);
    s.Opad = (int32_t)round_up(cs.O, kConvMfmaOPad);
    s.RB = (int32_t)RB; s.XB = (int32_t)XB;
    s.tiles_y = (int32_t)ty; s.tiles_x = (int32_t)tx; s.tiles_o = (int32_t)to;
    s.BR = (int32_t)BR; s.BC = (int32_t)BC; s.TG = (int32_t)TG;
    s.pool = pool;
    s.PH = (int32_t)(cs.OH / 2); s.PW = (int32_t)(cs.OW / 2);
    s.pbh = (int32_t)(RB / 2); s.pbw = (int32_t)(XB / 2);
    s.mBC = magic_of(BC); s.mBR = magic_of(BR); s.mXB = magic_of(XB);
    s.mPW = pool ? magic_of(XB / 2) : 0;
    s.mPer = pool ? magic_of((RB / 2) * (XB / 2)) : 0;  // at most 64 x 64 outputs: below 2^16
    s.wbase = (int32_t)band;
    *out = g;
    if (grid >= 384) break;
    if (smaller >= 1)
      pn = smaller;
    else if (ocf > 1 && 4 * BR * BC <= 2048 && cs.n * ty * tx * ((cs.O + ob / 2 - 1) / (ob / 2)) <= 512)
      ocf /= 2;
    else
      break;
  }
  return out->ocf != 0;
}

bool conv_mfma_supported(const ConvShape& cs, bool f16, bool pool) {
  ConvMfmaTile g;
  return conv_mfma_tile(cs, f16, pool, &g);
}

// A workgroup walks all of K (a tap of a channel block ~0.1 us, the next block's
// band ~1.2), where im2col + GEMM splits it over the chip for four launches: deep
// layers on few pixels are faster there (3 x 3 on 7 x 7 images, 512 -> 512 channels,
// one image: FP32 65 against 49 us, FP16 38 against 32; 256 -> 256 FP32 38 against
// 32, but on 16 images 40 against 51).
bool conv_mfma_better(const ConvShape& cs, bool f16) {
  const int64_t per = f16 ? 32 : 16, blocks = (cs.C + per - 1) / per, walk = blocks * (cs.k * cs.k + 12);
  const int64_t pixels = cs.n * cs.OH * cs.OW;
  return f16 ? walk < 160 || pixels > 4 * (walk - 110) : walk < 320 || pixels > 2 * (walk - 200);
}

template <int MODE, int OCF, int PN>
static void launch_cmf_t(const ConvMfmaTile& g, const float* x, const int8_t* w, const Epilogue& ep, hipStream_t s) {
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&conv_mfma_kernel<MODE, OCF, PN>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, cmf::kMaxLds);
  if (attr != hipSuccess) throw std::runtime_error("MFMA conv: the device refuses its LDS size");
  RG_LAUNCH((conv_mfma_kernel<MODE, OCF, PN>), dim3((unsigned)g.grid), dim3(cmf::kThreads), (unsigned)g.lds, s, x, w,
            g.s, ep);
}

template <int MODE, int OCF>
static void launch_cmf(const ConvMfmaTile& g, const float* x, const int8_t* w, const Epilogue& ep, hipStream_t s) {
  if (g.pn == 4) launch_cmf_t<MODE, OCF, 4>(g, x, w, ep, s);
  else if (g.pn == 2) launch_cmf_t<MODE, OCF, 2>(g, x, w, ep, s);
  else launch_cmf_t<MODE, OCF, 1>(g, x, w, ep, s);
}

void launch_conv_mfma(const float* x, const void* w, const ConvShape& cs, bool f16, bool pool, const Epilogue& ep,
                      hipStream_t s) {
  ConvMfmaTile g;
  if (!conv_mfma_tile(cs, f16, pool, &g)) throw std::logic_error("MFMA conv: unsupported shape");
  if (ep.h_out && (!f16 || !pool)) throw std::logic_error("MFMA conv: the operand hand-off is FP16 after a pool");
  const int8_t* const wb = reinterpret_cast<const int8_t*>(w);
  if (f16) {
    if (g.ocf == 1) launch_cmf<kModeF16, 1>(g, x, wb, ep, s);
    else if (g.ocf == 2) launch_cmf<kModeF16, 2>(g, x, wb, ep, s);
    else launch_cmf<kModeF16, 4>(g, x, wb, ep, s);
  } else {
    if (g.ocf == 1) launch_cmf<kModeF32, 1>(g, x, wb, ep, s);
    else if (g.ocf == 2) launch_cmf<kModeF32, 2>(g, x, wb, ep, s);
    else launch_cmf<kModeF32, 4>(g, x, wb, ep, s);
  }
}

// This translation unit's code object, loaded at program creation.
__global__ void conv_mfma_load_probe_kernel() {}

void load_conv_mfma_code_object(hipStream_t s) {
  hipLaunchKernelGGL(conv_mfma_load_probe_kernel, dim3(1), dim3(64), 0, s);
}

}  // namespace rgnpu
