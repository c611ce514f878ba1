// mid.hip -- the Linear GEMM for batches between the GEMV's 8 rows and the
// sizes that fill the chip with 128 x 128 tiles: C[M, N] = A[M, K] . B[N, K]^T
// with the fused epilogue, in the three operand modes.
//
// What bounds these calls is the latency of a CU's loads and the bytes it
// loads (FP32: the matrix cores): a few rows of a 4096-wide layer have 32 to
// 100 tiles of 128 x 128, and splitting K over more workgroups costs a second
// kernel and a round trip of the partial sums through memory.  Here one
// workgroup of 8 waves owns a small TM x TN output tile (16 to 128 rows and
// columns, as many tiles as CUs where that can be) and all of K.  Measured
// against 128 x 128 tiles with split K and its epilogue kernel (us, kernels
// only): 100 x 4096 x 4096 i8 18.3 -> 7.8, f16 22.6 -> 12.2, f32 75 -> 46;
// 1000 x 1024 x 1024 i8 17.6 -> 5.8, f16 21.8 -> 7.4, f32 33.8 -> 23.8;
// 12 x 4096 x 4096 i8 16.2 -> 4.2 (16.8 MB of weights: 4.0 TB/s).
//  * K is walked in stages of KS x 64 bytes per row.  The stage's rows travel
//    global -> LDS by buffer loads with the LDS as destination, 1 KiB per
//    instruction (runs of 256 or 512 contiguous bytes of a row), STAGES - 1
//    stages ahead.  Rows past M or N and bytes past a row's end get an offset
//    past the buffer: they are not fetched and land as zeros, so ragged
//    shapes need no padded operand and load no padding.
//  * The waves split the stage's K: wave w multiplies the 64-byte K block
//    w % KS of all TN columns and of its share of the TM rows, so each staged
//    byte is read from LDS once per wave row group (a split of the tile over
//    the waves would read it 2 to 4 times).  The KS partial tiles are added
//    through LDS at the end (integers: exact; f32: in a fixed order).
//  * 16-byte chunks are stored at chunk ^ (row & 15) of their row: the 16 rows
//    of a fragment read fall in 16 different bank groups.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <stdexcept>
#include <type_traits>

#include "devmath.h"
#include "gemm_core.h"
#include "rgnpu_internal.h"

namespace rgnpu {

namespace mid {
constexpr int kWaves = 8, kThreads = kWaves * 64;
}  // namespace mid

struct MidShape {
  int64_t lda;           // bytes between rows of A
  int32_t ka, kb;        // bytes of a row of A that exist, bytes of a row of B (its padded length)
  int32_t M, N;
  int32_t tiles_m, tiles_n;
  int32_t vec;           // y rows take 16-byte stores
  int32_t run;           // FP16, FP32: stages summed from zero before they join the total
};

// One buffer load of 16 bytes per lane into LDS, lane i at lds + 16 i; lanes
// with an offset past the buffer write zeros.
__device__ __forceinline__ void dma16_buf(__amdgpu_buffer_rsrc_t r, int8_t* lds, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (RG_LDS_AS void*)lds, 16, (int)off, 0, 0, 0);
}

// The workgroup's TM x TN outputs from the KS partial tiles in LDS: 4
// consecutive columns per thread.  Returns the thread's largest |y|.
template <int MODE, int ACT, int TM, int TN, int KS>
__device__ __forceinline__ float mid_epilogue(const int32_t* red, const MidShape& s, const Epilogue& ep, float cs,
                                              int m0, int n0, v4f b) {
  constexpr int LD = TN + 4, Q = TN / 4;
  static_assert(mid::kThreads % Q == 0, "a thread's outputs share their columns");
  const int c = ((int)threadIdx.x % Q) * 4, col = n0 + c;
  float amax = 0.0f;
  for (int r = (int)threadIdx.x / Q; r < TM; r += mid::kThreads / Q) {
    const int row = m0 + r;
    if (row >= s.M) break;
    v4i p[KS];
#pragma unroll
    for (int k = 0; k < KS; k++) p[k] = *reinterpret_cast<const v4i*>(red + (k * TM + r) * LD + c);
#pragma unroll
    for (int d = KS / 2; d >= 1; d /= 2)  // pairwise: log2 KS roundings of a f32 sum
#pragma unroll
      for (int k = 0; k < d; k++) {
        if constexpr (MODE == kModeI8)
          p[k] += p[k + d];
        else
          p[k] = __builtin_bit_cast(v4i, __builtin_bit_cast(v4f, p[k]) + __builtin_bit_cast(v4f, p[k + d]));
      }
    const v4i sum = p[0];
    v4f v;
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = epi_word<ACT, MODE>(sum[e], cs, b[e], ep.act_param);
    if constexpr (MODE == kModeF16) {
      if (ep.h_out) {  // the next Linear's operand, zero past N
        uint32_t h[4];
#pragma unroll
        for (int e = 0; e < 4; e++) h[e] = col + e < s.N ? rgmath::half_bits(v[e]) : 0u;
        if (col < ep.ldh)
          *reinterpret_cast<uint2*>(ep.h_out + (int64_t)row * ep.ldh + col) =
              make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
        continue;
      }
    }
    float* y = ep.y + (int64_t)row * s.N + col;
    if (s.vec && col + 4 <= s.N) {
      *reinterpret_cast<v4f*>(y) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (col + e < s.N) y[e] = v[e];
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (col + e < s.N) {
        if (ep.acc_out) ep.acc_out[(int64_t)row * s.N + col + e] = sum[e];
        amax = __builtin_fmaxf(amax, __builtin_fabsf(v[e]));  // NaN ignored, like f32::max
      }
  }
  return amax;
}

template <int MODE, int FM, int FN, int KS, int STAGES>
__global__ __launch_bounds__(mid::kThreads) void gemm_mid_kernel(const int8_t* __restrict__ A,
                                                                 const int8_t* __restrict__ B, MidShape s,
                                                                 Epilogue ep) {
  using namespace mid;
  constexpr int TM = 16 * FM, TN = 16 * FN, WM = kWaves / KS, FW = FM / WM;
  constexpr int SB = 64 * KS, CH = SB / 16;       // bytes and 16-byte chunks per row and stage
  constexpr int RI = 1024 / SB;                   // rows per DMA instruction
  constexpr int IA = TM / RI / kWaves, IB = TN / RI / kWaves;  // instructions per wave and stage
  constexpr int ST = (TM + TN) * SB, LD = TN + 4;
  static_assert(FW * WM == FM && IA * RI * kWaves == TM, "split of A");
  static_assert(IB * RI * kWaves == TN, "split of B");
  constexpr int NI = IA + IB;
  constexpr int RED = KS * TM * LD * 4, RING = STAGES * ST;
  constexpr int SCALE = RING > RED ? RING : RED;  // byte offset of the scale product
  __shared__ __attribute__((aligned(1024))) int8_t smem[SCALE + 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ksub = wave % KS, wm = wave / KS;
  // Workgroups of one XCD (dealt round-robin) take a contiguous run of tiles,
  // rows fastest: a column strip of B is read from memory by one XCD.
  const int total = s.tiles_m * s.tiles_n;
  const int xcd = (int)blockIdx.x & 7, q = total >> 3, rem = total & 7;
  const int t = (xcd < rem ? xcd * (q + 1) : rem * (q + 1) + (xcd - rem) * q) + ((int)blockIdx.x >> 3);
  const int tn = t / s.tiles_m, tm = t - tn * s.tiles_m;
  const int m0 = tm * TM, n0 = tn * TN;
  // The epilogue's operands (bias is padded to whole tiles) arrive during the K loop.
  const v4f bias = *reinterpret_cast<const v4f*>(ep.bias + n0 + (tid % (TN / 4)) * 4);
  uint32_t part = 0;
  // one wave reads the slot: 64 lines that every workgroup reads
  if (MODE == kModeI8 && wave == 0) part = tensor_absmax_part(ep.absmax_in);
  const __amdgpu_buffer_rsrc_t ra = bounded_rsrc(A + (int64_t)m0 * s.lda);
  const __amdgpu_buffer_rsrc_t rb = bounded_rsrc(B + (int64_t)n0 * s.kb);
  // DMA instruction j = i * 8 + wave fills rows [j RI, (j + 1) RI) of the
  // stage (A's rows, then B's); lane l its row's chunk slot l % CH.
  const int lr = lane / CH, lc = lane % CH;
  uint32_t base[NI], kk[NI], lim[NI];
#pragma unroll
  for (int i = 0; i < NI; i++) {
    const int r = (i * kWaves + wave) * RI + lr;
    const bool is_a = i < IA;
    const int rr = is_a ? r : r - TM;
    kk[i] = (uint32_t)((lc ^ (r & 15)) * 16);
    const bool ok = is_a ? m0 + rr < s.M : n0 + rr < s.N;
    base[i] = is_a ? (uint32_t)(rr * (int32_t)s.lda) : (uint32_t)(rr * s.kb);
    lim[i] = ok ? (uint32_t)(is_a ? s.ka : s.kb) : 0u;
  }
  const int nst = (s.kb + SB - 1) / SB;
  auto issue = [&](int st, int slot) {
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const uint32_t k = kk[i] + (uint32_t)(st * SB);
      const uint32_t off = k < lim[i] ? base[i] + k : kDropOffset;
      int8_t* const dst = smem + slot * ST + (i * kWaves + wave) * 1024;
      if (i < IA)
        dma16_buf(ra, dst, off);
      else
        dma16_buf(rb, dst, off);
    }
  };
  // An f32 sum rounds at every step, so long chains lose what the GEMV's and the
  // split tiles' short ones did not: s.run stages are summed from zero (FP32:
  // the even and odd halves of a chunk apart), then join a total; the waves'
  // totals meet pairwise.  Against 64 bits: FP32 1000 x 1024 x 10 in runs of 8
  // stages 1.6e-7, now 9.9e-8 (one row per wave 1.0e-7), 3 x 4096 x 14336 1.64e-7
  // and 1.22e-7 (GEMV 1.61e-7); FP16 outputs that are not the rounded exact sum,
  // per mille, as one chain per wave and now: 100 x 4096 x 256 1.10 and 0.66 (split
  // K 0.75), 5 x 14336 x 4096 2.2 and 0.8 (GEMV 1.7).  A FP16 run's first stage
  // starts from zero instead of clearing acc (1000 x 1024 x 1024: 6.9 us as one
  // chain, 7.2; 7.7 with clears).
  constexpr bool TOTAL = MODE != kModeI8;
  constexpr int NA = MODE == kModeF32 ? 2 : 1;
  v4f tot[TOTAL ? FW : 1][TOTAL ? FN : 1] = {};
  v4i acc[NA][FW][FN];
#pragma unroll
  for (int a = 0; a < NA; a++)
#pragma unroll
    for (int i = 0; i < FW; i++)
#pragma unroll
      for (int j = 0; j < FN; j++) acc[a][i][j] = v4i{0, 0, 0, 0};
  const uint32_t rd = (uint32_t)((lane & 15) * SB + (((ksub * 4 + (lane >> 4)) ^ (lane & 15)) << 4));
  const uint32_t rda = rd + (uint32_t)(wm * FW * 16 * SB), rdb = rd + (uint32_t)(TM * SB);
#pragma unroll
  for (int p = 0; p < STAGES - 1; p++) issue(p, p);  // stages past the last load nothing
  int slot_rd = 0, slot_is = STAGES - 1;
  // Stage st's products onto acc, or from zero with `first`.
  auto stage = [&](int st, auto first) {
    wait_vmcnt<(STAGES - 2) * NI>();  // this wave's copies of stage st have landed
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(st + STAGES - 1, slot_is);
    const int8_t* const sp = smem + slot_rd * ST;
    v4i bf[FN], af[FW];
#pragma unroll
    for (int j = 0; j < FN; j++) bf[j] = *reinterpret_cast<const v4i*>(sp + rdb + j * 16 * SB);
#pragma unroll
    for (int i = 0; i < FW; i++) af[i] = *reinterpret_cast<const v4i*>(sp + rda + i * 16 * SB);
#pragma unroll
    for (int c = 0; c < (MODE == kModeF32 ? 4 : 1); c++)
#pragma unroll
      for (int i = 0; i < FW; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) {
          v4i& a = acc[c & (NA - 1)][i][j];
          const v4i from = first.value && c < NA ? v4i{0, 0, 0, 0} : a;
          if constexpr (MODE == kModeF32) {
            const v4f fa = __builtin_bit_cast(v4f, af[i]), fb = __builtin_bit_cast(v4f, bf[j]);
            a = __builtin_bit_cast(
                v4i, __builtin_amdgcn_mfma_f32_16x16x4f32(fa[c], fb[c], __builtin_bit_cast(v4f, from), 0, 0, 0));
          } else {
            a = mma_block<MODE>(af[i], bf[j], from);
          }
        }
    slot_rd = slot_rd == STAGES - 1 ? 0 : slot_rd + 1;
    slot_is = slot_is == STAGES - 1 ? 0 : slot_is + 1;
  };
  auto add_run = [&](auto zero) {
#pragma unroll
    for (int i = 0; i < FW; i++)
#pragma unroll
      for (int j = 0; j < FN; j++) {
        v4f sum = __builtin_bit_cast(v4f, acc[0][i][j]);
        if constexpr (NA == 2) sum += __builtin_bit_cast(v4f, acc[1][i][j]);
        tot[i][j] += sum;
        if constexpr (zero.value) acc[0][i][j] = acc[NA - 1][i][j] = v4i{0, 0, 0, 0};
      }
  };
  if constexpr (MODE == kModeF16) {
    for (int st = 0; st < nst;) {
      const int end = min(st + s.run, nst);
      stage(st, std::true_type{});
      for (st++; st < end; st++) stage(st, std::false_type{});
      add_run(std::false_type{});
    }
  } else {  // FP32 has no registers for a second form of its stage
    int left = s.run;
    for (int st = 0; st < nst; st++) {
      stage(st, std::false_type{});
      if (MODE == kModeF32 && --left == 0) {
        add_run(std::true_type{});
        left = s.run;
      }
    }
    if constexpr (MODE == kModeF32) add_run(std::false_type{});
  }
  // every copy has landed and every wave has read its last fragments: the
  // ring's memory takes the partial tiles
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int32_t* const red = reinterpret_cast<int32_t*>(smem);
#pragma unroll
  for (int i = 0; i < FW; i++)
#pragma unroll
    for (int j = 0; j < FN; j++) {
      v4i sum = acc[0][i][j];
      if constexpr (TOTAL) sum = __builtin_bit_cast(v4i, tot[i][j]);
#pragma unroll
      for (int e = 0; e < 4; e++)
        red[(ksub * TM + (wm * FW + i) * 16 + 4 * (lane >> 4) + e) * LD + j * 16 + (lane & 15)] = sum[e];
    }
  float* const scale = reinterpret_cast<float*>(smem + SCALE);
  if (MODE == kModeI8 && wave == 0) {
    const float cs0 = rgmath::scale_from_absmax(rgmath::bitsf(wave_max_u32(part))) * ep.w_scale;
    if (lane == 0) *scale = cs0;
  }
  __syncthreads();
  const float cs = MODE == kModeI8 ? *scale : 1.0f;
  float amax = 0.0f;
#define RG_MID_EPI(ACTV) mid_epilogue<MODE, ACTV, TM, TN, KS>(red, s, ep, cs, m0, n0, bias)
  switch (ep.act) {
    case rgmath::ACT_RELU: amax = RG_MID_EPI(rgmath::ACT_RELU); break;
    case rgmath::ACT_SIGMOID: amax = RG_MID_EPI(rgmath::ACT_SIGMOID); break;
    case rgmath::ACT_TANH: amax = RG_MID_EPI(rgmath::ACT_TANH); break;
    case rgmath::ACT_GELU: amax = RG_MID_EPI(rgmath::ACT_GELU); break;
    case rgmath::ACT_LEAKY_RELU: amax = RG_MID_EPI(rgmath::ACT_LEAKY_RELU); break;
    case rgmath::ACT_SILU: amax = RG_MID_EPI(rgmath::ACT_SILU); break;
    default: amax = RG_MID_EPI(rgmath::ACT_NONE); break;
  }
#undef RG_MID_EPI
  if (MODE == kModeI8 && ep.absmax_out) {
    // one atomic per workgroup into its partial of the spread slot
    const uint32_t mw = wave_max_u32(rgmath::fbits(amax));
    __syncthreads();  // the partial tiles have been read
    if (lane == 0) red[wave] = (int32_t)mw;
    __syncthreads();
    if (tid == 0) {
      uint32_t m = 0;
#pragma unroll
      for (int w = 0; w < kWaves; w++) m = (uint32_t)red[w] > m ? (uint32_t)red[w] : m;
      if (m) atomicMax(ep.absmax_out + (blockIdx.x & (kSpread - 1)) * kSpreadStride, m);
    }
  }
}

// The tile shapes.
struct MidTile {
  int tm, tn;
};
static constexpr MidTile kMidTiles[] = {{16, 16}, {16, 32}, {16, 64}, {32, 32}, {64, 32},
                                        {32, 64}, {64, 64}, {128, 64}, {64, 128}};
static_assert(sizeof kMidTiles / sizeof kMidTiles[0] == kMidTileCount, "tile indexes");

// Rounds of one workgroup on each of the 256 CUs (a workgroup's LDS leaves
// room for no second one).
static int64_t mid_rounds(const MidTile& t, int64_t M, int64_t N) {
  return (((M + t.tm - 1) / t.tm) * ((N + t.tn - 1) / t.tn) + 255) / 256;
}

// A grid holds fewer than 2^32 threads (an operand's zero columns may take one
// more column of tiles).
static bool mid_grid_fits(const MidTile& t, int64_t M, int64_t N) {
  return ((M + t.tm - 1) / t.tm) * ((N + t.tn - 1) / t.tn + 1) * mid::kThreads < (int64_t(1) << 32);
}

// The tile with the least estimated time: a CU's K blocks at 40 bytes a clock
// of loads or one MFMA every 16 clocks per SIMD, whichever is more, over the
// rounds of one workgroup per CU, plus 1 us a round and 2.5 us a launch.  FP32
// takes an MFMA's 32 clocks and the loads one after the other, and its rounds end
// with more partial sums to write (4096 x 4096, us per round, estimated and
// measured: 16 x 16 10.0 and 10.2, 32 x 32 26 and 26, 64 x 64 79 and 81, 128 x 64
// 147 and 146).  Over 27 shapes (9 to 2000 rows, each precision) the tile it takes
// was the fastest of the nine or within 6% of it; of 87 FP32 shapes (200 to 8192
// rows) it and gemm_f32_us together took the fastest kernel or one within 1% on
// average, 14% at most.
int mid_choice(int mode, int64_t M, int64_t N, int64_t kb, double* us) {
  int best = -1;
  double best_us = 0.0;
  for (int i = 0; i < kMidTileCount; i++) {
    const MidTile& t = kMidTiles[i];
    if (!mid_grid_fits(t, M, N)) continue;
    const double rounds = (double)mid_rounds(t, M, N), steps = (double)(kb / 64);
    const double load = steps * (t.tm + t.tn) * 64.0 / 40.0;
    const double mfma = steps * (t.tm / 16) * (t.tn / 16) * (mode == kModeF32 ? 128.0 : 16.0) / 4.0;
    const double work = mode == kModeF32 ? load + mfma + t.tm * t.tn : load > mfma ? load : mfma;
    const double c = 2.5 + rounds * (1.0 + work / 2400.0);
    if (best < 0 || c < best_us) {
      best = i;
      best_us = c;
    }
  }
  if (us) *us = best_us;
  return best < 0 ? 0 : best;
}

bool gemm_mid_supported(int64_t M, int64_t N, int64_t lda, int64_t kb) {
  // 32-bit offsets within a tile's rows, 32-bit sizes
  return M > 0 && N > 0 && M < (int64_t(1) << 31) - 256 && N < (int64_t(1) << 31) - 256 && kb > 0 && kb % 64 == 0 &&
         lda % 16 == 0 && 128 * lda < (int64_t(1) << 31) && 128 * kb < (int64_t(1) << 31) &&
         (mid_grid_fits({128, 64}, M, N) || mid_grid_fits({64, 128}, M, N));
}

template <int MODE, int FM, int FN, int KS, int STAGES>
static void launch_mid_t(const int8_t* A, const int8_t* B, MidShape s, const Epilogue& ep, hipStream_t st) {
  s.tiles_m = (s.M + 16 * FM - 1) / (16 * FM);
  const int64_t cols = ep.h_out && ep.ldh > s.N ? ep.ldh : s.N;  // the operand's zero columns too
  s.tiles_n = (int32_t)((cols + 16 * FN - 1) / (16 * FN));
  // Wide FP32 layers: 8 stages, more of them a total's addition; where the
  // GEMV or the one-row-per-wave heads summed in shorter chains, the best.
  const int64_t stages = (s.kb + 64 * KS - 1) / (64 * KS);
  s.run = MODE == kModeF16 ? sum_run(stages, 3) : s.N <= kNarrowMaxN || s.M <= 8 ? sum_run(stages, 10) : 8;
  RG_LAUNCH((gemm_mid_kernel<MODE, FM, FN, KS, STAGES>), dim3((unsigned)((int64_t)s.tiles_m * s.tiles_n)),
            dim3(mid::kThreads), 0, st, A, B, s, ep);
}

template <int MODE>
static void launch_mid_mode(const int8_t* A, int64_t lda, int64_t ka, const int8_t* B, int64_t M, int64_t N, int64_t kb,
                            int tile, const Epilogue& ep, hipStream_t st) {
  if (!gemm_mid_supported(M, N, lda, kb) || ka > kb || ka % 16 || (reinterpret_cast<uintptr_t>(A) & 15))
    throw std::logic_error("mid GEMM: unsupported shape or unaligned operand");
  if (ep.h_out && (ep.ldh % 4 || MODE != kModeF16)) throw std::logic_error("mid GEMM: operand hand-off is FP16 only");
  const MidShape s{lda,        (int32_t)ka, (int32_t)kb, (int32_t)M,
                   (int32_t)N, 0,           0,           N % 4 == 0 && (reinterpret_cast<uintptr_t>(ep.y) & 15) == 0,
                   1};
  switch (tile) {
    case 0: launch_mid_t<MODE, 1, 1, 8, 6>(A, B, s, ep, st); break;
    case 1: launch_mid_t<MODE, 1, 2, 8, 5>(A, B, s, ep, st); break;
    case 2: launch_mid_t<MODE, 1, 4, 8, 3>(A, B, s, ep, st); break;
    case 3: launch_mid_t<MODE, 2, 2, 4, 6>(A, B, s, ep, st); break;
    case 4: launch_mid_t<MODE, 4, 2, 4, 5>(A, B, s, ep, st); break;
    case 5: launch_mid_t<MODE, 2, 4, 4, 5>(A, B, s, ep, st); break;
    case 6: launch_mid_t<MODE, 4, 4, 4, 4>(A, B, s, ep, st); break;
    case 7: launch_mid_t<MODE, 8, 4, 4, 3>(A, B, s, ep, st); break;
    default: launch_mid_t<MODE, 4, 8, 4, 3>(A, B, s, ep, st); break;
  }
}

void launch_gemm_mid(const int8_t* A, const int8_t* B, int64_t M, int64_t N, int64_t Kpad, int tile,
                     const Epilogue& ep, hipStream_t s) {
  if (!ep.absmax_in) throw std::logic_error("mid GEMM: no absmax slot");
  launch_mid_mode<kModeI8>(A, Kpad, Kpad, B, M, N, Kpad, tile, ep, s);
}

void launch_gemm_mid_f16(const uint16_t* A, const uint16_t* B, int64_t M, int64_t N, int64_t Kpad_h,
                         int tile, const Epilogue& ep, hipStream_t s) {
  launch_mid_mode<kModeF16>(reinterpret_cast<const int8_t*>(A), 2 * Kpad_h, 2 * Kpad_h,
                            reinterpret_cast<const int8_t*>(B), M, N, 2 * Kpad_h, tile, ep, s);
}

void launch_gemm_mid_f32(const float* A, int64_t lda, int64_t K, const float* B, int64_t M, int64_t N, int64_t Kpad_f,
                         int tile, const Epilogue& ep, hipStream_t s) {
  launch_mid_mode<kModeF32>(reinterpret_cast<const int8_t*>(A), 4 * lda, 4 * K, reinterpret_cast<const int8_t*>(B), M,
                            N, 4 * Kpad_f, tile, ep, s);
}

// This translation unit's code object, loaded at program creation.
__global__ void mid_load_probe_kernel() {}

void load_mid_code_object(hipStream_t s) { hipLaunchKernelGGL(mid_load_probe_kernel, dim3(1), dim3(64), 0, s); }

}  // namespace rgnpu
