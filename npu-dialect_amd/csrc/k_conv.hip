// k_conv.hip -- group `pad -> fill -> conv_2d_nhwc_fhwc -> generic(bias, act)`.
//
// Implicit GEMM on MFMA: rows = output pixels (n, oh, ow), columns = filters
// f, reduction = (kh, kw, c).  NHWC activations and FHWC filters both keep
// the channel dimension contiguous, so every lane's MFMA operand is one
// 16-byte run of channels of one pixel (A) or one filter (B) -- no transpose
// and no im2col buffer.  tensor.pad (test/conv2d_relu.mlir:13-16) is not
// materialised: out-of-image taps load zeros (predicated halo loads).  The
// spatial split the reference picks over Co (test/lit/spatial_tiling_conv2d.mlir:28-34)
// becomes the grid's y dimension; the pixel dimension is the grid's x.
//
// A workgroup of 2 x 2 waves owns BM pixels x BN filters.  The reduction walks
// the taps and, within a tap, chunks of 128 bytes of channels (or, for few
// channels, the 16-byte runs of all taps one after the other); per step the
// pixels' runs (zero outside the image and past C) and the filters' runs are
// staged in LDS, double-buffered, the next two steps' loads in flight while
// the current one is multiplied, one barrier per step.  The filter fragment is
// the MFMA's first operand where F is a multiple of 4, so a lane ends with four
// consecutive filters of one pixel: the epilogue (bias add, residual add, act,
// and the bf16 rounding of the bf16 variant) runs on the accumulators and stores
// 8 or 16 bytes.
// C need not be a multiple of an MFMA fragment's 16 (f32) or 32 (bf16)
// channels: a 16-byte run past C is staged as zero.  F need not be a multiple
// of 16 either: filters past F read filter F - 1 and are not stored.
#include "kernels.hpp"
#include "npu_device.hpp"
#include "persistent.hpp"
#include "plans.hpp"

namespace npu {

namespace {

// How the steps of 128 bytes of a filter walk the reduction: a tap's channels in
// chunks, the last one zero past C; the 16-byte runs of all taps one after the
// other; or the runs of one step.
enum class Walk { kTapChunks, kRuns, kOneStep };
constexpr const char *kWalkName[] = {"conv2d_nhwc", "conv2d_nhwc_runs", "conv2d_nhwc_one_step"};

struct ConvTileArgs {
  const void *x, *w, *res;
  const float *bias;
  void *out;
  int H, W, C, F, KW, taps, pad, Ho, Wo, act, P, npt, nft;
  int runs;              // 16-byte runs of a filter
  FastDiv by_run, by_kw;  // runs of a tap, filter columns
};

template <class MM, typename T, int BM, int BN, bool VEC, Walk WALK>
__global__ __launch_bounds__(256, 2) void conv2d_nhwc_kernel(const ConvTileArgs a) {
  constexpr int ES = sizeof(T), RUN = 16 / ES;        // elements of a 16-byte run
  constexpr int KC = 128 / ES;                        // channels of a step
  constexpr int REC = 128 + 32;                       // LDS row: 32 mod 64 bytes
  constexpr int TM = BM / 32, TN = BN / 32;           // 16 x 16 blocks of a wave
  constexpr int AR = BM / 32, BR = BN / 32;           // runs per thread and step
  constexpr int BUF = (BM + BN) * REC;
  constexpr bool FLAT = WALK != Walk::kTapChunks;
  constexpr int SETS = WALK == Walk::kOneStep ? 1 : 2;  // register sets and LDS buffers
  __shared__ __attribute__((aligned(16))) unsigned char lds[SETS * BUF];
  const int per = gridDim.x / kXcds, t = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
  if (t >= a.npt * a.nft) return;
  const int pt = t / a.nft, ft = t - pt * a.nft;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int wp = wave & 1, wf = wave >> 1;
  const int p0 = pt * BM, f0 = ft * BN;
  const T *const x = static_cast<const T *>(a.x);
  const T *const w = static_cast<const T *>(a.w);

  // staging: this thread's 16-byte run `seg` of rows tid / 8 + 32 i.  Offsets
  // are 32-bit words from the tensors' bases (an operand has less than 2^31
  // elements): a lane part that is fixed for the launch plus a step part that
  // is uniform, so a load's address is one vector addition.  us, with 64-bit
  // products of the coordinates instead / so: bf16 28x28x128 batch 32 21.8 /
  // 21.1, 7x7x512 33.9 / 32.2, 5x5 30x30x64 batch 2 9.56 / 9.27.
  const int seg = tid & 7, row0 = tid >> 3;
  int abase[AR], aoh[AR], aow[AR], bbase[BR];
#pragma unroll
  for (int i = 0; i < AR; ++i) {
    const int p = min(p0 + row0 + 32 * i, a.P - 1);
    const int n = p / (a.Ho * a.Wo), rem = p - n * a.Ho * a.Wo;
    const int oh = rem / a.Wo;
    aoh[i] = oh - a.pad;
    aow[i] = rem - oh * a.Wo - a.pad;
    abase[i] = ((n * a.H + aoh[i]) * a.W + aow[i]) * a.C;
  }
#pragma unroll
  for (int i = 0; i < BR; ++i) bbase[i] = min(f0 + row0 + 32 * i, a.F - 1) * a.taps * a.C;
  // Loads from clamped addresses now, zeros chosen when the runs are written
  // (a select on a loaded value would make the wave wait for it there).
  u32x4 av[SETS][AR], bv[SETS][BR];
  uint32_t keep[SETS];
  // run g of a filter is run g % by_run.d of tap g / by_run.d: the lanes of a
  // step may be on different taps
  auto fetch_flat = [&](int set, int step) __attribute__((always_inline)) {
    const int g = step * 8 + seg;
    const bool cin = g < a.runs;
    const int gc = cin ? g : 0, tap = a.by_run.div(gc), kh = a.by_kw.div(tap), kw = tap - kh * a.KW;
    const int xoff = (kh * a.W + kw) * a.C + (gc - tap * (int)a.by_run.d) * RUN;
    keep[set] = (uint32_t)cin << AR;
#pragma unroll
    for (int i = 0; i < AR; ++i) {
      const bool in = (unsigned)(aoh[i] + kh) < (unsigned)a.H && (unsigned)(aow[i] + kw) < (unsigned)a.W;
      av[set][i] = *reinterpret_cast<const u32x4 *>(x + (uint32_t)(in ? abase[i] + xoff : 0));
      keep[set] |= (uint32_t)(in && cin) << i;
    }
#pragma unroll
    for (int i = 0; i < BR; ++i)
      bv[set][i] = *reinterpret_cast<const u32x4 *>(w + (uint32_t)(bbase[i] + gc * RUN));
  };
  auto fetch = [&](int set, int kh, int kw, int c0) __attribute__((always_inline)) {
    const bool cin = c0 + seg * RUN < a.C;
    const int lc = cin ? seg * RUN : 0;
    const int xoff = (kh * a.W + kw) * a.C + c0, woff = (kh * a.KW + kw) * a.C + c0;
    keep[set] = (uint32_t)cin << AR;
#pragma unroll
    for (int i = 0; i < AR; ++i) {
      const bool in = (unsigned)(aoh[i] + kh) < (unsigned)a.H && (unsigned)(aow[i] + kw) < (unsigned)a.W;
      av[set][i] = *reinterpret_cast<const u32x4 *>(x + (uint32_t)(in ? abase[i] + xoff + lc : 0));
      keep[set] |= (uint32_t)(in && cin) << i;
    }
#pragma unroll
    for (int i = 0; i < BR; ++i)
      bv[set][i] = *reinterpret_cast<const u32x4 *>(w + (uint32_t)(bbase[i] + woff + lc));
  };
  unsigned char *const dst = lds + row0 * REC + seg * 16;
  auto commit = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AR; ++i)
      *reinterpret_cast<u32x4 *>(dst + buf * BUF + 32 * i * REC) = masked(av[buf][i], (keep[buf] >> i) & 1u);
#pragma unroll
    for (int i = 0; i < BR; ++i)
      *reinterpret_cast<u32x4 *>(dst + buf * BUF + (BM + 32 * i) * REC) = masked(bv[buf][i], (keep[buf] >> AR) & 1u);
  };

  typename MM::acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = typename MM::acc_t{0, 0, 0, 0};

  // steps in order (kh, kw, channel chunk); the coordinates of the step being
  // fetched run ahead, and stay in the last filter row past the end
  const int chunks = (a.C + KC - 1) / KC, KH = a.taps / a.KW;
  const int steps = FLAT ? (a.runs + 7) / 8 : a.taps * chunks;
  int kh = 0, kw = 0, ch = 0, fstep = 0;
  auto advance = [&]() __attribute__((always_inline)) {
    if (++ch == chunks) {
      ch = 0;
      if (++kw == a.KW) kw = 0, kh = min(kh + 1, KH - 1);
    }
  };
  const unsigned char *const arow = lds + (wp * (BM / 2) + r) * REC + q * 16;
  const unsigned char *const brow = lds + (BM + wf * (BN / 2) + r) * REC + q * 16;
  int mch = 0;  // channel chunk (FLAT: index) of the step being multiplied
  auto multiply = [&](int buf) __attribute__((always_inline)) {
    const int off = buf * BUF;
    const int frags = min(2, FLAT ? (a.runs - mch * 8 + 3) / 4 : (a.C - mch * KC + KC / 2 - 1) / (KC / 2));
    if (++mch == chunks && !FLAT) mch = 0;
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      if (f < frags) {  // uniform: the last chunk's second half may lie past C
        Frag16 af[TM], bf[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) af[i].u = *reinterpret_cast<const u32x4 *>(arow + off + 16 * i * REC + 64 * f);
#pragma unroll
        for (int j = 0; j < TN; ++j) bf[j].u = *reinterpret_cast<const u32x4 *>(brow + off + 16 * j * REC + 64 * f);
#pragma unroll
        for (int st = 0; st < MM::kSteps; ++st)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) VEC ? MM::step(acc[i][j], bf[j], af[i], st) : MM::step(acc[i][j], af[i], bf[j], st);
      }
    }
  };
  auto fetch_next = [&](int set) __attribute__((always_inline)) {
    if constexpr (FLAT) {
      fetch_flat(set, fstep++);
    } else {
      fetch(set, kh, kw, ch * KC);
      advance();
    }
  };
  // Step s is in buffer s % 2 and passed through register set s % 2: its loads
  // are issued two steps before they are committed (a step's MFMAs take less
  // time than a load from L2; us with one step / two: bf16 7x7x512 batch 32
  // 35.5 / 33.4, 28x28x128 batch 4 8.6 / 8.05, 5x5 30x30x64 batch 2 10.4 /
  // 9.55, f32 14x14x256 97 / 90; with more workgroups per CU, 28x28x128 batch
  // 32, the fragments' LDS reads bound it and it stays at 21.8).  Past the last step the
  // loads stay inside the filter's last row and are never committed.
  if constexpr (WALK == Walk::kOneStep) {
    fetch_next(0);
    commit(0);
    __syncthreads();
    multiply(0);
  } else {
    fetch_next(0);
    fetch_next(1);
    commit(0);
    fetch_next(0);
    __syncthreads();
    int s = 0;
    for (; s + 2 < steps; s += 2) {
      multiply(0);
      commit(1);
      fetch_next(1);
      __syncthreads();
      multiply(1);
      commit(0);
      fetch_next(0);
      __syncthreads();
    }
    multiply(0);
    if (s + 1 < steps) {
      commit(1);
      __syncthreads();
      multiply(1);
    }
  }

  // Epilogue: pixel r of each block, its filters 4q .. +3.
  const ActBounds ab = act_bounds(a.act);
  const T *const res = static_cast<const T *>(a.res);
  T *const out = static_cast<T *>(a.out);
  if constexpr (!VEC) {
    // pixels 4q .. +3 of each block, its filter r: sixteen lanes on
    // consecutive filters.  us, lanes on four filters of a pixel / so: bf16
    // 1x1 34x35x16 -> 481 with residual at batch 13 27.2 / 17.4.
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int f = f0 + wf * (BN / 2) + 16 * j + r;
      if (f >= a.F) continue;
      const float bj = a.bias ? a.bias[f] : 0.0f;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int p = p0 + wp * (BM / 2) + 16 * i + 4 * q + e;
          if (p >= a.P) continue;
          const size_t o = (size_t)p * a.F + f;
          const float v = acc[i][j][e] + bj;
          if constexpr (sizeof(T) == 4) out[o] = act_clamp(res ? v + res[o] : v, ab);
          else out[o] = f32_to_bf16(act_clamp(res ? v + bf16_to_f32(res[o]) : v, ab));
        }
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int f = f0 + wf * (BN / 2) + 16 * j + 4 * q;
    f32x4 bj = {0.f, 0.f, 0.f, 0.f};
    if (a.bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) bj[e] = a.bias[min(f + e, a.F - 1)];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int p = p0 + wp * (BM / 2) + 16 * i + r;
      if (p >= a.P || f >= a.F) continue;
      const size_t o = (size_t)p * a.F + f;
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[i][j][e] + bj[e];
      if constexpr (sizeof(T) == 4) {
        if (res) v += *reinterpret_cast<const f32x4 *>(res + o);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = act_clamp(v[e], ab);
        *reinterpret_cast<f32x4 *>(out + o) = v;
      } else {
        if (res) {
          const uint2 u = *reinterpret_cast<const uint2 *>(res + o);
          v[0] += __uint_as_float(u.x << 16);
          v[1] += __uint_as_float(u.x & 0xffff0000u);
          v[2] += __uint_as_float(u.y << 16);
          v[3] += __uint_as_float(u.y & 0xffff0000u);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = act_clamp(v[e], ab);
        *reinterpret_cast<uint2 *>(out + o) = make_uint2(cvt_pk_bf16(v[0], v[1]), cvt_pk_bf16(v[2], v[3]));
      }
    }
  }
}

template <class MM, typename T, int BM, int BN, bool VEC, Walk WALK>
hipError_t launch_tile(const ConvArgs &c, hipStream_t s) {
  auto kern = conv2d_nhwc_kernel<MM, T, BM, BN, VEC, WALK>;
  constexpr int RUN = 16 / sizeof(T);
  ConvTileArgs a{c.x, c.w, c.res, c.bias, c.out, c.H, c.W, c.C, c.F, c.KW, c.KH * c.KW, c.pad, c.Ho, c.Wo, c.act,
                 c.N * c.Ho * c.Wo, 0, 0, c.KH * c.KW * (c.C / RUN), FastDiv(c.C / RUN), FastDiv(c.KW)};
  a.npt = (a.P + BM - 1) / BM;
  a.nft = (a.F + BN - 1) / BN;
  const int G = a.npt * a.nft, grid = (G + kXcds - 1) / kXcds * kXcds;
  const double steps = WALK != Walk::kTapChunks ? (a.runs + 7) / 8 : (double)a.taps * ((a.C + 8 * RUN - 1) / (8 * RUN));
  npu_launch_plan p = make_plan(kWalkName[(int)WALK], G, wg_per_cu(kern), G, 8 * sizeof(T));
  p.load_phases = 1;  // a step's loads are in flight during the two before
  p.tile_macs = (double)BM * BN * steps * 128 / sizeof(T);
  p.tile_valu = 4.0 * (steps * (10.0 * (BM + BN) / 32 + 20.0) + 12.0 * BM * BN / 1024 + 120.0);
  p.tile_lds_bytes = steps * (128.0 * (BM + BN) + 4.0 * 2 * 1024 * (BM + BN) / 32);
  p.tile_load_bytes = steps * 128.0 * (BM + BN);
  p.tile_store_bytes = (double)BM * BN * sizeof(T);
  p.hbm_bytes = (double)sizeof(T) * ((double)c.N * c.H * c.W * c.C + (double)c.F * c.KH * c.KW * c.C +
                                     (double)a.P * c.F * (c.res ? 2 : 1)) + (c.bias ? 4.0 * c.F : 0.0);
  plans_add(p);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, a);
  return hipGetLastError();
}

template <class MM, typename T, int BM, int BN, Walk WALK>
hipError_t launch_tile(const ConvArgs &c, hipStream_t s) {
  return c.F % 4 == 0 ? launch_tile<MM, T, BM, BN, true, WALK>(c, s) : launch_tile<MM, T, BM, BN, false, WALK>(c, s);
}

// The walk over runs where it saves a quarter of the steps, which are mostly
// padding for few channels; filters of a single step load and stage it once, in
// one LDS buffer (twice the workgroups on a CU).  Measured, us, the kernel before
// the tiles (operands straight from L2) / tap chunks / so: bf16 5x5 34x35x8 ->
// 267 at batch 13 25.2 / 37.5 / 13.3, 5x5 40x41x16 -> 267 batch 3 15.2 / 17.7 /
// 8.8, 3x3 34x35x32 -> 481 batch 13 26.9 / 25.9 / 20.6; f32 5x5 34x35x16 -> 64 19.8 /
// 18.7 / 14.7; one step: bf16 1x1 34x35x16 -> 481 12.1 / 14.2 / 11.0, f32 1x1
// 34x35x8 -> 267 10.7 / 11.9 / 10.2.
template <class MM, typename T, int BM, int BN>
hipError_t launch_tile(const ConvArgs &c, hipStream_t s) {
  const long long run = c.C * (long long)sizeof(T) / 16, taps = (long long)c.KH * c.KW, runs = taps * run;
  if (runs <= 8) return launch_tile<MM, T, BM, BN, Walk::kOneStep>(c, s);
  // (run and runs within FastDiv's range)
  if (run < 64 && runs < 60000 && 4 * ((runs + 7) / 8) <= 3 * taps * ((run + 7) / 8))
    return launch_tile<MM, T, BM, BN, Walk::kRuns>(c, s);
  return launch_tile<MM, T, BM, BN, Walk::kTapChunks>(c, s);
}

// Tiles of 64 pixels x 64 filters when there are enough to keep more than one
// workgroup on a CU, with 32 filters where 64 would compute a tenth more
// padding; then 64 x 32; then 32 x 32.  Measured, us, as 64x64 / 64x32 / 32x32
// (workgroups of the first), against the kernel before (operands straight from
// L2): bf16 3x3 28x28x128 at batch 32 (784) 22.7 / 27.7 / 28.9, before 71.3;
// 14x14x256 (392) 26.2 / 30.1 / 30.6, before 70.5; 7x7x512 (200) 40.9 / 38.2 /
// 36.9, before 70.0; 28x28x128 at batch 4 (98) 12.1 / 10.4 / 9.3, before 21.7;
// 1x1 68x67x80 -> 150 at batch 11 (2376) 31.4 / 27.3 / 29.2, before 29.7; f32
// 1x1 56x56x64 -> 256 at batch 32 (6272) 60.9 / 62.5 / 67.8, before 93.6.
// Tiles of 128 pixels or filters were slower (fewer workgroups per CU).
constexpr long long kMinTiles = 384;

template <class MM, typename T>
hipError_t launch_conv(const ConvArgs &a, hipStream_t s) {
  const long long pt = ((long long)a.N * a.Ho * a.Wo + 63) / 64;
  const int f64 = (a.F + 63) / 64, f32 = (a.F + 31) / 32;
  if (pt * f64 >= kMinTiles && 2 * f64 * 10 <= f32 * 11) return launch_tile<MM, T, 64, 64>(a, s);
  if (pt * f32 >= kMinTiles) return launch_tile<MM, T, 64, 32>(a, s);
  return launch_tile<MM, T, 32, 32>(a, s);
}

}  // namespace

hipError_t launch_conv2d_nhwc_f32(const ConvArgs &a, hipStream_t s) {
  return launch_conv<MfmaF32, float>(a, s);
}
hipError_t launch_conv2d_nhwc_bf16(const ConvArgs &a, hipStream_t s) {
  return launch_conv<MfmaBF16, uint16_t>(a, s);
}

}  // namespace npu
