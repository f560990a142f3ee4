// k_conv_nchw.hip -- the reference's own conv group kind:
// `fill -> conv_2d_nchw_fchw -> generic...`, outlined as
// @fused_fill_conv2d_generic[_generic]_<idx> (test/conv2d_relu.mlir:7-42,
// test/resnet_block.mlir, test/resnet50_block.mlir, test/mobilenet_block.mlir;
// lib/Transforms/OutlineFusedGroupsPass.cpp:69-82).  NCHW activations, FCHW
// filters, any stride, the feeding tensor.pad folded into the halo loads and the
// layout kept on both sides: no transposed copy of either tensor in HBM.
//
// Implicit GEMM on the f32 MFMA: rows = output pixels, columns = filters,
// reduction k = (c, kh, kw) in FCHW order, so a filter's operand is its own
// row, loaded 16 bytes per lane straight into registers, and any filter size
// and stride run the same code.  A workgroup owns 16 NB pixels x 16 WF filters
// and splits K over WK groups of its waves: at batch 1 a layer has only 128 to
// 784 16x16 output blocks, so a workgroup per block with its waves along K is
// what fills the chip.  Per chunk of channels it stages the input patch its
// pixels see, zero outside the image (the folded tensor.pad); a table in LDS
// says where k lies in the patch, and lane (r, q) of MFMA step s reads pixel
// r's word of k = 16 step + 4q + s.  The K parts' sums meet in LDS and are
// finished with the bias, the residual and the activation, stored along the
// pixels.
//
// What bounds it: at batch 1 the patches' loads, one word per lane (about 28
// clocks of the CU's load path each), and the fetch of code that runs once;
// at larger batches the chain of a k step (its LDS reads, then its MFMAs: a
// third of the f32 matrix rate).  Measured against the
// kernel before it (row segments of 32 or 64 pixels x 64 filters, 16-channel
// chunks of halo and filters staged between two barriers): 3x3 at batch 1
// 56x56x64 31.7 -> 8.5 us, 28x28x128 57.6 -> 10.4, 14x14x256 110 -> 16,
// 7x7x512 215 -> 20, the 7x7/2 stem 31.7 -> 9.5; 56x56x64 at batch 8 with
// residual 84 -> 36 us, without 82 -> 34.
#include <cmath>
#include <type_traits>

#include "kernels.hpp"
#include "npu_device.hpp"
#include "persistent.hpp"
#include "plans.hpp"

namespace npu {

namespace {

struct NchwArgs {
  const float *x, *w, *bias, *res;
  float *out;
  int C, H, W, F, T, K, pad, st, Ho, Wo, act;
  int tw, nstrips;       // strip width, strips per image
  int tiles;             // pixel tiles per strip
  int npt, grid;         // pixel tiles of the launch, workgroups
  int hc, ps, npl;       // patch columns, patch words per channel, loads per channel
  int pstep, istep;      // between neighbouring pixels in the patch, patch words in the image
  int words;             // patch words past this are not loaded
  int cc, nchunks;       // channels per chunk
  FastDiv by_hc, by_tw, by_t, by_kw;
};

constexpr int kStage = 16;  // patch words a thread holds in flight per chunk
constexpr int kRing = 4;    // k steps whose filters a wave holds in flight
// LDS words between the patches of consecutive channels, for NPL loads of 64
// words each: 4 mod 64, so a 1x1 filter's four lane groups (channels 4 apart)
// read 16 banks apart.
constexpr int patch_stride(int npl) { return 64 * npl + 4; }

// An unaligned-by-16 run of four floats (filter rows of K % 4 != 0 words);
// global loads need 4-byte alignment only.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

template <int NB, int WF, int WK, int NPL>
__global__ __launch_bounds__(64 * WF * WK, WF * WK == 8 && NB * NPL <= 16 ? 4 : 2)
void conv2d_nchw_split_kernel(const NchwArgs a) {
  constexpr int NW = WF * WK, NT = 64 * NW, PX = 16 * NB;
  constexpr int CPW = kStage / NPL;  // channels a wave stages per chunk
  constexpr int PS = patch_stride(NPL);
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int KC = a.cc * a.T;                       // reduction length of a whole chunk
  const int KT = (KC + 15) & ~15;
  int *const ktab = reinterpret_cast<int *>(smem);             // byte offset of k in a patch
  float *const patch = reinterpret_cast<float *>(ktab + KT);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int wf = wave % WF, wk = wave / WF;
  // filter blocks outermost, cut into eight contiguous ranges, one per XCD:
  // the pixel tiles that read the same filters share an L2
  const int per = (a.grid + kXcds - 1) / kXcds, t0 = (blockIdx.x % kXcds) * per + blockIdx.x / kXcds;
  if (t0 >= a.grid) return;
  const int fb = t0 / a.npt, pt = t0 - fb * a.npt;
  const int strip = pt % a.nstrips, t1 = pt / a.nstrips;
  const int n = t1 / a.tiles, p0 = (t1 - n * a.tiles) * PX;
  const int ox0 = strip * a.tw, tw = min(a.tw, a.Wo - ox0);  // tw < a.tw: the last strip
  const int oy0 = a.by_tw.div(p0);
  const int f0 = (fb * WF + wf) * 16;

  // ---- filters: lane (r, q) holds filter r, k = 16 step + 4q .. +3, straight
  //      from its row of FCHW, in a ring of kRing steps.  Every load is
  //      unconditional (one under a branch, even a uniform one, makes the
  //      wave wait for it there).  A run that crosses the end of its row reads
  //      on into the next row; the last row's is moved back into the buffer.
  const int wrow = min(f0 + r, a.F - 1) * a.K + 4 * q, wlast = a.F * a.K - 4;
  auto load_w = [&](int k) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4u *>(a.w + min(wrow + k, wlast));
  };
  constexpr int KSTEP = 16 * WK;
  f32x4 wv[kRing];
  auto fill_ring = [&](int kbase) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kRing; ++u) wv[u] = load_w(min(kbase + 16 * wk + KSTEP * u, a.K));
  };
  fill_ring(0);

  // ---- staging: this wave's load (j, i) is patch words 64 i + lane of
  //      channel wave + NW j of the chunk.  A word's place in the plane does
  //      not depend on the channel, so a load is a uniform base plus a lane
  //      offset fixed for the whole launch.  Words outside the image load
  //      the plane's first word and are zeroed on commit.  Channels past C
  //      (the last chunk's) hold channel C - 1 again: their k are never used.
  int off[NPL];
  uint32_t keep = 0;
#pragma unroll
  for (int i = 0; i < NPL; ++i) {
    const int e = 64 * i + lane, hy = a.by_hc.div(e), hx = e - hy * a.hc;
    const int iy = oy0 * a.st - a.pad + __mul24(hy, a.istep), ix = ox0 * a.st - a.pad + __mul24(hx, a.istep);
    const bool in = e < a.words && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
    off[i] = in ? iy * a.W + ix : 0;
    keep |= (uint32_t)in << i;
  }
  const int plane = a.H * a.W;
  const float *const xn = a.x + (size_t)n * a.C * plane;
  float st[CPW][NPL];
  auto stage = [&](int c0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      const float *const xc = xn + min(c0 + wave + NW * j, a.C - 1) * plane;
#pragma unroll
      for (int i = 0; i < NPL; ++i) st[j][i] = xc[off[i]];
    }
  };
  auto commit = [&](float *buf) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
      if (wave + NW * j < a.cc) {
        float *const row = buf + (wave + NW * j) * PS + lane;
#pragma unroll
        for (int i = 0; i < NPL; ++i) row[64 * i] = (keep >> i) & 1u ? st[j][i] : 0.0f;
      }
    }
  };
  stage(0);

  // ---- the outputs this thread finishes, and their bias and residual: with
  //      few of them they are loaded here, so that the epilogue does not wait
  //      for memory once per output.  Outputs that do not exist, and operands
  //      that are absent, load the input's first word instead.
  constexpr int NE = (16 * WF * PX + NT - 1) / NT;  // outputs per thread
  constexpr bool PRE = NE <= 4;
  // output e (filter e / PX of the workgroup's, pixel e % PX): its index, or -1
  auto out_at = [&](int e, int &f) __attribute__((always_inline)) {
    const int px = e % PX, p = p0 + px, oy = a.by_tw.div(p), ox = p - oy * a.tw;
    f = fb * WF * 16 + e / PX;
    const bool ok = e < 16 * WF * PX && oy < a.Ho && ox < tw && f < a.F;
    return ok ? ((n * a.F + f) * a.Ho + oy) * a.Wo + ox0 + ox : -1;
  };
  float rv[PRE ? NE : 1], bv[PRE ? NE : 1];
  if constexpr (PRE) {
    const float *const rp = a.res ? a.res : a.x, *const bp = a.bias ? a.bias : a.x;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      int f;
      const int o = out_at(tid + NT * i, f);
      rv[i] = rp[o >= 0 && a.res ? o : 0];
      bv[i] = bp[o >= 0 && a.bias ? f : 0];
    }
  }

  // ---- where k lies in the patches
  for (int k = tid; k < KT; k += NT) {
    const int c = a.by_t.div(k), t = k - c * a.T, kh = a.by_kw.div(t), kw = t - kh * (int)a.by_kw.d;
    ktab[k] = k < KC ? (c * PS + kh * a.hc + kw) * 4 : 0;
  }
  // patch byte offset of this lane's pixel of each block
  const int npx = a.tw * a.Ho;  // pixel slots of a strip, the last strip's spare columns among them
  int pb[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int p = min(p0 + 16 * i + r, npx - 1);
    const int oy = a.by_tw.div(p), ox = p - oy * a.tw;
    pb[i] = ((oy - oy0) * a.hc + min(ox, tw - 1)) * a.pstep * 4;
  }
  f32x4 acc[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int ch = 0; ch < a.nchunks; ++ch) {
    float *const buf = patch + (ch & 1) * a.cc * PS;
    commit(buf);
    // one barrier per chunk: the buffer written next is the one read a chunk ago
    __syncthreads();
    if (ch + 1 < a.nchunks) stage((ch + 1) * a.cc);
    const char *const xb = reinterpret_cast<const char *>(buf);
    const int kbase = ch * KC, kend = min(KC, a.K - kbase);  // this chunk's k: [0, kend)
    const int kfull = kend & ~15, klast = a.K - 16;
    // k steps wk, wk + WK, ... of the chunk, kRing at a time and then the
    // rest.  No early exit from the ring's loop (its registers would be moved
    // at the exits, each move waiting for its load), and no second copy of it:
    // the kernel runs its code once or twice, so its instruction fetches count.
    auto step = [&](int k, f32x4 &ring) __attribute__((always_inline)) {
      const i32x4 ko = *reinterpret_cast<const i32x4 *>(ktab + k + 4 * q);
      float v[4][NB];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < NB; ++i) v[s][i] = *reinterpret_cast<const float *>(xb + pb[i] + ko[s]);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < NB; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[s][i], ring[s], acc[i], 0, 0, 0);
      ring = load_w(min(kbase + k + KSTEP * kRing, klast));
    };
    int k = 16 * wk;
    for (; k + KSTEP * (kRing - 1) < kfull; k += KSTEP * kRing)
#pragma unroll
      for (int u = 0; u < kRing; ++u) step(k + KSTEP * u, wv[u]);
#pragma unroll
    for (int u = 0; u + 1 < kRing; ++u)
      if (k + KSTEP * u < kfull) step(k + KSTEP * u, wv[u]);
    // the end of K (its length no multiple of 16): words past it count as
    // zero on both sides
    if (kfull < kend && (kfull >> 4) % WK == wk) {
      const int d = wrow + kbase + kfull - wlast;  // > 0: the run was moved back by d
      f32x4 wq = load_w(kbase + kfull);
      if (d > 0) wq = d == 1 ? f32x4{wq[1], wq[2], wq[3], 0.f} : d == 2 ? f32x4{wq[2], wq[3], 0.f, 0.f}
                                                               : f32x4{wq[3], 0.f, 0.f, 0.f};
      for (int s = 0; s < 4; ++s) {
        const bool ok = kfull + 4 * q + s < kend;
        const int ko = ktab[kfull + 4 * q + s];
        const float b = s == 0 ? wq[0] : s == 1 ? wq[1] : s == 2 ? wq[2] : wq[3];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const float v = *reinterpret_cast<const float *>(xb + pb[i] + ko);
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(ok ? v : 0.0f, ok ? b : 0.0f, acc[i], 0, 0, 0);
        }
      }
    }
    if (ch + 1 < a.nchunks) fill_ring(kbase + KC);
  }

  // ---- partial sums of the K parts through LDS, [wk][wf][filter][pixel]
  constexpr int RS = PX + 4;
  __syncthreads();
  float *const red = smem;
#pragma unroll
  for (int i = 0; i < NB; ++i)
    *reinterpret_cast<f32x4 *>(red + ((size_t)wave * 16 + r) * RS + 16 * i + 4 * q) = acc[i];
  __syncthreads();
  const ActBounds ab = act_bounds(a.act);
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const int e = tid + NT * i, px = e % PX, fl = e / PX;  // filter fl: wave fl / 16's block, row fl % 16
    int f;
    const int o = out_at(e, f);
    if (o >= 0) {
      float v = 0.0f;
#pragma unroll
      for (int k = 0; k < WK; ++k) v += red[((size_t)(k * WF) * 16 + fl) * RS + px];
      if (a.bias) v += PRE ? bv[PRE ? i : 0] : a.bias[f];
      if (a.res) v += PRE ? rv[PRE ? i : 0] : a.res[o];
      a.out[o] = act_clamp(v, ab);
    }
  }
}

template <int NB, int WF, int WK>
bool split_shape(const ConvArgs &c, NchwArgs &a, size_t &lds) {
  constexpr int NW = WF * WK, PX = 16 * NB;
  a.x = static_cast<const float *>(c.x); a.w = static_cast<const float *>(c.w);
  a.bias = c.bias; a.res = static_cast<const float *>(c.res); a.out = static_cast<float *>(c.out);
  a.C = c.C; a.H = c.H; a.W = c.W; a.F = c.F; a.T = c.KH * c.KW; a.K = c.C * a.T;
  a.pad = c.pad; a.st = c.stride; a.Ho = c.Ho; a.Wo = c.Wo; a.act = c.act;
  a.nstrips = (c.Wo + 15) / 16;
  a.tw = (c.Wo + a.nstrips - 1) / a.nstrips;
  a.nstrips = (c.Wo + a.tw - 1) / a.tw;
  const long long npx = (long long)a.tw * c.Ho;
  // by_tw's range (tw <= 16); 3x3 16 -> 16 at 4200x600 495 us (the direct
  // kernel, where taller images would go, reads each input word nine times)
  if (npx + PX >= 1 << 28) return false;
  a.tiles = (int)((npx + PX - 1) / PX);
  const long long npt = (long long)c.N * a.nstrips * a.tiles, grid = npt * ((c.F + 16 * WF - 1) / (16 * WF));
  if (grid > 0x7fffffff - kXcds) return false;
  a.npt = (int)npt;
  a.grid = (int)grid;
  int span = PX % a.tw == 0 ? PX / a.tw : (PX - 2) / a.tw + 2;  // output rows a tile touches
  if (span > c.Ho) span = c.Ho;
  // A 1x1 filter's patch holds the pixels it reads only; with few channels the
  // whole rows, whose channels' loads are fewer (16 -> 16 1x1/4 4.5 against 5.3
  // us).  us, the kernel before / whole rows / so: 1x1/2 56x56x64 -> 64 at batch 8
  // 9.3 / 11.0 / 7.0, 1x1/3 64 -> 256 24.4 / 50.5 / 8.7, 1x1/4 256 -> 128 at
  // 112x112 and batch 2 74 / 93 / 19.
  const bool skip = a.T == 1 && c.C > 24 && c.stride < 4096;
  a.pstep = skip ? 1 : c.stride;
  a.istep = skip ? c.stride : 1;
  const long long hr = (long long)(span - 1) * a.pstep + c.KH;
  const long long hc = (long long)(a.tw - 1) * a.pstep + c.KW;
  const long long wwords = (long long)c.F * a.K;  // filter indices stay below 2^31 past a row's end
  if (hr * hc > 64 * kStage || a.T > 4096 || wwords < 4 || wwords > (1LL << 31) - 4096) return false;
  a.hc = (int)hc;
  a.ps = (int)(hr * hc);
  a.words = skip ? a.ps : 64 * kStage;  // (other patches end near a load's end)
  const int need = (a.ps + 63) / 64;
  for (int v : {1, 2, 3, 4, 5, 8, 16})
    if (need <= (a.npl = v)) break;
  int cmax = kStage / a.npl * NW;
  for (;; cmax -= 16) {
    if (c.C <= cmax) {
      a.cc = c.C;
      a.nchunks = 1;
    } else {
      if (cmax < 16) return false;
      const int n = (c.C + cmax / 16 * 16 - 1) / (cmax / 16 * 16);
      a.cc = ((c.C + n - 1) / n + 15) / 16 * 16;
      a.nchunks = (c.C + a.cc - 1) / a.cc;
    }
    const size_t kt = ((size_t)a.cc * a.T + 15) / 16 * 16;
    lds = 4 * (kt + (size_t)(a.nchunks > 1 ? 2 : 1) * a.cc * patch_stride(a.npl));
    if (kt <= 8192 && lds <= 80 * 1024) break;
    if (cmax <= 16) return false;
  }
  const size_t red = (size_t)NW * 16 * (PX + 4) * 4;
  if (red > lds) lds = red;
  a.by_hc = FastDiv(a.hc); a.by_tw = FastDiv(a.tw); a.by_t = FastDiv(a.T); a.by_kw = FastDiv(c.KW);
  return true;
}

template <int NB, int WF, int WK, int NPL>
hipError_t launch_split(const ConvArgs &c, const NchwArgs &a, size_t lds, hipStream_t s) {
  auto kern = conv2d_nchw_split_kernel<NB, WF, WK, NPL>;
  constexpr int NW = WF * WK, PX = 16 * NB;
  // the dynamic LDS limit, raised once per device
  const int ok = cached_per_kernel(reinterpret_cast<const void *>(kern), [&](int) {
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024) == hipSuccess
               ? 1 : 0;
  });
  if (!ok) return hipErrorInvalidValue;
  const dim3 grid((a.grid + kXcds - 1) / kXcds * kXcds);
  const double units = NW / 4.0, steps = (a.K + 15) / 16;
  const int wgs = (int)std::ceil(a.grid * units);
  npu_launch_plan p = make_plan("conv2d_nchw", wgs, wg_per_cu(kern, 64 * NW, lds), wgs, 32);
  p.load_phases = a.nchunks;
  p.tile_macs = 16.0 * WF * PX * a.K / units;
  p.tile_valu = 4.0 * (steps / WK * (8.0 + 4.0 * (NB + 2)) + 12.0 * kStage * a.nchunks + 120.0);
  p.tile_lds_bytes = (4.0 * a.C * a.ps + WF * steps * 4.0 * 256 * (NB + 4) + 2.0 * NW * 16 * PX * 4) / units;
  p.tile_load_bytes = (4.0 * a.C * a.ps + 4.0 * 16 * WF * a.K) / units;
  p.tile_store_bytes = 4.0 * PX * 16 * WF * (c.res ? 2 : 1) / units;
  p.hbm_bytes = 4.0 * ((double)c.N * c.C * c.H * c.W + (double)c.F * a.K +
                       (double)c.N * c.F * c.Ho * c.Wo * (c.res ? 2 : 1)) + (c.bias ? 4.0 * c.F : 0.0);
  plans_add(p);
  hipLaunchKernelGGL(kern, grid, dim3(64 * NW), lds, s, a);
  return hipGetLastError();
}

// A window that is the whole input (no pad, one output pixel: the model zoo's
// classifiers, 7x7 over the last feature map): out[n, f] = x[n] . w[f], both
// contiguous in the same (c, kh, kw) order.  What bounds it is reading the
// filters once from HBM.  A workgroup of eight waves takes FW filters and
// splits K over its waves; a wave streams FW rows at a time in whole
// 1 KiB runs, several in flight, and multiplies each by the NI images' run.
// 512x7x7 -> 1000 at batch 1 (103 MB of filters): 2950 us on the direct
// kernel (16 workgroups, a load round trip per 16 k), 16.5 us here, 6.2 TB/s.
template <int FW, int NI, bool VEC>
__global__ __launch_bounds__(512) void conv2d_nchw_dot_kernel(
    const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
    const float *__restrict__ res, float *__restrict__ out, int N, int F, int K, int act) {
  constexpr int NW = 8, EPL = VEC ? 4 : 1;
  __shared__ float red[NW][FW * NI];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int f0 = blockIdx.x * FW, n0 = blockIdx.y * NI;
  const float *wr[FW], *xr[NI];
#pragma unroll
  for (int j = 0; j < FW; ++j) wr[j] = w + (size_t)min(f0 + j, F - 1) * K;
#pragma unroll
  for (int i = 0; i < NI; ++i) xr[i] = x + (size_t)min(n0 + i, N - 1) * K;
  float acc[FW][NI];
#pragma unroll
  for (int j = 0; j < FW; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) acc[j][i] = 0.0f;
  constexpr int RUN = 64 * EPL;  // elements of one wave load
  constexpr int U = NI == 1 ? 4 : 2;
  // runs wave, wave + NW, ... of K, U at a time; lanes past K take no part
  auto step = [&](int k0, auto full) __attribute__((always_inline)) {
    f32x4 wv[U][FW], xv[U][NI];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + u * NW * RUN + EPL * lane;
      const int kc = decltype(full)::value ? k : min(k, K - EPL);
#pragma unroll
      for (int j = 0; j < FW; ++j) {
        if constexpr (VEC) wv[u][j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(wr[j] + kc));
        else wv[u][j][0] = wr[j][kc];
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        if constexpr (VEC) xv[u][i] = *reinterpret_cast<const f32x4 *>(xr[i] + kc);
        else xv[u][i][0] = xr[i][kc];
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool ok = decltype(full)::value || k0 + u * NW * RUN + EPL * lane < K;
#pragma unroll
      for (int j = 0; j < FW; ++j)
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
          for (int e = 0; e < EPL; ++e)
            acc[j][i] = fmaf(ok ? wv[u][j][e] : 0.0f, ok ? xv[u][i][e] : 0.0f, acc[j][i]);
    }
  };
  int k0 = wave * RUN;
  for (; k0 + (U - 1) * NW * RUN + RUN <= K; k0 += U * NW * RUN) step(k0, std::true_type{});
  if (k0 < K) step(k0, std::false_type{});
#pragma unroll
  for (int j = 0; j < FW; ++j)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const float v = wave_sum(acc[j][i]);
      if (lane == 0) red[wave][j * NI + i] = v;
    }
  __syncthreads();
  if (tid < FW * NI) {
    const int f = f0 + tid / NI, n = n0 + tid % NI;
    float v = 0.0f;
#pragma unroll
    for (int k = 0; k < NW; ++k) v += red[k][tid];
    if (f < F && n < N) {
      const size_t o = (size_t)n * F + f;
      if (bias) v += bias[f];
      if (res) v += res[o];
      out[o] = act_clamp(v, act_bounds(act));
    }
  }
}

template <int FW, int NI, bool VEC>
hipError_t launch_dot(const ConvArgs &a, int K, hipStream_t s) {
  const dim3 grid((a.F + FW - 1) / FW, (a.N + NI - 1) / NI);
  npu_launch_plan p = make_plan("conv2d_nchw_dot", grid.x * grid.y * 2,
                                wg_per_cu(conv2d_nchw_dot_kernel<FW, NI, VEC>, 512), grid.x * grid.y * 2, 32);
  p.tile_valu = 4.0 * (K / 512.0 * (FW * NI + FW + NI) + 60.0);
  p.tile_load_bytes = 4.0 * K * (FW + NI) / 2;
  p.tile_store_bytes = 4.0 * FW * NI / 2;
  p.hbm_bytes = 4.0 * ((double)a.N * K + (double)a.F * K + (double)a.N * a.F * (a.res ? 2 : 1)) +
                (a.bias ? 4.0 * a.F : 0.0);
  plans_add(p);
  hipLaunchKernelGGL((conv2d_nchw_dot_kernel<FW, NI, VEC>), grid, dim3(512), 0, s,
                     static_cast<const float *>(a.x), static_cast<const float *>(a.w), a.bias,
                     static_cast<const float *>(a.res), static_cast<float *>(a.out), a.N, a.F, K, a.act);
  return hipGetLastError();
}

// 1x1 filters of at most CMAX channels: a lane per output pixel, its channels in
// registers, kPwF filters (uniform: scalar loads) multiplied into them and
// stored along the pixels.  What bounds it: the outputs' stores, and below a few
// thousand pixels the launch; the split kernel's table, staging and partial
// sums cost more than such a product.  us, 64-pixel x 64-filter MFMA tiles (the
// kernel before) / split / here: 67x67x2 -> 59 5.2 / 7.2 / 3.7, 88x88x1 -> 3 with
// residual at batch 12 13.6 / 16.9 / 3.6, 112x112x8 -> 8 at batch 4 8.8 / 8.4 /
// 4.4, 111x111x4 -> 253 at batch 2 21.2 / 17.8 / 12.4.
constexpr int kPwF = 4, kPwThreads = 128;

template <int CMAX>
__global__ __launch_bounds__(kPwThreads) void conv2d_nchw_pointwise_kernel(
    const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
    const float *__restrict__ res, float *__restrict__ out, int P, int C, int H, int W, int F, int st,
    int pad, int Ho, int Wo, int act) {
  const int p = blockIdx.x * kPwThreads + threadIdx.x;
  if (p >= P) return;
  const int n = p / (Ho * Wo), hw = p - n * Ho * Wo, oy = hw / Wo, ox = hw - oy * Wo;
  const int iy = oy * st - pad, ix = ox * st - pad, plane = H * W;
  const bool in = (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
  const float *const xp = x + (size_t)n * C * plane + (in ? iy * W + ix : 0);
  float v[CMAX];
#pragma unroll
  for (int c = 0; c < CMAX; ++c) {
    const float u = xp[(size_t)min(c, C - 1) * plane];
    v[c] = in ? u : 0.0f;
  }
  const int f0 = blockIdx.y * kPwF;
  const size_t map = (size_t)Ho * Wo, o = ((size_t)n * F + f0) * map + hw;
  float r[kPwF], acc[kPwF];
#pragma unroll
  for (int j = 0; j < kPwF; ++j) r[j] = res && f0 + j < F ? res[o + j * map] : 0.0f;
#pragma unroll
  for (int j = 0; j < kPwF; ++j) {
    const int f = min(f0 + j, F - 1);
    acc[j] = 0.0f;
#pragma unroll
    for (int c = 0; c < CMAX; ++c) acc[j] = c < C ? fmaf(v[c], w[(size_t)f * C + min(c, C - 1)], acc[j]) : acc[j];
    if (bias) acc[j] += bias[f];
  }
  const ActBounds ab = act_bounds(act);
#pragma unroll
  for (int j = 0; j < kPwF; ++j)
    if (f0 + j < F) out[o + j * map] = act_clamp(res ? acc[j] + r[j] : acc[j], ab);
}

template <int CMAX>
hipError_t launch_pointwise(const ConvArgs &a, hipStream_t s) {
  const int P = a.N * a.Ho * a.Wo;
  const dim3 grid((P + kPwThreads - 1) / kPwThreads, (a.F + kPwF - 1) / kPwF);
  // in units of four waves
  const int wgs = (int)(((long long)grid.x * grid.y * kPwThreads + 255) / 256);
  npu_launch_plan p = make_plan("conv2d_nchw_pointwise", wgs, wg_per_cu(conv2d_nchw_pointwise_kernel<CMAX>, kPwThreads),
                                wgs, 32);
  p.tile_valu = 4.0 * (60.0 + 3.0 * CMAX + kPwF * (12.0 + a.C));
  p.tile_load_bytes = 256.0 * 4 * (a.C + (a.res ? kPwF : 0));
  p.tile_store_bytes = 256.0 * 4 * kPwF;
  p.hbm_bytes = 4.0 * ((double)a.N * a.C * a.H * a.W + (double)a.F * a.C + (double)P * a.F * (a.res ? 2 : 1)) +
                (a.bias ? 4.0 * a.F : 0.0);
  plans_add(p);
  hipLaunchKernelGGL((conv2d_nchw_pointwise_kernel<CMAX>), grid, dim3(kPwThreads), 0, s,
                     static_cast<const float *>(a.x), static_cast<const float *>(a.w), a.bias,
                     static_cast<const float *>(a.res), static_cast<float *>(a.out), P, a.C, a.H, a.W, a.F,
                     a.stride, a.pad, a.Ho, a.Wo, a.act);
  return hipGetLastError();
}

// What the split kernel's patches do not hold (more than 1024 words per
// channel: long strides or very large filters) or its index ranges: implicit
// GEMM with the reduction index k = (c, kh, kw) in FCHW order, so a
// filter's operand is its own contiguous run of k, and each MFMA step's A
// word is the input pixel that k and the output pixel address (zero in the
// pad).  Operands come straight from L2: no staging, no halo reuse.
// Workgroup tile: 64 output pixels (flattened n, oh, ow) x 64 filters, waves
// as 2 x 2, each 32 x 32 = four 16x16 MFMA tiles; accumulator rows are
// pixels, so a lane's four values are consecutive pixels of one filter.
__global__ __launch_bounds__(256) void conv2d_nchw_direct_kernel(
    const float *__restrict__ x, const float *__restrict__ w, const float *__restrict__ bias,
    const float *__restrict__ res, float *__restrict__ out, int N, int C, int H, int W, int F,
    int KH, int KW, int st, int pad, int Ho, int Wo, int act) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int P = N * Ho * Wo, K = C * KH * KW, T = KH * KW;
  const int p0 = blockIdx.x * 64 + (wave & 1) * 32;
  const int f0 = blockIdx.y * 64 + (wave >> 1) * 32;
  int pn[2], ph[2], pw[2];
  bool pok[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int p = p0 + 16 * i + r;
    pok[i] = p < P;
    const int pp = pok[i] ? p : 0;
    pn[i] = pp / (Ho * Wo);
    const int rem = pp - pn[i] * Ho * Wo;
    ph[i] = (rem / Wo) * st - pad;
    pw[i] = (rem - (rem / Wo) * Wo) * st - pad;
  }
  const float *wr[2];
  bool fok[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int f = f0 + 16 * j + r;
    fok[j] = f < F;
    wr[j] = w + (size_t)(fok[j] ? f : 0) * K;
  }
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // lane group q takes k = k0 + 4q + s; (c, kh, kw) of each k is kept and
  // advanced by 16 per step instead of divided out
  int kc[4], kh_[4], kw_[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int k = 4 * q + s;
    kc[s] = k / T;
    kh_[s] = (k - kc[s] * T) / KW;
    kw_[s] = k - kc[s] * T - kh_[s] * KW;
  }
  for (int k0 = 0; k0 < K; k0 += 16) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 4 * q + s;
      const bool kin = k < K;
      float a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int ih = ph[i] + kh_[s], iw = pw[i] + kw_[s];
        const bool in = kin && pok[i] && ih >= 0 && ih < H && iw >= 0 && iw < W;
        a[i] = in ? x[((size_t)(pn[i] * C + kc[s]) * H + ih) * W + iw] : 0.0f;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) b[j] = kin && fok[j] ? wr[j][k] : 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
      // advance this slot's k by 16
      kw_[s] += 16;
      while (kw_[s] >= KW) {
        kw_[s] -= KW;
        if (++kh_[s] == KH) {
          kh_[s] = 0;
          ++kc[s];
        }
      }
    }
  }
  const ActBounds ab = act_bounds(act);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int f = f0 + 16 * j + r;
    if (f >= F) continue;
    const float bv = bias ? bias[f] : 0.0f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int p = p0 + 16 * i + 4 * q + e;
        if (p >= P) continue;
        const int n = p / (Ho * Wo), hw = p - n * Ho * Wo;
        const size_t o = (size_t)(n * F + f) * Ho * Wo + hw;
        float v = acc[i][j][e] + bv;
        if (res) v += res[o];
        out[o] = act_clamp(v, ab);
      }
  }
}

hipError_t launch_nchw_direct(const ConvArgs &a, hipStream_t s) {
  const int P = a.N * a.Ho * a.Wo;
  dim3 grid((P + 63) / 64, (a.F + 63) / 64);
  const double K = (double)a.C * a.KH * a.KW, steps = (K + 15) / 16;
  npu_launch_plan p = make_plan("conv2d_nchw_direct", grid.x * grid.y,
                                wg_per_cu(conv2d_nchw_direct_kernel), grid.x * grid.y, 32);
  p.load_phases = (int)steps;  // each k step loads, then multiplies
  p.tile_macs = 64.0 * 64 * K;
  p.tile_valu = 4.0 * (steps * 4 * 24.0 + 80.0);  // per wave: per k slot addresses, bounds, k advance
  p.tile_load_bytes = steps * 4 * 4.0 * 256 * 4;  // four words per lane and k slot, four waves
  p.tile_store_bytes = 4.0 * 64 * 64 * (a.res ? 2 : 1);
  p.hbm_bytes = 4.0 * ((double)a.N * a.C * a.H * a.W + (double)a.F * K +
                       (double)P * a.F * (a.res ? 2 : 1)) + (a.bias ? 4.0 * a.F : 0.0);
  plans_add(p);
  hipLaunchKernelGGL(conv2d_nchw_direct_kernel, grid, dim3(256), 0, s,
                     static_cast<const float *>(a.x), static_cast<const float *>(a.w), a.bias,
                     static_cast<const float *>(a.res), static_cast<float *>(a.out), a.N, a.C, a.H,
                     a.W, a.F, a.KH, a.KW, a.stride, a.pad, a.Ho, a.Wo, a.act);
  return hipGetLastError();
}

// The split kernel's shapes, largest tile first (pixels x filters per
// workgroup 64 x 64, 64 x 32, 64 x 16, 32 x 16, 16 x 16): the first that has
// kMinWgs workgroups, else the smallest.  Measured at batch 1, 3x3, us: the
// 112 -> 56 layer of 64 channels (49 / 98 / 196 workgroups of the first three)
// 22.1 / 15.5 / 12.5; 28x28x128 (28 / 56 / 112 / 200) 29.5 / 18.2 / 12.8 /
// 10.4; 14x14x256 (16 / .. / 64 / 112 / 208) 53 / 31 / 21.6 / 17.0 / 16.1;
// batch 8 14x14x256 (128 / 256) 55.7 / 33.3.  Sixteen waves per workgroup
// were slower than eight (7x7x512 27 against 20 us): their loads queue.  With
// twice kMinWgs tiles of 64 x 64, K is not split: it takes the same time
// (56x56x64 at batch 8 33.2 against 32.2 us, 28x28x128 at batch 16 56.8 against
// 57.4) and every sum runs in k order.
constexpr long long kMinWgs = 160;

// A whole-window conv of filters up to kDotShort long takes the direct kernel
// past kDotOutputs images x filters: the dot kernel's time grows with the
// images (its filters are read once per eight), the direct kernel's first
// with the filter's length only.  Measured, us, 1000 filters: of 512 words, dot
// 66 at 256 images, 128 at 512, 502 at 2048, direct 138 at 300, 141 at 512,
// 166 at 2048; of 1024, dot 69 at 256, direct 155 at 300, 159 at 1024; of
// 2048, dot 205 at 512, 388 at 1024, direct 677 at 2200; of 25088, dot 1375 at
// 512, 5469 at 2048, direct 3503 and 5449: there the two end at the same rate.
// kDotImages: the launch's y range.
constexpr long long kPwPixels = 4096;  // pointwise kernel past 8 channels: see below
constexpr long long kDotOutputs = 1 << 19, kDotShort = 2048;
constexpr int kDotImages = 8 * 65535;
template <int NB, int WF, int WK>
bool try_split(const ConvArgs &a, long long min_wgs, hipStream_t s, hipError_t &e) {
  NchwArgs n;
  size_t lds;
  if (!split_shape<NB, WF, WK>(a, n, lds)) return false;
  if (n.grid < min_wgs) return false;
  // Patches past 512 words hold at most eight channels, each staged by one wave:
  // the workgroups' time is the staging's, and many of them take longer than the
  // direct kernel on a short reduction.  Both estimates in us, from 7x7/4, 5x5/5
  // and 9x9/3 filters of 1 to 8 channels; split / direct: 7x7/4 168x168x1 -> 42 at
  // batch 13 37.7 / 17.0, 224x224x3 -> 64 at batch 8 52.8 / 31.2 and at batch 2
  // 17.8 / 26.3, 112x112x8 -> 64 at batch 32 66 / 78.
  if (n.npl == 16) {
    const double steps = (n.K + 15) / 16, tiles = ((double)a.N * a.Ho * a.Wo / 64 + 1) * ((a.F + 63) / 64);
    if (7.0 + steps * (1.8 + 0.0033 * tiles) < 4.0 + 0.0085 * n.grid) {
      e = launch_nchw_direct(a, s);
      return true;
    }
  }
  switch (n.npl) {
    case 1: e = launch_split<NB, WF, WK, 1>(a, n, lds, s); break;
    case 2: e = launch_split<NB, WF, WK, 2>(a, n, lds, s); break;
    case 3: e = launch_split<NB, WF, WK, 3>(a, n, lds, s); break;
    case 4: e = launch_split<NB, WF, WK, 4>(a, n, lds, s); break;
    case 5: e = launch_split<NB, WF, WK, 5>(a, n, lds, s); break;
    case 8: e = launch_split<NB, WF, WK, 8>(a, n, lds, s); break;
    default: e = launch_split<NB, WF, WK, 16>(a, n, lds, s); break;
  }
  return true;
}

}  // namespace

hipError_t launch_conv2d_nchw_f32(const ConvArgs &a, hipStream_t s) {
  const long long K = (long long)a.C * a.KH * a.KW;
  if (a.Ho == 1 && a.Wo == 1 && a.pad == 0 && a.KH == a.H && a.KW == a.W && K < (1 << 30)) {
    if (a.N > kDotImages || (K <= kDotShort && (long long)a.N * a.F > kDotOutputs)) return launch_nchw_direct(a, s);
    if (K % 4 == 0) return a.N == 1 ? launch_dot<4, 1, true>(a, (int)K, s) : launch_dot<4, 8, true>(a, (int)K, s);
    return launch_dot<4, 8, false>(a, (int)K, s);
  }
  // The pointwise kernel's time grows with the channels that a lane loads one
  // after the other: of 16, 5.0 us at 67x67 against 6.5, but 5.1 against 4.5 at
  // 28x28; of 25 -> 13 filters 13.1 against 10.1 (its channels are loaded again
  // for every four), of 24 -> 2 10.4 against 31.6.
  const long long pixels = (long long)a.N * a.Ho * a.Wo;
  if (K == a.C && a.F <= kPwF * 65535 && (a.C <= 8 || (pixels >= (a.stride > 1 ? 2 : 1) * kPwPixels &&
                                (a.C <= 16 || (a.C <= 32 && a.F <= 8)))))
    return a.C <= 4    ? launch_pointwise<4>(a, s)
           : a.C <= 8  ? launch_pointwise<8>(a, s)
           : a.C <= 16 ? launch_pointwise<16>(a, s)
                       : launch_pointwise<32>(a, s);
  hipError_t e = hipSuccess;
  if (try_split<4, 4, 1>(a, 2 * kMinWgs, s, e) || try_split<4, 4, 2>(a, kMinWgs, s, e) ||
      try_split<4, 2, 4>(a, kMinWgs, s, e) || try_split<4, 1, 8>(a, kMinWgs, s, e) ||
      try_split<2, 1, 8>(a, kMinWgs, s, e) || try_split<1, 1, 8>(a, 1, s, e))
    return e;
  return launch_nchw_direct(a, s);
}

}  // namespace npu
