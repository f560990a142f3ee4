// k_qbottleneck.hip -- int8 ResNet-50 bottleneck as ONE fused group:
//   y1  = clamp(requant(conv1x1(x, w1)), 0, 127)          [N,H,W,M1]
//   y2  = clamp(requant(conv3x3(pad(y1), w2)), 0, 127)    [N,H,W,M1]
//   out = clamp(requant(conv1x1(y2, w3)) + x, 0, 127)     [N,H,W,C]
// (the int8 restatement of test/resnet50_block.mlir:5-105; requant is TOSA
// apply_scale_32 with single rounding, per output channel).
//
// The reference cannot fuse across the tensor.pad that separates conv1 from
// conv2 (OutlineFusedGroupsPass.cpp:140-144 only unites linalg producers), so
// it would run three groups and round-trip y1 and y2 through DRAM.  Here the
// pad is folded into the halo: a tile is 7 output rows x 14 columns of one
// image, whose 9 x 16 halo is exactly nine 16-pixel MFMA blocks (one per halo
// row, lane = halo column); conv1 is recomputed on the halo and y1, y2 stay
// in LDS.  HBM sees x once (halo re-reads hit L2) and out once.
//
// The kernel is persistent: each wave loads its share of the three filters
// into registers once and the workgroup walks its tiles, prefetching the next
// tile's halo into registers while the current tile is computed.  A 56 x 56
// image is 32 such tiles, so 32 images are 1024 tiles: two per workgroup at
// two workgroups per CU, no CU carrying an extra tile.
//
// MFMA: v_mfma_i32_16x16x64_i8 with the filters as the A operand, so a lane's
// accumulator holds four consecutive output channels of one pixel.  Integer
// accumulation is exact, so any summation order gives the oracle's result bit
// for bit.
#include <type_traits>

#include "kernels.hpp"
#include "npu_device.hpp"
#include "persistent.hpp"
#include "plans.hpp"

namespace npu {

namespace {

constexpr int TH = 7, TW = 14;                 // output tile
constexpr int HH = TH + 2, HW = 16;            // halo tile: HW = TW + 2 = one MFMA block
constexpr int HP = HH * HW;                    // 144 halo pixels = 9 blocks

// TOSA apply_scale_32, single rounding: (acc * m + 2^(s-1)) >> s in 64 bits,
// truncated to 32.  `rnd` is 2^(s-1), prepared once per channel.
__device__ __forceinline__ int requant(int acc, int m, long long rnd, int s) {
  return (int)(((long long)acc * (long long)m + rnd) >> s);
}
__device__ __forceinline__ int clamp_i(int v, int lo, int hi) {
  return v < lo ? lo : (v > hi ? hi : v);
}

// Per-channel requant parameters of the four channels a lane's accumulator
// holds, read from the workgroup's LDS tables.
struct Scale4 {
  i32x4 m, s;
  long long r[4];
};
__device__ __forceinline__ Scale4 scale4(const int32_t *m, const int32_t *s, const long long *r,
                                         int c) {
  Scale4 q;
  q.m = *reinterpret_cast<const i32x4 *>(m + c);
  q.s = *reinterpret_cast<const i32x4 *>(s + c);
#pragma unroll
  for (int e = 0; e < 4; ++e) q.r[e] = r[c + e];
  return q;
}

// Requantize four accumulators (channels c..c+3 of one pixel), clamp to
// [0, 127] and pack them as four bytes, channel c in the low byte.
__device__ __forceinline__ uint32_t requant4(const i32x4 &acc, const Scale4 &q) {
  uint32_t packed = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    packed |= (uint32_t)clamp_i(requant(acc[e], q.m[e], q.r[e], q.s[e]), 0, 127) << (8 * e);
  return packed;
}

template <int C, int M1>
__global__ __launch_bounds__(256, 2) void qbottleneck_kernel(
    const int8_t *__restrict__ x, const int8_t *__restrict__ w1, const int8_t *__restrict__ w2,
    const int8_t *__restrict__ w3, const int32_t *__restrict__ m1, const int32_t *__restrict__ s1,
    const int32_t *__restrict__ m2, const int32_t *__restrict__ s2,
    const int32_t *__restrict__ m3, const int32_t *__restrict__ s3, int8_t *__restrict__ out,
    int H, int W, int tiles_w, int tiles_img, int ntiles) {
  static_assert(C % 64 == 0 && C <= 256 && M1 == 64, "C must be 64, 128 or 256 and M1 = 64");
  constexpr int XS = C + 32;    // LDS row strides: 32 mod 64 bytes keeps the 16-row
  constexpr int YS = M1 + 32;   // 16-byte operand reads free of bank conflicts
  constexpr int XCH = C / 16;   // 16-byte runs per pixel
  constexpr int NSEG = HP * XCH;
  constexpr int SEGS = (NSEG + 255) / 256;
  constexpr int FB3 = C / 64;   // conv3 filter blocks per wave
  __shared__ __attribute__((aligned(16))) int8_t xs[HP * XS];
  // conv2 reads three columns past a block's 16 lanes for lanes 14 and 15
  // (outputs that are never stored): one spare block keeps them in bounds.
  __shared__ __attribute__((aligned(16))) int8_t y1[(HP + 16) * YS];
  __shared__ __attribute__((aligned(16))) int8_t y2[TH * 16 * YS];
  // requant tables: conv1 channels 0..M1-1, conv2 M1..2M1-1, conv3 2M1..
  constexpr int NQ = 2 * M1 + C;
  __shared__ __attribute__((aligned(16))) int32_t qm[NQ], qs[NQ];
  __shared__ __attribute__((aligned(16))) long long qr[NQ];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const TileWalk walk = tile_walk(ntiles);

  // Halo runs: with 256 threads and XCH 16-byte runs per pixel, thread t
  // loads run t % XCH of halo column (t / XCH) % 16 in every segment s, on
  // halo row t / (16 XCH) + s * 16 / XCH.  Runs outside the image are loaded
  // from a clamped address and zeroed when they are committed to LDS (bit s
  // of `keep`): masking at the load would make the wave wait for it there.
  constexpr int RSTEP = 16 / XCH;
  const int hx = (tid / XCH) % HW, hch = tid % XCH, hy0 = tid / (HW * XCH);
  auto halo_load = [&](int tile, u32x4 (&st)[SEGS], uint32_t &keep) {
    const int n = tile / tiles_img, tt = tile - n * tiles_img;
    const int iy0 = (tt / tiles_w) * TH - 1 + hy0, ix = (tt % tiles_w) * TW - 1 + hx;
    const bool col_in = (unsigned)ix < (unsigned)W;
    const int8_t *base = x + ((size_t)n * H * W + min(max(ix, 0), W - 1)) * C + hch * 16;
    keep = 0;
#pragma unroll
    for (int s = 0; s < SEGS; ++s) {
      const int iy = iy0 + s * RSTEP;
      keep |= (uint32_t)(col_in && (unsigned)iy < (unsigned)H) << s;
      st[s] = *reinterpret_cast<const u32x4 *>(base + (size_t)min(max(iy, 0), H - 1) * W * C);
    }
  };

  // requant tables: loads first, LDS writes after the other prologue loads
  // are issued
  int32_t tm[(NQ + 255) / 256], ts[(NQ + 255) / 256];
#pragma unroll
  for (int k = 0; k < (NQ + 255) / 256; ++k) {
    const int c = min(tid + 256 * k, NQ - 1);
    tm[k] = c < M1 ? m1[c] : c < 2 * M1 ? m2[c - M1] : m3[c - 2 * M1];
    ts[k] = c < M1 ? s1[c] : c < 2 * M1 ? s2[c - M1] : s3[c - 2 * M1];
  }

  u32x4 st[SEGS];
  uint32_t keep = 0;
  if (walk.first < walk.end) halo_load(walk.first, st, keep);

  // Filters as each MFMA's A operand: wave w owns conv1 / conv2 output
  // channels 16w..16w+15 and conv3 output blocks w, w + 4, ...
  const int f12 = wave * 16 + r;
  Frag16 b1[C / 64], b2[9], b3[FB3];
#pragma unroll
  for (int kc = 0; kc < C / 64; ++kc) b1[kc] = load16(w1 + f12 * C + kc * 64 + 16 * q);
#pragma unroll
  for (int t = 0; t < 9; ++t) b2[t] = load16(w2 + (f12 * 9 + t) * M1 + 16 * q);
#pragma unroll
  for (int j = 0; j < FB3; ++j) b3[j] = load16(w3 + ((wave + 4 * j) * 16 + r) * M1 + 16 * q);
  const int fq = wave * 16 + 4 * q;
#pragma unroll
  for (int k = 0; k < (NQ + 255) / 256; ++k) {
    const int c = tid + 256 * k;
    if (c < NQ) {
      qm[c] = tm[k];
      qs[c] = ts[k];
      qr[c] = 1LL << (ts[k] - 1);
    }
  }
#pragma unroll
  for (int kc = 0; kc < C / 64; ++kc) settle(b1[kc].u);
#pragma unroll
  for (int t = 0; t < 9; ++t) settle(b2[t].u);
#pragma unroll
  for (int j = 0; j < FB3; ++j) settle(b3[j].u);

  for (int tile = walk.first; tile < walk.end; tile += walk.step) {
    const int n = tile / tiles_img, tt = tile - n * tiles_img;
    const int ty0 = (tt / tiles_w) * TH, tx0 = (tt % tiles_w) * TW;
    // addressing recomputed per tile rather than held across the loop
    const int ti = opaque(tid);

    // ---- the halo of this tile into LDS; the next tile's loads go out
#pragma unroll
    for (int s = 0; s < SEGS; ++s) {
      const int hy = hy0 + s * RSTEP;
      if (hy < HH)
        *reinterpret_cast<u32x4 *>(xs + (hy * HW + hx) * XS + hch * 16) = masked(st[s], (keep >> s) & 1);
    }
    __syncthreads();
    if (tile + walk.step < walk.end) halo_load(tile + walk.step, st, keep);

    // ---- conv1 (1x1, C -> M1) on the 9 halo rows, requant + ReLU into y1
    //      (zero for halo pixels outside the image: the pad before conv2)
    const bool col_in = (unsigned)(tx0 - 1 + r) < (unsigned)W;
#pragma unroll
    for (int pb = 0; pb < HH; ++pb) {
      i32x4 acc = {0, 0, 0, 0};
#pragma unroll
      for (int kc = 0; kc < C / 64; ++kc)
        MfmaI8::mma(acc, b1[kc], load16(xs + (pb * 16 + r) * XS + kc * 64 + 16 * q));
      const bool inside = col_in && (unsigned)(ty0 - 1 + pb) < (unsigned)H;
      const uint32_t v = requant4(acc, scale4(qm, qs, qr, fq));
      *reinterpret_cast<uint32_t *>(y1 + (pb * 16 + r) * YS + fq) = inside ? v : 0u;
    }
    __syncthreads();

    // ---- conv2 (3x3, M1 -> M1): output row i, column r reads halo rows
    //      i..i+2, columns r..r+2
#pragma unroll
    for (int i = 0; i < TH; ++i) {
      i32x4 acc = {0, 0, 0, 0};
#pragma unroll
      for (int t = 0; t < 9; ++t)
        MfmaI8::mma(acc, b2[t], load16(y1 + ((i + t / 3) * 16 + r + t % 3) * YS + 16 * q));
      *reinterpret_cast<uint32_t *>(y2 + (i * 16 + r) * YS + fq) = requant4(acc, scale4(qm, qs, qr, M1 + fq));
    }
    __syncthreads();

    // ---- conv3 (1x1, M1 -> C), requant + residual + ReLU.  The result
    //      overwrites the residual's own slot in the halo tile (each element
    //      is read and written by the same lane); lanes 14, 15 hold no output.
#pragma unroll
    for (int j = 0; j < FB3; ++j) {
      const int f4 = (wave + 4 * j) * 16 + 4 * q;
      const Scale4 sc = scale4(qm, qs, qr, 2 * M1 + f4);
#pragma unroll
      for (int i = 0; i < TH; ++i) {
        i32x4 acc = {0, 0, 0, 0};
        MfmaI8::mma(acc, b3[j], load16(y2 + (i * 16 + r) * YS + 16 * q));
        if (r < TW) {
          uint32_t *slot = reinterpret_cast<uint32_t *>(xs + ((i + 1) * 16 + r + 1) * XS + f4);
          const uint32_t res = *slot;
          uint32_t packed = 0;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int v = requant(acc[e], sc.m[e], sc.r[e], sc.s[e]) + (int)(int8_t)(res >> (8 * e));
            packed |= (uint32_t)clamp_i(v, 0, 127) << (8 * e);
          }
          *slot = packed;
        }
      }
    }
    __syncthreads();

    // ---- coalesced 16-byte stores of the output tile, RPI rows per pass.
    //      Every thread stores unconditionally: a run past the tile or the
    //      image stores the clamped pixel's own bytes again (the same value
    //      to the same address), so the stores are straight-line code and
    //      the wait for the next halo, which was loaded before them, can
    //      leave them in flight (the vector-memory counter covers loads and
    //      stores).
    {
      constexpr int RUNS = TW * XCH, RPI = 256 / RUNS;
      const int u = min(ti % RUNS + (ti / RUNS >= RPI ? RUNS : 0), RUNS - 1);
      const int sr = min(ti / RUNS, RPI - 1);
      const int c = min(u / XCH, W - 1 - tx0), ch = u % XCH;
      const int rows = min(TH, H - ty0);
      int8_t *obase = out + ((size_t)(n * H + ty0) * W + tx0 + c) * C + ch * 16;
      const int8_t *lbase = xs + (16 + c + 1) * XS + ch * 16;
#pragma unroll
      for (int k = 0; k < (TH + RPI - 1) / RPI; ++k) {
        const int i = min(k * RPI + sr, rows - 1);
        *reinterpret_cast<u32x4 *>(obase + (size_t)i * W * C) =
            *reinterpret_cast<const u32x4 *>(lbase + i * 16 * XS);
      }
    }
    __syncthreads();
  }
}

template <int C, int M1>
hipError_t launch_qb(const QBottleneckArgs &a, hipStream_t s) {
  const int tiles_w = (a.W + TW - 1) / TW, tiles_h = (a.H + TH - 1) / TH;
  const int tiles_img = tiles_w * tiles_h, ntiles = a.N * tiles_img;
  auto kern = qbottleneck_kernel<C, M1>;
  const int full = persistent_grid(kern);
  if (full <= 0) return hipErrorInvalidValue;
  // one tile per workgroup when there are fewer tiles than resident slots
  // (rounded up to whole XCD rounds: the walk gives the spare ones nothing)
  const int grid = ntiles < full ? (ntiles + kXcds - 1) / kXcds * kXcds : full;
  {
    npu_launch_plan p = make_plan("int8_bottleneck", grid, wg_per_cu(kern), ntiles, 8);
    p.load_phases = 1;  // the halo of the next tile is fetched during this one
    p.tile_macs = (double)HP * M1 * C + (double)TH * 16 * M1 * 9 * M1 + (double)TH * 16 * C * M1;
    // per wave: 4.75 vector instructions per requantized channel value
    // (64-bit multiply-add, shift, clamp, packing), four values per lane and
    // block, over conv1's HH halo blocks, conv2's TH blocks and conv3's TH
    // blocks x C/64 filter blocks; 12 per halo run committed and per output
    // row stored (addresses)
    const double vals = 4.0 * (HH + TH + TH * C / 64);
    const int segs = (HP * C / 16 + 255) / 256;
    p.tile_valu = 4.0 * (vals * 4.75 + 12.0 * (segs + TH));
    // LDS: halo written; 1 KiB per wave and MFMA operand read (conv1 HH x
    // C/64, conv2 TH x 9 taps, conv3 TH x C/64); y1 and y2 written; the
    // residual read and overwritten; the output read for the stores; the
    // requant parameters (64 bytes per lane and scale set: conv1, conv2 and
    // one per conv3 filter block)
    p.tile_lds_bytes = HP * (double)C + 4.0 * 1024 * (HH * C / 64 + TH * 9 + TH * C / 64) +
                       (HP + TH * 16.0) * M1 + 2.0 * TH * TW * C + (double)TH * TW * C +
                       (2.0 + C / 64) * 256 * 64;
    // set-up: every workgroup loads the three filters (its waves' shares)
    // and the requant tables, and fills the tables (192 per wave)
    p.wg_setup_bytes = (double)M1 * C * 2 + 9.0 * M1 * M1 + 2.0 * 4 * (2 * M1 + C);
    p.wg_setup_valu = 4.0 * 192.0;
    p.tile_load_bytes = HP * (double)C;
    p.tile_store_bytes = (double)TH * TW * C;
    p.hbm_bytes = 2.0 * a.N * a.H * a.W * C + (double)M1 * C * 2 + 9.0 * M1 * M1 + 4.0 * 2 * (2 * M1 + C);
    plans_add(p);
  }
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, a.x, a.w1, a.w2, a.w3, a.m1, a.s1, a.m2,
                     a.s2, a.m3, a.s3, a.out, a.H, a.W, tiles_w, tiles_img, ntiles);
  return hipGetLastError();
}

// Large filters (launch_qbottleneck_i8: ResNet-50's 512/128, 1024/256 and
// 2048/512): any C <= 2048 and M1 <= 512 that are multiples of 64, M1 >= 128.
// Sixteen waves walk 4 x 7 output tiles (6 x 9 halo pixels); y1 and y2 stay in
// LDS.  Each of the three convolutions is a matrix product that streams its
// filters through LDS in chunks of 256 rows of 128 bytes (KP = 1), or, for
// M1 = 128, of 128 rows of two such runs (KP = 2), conv1 its halo pixels'
// channels with them; two LDS buffers, two more chunks in registers, one
// barrier per chunk.  conv3 goes 256 output channels at a time: the residual's
// tile is staged in LDS, finished in place and stored in 16-byte runs while the
// next channels are multiplied.
//
// Filter chunks lie unpadded, the 16-byte piece p of row f at p ^ (f / 2 % 8),
// so that 16 rows' reads and a row's writes use every bank once.
//
// What bounds it: the instructions around each chunk's four MFMAs per wave
// (about 1 700 clocks a chunk, 34 chunks a tile at 1024/256).  Loaded straight as
// MFMA fragments, 16 rows of 64 bytes per instruction, the filters cost the CU's
// load path 70 clocks per KB (60 us at 1024/256); one chunk in registers instead
// of two 38.4 us.  Measured, batch 32, us, before (4 x 4 tiles, fragments from
// L2) and now: 14x14x1024/256 122 -> 36.3, 28x28x512/128 133 -> 68,
// 7x7x2048/512 367 -> 101.
constexpr int STH = 4, STW = 7, SHW = STW + 2, SHP = SHW * (STH + 2);  // 54 halo pixels
constexpr int SOP = STH * STW;                                         // 28 output pixels
constexpr int SNT = 1024, SROWS = 256;                                 // lanes, filter rows of a chunk
constexpr int SOS = SROWS + 16;                                        // output tile row (bytes)

struct QStreamArgs {
  const int8_t *x, *w1, *w2, *w3;
  const int32_t *m1, *s1, *m2, *s2, *m3, *s3;
  int8_t *out;
  int H, W, C, M1, tiles_w, tiles_img, ntiles;
  FastDiv by_mk;
};

template <int KP>
struct QStreamShape {
  static constexpr int NF1 = 2, NP1 = KP == 1 ? 2 : 1, NF2 = KP == 1 ? 2 : 1;
  static constexpr int XS = KP * 128 + 32;            // x chunk row: 32 mod 64 bytes
  static constexpr int XBUF = SHP * XS, XR = (SHP * 8 * KP + SNT - 1) / SNT;
  static constexpr int NOB = 2;                       // output tiles in LDS
  static constexpr int FBUF = SROWS * 128;
  static_assert(NOB * SOP * SOS <= 2 * XBUF, "output tiles fit the x chunks' space");
  static size_t lds(int M1) { return 2 * FBUF + 2 * XBUF + (size_t)(SHP + 32) * (M1 + 32); }
};

template <int KP>
__global__ __launch_bounds__(SNT, 4) void qb_stream_kernel(const QStreamArgs a) {
  using S = QStreamShape<KP>;
  constexpr int NF1 = S::NF1, NP1 = S::NP1, NF2 = S::NF2, XS = S::XS, XR = S::XR;
  extern __shared__ __attribute__((aligned(16))) int8_t qmem[];
  int8_t *const fbuf = qmem;                     // [2][SROWS][128]
  int8_t *const xbuf = fbuf + 2 * S::FBUF;       // [2][SHP][XS]; conv3: [NOB][SOP][SOS]
  int8_t *const y1 = xbuf + 2 * S::XBUF;         // [SHP][YS]
  const int C = a.C, M1 = a.M1, YS = M1 + 32;
  int8_t *const y2 = y1 + SHP * YS;              // [32][YS]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int R = min(M1, SROWS), rg = (M1 + R - 1) / R, mk = M1 / 64;  // filter rows of a chunk, row groups
  // k chunks of a row group, made even (an odd count's last chunk is empty):
  // chunks go by pairs, each with its own LDS buffer and registers
  const int kc1 = (C + 256 * KP - 1) / (256 * KP) * 2, kc2 = (9 * M1 + 256 * KP - 1) / (256 * KP) * 2;
  const int kc3 = (M1 + 255) / 256 * 2, rg3 = (C + SROWS - 1) / SROWS;

  // ---- filter chunks: this thread's 16-byte piece `piece` of slots srow and
  //      srow + 128 (slot = kpart R + row).  Rows and k past the end load
  //      from clamped addresses; the first are not stored, the second skipped.
  const int piece = tid & 7, srow = tid >> 3;
  const int fdst0 = srow * 128 + 16 * (piece ^ ((srow >> 1) & 7)), fdst1 = fdst0 + 128 * 128;
  struct Pair {
    u32x4 lo, hi;
  } fr0, fr1;  // of the even and the odd chunks
  auto commit = [&](int buf, const Pair &f) __attribute__((always_inline)) {
    *reinterpret_cast<u32x4 *>(fbuf + buf * S::FBUF + fdst0) = f.lo;
    *reinterpret_cast<u32x4 *>(fbuf + buf * S::FBUF + fdst1) = f.hi;
  };
  // filter fragment: slot row f (= r mod 16), 64-byte step h of its 128 bytes
  const int sw = (r >> 1) & 7;
  auto ffrag = [&](int buf, int f, int h) __attribute__((always_inline)) {
    return load16(fbuf + buf * S::FBUF + f * 128 + 16 * ((4 * h + q) ^ sw));
  };
  // chunk i of the tile's walk over conv1's, conv2's and conv3's chunks
  const int n1 = rg * kc1, n2 = n1 + rg * kc2, n3 = n2 + rg3 * kc3;
  // the chunk to fetch next: its place in the walk, its filters' rows, bytes
  // per row, rows per chunk, k chunks and bytes of k per chunk
  int fi, fk, fg, f_rows, f_kbytes, f_rper, f_kcn, f_kstep;
  const int8_t *f_w;
  auto fetch_start = [&]() __attribute__((always_inline)) {
    fi = fk = fg = 0;
    f_w = a.w1, f_rows = M1, f_kbytes = C, f_rper = R, f_kcn = kc1, f_kstep = 128 * KP;
  };
  auto fetch_next = [&](Pair &f) __attribute__((always_inline)) {
    const int kp0 = KP == 1 ? 0 : srow / f_rper, kp1 = KP == 1 ? 0 : (srow + 128) / f_rper;
    const int row0 = min(fg * f_rper + srow - kp0 * f_rper, f_rows - 1), kb0 = fk * f_kstep + kp0 * 128 + piece * 16;
    const int row1 = min(fg * f_rper + srow + 128 - kp1 * f_rper, f_rows - 1), kb1 = fk * f_kstep + kp1 * 128 + piece * 16;
    f.lo = *reinterpret_cast<const u32x4 *>(f_w + (row0 * f_kbytes + (kb0 < f_kbytes ? kb0 : 0)));
    f.hi = *reinterpret_cast<const u32x4 *>(f_w + (row1 * f_kbytes + (kb1 < f_kbytes ? kb1 : 0)));
    if (fi + 1 < n3) {
      ++fi;
      if (++fk == f_kcn) fk = 0, ++fg;
      if (fi == n1) {
        fg = 0;
        f_w = a.w2, f_kbytes = 9 * M1, f_kcn = kc2;
      } else if (fi == n2) {
        fg = 0;
        f_w = a.w3, f_rows = C, f_kbytes = M1, f_rper = SROWS, f_kcn = kc3, f_kstep = 128;
      }
    }
  };
  struct Mul4 {
    i32x4 m, s;
  };
  auto load_params = [&](const int32_t *m, const int32_t *sh, int c) __attribute__((always_inline)) {
    return Mul4{*reinterpret_cast<const i32x4 *>(m + c), *reinterpret_cast<const i32x4 *>(sh + c)};
  };
  auto scale = [&](const Mul4 &p) __attribute__((always_inline)) {
    Scale4 sc;
    sc.m = p.m;
    sc.s = p.s;
#pragma unroll
    for (int e = 0; e < 4; ++e) sc.r[e] = 1LL << (p.s[e] - 1);
    return sc;
  };

  const TileWalk walk = tile_walk(a.ntiles);
  for (int t = walk.first; t < walk.end; t += walk.step) {
    const int n = t / a.tiles_img, tt = t - n * a.tiles_img;
    const int ty0 = (tt / a.tiles_w) * STH, tx0 = (tt - (tt / a.tiles_w) * a.tiles_w) * STW;
    const int8_t *const xn = a.x + (size_t)n * a.H * a.W * C;
    // x chunks: run `e` of the 8 KP 16-byte runs of each halo pixel, clamped into
    // the image (what lies outside only feeds y1 values that are zeroed)
    int xoff[XR], xdst[XR], xkb[XR];
#pragma unroll
    for (int j = 0; j < XR; ++j) {
      const int e = min(opaque(tid) + SNT * j, SHP * 8 * KP - 1), hp = e / (8 * KP), hy = hp / SHW, hx = hp - hy * SHW;
      const int iy = min(max(ty0 + hy - 1, 0), a.H - 1), ix = min(max(tx0 + hx - 1, 0), a.W - 1);
      xkb[j] = (e - hp * 8 * KP) * 16;
      xoff[j] = (iy * a.W + ix) * C;
      xdst[j] = hp * XS + xkb[j];
    }
    u32x4 xr0[XR], xr1[XR];
    auto xfetch = [&](int k, u32x4 (&xr)[XR]) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < XR; ++j) {
        const int kb = k * 128 * KP + xkb[j];
        xr[j] = *reinterpret_cast<const u32x4 *>(xn + (xoff[j] + (kb < C ? kb : 0)));
      }
    };
    auto xcommit = [&](int buf, const u32x4 (&xr)[XR]) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < XR; ++j) *reinterpret_cast<u32x4 *>(xbuf + buf * S::XBUF + xdst[j]) = xr[j];
    };
    fetch_start();
    fetch_next(fr0);
    xfetch(0, xr0);
    fetch_next(fr1);
    xfetch(1, xr1);
    commit(0, fr0);
    xcommit(0, xr0);
    fetch_next(fr0);
    xfetch(kc1 > 2 ? 2 : 0, xr0);
    __syncthreads();

    // ---- conv1 on the halo: requant + ReLU clamp into y1, zero outside the image
    {
      // recomputed per tile: hoisted out of the tile loop, every phase's
      // addresses would be held at once
      const int ol = opaque(lane), r = ol & 15, q = ol >> 4;
      constexpr int FGW = KP == 1 ? 8 : 4;  // waves along the filters
      const int fw = wave % FGW * 16 * NF1, pw = wave / FGW * NP1;
      int px[NP1];
#pragma unroll
      for (int p = 0; p < NP1; ++p) px[p] = min((pw + p) * 16 + r, SHP - 1) * XS + 16 * q;
      for (int g = 0; g < rg; ++g) {
        i32x4 acc[NF1][NP1] = {};
        auto chunk = [&](int k, auto odd) __attribute__((always_inline)) {
          constexpr bool ODD = decltype(odd)::value;
          constexpr int buf = ODD;
          // the next chunk to LDS, the one three ahead on its way
          commit(buf ^ 1, ODD ? fr0 : fr1);
          fetch_next(ODD ? fr0 : fr1);
          xcommit(buf ^ 1, ODD ? xr0 : xr1);
          // chunk (k + 3) mod kc1 of this row group or the next (kc1 >= 2)
          xfetch(k + 3 < kc1 ? k + 3 : k + 3 < 2 * kc1 ? k + 3 - kc1 : k + 3 - 2 * kc1, ODD ? xr0 : xr1);
          const int steps = min(2 * KP, C / 64 - k * 2 * KP);
#pragma unroll
          for (int s = 0; s < 2 * KP; ++s)
            if (s < steps) {  // uniform
              Frag16 f[NF1];
#pragma unroll
              for (int b = 0; b < NF1; ++b) f[b] = ffrag(buf, (s >> 1) * R + fw + 16 * b + r, s & 1);
#pragma unroll
              for (int p = 0; p < NP1; ++p) {
                const Frag16 v = load16(xbuf + buf * S::XBUF + px[p] + s * 64);
#pragma unroll
                for (int b = 0; b < NF1; ++b) MfmaI8::mma(acc[b][p], f[b], v);
              }
            }
          if constexpr (ODD) {
           if (k + 1 == kc1) {
#pragma unroll
            for (int b = 0; b < NF1; ++b) {
              const int f0 = g * R + fw + 16 * b;
              const Scale4 s4 = scale(load_params(a.m1, a.s1, min(f0, M1 - 16) + 4 * q));
#pragma unroll
              for (int p = 0; p < NP1; ++p) {
                const int hp = (pw + p) * 16 + r, hy = hp / SHW, hx = hp - hy * SHW;
                const bool inside = (unsigned)(ty0 + hy - 1) < (unsigned)a.H && (unsigned)(tx0 + hx - 1) < (unsigned)a.W;
                const uint32_t v = requant4(acc[b][p], s4);
                if (hp < SHP && fw + 16 * b < R && f0 < M1)
                  *reinterpret_cast<uint32_t *>(y1 + hp * YS + f0 + 4 * q) = inside ? v : 0u;
                __builtin_amdgcn_sched_barrier(0);  // one block's 64-bit values at a time
              }
            }
          }
          }
          __syncthreads();
        };
        for (int k = 0; k < kc1; k += 2) {
          chunk(k, std::false_type{});
          chunk(k + 1, std::true_type{});
        }
      }
    }

    // the residual's tile of 256 channels, one group ahead: this thread's
    // 16-byte run, its place in the tile and in the image (recomputed at each use)
    u32x4 rr;
    auto rplace = [&](int &lds, int &off, int &c) __attribute__((always_inline)) {
      const int rt = opaque(tid), o = min(rt >> 4, SOP - 1), oy = o / STW, ox = o - oy * STW;
      c = (rt & 15) * 16;
      lds = o * SOS + c;
      const bool in = rt < SOP * 16 && ty0 + oy < a.H && tx0 + ox < a.W;
      off = in ? ((ty0 + oy) * a.W + tx0 + ox) * C : 0;
      return in;
    };
    auto rfetch = [&](int g) __attribute__((always_inline)) {
      int lds, off, c;
      rplace(lds, off, c);
      c += g * SROWS;
      rr = *reinterpret_cast<const u32x4 *>(xn + (off + (c < C ? c : 0)));
    };
    auto rcommit = [&](int g) __attribute__((always_inline)) {
      int lds, off, c;
      rplace(lds, off, c);
      if (tid < SOP * 16) *reinterpret_cast<u32x4 *>(xbuf + (g % S::NOB) * SOP * SOS + lds) = rr;
    };

    // ---- conv2 (3x3) on the output pixels, k steps tap by tap
    {
      const int ol = opaque(lane), r = ol & 15, q = ol >> 4;
      constexpr int FGW = 8;
      const int fw = wave % FGW * 16 * NF2, pw = wave / FGW;
      const int o = min(pw * 16 + r, SOP - 1), oy = o / STW;
      const int px = (oy * SHW + o - oy * STW) * YS + 16 * q;
      const bool on = fw < R;  // uniform
      for (int g = 0; g < rg; ++g) {
        i32x4 acc[NF2] = {};
        Mul4 sc[NF2];
#pragma unroll
        for (int b = 0; b < NF2; ++b) sc[b] = load_params(a.m2, a.s2, min(g * R + fw + 16 * b, M1 - 16) + 4 * q);
        auto chunk = [&](int k, auto odd) __attribute__((always_inline)) {
          constexpr bool ODD = decltype(odd)::value;
          constexpr int buf = ODD;
          commit(buf ^ 1, ODD ? fr0 : fr1);
          fetch_next(ODD ? fr0 : fr1);
          if (g + 1 == rg && k + (ODD ? 1 : 2) == kc2) {  // the last pair
            if constexpr (ODD) rcommit(0);
            rfetch(ODD && rg3 > 1 ? 1 : 0);
          }
          const int ks = k * 2 * KP, steps = on ? min(2 * KP, 9 * mk - ks) : 0;
#pragma unroll
          for (int s = 0; s < 2 * KP; ++s)
            if (s < steps) {
              const int tap = a.by_mk.div(ks + s), kh = tap / 3;
              const Frag16 v = load16(y1 + px + (kh * SHW + tap - 3 * kh) * YS + (ks + s - tap * mk) * 64);
#pragma unroll
              for (int b = 0; b < NF2; ++b)
                MfmaI8::mma(acc[b], ffrag(buf, (s >> 1) * R + fw + 16 * b + r, s & 1), v);
            }
          if constexpr (ODD) {
            if (k + 1 == kc2 && on) {
#pragma unroll
              for (int b = 0; b < NF2; ++b)
                if (fw + 16 * b < R && g * R + fw + 16 * b < M1)
                  *reinterpret_cast<uint32_t *>(y2 + (pw * 16 + r) * YS + g * R + fw + 16 * b + 4 * q) =
                      requant4(acc[b], scale(sc[b]));
            }
          }
          __syncthreads();
        };
        for (int k = 0; k < kc2; k += 2) {
          chunk(k, std::false_type{});
          chunk(k + 1, std::true_type{});
        }
      }
    }

    // ---- conv3 + requant + residual + clamp, 256 channels at a time
    {
      const int ol = opaque(lane), r = ol & 15, q = ol >> 4;
      const int fw = wave % 8 * 32, pw = wave / 8, o = pw * 16 + r;
      const int px = o * YS + 16 * q;
      auto store = [&](int g) __attribute__((always_inline)) {
        int lds, off, c;
        const bool in = rplace(lds, off, c);
        if (in && g * SROWS + c < C)
          *reinterpret_cast<u32x4 *>(a.out + (size_t)n * a.H * a.W * C + (off + g * SROWS + c)) =
              *reinterpret_cast<const u32x4 *>(xbuf + (g % S::NOB) * SOP * SOS + lds);
      };
      for (int g = 0; g < rg3; ++g) {
        i32x4 acc[2] = {};
        Mul4 sc[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) sc[b] = load_params(a.m3, a.s3, min(g * SROWS + fw + 16 * b, C - 16) + 4 * q);
        auto chunk = [&](int k, auto odd) __attribute__((always_inline)) {
          constexpr bool ODD = decltype(odd)::value;
          constexpr int buf = ODD;
          commit(buf ^ 1, ODD ? fr0 : fr1);
          fetch_next(ODD ? fr0 : fr1);
          if (k == 0 && g > 0) store(g - 1);
          const int steps = min(2, mk - 2 * k);
#pragma unroll
          for (int s = 0; s < 2; ++s)
            if (s < steps) {
              const Frag16 v = load16(y2 + px + (2 * k + s) * 64);
#pragma unroll
              for (int b = 0; b < 2; ++b) MfmaI8::mma(acc[b], ffrag(buf, fw + 16 * b + r, s), v);
            }
          if constexpr (ODD) {
           if (k + 1 == kc3) {
            int8_t *const ob = xbuf + (g % S::NOB) * SOP * SOS + o * SOS;
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              if (o < SOP) {
                const Scale4 s4 = scale(sc[b]);
                uint32_t *slot = reinterpret_cast<uint32_t *>(ob + fw + 16 * b + 4 * q);
                const uint32_t res = *slot;
                uint32_t packed = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  const int v = requant(acc[b][e], s4.m[e], s4.r[e], s4.s[e]) + (int)(int8_t)(res >> (8 * e));
                  packed |= (uint32_t)clamp_i(v, 0, 127) << (8 * e);
                }
                *slot = packed;
              }
            }
            if (g + 1 < rg3) {
              rcommit(g + 1);
              if (g + 2 < rg3) rfetch(g + 2);
            }
          }
          }
          __syncthreads();
        };
        for (int k = 0; k < kc3; k += 2) {
          chunk(k, std::false_type{});
          chunk(k + 1, std::true_type{});
        }
      }
      store(rg3 - 1);
    }
    __syncthreads();  // the buffers are the next tile's
  }
}

template <int KP>
hipError_t launch_qb_stream(const QBottleneckArgs &c, hipStream_t s) {
  using S = QStreamShape<KP>;
  auto kern = qb_stream_kernel<KP>;
  QStreamArgs a{c.x, c.w1, c.w2, c.w3, c.m1, c.s1, c.m2, c.s2, c.m3, c.s3, c.out, c.H, c.W, c.C, c.M1,
                (c.W + STW - 1) / STW, 0, 0, FastDiv(c.M1 / 64)};
  a.tiles_img = a.tiles_w * ((c.H + STH - 1) / STH);
  a.ntiles = c.N * a.tiles_img;
  const size_t lds = S::lds(c.M1);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  const int cus = cached_per_kernel(reinterpret_cast<const void *>(kern), [&](int dev) {
    int n = 0;
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) == hipSuccess &&
                   hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess
               ? n : 0;
  });
  if (cus <= 0) return hipErrorInvalidValue;
  const int full = cus / kXcds * kXcds;  // one workgroup per CU: its LDS
  const int grid = a.ntiles < full ? (a.ntiles + kXcds - 1) / kXcds * kXcds : full;
  {
    npu_launch_plan p = make_plan("int8_bottleneck_stream", grid, 4, a.ntiles, 8);
    p.unit_waves = 16;
    p.load_phases = 1;  // the first chunk; later ones are in flight ahead of their use
    const double wbytes = 2.0 * c.M1 * c.C + 9.0 * c.M1 * c.M1;
    p.tile_macs = 64.0 * c.M1 * c.C + 32.0 * 9 * c.M1 * c.M1 + 32.0 * c.C * c.M1;
    p.tile_valu = 16.0 * (60.0 + 30.0 * wbytes / 32768 + 20.0 * (64.0 * c.M1 + 32.0 * c.M1 + 32.0 * c.C) / 16 / 64 / 4);
    p.tile_lds_bytes = wbytes + 2.0 * SHP * c.C + 2.0 * p.tile_macs / 16.0 / 16.0 / 64.0 * 1024;
    p.tile_load_bytes = (double)(SHP + SOP) * c.C + wbytes;
    p.tile_store_bytes = (double)SOP * c.C;
    p.hbm_bytes = 2.0 * c.N * c.H * c.W * c.C + wbytes + 4.0 * 2 * (2 * c.M1 + c.C);
    plans_add(p);
  }
  hipLaunchKernelGGL(kern, dim3(grid), dim3(SNT), lds, s, a);
  return hipGetLastError();
}

// Small filters that the tuned instances above do not cover (M1 = 64, M1 = 128
// with few channels, see launch_qbottleneck_i8): every filter block is read from L2 where it is
// used, so nothing scales the registers with the channel counts.  A workgroup
// walks 4 x 4 output tiles; per tile: the x halo (6 x 6 pixels, all C channels,
// zero outside the image) to LDS; conv1 on the halo, one unit = 16 output
// channels x 16 halo pixels, requant + ReLU clamp into y1 (zero outside the
// image: the pad before conv2); conv2, one unit = 16 channels of the 16 output
// pixels, into y2; conv3, one unit = 16 output channels, with requant, the
// residual from the halo and the clamp, stored.  The units of a phase are dealt
// round-robin over the four waves, one barrier per phase.
template <int MMAX>
__global__ __launch_bounds__(256, 1) void qb_direct_kernel(
    const int8_t *__restrict__ x, const int8_t *__restrict__ w1, const int8_t *__restrict__ w2,
    const int8_t *__restrict__ w3, const int32_t *__restrict__ m1, const int32_t *__restrict__ s1,
    const int32_t *__restrict__ m2, const int32_t *__restrict__ s2,
    const int32_t *__restrict__ m3, const int32_t *__restrict__ s3, int8_t *__restrict__ out,
    int H, int W, int C, int M1, int tiles_w, int tiles_img, int ntiles) {
  constexpr int SHW = 6, SHP = 36, SHPB = 3, CMAX = 2048;
  __shared__ __attribute__((aligned(16))) int8_t xs[SHP * (CMAX + 32)];
  __shared__ __attribute__((aligned(16))) int8_t y1[SHPB * 16 * (MMAX + 32)];
  __shared__ __attribute__((aligned(16))) int8_t y2[16 * (MMAX + 32)];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int XS = C + 32, YS = M1 + 32;  // 16-byte row reads: 32 mod 64 bytes
  const int XV = C / 16;                // 16-byte runs per halo pixel
  const int py = r / 4, px = r - py * 4, hb = py * SHW + px;
  auto params = [&](const int32_t *m, const int32_t *sh, int c) {
    Scale4 sc;
    sc.m = *reinterpret_cast<const i32x4 *>(m + c);
    sc.s = *reinterpret_cast<const i32x4 *>(sh + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) sc.r[e] = 1LL << (sc.s[e] - 1);
    return sc;
  };
  const TileWalk walk = tile_walk(ntiles);
  for (int t = walk.first; t < walk.end; t += walk.step) {
    const int n = t / tiles_img, tt = t - n * tiles_img;
    const int ty0 = (tt / tiles_w) * 4, tx0 = (tt - (tt / tiles_w) * tiles_w) * 4;
    for (int idx = tid; idx < SHP * XV; idx += 256) {
      const int hp = idx / XV, cv = idx - hp * XV, hy = hp / SHW, hx = hp - hy * SHW;
      const int iy = ty0 + hy - 1, ix = tx0 + hx - 1;
      const bool inside = (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
      const int8_t *src = x + ((size_t)(n * H + (inside ? iy : 0)) * W + (inside ? ix : 0)) * C + 16 * cv;
      *reinterpret_cast<u32x4 *>(xs + hp * XS + 16 * cv) = masked(*reinterpret_cast<const u32x4 *>(src), inside);
    }
    __syncthreads();
    // conv1: unit u = (filter block fb, halo block pb)
    for (int u = wave; u < (M1 / 16) * SHPB; u += 4) {
      const int fb = u / SHPB, pb = u - fb * SHPB;
      i32x4 acc = {0, 0, 0, 0};
      for (int c0 = 0; c0 < C; c0 += 64)
        MfmaI8::mma(acc, load16(w1 + (size_t)(fb * 16 + r) * C + c0 + 16 * q),
                    load16(xs + min(pb * 16 + r, SHP - 1) * XS + c0 + 16 * q));
      const int hp = pb * 16 + r, hy = hp / SHW, hx = hp - hy * SHW;
      const bool inside = hp < SHP && (unsigned)(ty0 + hy - 1) < (unsigned)H &&
                          (unsigned)(tx0 + hx - 1) < (unsigned)W;
      const uint32_t v = requant4(acc, params(m1, s1, fb * 16 + 4 * q));
      *reinterpret_cast<uint32_t *>(y1 + hp * YS + fb * 16 + 4 * q) = inside ? v : 0u;
    }
    __syncthreads();
    // conv2: unit = filter block fb on the 16 output pixels (pixel r: halo hb)
    for (int fb = wave; fb < M1 / 16; fb += 4) {
      i32x4 acc = {0, 0, 0, 0};
      for (int tap = 0; tap < 9; ++tap)
        for (int c0 = 0; c0 < M1; c0 += 64)
          MfmaI8::mma(acc, load16(w2 + ((size_t)(fb * 16 + r) * 9 + tap) * M1 + c0 + 16 * q),
                      load16(y1 + (hb + (tap / 3) * SHW + tap % 3) * YS + c0 + 16 * q));
      *reinterpret_cast<uint32_t *>(y2 + r * YS + fb * 16 + 4 * q) =
          requant4(acc, params(m2, s2, fb * 16 + 4 * q));
    }
    __syncthreads();
    // conv3 + requant + residual + clamp: unit = output channel block cb
    for (int cb = wave; cb < C / 16; cb += 4) {
      i32x4 acc = {0, 0, 0, 0};
      for (int c0 = 0; c0 < M1; c0 += 64)
        MfmaI8::mma(acc, load16(w3 + (size_t)(cb * 16 + r) * M1 + c0 + 16 * q),
                    load16(y2 + r * YS + c0 + 16 * q));
      const int c = cb * 16 + 4 * q;
      const Scale4 sc = params(m3, s3, c);
      const uint32_t res = *reinterpret_cast<const uint32_t *>(xs + (hb + SHW + 1) * XS + c);
      uint32_t packed = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int v = requant(acc[e], sc.m[e], sc.r[e], sc.s[e]) + (int)(int8_t)(res >> (8 * e));
        packed |= (uint32_t)clamp_i(v, 0, 127) << (8 * e);
      }
      if (ty0 + py < H && tx0 + px < W)
        *reinterpret_cast<uint32_t *>(out + ((size_t)(n * H + ty0 + py) * W + tx0 + px) * C + c) = packed;
    }
    __syncthreads();  // xs, y1 and y2 are the next tile's
  }
}

template <int MMAX>
hipError_t launch_qb_direct(const QBottleneckArgs &a, hipStream_t s) {
  const int tiles_w = (a.W + 3) / 4, tiles_img = tiles_w * ((a.H + 3) / 4), ntiles = a.N * tiles_img;
  auto kern = qb_direct_kernel<MMAX>;
  const int full = persistent_grid(kern);
  if (full <= 0) return hipErrorInvalidValue;
  const int grid = ntiles < full ? (ntiles + kXcds - 1) / kXcds * kXcds : full;
  {
    npu_launch_plan p = make_plan("int8_bottleneck_direct", grid, wg_per_cu(kern), ntiles, 8);
    p.load_phases = 4;  // the halo, then each phase's filters from L2
    p.tile_macs = 48.0 * a.M1 * a.C + 16.0 * 9 * a.M1 * a.M1 + 16.0 * a.C * a.M1;
    p.tile_valu = 4.0 * (40.0 + 30.0 * (3 * a.M1 / 16 + a.M1 / 16 + a.C / 16) / 4.0);
    p.tile_lds_bytes = 2.0 * 36 * a.C + 1024.0 * (3 * a.M1 / 16 * a.C / 64 + a.M1 / 16 * 9 * a.M1 / 64 +
                                                  a.C / 16 * a.M1 / 64);
    p.tile_load_bytes = 36.0 * a.C + 48.0 * a.M1 * a.C / 16 + 9.0 * a.M1 * a.M1 + (double)a.C * a.M1;
    p.tile_store_bytes = 16.0 * a.C;
    p.hbm_bytes = 2.0 * a.N * a.H * a.W * a.C + (double)a.M1 * a.C * 2 + 9.0 * a.M1 * a.M1 +
                  4.0 * 2 * (2 * a.M1 + a.C);
    plans_add(p);
  }
  hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, a.x, a.w1, a.w2, a.w3, a.m1,
                     a.s1, a.m2, a.s2, a.m3, a.s3, a.out, a.H, a.W, a.C, a.M1, tiles_w, tiles_img,
                     ntiles);
  return hipGetLastError();
}

bool qb_tuned(int C, int M1) {
  return (C == 256 && M1 == 64) || (C == 128 && M1 == 64) || (C == 64 && M1 == 64);
}

}  // namespace

bool qbottleneck_supported(int C, int M1) {
  return qb_tuned(C, M1) || (C >= 64 && C % 64 == 0 && C <= 2048 && M1 >= 64 && M1 % 64 == 0 && M1 <= 512);
}

hipError_t launch_qbottleneck_i8(const QBottleneckArgs &a, hipStream_t s) {
  if (a.C == 256 && a.M1 == 64) return launch_qb<256, 64>(a, s);
  if (a.C == 128 && a.M1 == 64) return launch_qb<128, 64>(a, s);
  if (a.C == 64 && a.M1 == 64) return launch_qb<64, 64>(a, s);
  if (!qbottleneck_supported(a.C, a.M1)) return hipErrorInvalidValue;
  // Filters streamed through LDS from 256 KB on.  Measured, us, streamed / read
  // from L2: 512/128 (279 KB) one 14x14 image 17.7 / 20.4, batch 32 of 7x7
  // 18.1 / 20.5; 192/192 (406 KB) 17.9 / 19.7; 1024/256 (1.1 MB) one 7x7 image
  // 30.7 / 59.6; 320/128 (229 KB) 17.5 / 15.3; 320/64 (78 KB) 14.4 / 9.2.
  const double bytes = 2.0 * a.M1 * a.C + 9.0 * a.M1 * a.M1;
  if (a.M1 < 128 || bytes < 256 * 1024) return launch_qb_direct<128>(a, s);
  // With a CU for every 4 x 4 tile, row groups that fill little of their last
  // chunks (320 filters are chunks of 256 and 64, 192 one of 192) are not worth
  // streaming for few channels: 64/320 36.1 from L2 / 41.9 streamed, 192/320 40.6
  // / 42.3, 256/320 44.0 / 42.3, 64/192 17.1 / 18.3, 128/192 19.0 / 18.5, 64/384
  // 49.8 / 47.1; in rounds 64/320 14x14 at batch 32 72.6 / 47.2.  The estimates,
  // in us: a tile's filters and channels at L2's rate, or its chunks.
  if (a.M1 <= 320 && (long long)a.N * ((a.H + 3) / 4) * ((a.W + 3) / 4) <= device_cus()) {
    const int rg = (a.M1 + SROWS - 1) / SROWS;
    const int chunks = 2 * (rg * ((a.C + 255) / 256 + (9 * a.M1 + 255) / 256) +
                            (a.C + SROWS - 1) / SROWS * ((a.M1 + 255) / 256));
    if (a.M1 >= 192 && 4.3 + 31.8e-6 * bytes + 0.0175 * a.C < 6.5 + 0.635 * chunks) return launch_qb_direct<320>(a, s);
  }
  return a.M1 >= 192 ? launch_qb_stream<1>(a, s) : launch_qb_stream<2>(a, s);
}

}  // namespace npu
