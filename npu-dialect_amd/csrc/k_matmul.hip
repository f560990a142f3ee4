// k_matmul.hip -- group `fill -> matmul -> generic(bias, act)` in f32: small
// outputs on split-K tiles of 16 x 16, large ones on tiles of the bf16 matrix
// pipe (below).
//
// Replaces the tile loops the reference wraps around the outlined call
// (FusionPass.cpp:306-359 tile-and-fuse of the consumer generic, then
// OutlineFusedGroupsPass.cpp:306-316): one launch covers the whole output.
//
// Decomposition.  The matmul+bias+ReLU shape (256x512 . 512x256) has only
// 256 output tiles of 16x16, one per CU, so each workgroup owns one 16x16
// tile and splits K across its 4 waves (split-K inside the workgroup; the
// reference's analogue is a K split with a reduce penalty,
// CostModel.cpp:798-812).  Each wave runs v_mfma_f32_16x16x4_f32 over its K
// share, the partial tiles meet in LDS, and the epilogue (bias add, act) is
// applied once while the tile is in registers: the matmul result never
// reaches HBM.
#include <type_traits>

#include "kernels.hpp"
#include "npu_device.hpp"
#include "persistent.hpp"
#include "plans.hpp"

namespace npu {

namespace {

constexpr int kWaves = 4;
constexpr int kBatch = 8;   // K chunks whose loads are all issued before their MFMAs
constexpr int kBRow = 20;   // LDS row stride of a staged B chunk, in floats (80 bytes)

// B operand staging.  The MFMA wants, per lane (column j, group q), the
// values B[k][j] of four consecutive k: a column walk, one 4-byte load per
// value.  Instead each wave loads its B rows whole -- lane l takes 16 bytes
// of row l/4 of a chunk (columns 4(l%4)..+3 of the tile), so one
// instruction moves a chunk's 16 rows x 64 bytes -- parks them in its own
// LDS slice and reads the column runs back (four 4-byte LDS reads per
// chunk).  The 80-byte row stride puts rows 4q + s of the four lane groups
// 16 banks apart: the reads are free of bank conflicts.  Each wave only
// reads what it wrote, so no barrier is needed (a wave's LDS operations
// complete in order).
//
// VEC: N % 4 == 0, so a 16-byte run is all inside a row or all past it; else
// four 4-byte loads with the column clamped.
template <bool VEC>
__global__ __launch_bounds__(kWaves * 64) void matmul_bias_act_f32_kernel(
    const float *__restrict__ A, const float *__restrict__ B,
    const float *__restrict__ bias, float *__restrict__ out, int M, int N, int K,
    int act, int tiles_n) {
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = lane & 15, q = lane >> 4;
  // Tiles in XCD-contiguous ranges (consecutive workgroups go to the eight
  // XCDs in turn, each with its own L2): an XCD's tiles share rows of A.
  const int nb = gridDim.x, b = blockIdx.x;
  const int t = nb % kXcds == 0 ? (b % kXcds) * (nb / kXcds) + b / kXcds : b;
  const int m0 = (t / tiles_n) * 16, n0 = (t % tiles_n) * 16;
  // Rows past M and columns past N read row M-1 / the last columns: they
  // only feed outputs that are never stored.  Every load is issued
  // unconditionally from a valid address and masked afterwards (a load
  // under a divergent branch would make the compiler wait for all
  // outstanding loads).
  const float *arow = A + (size_t)min(m0 + r, M - 1) * K;
  const int br = lane >> 2, bq = lane & 3;
  const int bcol = n0 + 4 * bq;
  const int bcol_v = min(bcol, N - 4);  // VEC: N >= 4
  __shared__ __attribute__((aligned(16))) float bs[kWaves][kBatch * 16 * kBRow];
  float *const myb = bs[wave];

  // K is walked in chunks of 16 (four MFMA k-steps); waves take contiguous
  // chunk ranges.  K % 4 == 0, so a lane's 4-element run of A is all in or
  // all out; a B row is in when its k is.
  const int nchunks = (K + 15) >> 4;
  const int c_begin = (wave * nchunks) / kWaves;
  const int c_end = ((wave + 1) * nchunks) / kWaves;

  // this thread's epilogue element is (row e / 16, column e % 16) of the
  // tile, e = threadIdx.x: its bias is fetched now, not after the K loop
  const int ecol = n0 + (threadIdx.x & 15);
  const float bias_e = bias ? bias[min(ecol, N - 1)] : 0.0f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  // One batch of kBatch chunks from chunk c: loads, B staged, MFMAs.  MASK:
  // the batch runs past the wave's range or past K (its last, partial
  // batch), so indices are clamped and values masked; full batches (a
  // uniform test) skip both.
  auto batch = [&](int c, auto mask) __attribute__((always_inline)) {
    constexpr bool MASK = decltype(mask)::value;
    Frag16 a[kBatch], bv[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int k = (c + u) * 16 + 4 * q, kb = (c + u) * 16 + br;
      const bool ok = !MASK || (c + u < c_end && k < K), okb = !MASK || (c + u < c_end && kb < K);
      a[u] = load16(arow + (ok ? k : 0));
      const float *brow = B + (size_t)(okb ? kb : 0) * N;
      if constexpr (VEC) {
        bv[u] = load16(brow + bcol_v);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[u].f[e] = brow[min(bcol + e, N - 1)];
      }
      if constexpr (MASK) {
        a[u].u = masked(a[u].u, ok);
        bv[u].u = masked(bv[u].u, okb);
      }
    }
    // chunk by chunk, so each chunk's MFMAs wait only for its own loads
    // (issued in order) and run while the later chunks arrive
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      *reinterpret_cast<u32x4 *>(myb + (u * 16 + br) * kBRow + 4 * bq) = bv[u].u;
      // the reads below take values other lanes of this wave just wrote:
      // order them after the writes explicitly
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
      for (int s = 0; s < 4; ++s)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u].f[s], myb[(u * 16 + 4 * q + s) * kBRow + r], acc, 0, 0, 0);
    }
  };
  for (int c = c_begin; c < c_end; c += kBatch) {
    if (c + kBatch <= c_end && (c + kBatch) * 16 <= K)
      batch(c, std::false_type{});
    else
      batch(c, std::true_type{});
  }

  // Split-K reduction through LDS, then the fused epilogue.
  __shared__ float red[kWaves][256];
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][(4 * q + i) * 16 + r] = acc[i];
  __syncthreads();
  const ActBounds ab = act_bounds(act);
  static_assert(kWaves * 64 == 256, "one epilogue element per thread");
  const int e = threadIdx.x;
  float sum = red[0][e];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) sum += red[w][e];
  const int row = m0 + (e >> 4);
  if (row < M && ecol < N) out[(size_t)row * N + ecol] = act_clamp(bias ? sum + bias_e : sum, ab);
}

// ---- large outputs: tiles on the bf16 matrix pipe ------------------------------
//
// A BM x BN tile per workgroup of WR x WC waves, K in steps of 32.  Each
// value is split into its three bf16 parts as it is staged (npu_device.hpp; the
// first part rounded to nearest, as truncating it lost up to two bits of a
// product: 80.0 us against 78.6 at 2000x1024x3000) and a product takes six bf16
// MFMAs, 2.7 times the f32 matrix rate, at f32 accuracy.  A's rows go to LDS as
// records of three 64-byte part runs; B's rows as 16-column strips per part,
// read back as column runs by the transposing LDS read.  The operands are
// swapped (B's fragment first), so a lane ends with four consecutive columns of
// one row: 16-byte stores.  Two LDS buffers, one barrier per step: the next
// step's runs are split and written and the one after's loaded while this one
// is multiplied.
//
// What bounds it: the MFMAs and the split's vector work (34 instructions per
// 16-byte run), which two waves per SIMD overlap; the larger the tile, the
// fewer splits per product.
//
// A value outside the split's domain (Inf, NaN, |v| >= 2^55, 0 < |v| < 2^-55: the
// tail of an exponential) makes its workgroup start over, soon after staging it,
// with f32 MFMAs on the same tiles staged unsplit.  us with such a value in every
// row's first (middle) k, 16x16 tiles / six products first and the operands then
// from memory / so: 1024x1024x1024 44 / 94 / 33 (58), 1024x512x1024 24 / 52 / 21
// (26), 20000x512x64 28 / 88 / 28 (37), 2000x1024x3000 410 / 323 / 117 (182); the
// tests for it take 2 % where there is none.
template <int BM, int BN, int WR, int WC>
struct X6Shape {
  static constexpr int NT = 64 * WR * WC, KC = 32;
  static constexpr int TM = BM / WR / 16, TN = BN / WC / 16;  // 16 x 16 blocks of a wave
  static constexpr int AREC = 3 * 64 + 32;                    // A row: 32 mod 64 bytes
  static constexpr int STRIPS = BN / 16, SB = KC * 32 + 32;   // B strip: 8 banks past a multiple of 64
  static constexpr int ABYTES = BM * AREC, BUF = ABYTES + 3 * STRIPS * SB;
  static constexpr int AR = BM * 8 / NT;                      // 16-byte runs per thread and step
  static constexpr int BITEMS = KC * BN / 4, BR = (BITEMS + NT - 1) / NT;
  // unsplit: A rows 16 bytes past 128, B rows 16 past a multiple of 128 (a lane
  // group's 16 words of four rows use every bank once)
  static constexpr int AF = KC * 4 + 16, BF = BN * 4 + 16;
  static_assert(BM * AF + KC * BF <= BUF, "the unsplit tile fits a buffer");
  static_assert(BM * 8 % NT == 0 && TM >= 1 && TN >= 1, "whole runs, whole blocks");
};

template <int BM, int BN, int WR, int WC, bool VEC>
__global__ __launch_bounds__(64 * WR * WC, 2) void matmul_x6_kernel(
    const float *__restrict__ A, const float *__restrict__ B, const float *__restrict__ bias,
    float *__restrict__ out, int M, int N, int K, int act, int tiles_m, int tiles_n, int xm) {
  using S = X6Shape<BM, BN, WR, WC>;
  constexpr int NT = S::NT, TM = S::TM, TN = S::TN, KC = S::KC;
  extern __shared__ __attribute__((aligned(16))) unsigned char x6mem[];
  __shared__ int missed;
  int tm, tn;
  if (!xcd_tile(tiles_m, tiles_n, xm, tm, tn)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, q = lane >> 4;
  const int m0 = tm * BM, n0 = tn * BN;
  const int wr = wave % WR, wc = wave / WR;
  if (tid == 0) missed = 0;

  // Runs past M or N read the last row or columns (they feed outputs that
  // are not stored); runs past K are zeroed when they are split.
  const float *ap[S::AR];
  uint32_t adst[S::AR];
  const int ak = (tid & 7) * 4;
#pragma unroll
  for (int i = 0; i < S::AR; ++i) {
    const int row = (tid + NT * i) >> 3;
    ap[i] = A + (size_t)min(m0 + row, M - 1) * K;
    adst[i] = (uint32_t)(row * S::AREC + ak * 2);
  }
  int bk[S::BR], bcol[S::BR];
  uint32_t bdst[S::BR];
#pragma unroll
  for (int i = 0; i < S::BR; ++i) {
    const int it = min(tid + NT * i, S::BITEMS - 1);
    const int c = it % (BN / 4) * 4;
    bk[i] = it / (BN / 4);
    bcol[i] = n0 + c;
    bdst[i] = (uint32_t)(S::ABYTES + (c >> 4) * S::SB + strip_row(bk[i]) * 32 + (c & 15) * 2);
  }
  u32x4 av[S::AR], bv[S::BR];
  auto fetch = [&](int k0) __attribute__((always_inline)) {
    const int ka = min(k0 + ak, K - 4);
#pragma unroll
    for (int i = 0; i < S::AR; ++i) av[i] = *reinterpret_cast<const u32x4 *>(ap[i] + ka);
#pragma unroll
    for (int i = 0; i < S::BR; ++i) {
      const float *row = B + (size_t)min(k0 + bk[i], K - 1) * N;
      if constexpr (VEC) {
        bv[i] = *reinterpret_cast<const u32x4 *>(row + min(bcol[i], N - 4));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) bv[i][e] = __float_as_uint(row[min(bcol[i] + e, N - 1)]);
      }
    }
  };
  SplitDomainBounds dom;
  auto commit = [&](int k0, unsigned char *buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < S::AR; ++i) {
      const u32x4 v = masked(av[i], k0 + ak < K);
      dom.fold(v);
      const Parts4 p = split_parts_rn(v);
      *reinterpret_cast<uint2 *>(buf + adst[i]) = p.h;
      *reinterpret_cast<uint2 *>(buf + adst[i] + 64) = p.m;
      *reinterpret_cast<uint2 *>(buf + adst[i] + 128) = p.l;
    }
#pragma unroll
    for (int i = 0; i < S::BR; ++i) {
      const u32x4 v = masked(bv[i], k0 + bk[i] < K);
      dom.fold(v);
      const Parts4 p = split_parts_rn(v);
      if (NT * (i + 1) <= S::BITEMS || tid + NT * i < S::BITEMS) {
        *reinterpret_cast<uint2 *>(buf + bdst[i]) = p.h;
        *reinterpret_cast<uint2 *>(buf + bdst[i] + S::STRIPS * S::SB) = p.m;
        *reinterpret_cast<uint2 *>(buf + bdst[i] + 2 * S::STRIPS * S::SB) = p.l;
      }
    }
  };

  f32x4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const unsigned char *buf) __attribute__((always_inline)) {
    Frag16 b[TN][3];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int p = 0; p < 3; ++p)
        b[j][p] = read_wfrag(buf + S::ABYTES + (p * S::STRIPS + wc * TN + j) * S::SB, 0, lane);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      Frag16 a[3];
      const unsigned char *rec = buf + (wr * (BM / WR) + 16 * i + r) * S::AREC + q * 16;
#pragma unroll
      for (int p = 0; p < 3; ++p) a[p].u = *reinterpret_cast<const u32x4 *>(rec + 64 * p);
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += dot_x6(b[j], a);
    }
  };
  const int steps = (K + KC - 1) / KC;
  fetch(0);
  commit(0, x6mem);
  fetch(KC);
  __syncthreads();
  // The domain is tested after 2, 8, 32, ... steps (a test costs about 0.1 us):
  // data that has such values mostly has them throughout, and one that is
  // staged later costs the steps done before it.
  bool out_of_domain = false;
  for (int s = 0; s < steps && !out_of_domain;) {
    for (const int end = min(max(2, 4 * s), steps); s < end; ++s) {
      multiply(x6mem + (s & 1) * S::BUF);
      if (s + 1 < steps) {
        commit((s + 1) * KC, x6mem + ((s + 1) & 1) * S::BUF);
        fetch((s + 2) * KC);
      }
      __syncthreads();
    }
    if (__builtin_amdgcn_ballot_w64(dom.miss()) != 0 && lane == 0) missed = 1;
    __syncthreads();
    out_of_domain = missed;
  }
  if (out_of_domain) {
    // f32 MFMAs: step t of a run of 16 takes k = 4q + t of lane group q
    // (places in LDS from an opaque lane: none is held through the loop above)
    const int tid = opaque(threadIdx.x), r = tid & 15, q = (tid >> 4) & 3;
    auto commit_f32 = [&](int k0, unsigned char *buf) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < S::AR; ++i)
        *reinterpret_cast<u32x4 *>(buf + ((tid + NT * i) >> 3) * S::AF + ak * 4) = masked(av[i], k0 + ak < K);
#pragma unroll
      for (int i = 0; i < S::BR; ++i)
        if (NT * (i + 1) <= S::BITEMS || tid + NT * i < S::BITEMS)
          *reinterpret_cast<u32x4 *>(buf + BM * S::AF + (tid + NT * i) / (BN / 4) * S::BF + (tid + NT * i) % (BN / 4) * 16) =
              masked(bv[i], k0 + bk[i] < K);
    };
    auto multiply_f32 = [&](const unsigned char *buf) __attribute__((always_inline)) {
#pragma unroll
      for (int run = 0; run < KC / 16; ++run) {
        Frag16 af[TM], bf[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
          af[i] = load16(buf + (wr * (BM / WR) + 16 * i + r) * S::AF + run * 64 + q * 16);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t)
            bf[j].f[t] = *reinterpret_cast<const float *>(buf + BM * S::AF + (run * 16 + 4 * q + t) * S::BF +
                                                          (wc * (BN / WC) + 16 * j + r) * 4);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) MfmaF32::step(acc[i][j], bf[j], af[i], t);
      }
    };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    fetch(0);
    commit_f32(0, x6mem);
    fetch(KC);
    __syncthreads();
    for (int s = 0; s < steps; ++s) {
      multiply_f32(x6mem + (s & 1) * S::BUF);
      if (s + 1 < steps) {
        commit_f32((s + 1) * KC, x6mem + ((s + 1) & 1) * S::BUF);
        fetch((s + 2) * KC);
      }
      __syncthreads();
    }
  }

  const ActBounds ab = act_bounds(act);
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wc * (BN / WC) + 16 * j + 4 * q;
    f32x4 bj = {0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma unroll
      for (int e = 0; e < 4; ++e) bj[e] = bias[min(n + e, N - 1)];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + wr * (BM / WR) + 16 * i + r;
      if (m >= M) continue;
      f32x4 v = acc[i][j];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = act_clamp(bias ? v[e] + bj[e] : v[e], ab);
      float *o = out + (size_t)m * N + n;
      if constexpr (VEC) {
        if (n < N) *reinterpret_cast<f32x4 *>(o) = v;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) o[e] = v[e];
      }
    }
  }
}

template <int BM, int BN, int WR, int WC, bool VEC>
hipError_t launch_x6(const char *name, const MatmulArgs &a, hipStream_t s) {
  using S = X6Shape<BM, BN, WR, WC>;
  auto kern = matmul_x6_kernel<BM, BN, WR, WC, VEC>;
  // the dynamic LDS limit, raised once per device
  const int ok = cached_per_kernel(reinterpret_cast<const void *>(kern), [&](int) {
    return hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                               hipFuncAttributeMaxDynamicSharedMemorySize, 2 * S::BUF) == hipSuccess
               ? 1 : 0;
  });
  if (!ok) return hipErrorInvalidValue;
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  const int G = tiles_m * tiles_n, grid = (G + kXcds - 1) / kXcds * kXcds;
  const double steps = (a.K + S::KC - 1) / S::KC;
  npu_launch_plan p = make_plan(name, G, wg_per_cu(kern, S::NT, 2 * S::BUF), G, 16);
  p.unit_waves = WR * WC;
  p.load_phases = 1;
  p.tile_macs = 6.0 * BM * BN * S::KC * steps;
  p.tile_valu = WR * WC * (steps * (34.0 * (S::AR + S::BR) + 30.0) + 16.0 * S::TM * S::TN + 100.0);
  p.tile_lds_bytes = steps * (S::BUF + WR * WC * 3.0 * 1024 * (S::TM + S::TN));
  p.tile_load_bytes = steps * 4.0 * S::KC * (BM + BN);
  p.tile_store_bytes = 4.0 * BM * BN;
  p.hbm_bytes = 4.0 * ((double)a.M * a.K + (double)a.K * a.N + (double)a.M * a.N + (a.bias ? a.N : 0));
  plans_add(p);
  const int xm = xcd_block_grid(tiles_m, tiles_n, BM, BN, true);
  hipLaunchKernelGGL(kern, dim3(grid), dim3(S::NT), 2 * S::BUF, s, a.A, a.B, a.bias, a.out, a.M, a.N,
                     a.K, a.act, tiles_m, tiles_n, xm);
  return hipGetLastError();
}

template <int BM, int BN, int WR, int WC>
hipError_t launch_x6(const char *name, const MatmulArgs &a, hipStream_t s) {
  return a.N % 4 == 0 ? launch_x6<BM, BN, WR, WC, true>(name, a, s) : launch_x6<BM, BN, WR, WC, false>(name, a, s);
}

// Which tiles: the ones whose rounds over the CUs take the least time, by the
// rates measured for each (us per k step of 32 and round, and per tile of
// 16 x 16).  A count of tiles alone does not tell: one row against 32 000
// columns counts 334 tiles of 256 x 96, of which hardly anything lies inside
// the matrix.  So the split-K tiles of 16 x 16 are kept below 48 rows or 32
// columns (three quarters and half of a 64 x 64 tile), and below kMinMid tiles of
// 64 x 64, where the rates are least certain, for anything thinner than a tile
// or without a fifth to gain.  Over 260 shapes the choice takes 1.2 % longer than
// the fastest of the three (geometric mean).  Measured, us, as 16x16 / 64x64 / 256x96:
// 2000x1024x3000 (256 tiles of 256 x 96) 420 / 124 / 83; 1500x1024x4096 (258)
// 255 / 119 / 147; 2026x384x6040 (504) 318 / 94 / 69; 1024x1024x1024 (256 of
// 64 x 64) 43 / 29 / 73; 225x1520x2234 (140) 87 / 51 / 117; 1x512x32000 (500)
// 12.7 / 22.7 / 76; 16x512x32000 15.5 / 23.1 / 76; 32x512x32000 26.2 / 24.4 / 77;
// 64x512x32000 48 / 24 / 79; 50000x256x32 (782) 36.5 / 24.7 / 24;
// 50000x256x10 (782) 27.3 / 27.5 / 25; 4521x508x36 (71) 8.3 / 16.0 / -;
// 1x484x28358 (444) 23.9 / 27.3 / -; 1980x360x158 (93) 14.3 / 16.3 / -.
// Error against 64 bits, relative 2-norm, x6 tiles / 16x16: K = 4 2.9e-8 /
// 4.0e-8, 44 4.4e-8 / 8.0e-8, 256 6.8e-8 / 1.5e-7, 1024 1.1e-7 / 2.9e-7.
enum class MatmulTile { k16x16, k64x64, k256x96 };

constexpr int kMinMid = 176;

MatmulTile matmul_tile(const MatmulArgs &a) {
  const int cus = device_cus();
  auto tiles = [&](int bm, int bn) { return (long long)((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn); };
  auto rounds = [&](long long t) { return (double)((t + cus - 1) / cus); };
  const long long mid = tiles(64, 64);
  const int least = mid < kMinMid ? 64 : 32;
  if (a.M < (least > 48 ? least : 48) || a.N < least) return MatmulTile::k16x16;
  const double steps = (a.K + 31) / 32;
  // a row of B that is no multiple of 16 bytes is loaded word by word
  const double t16 = 4.0 + tiles(16, 16) * (a.N % 4 == 0 ? 0.003 + 0.0003 * steps : 0.004 + 0.0006 * steps);
  // two workgroups of 64 x 64 share a CU, one of 256 x 96 has it alone
  const double t64 = 5.0 + steps * (mid <= cus ? 0.88 : 0.58 * rounds(mid));
  const double t256 = 6.0 + steps * 2.3 * rounds(tiles(256, 96));
  if (t16 * (mid < kMinMid ? 0.8 : 1.0) <= (t64 < t256 ? t64 : t256)) return MatmulTile::k16x16;
  return t64 <= t256 ? MatmulTile::k64x64 : MatmulTile::k256x96;
}

}  // namespace

hipError_t launch_matmul_bias_act_f32(const MatmulArgs &a, hipStream_t s) {
  const MatmulTile tile = matmul_tile(a);
  if (tile == MatmulTile::k256x96) return launch_x6<256, 96, 4, 2>("matmul_f32_bf16x6_256x96", a, s);
  if (tile == MatmulTile::k64x64) return launch_x6<64, 64, 2, 2>("matmul_f32_bf16x6_64x64", a, s);
  const int tiles_n = (a.N + 15) / 16, tiles = tiles_n * ((a.M + 15) / 16);
  const int nchunks = (a.K + 15) / 16;
  const bool vec = a.N % 4 == 0;
  auto kern = vec ? matmul_bias_act_f32_kernel<true> : matmul_bias_act_f32_kernel<false>;
  npu_launch_plan p = make_plan("matmul_bias_act_f32", tiles, wg_per_cu(kern), tiles, 32);
  const int batches = ((nchunks + kWaves - 1) / kWaves + kBatch - 1) / kBatch;
  p.load_phases = batches;
  p.tile_macs = 16.0 * 16 * nchunks * 16;
  // Vector instructions per wave, from the compiled loops: 60 to set up and
  // write the split-K partials; 62 per full batch of kBatch K chunks (the
  // B rows' 64-bit addresses, LDS offsets), 146 for a partial one (indices
  // clamped, values masked); 19 per epilogue pass.
  const int cpw = (nchunks + kWaves - 1) / kWaves;
  const bool partial = cpw % kBatch != 0 || nchunks % kWaves != 0 || a.K % 16 != 0;
  p.tile_valu = kWaves * (60.0 + 62.0 * batches + (partial ? 84.0 : 0.0) +
                          19.0 * ((256 + kWaves * 64 - 1) / (kWaves * 64)));
  p.tile_lds_bytes = 2.0 * 16 * nchunks * 16 * 4 +           // B chunks staged, read back
                     2.0 * kWaves * 256 * 4;                  // partials written, read
  p.tile_load_bytes = 2.0 * 16 * nchunks * 16 * 4;           // 16 rows of A, 16 columns of B
  p.tile_store_bytes = 16.0 * 16 * 4;
  p.hbm_bytes = 4.0 * ((double)a.M * a.K + (double)a.K * a.N + (double)a.M * a.N + (a.bias ? a.N : 0));
  plans_add(p);
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(kWaves * 64), 0, s, a.A, a.B, a.bias, a.out, a.M, a.N,
                     a.K, a.act, tiles_n);
  return hipGetLastError();
}

}  // namespace npu
