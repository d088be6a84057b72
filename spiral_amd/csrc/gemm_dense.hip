// Prefill products of many rows: Y[m][n] = sum_k X[m][k] * W[n][k] over weights
// dequantized once to bf16 in the caller's workspace (spiral_dequant_bf16), then
// one bf16 MFMA product with both operands brought to LDS by direct loads.
//
// The fused GEMM (gemm.hip) turns each weight into bf16 once per 128 rows of X,
// and that VALU work adds to its MFMA time. From a few hundred rows on one
// pass over the matrix (a quarter of its bytes in, two bytes a weight out)
// costs less than repeating it.
//
// dense_kernel: one workgroup of 8 waves per BM x BN tile (BM = 64 MF, BN =
// 32 NF), k steps of 64, two or three LDS stages of each operand (Stages; 160 KiB
// at 256 x 256), one workgroup a CU, two waves a SIMD.
//  - Staging: buffer loads straight into LDS, 1 KiB an instruction: 8 rows of
//    128 bytes, so a lane group of 8 reads one whole line. The 16-byte chunks
//    of a row are stored permuted (chunk c of row r at c ^ (r / 2 % 8)) so that
//    the MFMA operand reads, 16 rows x one chunk, touch every bank once. The
//    permutation is in the lanes' global offsets; LDS is written linearly.
//  - Wave (wm, wn) = (w / 2, w % 2) owns 16 MF rows of X and 16 NF rows of W.
//    v_mfma_f32_16x16x32_bf16 takes W as its first operand, so a lane's four
//    results are four consecutive outputs of one row of Y.
//  - A step's two k halves have an operand register set each. Half 1 is read
//    from LDS while half 0 multiplies, and the next step's half 0 while half 1
//    multiplies; the barrier lies between them, when the wave holds all of the
//    step's operands in registers. So one barrier a step both publishes the
//    next stage and frees this one. LDS reads and direct loads are issued one
//    at a time between MFMAs: issued together they fill their queues, and the
//    wave's next MFMA waits behind them.
//
// Measured, Q4_K 14336 x 4096, 2048 rows of x, bf16 out: 344 us fused, 217 us
// here (28 us the dequantization, 190 us the product, 1.27 PFLOP/s; a dense
// library product of this shape takes 209 us). What bounds it: with the direct
// loads left out the product takes 172 us, at the 1.95 GHz the clock falls to
// under this load; with the MFMAs and LDS reads left out, 174 us. The loads are
// bound by the lines a CU keeps in flight (about 80) against the latency of
// filling L2: reading four k steps over and over, from L2, they take 86 us.
// K-sliced weights and plain stores of the dequantized weights made no difference.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "dequant_impl.h"

namespace spiral {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr int kThreads = 512, kBK = 64;
constexpr int kRowBytes = kBK * 2;
constexpr int kWaitLds = 0xC07F;  // s_waitcnt lgkmcnt(0)

// Tile index for workgroup b: consecutive workgroups go to consecutive XCDs,
// so XCD x gets a contiguous range of the tile order (the first `grid % 8`
// XCDs one more).
__device__ __forceinline__ uint32_t xcd_order(uint32_t b, uint32_t grid) {
  const uint32_t x = b & 7u, q = grid >> 3, r = grid & 7u;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// Bytes of an X and a W stage (W rows rounded up to whole loads by all waves),
// and how many of each LDS holds: three where both fit, else two of X and, where
// they fit, three of W. (4096 x 4096, 768 rows, 128 x 128 tiles: two of X and three
// of W 60 us, three of both 50.8, five 50.9.)
constexpr int kLdsBytes = 160 * 1024;
template <int MF, int NF>
struct Stages {
  static constexpr int kX = 64 * MF * kRowBytes, kW = 64 * ((NF + 1) / 2) * kRowBytes;
  static constexpr int kNX = 3 * (kX + kW) <= kLdsBytes ? 3 : 2;
  static constexpr int kNW = kNX * kX + 3 * kW <= kLdsBytes ? 3 : 2;
  static constexpr int kBytes = kNX * kX + kNW * kW;
};

// Scheduling of one k half: a load and an LDS read behind each of the first
// MFMAs, so that neither queue blocks the wave's issue while the matrix core idles.
template <int MFMAS, int READS, int LOADS>
__device__ __forceinline__ void interleave() {
  constexpr int kMfma = 0x8, kVmem = 0x10, kDsRead = 0x100;
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    __builtin_amdgcn_sched_group_barrier(kMfma, 1, 0);
    __builtin_amdgcn_sched_group_barrier(kVmem, 1, 0);
  }
#pragma unroll
  for (int i = 0; i < READS; ++i) {
    __builtin_amdgcn_sched_group_barrier(kMfma, LOADS > 0 ? 1 : 2, 0);
    __builtin_amdgcn_sched_group_barrier(kDsRead, 1, 0);
  }
  __builtin_amdgcn_sched_group_barrier(kMfma, MFMAS, 0);
  __builtin_amdgcn_sched_barrier(0);
}

template <int MF, int NF, bool F32_OUT>
__global__ void __launch_bounds__(kThreads, 2)
    dense_kernel(const uint16_t* __restrict__ x, uint32_t ldx, uint32_t m, const uint16_t* __restrict__ wb, uint32_t n,
                 uint32_t k, void* __restrict__ y, int64_t ldy, uint32_t tiles_m, uint32_t tiles_n,
                 uint32_t flush_steps) {
  constexpr int BM = 64 * MF, BN = 32 * NF;
  using S = Stages<MF, NF>;
  extern __shared__ __align__(1024) uint8_t smem[];
  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wm = wave >> 1, wn = wave & 1u;

  // Tiles in column blocks of 8 n-tiles, m fastest inside a block: the tiles
  // an XCD runs together share X and W rows in its L2.
  const uint32_t t = xcd_order(blockIdx.x, gridDim.x);
  const uint32_t per = 8 * tiles_m, blk = t / per, in = t - blk * per;
  const uint32_t bw = min(8u, tiles_n - 8 * blk);
  const uint32_t tm = in / bw, tn = 8 * blk + (in - tm * bw);
  const uint32_t m0 = tm * BM, n0 = tn * BN;

  // Rows past m or n are clamped to the last row: their products are not stored.
  const uint32_t xr = min(m - 1 - m0, BM - 1u), wr = min(n - 1 - n0, BN - 1u);  // last rows of the tile
  const __amdgpu_buffer_rsrc_t X = buffer_rsrc(x + static_cast<int64_t>(m0) * ldx, (xr * ldx + k) * 2);
  const __amdgpu_buffer_rsrc_t W = buffer_rsrc(wb + static_cast<int64_t>(n0) * k, (wr * k + k) * 2);
  // Lane's offsets: the wave's i-th X (W) instruction brings rows 64 i + 8 wave
  // .. + 7 of the tile's X (W) rows. With an odd NF the last W load of waves
  // 4..7 lies outside the tile: past the buffer's end, so it fetches nothing.
  constexpr int kWi = (NF + 1) / 2;
  const uint32_t r0 = 8 * wave + (lane >> 3), c0 = ((lane & 7u) ^ ((r0 >> 1) & 7u)) * 16;
  uint32_t xoff[MF], woff[kWi];
#pragma unroll
  for (int i = 0; i < MF; ++i) xoff[i] = min(64 * i + r0, xr) * ldx * 2 + c0;
#pragma unroll
  for (int i = 0; i < kWi; ++i) woff[i] = 64 * i + r0 < BN ? min(64 * i + r0, wr) * k * 2 + c0 : 0x80000000u;
  // X stages, then W stages; a stage is named by its byte offset.
  auto load_x = [&](uint32_t at, uint32_t step) {
#pragma unroll
    for (int i = 0; i < MF; ++i) dma16(X, smem + at + wave * 1024 + i * 8192, xoff[i], step * kRowBytes);
  };
  auto load_w = [&](uint32_t at, uint32_t step) {
#pragma unroll
    for (int i = 0; i < kWi; ++i)
      dma16(W, smem + S::kNX * S::kX + at + wave * 1024 + i * 8192, woff[i], step * kRowBytes);
  };

  // Operand reads: fragment row l % 16, chunk 4 h + l / 16 of k half h. Rows
  // are 16 apart from fragment to fragment, so the permutation is the lane's.
  const uint32_t fr = lane & 15u;
  const uint32_t rd = fr * kRowBytes + (((lane >> 4) ^ ((fr >> 1) & 7u)) * 16);
  const uint32_t rx = (wm * 16 * MF) * kRowBytes + rd, rw = S::kNX * S::kX + (wn * 16 * NF) * kRowBytes + rd;
  struct Frags {
    bf16x8_t x[MF], w[NF];
  };
  auto read = [&](Frags& f, uint32_t xat, uint32_t wat, int h) {
#pragma unroll
    for (int j = 0; j < NF; ++j)
      f.w[j] = *reinterpret_cast<const bf16x8_t*>(smem + wat + ((rw ^ (h * 64)) + j * 16 * kRowBytes));
#pragma unroll
    for (int i = 0; i < MF; ++i)
      f.x[i] = *reinterpret_cast<const bf16x8_t*>(smem + xat + ((rx ^ (h * 64)) + i * 16 * kRowBytes));
  };
  f32x4_t acc[NF][MF];
#pragma unroll
  for (int j = 0; j < NF; ++j)
#pragma unroll
    for (int i = 0; i < MF; ++i) acc[j][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int i = 0; i < MF; ++i)
        acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[j], f.x[i], acc[j][i], 0, 0, 0);
  };
  // The wave's loads up to the next step's have landed (they retire in order;
  // `newer` later ones may be in flight) and its LDS reads are done, then the
  // same of every wave.
  auto publish = [&](auto newer) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(newer)::value) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // Loads behind the next step's at a publish: the whole of the steps after it,
  // or the W of the one after it, which is requested last.
  constexpr int kNewer = (S::kNX - 2) * MF + (S::kNW - 2) * kWi;
  auto wrap = [](uint32_t at, uint32_t by, uint32_t end) { return at + by == end ? 0u : at + by; };

  // F32 results keep short chains of fp32 additions: every `flush_steps` steps
  // the accumulators are added to a second set and cleared. bf16 results are one
  // chain over the k range and keep the registers for a wider tile.
  f32x4_t sum[F32_OUT ? NF : 1][F32_OUT ? MF : 1];
  auto flush = [&]() {
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int i = 0; i < MF; ++i) {
        sum[j][i] += acc[j][i];
        acc[j][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
  };
  if constexpr (F32_OUT) {
#pragma unroll
    for (int j = 0; j < NF; ++j)
#pragma unroll
      for (int i = 0; i < MF; ++i) sum[j][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }

  const uint32_t steps = k / kBK;
  Frags f0, f1;
#pragma unroll
  for (int i = 0; i < S::kNW; ++i) {
    if (i < S::kNX) load_x(i * S::kX, min(static_cast<uint32_t>(i), steps - 1));
    if (i < S::kNW) load_w(i * S::kW, min(static_cast<uint32_t>(i), steps - 1));
  }
  publish(std::integral_constant<int, MF + kWi + kNewer>());
  read(f0, 0, 0, 0);
  uint32_t xat = 0, wat = 0, left = flush_steps;
#pragma unroll 1
  for (uint32_t s = 0; s + 1 < steps; ++s) {
    const uint32_t xn = wrap(xat, S::kX, S::kNX * S::kX), wn_ = wrap(wat, S::kW, S::kNW * S::kW);
    // f0's reads ran under the multiplies of f1: waiting for them here, before
    // f1's reads are issued, keeps the compiler from waiting for both below.
    __builtin_amdgcn_s_waitcnt(kWaitLds);
    read(f1, xat, wat, 1);
    multiply(f0);
    interleave<MF * NF, MF + NF, 0>();
    publish(std::integral_constant<int, kNewer>());
    // Past the last step the last one is loaded again, which keeps the counts.
    load_x(xat, min(s + S::kNX, steps - 1));
    load_w(wat, min(s + S::kNW, steps - 1));
    xat = xn, wat = wn_;
    read(f0, xat, wat, 0);
    multiply(f1);
    interleave<MF * NF, MF + NF, MF + kWi>();
    if constexpr (F32_OUT) {
      if (--left == 0) {
        flush();
        left = flush_steps;
      }
    }
  }
  read(f1, xat, wat, 1);
  multiply(f0);
  multiply(f1);
  if constexpr (F32_OUT) flush();
  publish(std::integral_constant<int, 0>());  // no load may be in flight when the workgroup's LDS is given back

  // Lane l holds Y[.. + l % 16][.. + 4 (l / 16) + e] of each fragment.
  using OutT = typename std::conditional<F32_OUT, float, uint16_t>::type;
  OutT* Y = static_cast<OutT*>(y);
#pragma unroll
  for (int i = 0; i < MF; ++i) {
    const uint32_t gm = m0 + (wm * MF + i) * 16 + fr;
    if (gm >= m) continue;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      const uint32_t gn = n0 + (wn * NF + j) * 16 + 4 * (lane >> 4);
      OutT* dst = Y + gm * ldy + gn;
      if constexpr (F32_OUT) {
        const f32x4_t a = sum[j][i];
        if (gn + 4 <= n && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
          *reinterpret_cast<f32x4_t*>(dst) = a;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (gn + e < n) dst[e] = a[e];
        }
      } else {
        const f32x4_t a = acc[j][i];
        const uint32_t lo = pack_bf16x2(a[0], a[1]), hi = pack_bf16x2(a[2], a[3]);
        if (gn + 4 <= n && (reinterpret_cast<uintptr_t>(dst) & 7u) == 0) {
          *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
        } else {
          const uint32_t v[2] = {lo, hi};
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (gn + e < n) dst[e] = static_cast<uint16_t>(v[e / 2] >> (16 * (e & 1)));
        }
      }
    }
  }
}

// Tiles (64 MF rows of X x 32 NF rows of W) and their average k step, ns; F32
// results need registers for two accumulator sets, so their tiles stop at NF = 5.
struct Tile {
  int mf, nf, step_ns;
};
constexpr Tile kTiles[] = {{4, 8, 1330}, {4, 7, 1200}, {4, 6, 1030}, {4, 5, 960}, {4, 4, 730}, {2, 4, 510}};

// Estimated nanoseconds of the product with tile t: rounds of one workgroup a
// CU, whose steps take their MFMAs (16 clocks each, two waves a SIMD, and the
// barrier) or their loads. A CU keeps about 80 lines in flight, so loads run at
// about 25 bytes a clock while L2 is being filled (47 when every line is in L2
// already). Measured steps: 256 x 224 1.45 us, 256 x 128 0.90 us, 128 x 128 0.62 us.
int64_t tile_ns(const Tile& t, int64_t m, int64_t n, int64_t k) {
  const int64_t rounds = ceil_div(ceil_div(m, 64 * t.mf) * ceil_div(n, 32 * t.nf), device_cu_count());
  const int64_t mfma = 80 * t.mf * t.nf + 300, load = (64 * t.mf + 32 * t.nf) * kRowBytes / 25;
  return rounds * (k / kBK * std::max(mfma, load) * 10 / 21 + 2000);
}

Tile choose_tile(int64_t m, int64_t n, int64_t k, bool f32) {
  Tile best = kTiles[4];
  for (const Tile& t : kTiles)
    if (!(f32 && t.nf > 5) && tile_ns(t, m, n, k) < tile_ns(best, m, n, k)) best = t;
  return best;
}

constexpr int64_t kMaxChunkBytes = int64_t(256) << 20;

// Weight rows dequantized at a time: all of them up to 256 MiB of bf16 (256 rows
// at least, which dense_fits() holds below that).
int64_t chunk_rows(int64_t n_rows, int64_t k) {
  const int64_t cap = std::max<int64_t>(kMaxChunkBytes / (2 * k) / 256 * 256, 256);
  if (n_rows <= cap) return n_rows;
  return ceil_div(ceil_div(n_rows, ceil_div(n_rows, cap)), 256) * 256;
}

// Steps between flushes of an F32 product: chains of at most k / 128 MFMAs, the
// length of the fused GEMM's four k quarters, and of at most 32. Root mean square
// error against float64, this form over the fused one, Q4_0, 2048 x 2048 outputs,
// at k = 256, 512, 1024, 2048, 4096 and 14336: 1.00, 1.00, 1.00, 1.00, 1.00 and
// 0.53 (flushed every 16 steps whatever k: 1.42, 1.68, 1.93, 1.41, 1.00, 0.53; one
// chain: 1.42, 1.68, 1.93, 2.09, 2.16, 2.15). Four flushes cost up to 1 % of the
// product's time at k = 1024, eight 2.5 %. The chain of a bf16 result is lost in
// its rounding: error 1.655e-3 of the outputs in both forms at k = 14336, equal to
// 1e-7 of itself, and outputs that are not the nearest bf16 5.0e-4 of all against
// 4.0e-4.
uint32_t flush_steps(int64_t k) {
  return static_cast<uint32_t>(std::max<int64_t>(1, std::min<int64_t>(16, k / (4 * kBK))));
}

template <int MF, int NF, bool F32_OUT>
int launch(const uint16_t* x, int64_t ldx, int64_t m, const uint16_t* wb, int64_t n, int64_t k, void* y, int64_t ldy,
           hipStream_t s) {
  const void* fn = reinterpret_cast<const void*>(&dense_kernel<MF, NF, F32_OUT>);
  constexpr int lds = Stages<MF, NF>::kBytes;
  const int rc = allow_dynamic_lds(fn, lds);
  if (rc != SPIRAL_OK) return rc;
  const int64_t tm = ceil_div(m, 64 * MF), tn = ceil_div(n, 32 * NF);
  hipLaunchKernelGGL((dense_kernel<MF, NF, F32_OUT>), dim3(static_cast<unsigned>(tm * tn)), dim3(kThreads), lds, s, x,
                     static_cast<uint32_t>(ldx), static_cast<uint32_t>(m), wb, static_cast<uint32_t>(n),
                     static_cast<uint32_t>(k), y, ldy, static_cast<uint32_t>(tm), static_cast<uint32_t>(tn),
                     flush_steps(k));
  return launch_status();
}

int launch_bf16(Tile t, const uint16_t* x, int64_t ldx, int64_t m, const uint16_t* wb, int64_t n, int64_t k, void* y,
                int64_t ldy, hipStream_t s) {
  if (t.mf == 2) return launch<2, 4, false>(x, ldx, m, wb, n, k, y, ldy, s);
  switch (t.nf) {
    case 8: return launch<4, 8, false>(x, ldx, m, wb, n, k, y, ldy, s);
    case 7: return launch<4, 7, false>(x, ldx, m, wb, n, k, y, ldy, s);
    case 6: return launch<4, 6, false>(x, ldx, m, wb, n, k, y, ldy, s);
    case 5: return launch<4, 5, false>(x, ldx, m, wb, n, k, y, ldy, s);
    default: return launch<4, 4, false>(x, ldx, m, wb, n, k, y, ldy, s);
  }
}

int launch_f32(Tile t, const uint16_t* x, int64_t ldx, int64_t m, const uint16_t* wb, int64_t n, int64_t k, void* y,
               int64_t ldy, hipStream_t s) {
  if (t.mf == 2) return launch<2, 4, true>(x, ldx, m, wb, n, k, y, ldy, s);
  return t.nf == 5 ? launch<4, 5, true>(x, ldx, m, wb, n, k, y, ldy, s)
                   : launch<4, 4, true>(x, ldx, m, wb, n, k, y, ldy, s);
}

// Estimated nanoseconds of the fused GEMM (gemm.hip, one range of k): packing x,
// then rounds of one 128 x 64 tile a CU, whose time a k follows the format's
// dequantization; weights that the 256 MiB cache does not hold come from HBM again
// for every 128 rows.
int64_t fused_ns(int type, int64_t m, int64_t n, int64_t k, int64_t w_bytes, int64_t y_bytes) {
  const int64_t tm = ceil_div(m, 128), tiles = tm * ceil_div(n, 64), rounds = ceil_div(tiles, device_cu_count());
  const int64_t ps = type == SPIRAL_TYPE_Q4_0     ? 3590
                     : type == SPIRAL_TYPE_Q8_0   ? 3870
                     : type == SPIRAL_TYPE_IQ4_NL ? 4050
                     : type == SPIRAL_TYPE_IQ4_XS ? 4240
                     : type == SPIRAL_TYPE_Q4_K   ? 4400
                     : type == SPIRAL_TYPE_Q5_K   ? 4710
                                                  : 4790;
  return 3560 + 3310 * rounds + 2 * m * k / 4000 + y_bytes / 8450 + tiles * k / 270 + rounds * k * ps / 1000 +
         tm * std::max<int64_t>(0, w_bytes - 200000000) / 9000;
}

// Of this form: for each chunk of rows that gemm_dense() takes, its bytes
// written and read, and the product's rounds at the tile's measured step.
int64_t dense_ns(int64_t m, int64_t n, int64_t k, bool f32) {
  const int64_t chunk = chunk_rows(n, k);
  int64_t ns = 0;
  for (int64_t r = 0; r < n; r += chunk) {
    const int64_t nc = std::min(chunk, n - r);
    const Tile t = choose_tile(m, nc, k, f32);
    const int64_t rounds = ceil_div(ceil_div(m, 64 * t.mf) * ceil_div(nc, 32 * t.nf), device_cu_count());
    ns += 7000 + 2 * nc * k / 3500 + m * nc * (f32 ? 4 : 2) / 3200 + rounds * (k / kBK) * t.step_ns;
  }
  return ns;
}

}  // namespace

// Whether the dequantize-once form takes this product: 32-bit row offsets, and
// estimated to beat the fused GEMM by 4 %. Both estimates were fitted to 2660
// measured pairs (seven formats, 17 matrices from 1024 x 1024 to 12288 x 36864,
// 256 to 3072 rows, bf16 and F32); of those and 970 others it sends 44 to a form
// more than 3 % slower than the fused one (the worst by 12 %). Where they cross,
// us, fused and this form: Q4_0 4096 x 4096, 768 rows 46 and 51, 1536 rows 73 and
// 65; Q6_K the same 768 rows 54 and 51; Q4_K 6912 x 2560, 512 rows 37 and 45, 1024
// rows 70 and 54; Q4_K 16384 x 53248 (eight chunks), 1024 rows 2439 and 4057; Q4_K
// 49152 x 12288 (five), 512 rows 843 and 1103, 2048 rows 3266 and 2467. No matrix
// gained at 256 rows: two rows of fused tiles, one of these.
bool dense_fits(int type, int64_t n_rows, int64_t k, int64_t m, int64_t ldx, bool f32) {
  if (m <= 256 || n_rows < 256 || k % kBK != 0 || k > kMaxChunkBytes / 512 || m > (int64_t(1) << 24) ||
      n_rows > (int64_t(1) << 24) || ldx >= (int64_t(1) << 22))
    return false;
  // Shorter F32 rows: one chain of two or four MFMAs is less exact than the fused
  // form's quarters (error 1.12 and 1.03 times at k = 64 and 128).
  if (f32 && k < 192) return false;
  const int64_t wbytes = spiral_tensor_bytes(type, n_rows, k);
  if (wbytes == 0 || wbytes >= (int64_t(1) << 32)) return false;  // the fused GEMM's limit
  return dense_ns(m, n_rows, k, f32) * 104 < fused_ns(type, m, n_rows, k, wbytes, m * n_rows * (f32 ? 4 : 2)) * 100;
}

int64_t dense_workspace_bytes(int64_t n_rows, int64_t k) { return chunk_rows(n_rows, k) * k * 2; }

// Y = X W^T; arguments validated by the caller, dense_fits(), workspace of
// dense_workspace_bytes(n_rows, k) bytes, 16-byte aligned.
int gemm_dense(int type, const void* w, int64_t n_rows, int64_t k, const uint16_t* x, int64_t ldx, int64_t m, void* y,
               int y_type, int64_t ldy, void* workspace, hipStream_t s) {
  uint16_t* wb = static_cast<uint16_t*>(workspace);
  const int64_t chunk = chunk_rows(n_rows, k);
  for (int64_t r = 0; r < n_rows; r += chunk) {
    const int64_t nc = std::min(chunk, n_rows - r);
    int rc = dequant_rows(type, w, n_rows, k, r, nc, wb, k, s);
    if (rc != SPIRAL_OK) return rc;
    const bool f32 = y_type == SPIRAL_TYPE_F32;
    void* yc = static_cast<uint8_t*>(y) + r * (f32 ? 4 : 2);
    const Tile t = choose_tile(m, nc, k, f32);
    rc = f32 ? launch_f32(t, x, ldx, m, wb, nc, k, yc, ldy, s) : launch_bf16(t, x, ldx, m, wb, nc, k, yc, ldy, s);
    if (rc != SPIRAL_OK) return rc;
  }
  return SPIRAL_OK;
}

}  // namespace spiral
