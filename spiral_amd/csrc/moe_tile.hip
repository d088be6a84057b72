// MUL_MAT_ID for batches that route tens of tokens to an expert (prefill): one
// workgroup takes up to 80 of an expert's routed tokens against 96 of its weight
// rows over the whole k, so a weight is read and dequantized once for all of them.
//
// The streaming form (moe.hip) holds a pass's activations over the whole k in
// LDS, which caps a pass at 32 tokens at k = 2048 (the fused GLU form at 32 for
// any k): an expert's weights went by two or three times. Here the activations
// pass through LDS 128 k at a time.
//
// moe_tile_kernel: 4 waves, two workgroups a CU (at most 80 KiB of LDS each).
//  - Every load goes straight to LDS: the routed rows of x, 128 k a step, two
//    stages; 96 weight rows' codes (128 bytes a row: 256 k), their scale entries
//    and Q5_K's high bits, two stages. x chunks are stored permuted within their
//    256-byte row and code chunks within their 128-byte row, so that operand
//    reads spread over the banks.
//  - Wave s forms MFMA s of every 128-wide step (moe_piece.h) for all 96 rows:
//    each (row, token) sum is the streaming form's four chains added in its
//    order, so both forms give the same bits (moe_kernel, which takes small batches
//    past k = 4096, sums in another order). (The eight elements of a lane may
//    come in any order and the two operands may change places: both measured
//    bit-equal on gfx950; elements moved between lane groups are not.) Every code
//    and every x element is then read from LDS by one wave only.
//  - A lane takes eight weights of a row's 32-weight group, so scales are decoded
//    once per 256 k by the whole workgroup into (scale, offset) pairs in LDS.
//  - GLU: 48 gate rows and the same 48 up rows, activated where the chains meet.
//  - LDS is read through native vector types: behind a direct load the compiler
//    waits for every load in flight before a read through HIP's uint2 or float2.
//
// Measured, gate_up + SwiGLU and down, streaming form against this one, us: 128
// experts, 2048 / 768, top-8, 1000 tokens, Q4_K 332 and 216; 8 experts, 4096 /
// 7168, top-2, 400 tokens, Q4_K 1036 and 367; 60 experts, 3072 / 1536, top-4, 1020
// tokens, Q4_0 583 and 293. What bounds it: VALU 40 % and MFMA 17 % of a SIMD's
// time, the rest latency that two workgroups a CU do not cover (about 4 us a
// workgroup outside its k loop). One workgroup of 8 waves with half the x loads
// and three x stages was slower (157 against 150 us for gate_up), a second stage
// of decoded scales in place of the barrier behind them made no difference.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "dequant_impl.h"
#include "glu.h"

namespace spiral {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

constexpr int kThreads = 256, kGroups = 6, kRows = 16 * kGroups, kTokens = 80;
constexpr uint32_t kNone = 0x80000000u;  // past every buffer: fetches nothing

template <int TYPE>
constexpr bool kHighBits = TYPE == SPIRAL_TYPE_Q5_K;
template <int TYPE>
constexpr bool kSplitX = TYPE == SPIRAL_TYPE_Q4_0 || is_iq4(TYPE);
// Bytes of a row's scale entry for 256 k.
template <int TYPE>
constexpr int kEntry = TYPE == SPIRAL_TYPE_IQ4_XS ? 8 : 16;

// LDS: x stages, code stages, scale-entry stages, [high-bit stages], decoded scales.
constexpr int kXStage = kTokens * 256, kQStage = kRows * 128, kMStage = kRows * 16, kHStage = kRows * 32;
template <int TYPE>
struct Lds {
  static constexpr int kX = 0, kQ = 2 * kXStage, kM = kQ + 2 * kQStage, kH = kM + 2 * kMStage;
  static constexpr int kS = kH + (kHighBits<TYPE> ? 2 * kHStage : 0), kPairs = kS + kRows * 64;
  static constexpr int kBytes = kPairs + kTokens * 4;
};
static_assert(Lds<SPIRAL_TYPE_Q5_K>::kBytes <= 80 * 1024, "two workgroups a CU");

// (scale, offset) of 32-weight group j of a row from its entry: Q4_0 and IQ4_NL
// eight fp16 d, the K-quants d, dmin and the packed scales, IQ4_XS d and its own.
template <int TYPE>
__device__ __forceinline__ f32x2_t decode_scale(const uint8_t* entry, int j) {
  if constexpr (is_kquant(TYPE)) {
    const u32x4_t m = *reinterpret_cast<const u32x4_t*>(entry);
    const uint32_t sm = kq_chunk_scales(m.y, m.z, m.w, static_cast<uint32_t>(j) >> 1) >> (16 * (j & 1));
    return f32x2_t{fp16_ieee(m.x & 0xffffu) * 16777216.0f * static_cast<float>(sm & 0xffu),
                       -(fp16_ieee(m.x >> 16) * static_cast<float>((sm >> 8) & 0xffu))};
  } else if constexpr (TYPE == SPIRAL_TYPE_IQ4_XS) {
    const u32x2_t m = *reinterpret_cast<const u32x2_t*>(entry);
    const float sc = iq4xs_scale(make_uint2(m.x, m.y), j);
    return f32x2_t{sc, -1152.0f * sc};
  } else {
    const uint32_t d = reinterpret_cast<const uint16_t*>(entry)[j];
    const float m = TYPE == SPIRAL_TYPE_Q4_0 ? fp16_scale(d) : fp16_ieee(d);
    return f32x2_t{m, (TYPE == SPIRAL_TYPE_Q4_0 ? -1032.0f : -1152.0f) * m};
  }
}

// Four codes (a byte each) under the fp16 high byte of `magic`, times scale plus
// offset: four bf16 weights, each rounded once.
__device__ __forceinline__ uint2 weights4(uint32_t codes, uint32_t magic, float scale, float off) {
  const f16x2_t a = __builtin_bit_cast(f16x2_t, __builtin_amdgcn_perm(magic, codes, 0x04010400u));
  const f16x2_t b = __builtin_bit_cast(f16x2_t, __builtin_amdgcn_perm(magic, codes, 0x04030402u));
  return make_uint2(pack_bf16x2(__builtin_fmaf(static_cast<float>(a.x), scale, off),
                                __builtin_fmaf(static_cast<float>(a.y), scale, off)),
                    pack_bf16x2(__builtin_fmaf(static_cast<float>(b.x), scale, off),
                                __builtin_fmaf(static_cast<float>(b.y), scale, off)));
}

template <int TYPE, bool F32_OUT, bool GLU>
__global__ void __launch_bounds__(kThreads, 2)
    moe_tile_kernel(const uint8_t* __restrict__ w, const uint8_t* __restrict__ w_up, int64_t expert_stride,
                    uint32_t mat_rows, uint32_t feat, uint32_t k, const uint16_t* __restrict__ x, uint32_t x_bytes,
                    uint32_t x_slots, uint32_t top_k, const int32_t* __restrict__ offsets,
                    const int32_t* __restrict__ list, void* __restrict__ y, int glu_op, int swapped) {
  using L = Lds<TYPE>;
  constexpr int kFeat = GLU ? kRows / 2 : kRows;  // output columns of a workgroup
  extern __shared__ __align__(1024) uint8_t smem[];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, r = lane & 15u, g = lane >> 4;
  const uint32_t s = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave: MFMA s of a step
  const uint32_t e = blockIdx.y, f0 = blockIdx.x * kFeat;
  const int32_t begin = offsets[e], count = offsets[e + 1] - begin;
  const uint32_t nsb = k / 256, steps = 2 * nsb;
  int32_t* s_pair = reinterpret_cast<int32_t*>(smem + L::kPairs);

  // Planes of this expert: codes, scale entries, high bits. Lower half of the
  // workgroup's rows (d < kRows / 2) from `lo`, upper half from `hi` (GLU: up rows).
  const uint32_t codes = mat_rows * nsb * 128, hbytes = kHighBits<TYPE> ? mat_rows * nsb * 32 : 0;
  struct Matrix {
    __amdgpu_buffer_rsrc_t q, m, h;
  };
  const auto matrix = [&](const uint8_t* base) {
    const uint8_t* p = base + e * expert_stride;
    Matrix M;
    M.q = buffer_rsrc(p, codes);
    M.h = kHighBits<TYPE> ? buffer_rsrc(p + codes, hbytes) : M.q;
    M.m = buffer_rsrc(p + codes + hbytes, mat_rows * nsb * kEntry<TYPE>);
    return M;
  };
  const bool split = GLU && w_up != nullptr;
  const Matrix lo = matrix(w), hi = split ? matrix(w_up) : lo;
  // Matrix row of local row lr; rows past the end repeat the last one.
  const auto row_of = [&](uint32_t lr) -> uint32_t {
    if (!GLU) return min(f0 + lr, mat_rows - 1);
    const uint32_t f = min(f0 + (lr < kRows / 2 ? lr : lr - kRows / 2), feat - 1);
    return lr < kRows / 2 || split ? f : f + feat;
  };
  // The lane's load offsets: codes, 8 rows an instruction (three a wave: local
  // rows 24 s .. + 23); entries and high bits, the same 24 rows in one each.
  uint32_t qoff[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const uint32_t lr = 24 * s + 8 * i + (lane >> 3);
    qoff[i] = row_of(lr) * (nsb * 128) + (((lane & 7u) ^ ((lr >> 1) & 7u)) * 16);
  }
  // (IQ4_XS's 8-byte entries go a dword a lane)
  constexpr uint32_t kMLane = kEntry<TYPE> == 8 ? 2 : 1;
  const uint32_t moff = row_of(24 * s + min(lane / kMLane, 23u)) * (nsb * kEntry<TYPE>) + (lane % kMLane) * 4;
  const uint32_t hoff = kHighBits<TYPE> ? row_of(24 * s + min(lane >> 1, 23u)) * (nsb * 32) + (lane & 1u) * 16 : 0;
  const auto load_w = [&](uint32_t sb) {
    const uint32_t st = sb & 1u;
    const Matrix& M = s < 2 ? lo : hi;
#pragma unroll
    for (int i = 0; i < 3; ++i) dma16(M.q, smem + L::kQ + st * kQStage + (24 * s + 8 * i) * 128, qoff[i], sb * 128);
    uint8_t* entries = smem + L::kM + st * kMStage + 24 * s * kEntry<TYPE>;
    if constexpr (kEntry<TYPE> == 8) {
      if (lane < 48) dma4(M.m, entries, moff, sb * 8);
    } else {
      if (lane < 24) dma16(M.m, entries, moff, sb * 16);
    }
    if constexpr (kHighBits<TYPE>) {
      if (lane < 48) dma16(M.h, smem + L::kH + st * kHStage + 24 * s * 32, hoff, sb * 32);
    }
  };
  constexpr int kWLoads = kHighBits<TYPE> ? 5 : 4;
  const __amdgpu_buffer_rsrc_t X = buffer_rsrc(x, x_bytes);

  // Operand reads. x: chunk(s) of the lane group's eight elements; codes: chunk
  // 4 h + g of the row's 128 bytes.
  const uint32_t cx = kSplitX<TYPE> ? 4 * g + (s >> 1) : 8 * (g >> 1) + 2 * (g & 1u) + (s & 1u) + 4 * (s >> 1);
  const uint32_t xr0 = r * 256 + ((cx ^ r) * 16) + (kSplitX<TYPE> ? (s & 1u) * 8 : 0);
  const uint32_t xr1 = r * 256 + (((cx + 2) ^ r) * 16) + (s & 1u) * 8;  // kSplitX: elements 16 further on
  const uint32_t qr = r * 128 + ((g ^ ((r >> 1) & 7u)) * 16) + (kSplitX<TYPE> ? s * 4 : (s & 1u) * 8);
  const uint32_t hr = r * 32 + (g & 1u) * 16 + (s & 1u) * 8;

  // The expert's tokens in equal tiles of at most kTokens.
  const int32_t tiles = (count + kTokens - 1) / kTokens;
  const int32_t per = tiles > 0 ? (count + tiles - 1) / tiles : 0;

  const auto tile = [&](auto frags, int32_t t0, int32_t nt) {
    constexpr int NF = decltype(frags)::value;
    uint32_t xoff[NF];
#pragma unroll
    for (int i = 0; i < NF; ++i) {
      const uint32_t t = 4 * (s + 4 * i) + (lane >> 4);  // token of the tile
      const uint32_t p = static_cast<uint32_t>(s_pair[t]);
      const uint32_t tok = p / top_k, slot = p - tok * top_k;
      const uint32_t row = tok * x_slots + (x_slots == 1 ? 0u : slot);
      xoff[i] = static_cast<int32_t>(t) < nt ? row * k * 2 + (((lane & 15u) ^ (t & 15u)) * 16) : kNone;
    }
    const auto load_x = [&](uint32_t st) {
#pragma unroll
      for (int i = 0; i < NF; ++i) dma16(X, smem + L::kX + (st & 1u) * kXStage + (s + 4 * i) * 1024, xoff[i], st * 256);
    };
    f32x4_t acc[kGroups][NF];
#pragma unroll
    for (int q = 0; q < kGroups; ++q)
#pragma unroll
      for (int i = 0; i < NF; ++i) acc[q][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    load_w(0);
    load_x(0);
#pragma unroll 1
    for (uint32_t st = 0; st < steps; ++st) {
      const uint32_t sb = st >> 1, h = st & 1u;
      // x of this step, and at h = 0 the weights of this super-block, have
      // landed; at h = 1 the next super-block's (requested last) may be in flight.
      if (h != 0 && sb + 1 < nsb)
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kWLoads) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (st + 1 < steps) load_x(st + 1);
      __builtin_amdgcn_sched_barrier(0);  // the wait above counts on this order
      if (h == 0) {
        if (sb + 1 < nsb) load_w(sb + 1);
        // Decoded scales: entry j of row lr at lr * 64 + (j ^ 2 (lr / 4 % 4)) * 8.
#pragma unroll
        for (int i = 0; i < kRows * 8 / kThreads; ++i) {
          const uint32_t n = tid + kThreads * i, lr = n >> 3, j = n & 7u;
          *reinterpret_cast<f32x2_t*>(smem + L::kS + lr * 64 + ((j ^ (2 * ((lr >> 2) & 3u))) * 8)) =
              decode_scale<TYPE>(smem + L::kM + (sb & 1u) * kMStage + lr * kEntry<TYPE>, static_cast<int>(j));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
      }
      const uint8_t* xs = smem + L::kX + (st & 1u) * kXStage;
      bf16x8_t xf[NF];
#pragma unroll
      for (int i = 0; i < NF; ++i) {
        if constexpr (kSplitX<TYPE>) {
          const u32x2_t a = *reinterpret_cast<const u32x2_t*>(xs + xr0 + i * 4096);
          const u32x2_t b = *reinterpret_cast<const u32x2_t*>(xs + xr1 + i * 4096);
          xf[i] = __builtin_bit_cast(bf16x8_t, make_uint4(a.x, a.y, b.x, b.y));
        } else {
          xf[i] = *reinterpret_cast<const bf16x8_t*>(xs + xr0 + i * 4096);
        }
      }
      const uint8_t* qs = smem + L::kQ + (sb & 1u) * kQStage + (qr ^ (h * 64));
      // scale entry of the lane's group: 4 h + g, K-quants 4 h + 2 (g / 2) + s / 2
      const uint32_t j = is_kquant(TYPE) ? 4 * h + (g & 2u) + (s >> 1) : 4 * h + g;
      const uint8_t* ss = smem + L::kS + r * 64 + ((j ^ (2 * ((r >> 2) & 3u))) * 8);
#pragma unroll
      for (int q = 0; q < kGroups; ++q) {
        const f32x2_t sc = *reinterpret_cast<const f32x2_t*>(ss + q * 1024);
        uint2 o0, o1;
        if constexpr (is_kquant(TYPE)) {
          const u32x2_t c = *reinterpret_cast<const u32x2_t*>(qs + q * 2048);
          const uint32_t sh = (s >> 1) * 4;
          uint32_t c0 = (c.x >> sh) & 0x0F0F0F0Fu, c1 = (c.y >> sh) & 0x0F0F0F0Fu;
          if constexpr (kHighBits<TYPE>) {
            const u32x2_t b = *reinterpret_cast<const u32x2_t*>(smem + L::kH + (sb & 1u) * kHStage + hr + q * 512);
            c0 |= ((b.x >> j) & 0x01010101u) << 4;
            c1 |= ((b.y >> j) & 0x01010101u) << 4;
          }
          o0 = weights4(c0, 0u, sc.x, sc.y);
          o1 = weights4(c1, 0u, sc.x, sc.y);
        } else {
          const uint32_t c = *reinterpret_cast<const uint32_t*>(qs + q * 2048);
          if constexpr (TYPE == SPIRAL_TYPE_Q4_0) {
            o0 = weights4(c & 0x0F0F0F0Fu, 0x64646464u, sc.x, sc.y);
            o1 = weights4(c & 0xF0F0F0F0u, 0x54545454u, sc.x, -72.0f * sc.x);  // 16 c: the fp16 64 + c
          } else {
            o0 = weights4(iq4_lut(c & 0x0F0F0F0Fu), 0x64646464u, sc.x, sc.y);
            o1 = weights4(iq4_lut((c >> 4) & 0x0F0F0F0Fu), 0x64646464u, sc.x, sc.y);
          }
        }
        const bf16x8_t wf = __builtin_bit_cast(bf16x8_t, make_uint4(o0.x, o0.y, o1.x, o1.y));
#pragma unroll
        for (int i = 0; i < NF; ++i) acc[q][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xf[i], acc[q][i], 0, 0, 0);
      }
    }

    // The chains meet in LDS, two row groups at a time (GLU: a gate group and
    // its up group), NF KiB a wave and group, and each sum goes to one wave:
    // lane l holds column 4 (l / 16) + i of token l % 16.
    const auto sum4 = [&](int slot, int i) {
      const f32x4_t* p = reinterpret_cast<const f32x4_t*>(smem) + (slot * NF + i) * 64 + lane;
      constexpr int kWave = 2 * NF * 64;
      return (p[0] + p[kWave]) + (p[2 * kWave] + p[3 * kWave]);
    };
    const auto store = [&](uint32_t col, int i, f32x4_t v) {
      const int32_t t = 16 * i + static_cast<int32_t>(r);
      const uint32_t n = f0 + col + 4 * g;
      if (t >= nt || n >= feat) return;
      const int64_t at = static_cast<int64_t>(s_pair[t]) * feat + n;
      if constexpr (F32_OUT) {
        float* dst = static_cast<float*>(y) + at;
        if (n + 4 <= feat && (reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
          *reinterpret_cast<f32x4_t*>(dst) = v;
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (n + c < feat) dst[c] = v[c];
        }
      } else {
        uint16_t* dst = static_cast<uint16_t*>(y) + at;
        const uint32_t b[2] = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        if (n + 4 <= feat && (reinterpret_cast<uintptr_t>(dst) & 7u) == 0) {
          *reinterpret_cast<uint2*>(dst) = make_uint2(b[0], b[1]);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (n + c < feat) dst[c] = static_cast<uint16_t>(b[c / 2] >> (16 * (c & 1)));
        }
      }
    };
#pragma unroll
    for (int p = 0; p < kGroups / 2; ++p) {
      __syncthreads();
      f32x4_t* mine = reinterpret_cast<f32x4_t*>(smem) + s * (2 * NF * 64) + lane;
#pragma unroll
      for (int i = 0; i < NF; ++i) {
        mine[i * 64] = acc[GLU ? p : 2 * p][i];
        mine[(NF + i) * 64] = acc[GLU ? kGroups / 2 + p : 2 * p + 1][i];
      }
      __syncthreads();
      if constexpr (GLU) {
        for (int i = s; i < NF; i += 4) {
          const f32x4_t a = sum4(0, i), b = sum4(1, i);
          f32x4_t v;
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] = swapped ? glu_act(glu_op, b[c]) * a[c] : glu_act(glu_op, a[c]) * b[c];
          store(16 * p, i, v);
        }
      } else {
        for (int i = s; i < 2 * NF; i += 4) store(32 * p + (i < NF ? 0 : 16), i < NF ? i : i - NF, sum4(0, i));
      }
    }
    __syncthreads();  // before the next tile's loads and token list
  };

  for (int32_t z = blockIdx.z; z < tiles; z += gridDim.z) {
    const int32_t t0 = z * per, nt = min(per, count - t0);
    if (nt <= 0) break;
    if (tid < kTokens) s_pair[tid] = list[begin + t0 + min(static_cast<int32_t>(tid), nt - 1)];
    __syncthreads();
    if (nt <= 32)
      tile(std::integral_constant<int, 2>(), t0, nt);
    else if (nt <= 64)
      tile(std::integral_constant<int, 4>(), t0, nt);
    else
      tile(std::integral_constant<int, 5>(), t0, nt);
  }
}

template <int TYPE, bool F32_OUT, bool GLU>
int launch_tile(const void* w, const void* w_up, int64_t expert_stride, int64_t n_expert, int64_t n_rows, int64_t k,
                const uint16_t* x, int64_t x_slots, int64_t n_pairs, int64_t top_k, const int32_t* offsets,
                const int32_t* list, void* y, int glu_op, int swapped, hipStream_t s) {
  const auto kern = moe_tile_kernel<TYPE, F32_OUT, GLU>;
  constexpr int lds = Lds<TYPE>::kBytes;
  const int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds);
  if (rc != SPIRAL_OK) return rc;
  const int64_t feat = GLU ? n_rows / 2 : n_rows, rows = GLU && w_up != nullptr ? feat : n_rows;
  const int64_t lanes = std::min<int64_t>(64, ceil_div(n_pairs, n_expert * kTokens));
  const dim3 grid(static_cast<unsigned>(ceil_div(feat, GLU ? kRows / 2 : kRows)), static_cast<unsigned>(n_expert),
                  static_cast<unsigned>(lanes));
  hipLaunchKernelGGL(kern, grid, dim3(kThreads), lds, s, static_cast<const uint8_t*>(w),
                     static_cast<const uint8_t*>(w_up), expert_stride, static_cast<uint32_t>(rows),
                     static_cast<uint32_t>(feat), static_cast<uint32_t>(k), x,
                     static_cast<uint32_t>(n_pairs / top_k * x_slots * k * 2), static_cast<uint32_t>(x_slots),
                     static_cast<uint32_t>(top_k), offsets, list, y, glu_op, swapped);
  return launch_status();
}

}  // namespace

// Whether the tiled form takes this MUL_MAT_ID: formats of 4-bit codes (and Q5_K),
// 32-bit offsets, and enough tokens an expert. Below that the streaming form reads
// its weights ahead better: gate_up and down of 128 experts, 2048 / 768, us,
// streaming against this form at 17, 20 and 24 tokens an expert (its passes take
// 32): Q4_K 142 and 166, 145 and 167, 237 and 176; Q4_0 123 and 160, 162 and 164,
// 199 and 173; IQ4_XS 159 and 189, 210 and 185, 267 and 194. The two products apart
// at 20 and 24: Q5_K 172 and 114, 173 and 116 (gate_up), 43 and 65, 71 and 67
// (down); IQ4_NL 95 and 101, 167 and 106, 42 and 59, 69 and 63. Past k = 2304 the
// streaming form's passes stay at 16: 60 experts, 3072 / 1536, 13 tokens: Q4_K 310
// and 221, Q4_0 246 and 203, IQ4_XS 264 and 239; one product at 13: Q5_K 60 experts
// of 2048 x 2560 128 and 91, 16 of 4096 x 4096 102 and 79, 8 of 4096 x 14336 177
// and 152, IQ4_NL 87 and 82, 82 and 71, 167 and 138; at 10 Q4_K 1.57 times the
// streaming form's time in 16 of 4096 x 4096.
//
// short_rows: a product without GLU whose rows leave LDS for the streaming form's
// passes of 64 tokens. It stays with that form while the average expert fills at
// most 0.7 of its passes, so that evenly routed experts take one pass each, side
// by side (for several passes, while there are row groups enough for the chip):
// 128 experts of 2048 x 768, us, streaming and this form at 36, 40, 48, 56, 80 and
// 128 tokens an expert, Q4_K 51 and 70, 52 and 72, 80 and 73, 82 and 78, 95 and 112,
// 139 and 152; Q4_0 50 and 71, 51 and 73, 74 and 74, 74 and 78, 93 and 117, 130 and
// 154. An expert of several times the average takes its passes one after another
// there: with popularities spread over e^0.25 (the busiest of 128 at twice the
// average) the two forms meet, over e^0.5 this one leads (40 tokens: 92 and 73).
bool moe_tile_fits(int type, int64_t n_expert, int64_t n_rows, int64_t k, int64_t x_slots, int64_t n_pairs,
                   int64_t top_k, bool short_rows) {
  if (type != SPIRAL_TYPE_Q4_0 && !is_iq4(type) && !is_kquant(type)) return false;
  if (k % 256 != 0 || n_expert > 65535 || n_pairs / top_k * x_slots * k * 2 >= (int64_t(1) << 31)) return false;
  if (n_pairs < (k > 2304 ? 13 : 24) * n_expert) return false;
  const int64_t avg = ceil_div(n_pairs, n_expert), passes = ceil_div(avg, 64);
  return !(short_rows && avg > 32 && 10 * avg <= 7 * 64 * passes && (passes == 1 || n_expert * n_rows >= 120000));
}

// Arguments validated by the caller (moe); offsets and list from the route kernel.
int moe_tile(int type, const void* w, const void* w_up, int64_t expert_stride, int64_t n_expert, int64_t n_rows,
             int64_t k, const uint16_t* x, int64_t x_slots, int64_t n_pairs, int64_t top_k, const int32_t* offsets,
             const int32_t* list, void* y, bool f32, int glu_op, int swapped, hipStream_t s) {
#define SPIRAL_TILE_AS(T, F, G)                                                                                    \
  launch_tile<T, F, G>(w, w_up, expert_stride, n_expert, n_rows, k, x, x_slots, n_pairs, top_k, offsets, list, y, \
                       glu_op, swapped, s)
#define SPIRAL_TILE(T)                                                                 \
  case T:                                                                              \
    if (glu_op >= 0) return f32 ? SPIRAL_TILE_AS(T, true, true) : SPIRAL_TILE_AS(T, false, true); \
    return f32 ? SPIRAL_TILE_AS(T, true, false) : SPIRAL_TILE_AS(T, false, false)
  switch (type) {
    SPIRAL_TILE(SPIRAL_TYPE_Q4_0);
    SPIRAL_TILE(SPIRAL_TYPE_Q4_K);
    SPIRAL_TILE(SPIRAL_TYPE_Q5_K);
    SPIRAL_TILE(SPIRAL_TYPE_IQ4_NL);
    SPIRAL_TILE(SPIRAL_TYPE_IQ4_XS);
    default: return SPIRAL_ERR_TYPE;
  }
#undef SPIRAL_TILE
#undef SPIRAL_TILE_AS
}

}  // namespace spiral
