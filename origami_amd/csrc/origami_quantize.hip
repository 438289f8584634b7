// origami_quantize.hip -- MI355X (gfx950) kernels for the quantized saves: one layer's
// K/V read once and its CacheGen or KIVI payload written once (the quantizers of the
// reference's cachegen_adapter.py:246-340 and kivi_adapter.py:229-450, which are chains
// of float32 tensor operations).
//
// Arithmetic is that of the tensor expressions, operation by operation in binary32
// without contraction, so payloads are the same bytes: a scalar divided by a tensor is
// the tensor's reciprocal times the scalar, a tensor divided by a scalar is the tensor
// times the scalar's reciprocal, and a minimum or maximum with a NaN is that NaN (whose
// symbols are 0).  One value may have other bytes: the zero point of a KIVI group whose
// least values are zeros of both signs is -0 here, and there the zero that the reduction's
// order leaves; both decode to the same values.  The K/V tensor may have any of the layouts
// the adapters accept: head_dim is its fastest axis, everything else is a stride
// (KvStrides).
//
// HBM bounds CacheGen, its own arithmetic KIVI; 4 bytes are read and b / 4 bytes written
// per (K, V) pair of 16-bit values.  16384 tokens of 8 heads x 128, bf16, with the copy of
// the payload into its stored chunks: CacheGen 573 -> 26.7 us, KIVI (2 bits) 1025 -> 30.0 us.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <type_traits>

#include "origami_internal.h"
#include "origami_layout.h"

using namespace origami_internal;

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4u __attribute__((ext_vector_type(4), aligned(1)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int kQThreads = 256;
constexpr int kQWaves = kQThreads / 64;

// Element strides of a K/V tensor: element (half, token t, head h, dim d) is at
// half * half + (t / block_tokens) * block + (t % block_tokens) * token + h * head + d.
struct KvStrides {
  int64_t half, block, token, head;
  uint32_t block_tokens;
};

__device__ __forceinline__ int64_t token_offset(const KvStrides& s, uint32_t t) {
  const uint32_t blk = t / s.block_tokens;
  return static_cast<int64_t>(blk) * s.block +
         static_cast<int64_t>(t - blk * s.block_tokens) * s.token;
}

// Eight consecutive elements as binary32: 16 bytes of a 16-bit type, 32 of float32.
template <int DT>
struct Eight {
  static constexpr int kWords = DT == ORIGAMI_DTYPE_FLOAT32 ? 8 : 4;
  uint32_t w[kWords];

  __device__ __forceinline__ void load(const void* base, int64_t element) {
    const u32x4* src = reinterpret_cast<const u32x4*>(
        static_cast<const uint8_t*>(base) + element * (kWords / 2));
#pragma unroll
    for (int i = 0; i < kWords / 4; ++i) {
      const u32x4 x = __builtin_nontemporal_load(src + i);
      w[4 * i] = x.x;
      w[4 * i + 1] = x.y;
      w[4 * i + 2] = x.z;
      w[4 * i + 3] = x.w;
    }
  }
  __device__ __forceinline__ float get(int i) const {
    if constexpr (DT == ORIGAMI_DTYPE_FLOAT32) {
      return __builtin_bit_cast(float, w[i]);
    } else if constexpr (DT == ORIGAMI_DTYPE_BFLOAT16) {
      return __builtin_bit_cast(float, i & 1 ? w[i >> 1] & 0xffff0000u : w[i >> 1] << 16);
    } else {
      return static_cast<float>(
          __builtin_bit_cast(_Float16, static_cast<uint16_t>(w[i >> 1] >> (16 * (i & 1)))));
    }
  }
};

__device__ __forceinline__ uint16_t half_bits(float v) {
  asm("" : "+v"(v));  // an already rounded binary32 value (no fused convert)
  return __builtin_bit_cast(uint16_t, static_cast<_Float16>(v));
}

// ---------------------------------------------------------------------------
// CacheGen
// ---------------------------------------------------------------------------

struct CacheGenQuantParams {
  const void* kv;
  KvStrides s;
  uint32_t tokens;
  int32_t row_lanes;   // lanes of a token row: a power of two, at most 64
  int32_t groups;      // 8-channel groups of a row
  int32_t head_groups; // groups of a head
  int32_t bits[2];
  float center[2];
  uint8_t* stream[2];
  uint16_t* peak[2];
  uint8_t* pad;        // a byte between the streams and the maxima, or null
};

// A wave holds whole token rows, row_lanes lanes each with NV 8-channel groups, so the
// row maximum is a butterfly inside the wave and each value is read once.  A lane
// packs its 8 symbols into b bytes; the tile's rows are one stretch of the stream, put
// together in LDS so that the stream is written in whole 16-byte chunks.  R row steps
// are loaded before the first is reduced.
template <int DT, int NV, int R>
__global__ __launch_bounds__(kQThreads) void cachegen_quantize_kernel(CacheGenQuantParams p) {
  extern __shared__ __align__(16) uint8_t stage[];
  const int half = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int RL = p.row_lanes, step_rows = 64 / RL, sub = lane / RL, li = lane & (RL - 1);
  const uint32_t tile_rows = kQWaves * R * step_rows;
  const uint32_t t0 = blockIdx.x * tile_rows;
  const int bits = p.bits[half];
  const float center = p.center[half];

  // Every lane loads: one past the row's groups takes the last group again and one past
  // the last token that token, which changes no maximum, so no branch keeps the R * NV
  // loads from being in flight together (with branches the compiler moved them down to
  // their uses: the save of 16384 tokens took 30.8 us, 26.7 without).
  int64_t at[NV];  // this lane's groups in a row
  bool live[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    live[v] = li + v * RL < p.groups;
    const int g = live[v] ? li + v * RL : p.groups - 1;
    const int h = g / p.head_groups;
    at[v] = half * p.s.half + h * p.s.head + static_cast<int64_t>(g - h * p.head_groups) * 8;
  }
  Eight<DT> x[R][NV];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t t = t0 + (wave * R + r) * step_rows + sub;
    const int64_t row = token_offset(p.s, t < p.tokens ? t : p.tokens - 1);
#pragma unroll
    for (int v = 0; v < NV; ++v) x[r][v].load(p.kv, row + at[v]);
  }
  asm volatile("" ::: "memory");

  const uint32_t rows = p.tokens - t0 < tile_rows ? p.tokens - t0 : tile_rows;
  const int64_t row_bytes = static_cast<int64_t>(p.groups) * bits;
  uint8_t* const dst = p.stream[half] + t0 * row_bytes;
  const int mis = static_cast<int>(reinterpret_cast<uintptr_t>(dst) & 15);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const uint32_t local = (wave * R + r) * step_rows + sub;
    // |x| as an integer: ordered like the value, a NaN above infinity
    uint32_t top = 0;
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t a = __builtin_bit_cast(uint32_t, x[r][v].get(i)) & 0x7fffffffu;
        top = top > a ? top : a;
      }
    for (int m = 1; m < RL; m <<= 1) {
      const uint32_t o = __shfl_xor(top, m);
      top = top > o ? top : o;
    }
    const float least = 1e-6f;
    float peak = __builtin_bit_cast(float, top);
    if (peak < least) peak = least;
    const float scale = __fmul_rn(__fdiv_rn(1.0f, peak), center);
    if (local >= rows) continue;
    if (li == 0) p.peak[half][t0 + local] = half_bits(peak);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (!live[v]) continue;
      uint32_t q[2] = {0, 0};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        // |x| <= peak, so the rounded value lies in [0, 2 * center]; the maximum is for
        // NaNs, which become 0
        const float y = __builtin_rintf(__fadd_rn(__fmul_rn(x[r][v].get(i), scale), center));
        q[i >> 2] |= static_cast<uint32_t>(fmaxf(y, 0.0f)) << (bits * (i & 3));
      }
      const uint64_t packed = q[0] | (static_cast<uint64_t>(q[1]) << (4 * bits));
      uint8_t* o = stage + mis + local * row_bytes + (li + v * RL) * bits;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (i < bits) o[i] = static_cast<uint8_t>(packed >> (8 * i));
    }
  }
  __syncthreads();
  const int total = mis + static_cast<int>(rows * row_bytes);
  for (int c = threadIdx.x * 16; c < total; c += kQThreads * 16) {
    uint8_t* const o = dst - mis + c;
    if (c >= mis && c + 16 <= total) {
      *reinterpret_cast<u32x4*>(o) = *reinterpret_cast<const u32x4*>(stage + c);
    } else {  // the tile's ends: the rest of the chunk is another tile's
      for (int i = 0; i < 16; ++i)
        if (c + i >= mis && c + i < total) o[i] = stage[c + i];
    }
  }
  if (p.pad && blockIdx.x == 0 && half == 0 && threadIdx.x == 0) *p.pad = 0;
}

template <int DT, int NV, int R>
int launch_cachegen(const CacheGenQuantParams& p, hipStream_t stream) {
  const uint32_t tile_rows = kQWaves * R * (64 / p.row_lanes);
  const dim3 grid((p.tokens + tile_rows - 1) / tile_rows, 2);
  const size_t lds = static_cast<size_t>(tile_rows) * p.groups * 8 + 32;
  hipLaunchKernelGGL((cachegen_quantize_kernel<DT, NV, R>), grid, dim3(kQThreads), lds, stream, p);
  return check_launch("cachegen_quantize_kernel");
}

// Groups per lane by row length (at most 4096 channels), and several row steps in flight
// per wave in long launches.  us with 1 / 4 steps, bf16 not in a cache: 8 heads x 128, 4096
// tokens 7.4 / 9.0, 8192 12.0 / 12.8, 12288 16.7 / 16.9, 16384 20.6 / 20.0, 32768 36.8 /
// 33.6; 4 x 128, 6144 tokens 7.2 / 7.6, 8192 8.8 / 8.6, 16384 15.3 / 13.4; 2 x 64, 24576
// tokens 7.0 / 7.3, 32768 8.5 / 8.0.
template <int DT>
int launch_cachegen_rows(const CacheGenQuantParams& p, hipStream_t stream) {
  const int64_t steps = (static_cast<int64_t>(p.tokens) * p.row_lanes / 64) * 2 / kQWaves;
  if (p.groups <= 64)
    return steps >= 4096 ? launch_cachegen<DT, 1, 4>(p, stream)
                            : launch_cachegen<DT, 1, 1>(p, stream);
  if (p.groups <= 128)
    return steps >= 8192 ? launch_cachegen<DT, 2, 4>(p, stream)
                            : launch_cachegen<DT, 2, 1>(p, stream);
  if (p.groups <= 256) return launch_cachegen<DT, 4, 1>(p, stream);
  return launch_cachegen<DT, 8, 1>(p, stream);
}

// ---------------------------------------------------------------------------
// KIVI
// ---------------------------------------------------------------------------

struct KiviQuantParams {
  const void* kv;
  KvStrides s;
  uint32_t tokens, sink, body;
  int32_t H, D, C;
  int32_t group;        // 16, 32, 64 or 128
  int32_t vgroups;
  float inv_levels;
  uint8_t* stream[2];   // packed streams, or one byte per symbol (workspace)
  uint16_t* scale[2];
  uint16_t* zero[2];
  uint16_t* sink_rows[2];
  uint8_t* pad[8];      // bytes between parts that are written as 0 (null: none)
  int32_t tiles[2];     // workgroups of the keys, then the values, then the sink rows
  int32_t chan_tiles[2];
};

constexpr int kQTokens = 16;  // tokens of a lane

// The ranges are taken on pairs, two float16 values per register: the least and the
// greatest of three, NaN if one is a NaN (gfx950's IEEE 754-2019 minimum and maximum).
__device__ __forceinline__ uint32_t pk_min3(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_pk_minimum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ uint32_t pk_max3(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_pk_maximum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ float low_half(uint32_t v) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(v)));
}
__device__ __forceinline__ float high_half(uint32_t v) {
  return static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(v >> 16)));
}

// One quantization group: zero point (its minimum), scale and the scale's reciprocal.
struct Group {
  float zero, scale, inv;
};

// `range` holds the minimum (low) and the negated maximum (high).  A NaN keeps its sign and
// payload through both and through the subtraction, as in the tensor operations.
__device__ __forceinline__ Group make_group(uint32_t range, float inv_levels) {
  const float tiny = 1.17549435e-38f;  // the least normal binary32
  Group g;
  g.zero = low_half(range);
  const float s = __fmul_rn(__fsub_rn(high_half(range ^ 0x80000000u), g.zero), inv_levels);
  g.scale = s < tiny ? tiny : s;
  g.inv = __fdiv_rn(1.0f, g.scale);
  return g;
}

// round((x - zero) / scale) in [0, levels], with the correctly rounded quotient: the
// product with the correctly rounded reciprocal, corrected twice by its remainder
// (Markstein's division; nothing underflows here, as a scale is the least normal number
// where the group has one value, and at least 2^-32 elsewhere).  An infinite or NaN
// scale gives a NaN, whose symbol is 0 like that of the quotient.
// x is the low or high half of `pair`: one v_fma_mix converts it and takes off the zero
// point (x * 1 - zero, rounded once, as the subtraction).
template <bool HIGH>
__device__ __forceinline__ float kivi_symbol(uint32_t pair, const Group& g) {
  float d;
  if constexpr (HIGH)
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
        : "=v"(d) : "v"(pair), "v"(g.zero));
  else
    asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(d) : "v"(pair), "v"(g.zero));
  const float q0 = __fmul_rn(d, g.inv);
  const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, g.scale, d), g.inv, q0);
  const float q2 = __builtin_fmaf(__builtin_fmaf(-q1, g.scale, d), g.inv, q1);
  return __builtin_rintf(fmaxf(q2, 0.0f));
}

// Eight values as float16 at any even address.
__device__ __forceinline__ void store_halves(uint16_t* dst, const float (&v)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const f32x2 pair = {v[2 * k], v[2 * k + 1]};
    w[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, f16x2));
  }
  *reinterpret_cast<u32x4u*>(dst) = u32x4u{w[0], w[1], w[2], w[3]};
}

// A lane's run of one plane: 16 symbols of W bits, gathered as exact binary32 sums of
// 16 / W symbols each.
template <int W>
struct PlaneRun {
  static constexpr int kPer = 16 / W;         // symbols of a sum
  static constexpr int kSums = 16 / kPer;
  float sum[kSums];

  template <int J>
  __device__ __forceinline__ void put(float symbol) {
    constexpr float weight = static_cast<float>(1u << (W * (J % kPer)));
    if constexpr (J % kPer == 0)
      sum[J / kPer] = symbol;
    else
      sum[J / kPer] = __builtin_fmaf(symbol, weight, sum[J / kPer]);
  }
  __device__ __forceinline__ uint32_t word(int i) const {
    return static_cast<uint32_t>(sum[2 * i]) | (static_cast<uint32_t>(sum[2 * i + 1]) << 16);
  }
};

// Writes a run at symbol `symbol` of its stream.  BYTES: W = 8 at any address, `nv`
// symbols (the packer follows); else a whole run on an aligned word.
template <int W, bool BYTES>
__device__ __forceinline__ void store_run(uint8_t* stream, int64_t symbol, const PlaneRun<W>& r,
                                          int nv) {
  uint8_t* const o = stream + (symbol * W >> 3);
  if constexpr (BYTES) {
    const uint32_t w[4] = {r.word(0), r.word(1), r.word(2), r.word(3)};
    if (nv == kQTokens) {
      *reinterpret_cast<u32x4u*>(o) = u32x4u{w[0], w[1], w[2], w[3]};
    } else {
#pragma unroll
      for (int j = 0; j < kQTokens; ++j)
        if (j < nv) o[j] = static_cast<uint8_t>(w[j >> 2] >> (8 * (j & 3)));
    }
  } else if constexpr (W == 8) {
    *reinterpret_cast<u32x4*>(o) = u32x4{r.word(0), r.word(1), r.word(2), r.word(3)};
  } else if constexpr (W == 4) {
    *reinterpret_cast<u32x2*>(o) = u32x2{r.word(0), r.word(1)};
  } else {
    *reinterpret_cast<uint32_t*>(o) = r.word(0);
  }
}

// Calls f(std::integral_constant<int, i>) for i = 0 .. N - 1.
template <int N, typename F>
__device__ __forceinline__ void each(F&& f) {
  if constexpr (N > 0) {
    each<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

// A lane owns 8 channels x 16 tokens: it loads 16 row segments of 16 bytes, rounds them
// to float16 pairs, takes the group ranges, and holds each plane's run of 16 tokens,
// which it writes packed.  Key tiles (groups along tokens) are 8 lanes along channels x
// 8 along tokens per wave, value tiles (groups along channels) 16 x 4; a workgroup's
// waves go along tokens, so a plane's stretch of 2-bit symbols is a whole 128-byte line
// of keys (64 bytes of values) written by one workgroup.  Lanes past the last token or
// channel load the last one again, which changes no range of a group they share.
// With the loads in flight the arithmetic bounds it: ranges on pairs, a branch-free
// division and symbols gathered by fused multiply-adds took the save of 16384 tokens
// from 61.0 us (scalar ranges, a branch per quotient, shifts) to 33.3; ranges by the
// three-operand minimum and maximum, which carry NaNs, the subtraction of the zero point
// folded into the conversion and one address per lane to 30.1.  It runs three waves per
// SIMD at 164-172 registers (two at 8 bits of bfloat16); a cap at four waves spills 58-69 of
// them, one at five waves took 58 us.
template <int HALF, int DT, int W, bool BYTES>
__device__ __forceinline__ void kivi_quantize_tile(const KiviQuantParams& p, uint32_t tile) {
  constexpr int CL = HALF == 0 ? 8 : 16, TL = 64 / CL;  // lanes along channels, tokens
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t ct = tile % p.chan_tiles[HALF], tt = tile / p.chan_tiles[HALF];
  const int c0 = (ct * CL + (lane & (CL - 1))) * 8;
  const uint32_t bt0 = ((tt * kQWaves + wave) * TL + lane / CL) * kQTokens;
  const bool chan_ok = c0 < p.C;
  const int nv = !chan_ok || bt0 >= p.body
                     ? 0
                     : (p.body - bt0 < kQTokens ? static_cast<int>(p.body - bt0) : kQTokens);
  const int cl = chan_ok ? c0 : p.C - 8;
  const int h = cl / p.D, d0 = cl - h * p.D;
  const int64_t col = HALF * p.s.half + h * p.s.head + d0;

  uint32_t v[kQTokens][4];  // float16 pairs
  {
    const uint32_t last = p.tokens - 1;
    uint32_t t = p.sink + bt0 < last ? p.sink + bt0 : last;
    uint32_t blk = t / p.s.block_tokens, off = t - blk * p.s.block_tokens;
    Eight<DT> x[kQTokens];
    if (__all(t + kQTokens - 1 <= last && off + kQTokens <= p.s.block_tokens)) {
      // every lane's tokens are rows of one block: one address, a uniform step
      const int64_t row = static_cast<int64_t>(blk) * p.s.block +
                          static_cast<int64_t>(off) * p.s.token + col;
#pragma unroll
      for (int j = 0; j < kQTokens; ++j) x[j].load(p.kv, row + j * p.s.token);
    } else {
#pragma unroll
      for (int j = 0; j < kQTokens; ++j) {
        x[j].load(p.kv, static_cast<int64_t>(blk) * p.s.block +
                            static_cast<int64_t>(off) * p.s.token + col);
        if (t < last) {
          ++t;
          if (++off == p.s.block_tokens) {
            off = 0;
            ++blk;
          }
        }
      }
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < kQTokens; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if constexpr (DT == ORIGAMI_DTYPE_FLOAT16) {
          v[j][k] = x[j].w[k];
        } else {
          const f32x2 pair = {x[j].get(2 * k), x[j].get(2 * k + 1)};
          v[j][k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, f16x2));
        }
      }
  }

  PlaneRun<W> run[8];
  const uint32_t kNegHigh = 0x80000000u;
  if constexpr (HALF == 0) {
    const int lanes = p.group / kQTokens;  // token lanes of a group
    uint32_t range[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint32_t lo = v[0][k], hi = v[0][k];
#pragma unroll
      for (int j = 1; j < kQTokens; j += 2) {
        const uint32_t a = v[j][k], b = v[j + 1 < kQTokens ? j + 1 : j][k];
        lo = pk_min3(lo, a, b);
        hi = pk_max3(hi, a, b);
      }
      range[2 * k] = __builtin_amdgcn_perm(hi, lo, 0x05040100u) ^ kNegHigh;
      range[2 * k + 1] = __builtin_amdgcn_perm(hi, lo, 0x07060302u) ^ kNegHigh;
    }
    for (int m = 1; m < lanes; m <<= 1)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t o = __shfl_xor(range[i], m * CL);
        range[i] = pk_min3(range[i], o, o);
      }
    const int64_t meta = static_cast<int64_t>(bt0 / p.group) * p.C + c0;
    const bool lead = nv > 0 && bt0 % p.group == 0;
    float scales[8], zeros[8];
    each<8>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const Group g = make_group(range[i], p.inv_levels);
      scales[i] = g.scale;
      zeros[i] = g.zero;
      each<kQTokens>([&](auto jc) {
        constexpr int j = decltype(jc)::value;
        run[i].template put<j>(kivi_symbol<(i & 1) != 0>(v[j][i >> 1], g));
      });
    });
    if (lead) {
      store_halves(p.scale[0] + meta, scales);
      store_halves(p.zero[0] + meta, zeros);
    }
  } else {
    const int lanes = p.group / 8;  // channel lanes of a group
    uint32_t range[kQTokens];
#pragma unroll
    for (int j = 0; j < kQTokens; ++j) {
      const uint32_t lo = pk_min3(pk_min3(v[j][0], v[j][1], v[j][2]), v[j][3], v[j][3]);
      const uint32_t hi = pk_max3(pk_max3(v[j][0], v[j][1], v[j][2]), v[j][3], v[j][3]);
      const uint32_t a = __builtin_amdgcn_perm(hi, lo, 0x05040100u) ^ kNegHigh;
      const uint32_t b = __builtin_amdgcn_perm(hi, lo, 0x07060302u) ^ kNegHigh;
      range[j] = pk_min3(a, b, b);
    }
    for (int m = 1; m < lanes; m <<= 1)
#pragma unroll
      for (int j = 0; j < kQTokens; ++j) {
        const uint32_t o = __shfl_xor(range[j], m);
        range[j] = pk_min3(range[j], o, o);
      }
    const bool lead = chan_ok && c0 % p.group == 0;
    const int64_t meta = static_cast<int64_t>(bt0) * p.vgroups + c0 / p.group;
    each<kQTokens>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const Group g = make_group(range[j], p.inv_levels);
      if (lead && j < nv) {
        p.scale[1][meta + static_cast<int64_t>(j) * p.vgroups] = half_bits(g.scale);
        p.zero[1][meta + static_cast<int64_t>(j) * p.vgroups] = half_bits(g.zero);
      }
      each<8>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        run[i].template put<j>(kivi_symbol<(i & 1) != 0>(v[j][i >> 1], g));
      });
    });
  }
  if (nv == 0) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int64_t plane = HALF == 0 ? static_cast<int64_t>(d0 + i) * p.H + h : c0 + i;
    store_run<W, BYTES>(p.stream[HALF], plane * p.body + bt0, run[i], nv);
  }
}

template <int DT, int W, bool BYTES>
__global__ __launch_bounds__(kQThreads) void kivi_quantize_kernel(KiviQuantParams p) {
  uint32_t tile = blockIdx.x;
  if (tile < static_cast<uint32_t>(p.tiles[0])) {
    kivi_quantize_tile<0, DT, W, BYTES>(p, tile);
    return;
  }
  tile -= p.tiles[0];
  if (tile < static_cast<uint32_t>(p.tiles[1])) {
    kivi_quantize_tile<1, DT, W, BYTES>(p, tile);
    return;
  }
  // sink rows of both halves, 8 channels per thread, and the pad bytes
  tile -= p.tiles[1];
  if (tile == 0 && threadIdx.x < 8 && p.pad[threadIdx.x]) *p.pad[threadIdx.x] = 0;
  const uint32_t G = p.C / 8, n = p.sink * G;
  const uint32_t i = tile * kQThreads + threadIdx.x;
  if (i >= 2 * n) return;
  const int half = i >= n;
  const uint32_t k = i - half * n, t = k / G, c0 = (k - t * G) * 8;
  const int h = c0 / p.D, d0 = c0 - h * p.D;
  Eight<DT> x;
  x.load(p.kv, half * p.s.half + token_offset(p.s, t) + h * p.s.head + d0);
  uint16_t* const o = p.sink_rows[half] + static_cast<int64_t>(t) * p.C + c0;
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = half_bits(x.get(j));
}

template <int DT>
int launch_kivi(const KiviQuantParams& p, int sb, bool bytes, hipStream_t stream) {
  const uint32_t sink_tiles = (2 * p.sink * (p.C / 8) + kQThreads - 1) / kQThreads;
  const dim3 grid(p.tiles[0] + p.tiles[1] + (sink_tiles > 0 ? sink_tiles : 1)), block(kQThreads);
  if (bytes)
    hipLaunchKernelGGL((kivi_quantize_kernel<DT, 8, true>), grid, block, 0, stream, p);
  else if (sb == 2)
    hipLaunchKernelGGL((kivi_quantize_kernel<DT, 2, false>), grid, block, 0, stream, p);
  else if (sb == 4)
    hipLaunchKernelGGL((kivi_quantize_kernel<DT, 4, false>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((kivi_quantize_kernel<DT, 8, false>), grid, block, 0, stream, p);
  return check_launch("kivi_quantize_kernel");
}

// Checks that both quantizers share; fills `s`.  kv is 16-byte aligned and every row
// segment of 8 channels with it.
int check_kv(const void* kv, int64_t dtype, int64_t tokens, int64_t heads, int64_t head_dim,
             const int64_t* strides, KvStrides* s) {
  ORIGAMI_REQUIRE(dtype == ORIGAMI_DTYPE_FLOAT16 || dtype == ORIGAMI_DTYPE_BFLOAT16 ||
                      dtype == ORIGAMI_DTYPE_FLOAT32,
                  "K/V must be float16, bfloat16 or float32");
  ORIGAMI_REQUIRE(tokens > 0 && heads > 0 && head_dim > 0,
                  "tokens, heads, and head_dim must be positive");
  for (int i = 0; i < 4; ++i)
    ORIGAMI_REQUIRE(strides[i] >= 0, "K/V strides must be non-negative");
  ORIGAMI_REQUIRE(strides[4] > 0, "K/V block size must be positive");
  if (!aligned16(kv) || head_dim % 8 != 0 || strides[0] % 8 != 0 || strides[1] % 8 != 0 ||
      strides[2] % 8 != 0 || strides[3] % 8 != 0 || tokens > (int64_t(1) << 30) ||
      heads * head_dim > (int64_t(1) << 24) || strides[4] > UINT32_MAX)
    return fail(ORIGAMI_ERR_UNSUPPORTED, "the fused quantizers need 16-byte channel groups");
  *s = KvStrides{strides[0], strides[1], strides[2], strides[3],
                 static_cast<uint32_t>(strides[4])};
  return ORIGAMI_OK;
}

}  // namespace

extern "C" {

int origami_cachegen_quantize(const void* kv, int64_t dtype, int64_t tokens, int64_t heads,
                              int64_t head_dim, const int64_t* strides, int64_t key_bits,
                              int64_t value_bits, int64_t key_bins, int64_t value_bins,
                              uint8_t* payload, int64_t payload_bytes, int64_t value_offset,
                              int64_t key_max_offset, int64_t value_max_offset,
                              origami_stream_t stream_) {
  CacheGenQuantParams p{};
  if (int rc = check_kv(kv, dtype, tokens, heads, head_dim, strides, &p.s)) return rc;
  const int64_t C = heads * head_dim;
  const int64_t bits[2] = {key_bits, value_bits}, bins[2] = {key_bins, value_bins};
  const int64_t streams[2] = {0, value_offset}, maxima[2] = {key_max_offset, value_max_offset};
  for (int i = 0; i < 2; ++i) {
    ORIGAMI_REQUIRE(bits[i] >= 1 && bits[i] <= 8,
                    "Origami CUDA bitpack supports only 1..8 bit symbols");
    ORIGAMI_REQUIRE(bins[i] > 3 && bins[i] - 2 < (int64_t(1) << bits[i]),
                    "CacheGen bins do not fit the symbol width");
  }
  if (C > 4096) return fail(ORIGAMI_ERR_UNSUPPORTED, "CacheGen rows of at most 4096 channels");
  const int64_t bytes[2] = {tokens * C / 8 * key_bits, tokens * C / 8 * value_bits};
  ORIGAMI_REQUIRE(value_offset >= bytes[0] && key_max_offset >= value_offset + bytes[1] &&
                      value_max_offset >= key_max_offset + 2 * tokens &&
                      value_max_offset + 2 * tokens <= payload_bytes,
                  "CacheGen payload parts overlap or exceed the payload");
  ORIGAMI_REQUIRE((reinterpret_cast<uintptr_t>(payload) + key_max_offset) % 2 == 0 &&
                      (reinterpret_cast<uintptr_t>(payload) + value_max_offset) % 2 == 0,
                  "CacheGen maxima must be at even addresses");
  p.kv = kv;
  p.tokens = static_cast<uint32_t>(tokens);
  p.groups = static_cast<int32_t>(C / 8);
  p.head_groups = static_cast<int32_t>(head_dim / 8);
  p.row_lanes = 1;
  while (p.row_lanes < 64 && p.row_lanes < p.groups) p.row_lanes *= 2;
  for (int i = 0; i < 2; ++i) {
    p.bits[i] = static_cast<int32_t>(bits[i]);
    p.center[i] = static_cast<float>(bins[i] / 2 - 1);
    p.stream[i] = payload + streams[i];
    p.peak[i] = reinterpret_cast<uint16_t*>(payload + maxima[i]);
  }
  ORIGAMI_REQUIRE(key_max_offset - value_offset - bytes[1] <= 1,
                  "CacheGen payload has at most one pad byte");
  if (key_max_offset > value_offset + bytes[1]) p.pad = payload + key_max_offset - 1;
  const hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (dtype == ORIGAMI_DTYPE_FLOAT32)
    return launch_cachegen_rows<ORIGAMI_DTYPE_FLOAT32>(p, stream);
  if (dtype == ORIGAMI_DTYPE_BFLOAT16)
    return launch_cachegen_rows<ORIGAMI_DTYPE_BFLOAT16>(p, stream);
  return launch_cachegen_rows<ORIGAMI_DTYPE_FLOAT16>(p, stream);
}

int origami_kivi_quantize(const void* kv, int64_t dtype, int64_t tokens, int64_t heads,
                          int64_t head_dim, const int64_t* strides, int64_t bits,
                          int64_t group_size, int64_t sink_tokens, uint8_t* payload,
                          int64_t payload_bytes, const int64_t* offsets, uint8_t* workspace,
                          int64_t workspace_bytes, origami_stream_t stream_) {
  KiviQuantParams p{};
  if (int rc = check_kv(kv, dtype, tokens, heads, head_dim, strides, &p.s)) return rc;
  ORIGAMI_REQUIRE(bits == 2 || bits == 3 || bits == 4 || bits == 8,
                  "KIVI packs 2, 3, 4 or 8 bits");
  ORIGAMI_REQUIRE(group_size > 0 && sink_tokens >= 0 && sink_tokens < tokens,
                  "KIVI needs a positive group and a body token");
  const int64_t C = heads * head_dim, body = tokens - sink_tokens;
  if (group_size != 16 && group_size != 32 && group_size != 64 && group_size != 128)
    return fail(ORIGAMI_ERR_UNSUPPORTED, "fused KIVI groups are 16, 32, 64 or 128");
  const int sb = bits == 3 ? 4 : static_cast<int>(bits);
  const int64_t key_groups = (body + group_size - 1) / group_size;
  const int64_t value_groups = (C + group_size - 1) / group_size;
  const int64_t part[8] = {(C * body * sb + 7) / 8,     (C * body * sb + 7) / 8,
                           2 * key_groups * C,           2 * key_groups * C,
                           2 * body * value_groups,      2 * body * value_groups,
                           2 * sink_tokens * C,          2 * sink_tokens * C};
  int64_t end = 0;
  for (int i = 0; i < 8; ++i) {
    ORIGAMI_REQUIRE(offsets[i] >= end && offsets[i] - end <= 1,
                    "KIVI payload parts overlap or leave more than a pad byte");
    if (offsets[i] > end) p.pad[i] = payload + end;
    ORIGAMI_REQUIRE(i < 2 || (reinterpret_cast<uintptr_t>(payload) + offsets[i]) % 2 == 0,
                    "KIVI metadata must be at even addresses");
    end = offsets[i] + part[i];
  }
  ORIGAMI_REQUIRE(end <= payload_bytes, "KIVI payload is too small");

  // A lane's run of 16 symbols is whole aligned words of the stream when the planes are
  // whole runs; otherwise symbols go through the workspace, one per byte, and each
  // stream is packed from there (2 more bytes of traffic per symbol, but planes may start at any
  // bit).
  const bool direct = body % kQTokens == 0 && aligned16(payload) && offsets[1] % 16 == 0;
  SymbolRun runs[2];
  if (!direct) {
    ORIGAMI_REQUIRE(workspace != nullptr && workspace_bytes >= 2 * C * body,
                    "KIVI workspace is too small");
    for (int i = 0; i < 2; ++i) {
      runs[i] = SymbolRun{i * C * body, offsets[i], C * body};
      if (!pack_runs_aligned(workspace, payload, &runs[i], 1))
        return fail(ORIGAMI_ERR_UNSUPPORTED, "fused KIVI streams must start on dwords");
    }
  }
  p.kv = kv;
  p.tokens = static_cast<uint32_t>(tokens);
  p.sink = static_cast<uint32_t>(sink_tokens);
  p.body = static_cast<uint32_t>(body);
  p.H = static_cast<int32_t>(heads);
  p.D = static_cast<int32_t>(head_dim);
  p.C = static_cast<int32_t>(C);
  p.group = static_cast<int32_t>(group_size);
  p.vgroups = static_cast<int32_t>(value_groups);
  p.inv_levels = 1.0f / static_cast<float>((1 << bits) - 1);
  int64_t grid = 0;
  for (int i = 0; i < 2; ++i) {
    p.stream[i] = direct ? payload + offsets[i] : workspace + i * C * body;
    p.scale[i] = reinterpret_cast<uint16_t*>(payload + offsets[2 + 2 * i]);
    p.zero[i] = reinterpret_cast<uint16_t*>(payload + offsets[3 + 2 * i]);
    p.sink_rows[i] = reinterpret_cast<uint16_t*>(payload + offsets[6 + i]);
    const int64_t chan_lanes = i == 0 ? 8 : 16, tile_tokens = kQWaves * kQTokens * 64 / chan_lanes;
    p.chan_tiles[i] = static_cast<int32_t>((C + 8 * chan_lanes - 1) / (8 * chan_lanes));
    const int64_t tiles = p.chan_tiles[i] * ((body + tile_tokens - 1) / tile_tokens);
    grid += tiles;
    p.tiles[i] = static_cast<int32_t>(tiles);
  }
  if (grid + 2 * sink_tokens * C / 8 / kQThreads + 2 > INT32_MAX ||
      2 * sink_tokens * (C / 8) > INT32_MAX)
    return fail(ORIGAMI_ERR_UNSUPPORTED, "KIVI layer exceeds the launch grid");
  const hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  int rc = ORIGAMI_OK;
  if (dtype == ORIGAMI_DTYPE_FLOAT32)
    rc = launch_kivi<ORIGAMI_DTYPE_FLOAT32>(p, sb, !direct, stream);
  else if (dtype == ORIGAMI_DTYPE_BFLOAT16)
    rc = launch_kivi<ORIGAMI_DTYPE_BFLOAT16>(p, sb, !direct, stream);
  else
    rc = launch_kivi<ORIGAMI_DTYPE_FLOAT16>(p, sb, !direct, stream);
  for (int i = 0; i < 2 && !direct && rc == ORIGAMI_OK; ++i)
    rc = launch_pack_runs(workspace, &runs[i], 1, sb, payload, stream);
  return rc;
}

}  // extern "C"
