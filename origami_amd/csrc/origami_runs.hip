// origami_runs.hip -- MI355X (gfx950) kernels for symbol runs: stretches of a
// canonical stream whose symbols are consecutive bytes of the symbol tensor, in
// stream order.  Plain bit streams (a [1, 1, n] tensor: CacheGen symbols, quantized
// payloads stored as bytes) and token-fastest symbol tensors are such runs; the row
// kernels serve the token-major tensors, whose planes are strided.
//
// Both directions move each byte once, so HBM bounds them.  A lane owns 16 (or 32)
// consecutive symbols, so symbol accesses are 16 bytes per lane and a wave covers
// 1 KiB; the packed side is the lane's 2b (4b) bytes, adjacent to its neighbours'.
// Large unpacks and 8-bit packs keep kRunUnroll groups in flight per lane.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include "origami_internal.h"
#include "origami_layout.h"

using namespace origami_internal;

namespace {

constexpr int kRunThreads = 256;
// Groups of one lane in flight in the unpack and the 8-bit pack (the copy of a payload into
// its chunks), kRunThreads apart: 4 when the launch has at least kRunUnrollGroups groups,
// else 1.  us with 1 / 4, 5-bit symbols not in a cache: 8.4M 4.3 / 5.3, 16.8M 6.4 / 6.1,
// 33.6M 10.2 / 9.7, 67M 17.8 / 17.4, 134M 32.7 / 32.8 (8 bits: 4.6 / 4.4, 6.8 / 7.1, 12.2 /
// 11.8, 21.6 / 20.7, 45.1 / 46.5).  CacheGen saves, whose payload was just written: 10.6 MB
// 18.4 / 20.3, 21 MB 28.6 / 27.0, 42 MB 46.4 / 45.5.  The other packs keep 1: 5 bits, 8.4M
// 4.7 / 5.6, 33.6M 12.7 / 13.6, 134M 40.3 / 42.7.
constexpr int kRunUnroll = 4;
constexpr int64_t kRunUnrollGroups = int64_t(1) << 20;

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef unsigned int u32x3a4 __attribute__((ext_vector_type(3), aligned(4)));
typedef unsigned int u32x4a4 __attribute__((ext_vector_type(4), aligned(4)));

struct RunParams {
  const uint8_t* stream;  // unpack: 4-byte aligned base; pack: unused
  int64_t stream_bytes;   // unpack: readable bytes from `stream`
  int64_t bit_bias;       // unpack: (caller's stream - stream) * 8
  uint8_t* flat;          // pack: the caller's stream
  uint8_t* symbols;
  SymbolRun run[kMaxSymbolRuns];  // blockIdx.y
};

// N (1..5) dwords from a 4-byte aligned address.
template <int N>
__device__ __forceinline__ void load_dwords(const uint8_t* src, uint32_t* w) {
  if constexpr (N == 1) {
    w[0] = *reinterpret_cast<const uint32_t*>(src);
  } else if constexpr (N == 2) {
    const u32x2a4 x = *reinterpret_cast<const u32x2a4*>(src);
    w[0] = x.x;
    w[1] = x.y;
  } else if constexpr (N == 3) {
    const u32x3a4 x = *reinterpret_cast<const u32x3a4*>(src);
    w[0] = x.x;
    w[1] = x.y;
    w[2] = x.z;
  } else {
    const u32x4a4 x = *reinterpret_cast<const u32x4a4*>(src);
    w[0] = x.x;
    w[1] = x.y;
    w[2] = x.z;
    w[3] = x.w;
    if constexpr (N == 5) w[4] = *reinterpret_cast<const uint32_t*>(src + 16);
  }
}

// N (1..8) dwords to a 4-byte aligned address.
template <int N>
__device__ __forceinline__ void store_dwords(uint8_t* dst, const uint32_t* w) {
  if constexpr (N >= 4) {
    *reinterpret_cast<u32x4a4*>(dst) = u32x4a4{w[0], w[1], w[2], w[3]};
    if constexpr (N > 4) store_dwords<N - 4>(dst + 16, w + 4);
  } else if constexpr (N == 3) {
    *reinterpret_cast<u32x3a4*>(dst) = u32x3a4{w[0], w[1], w[2]};
  } else if constexpr (N == 2) {
    *reinterpret_cast<u32x2a4*>(dst) = u32x2a4{w[0], w[1]};
  } else {
    *reinterpret_cast<uint32_t*>(dst) = w[0];
  }
}

// The symbols of group s .. s + 15 that lie in [0, count), one byte each: a run's first
// or last group, or one whose dwords pass the end of the stream.  Its loads go out
// together (symbol by symbol, two loads and a store each in turn, a stream of 100 5-bit
// symbols took 5.2 us; now 2.6).
template <int BITS>
__device__ __forceinline__ void unpack_part(const RunParams& p, int64_t bit0, int64_t s,
                                            int64_t count, uint8_t* out) {
  constexpr int NU = (16 * BITS + 31) / 32;
  const int64_t bit = bit0 + s * BITS;  // negative before a stream's first symbol
  const int64_t byte = (bit >> 5) * 4;
  uint32_t w[NU + 1], x[NU > 4 ? NU : 4], o[4];
#pragma unroll
  for (int i = 0; i <= NU; ++i) {
    const int64_t at = byte + 4 * i;
    w[i] = at < 0 ? 0 : load_dword_guarded(p.stream, at, p.stream_bytes);
  }
#pragma unroll
  for (int i = 0; i < NU; ++i)
    x[i] = __builtin_amdgcn_alignbit(w[i + 1], w[i], static_cast<uint32_t>(bit & 31));
  expand16<BITS>(x, o);
#pragma unroll
  for (int j = 0; j < 16; ++j)
    if (s + j >= 0 && s + j < count) out[s + j] = static_cast<uint8_t>(o[j >> 2] >> (8 * (j & 3)));
}

// Stream -> symbols.  Group g holds the 16 symbols whose bytes are the g-th aligned
// 16 bytes from the run's first symbol byte rounded down, so every whole group is one
// aligned store whatever the run's alignment; its bits start anywhere and are funnel
// shifted.  DWORD: every group's bits start on a dword (b even), no shift and no
// extra dword.
template <int BITS, bool DWORD, int U>
__global__ __launch_bounds__(kRunThreads) void runs_unpack_kernel(RunParams p) {
  constexpr int NU = (16 * BITS + 31) / 32, NW = DWORD ? NU : NU + 1;
  const SymbolRun r = p.run[blockIdx.y];
  uint8_t* const out = p.symbols + r.symbol;
  const int lead = static_cast<int>(reinterpret_cast<uintptr_t>(out) & 15);
  const int64_t groups = (r.count + lead + 15) >> 4;
  const int64_t bit0 = p.bit_bias + r.byte * 8;
  const int64_t step = static_cast<int64_t>(gridDim.x) * kRunThreads * U;
  for (int64_t g0 = (static_cast<int64_t>(blockIdx.x) * U) * kRunThreads + threadIdx.x;
       g0 < groups; g0 += step) {
    uint32_t w[U][5];
    uint32_t whole = 0;  // bit u: group u is whole and its dwords lie in the stream
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t s = (g0 + u * kRunThreads) * 16 - lead;
      const int64_t byte = ((bit0 + s * BITS) >> 5) * 4;
      if (s >= 0 && s + 16 <= r.count && byte + 4 * NW <= p.stream_bytes) {
        whole |= 1u << u;
        load_dwords<NW>(p.stream + byte, w[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t s = (g0 + u * kRunThreads) * 16 - lead;
      if (whole & (1u << u)) {
        uint32_t x[NU > 4 ? NU : 4], o[4];
        const uint32_t sh = static_cast<uint32_t>((bit0 + s * BITS) & 31);
#pragma unroll
        for (int i = 0; i < NU; ++i)
          x[i] = DWORD ? w[u][i] : __builtin_amdgcn_alignbit(w[u][i + 1], w[u][i], sh);
        expand16<BITS>(x, o);
        __builtin_nontemporal_store(u32x4{o[0], o[1], o[2], o[3]},
                                    reinterpret_cast<u32x4*>(out + s));
      } else if (s < r.count) {
        unpack_part<BITS>(p, bit0, s, r.count, out);
      }
    }
  }
}

// Symbols -> stream.  A lane packs GS symbols, the fewest that fill whole dwords (16
// for even b, 32 for odd), so lanes never share a dword; the run's last group, if it
// is not whole, is written byte by byte with zero pad bits.  The run's symbols and
// its stream bytes start on dwords.
template <int BITS, int U>
__global__ __launch_bounds__(kRunThreads) void runs_pack_kernel(RunParams p) {
  constexpr int GS = BITS % 2 == 0 ? 16 : 32, NV = GS / 16, ND = GS * BITS / 32;
  // The last group of odd widths, up to 31 symbols, is loaded together and packed like the
  // others: 10007 7-bit symbols 4.6 -> 3.0 us.  Up to 15 symbols go one by one: as fast, and
  // the kernels of even widths are 2-5% faster with the shorter code (4.2M symbols 2.9 -> 2.75).
  constexpr bool kWholeTail = BITS % 2 == 1;
  const SymbolRun r = p.run[blockIdx.y];
  const uint8_t* const src = p.symbols + r.symbol;
  uint8_t* const dst = p.flat + r.byte;
  const int64_t groups = (r.count + GS - 1) / GS;
  const int64_t step = static_cast<int64_t>(gridDim.x) * kRunThreads * U;
  for (int64_t g0 = (static_cast<int64_t>(blockIdx.x) * U) * kRunThreads + threadIdx.x; g0 < groups;
       g0 += step) {
    uint32_t w[U][NV][4];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t s = (g0 + u * kRunThreads) * GS;
      if (s + GS <= r.count) {
#pragma unroll
        for (int v = 0; v < NV; ++v) load_dwords<4>(src + s + 16 * v, w[u][v]);
      } else {  // the run's last symbols, zeros past them
#pragma unroll
        for (int q = 0; q < GS / 4; ++q)
          w[u][q >> 2][q & 3] = kWholeTail ? load_dword_guarded(src, s + 4 * q, r.count) : 0;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t s = (g0 + u * kRunThreads) * GS;
      if (s >= r.count) continue;
      if (!kWholeTail && s + GS > r.count) {
        uint8_t* o = dst + s / GS * (4 * ND);
        uint32_t acc = 0;
        int n = 0;
        for (int64_t i = s; i < r.count; ++i) {
          acc |= (src[i] & ((1u << BITS) - 1u)) << n;
          n += BITS;
          if (n >= 8) {
            *o++ = static_cast<uint8_t>(acc);
            acc >>= 8;
            n -= 8;
          }
        }
        if (n > 0) *o = static_cast<uint8_t>(acc);
        continue;
      }
      uint32_t d[ND] = {};
#pragma unroll
      for (int j = 0; j < GS; ++j) {
        const uint32_t sym = (w[u][j >> 4][(j >> 2) & 3] >> (8 * (j & 3))) & ((1u << BITS) - 1u);
        const int dw = (j * BITS) >> 5, off = (j * BITS) & 31;
        d[dw] |= sym << off;
        if (off + BITS > 32) d[dw + 1] |= sym >> (32 - off);
      }
      uint8_t* const o = dst + s / GS * (4 * ND);
      if (s + GS <= r.count) {
        store_dwords<ND>(o, d);
      } else {
        const int n = static_cast<int>(((r.count - s) * BITS + 7) >> 3);
#pragma unroll
        for (int i = 0; i < 4 * ND; ++i)
          if (i < n) o[i] = static_cast<uint8_t>(d[i >> 2] >> (8 * (i & 3)));
      }
    }
  }
}

template <int BITS>
int launch_unpack(const RunParams& p, int nrun, int64_t groups, bool dword, hipStream_t stream) {
  const bool many = groups * nrun >= kRunUnrollGroups;
  const dim3 grid(grid_for(groups, int64_t(kRunThreads) * (many ? kRunUnroll : 1), 65536), nrun);
  const dim3 block(kRunThreads);
  if constexpr (BITS % 2 == 0) {
    if (dword) {
      if (many)
        hipLaunchKernelGGL((runs_unpack_kernel<BITS, true, kRunUnroll>), grid, block, 0, stream, p);
      else
        hipLaunchKernelGGL((runs_unpack_kernel<BITS, true, 1>), grid, block, 0, stream, p);
      return check_launch("runs_unpack_kernel");
    }
  }
  if (many)
    hipLaunchKernelGGL((runs_unpack_kernel<BITS, false, kRunUnroll>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((runs_unpack_kernel<BITS, false, 1>), grid, block, 0, stream, p);
  return check_launch("runs_unpack_kernel");
}

template <int BITS>
int launch_pack(const RunParams& p, int nrun, int64_t symbols, hipStream_t stream) {
  constexpr int GS = BITS % 2 == 0 ? 16 : 32;
  const int64_t groups = (symbols + GS - 1) / GS;
  const bool many = BITS == 8 && groups * nrun >= kRunUnrollGroups;
  const dim3 grid(grid_for(groups, int64_t(kRunThreads) * (many ? kRunUnroll : 1), 65536), nrun),
      block(kRunThreads);
  if constexpr (BITS == 8) {
    if (many) {
      hipLaunchKernelGGL((runs_pack_kernel<8, kRunUnroll>), grid, block, 0, stream, p);
      return check_launch("runs_pack_kernel");
    }
  }
  hipLaunchKernelGGL((runs_pack_kernel<BITS, 1>), grid, block, 0, stream, p);
  return check_launch("runs_pack_kernel");
}

}  // namespace

namespace origami_internal {

int collect_symbol_runs(const int64_t* offsets, const int64_t* bits, const int64_t* specs,
                        int64_t n, int64_t stride_token, int64_t stride_head,
                        int64_t stride_channel, SymbolRun (&runs)[kMaxSymbolRuns]) {
  int nrun = 0;
  for (int64_t k = 0; k < n; ++k) {
    if (bits[k] != bits[0]) return 0;
    const int64_t* s = specs + 6 * k;
    const int64_t Hc = s[1] - s[0], Cc = s[3] - s[2], Tc = s[5] - s[4];
    // stream order (head, channel, token fastest) is memory order
    if ((Tc > 1 && stride_token != 1) || (Cc > 1 && stride_channel != Tc) ||
        (Hc > 1 && stride_head != Cc * Tc))
      return 0;
    const int64_t symbol = s[4] * stride_token + s[0] * stride_head + s[2] * stride_channel;
    const int64_t count = Hc * Cc * Tc;
    if (nrun > 0) {
      SymbolRun& last = runs[nrun - 1];
      if (last.symbol + last.count == symbol && (last.count * bits[0]) % 8 == 0 &&
          last.byte + last.count * bits[0] / 8 == offsets[k]) {
        last.count += count;
        continue;
      }
    }
    if (nrun == kMaxSymbolRuns) return 0;
    runs[nrun++] = SymbolRun{symbol, offsets[k], count};
  }
  return nrun;
}

int launch_unpack_runs(const uint8_t* flat, int64_t flat_bytes, const SymbolRun* runs, int nrun,
                       int bits, uint8_t* symbols, hipStream_t stream) {
  RunParams p{};
  const uintptr_t addr = reinterpret_cast<uintptr_t>(flat), base = addr & ~uintptr_t(3);
  p.stream = reinterpret_cast<const uint8_t*>(base);
  p.bit_bias = static_cast<int64_t>(addr - base) * 8;
  p.stream_bytes = flat_bytes + static_cast<int64_t>(addr - base);
  p.symbols = symbols;
  int64_t groups = 0;
  bool dword = bits % 2 == 0;
  for (int i = 0; i < nrun; ++i) {
    p.run[i] = runs[i];
    const int64_t lead = (reinterpret_cast<uintptr_t>(symbols) + runs[i].symbol) & 15;
    groups = groups > (runs[i].count + lead + 15) / 16 ? groups : (runs[i].count + lead + 15) / 16;
    dword = dword && (p.bit_bias + runs[i].byte * 8 - lead * bits) % 32 == 0;
  }
  switch (bits) {
    case 1: return launch_unpack<1>(p, nrun, groups, dword, stream);
    case 2: return launch_unpack<2>(p, nrun, groups, dword, stream);
    case 3: return launch_unpack<3>(p, nrun, groups, dword, stream);
    case 4: return launch_unpack<4>(p, nrun, groups, dword, stream);
    case 5: return launch_unpack<5>(p, nrun, groups, dword, stream);
    case 6: return launch_unpack<6>(p, nrun, groups, dword, stream);
    case 7: return launch_unpack<7>(p, nrun, groups, dword, stream);
    case 8: return launch_unpack<8>(p, nrun, groups, dword, stream);
    default:
      return fail(ORIGAMI_ERR_INVALID, "Origami CUDA bitpack supports only 1..8 bit symbols");
  }
}

bool pack_runs_aligned(const uint8_t* symbols, const uint8_t* flat, const SymbolRun* runs,
                       int nrun) {
  for (int i = 0; i < nrun; ++i)
    if (((reinterpret_cast<uintptr_t>(symbols) + runs[i].symbol) & 3) != 0 ||
        ((reinterpret_cast<uintptr_t>(flat) + runs[i].byte) & 3) != 0)
      return false;
  return true;
}

int launch_pack_runs(const uint8_t* symbols, const SymbolRun* runs, int nrun, int bits,
                     uint8_t* flat, hipStream_t stream) {
  RunParams p{};
  p.symbols = const_cast<uint8_t*>(symbols);
  p.flat = flat;
  int64_t most = 0;
  for (int i = 0; i < nrun; ++i) {
    p.run[i] = runs[i];
    most = most > runs[i].count ? most : runs[i].count;
  }
  switch (bits) {
    case 1: return launch_pack<1>(p, nrun, most, stream);
    case 2: return launch_pack<2>(p, nrun, most, stream);
    case 3: return launch_pack<3>(p, nrun, most, stream);
    case 4: return launch_pack<4>(p, nrun, most, stream);
    case 5: return launch_pack<5>(p, nrun, most, stream);
    case 6: return launch_pack<6>(p, nrun, most, stream);
    case 7: return launch_pack<7>(p, nrun, most, stream);
    case 8: return launch_pack<8>(p, nrun, most, stream);
    default:
      return fail(ORIGAMI_ERR_INVALID, "Origami CUDA bitpack supports only 1..8 bit symbols");
  }
}

}  // namespace origami_internal
