// Weight quantize/pack kernels: fp32 [N, K] -> canonical W8 / W4-g128 tensors.
// Every operation that decides an integer is IEEE binary32, round-to-nearest-even,
// so the outputs are bit-identical to the CPU statement of the scheme.
#pragma once
#include "ajq_common.h"

namespace ajq {

// Codes of many weights over one d, the common case: |w / d| <= 2^21 and d one of fp16's finite positive values.  Then the three-
// instruction quotient of `Divisor` is the correctly rounded one (a numerator small enough to lose its residual to underflow
// rounds to code 0 either way), and adding 1.5 * 2^23 rounds it to the nearest integer, ties to even, which lies in the sum's
// low bits: no rounding, conversion or masking instruction.  Anything else takes the division.  The choice is made once per
// wavefront and run of weights.
constexpr float kRoundingBias = 12582912.0f;
__device__ __forceinline__ bool plain_quotients(float d, float largest) { return __all(largest <= 2097152.0f * d && d <= 65504.0f); }
// the bits of rint(w / d) + the bias, between two bounds that include it
__device__ __forceinline__ uint32_t biased_code(const Divisor& by, float w, float lo, float hi) {
  return __float_as_uint(fminf(fmaxf(by.divide(w) + kRoundingBias, lo), hi));
}

// ---------------------------------------------------------------- W8 ------
// Place (in dwords) of the four codes of row n at column k = 4 word in the private tensor of K128 columns.
__device__ __forceinline__ size_t w8_private_word(int n, int word, int K128) {
  const int t = word >> 4, r = word & 15;  // 64-k tile, dword within it
  return ((size_t)((n >> 4) * (size_t)(K128 / kW8TileK) + t) * 64 + 16 * ((r >> 1) & 3) + (n & 15)) * 4 + 2 * (r >> 3) + (r & 1);
}

// q = clamp(rint(w / float(scale)), -127, 127), scale = fp16(absmax / 127).  One workgroup per output row, the row read once
// and held in registers (NV vectors of four per thread: K <= 1024 NV), the codes written in both layouts.  wq (may be null):
// rows N .. and columns K .. K128 of the private tensor become zero codes.  Bound: HBM (4 bytes in, 1 + 1 out per weight).
// The 16 rows of a private tile go to one XCD, whose L2 puts their 16-byte pieces of a line together: workgroups are dealt to
// the 8 XCDs in turn.  The row read twice, a division per code and a repack launch behind it: 94 + 50 us on
// 4096 x 14336.
template <int NV>
__global__ __launch_bounds__(256) void quantize_w8_row_kernel(const float* __restrict__ W, int N, int K, int K128,
                                                              uint32_t* __restrict__ q, uint16_t* __restrict__ scales,
                                                              uint32_t* __restrict__ wq) {
  const int unit = blockIdx.x >> 3;
  const int n = ((unit >> 4) * 8 + (blockIdx.x & 7)) * kTileN + (unit & 15);
  const int n16 = (N + kTileN - 1) / kTileN * kTileN;
  if (n >= n16) return;
  const int words = K >> 2, padded = K128 >> 2;
  if (n >= N) {
    if (wq)
      for (int i = threadIdx.x; i < padded; i += 256) wq[w8_private_word(n, i, K128)] = 0u;
    return;
  }
  const f32x4_t* row = reinterpret_cast<const f32x4_t*>(W + (size_t)n * K);
  f32x4_t v[NV];
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = threadIdx.x + 256 * j;
    v[j] = i < words ? __builtin_nontemporal_load(row + i) : f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int j = 0; j < NV; ++j) amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[j].x), fabsf(v[j].y)), fmaxf(fabsf(v[j].z), fabsf(v[j].w))));
  for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  __shared__ float wave_max[4];
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));
  const __half hs = __float2half_rn(amax / 127.0f);
  if (threadIdx.x == 0) scales[n] = __half_as_ushort(hs);
  float d = __half2float(hs);
  if (d == 0.0f) d = 1.0f;
  auto store = [&](auto code) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = threadIdx.x + 256 * j;
      const uint32_t word = __builtin_amdgcn_perm(__builtin_amdgcn_perm(code(v[j].w), code(v[j].z), 0x0C0C0400u),
                                                  __builtin_amdgcn_perm(code(v[j].y), code(v[j].x), 0x0C0C0400u), 0x05040100u);
      if (i < words) q[(size_t)n * words + i] = word;
      if (wq && i < padded) wq[w8_private_word(n, i, K128)] = i < words ? word : 0u;
    }
  };
  if (plain_quotients(d, amax)) {
    const Divisor by(d);
    store([by](float w) { return biased_code(by, w, kRoundingBias - 127.0f, kRoundingBias + 127.0f); });
  } else {
    store([d](float w) { return (uint32_t)(int)fminf(fmaxf(rintf(w / d), -127.0f), 127.0f); });
  }
}

// The same for rows that do not fit the registers and for short ones (canonical codes only): the second read of a row hits a cache.
__global__ __launch_bounds__(256) void quantize_w8_kernel(const float* __restrict__ W, int K,
                                                          int8_t* __restrict__ q,
                                                          uint16_t* __restrict__ scales) {
  const int n = blockIdx.x;
  const float4* row = reinterpret_cast<const float4*>(W + (size_t)n * K);
  const int k4 = K >> 2;
  float amax = 0.0f;
  for (int i = threadIdx.x; i < k4; i += 256) {
    float4 v = row[i];
    amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
  }
  for (int off = 32; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off));
  __shared__ float wave_max[4];
  if ((threadIdx.x & 63) == 0) wave_max[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(wave_max[0], wave_max[1]), fmaxf(wave_max[2], wave_max[3]));

  const __half hs = __float2half_rn(amax / 127.0f);
  if (threadIdx.x == 0) scales[n] = __half_as_ushort(hs);
  float d = __half2float(hs);
  if (d == 0.0f) d = 1.0f;

  uint32_t* qrow = reinterpret_cast<uint32_t*>(q + (size_t)n * K);
  for (int i = threadIdx.x; i < k4; i += 256) {
    float4 v = row[i];
    int a = (int)fminf(fmaxf(rintf(v.x / d), -127.0f), 127.0f);
    int b = (int)fminf(fmaxf(rintf(v.y / d), -127.0f), 127.0f);
    int c = (int)fminf(fmaxf(rintf(v.z / d), -127.0f), 127.0f);
    int e = (int)fminf(fmaxf(rintf(v.w / d), -127.0f), 127.0f);
    qrow[i] = (uint32_t)(a & 0xFF) | ((uint32_t)(b & 0xFF) << 8) | ((uint32_t)(c & 0xFF) << 16) |
              ((uint32_t)(e & 0xFF) << 24);
  }
}

// ---------------------------------------------------------------- W4 ------
// The canonical tensors alone: 16 lanes own one 128-wide group (8 consecutive weights per lane, one packed word out), a workgroup 16
// consecutive groups of all.  Bound: HBM; no tile is put together, and many small workgroups beat the few large ones of the kernel below
// (16 x 4096: 2.4 us, 4.1 below; 4096 x 4096: 15.5 / 19.2; 14336 x 4096: 44.3 / 50.4).
__global__ __launch_bounds__(256) void quantize_w4_codes_kernel(const float* __restrict__ W, long long groups, uint32_t* __restrict__ qweight,
                                                                uint16_t* __restrict__ scales, uint8_t* __restrict__ zeros) {
  const long long g = (long long)blockIdx.x * 16 + (threadIdx.x >> 4);
  if (g >= groups) return;  // the 16 lanes of a group leave together
  const int sub = threadIdx.x & 15;
  const float4* src = reinterpret_cast<const float4*>(W + g * kGroup + sub * 8);
  const float4 v0 = src[0], v1 = src[1];
  const float w[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
  float mn = w[0], mx = w[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) {
    mn = fminf(mn, w[i]);
    mx = fmaxf(mx, w[i]);
  }
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) {
    mn = fminf(mn, __shfl_xor(mn, off));
    mx = fmaxf(mx, __shfl_xor(mx, off));
  }
  const __half hs = __float2half_rn((mx - mn) / 15.0f);
  float d = __half2float(hs);
  if (d == 0.0f) d = 1.0f;
  const float zf = fminf(fmaxf(rintf(-mn / d), 0.0f), 15.0f);
  uint32_t word = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i) word |= (uint32_t)(int)fminf(fmaxf(rintf(w[i] / d) + zf, 0.0f), 15.0f) << (4 * i);
  qweight[g * 16 + sub] = word;
  if (sub == 0) {
    scales[g] = __half_as_ushort(hs);
    zeros[g] = (uint8_t)(int)zf;
  }
}

// With the private tiles: 16 lanes own one 128-wide group (8 consecutive weights per lane, one packed word out); a workgroup takes the 16 rows of a
// private tile and four consecutive groups, a wavefront four of the rows (2 KiB of each at a time), and writes the codes in
// both layouts: the canonical tensors, and the private tiles, put together in LDS and written as whole
// lines; their rows N .. are zero codes with zero scales.  Bound: HBM (4 bytes in, 0.5 + 0.5 out per weight).  14336 x 4096: 54
// us = 5.5 TB/s, the rate of a large copy; codes, tiles and meta words as three launches with 16-byte loads 32 bytes apart took
// 70, the same loads in this one launch 60, a range of its own per XCD 56.
constexpr int kQuantizeGroups = 4;
// the value of the other lane of a pair (DPP quad_perm [1, 0, 3, 2]); of lane ^ 16 (within a half wavefront)
__device__ __forceinline__ float neighbour(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}
__device__ __forceinline__ float other_row(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_ds_swizzle(__builtin_bit_cast(int, v), 0x401F));
}
__global__ __launch_bounds__(256) void quantize_w4_kernel(const float* __restrict__ W, int N, int G, uint32_t* __restrict__ qweight,
                                                          uint16_t* __restrict__ scales, uint8_t* __restrict__ zeros,
                                                          u32x4_t* __restrict__ wq, uint32_t* __restrict__ meta) {
  constexpr int kRows = 4;
  __shared__ __attribute__((aligned(16))) uint32_t tile_s[kQuantizeGroups * 256];
  const int chunks = (G + kQuantizeGroups - 1) / kQuantizeGroups;
  const int nt = blockIdx.x / chunks, g0 = blockIdx.x % chunks * kQuantizeGroups;
  // A wavefront's loads cover a row's 2 KiB as two whole KiB; then neighbours trade a vector each, so that the even lanes of a
  // half hold 32 consecutive bytes each of one of the first two groups, the odd ones of the last two.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, team = 2 * (lane & 1) + (lane >> 5), sub = (lane & 31) >> 1, g = g0 + team;
  const bool odd = lane & 1;
  f32x4_t v[kRows][2];
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const int n = nt * kTileN + kRows * wave + i;
    const f32x4_t* p = reinterpret_cast<const f32x4_t*>(W + ((size_t)n * G + g0) * kGroup) + lane;
#pragma unroll
    for (int h = 0; h < 2; ++h)
      v[i][h] = n < N && g0 + 2 * h + (lane >> 5) < G ? __builtin_nontemporal_load(p + 64 * h) : f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int i = 0; i < kRows; ++i) {
    const int nl = kRows * wave + i, n = nt * kTileN + nl;
    float w[8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float other = neighbour(odd ? v[i][0][e] : v[i][1][e]);
      w[e] = odd ? other : v[i][0][e];
      w[4 + e] = odd ? v[i][1][e] : other;
    }
    float mn = w[0], mx = w[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) {
      mn = fminf(mn, w[e]);
      mx = fmaxf(mx, w[e]);
    }
    mn = fminf(mn, row_ror<8>(mn)); mx = fmaxf(mx, row_ror<8>(mx));
    mn = fminf(mn, row_ror<4>(mn)); mx = fmaxf(mx, row_ror<4>(mx));
    mn = fminf(mn, row_ror<2>(mn)); mx = fmaxf(mx, row_ror<2>(mx));
    mn = fminf(mn, other_row(mn)); mx = fmaxf(mx, other_row(mx));
    const __half hs = __float2half_rn((mx - mn) / 15.0f);
    float d = __half2float(hs);
    if (d == 0.0f) d = 1.0f;
    float zf;
    uint32_t word = 0, tile = 0;
    auto tile_shift = [](int e) { return 4 * ((e >> 1) + 4 * (e & 1)); };
    if (plain_quotients(d, fmaxf(fabsf(mn), fabsf(mx)))) {
      const Divisor by(d);
      zf = __uint_as_float(biased_code(by, -mn, kRoundingBias, kRoundingBias + 15.0f)) - kRoundingBias;
      const float lo = kRoundingBias - zf;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t code = biased_code(by, w[e], lo, lo + 15.0f);
        word += code << (4 * e);
        tile += code << tile_shift(e);
      }
      word -= __float_as_uint(lo) * 0x11111111u;  // eight times the bits of lo, each at its own nibble
      tile -= __float_as_uint(lo) * 0x11111111u;
    } else {
      zf = fminf(fmaxf(rintf(-mn / d), 0.0f), 15.0f);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t code = (uint32_t)(int)fminf(fmaxf(rintf(w[e] / d) + zf, 0.0f), 15.0f);
        word |= code << (4 * e);
        tile |= code << tile_shift(e);
      }
    }
    tile_s[team * 256 + (16 * (sub & 3) + nl) * 4 + (sub >> 2)] = n < N ? tile : 0u;
    if (g < G) {
      if (n < N) {
        qweight[((size_t)n * G + g) * 16 + sub] = word;
        if (sub == 0) {
          scales[(size_t)n * G + g] = __half_as_ushort(hs);
          zeros[(size_t)n * G + g] = (uint8_t)(int)zf;
        }
      }
      const __half zc = __float2half_rn(128.0f + zf);  // <= 143: exact
      if (sub == 0) meta[((size_t)nt * G + g) * kTileN + nl] = (uint32_t)__half_as_ushort(hs) | (uint32_t)__half_as_ushort(zc) << 16;
    }
  }
  __syncthreads();
  if (g0 + wave < G) wq[((size_t)nt * G + g0) * 64 + threadIdx.x] = reinterpret_cast<const u32x4_t*>(tile_s)[threadIdx.x];
}

// ------------------------------------------------------------ repack ------
// canonical W4 -> private tiles.  One thread per private dword.
__global__ __launch_bounds__(256) void repack_w4_kernel(const uint32_t* __restrict__ qweight, int N,
                                                        int K, uint32_t* __restrict__ wq) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long total = (long long)N * (K / 8);
  if (idx >= total) return;
  const int G = K / kGroup;
  const int j = idx & 3;
  const int lane = (idx >> 2) & 63;
  const long long tile = idx >> 8;
  const int g = (int)(tile % G);
  const int nt = (int)(tile / G);
  const int nl = lane & 15, kc = lane >> 4;
  const int n = nt * kTileN + nl;
  const int k = g * kGroup + 32 * j + 8 * kc;
  const uint32_t w = qweight[(size_t)n * (K / 8) + (k >> 3)];
  uint32_t out = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t v = (w >> (4 * e)) & 0xFu;
    out |= v << (4 * ((e >> 1) + 4 * (e & 1)));
  }
  wq[idx] = out;
}

__global__ __launch_bounds__(256) void repack_w4_meta_kernel(const uint16_t* __restrict__ scales,
                                                             const uint8_t* __restrict__ zeros, int N,
                                                             int G, uint32_t* __restrict__ meta) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long long)N * G) return;
  const int nl = idx & 15;
  const long long tile = idx >> 4;
  const int g = (int)(tile % G);
  const int nt = (int)(tile / G);
  const size_t src = (size_t)(nt * kTileN + nl) * G + g;
  const __half zc = __float2half_rn(128.0f + (float)zeros[src]);  // <= 143: exact
  meta[idx] = (uint32_t)scales[src] | ((uint32_t)__half_as_ushort(zc) << 16);
}

__global__ __launch_bounds__(256) void unrepack_w4_kernel(const uint32_t* __restrict__ wq, int N, int K,
                                                          uint32_t* __restrict__ qweight) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long total = (long long)N * (K / 8);
  if (idx >= total) return;
  const int G = K / kGroup;
  const int j = idx & 3;
  const int lane = (idx >> 2) & 63;
  const long long tile = idx >> 8;
  const int g = (int)(tile % G);
  const int nt = (int)(tile / G);
  const int nl = lane & 15, kc = lane >> 4;
  const int n = nt * kTileN + nl;
  const int k = g * kGroup + 32 * j + 8 * kc;
  const uint32_t w = wq[idx];
  uint32_t out = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t v = (w >> (4 * ((e >> 1) + 4 * (e & 1)))) & 0xFu;
    out |= v << (4 * e);
  }
  qweight[(size_t)n * (K / 8) + (k >> 3)] = out;
}

__global__ __launch_bounds__(256) void unrepack_w4_meta_kernel(const uint32_t* __restrict__ meta, int N,
                                                               int G, uint16_t* __restrict__ scales,
                                                               uint8_t* __restrict__ zeros) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long long)N * G) return;
  const int nl = idx & 15;
  const long long tile = idx >> 4;
  const int g = (int)(tile % G);
  const int nt = (int)(tile / G);
  const size_t dst = (size_t)(nt * kTileN + nl) * G + g;
  const uint32_t m = meta[idx];
  scales[dst] = (uint16_t)(m & 0xFFFFu);
  zeros[dst] = (uint8_t)(int)(f16_bits_to_f32(m >> 16) - 128.0f);
}

// canonical W8 [N, K] int8 -> private tiles.  One thread per private dword.
// dword (tile (nt, t), lane (kc, nl), d) holds k = 64t + 32*(d>>1) + 8kc + 4*(d&1) .. +4
template <bool kInverse>
__global__ __launch_bounds__(256) void repack_w8_kernel(const uint32_t* __restrict__ src, int N, int K,
                                                        uint32_t* __restrict__ dst) {
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  const long long total = (long long)N * (K / 4);
  if (idx >= total) return;
  const int T = K / kW8TileK;
  const int d = idx & 3;
  const int lane = (idx >> 2) & 63;
  const long long tile = idx >> 8;
  const int t = (int)(tile % T);
  const int nt = (int)(tile / T);
  const int nl = lane & 15, kc = lane >> 4;
  const int n = nt * kTileN + nl;
  const int k = t * kW8TileK + 32 * (d >> 1) + 8 * kc + 4 * (d & 1);
  const size_t canon = (size_t)n * (K / 4) + (k >> 2);
  if (kInverse)
    dst[canon] = src[idx];
  else
    dst[idx] = src[canon];
}

}  // namespace ajq
