// Decode GEMV of up to four rows behind an RMSNorm whose sums of squares the producer of h left behind:
//
//   y = x W^T, x = bf16( (h / rms) * gain ), rms from ssq[rows][parts] (per row the sums over 16 columns; parts = K / 16)
//
// K == kWaves * TPW * 128.  A workgroup takes T neighbouring 16-row tiles of W: every workgroup forms the rows' norm for itself, which costs it as
// many bytes from L2 as a tile of int4 weights and a chain of its own (sums, divisor, products, LDS, group sums), so a CU's tiles share one
// workgroup and its norm instead of having one each.  Wave w owns k groups [w TPW, (w + 1) TPW) of all tiles: rows and sums are requested first, then
// the weights of all tiles, and the norm is formed while those travel; its A fragments stay in registers and meet every tile.  The waves'
// partial sums of all tiles meet in LDS once; wave t adds and stores tile t.
// us, one tile a workgroup -> T (graph chains, int4, K = 2048, 1 / 2 / 4 rows): 6144 columns, T = 2: 3.8 / 4.9 / 5.1 -> 3.6 / 3.9 / 4.5; 11264 gated,
// T = 3: 4.7 / 6.3 / 6.8 -> 4.5 / 5.0 / 5.9; 32000: 8.3 / 12.4 / 12.8 -> 8.1 (T = 2) / 8.4 / 9.3 (T = 4).
#pragma once
#include "gemv_fused_kernels.h"

namespace ajq {

template <int kWaves, int TPW, int MROWS, int T, bool kW4, bool kGate>
__global__ __launch_bounds__(kWaves * 64) void dequant_gemv_norm_kernel(
    const u32x4_t* __restrict__ wq, const uint32_t* __restrict__ meta, int K, int m_flags, int N, void* __restrict__ y,
    const uint16_t* __restrict__ scales8, const float* __restrict__ h, const float* __restrict__ ssq, const float* __restrict__ gain,
    float eps, int parts) {
  const int M = m_flags & 0xFF;
  const bool out_f32 = (m_flags >> 8) != 0;
  constexpr int kSlice = TPW * kGroup, kStride = kSlice + 8, kVecPerRow = kSlice / 8, kVecs = MROWS * kVecPerRow;
  constexpr int kXLoads = (kVecs + 63) / 64, kLoadsPerGroup = kW4 ? 1 : 2, kRowQuads = (MROWS + 3) / 4;
  static_assert(kVecPerRow <= 64 && T <= kWaves, "a row's slice fits one wave-wide load, and every tile has a wave");
  extern __shared__ u32x4_t smem_raw[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nl = lane & 15, kc = lane >> 4, G = K >> 7, tiles = N / kTileN, nt0 = blockIdx.x * T, g0 = wave * TPW;
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem_raw) + wave * (MROWS * kStride);
  float* red = reinterpret_cast<float*>(reinterpret_cast<uint16_t*>(smem_raw) + kWaves * (MROWS * kStride));
  // ---- requests: the sums, the rows, meta, weights (vector loads return in issue order)
  u32x4_t w[T][TPW][kLoadsPerGroup];
  uint32_t mw[T][TPW];
  float4 a0[kXLoads][2], a2[kXLoads][2];
  __builtin_amdgcn_sched_barrier(0);
  constexpr int kLanesPerRow = 64 / MROWS, kPartLoads = (64 + kLanesPerRow - 1) / kLanesPerRow;
  float4 sums[kPartLoads];
  {
    const int row = lane / kLanesPerRow, piece = lane % kLanesPerRow;
#pragma unroll
    for (int u = 0; u < kPartLoads; ++u) {
      const int j = piece + u * kLanesPerRow;
      const bool live = 4 * j < parts && row < M;
      sums[u] = *reinterpret_cast<const float4*>(ssq + (live ? (size_t)row * parts + 4 * j : 0));
    }
  }
#pragma unroll
  for (int i = 0; i < kXLoads; ++i) {
    const int v = min(lane + 64 * i, kVecs - 1), m = min(v / kVecPerRow, M - 1), k = g0 * kGroup + 8 * (v % kVecPerRow);
    const float4* ph = reinterpret_cast<const float4*>(h + (size_t)m * K + k);
    const float4* pg = reinterpret_cast<const float4*>(gain + k);
    a0[i][0] = ph[0]; a0[i][1] = ph[1]; a2[i][0] = pg[0]; a2[i][1] = pg[1];
  }
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const size_t at = (size_t)(T > 1 ? min(nt0 + t, tiles - 1) : nt0) * G + g0;
    if (kW4) {
#pragma unroll
      for (int p = 0; p < TPW; ++p) mw[t][p] = meta[(at + p) * 16 + nl];
    }
    const u32x4_t* wtile = wq + at * kLoadsPerGroup * 64 + lane;
#pragma unroll
    for (int p = 0; p < TPW; ++p)
#pragma unroll
      for (int q = 0; q < kLoadsPerGroup; ++q) w[t][p][q] = __builtin_nontemporal_load(wtile + (p * kLoadsPerGroup + q) * 64);
  }
  uint32_t scale_bits = 0;
  if (!kW4) scale_bits = scales8[(T > 1 ? min(nt0 + min(wave, T - 1), tiles - 1) : nt0) * kTileN + nl];
  __builtin_amdgcn_sched_barrier(0);
  // ---- a row's total in all of its lanes: the kLanesPerRow lanes of a row share the parts
  float total = 0.f;
#pragma unroll
  for (int u = 0; u < kPartLoads; ++u) {
    // (idle lanes' words are dropped here and not at the load, which would become a branch of its own)
    asm volatile("" : "+v"(sums[u].x), "+v"(sums[u].y), "+v"(sums[u].z), "+v"(sums[u].w));
    const bool live = 4 * (lane % kLanesPerRow + u * kLanesPerRow) < parts && lane / kLanesPerRow < M;
    total += live ? (sums[u].x + sums[u].y) + (sums[u].z + sums[u].w) : 0.f;
  }
  if (kLanesPerRow >= 16) {
    total = team_sum16(total);
    if (kLanesPerRow == 64) total = quad_sum(total);
    else if (kLanesPerRow == 32) total += __shfl_xor(total, 16);
  } else {
#pragma unroll
    for (int off = kLanesPerRow / 2; off > 0; off >>= 1) total += __shfl_xor(total, off);
  }
  float* row_sum = red + wave * 16;  // (the wave's own words, ahead of the reduction's use of them)
  if (MROWS > 1) {
    if (lane % kLanesPerRow == 0) row_sum[lane / kLanesPerRow] = total;
    wave_lds_order();
  }
#pragma unroll
  for (int i = 0; i < kXLoads; ++i) {
    const int v = min(lane + 64 * i, kVecs - 1);
    const Divisor by_rms(sqrtf((MROWS > 1 ? row_sum[v / kVecPerRow] : total) / (float)(kWaves * kSlice) + eps));
    const float4 h0 = a0[i][0], h1 = a0[i][1], g0v = a2[i][0], g1v = a2[i][1];
    u32x4_t pk;
    pk.x = pack2_bf16(by_rms.divide(h0.x) * g0v.x, by_rms.divide(h0.y) * g0v.y);
    pk.y = pack2_bf16(by_rms.divide(h0.z) * g0v.z, by_rms.divide(h0.w) * g0v.w);
    pk.z = pack2_bf16(by_rms.divide(h1.x) * g1v.x, by_rms.divide(h1.y) * g1v.y);
    pk.w = pack2_bf16(by_rms.divide(h1.z) * g1v.z, by_rms.divide(h1.w) * g1v.w);
    *reinterpret_cast<u32x4_t*>(xs + (v / kVecPerRow) * kStride + 8 * (v % kVecPerRow)) = pk;
  }
  wave_lds_order();
  constexpr bool kValuSums = gemv_valu_group_sums(kW4, MROWS);
  const uint16_t* xrow = xs + min(nl, M - 1) * kStride + 8 * kc;
  float gs[kValuSums ? MROWS : 1][TPW];
  if constexpr (kValuSums) gemv_group_sums<TPW, MROWS>(xs, kStride, gs);
  u32x4_t frag[TPW][4];
  if (T > 1)
#pragma unroll
    for (int p = 0; p < TPW; ++p)
#pragma unroll
      for (int j = 0; j < 4; ++j) frag[p][j] = *reinterpret_cast<const u32x4_t*>(xrow + p * kGroup + 32 * j);
  __builtin_amdgcn_sched_barrier(0);
  auto fragment = [&](int p, int j) { return T > 1 ? frag[p][j] : *reinterpret_cast<const u32x4_t*>(xrow + p * kGroup + 32 * j); };
  const W4Consts w4c = w4_consts();
  const u32x4_t ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
  // Four waves of twice the groups keep the sums of their two halves apart: added up like those of eight waves, the outputs are
  // the same bit for bit.
  constexpr int kHalves = kWaves == 4 ? 2 : 1, kParts = kWaves * kHalves;
  static_assert(TPW % kHalves == 0, "whole groups per half");
  constexpr int kLive = MROWS < 4 ? MROWS : 4;
  typedef float live_t __attribute__((ext_vector_type(kLive == 3 ? 4 : kLive)));
  live_t* redv = reinterpret_cast<live_t*>(red + (MROWS > 1 ? kWaves * 16 : 0));
  f32x4_t acc[T][kHalves] = {};
  auto half = [](int p) { return p * kHalves / TPW; };
#pragma unroll
  for (int t = 0; t < T; ++t) {
    if (kW4) {
#pragma unroll
      for (int p = 0; p < TPW; ++p) {
        const float sc = f16_bits_to_f32(mw[t][p] & 0xFFFFu), zc = f16_bits_to_f32(mw[t][p] >> 16);
        f32x4_t part = {0.f, 0.f, 0.f, 0.f}, asum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u32x4_t a = fragment(p, j);
          part = mfma16(a, w4_unpack(w[t][p][0][j], w4c), part);
          if (!kValuSums) asum = mfma16(a, ones, asum);
        }
#pragma unroll
        for (int i = 0; i < kLive; ++i) acc[t][half(p)][i] += sc * (part[i] - zc * (kValuSums ? gs[kValuSums ? i : 0][p] : asum[i]));
      }
    } else {
#pragma unroll
      for (int p = 0; p < TPW; ++p)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u32x2_t lo = w8_to_bf16(w[t][p][j >> 1][2 * (j & 1)]), hi = w8_to_bf16(w[t][p][j >> 1][2 * (j & 1) + 1]);
          acc[t][half(p)] = mfma16(fragment(p, j), u32x4_t{lo.x, lo.y, hi.x, hi.y}, acc[t][half(p)]);
        }
    }
#pragma unroll
    for (int u = 0; u < kHalves; ++u) {
      asm volatile("" : "+v"(acc[t][u]));
      live_t mine;
#pragma unroll
      for (int i = 0; i < kLive; ++i) mine[i] = acc[t][u][i];
      if (kc < kRowQuads) redv[(t * kParts + wave * kHalves + u) * (16 * kRowQuads) + lane] = mine;
    }
  }
  if (!kW4) asm volatile("" : "+v"(scale_bits));
  __syncthreads();
  const int nt = nt0 + wave;
  if (wave >= T || (T > 1 && nt >= tiles) || kc >= kRowQuads) return;
  live_t sum = redv[wave * kParts * (16 * kRowQuads) + lane];
#pragma unroll
  for (int u = 1; u < kParts; ++u) sum += redv[(wave * kParts + u) * (16 * kRowQuads) + lane];
  const int n = nt * kTileN + nl;
  const float cs = kW4 ? 1.0f : f16_bits_to_f32(scale_bits);
#pragma unroll
  for (int i = 0; i < kLive; ++i) {
    const int m = 4 * kc + i;
    const float v = sum[i] * cs;
    if (kGate) {
      // columns 0..7 of the tile are gate projections, 8..15 the matching up projections
      const float other = row_ror<8>(v);
      if (nl < 8 && m < M) reinterpret_cast<uint16_t*>(y)[(size_t)m * (N >> 1) + nt * 8 + nl] = f32_to_bf16_rne(v * (1.0f / (1.0f + expf(-v))) * other);
    } else if (m < M) {
      if (out_f32) reinterpret_cast<float*>(y)[(size_t)m * N + n] = v;
      else reinterpret_cast<uint16_t*>(y)[(size_t)m * N + n] = f32_to_bf16_rne(v);
    }
  }
}
// activation slices, the rows' totals, the partial sums of all tiles
constexpr size_t gemv_norm_lds_bytes(int waves, int tpw, int mrows, int t) {
  return (size_t)waves * mrows * (tpw * kGroup + 8) * 2 + (mrows > 1 ? (size_t)waves * 64 : 0) +
         (size_t)t * waves * (waves == 4 ? 2 : 1) * (16 * ((mrows + 3) / 4)) * 4 * (mrows < 4 ? mrows : 4);
}

}  // namespace ajq
