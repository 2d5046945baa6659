// Matrix-vector products of one decode step for dense bf16 weights [N, K] (row-major, N % 16 == 0, K % 8 == 0) on
// MFMA, up to 16 sequences per workgroup (grid.y deals larger batches), with what surrounds them folded in:
//
//   dense_in_kernel      two weight matrices that read the same fp32 residual row through norms of their own: the layer
//                        norm is the prologue (or bf16 rows a norm launch left); the first matrix's outputs are stored
//                        in fp32, the second's go through an activation: gated pairs (8 gate rows and their 8 up rows per
//                        16-row tile), or every row by itself
//   latent_absorb_kernel per-head products of the unrotated query with the transposed key expansion, so that attention
//                        can run on the latents; beside them the rotation of the query, and the new cache row (RMS norm of
//                        the latent, rotation of the shared key part)
//   latent_expand_kernel merge of the attention's row chunks (with the sink), per-head value expansion, output gate
//   dense_out_kernel     product with the residual add (and whatever the next layer run adds first) as epilogue
//   dense_out_streams_kernel  product whose epilogue mixes it into several residual streams and forms what the next sublayer reads
//
// A 16 x 16 output tile (16 weight rows, 16 batch columns) belongs to a wave, or to kWaves waves that split K and meet in
// LDS.  The small products' lane l = 16 g + r loads 16 bytes of weight row r at k = 32 step + 8 g (`tile_steps`); the large
// ones stream whole lines (`stream_rows`).
#pragma once
#include "dense_kernels.h"
#include "latent_attention.h"
#include "stream_kernels.h"

namespace ajq {

constexpr int kGemvBatch = 16;

// acc += W[16 rows, steps begin .. end) x; `wrow` points at this lane's row, `x(step)` gives the B fragment (batch column r, k = 32
// step + 8 g ..), both zero past K.
template <typename XFn>
__device__ __forceinline__ void tile_steps(const uint16_t* __restrict__ wrow, int K, int begin, int end, int g, f32x4_t& acc, XFn&& x) {
  constexpr int kUnroll = 8;
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  for (int s0 = begin; s0 < end; s0 += kUnroll) {
    u32x4_t w[kUnroll], v[kUnroll];
#pragma unroll
    for (int i = 0; i < kUnroll; ++i) {
      const int k = 32 * (s0 + i) + 8 * g;
      w[i] = zero;
      if (s0 + i < end && k < K) w[i] = *reinterpret_cast<const u32x4_t*>(wrow + k);
    }
#pragma unroll
    for (int i = 0; i < kUnroll; ++i) {
      v[i] = zero;
      if (s0 + i < end && 32 * (s0 + i) + 8 * g < K) v[i] = x(s0 + i);
    }
#pragma unroll
    for (int i = 0; i < kUnroll; ++i) acc = mfma16(w[i], v[i], acc);
  }
}

// sum of the waves' tiles; tile (n, t) is valid in wave n BT + t
template <int kWaves, int RT, int BT>
__device__ __forceinline__ void meet(f32x4_t (&acc)[RT][BT], float* red, int wave, int lane) {
  if (kWaves == 1) return;
  static_assert(kWaves == 1 || RT * BT <= kWaves, "a wave per tile");
  float4* slot = reinterpret_cast<float4*>(red);
#pragma unroll
  for (int i = 0; i < RT * BT; ++i) {
    const f32x4_t& v = acc[i / BT][i % BT];
    if (wave != i) slot[(i * kWaves + wave) * 64 + lane] = float4{v[0], v[1], v[2], v[3]};
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RT * BT; ++i) {
    if (wave != i) continue;
    f32x4_t& v = acc[i / BT][i % BT];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      if (w == i) continue;
      const float4 o = slot[(i * kWaves + w) * 64 + lane];
      v[0] += o.x; v[1] += o.y; v[2] += o.z; v[3] += o.w;
    }
  }
}

// acc[n][t] += W[rows of tile n, :] x_t for RT tiles of ROWS (16 or 8) consecutive rows of a row-major W [.., K], K split over
// kWaves waves in blocks of 128 columns, UQ of them requested together.  `w`: the first row; `xrows`: the first of nb batch rows [.., K];
// `between` runs while the first blocks travel.  `lds`: stream_lds() bytes; the tiles' sums of all waves are complete in wave n BT + t (as
// `meet` leaves them).
//
// Bound: HBM.  What costs is how a row-major matrix is asked for: the product's own operand layout wants 64 bytes of each of 16
// rows per instruction, half a line everywhere, and streams at 4.4 TB/s; four rows of 256 bytes per instruction stream at 5.9
// (4096 x 18432, 8 sequences: 38.3 -> 25.7 us; 35424 x 4096: 63.0 -> 46.3; 2048 x 8192: 13.9 -> 7.9 with tiles of 8 rows on
// twice as many CUs).  The block then takes the operand layout on its way through wave-private LDS (no barrier; chunk c of row
// r lies in slot c ^ r, so that both the rows' writes and the operand reads meet all banks), while the next one travels.
//
// XQ: the batch rows go the same way, ahead of the weights, four rows per instruction: XQ = 1, 2 or 4 instructions per batch tile
// and block hold up to 4, 8 or 16 of them.  In the operand layout they were four instructions of half lines whatever the batch, as many
// as the weights' (twice as many for tiles of 8 rows).  us, before -> after: 2048 x 8192: 4 sequences 8.0 -> 7.5, 16 11.4 -> 9.7, 32 18.3 ->
// 12.8; 4096 x 18432: 16 29.9 -> 27.5, 32 44.7 -> 35.0; 35424 x 4096: 16 55.6 -> 51.3, 32 68.5 -> 57.6.
// XQ = kStreamDirect: `x(t, k)` gives the B fragment of batch tile t at columns k + 8 g .. of batch column r, from memory, asked for behind the
// weights: short rows, and many tiles with up to four sequences (16384 x 4096: 21.2 us, 21.7 staged); kStreamFrom: from LDS, behind `between`.
constexpr int kStreamBlock = 128;
enum { kStreamFrom = 0, kStreamDirect = -1 };
constexpr int stream_wave_lds(int rows, int rt, int bt, int uq, int xq) { return uq * (rt * rows + (xq > 0 ? bt * 4 * xq : 0)) * 256; }
constexpr int stream_lds(int waves, int rows, int rt, int bt, int uq, int xq) {
  const int blocks = waves * stream_wave_lds(rows, rt, bt, uq, xq), sums = rt * bt * waves * 1024;
  return blocks > sums ? blocks : sums;
}
template <int kWaves, int ROWS, int RT, int BT, int UQ, int XQ, typename Between, typename XFn>
__device__ __forceinline__ void stream_rows(const uint16_t* __restrict__ w, int K, int wave, int lane, unsigned char* lds,
                                            f32x4_t (&acc)[RT][BT], const uint16_t* __restrict__ xrows, int nb, Between&& between, XFn&& x) {
  static_assert(ROWS == 16 || ROWS == 8, "tiles of 16 or 8 rows");
  constexpr int kLoads = ROWS / 4;  // instructions of 1 KiB per tile and block
  constexpr bool kStaged = XQ > 0, kAhead = XQ != kStreamFrom;
  constexpr int kX = kStaged ? XQ : 4;
  const int r = lane & 15, g = lane >> 4, rr = ROWS == 16 ? r : r & 7;
  const int full = K / kStreamBlock, per = (full + kWaves - 1) / kWaves;
  const int begin = min(full, wave * per), count = min(full, begin + per) - begin;
  unsigned char* mine = lds + wave * stream_wave_lds(ROWS, RT, BT, UQ, XQ);
  unsigned char* mine_x = mine + UQ * RT * ROWS * 256;
  // row 4 j + lane / 16 of a tile, chunk (lane % 16) ^ row
  uint32_t at[kLoads], x_at[BT][kX];
#pragma unroll
  for (int j = 0; j < kLoads; ++j) at[j] = (uint32_t)(4 * j + g) * (2u * K) + 16u * (r ^ (4 * j + g));
  if (kStaged)
#pragma unroll
    for (int t = 0; t < BT; ++t)
#pragma unroll
      for (int j = 0; j < kX; ++j) x_at[t][j] = (uint32_t)min(16 * t + 4 * j + g, nb - 1) * (2u * K) + 16u * (r ^ (4 * j + g));
  const unsigned char* base = reinterpret_cast<const unsigned char*>(w);
  const unsigned char* x_base = reinterpret_cast<const unsigned char*>(xrows);
  const size_t tile = (size_t)ROWS * 2 * K;
  u32x4_t wr[2][UQ][RT][kLoads], xr[2][UQ][BT][kX];
  auto load_w = [&](int buf, int q) {
#pragma unroll
    for (int i = 0; i < UQ; ++i)
#pragma unroll
      for (int n = 0; n < RT; ++n)
#pragma unroll
        for (int j = 0; j < kLoads; ++j)
          wr[buf][i][n][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(base + n * tile + (size_t)(q + i) * 256 + at[j]));
  };
  auto load_x = [&](int buf, int q) {
#pragma unroll
    for (int i = 0; i < UQ; ++i)
#pragma unroll
      for (int t = 0; t < BT; ++t)
#pragma unroll
        for (int s = 0; s < kX; ++s) {
          if (kStaged) xr[buf][i][t][s] = *reinterpret_cast<const u32x4_t*>(x_base + (size_t)(q + i) * 256 + x_at[t][s]);
          else xr[buf][i][t][s] = x(t, kStreamBlock * (q + i) + 32 * s);
        }
  };
  auto put = [&](int i, int n, int j, const u32x4_t& v) {
    *reinterpret_cast<u32x4_t*>(mine + ((i * RT + n) * kLoads + j) * 1024 + lane * 16) = v;
  };
  auto put_x = [&](int i, int t, int j, const u32x4_t& v) { *reinterpret_cast<u32x4_t*>(mine_x + ((i * BT + t) * kX + j) * 1024 + lane * 16) = v; };
  auto operand = [&](int i, int n, int s) {
    return *reinterpret_cast<const u32x4_t*>(mine + (i * RT + n) * kLoads * 1024 + rr * 256 + ((4 * s + g) ^ rr) * 16);
  };
  const int rx = r & (4 * kX - 1);
  auto operand_x = [&](int i, int t, int s) {
    return *reinterpret_cast<const u32x4_t*>(mine_x + (i * BT + t) * kX * 1024 + rx * 256 + ((4 * s + g) ^ rx) * 16);
  };
  auto use = [&](int buf) {
#pragma unroll
    for (int i = 0; i < UQ; ++i) {
      if (kStaged)
#pragma unroll
        for (int t = 0; t < BT; ++t)
#pragma unroll
          for (int j = 0; j < kX; ++j) put_x(i, t, j, xr[buf][i][t][j]);
#pragma unroll
      for (int n = 0; n < RT; ++n)
#pragma unroll
        for (int j = 0; j < kLoads; ++j) put(i, n, j, wr[buf][i][n][j]);
    }
    wave_lds_order();
#pragma unroll
    for (int i = 0; i < UQ; ++i)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        u32x4_t v[BT];
#pragma unroll
        for (int t = 0; t < BT; ++t) v[t] = kStaged ? operand_x(i, t, s) : xr[buf][i][t][s & (kX - 1)];
#pragma unroll
        for (int n = 0; n < RT; ++n) {
          const u32x4_t f = operand(i, n, s);
#pragma unroll
          for (int t = 0; t < BT; ++t) acc[n][t] = mfma16(f, v[t], acc[n][t]);
        }
      }
    wave_lds_order();  // (the next block's puts overwrite what was read here)
  };
  auto load = [&](int buf, int q) {
    if (kStaged) load_x(buf, q);
    load_w(buf, q);
    if (!kStaged) load_x(buf, q);
  };
  if (count >= UQ) {
    if (kAhead) load(0, begin);
    else load_w(0, begin);
  }
  between();
  int s = begin, left = count;
  if (left >= UQ) {
    if (!kAhead) load_x(0, s);
    for (; left >= 3 * UQ; left -= 2 * UQ, s += 2 * UQ) {
      load(1, s + UQ);
      __builtin_amdgcn_sched_barrier(0);
      use(0);
      load(0, s + 2 * UQ);
      __builtin_amdgcn_sched_barrier(0);
      use(1);
    }
    if (left >= 2 * UQ) {
      load(1, s + UQ);
      __builtin_amdgcn_sched_barrier(0);
      use(0);
      use(1);
      left -= 2 * UQ;
      s += 2 * UQ;
    } else {
      use(0);
      left -= UQ;
      s += UQ;
    }
  }
  // A block at a time: what UQ leaves over, and (in the last wave) the columns of a block that K cuts short, zero past it.  All that a
  // block needs is requested at once, at columns held inside K, and cleared behind its arrival: with the loads inside the
  // conditions each was a round trip of its own (K = 1000, 4096 columns, 48 sequences: 13.1 us a launch, 7.0 now).
  const bool cut = wave == kWaves - 1 && K % kStreamBlock != 0;
  for (; left > 0 || (left == 0 && cut); --left) {
    const int q = left == 0 ? full : s++;
    u32x4_t wt[RT][kLoads], xt[BT][kX];
    auto inside = [&](int j) {  // this lane's column of row 4 j + g, held inside K: what to add to the row's offset
      const int c = 8 * (r ^ (4 * j + g));  // (of which at[j] holds 2 c already)
      return 2u * (uint32_t)(min(kStreamBlock * q + c, K - 8) - c);
    };
    auto live = [&](int j) { return kStreamBlock * q + 8 * (r ^ (4 * j + g)) < K; };
#pragma unroll
    for (int t = 0; t < BT; ++t)
#pragma unroll
      for (int k = 0; k < kX; ++k)
        xt[t][k] = kStaged ? *reinterpret_cast<const u32x4_t*>(x_base + (x_at[t][k] + inside(k))) : x(t, min(kStreamBlock * q + 32 * k, K - 8 - 8 * g));
#pragma unroll
    for (int n = 0; n < RT; ++n)
#pragma unroll
      for (int j = 0; j < kLoads; ++j)
        wt[n][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(base + n * tile + (at[j] + inside(j))));
    const u32x4_t zero = {0u, 0u, 0u, 0u};
    if (kStaged)
#pragma unroll
      for (int t = 0; t < BT; ++t)
#pragma unroll
        for (int j = 0; j < kX; ++j) {
          asm volatile("" : "+v"(xt[t][j]));
          put_x(0, t, j, live(j) ? xt[t][j] : zero);
        }
#pragma unroll
    for (int n = 0; n < RT; ++n)
#pragma unroll
      for (int j = 0; j < kLoads; ++j) {
        asm volatile("" : "+v"(wt[n][j]));
        put(0, n, j, live(j) ? wt[n][j] : zero);
      }
    wave_lds_order();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      u32x4_t v[BT];
#pragma unroll
      for (int t = 0; t < BT; ++t) {
        if (kStaged) {
          v[t] = operand_x(0, t, k);
        } else {
          asm volatile("" : "+v"(xt[t][k & (kX - 1)]));
          v[t] = kStreamBlock * q + 32 * k + 8 * g < K ? xt[t][k & (kX - 1)] : zero;
        }
      }
#pragma unroll
      for (int n = 0; n < RT; ++n) {
        const u32x4_t f = operand(0, n, k);
#pragma unroll
        for (int t = 0; t < BT; ++t) acc[n][t] = mfma16(f, v[t], acc[n][t]);
      }
    }
    wave_lds_order();
  }
  __syncthreads();
  meet<kWaves, RT, BT>(acc, reinterpret_cast<float*>(lds), wave, lane);
}

struct DenseIn {
  const float* x;           // [B, Dp] residual rows (norm prologue)
  const uint16_t* n1;       // or [B, Dp] bf16 rows already normed by gain 1 / gain 2
  const uint16_t* n2;
  const float* gain1;
  const float* gain2;
  const uint16_t* w1;       // [16 tiles1, Dp]
  const uint16_t* w2;       // [16 tiles2, Dp]; pairs: gate / up rows interleaved in blocks of 8
  float* y1;                // [B, 16 tiles1]
  uint16_t* gated;          // [B, gated_ld], column 8 * tile + j (pairs) or 16 * tile + j
  int batch, D, Dp, tiles1, tiles2, gated_ld, act, center, pairs;
  float eps;
  const float* sums;        // or null: n1 / n2 are rows times gain, not normed yet; [B, parts] holds their rows' sums of squares in parts,
  int parts;                // and the norm's factor goes to the outputs
};

// kNorm: the norm is formed here, for the rows of one batch block (dynamic LDS: rows x (Dp + 8) bf16).
// RT: row tiles per workgroup (grid.x counts workgroups of the first matrix, then of the second), BT: batch tiles; XQ, UQ as in stream_rows.
template <int kWaves, bool kNorm, int RT, int BT, int XQ, int UQ>
__global__ __launch_bounds__(64 * kWaves) void dense_in_kernel(DenseIn a) {
  extern __shared__ __attribute__((aligned(16))) uint16_t normed[];
  __shared__ __attribute__((aligned(16))) unsigned char lds[stream_lds(kWaves, 16, RT, BT, UQ, XQ)];
  __shared__ float stat[kNorm ? kWaves : kGemvBatch * BT];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int b0 = blockIdx.y * kGemvBatch * BT, nb = min(kGemvBatch * BT, a.batch - b0);
  const int groups1 = (a.tiles1 + RT - 1) / RT;
  const bool second = (int)blockIdx.x >= groups1;
  const int tiles = second ? a.tiles2 : a.tiles1;
  // the last workgroup of an odd matrix overlaps its neighbour: the same rows give the same values twice
  const int tile0 = max(0, min(RT * (second ? (int)blockIdx.x - groups1 : (int)blockIdx.x), tiles - RT));
  const uint16_t* wrow = (second ? a.w2 : a.w1) + (size_t)(16 * tile0) * a.Dp;
  f32x4_t acc[RT][BT] = {};
  if constexpr (kNorm) {
    const float* gain = second ? a.gain2 : a.gain1;
    constexpr int kThreads = 64 * kWaves, kKeep = 4;
    const int stride = a.Dp + 8;
    auto block_sum = [&](float v) {
      v = wave_sum(v);
      __syncthreads();
      if (lane == 0) stat[wave] = v;
      __syncthreads();
      float s = stat[0];
#pragma unroll
      for (int w = 1; w < kWaves; ++w) s += stat[w];
      return s;
    };
    auto norm = [&]() {
      for (int b = 0; b < nb; ++b) {
        const float* x = a.x + (size_t)(b0 + b) * a.Dp;
        float4 keep[kKeep];
        float sum = 0.f;
  #pragma unroll
        for (int j = 0; j < kKeep; ++j) {
          const int i = 4 * (threadIdx.x + kThreads * j);
          keep[j] = i < a.Dp ? load4(x + i) : float4{0.f, 0.f, 0.f, 0.f};
          sum += (keep[j].x + keep[j].y) + (keep[j].z + keep[j].w);
        }
        for (int i = 4 * (threadIdx.x + kThreads * kKeep); i < a.Dp; i += 4 * kThreads) {
          const float4 v = load4(x + i);
          sum += (v.x + v.y) + (v.z + v.w);
        }
        const float mean = a.center ? block_sum(sum) / (float)a.D : 0.f;
        float ss = 0.f;
        auto square = [&](int i, const float4& v) {
          const float p = v.x - mean, q = v.y - mean, s = v.z - mean, t = v.w - mean;
          if (i + 3 < a.D) {
            ss += (p * p + q * q) + (s * s + t * t);
          } else {
            if (i < a.D) ss += p * p;
            if (i + 1 < a.D) ss += q * q;
            if (i + 2 < a.D) ss += s * s;
          }
        };
  #pragma unroll
        for (int j = 0; j < kKeep; ++j) square(4 * (threadIdx.x + kThreads * j), keep[j]);
        for (int i = 4 * (threadIdx.x + kThreads * kKeep); i < a.Dp; i += 4 * kThreads) square(i, load4(x + i));
        const Divisor by(sqrtf(block_sum(ss) / (float)a.D + a.eps));
        auto put = [&](int i, const float4& v) {
          const float4 w = load4(gain + i);
          store4(normed + b * stride + i, float4{by.divide(v.x - mean) * w.x, by.divide(v.y - mean) * w.y,
                                                 by.divide(v.z - mean) * w.z, by.divide(v.w - mean) * w.w});
        };
  #pragma unroll
        for (int j = 0; j < kKeep; ++j) {
          const int i = 4 * (threadIdx.x + kThreads * j);
          if (i < a.Dp) put(i, keep[j]);
        }
        for (int i = 4 * (threadIdx.x + kThreads * kKeep); i < a.Dp; i += 4 * kThreads) put(i, load4(x + i));
      }
      __syncthreads();
    };
    static_assert(XQ == kStreamFrom, "formed rows lie in LDS");
    stream_rows<kWaves, 16, RT, BT, UQ, XQ>(wrow, a.Dp, wave, lane, lds, acc, nullptr, nb, norm, [&](int t, int k) {
      return *reinterpret_cast<const u32x4_t*>(normed + min(16 * t + r, nb - 1) * stride + 8 * g + k);
    });
  } else {
    const uint16_t *xr = (second ? a.n2 : a.n1) + (size_t)b0 * a.Dp, *xd = xr + 8 * g;
    // the rows' factors while the first weights travel: 16 lanes per row add its parts
    auto factors = [&]() {
      if (!a.sums) return;
      for (int row = threadIdx.x >> 4; row < nb; row += 4 * kWaves) {
        const float* part = a.sums + (size_t)(b0 + row) * a.parts;
        float ss = 0.f;
        constexpr int kTogether = 16;
        for (int i0 = r; i0 < a.parts; i0 += 16 * kTogether) {
          float p[kTogether];
#pragma unroll
          for (int k = 0; k < kTogether; ++k) p[k] = part[min(i0 + 16 * k, a.parts - 1)];
#pragma unroll
          for (int k = 0; k < kTogether; ++k) ss += i0 + 16 * k < a.parts ? p[k] : 0.f;
        }
        ss = team_sum16(ss);
        if (r == 0) stat[row] = 1.0f / sqrtf(ss / (float)a.D + a.eps);
      }
    };
    stream_rows<kWaves, 16, RT, BT, UQ, XQ>(wrow, a.Dp, wave, lane, lds, acc, xr, nb, factors, [&](int t, int k) {
      return *reinterpret_cast<const u32x4_t*>(xd + (size_t)min(16 * t + r, nb - 1) * a.Dp + k);
    });
  }
#pragma unroll
  for (int i = 0; i < RT * BT; ++i) {
    if (wave != i) continue;
    f32x4_t sum = acc[i / BT][i % BT];
    const int row = 16 * (i % BT) + r, tile = tile0 + i / BT;
    if (!kNorm && a.sums) sum *= stat[min(row, nb - 1)];
    if (!second) {
      if (row < nb) store4(a.y1 + (size_t)(b0 + row) * (16 * a.tiles1) + 16 * tile + 4 * g, float4{sum[0], sum[1], sum[2], sum[3]});
      continue;
    }
    if (!a.pairs) {
      if (row < nb)
        store4(a.gated + (size_t)(b0 + row) * a.gated_ld + 16 * tile + 4 * g,
               float4{activate(a.act, sum[0]), activate(a.act, sum[1]), activate(a.act, sum[2]), activate(a.act, sum[3])});
      continue;
    }
    // rows 0 .. 7 of the tile (lanes g < 2) are gates, rows 8 .. 15 (lanes g >= 2, 32 lanes on) the matching up rows
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = activate(a.act, sum[e]) * __shfl_xor(sum[e], 32);
    if (g < 2 && row < nb) store4(a.gated + (size_t)(b0 + row) * a.gated_ld + 8 * tile + 4 * g, float4{v[0], v[1], v[2], v[3]});
  }
}

struct DenseOut {
  const uint16_t* in;       // [B, K]
  const uint16_t* w;        // [Dp, K]
  float* x;                 // [B, Dp], updated in place
  const float* again;       // [B, Dp] or null, added too
  const float* step;        // [Dp] or null, added too
  int batch, K, Dp;
};
// ROWS, kWaves: tiles of 16 rows on four waves, or of 8 on eight (few tiles); UQ, XQ as in stream_rows.
template <int kWaves, int ROWS, int RT, int BT, int UQ, int XQ>
__global__ __launch_bounds__(64 * kWaves) void dense_out_kernel(DenseOut a) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[stream_lds(kWaves, ROWS, RT, BT, UQ, XQ)];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int b0 = blockIdx.y * kGemvBatch * BT, nb = min(kGemvBatch * BT, a.batch - b0);
  const int first = blockIdx.x * RT * ROWS;  // (RT divides the row tiles: x is updated in place)
  const uint16_t *xr = a.in + (size_t)b0 * a.K, *xd = xr + 8 * g;
  // what the product of tile wave = (row tile, batch tile) is added to, requested ahead of it by the wave that will write it
  const bool writes = wave < RT * BT && 4 * g < ROWS;
  const int row = 16 * (wave % BT) + r, column = first + ROWS * (wave / BT) + 4 * g;
  const size_t place = (size_t)(b0 + min(row, nb - 1)) * a.Dp + column;
  // (and added behind it: an addition here would have that wave wait before it asks for its first weights)
  float4 v = float4{0.f, 0.f, 0.f, 0.f}, again = v, step = v;
  if (writes) v = load4(a.x + place);
  if (writes && a.again) again = load4(a.again + place);
  if (writes && a.step) step = load4(a.step + column);
  f32x4_t acc[RT][BT] = {};
  stream_rows<kWaves, ROWS, RT, BT, UQ, XQ>(a.w + (size_t)first * a.K, a.K, wave, lane, lds, acc, xr, nb, [] {}, [&](int t, int k) {
    return *reinterpret_cast<const u32x4_t*>(xd + (size_t)min(16 * t + r, nb - 1) * a.K + k);
  });
  if (a.again) { v.x += again.x; v.y += again.y; v.z += again.z; v.w += again.w; }
  if (a.step) { v.x += step.x; v.y += step.y; v.z += step.z; v.w += step.w; }
#pragma unroll
  for (int i = 0; i < RT * BT; ++i) {
    const f32x4_t& sum = acc[i / BT][i % BT];
    if (wave == i && writes && row < nb) store4(a.x + place, float4{v.x + sum[0], v.y + sum[1], v.z + sum[2], v.w + sum[3]});
  }
}

struct DenseOutStreams {
  const uint16_t* in;       // [B, K]
  const uint16_t* w;        // [Dp, K]
  float* x;                 // [B, S, Dp], updated in place
  const float* scale;       // [Dp], a factor per column of the product
  const float* out;         // [S]
  const float* mix;         // [S, S]
  const float* next;        // [S], weights of the next reader; null: the plain sum
  float* u;                 // [B, Dp], what the next reader gets, or null and
  const float* gain;        // [Dp] its norm's gain,
  uint16_t* scaled;         // [B, Dp] bf16, what it gets times the gain,
  float* sums;              // [B, Dp / ROWS] its sums of squares per tile
  int batch, K, Dp, streams;
};
template <int kWaves, int ROWS, int RT, int BT, int UQ, int XQ, int MAXS>
__global__ __launch_bounds__(64 * kWaves) void dense_out_streams_kernel(DenseOutStreams a) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[stream_lds(kWaves, ROWS, RT, BT, UQ, XQ)];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int b0 = blockIdx.y * kGemvBatch * BT, nb = min(kGemvBatch * BT, a.batch - b0);
  const int first = blockIdx.x * RT * ROWS;
  const uint16_t *xr = a.in + (size_t)b0 * a.K, *xd = xr + 8 * g;
  // the streams at this lane's place of tile wave = (row tile, batch tile), requested ahead of the product
  const bool writes = wave < RT * BT && 4 * g < ROWS;
  const int row = 16 * (wave % BT) + r, column = first + ROWS * (wave / BT) + 4 * g;
  float* x = a.x + (size_t)(b0 + min(row, nb - 1)) * a.streams * a.Dp + column;
  float4 v[MAXS];
#pragma unroll
  for (int s = 0; s < MAXS; ++s)
    if (writes && s < a.streams) v[s] = load4(x + (size_t)s * a.Dp);
  // and the column's factors and, for few streams, the coefficients: fetched where the epilogue uses them they were five round trips
  // to memory, one after the other, at the end of every launch (4 sequences, K = 8192, 2048 columns, two streams: 7.9 us, 7.2 now)
  constexpr bool kHold = MAXS <= 4;
  constexpr int kC = kHold ? MAXS : 1;
  float4 f = float4{0.f, 0.f, 0.f, 0.f}, k = f;
  float c_out[kC], c_next[kC], c_mix[kC * kC];
  if (writes) f = load4(a.scale + column);
  if (writes && !a.u) k = load4(a.gain + column);
  if constexpr (kHold) {
#pragma unroll
    for (int t = 0; t < kC; ++t) {
      const int to = min(t, a.streams - 1);
      c_out[t] = a.out[to];
      c_next[t] = a.next ? a.next[to] : 1.f;
#pragma unroll
      for (int s = 0; s < kC; ++s) c_mix[s * kC + t] = a.mix[min(s, a.streams - 1) * a.streams + to];
    }
  }
  f32x4_t acc[RT][BT] = {};
  stream_rows<kWaves, ROWS, RT, BT, UQ, XQ>(a.w + (size_t)first * a.K, a.K, wave, lane, lds, acc, xr, nb, [] {}, [&](int t, int k) {
    return *reinterpret_cast<const u32x4_t*>(xd + (size_t)min(16 * t + r, nb - 1) * a.K + k);
  });
#pragma unroll
  for (int i = 0; i < RT * BT; ++i) {
    if (wave != i || !writes || row >= nb) continue;
    const f32x4_t& sum = acc[i / BT][i % BT];
    const float4 y = float4{sum[0] * f.x, sum[1] * f.y, sum[2] * f.z, sum[3] * f.w};
    if constexpr (kHold) mix_streams_by<MAXS>(v, a.streams, [&](int t) { return c_out[t]; }, [&](int s, int t) { return c_mix[s * kC + t]; }, y);
    else mix_streams<MAXS>(v, a.streams, a.out, a.mix, y);
#pragma unroll
    for (int s = 0; s < MAXS; ++s)
      if (s < a.streams) store4(x + (size_t)s * a.Dp, v[s]);
    float4 read;
    if constexpr (kHold) read = read_streams_by<MAXS>(v, a.streams, [&](int s) { return c_next[s]; });
    else read = read_streams<MAXS>(v, a.streams, a.next);
    if (a.u) {
      store4(a.u + (size_t)(b0 + row) * a.Dp + column, read);
      continue;
    }
    store4(a.scaled + (size_t)(b0 + row) * a.Dp + column, float4{read.x * k.x, read.y * k.y, read.z * k.z, read.w * k.w});
    // (the lanes of a row are 16 apart, and all of them here)
    float ss = (read.x * read.x + read.y * read.y) + (read.z * read.z + read.w * read.w);
    ss += __shfl_xor(ss, 16);
    if (ROWS == 16) ss += __shfl_xor(ss, 32);
    if (g == 0) a.sums[(size_t)(b0 + row) * (a.Dp / ROWS) + column / ROWS] = ss;
  }
}

struct LatentAbsorb {
  const float* y;           // [B, ldy] projection rows (see latent_split_kernel)
  const uint16_t* ukt;      // [H, rankp, dimp] transposed key expansion
  const float* latent_gain; // [rankp]
  const float* cosine;      // [table_rows, rot / 2]
  const float* sine;
  const long long* pos;
  uint16_t* q;              // [B, H, rankp + rotp]
  uint16_t* ring;           // [B, cap, rankp + rotp]
  int batch, ldy, table_rows, cap, groups;  // groups: workgroups per head (4 tiles of 16 latent columns each)
  LatentShape s;
};
// Grid (H * groups + 4 + H, batch blocks).  Behind the products' workgroups four make the cache rows, a wave each, and one per head
// rotates the rotated part of its queries: those hang on the position and then on its angles, two round trips more than a
// product takes.  A cache row's operands are requested at once (8 sequences, 32 heads, 512 + 64 columns: 4.9 us a launch, 5.5 with the
// rotations ahead of the first product of a head and a wait per 256 columns of a row).
__global__ __launch_bounds__(256) void latent_absorb_kernel(LatentAbsorb a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int b0 = blockIdx.y * kGemvBatch, nb = min(kGemvBatch, a.batch - b0);
  const LatentShape s = a.s;
  const int dq = s.dimp + s.rotp, width = s.rankp + s.rotp;
  const int p = clamped_position(a.pos, 0, a.table_rows);
  const float* cs = a.cosine + (size_t)p * (s.rot >> 1);
  const float* sn = a.sine + (size_t)p * (s.rot >> 1);
  const int extra = (int)blockIdx.x - s.heads * a.groups;
  if (extra >= 4) {
    const int head = extra - 4;
    for (int i = threadIdx.x; i < nb * s.rotp; i += 256) {
      const int b = b0 + i / s.rotp, d = i % s.rotp;
      a.q[((size_t)b * s.heads + head) * width + s.rankp + d] =
          f32_to_bf16_rne(rotated(a.y + (size_t)b * a.ldy + head * dq + s.dimp, d, s.rot, cs, sn));
    }
    return;
  }
  if (extra >= 0) {
    const int b = 4 * extra + wave;
    if (b < nb) {
      const float* lat = a.y + (size_t)(b0 + b) * a.ldy + s.heads * dq;
      uint16_t* dst = a.ring + ((size_t)(b0 + b) * a.cap + p % a.cap) * width;
      constexpr int kKeep = 2;  // the first 512 columns stay in registers
      float4 v[kKeep], w[kKeep];
#pragma unroll
      for (int j = 0; j < kKeep; ++j) {
        const int i = min(4 * lane + 256 * j, s.rankp - 4);
        v[j] = load4(lat + i);
        w[j] = load4(a.latent_gain + i);
      }
      for (int i = lane; i < s.rotp; i += 64) dst[s.rankp + i] = f32_to_bf16_rne(rotated(lat + s.rankp, i, s.rot, cs, sn));
      float ss = 0.f;
      auto square = [&](const float4& u) { ss += (u.x * u.x + u.y * u.y) + (u.z * u.z + u.w * u.w); };  // padding columns are zero
#pragma unroll
      for (int j = 0; j < kKeep; ++j)
        if (4 * lane + 256 * j < s.rankp) square(v[j]);
      for (int i = 4 * lane + 256 * kKeep; i < s.rankp; i += 256) square(load4(lat + i));
      const Divisor by(sqrtf(wave_sum(ss) / (float)s.rank + s.eps));
      auto put = [&](int i, const float4& u, const float4& k) {
        store4(dst + i, float4{by.divide(u.x) * k.x, by.divide(u.y) * k.y, by.divide(u.z) * k.z, by.divide(u.w) * k.w});
      };
#pragma unroll
      for (int j = 0; j < kKeep; ++j)
        if (4 * lane + 256 * j < s.rankp) put(4 * lane + 256 * j, v[j], w[j]);
      for (int i = 4 * lane + 256 * kKeep; i < s.rankp; i += 256) put(i, load4(lat + i), load4(a.latent_gain + i));
    }
    return;
  }
  const int h = blockIdx.x / a.groups, grp = blockIdx.x % a.groups;
  const int tile = 4 * grp + wave;
  if (16 * tile >= s.rankp) return;
  const uint16_t* wrow = a.ukt + ((size_t)h * s.rankp + 16 * tile + r) * s.dimp;
  const float* xr = a.y + (size_t)(b0 + min(r, nb - 1)) * a.ldy + h * dq;  // (columns past the batch repeat the last one, and are not stored)
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  // (as many steps together as a head has, at most four: repeated ones cost their loads, 5.6 us instead of 3.5 at 48 sequences, 20
  // heads of 32 columns, latents of 512)
  auto steps = [&](auto together, int k0) {
    constexpr int kSteps = decltype(together)::value;
    u32x4_t w[kSteps];
    float4 u[kSteps], v[kSteps];
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
      const int k = min(k0 + 32 * i, s.dimp - 8);
      w[i] = *reinterpret_cast<const u32x4_t*>(wrow + k);
      u[i] = load4(xr + k);
      v[i] = load4(xr + k + 4);
    }
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
      const u32x4_t none = {0u, 0u, 0u, 0u};
      const u32x4_t x = {pack2_bf16(u[i].x, u[i].y), pack2_bf16(u[i].z, u[i].w), pack2_bf16(v[i].x, v[i].y), pack2_bf16(v[i].z, v[i].w)};
      const bool live = k0 + 32 * i < s.dimp;
      acc = mfma16(live ? w[i] : none, live ? x : none, acc);
    }
  };
  if (s.dimp <= 32) {
    steps(std::integral_constant<int, 1>{}, 8 * g);
  } else if (s.dimp <= 64) {
    steps(std::integral_constant<int, 2>{}, 8 * g);
  } else {
    for (int k0 = 8 * g; k0 < s.dimp + 8 * g; k0 += 128) steps(std::integral_constant<int, 4>{}, k0);
  }
  if (r < nb)
    store4(a.q + ((size_t)(b0 + r) * s.heads + h) * width + 16 * tile + 4 * g, float4{acc[0], acc[1], acc[2], acc[3]});
}

// One chunk of cache rows against 16 HT heads of one sequence, in the latent space: row j of the ring
// (latent rankp | rotated rotp) is the key, its latent part the value, for every head, so a row is fetched once for all of
// the workgroup's heads and both products.  Four waves per head tile; blocks of 64 rows go into LDS by DMA, one block ahead.
//   S^T = K Q^T:    wave w takes keys 16 (w & 3) .. of the block; KS column steps, its head tile's queries in registers
//   U^T += C^T P^T: wave w takes every fourth 16-column tile of the latent (RT of them), latents by transposing LDS reads
// LDS holds the rows in panels of 128 bytes (64 rows x 8 chunks): chunk c of row k in slot c ^ (k & 6 | k >> 3 & 1), so that
// sixteen rows of one chunk and eight rows of one 32-byte segment (whose two chunks stay neighbours) meet every bank once.
// Partial result of (b, h, chunk): maximum and denominator (base-2 exponents) in `heads_out`, and rankp sums in `sums`, which
// holds [b][head tile][chunk][16-column tile][16 heads][16 columns] so that a wave stores whole lines; zeros for an empty chunk.
// Grid: chunks of sequences x head groups; the groups of a chunk are 8 workgroups apart, on one XCD and its L2.
struct LatentDecode {
  const uint16_t* q;        // [B, H, width]
  const uint16_t* ring;     // [B, cap, width]
  const long long* pos;
  float* sums;
  float2* heads_out;        // [B, H, S]
  int batch, heads, rankp, width, cap, chunks;
  int key_step;             // 32-column steps ahead of it meet zero query columns and are left out of the scores
  float scale2;
};
__host__ __device__ constexpr long long latent_sums_at(int b, int tile, int chunk, int heads, int chunks, int rankp) {
  return (((long long)b * ((heads + 15) / 16) + tile) * chunks + chunk) * 16 * rankp;
}
constexpr int kLatentRows = 64;
constexpr int kBufferWord3 = 0x00020000;  // last word of a raw buffer descriptor: 32-bit elements, no swizzle
constexpr int kLatentPBytes = (kLatentRows + 8) * 2;
constexpr int latent_decode_lds(int ks, int ht) { return ks * 8192 + ht * 16 * kLatentPBytes; }  // two stages of ks / 2 panels
// Where the queries come from, and which row of the ring the launch itself makes: rows of `q`, and none.
template <int KS>
struct LatentQueries {
  static constexpr bool kMakesRow = false;
  // Requested before the position is known and in one go, through a buffer descriptor of the sequence's queries: chunks past the
  // width are addressed past its end, which reads as zeros (left out by a branch, each was waited for before the next was
  // requested; cleared by selects, 18 of them cost a microsecond of arithmetic).
  __device__ __forceinline__ void request(const LatentDecode& a, int b, int h0, u32x4_t (&qf)[KS]) {
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, cw = a.width >> 3;
    const uint32_t q_bytes = 2u * (uint32_t)(a.heads * a.width);  // (a launch's queries of one sequence stay far below 2 GiB)
    const __amdgpu_buffer_rsrc_t q_rows =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(a.q) + (size_t)b * a.heads * a.width, 0, (int)q_bytes, kBufferWord3);
    const uint32_t q_at = 2u * (uint32_t)(min(h0 + r, a.heads - 1) * a.width);
#pragma unroll
    for (int s = 0; s < KS; ++s)
      qf[s] = __builtin_amdgcn_raw_buffer_load_b128(q_rows, (int)(4 * s + g < cw ? q_at + 16u * (uint32_t)(4 * s + g) : q_bytes), 0, 0);
  }
  // (the queries are waited for behind the first block's requests and not in the loop, where the wait would be for the block ahead as well)
  template <typename Fetch>
  __device__ __forceinline__ void ready(const LatentDecode&, int, int, int, u32x4_t (&qf)[KS], Fetch&& fetch) {
    fetch();
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[s]));
  }
};
template <int KS, int RT, int HT, typename Front>
__device__ __forceinline__ void latent_decode(const LatentDecode& a, Front& front) {
  constexpr int NP = KS / 2, kPanel = kLatentRows * 128, kStage = NP * kPanel, kWaves = 4 * HT;
  static_assert(KS % 2 == 0, "whole panels");
  extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
  __shared__ float smax[HT][4][16], ssum[HT][4][16];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(pf_lds_char_t*)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int part = wave & 3, ht = wave >> 2;
  const int groups = (a.heads + 16 * HT - 1) / (16 * HT), units = a.batch * a.chunks;
  int unit, group;
  if ((units & 7) == 0) {
    const int m = (int)(blockIdx.x >> 3);
    group = m % groups;
    unit = 8 * (m / groups) + (int)(blockIdx.x & 7);
  } else {
    group = (int)blockIdx.x % groups;
    unit = (int)blockIdx.x / groups;
  }
  const int b = unit / a.chunks, chunk = unit % a.chunks, h0 = 16 * (HT * group + ht);
  const int cw = a.width >> 3;
  u32x4_t qf[KS];
  front.request(a, b, h0, qf);
  const int position = (int)min(max(*a.pos, 0ll), 0x7FFFFFFEll), valid = min(position, a.cap - 1) + 1;  // (rows the ring holds)
  const int per = (((valid + a.chunks - 1) / a.chunks) + kLatentRows - 1) & ~(kLatentRows - 1);
  const int begin = chunk * per, end = min(valid, begin + per);
  float m = -INFINITY, l = 0.f;
  f32x4_t u[RT] = {};
  if (begin < end) {
    const char* ring = reinterpret_cast<const char*>(a.ring + (size_t)b * a.cap * a.width);
    // a request fills 8 rows of a panel: this lane row lane / 8, slot lane % 8.  Rows past the end repeat the last one (those
    // keys are masked), chunks past the width the last one (they meet zero query columns).
    const int chunk_of = (lane & 7) ^ (((lane >> 3) & 6) | (wave & 1));  // (a wave's requests all start at rows of one parity of 8)
    auto fetch = [&](int j0) {
      const uint32_t to = lds0 + (uint32_t)((((j0 - begin) / kLatentRows) & 1) * kStage);
#pragma unroll
      for (int i = 0; i < (8 * NP + kWaves - 1) / kWaves; ++i) {
        const int req = wave + kWaves * i;  // panel req / 8, rows 8 (req % 8) ..
        if ((8 * NP) % kWaves != 0 && req >= 8 * NP) continue;
        const uint32_t row = (uint32_t)min(j0 + 8 * (req & 7) + (lane >> 3), end - 1);
        const uint32_t c = (uint32_t)min(8 * (req >> 3) + chunk_of, cw - 1);
        dma16_gather(ring + (size_t)row * (uint32_t)(2 * a.width) + 16u * c, to + (uint32_t)(req * 1024));
      }
    };
    front.ready(a, position, begin, end, qf, [&]() __attribute__((always_inline)) { fetch(begin); });
    // keys: row 16 part + r, chunk 4 (s & 1) + g of panel s / 2
    const uint32_t k_rd[2] = {lds0 + (uint32_t)((16 * part + r) * 128 + 16 * (g ^ (r & 6 | r >> 3))),
                              lds0 + (uint32_t)((16 * part + r) * 128 + 16 * ((4 + g) ^ (r & 6 | r >> 3)))};
    // latents: this lane addresses 8 bytes (piece r & 3) of row 4 g + (r >> 2); tile part + 4 t is segment part of panel t
    const int vrow = 4 * g + (r >> 2);
    const uint32_t v_rd = lds0 + (uint32_t)(vrow * 128 + 16 * ((2 * part | (r & 3) >> 1) ^ (vrow & 6 | vrow >> 3)) + 8 * (r & 1));
    unsigned char* p_lds = lds + 2 * kStage + ht * 16 * kLatentPBytes + r * kLatentPBytes;
    for (int j0 = begin; j0 < end; j0 += kLatentRows) {
      // this block has landed; every wave is done with the one before, whose stage the next block goes to
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if constexpr (Front::kMakesRow) front.place(a, lds, (((j0 - begin) / kLatentRows) & 1) * kStage, j0, end);
      if (j0 + kLatentRows < end) fetch(j0 + kLatentRows);
      const uint32_t stage = (uint32_t)((((j0 - begin) / kLatentRows) & 1) * kStage);
      f32x4_t sc[2] = {};
      auto fragment = [&](int s) { return pf_read128(k_rd[s & 1] + stage + (uint32_t)((s >> 1) * kPanel)); };
      // the usual two starts: fragments are read kBatch at a time, ahead of the products of the ones before (left to the compiler,
      // and more so with a branch per step, each read waits for the product before it)
      auto scores_from = [&](auto from) {
        constexpr int kFrom = decltype(from)::value, kBatch = 4;
        u32x4_t ka[2][kBatch];
        auto read = [&](int s0) {
#pragma unroll
          for (int i = 0; i < kBatch; ++i)
            if (s0 + i < KS) ka[((s0 - kFrom) / kBatch) & 1][i] = fragment(s0 + i);
        };
        read(kFrom);
#pragma unroll
        for (int s0 = kFrom; s0 < KS; s0 += kBatch) {
          if (s0 + kBatch < KS) read(s0 + kBatch);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int i = 0; i < kBatch; ++i)
            if (s0 + i < KS) sc[(s0 + i) & 1] = mfma16(ka[((s0 - kFrom) / kBatch) & 1][i], qf[s0 + i], sc[(s0 + i) & 1]);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (a.key_step == 0) {
        scores_from(std::integral_constant<int, 0>{});
      } else if (a.key_step == KS / 2) {
        scores_from(std::integral_constant<int, KS / 2>{});
      } else {
#pragma unroll
        for (int s = 0; s < KS; ++s)
          if (s >= a.key_step) sc[s & 1] = mfma16(fragment(s), qf[s], sc[s & 1]);
      }
      // score i: key j0 + 16 part + 4 g + i, head h0 + r
      float p[4], mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = j0 + 16 * part + 4 * g + i < end ? (sc[0][i] + sc[1][i]) * a.scale2 : -INFINITY;
        mx = fmaxf(mx, p[i]);
      }
      mx = quad_max(mx);
      if (g == 0) smax[ht][part][r] = mx;
      __syncthreads();
      // (finite: the block's first row is valid)
      const float m_new = fmaxf(fmaxf(fmaxf(smax[ht][0][r], smax[ht][1][r]), fmaxf(smax[ht][2][r], smax[ht][3][r])), m);
      const float corr = __builtin_amdgcn_exp2f(m - m_new);
      m = m_new;
#pragma unroll
      for (int i = 0; i < 4; ++i) p[i] = __builtin_amdgcn_exp2f(p[i] - m);
      l = l * corr + ((p[0] + p[1]) + (p[2] + p[3]));
      store4(reinterpret_cast<uint16_t*>(p_lds) + 16 * part + 4 * g, float4{p[0], p[1], p[2], p[3]});
#pragma unroll
      for (int t = 0; t < RT; ++t) u[t] *= corr;
      __syncthreads();
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const unsigned char* pr = p_lds + 2 * (32 * hf + 4 * g);
        const u32x2_t plo = *reinterpret_cast<const u32x2_t*>(pr), phi = *reinterpret_cast<const u32x2_t*>(pr + 32);
        const u32x4_t pf = {plo.x, plo.y, phi.x, phi.y};
        const uint32_t at = v_rd + stage + (uint32_t)(hf * 4096);
        // (panels past the latent hold the rotated part, or nothing of this block: their sums are not written)
        u32x2_t lo[RT], hi[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          lo[t] = pf_read_tr(at + (uint32_t)(t * kPanel));
          hi[t] = pf_read_tr(at + (uint32_t)(t * kPanel + 2048));
        }
#pragma unroll
        for (int t = 0; t < RT; ++t) u[t] = mfma16(u32x4_t{lo[t].x, lo[t].y, hi[t].x, hi[t].y}, pf, u[t]);
      }
    }
    l = quad_sum(l);
    if (g == 0) ssum[ht][part][r] = l;
    __syncthreads();
    l = (ssum[ht][0][r] + ssum[ht][1][r]) + (ssum[ht][2][r] + ssum[ht][3][r]);
  }
  if (h0 >= a.heads) return;
  if (part == 0 && g == 0 && h0 + r < a.heads) a.heads_out[((size_t)b * a.heads + h0 + r) * a.chunks + chunk] = float2{m, l};
  float* out = a.sums + latent_sums_at(b, h0 >> 4, chunk, a.heads, a.chunks, a.rankp) + 16 * r + 4 * g;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int tile = part + 4 * t;
    if (16 * tile < a.rankp) store4(out + 256 * tile, float4{u[t][0], u[t][1], u[t][2], u[t][3]});
  }
}

template <int KS, int RT, int HT>
__global__ __launch_bounds__(256 * HT) void latent_decode_kernel(LatentDecode a) {
  LatentQueries<KS> front;
  latent_decode<KS, RT, HT>(a, front);
}

struct LatentExpand {
  const float* sums;        // as latent_decode_kernel leaves them
  const float2* heads_in;   // [B, H, S]
  const float* sink;        // [H] or null
  const float* gate;        // gate projections, [b * gate_ld + h], or null
  const uint16_t* uv;       // [H, vdimp, rankp]
  uint16_t* out;            // [B, out_ld], head h at column h * vdimp
  int batch, heads, chunks, rankp, vdimp, gate_ld, out_ld, groups;  // groups: workgroups per head
};
constexpr int kLatentMaxChunks = 32, kExpandRank = 512;
// A workgroup of 8 waves per (head, TW 16-column tiles of values, EB sequences): the chunks are merged by all threads, then
// 8 / TW waves per tile expand the merged latents, a part of them each; their weights are requested first.  One CU takes in
// some 40 KB per microsecond, and that is what bounds a launch: a head's weights (128 KB at 512 x 128) divided by the tiles, a
// sequence's chunks (2 KB each) times EB, which every workgroup of a head repeats.  Grid (H * groups, batch blocks).
template <int TW, int EB>
__global__ __launch_bounds__(512) void latent_expand_kernel(LatentExpand a) {
  constexpr int kParts = 8 / TW, kSteps = kExpandRank / 32 / kParts;
  extern __shared__ __attribute__((aligned(16))) uint16_t merged[];   // [EB][rankp + 8] bf16
  __shared__ float weight[EB][kLatentMaxChunks];
  __shared__ float4 part[512];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
  const int b0 = blockIdx.y * EB, nb = min(EB, a.batch - b0);
  const int h = blockIdx.x / a.groups, tile = TW * (blockIdx.x % a.groups) + wave / kParts;
  const int ld = a.rankp + 8;
  const u32x4_t zero = {0u, 0u, 0u, 0u};
  const bool active = 16 * tile < a.vdimp;
  const int k0 = 32 * kSteps * (wave % kParts) + 8 * g;
  u32x4_t w[kSteps];
  const uint16_t* wrow = a.uv + ((size_t)h * a.vdimp + (active ? 16 * tile : 0) + r) * a.rankp;
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    w[s] = zero;
    if (active && k0 + 32 * s < a.rankp) w[s] = *reinterpret_cast<const u32x4_t*>(wrow + k0 + 32 * s);
  }
  // merged[b] = sum over chunks; the threads of a column quad split the chunks where there are more threads than quads.
  // The first chunks' sums are requested before the chunks' weights are known.
  const int quads = a.rankp >> 2, items = nb * quads;
  const int split = items <= 128 ? 4 : items <= 256 ? 2 : 1, span = 512 / split;
  const int which = tid / span;
  constexpr int kAhead = 8;
  float4 ahead[kAhead];
  auto request = [&](int i, int s0) {
    const int b = min(i / quads, nb - 1), c = 4 * (i % quads);
    const float* src = a.sums + latent_sums_at(b0 + b, h >> 4, 0, a.heads, a.chunks, a.rankp) + 256 * (c >> 4) + 16 * (h & 15) + (c & 15);
#pragma unroll
    for (int k = 0; k < kAhead; ++k) ahead[k] = load4(src + (size_t)min(s0 + k * split, a.chunks - 1) * (16 * a.rankp));
  };
  request(tid % span, which);
  const float gate = a.gate ? a.gate[(size_t)(b0 + min(r, nb - 1)) * a.gate_ld + h] : 0.f;
  if (wave < nb) {  // a wave per sequence, a lane per chunk
    const bool mine = lane < a.chunks;
    const float2 ml = mine ? a.heads_in[((size_t)(b0 + wave) * a.heads + h) * a.chunks + lane] : float2{-INFINITY, 0.f};
    const float mx = ml.x, sum = ml.y;
    const float sink2 = a.sink ? a.sink[h] * kLog2eF : -INFINITY;
    const float top = fmaxf(wave_max64(mx), sink2);
    const float e = mx == -INFINITY ? 0.f : exp2f(mx - top);
    const float total = wave_sum(sum * e) + (a.sink ? exp2f(sink2 - top) : 0.f);
    if (lane < kLatentMaxChunks) weight[wave][lane] = mine ? e / total : 0.f;
  }
  __syncthreads();
  for (int i0 = 0; i0 < items; i0 += span) {
    const int i = i0 + tid % span, b = min(i / quads, nb - 1);
    float4 sum = float4{0.f, 0.f, 0.f, 0.f};
    for (int s0 = which; s0 < a.chunks; s0 += kAhead * split) {
      if (i0 > 0 || s0 > which) request(i, s0);
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int s = s0 + k * split;
        const float f = s < a.chunks ? weight[b][s] : 0.f;
        const float4 v = ahead[k];
        sum.x = fmaf(v.x, f, sum.x); sum.y = fmaf(v.y, f, sum.y); sum.z = fmaf(v.z, f, sum.z); sum.w = fmaf(v.w, f, sum.w);
      }
    }
    if (split > 1) {  // (one round: items <= span)
      part[tid] = sum;
      __syncthreads();
      for (int o = 1; o < split; ++o) {
        const float4 v = part[(tid + o * span) & 511];
        sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
      }
    }
    if (which == 0 && i < items) store4(merged + b * ld + 4 * (i % quads), sum);
  }
  __syncthreads();
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < kSteps; ++s) {
    u32x4_t v = zero;
    if (r < nb && k0 + 32 * s < a.rankp) v = *reinterpret_cast<const u32x4_t*>(merged + r * ld + k0 + 32 * s);
    acc = mfma16(w[s], v, acc);
  }
  if (kParts > 1) {
    part[tid] = float4{acc[0], acc[1], acc[2], acc[3]};  // (last read before the barrier above)
    __syncthreads();
  }
  if (wave % kParts != 0 || !active) return;
#pragma unroll
  for (int q = 1; q < kParts; ++q) {
    const float4 v = part[tid + 64 * q];
    acc[0] += v.x; acc[1] += v.y; acc[2] += v.z; acc[3] += v.w;
  }
  if (r >= nb) return;
  const float f = a.gate ? sigmoid_f32(gate) : 1.f;
  store4(a.out + (size_t)(b0 + r) * a.out_ld + (size_t)h * a.vdimp + 16 * tile + 4 * g,
         float4{acc[0] * f, acc[1] * f, acc[2] * f, acc[3] * f});
}

}  // namespace ajq
