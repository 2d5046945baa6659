// Dequant matmul of 17 to 64 rows where the activations do not stay resident in registers (skinny_resident_kernels.h: K = 2048 and
// 4096): one block of 16 MB rows x 128 columns, K cut into S parts.
//
// What it is for: dequant_skinny_kernel gives every workgroup of one to four 16-column tiles its own copy of 32 rows of activations,
// which the L2s deliver at 14 TB/s at most, twice as many bytes as int8 weights; rows past 32 read the weights again.
//  * four wavefronts split the columns: each owns two private 16-column tiles, which go from memory straight into its registers and
//    meet every row of the block there; two teams of four take a half of the workgroup's part of K each;
//  * the block's activations are shared: 128 columns of them at a time go through registers into LDS (two slots; chunk c of row r
//    in slot c ^ (r & 15): both the rows' writes and the operand reads meet all banks), one barrier per 128 columns;
//  * everything of the next 128 columns is requested ahead of the arithmetic of these;
//  * the weights are the A operand of v_mfma_f32_16x16x32_bf16, the activations the B operand: a lane ends with four consecutive
//    columns of one row;
//  * int4: products of 128 + q; per group acc += scale (part - (128 + zero) sum(x)), sums of x by a product against ones;
//  * S > 1: the parts' sums go to a workspace in fp32 and gemm_split_reduce_kernel adds them in order (no atomics), 3.5 us with
//    its launch.
// Bound: the trip to memory per 128 columns for few parts, then HBM.  int8 / int4, K = 14336, N = 4096: 37 rows 26.2 -> 18.4 / 20.7
// -> 16.9 us, 64 rows 25.4 -> 20.4; 8192 x 8192, 37 rows 26.8 -> 20.8 / 20.8 -> 17.7.  One team instead of two: the same for int8,
// 2 us more for int4; 256 columns per turn instead of 128: 1 us more (registers); non-temporal weights: 1-2 us more (the partial
// sums leave the caches).
#pragma once
#include "gemm128_kernels.h"

namespace ajq {

constexpr int kMidWaves = 4;   // wavefronts along the columns
constexpr int kMidTeams = 2;   // teams of them, each with a part of K
constexpr int kMidNW = 2;      // private weight tiles per wavefront
constexpr int kMidColumns = kMidWaves * kMidNW * kTileN;
// dynamic LDS: two slots of a group of activations per team; at the end the second team's sums
constexpr int mid_lds_bytes(int mb) { return kMidTeams * 2 * 16 * mb * 256; }

template <bool kW4, int MB>
__global__ __launch_bounds__(64 * kMidWaves * kMidTeams) void dequant_gemm_mid_kernel(
    const uint16_t* __restrict__ x, int M, int K, const u32x4_t* __restrict__ wq, const uint32_t* __restrict__ meta,
    const uint16_t* __restrict__ scales8, int N, int S, void* __restrict__ y, int out_f32, float* __restrict__ partial) {
  constexpr int NW = kMidNW, kRows = 16 * MB, kPieces = kW4 ? 1 : 2, kGroupBytes = kRows * 256;
  static_assert(kMidTeams == 2, "one team leaves its sums, the other adds them");
  extern __shared__ __attribute__((aligned(16))) unsigned char mid_lds[];
  const int lane = threadIdx.x & 63, nl = lane & 15, kc = lane >> 4;
  const int all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = all % kMidWaves, team = all / kMidWaves;
  const int ntiles = N / kTileN;
  const int nt0 = (int)blockIdx.x / S * (kMidWaves * NW) + wave * NW, split = (int)blockIdx.x % S;
  const int G = K / kGroup, part0 = split * kMidTeams + team, parts = S * kMidTeams;
  const int begin = (int)((long long)G * part0 / parts), count = (int)((long long)G * (part0 + 1) / parts) - begin;
  // (every team takes as many turns: the barriers are the workgroup's)
  const int turns = (G + parts - 1) / parts;

  // activations: this wave fills rows 4 MB wave .. of the block, four rows of 256 bytes per instruction
  uint32_t x_at[MB], x_to[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int row = 4 * (MB * wave + i) + kc;
    x_at[i] = (uint32_t)min(row, M - 1) * (2u * K) + 16u * nl;
    x_to[i] = (uint32_t)(row * 256 + ((nl ^ (row & 15)) << 4));
  }
  unsigned char* const slots = mid_lds + team * (2 * kGroupBytes);
  const unsigned char* xb = reinterpret_cast<const unsigned char*>(x);
  const u32x4_t* wt[NW];
  const uint32_t* mt[NW];
#pragma unroll
  for (int n = 0; n < NW; ++n) {
    const size_t first = (size_t)min(nt0 + n, ntiles - 1) * G;
    wt[n] = wq + first * (kPieces * 64);
    mt[n] = meta + first * kTileN;
  }
  u32x4_t w[2][NW][kPieces], mw[2][NW], xr[MB];
  auto request = [&](int buf, int turn) {
    const int g = min(begin + turn, G - 1);   // (past this part's groups one is requested, and not used)
#pragma unroll
    for (int i = 0; i < MB; ++i) xr[i] = *reinterpret_cast<const u32x4_t*>(xb + (size_t)g * 256 + x_at[i]);
#pragma unroll
    for (int n = 0; n < NW; ++n) {
#pragma unroll
      for (int p = 0; p < kPieces; ++p) w[buf][n][p] = wt[n][(size_t)(g * kPieces + p) * 64 + lane];
      if (kW4) mw[buf][n] = *reinterpret_cast<const u32x4_t*>(mt[n] + (size_t)g * kTileN + 4 * kc);
    }
  };
  auto put = [&](int slot) {
#pragma unroll
    for (int i = 0; i < MB; ++i) *reinterpret_cast<u32x4_t*>(slots + slot * kGroupBytes + x_to[i]) = xr[i];
  };
  f32x4_t acc[NW][MB] = {};
  const W4Consts consts = w4_consts();
  auto use = [&](int buf) {
    const unsigned char* slot = slots + buf * kGroupBytes;
    f32x4_t part[kW4 ? NW : 1][MB] = {}, sums[kW4 ? MB : 1] = {};
    const u32x4_t ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      u32x4_t xf[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) xf[i] = *reinterpret_cast<const u32x4_t*>(slot + (16 * i + nl) * 256 + (((4 * s + kc) ^ nl) << 4));
#pragma unroll
      for (int n = 0; n < NW; ++n) {
        u32x4_t f;
        if (kW4) {
          f = w4_unpack(w[buf][n][0][s], consts);
        } else {
          const u32x2_t lo = w8_to_bf16(w[buf][n][kPieces == 2 ? s >> 1 : 0][2 * (s & 1)]);
          const u32x2_t hi = w8_to_bf16(w[buf][n][kPieces == 2 ? s >> 1 : 0][2 * (s & 1) + 1]);
          f = u32x4_t{lo.x, lo.y, hi.x, hi.y};
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          if (kW4) part[n][i] = mfma16(f, xf[i], part[n][i]);
          else acc[n][i] = mfma16(f, xf[i], acc[n][i]);
        }
      }
      if (kW4)
#pragma unroll
        for (int i = 0; i < MB; ++i) sums[i] = mfma16(ones, xf[i], sums[i]);
    }
    if (kW4)
#pragma unroll
      for (int n = 0; n < NW; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float scale = f16_bits_to_f32(mw[buf][n][e] & 0xFFFFu), zero = f16_bits_to_f32(mw[buf][n][e] >> 16);
#pragma unroll
          for (int i = 0; i < MB; ++i) acc[n][i][e] = fmaf(scale, fmaf(-zero, sums[i][0], part[n][i][e]), acc[n][i][e]);
        }
  };
  request(0, 0);
  put(0);
  __syncthreads();
  auto step = [&](int buf, int turn) {
    request(buf ^ 1, turn + 1);
    __builtin_amdgcn_sched_barrier(0);
    if (turn < count) use(buf);
    put(buf ^ 1);
    __syncthreads();
  };
  int turn = 0;
  for (; turn + 1 < turns; turn += 2) {
    step(0, turn);
    step(1, turn + 1);
  }
  if (turn < turns) {
    if (turn < count) use(0);
    __syncthreads();
  }
  // the first team adds the second's sums
  f32x4_t* sums = reinterpret_cast<f32x4_t*>(mid_lds) + wave * (NW * MB * 64) + lane;
  static_assert(kMidWaves * NW * MB * 1024 <= mid_lds_bytes(MB), "the sums take the activations' place");
  if (team > 0)
#pragma unroll
    for (int j = 0; j < NW * MB; ++j) sums[64 * j] = acc[j / MB][j % MB];
  __syncthreads();
  if (team > 0) return;
#pragma unroll
  for (int j = 0; j < NW * MB; ++j) acc[j / MB][j % MB] += sums[64 * j];

#pragma unroll
  for (int n = 0; n < NW; ++n) {
    if (nt0 + n >= ntiles) break;
    const int col = (nt0 + n) * kTileN + 4 * kc;
    float cs[4] = {1.f, 1.f, 1.f, 1.f};
    if (!kW4) {
      const u32x2_t h = *reinterpret_cast<const u32x2_t*>(scales8 + col);
      cs[0] = f16_bits_to_f32(h.x & 0xFFFFu); cs[1] = f16_bits_to_f32(h.x >> 16);
      cs[2] = f16_bits_to_f32(h.y & 0xFFFFu); cs[3] = f16_bits_to_f32(h.y >> 16);
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int m = 16 * i + nl;
      if (m >= M) continue;
      const f32x4_t v = {acc[n][i][0] * cs[0], acc[n][i][1] * cs[1], acc[n][i][2] * cs[2], acc[n][i][3] * cs[3]};
      if (S > 1) *reinterpret_cast<f32x4_t*>(partial + ((size_t)split * M + m) * N + col) = v;
      else if (out_f32) *reinterpret_cast<f32x4_t*>(reinterpret_cast<float*>(y) + (size_t)m * N + col) = v;
      else *reinterpret_cast<u32x2_t*>(reinterpret_cast<uint16_t*>(y) + (size_t)m * N + col) = u32x2_t{pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3])};
    }
  }
}

}  // namespace ajq
