// Product of many rows in bf16: y[M, N] = x[M, K] w[N, K]^T, K % 64 == 0, fp32 accumulators, with the activation behind it where
// there is one.
//
// A workgroup of eight waves makes one tile of BM x BN.  Rows of both operands enter LDS by DMA, 64 k (whole 128-byte lines) at
// a time, in two buffers of four half tiles (rows 0, rows 1, columns 0, columns 1).  A wave owns a block of each of the four
// quadrants that the halves span and goes through them in the order (0, 0), (0, 1), (1, 1), (1, 0): every half is read into
// registers once per 64 k, one or none per quadrant, and two quadrants later its place takes the half 128 k further on.
//
// The two waves of a SIMD take turns: a quadrant is a part that reads LDS and asks for data and a part that is nothing but MFMA, a
// barrier ends each part, and the second four waves run one part behind the first.  So one wave's MFMA always runs beside the
// other's reads.  Eight waves that all read ahead of their own MFMAs (ring of four 32-k stages, one barrier per stage, the
// order left to the compiler) reached 1.31 PFLOP/s at 8192 x 8192 x 8192, this 1.62; there the clock is what limits (the
// vendor's product: 1.61 to 1.65).
//
// Hazards.  A request goes to a place that was read two quadrants before: the wave that is a part behind has waited for those
// reads (its products consumed them) ahead of a barrier that the requesting wave has passed.  A half is read in the quadrant after
// the one whose first part waits until at most the requests of four younger halves are in flight; both groups of waves have
// passed that wait, and a barrier, when the first of them reads.
#pragma once
#include <type_traits>

#include "dense_kernels.h"
#include "gemm_kernels.h"

namespace ajq {

struct DenseGemm {
  const uint16_t *x, *w;
  void* y;
  int m, n, k, ldx, ldy, act;
  int part;  // of k, a workgroup row's (gridDim.y); more than one: fp32 planes [parts][m][ldy]
};

// What becomes of the sums: fp32, bf16, bf16(act(sum)), or bf16(act(gate) * up) of w's rows in blocks of 8 gates and their 8 ups.
enum { kTileF32 = 0, kTileBf16 = 1, kTileAct = 2, kTilePairs = 3 };

constexpr int kTileThreads = 512;
constexpr int tile_lds_bytes(int bm, int bn, int epi) {
  const int stages = 2 * (bm + bn) * 128;
  const int out = epi == kTileF32 ? bm / 2 * (4 * bn + 16) : bm * ((epi == kTilePairs ? bn : 2 * bn) + 16);
  return stages > out ? stages : out;
}

// A quadrant of a wave: QM x QN blocks of 16 x 16; BM = 64 QM, BN = 128 QN.
template <int QM, int QN, int EPI>
__global__ __launch_bounds__(kTileThreads) void dense_gemm_kernel(DenseGemm a) {
  constexpr int BM = 64 * QM, BN = 128 * QN;
  constexpr int kHalfA = BM / 2 * 128, kHalfB = BN / 2 * 128;  // bytes of half a tile's rows, 64 k of them
  constexpr int kStage = 2 * (kHalfA + kHalfB);                // rows 0, rows 1, columns 0, columns 1
  constexpr int QA = kHalfA / 1024, QB = kHalfB / 1024;        // 1 KiB requests of a half
  constexpr int RA = (QA + 7) / 8, RB = (QB + 7) / 8;          // of a wave (some are made twice where 8 does not divide)
  extern __shared__ u32x4_t smem_raw[];
  char* lds = reinterpret_cast<char*>(smem_raw);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int r = lane & 15, g = lane >> 4;
  const int k0 = (int)blockIdx.y * a.part, steps = min(a.part, a.k - k0) >> 6;
  int tile_m, tile_n;
  tile_place((a.m + BM - 1) / BM, (a.n + BN - 1) / BN, tile_m, tile_n);
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  // ---- requests: eight rows of 128 bytes each; chunk c of a half's row r sits in slot c ^ ((r >> 1) & 7), so that the 16 rows
  // a fragment read meets lie in distinct banks.  Rows past the end repeat the last one.
  const char* a_base = reinterpret_cast<const char*>(a.x) + ((size_t)m0 * a.ldx + k0) * 2;
  const char* b_base = reinterpret_cast<const char*>(a.w) + ((size_t)n0 * a.k + k0) * 2;
  uint32_t a_voff[2][RA], b_voff[2][RB], a_to[RA], b_to[RB];
#pragma unroll
  for (int h = 0; h < RA; ++h) {
    const int q = min(h * 8 + wave, QA - 1), row = 8 * q + (lane >> 3);
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
    a_to[h] = (uint32_t)(q * 1024);
#pragma unroll
    for (int f = 0; f < 2; ++f) a_voff[f][h] = (uint32_t)(min(m0 + f * (BM / 2) + row, a.m - 1) - m0) * (uint32_t)a.ldx * 2u + chunk;
  }
#pragma unroll
  for (int h = 0; h < RB; ++h) {
    const int q = min(h * 8 + wave, QB - 1), row = 8 * q + (lane >> 3);
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
    b_to[h] = (uint32_t)(q * 1024);
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      // pairs: half 0 takes the gates, half 1 their ups
      const int from = EPI == kTilePairs ? 16 * (row >> 3) + (row & 7) + 8 * f : f * (BN / 2) + row;
      b_voff[f][h] = (uint32_t)(min(n0 + from, a.n - 1) - n0) * (uint32_t)a.k * 2u + chunk;
    }
  }
  auto request_a = [&](int step, int buffer, int f) {
#pragma unroll
    for (int h = 0; h < RA; ++h) dma16(a_base + (size_t)step * 128, a_voff[f][h], (uint32_t)(buffer * kStage + f * kHalfA) + a_to[h]);
  };
  auto request_b = [&](int step, int buffer, int f) {
#pragma unroll
    for (int h = 0; h < RB; ++h)
      dma16(b_base + (size_t)step * 128, b_voff[f][h], (uint32_t)(buffer * kStage + 2 * kHalfA + f * kHalfB) + b_to[h]);
  };

  f32x4_t acc[2][2][QM][QN];
#pragma unroll
  for (int ha = 0; ha < 2; ++ha)
#pragma unroll
    for (int hb = 0; hb < 2; ++hb)
#pragma unroll
      for (int i = 0; i < QM; ++i)
#pragma unroll
        for (int t = 0; t < QN; ++t) acc[ha][hb][i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // fragment of block b and 32-k half s: row 16 b + r, chunk 4 s + g
  uint32_t a_rel[2], b_rel[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const uint32_t c = (uint32_t)(((4 * s + g) ^ ((r >> 1) & 7)) * 16);
    a_rel[s] = (uint32_t)((wm * QM * 16 + r) * 128) + c;
    b_rel[s] = (uint32_t)(2 * kHalfA + (wn * QN * 16 + r) * 128) + c;
  }
  u32x4_t af[QM][2], bf[2][QN][2];
  auto read_a = [&](int buffer, int f) {
#pragma unroll
    for (int i = 0; i < QM; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) af[i][s] = lds_read128((uint32_t)(buffer * kStage + f * kHalfA + i * 2048) + a_rel[s]);
  };
  auto read_b = [&](int buffer, int f) {
#pragma unroll
    for (int t = 0; t < QN; ++t)
#pragma unroll
      for (int s = 0; s < 2; ++s) bf[f][t][s] = lds_read128((uint32_t)(buffer * kStage + f * kHalfB + t * 2048) + b_rel[s]);
  };
  // (the weights are the first operand: a lane then holds four neighbouring columns of a row)
  auto products = [&](int ha, int hb) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < QM; ++i)
#pragma unroll
        for (int t = 0; t < QN; ++t) acc[ha][hb][i][t] = mfma16(bf[hb][t][s], af[i][s], acc[ha][hb][i][t]);
    __builtin_amdgcn_s_setprio(0);
  };
  constexpr int kYounger = 2 * (RA + RB);
  const int last = steps - 1;
  request_a(0, 0, 0);
  request_b(0, 0, 0);
  request_b(0, 0, 1);
  request_a(0, 0, 1);
  request_a(min(1, last), 1, 0);
  request_b(min(1, last), 1, 0);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kYounger) : "memory");
  turn_barrier();
  if (wm == 1) turn_barrier();

  auto step = [&](int j, auto bc) {
    constexpr int cur = decltype(bc)::value, nxt = cur ^ 1;
    const int j1 = min(j + 1, last), j2 = min(j + 2, last);  // (past the end: the last ones again, not read)
    read_a(cur, 0);
    read_b(cur, 0);
    request_b(j1, nxt, 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kYounger) : "memory");
    turn_barrier();
    products(0, 0);
    turn_barrier();
    read_b(cur, 1);
    request_a(j1, nxt, 1);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kYounger) : "memory");
    turn_barrier();
    products(0, 1);
    turn_barrier();
    read_a(cur, 1);
    request_a(j2, cur, 0);
    turn_barrier();
    products(1, 1);
    turn_barrier();
    request_b(j2, cur, 0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kYounger) : "memory");
    turn_barrier();
    products(1, 0);
    turn_barrier();
  };
  for (int j = 0; j < steps; j += 2) {
    step(j, std::integral_constant<int, 0>{});
    if (j + 1 < steps) step(j + 1, std::integral_constant<int, 1>{});
  }
  if (wm == 0) turn_barrier();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- the result leaves through LDS in whole rows of the tile, 16 bytes per lane
  auto row_of = [&](int ha, int i) { return ha * (BM / 2) + (wm * QM + i) * 16 + r; };
  auto col_of = [&](int hb, int t) { return hb * (BN / 2) + (wn * QN + t) * 16 + 4 * g; };
  if constexpr (EPI == kTileF32) {
    constexpr int kStride = BN * 4 + 16, kPieces = BN / 4;
    float* y = reinterpret_cast<float*>(a.y) + (size_t)blockIdx.y * a.m * a.ldy;
#pragma unroll
    for (int ha = 0; ha < 2; ++ha) {  // (half the rows at a time)
      __syncthreads();
#pragma unroll
      for (int i = 0; i < QM; ++i)
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
#pragma unroll
          for (int t = 0; t < QN; ++t) *reinterpret_cast<f32x4_t*>(lds + row_of(0, i) * kStride + col_of(hb, t) * 4) = acc[ha][hb][i][t];
      __syncthreads();
#pragma unroll
      for (int at = 0; at < BM / 2 * kPieces; at += kTileThreads) {
        const int id = at + threadIdx.x, row = id / kPieces, n = n0 + id % kPieces * 4, m = m0 + ha * (BM / 2) + row;
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(lds + row * kStride + id % kPieces * 16);
        if (m < a.m && n < a.n) *reinterpret_cast<f32x4_t*>(y + (size_t)m * a.ldy + n) = v;
      }
    }
  } else {
    constexpr int cols = EPI == kTilePairs ? BN / 2 : BN;  // of the tile's result
    constexpr int kStride = cols * 2 + 16, kPieces = cols / 8;
    __syncthreads();
    auto put = [&](auto act) {
      constexpr int ACT = decltype(act)::value;
#pragma unroll
      for (int ha = 0; ha < 2; ++ha)
#pragma unroll
        for (int i = 0; i < QM; ++i)
#pragma unroll
          for (int hb = 0; hb < (EPI == kTilePairs ? 1 : 2); ++hb)
#pragma unroll
            for (int t = 0; t < QN; ++t) {
              float v[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float s = acc[ha][hb][i][t][e];
                v[e] = EPI == kTileBf16 ? s : EPI == kTileAct ? activate(ACT, s) : activate(ACT, s) * acc[ha][1][i][t][e];
              }
              *reinterpret_cast<u32x2_t*>(lds + row_of(ha, i) * kStride + col_of(hb, t) * 2) = u32x2_t{pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3])};
            }
    };
    // (one choice per tile: made per value it cost 15 us of 178 at 1500 x 16384 x 4096)
    if (EPI == kTileBf16 || a.act == kActRelu) put(std::integral_constant<int, kActRelu>{});
    else if (a.act == kActSquaredRelu) put(std::integral_constant<int, kActSquaredRelu>{});
    else if (a.act == kActSilu) put(std::integral_constant<int, kActSilu>{});
    else put(std::integral_constant<int, kActGeluTanh>{});
    __syncthreads();
    const int out_n = EPI == kTilePairs ? a.n / 2 : a.n, on0 = EPI == kTilePairs ? n0 / 2 : n0;
#pragma unroll
    for (int at = 0; at < BM * kPieces; at += kTileThreads) {
      const int id = at + threadIdx.x, row = id / kPieces, n = on0 + id % kPieces * 8;
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(lds + row * kStride + id % kPieces * 16);
      if (m0 + row < a.m && n < out_n) *reinterpret_cast<u32x4_t*>(reinterpret_cast<uint16_t*>(a.y) + (size_t)(m0 + row) * a.ldy + n) = v;
    }
  }
}

// y = the sum of a product's parts: eight columns of a row per thread.  Bound by its bytes, read where the parts have just been written
// (1500 x 4096 in two parts: 13.1 us, 5.6 TB/s).
template <typename O>
__global__ __launch_bounds__(256) void sum_parts_kernel(const float* planes, int parts, int m, int n, O* y, int ldy) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x, pieces = (size_t)m * (n / 8);
  if (i >= pieces) return;
  Float8 v = load8(planes + i * 8);
#pragma unroll 4
  for (int p = 1; p < parts; ++p) {
    const Float8 u = load8(planes + ((size_t)p * pieces + i) * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) v.v[e] += u.v[e];
  }
  store8(y + i / (n / 8) * ldy + i % (n / 8) * 8, v);
}

}  // namespace ajq
