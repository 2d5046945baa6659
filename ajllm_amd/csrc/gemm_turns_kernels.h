// Prefill dequant-GEMM, W8A16, on tiles of BM x BN, BM = 64 QM, BN = 128 QN, by waves that take turns.
//
//   y[M, N] = x[M, K] @ W_hat[N, K]^T,  K % 128 == 0; M >= 256 for tiles of 256 rows.
//
// Eight waves, two per SIMD.  64 k at a time, activations enter LDS by DMA in whole 128-byte lines; the packed weights come
// into registers (a private tile of 16 columns per wave and half of the columns), are dequantized ONCE per workgroup to exact
// bf16 integers and written to LDS as rows of the same form.  Channel scales are applied in the epilogue.
//
// LDS holds two buffers of four half tiles (rows 0, rows 1, columns 0, columns 1).  A wave owns a block of each of the four
// quadrants that the halves span and goes through them in the order (0, 0), (0, 1), (1, 1), (1, 0): every half is read into
// registers once per 64 k, one or none per quadrant, and two quadrants later its place is free for what comes 128 k further on.
// The two waves of a SIMD take turns: a quadrant is a part that reads LDS, writes what has been dequantized and asks for data,
// and a part of MFMA with the converts between them; a barrier ends each part, and the second four waves run one part behind the
// first.  So one wave's products always run beside the other's reads.
//
// What it measured (same process, us before -> after; before: eight waves that read ahead of their own MFMAs, ring of four 32-k
// stages): 8192 x 14336 x 4096 757 -> 688 (1.40 PFLOP/s), 5328 x 28672 x 4096 1055 -> 955.  With the converts in the reading
// part that part was longer than the products beside it: 689 and 985.  192 x 256 tiles fill the rounds of others: 5328 x 4096 x
// 4096 194 -> 160, 904 x 8672 x 9344 211 -> 150.  (int4, whose unpack is three times as long and whose accumulators change units
// every group, was no faster this way: 820 us against 973 at 8192 x 14336 x 4096.)
//
// Hazards.  What is written (by request or by ds_write) goes to a place that was read two quadrants or more before: the wave that
// is a part behind has waited for those reads (its products consumed them) ahead of a barrier that the writing wave has passed.
// Requested rows are read in the quadrant after the one whose first part waits for them.  Dequantized columns are read three
// quadrants or more after they were written, and LDS operations of a wave end in order: the reads that it waited for in between
// came after its writes.
#pragma once
#include <type_traits>

#include "gemm_split_kernels.h"  // lds_write128, load16_async, wait_loads

namespace ajq {

constexpr int kTurnsThreads = 512;
// buffers, or the output on its way out: bf16 rows of the tile, fp32 rows of half of it, 16 bytes apart
constexpr int gemm_turns_lds(int bm, int bn) {
  const int ring = 2 * (bm + bn) * 128, half = bm * (2 * bn + 16), full = bm / 2 * (4 * bn + 16);
  return ring > half ? (ring > full ? ring : full) : half > full ? half : full;
}
template <int kLeft>
__device__ __forceinline__ void wait_load(u32x4_t& a) {
  asm volatile("s_waitcnt vmcnt(%1)" : "+v"(a) : "n"(kLeft) : "memory");
}

// kGate: the weights are the w1 | w3 rows of a SwiGLU feed-forward (N = 2 F, F % 16 == 0).  The first half of a workgroup's
// columns are then gate projections and the second half the up projections of the SAME BN / 2 columns: a wave holds both factors,
// and writes bf16( silu(a) * u ), [M, F].
template <bool kGate, int QM, int QN>
__global__ __launch_bounds__(kTurnsThreads) void dequant_gemm_turns_kernel(const uint16_t* __restrict__ x, int M, int K,
                                                                           const u32x4_t* __restrict__ wq,
                                                                           const uint16_t* __restrict__ scales, int N,
                                                                           void* __restrict__ y, int out_f32) {
  constexpr int BM = 64 * QM, BN = 128 * QN;
  constexpr int kHalfA = BM / 2 * 128, kHalfB = BN / 2 * 128;  // bytes of half a tile's rows, 64 k of them
  constexpr int kColumns = 4 * kHalfA;                         // rows of both buffers, then columns of both
  constexpr int QA = kHalfA / 1024, RA = (QA + 7) / 8;         // 1 KiB requests of a half's rows, of a wave (some are made twice where 8 does not divide)
  constexpr bool kShift = QM == 4;
  extern __shared__ u32x4_t smem_raw[];
  char* lds = reinterpret_cast<char*>(smem_raw);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int r = lane & 15, g = lane >> 4;
  constexpr int tile_cols = kGate ? BN / 2 : BN;  // of the result
  const int cols = kGate ? N >> 1 : N;
  int tile_m, tile_n;
  tile_place((M + BM - 1) / BM, (cols + tile_cols - 1) / tile_cols, tile_m, tile_n);
  const int m0 = kShift ? min(tile_m * BM, M - BM) : tile_m * BM, n0 = tile_n * tile_cols;
  const int steps = K >> 6, last = steps - 1;  // (an even number)

  // ---- activations: eight rows of 128 bytes a request; chunk c of a half's row r sits in slot c ^ ((r >> 1) & 7), so that the 16
  // rows a fragment read meets lie in distinct banks.  Rows past the end repeat the last one; of tiles of 256 rows, whose registers are
  // few, the last is shifted up to end at row M instead.
  const char* a_base = reinterpret_cast<const char*>(x) + (size_t)m0 * K * 2;
  uint32_t a_voff[kShift ? 1 : 2][kShift ? 1 : RA];
#pragma unroll
  for (int h = 0; h < (kShift ? 1 : RA); ++h) {
    const int row = 8 * min(h * 8 + wave, QA - 1) + (lane >> 3);
    const uint32_t chunk = (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
#pragma unroll
    for (int f = 0; f < (kShift ? 1 : 2); ++f)
      a_voff[f][h] = (uint32_t)(kShift ? row : min(m0 + f * (BM / 2) + row, M - 1) - m0) * (uint32_t)K * 2u + chunk;
  }
  auto request_a = [&](int step, int buffer, int f) {
#pragma unroll
    for (int h = 0; h < RA; ++h) {
      const size_t rows = kShift ? (size_t)(f * (BM / 2) + 64 * h) * K * 2 : 0;
      dma16(a_base + rows + (size_t)step * 128, a_voff[kShift ? 0 : f][kShift ? 0 : h],
            (uint32_t)((2 * buffer + f) * kHalfA + min(h * 8 + wave, QA - 1) * 1024));
    }
  };
  // ---- weights: of half f, QN = 2: this wave's 16 columns, QN = 1: one 32-k half of the 16 columns it shares with another wave.
  // Tile lane (r, g) holds 8 consecutive k of column r from 8 g on, of each 32 k.
  const int strips = N / kTileN, mine = QN == 2 ? wave : wave & 3, part32 = wave >> 2;
  const u32x4_t* b_src[2];
#pragma unroll
  for (int f = 0; f < 2; ++f) {
    const int at = kGate ? f * (strips >> 1) + n0 / kTileN + mine : n0 / kTileN + f * 4 * QN + mine;
    b_src[f] = wq + (size_t)min(at, strips - 1) * steps * 64;
  }
  const uint32_t lane16 = (uint32_t)lane * 16u;
  auto fetch = [&](u32x4_t& words, int f, int step) { load16_async(words, b_src[f] + (size_t)min(step, last) * 64, lane16); };
  uint32_t b_wr[QN];  // where this lane's chunk of a step's first / second 32 k goes (QN = 1: of the wave's 32 k)
#pragma unroll
  for (int c = 0; c < QN; ++c) {
    const int row = mine * 16 + r, half = QN == 2 ? c : part32;
    b_wr[c] = (uint32_t)(kColumns + row * 128 + (((4 * half + g) ^ ((row >> 1) & 7)) * 16));
  }
  // chunk c of the packed words of 64 k, eight bf16.  (QN = 1: the words are selected, not branched to: they come from a load that is
  // waited for by name.)
  auto convert = [&](const u32x4_t& words, int c) {
    const u32x2_t lo = w8_to_bf16(QN == 2 ? words[2 * c] : part32 ? words[2] : words[0]);
    const u32x2_t hi = w8_to_bf16(QN == 2 ? words[2 * c + 1] : part32 ? words[3] : words[1]);
    return u32x4_t{lo.x, lo.y, hi.x, hi.y};
  };
  auto put = [&](const u32x4_t& v, int buffer, int f, int c) { lds_write128((uint32_t)((2 * buffer + f) * kHalfB) + b_wr[c], v); };

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
    b_rel[s] = (uint32_t)(kColumns + (wn * QN * 16 + r) * 128) + c;
  }
  u32x4_t af[QM][2], bf[2][QN][2];
  auto read_a = [&](int buffer, int f) {
#pragma unroll
    for (int i = 0; i < QM; ++i)
#pragma unroll
      for (int s = 0; s < 2; ++s) af[i][s] = lds_read128((uint32_t)((2 * buffer + f) * kHalfA + i * 2048) + a_rel[s]);
  };
  auto read_b = [&](int buffer, int f) {
#pragma unroll
    for (int t = 0; t < QN; ++t)
#pragma unroll
      for (int s = 0; s < 2; ++s) bf[f][t][s] = lds_read128((uint32_t)((2 * buffer + f) * kHalfB + t * 2048) + b_rel[s]);
  };
  // The weights are the first operand: a lane then holds four neighbouring columns of a row.  `beside`: the converts that issue between
  // the MFMAs (a SIMD issues VALU instructions of the wave under them).
  auto products = [&](int ha, int hb, auto beside) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < QM; ++i)
#pragma unroll
        for (int t = 0; t < QN; ++t) acc[ha][hb][i][t] = mfma16(bf[hb][t][s], af[i][s], acc[ha][hb][i][t]);
    beside();
#pragma unroll
    for (int i = 0; i < 2 * QM * QN; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two converts
    }
    __builtin_amdgcn_s_setprio(0);
  };

  // ---- A step asks for rows 1 of the next one and rows 0 of the one after, and dequantizes columns 1 of the next (beside its first two
  // quadrants) and columns 0 of the one after (beside the other two); what is dequantized beside one quadrant's products is written in
  // front of the next one's.  P, Q: the packed words of even / odd steps.
  u32x4_t P[2], Q[2], cv;
  request_a(0, 0, 0);
  request_a(0, 0, 1);
  request_a(1, 1, 0);
  {
    u32x4_t first[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      fetch(first[f], f, 0);
      fetch(Q[f], f, 1);
      fetch(P[f], f, 2);
    }
    wait_loads<0>(first);
    wait_loads<0>(P);
    wait_loads<0>(Q);
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int c = 0; c < QN; ++c) put(convert(first[f], c), 0, f, c);
    cv = convert(Q[0], 0);
    put(cv, 1, 0, 0);
    if (QN == 2) cv = convert(Q[0], 1);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  turn_barrier();
  if (wm == 1) turn_barrier();

  // E: packed words of steps of j's parity, O: of the others'.  Columns 0 of step j + 2 are in E[0], asked for in step j - 1; columns 1 of
  // step j + 1 in O[1], asked for in step j - 2.
  auto step = [&](int j, auto bc, u32x4_t (&E)[2], u32x4_t (&O)[2]) {
    constexpr int cur = decltype(bc)::value, nxt = cur ^ 1;
    const int j1 = min(j + 1, last), j2 = min(j + 2, last);  // (past the end: the last ones again, not read)
    if (QN == 2) put(cv, nxt, 0, 1);  // the rest of columns 0 of step j + 1
    fetch(O[0], 0, j + 3);
    read_a(cur, 0);
    read_b(cur, 0);
    request_a(j1, nxt, 1);
    wait_load<4 * RA + 3>(O[1]);
    turn_barrier();
    products(0, 0, [&] { cv = convert(O[1], 0); });
    turn_barrier();
    put(cv, nxt, 1, 0);
    read_b(cur, 1);
    // rows 1 of step j; younger: a load, rows 0 of step j + 1, a load, rows 1 of step j + 1
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * RA + 2) : "memory");
    turn_barrier();
    products(0, 1, [&] { if (QN == 2) cv = convert(O[1], QN - 1); });
    turn_barrier();
    if (QN == 2) put(cv, nxt, 1, QN - 1);
    fetch(O[1], 1, j + 3);
    read_a(cur, 1);
    request_a(j2, cur, 0);
    wait_load<4 * RA + 3>(E[0]);
    turn_barrier();
    products(1, 1, [&] { cv = convert(E[0], 0); });
    turn_barrier();
    put(cv, cur, 0, 0);
    // rows 0 of step j + 1; younger: a load, rows 1 of step j + 1, a load, rows 0 of step j + 2
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * RA + 2) : "memory");
    turn_barrier();
    products(1, 0, [&] { if (QN == 2) cv = convert(E[0], QN - 1); });
    turn_barrier();
  };
  for (int j = 0; j < steps; j += 2) {
    step(j, std::integral_constant<int, 0>{}, P, Q);
    step(j + 1, std::integral_constant<int, 1>{}, Q, P);
  }
  // The last steps' redundant loads are still in flight, and nothing reads their registers any more: unless the wait NAMES them,
  // the compiler hands those registers to the epilogue's first values in front of it.
  wait_loads<0>(P);
  wait_loads<0>(Q);
  if (wm == 0) turn_barrier();

  // ---- epilogue: through LDS, whole rows of the tile per store.  (The lane's place is counted again: kept through the loop it would
  // cost registers that the 256 x 256 tile does not have.)
  uint32_t zero = 0;
  asm volatile("" : "+v"(zero));
  const int thread = wave * 64 + (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
  const int er = thread & 15, eg = (thread >> 4) & 3;
  auto row_of = [&](int ha, int i) { return ha * (BM / 2) + (wm * QM + i) * 16 + er; };
  auto col_of = [&](int hb, int t) { return hb * (BN / 2) + (wn * QN + t) * 16 + 4 * eg; };
  float scale[2][QN][4];
#pragma unroll
  for (int hb = 0; hb < 2; ++hb)
#pragma unroll
    for (int t = 0; t < QN; ++t) {
      const int n = n0 + (kGate ? hb * (N >> 1) + col_of(0, t) : col_of(hb, t));
#pragma unroll
      for (int e = 0; e < 4; ++e) scale[hb][t][e] = f16_bits_to_f32(scales[min(n + e, N - 1)]);
    }
  auto value = [&](int ha, int hb, int i, int t, int e) -> float { return acc[ha][hb][i][t][e] * scale[hb][t][e]; };
  if (!kGate && out_f32) {
    constexpr int kStride = BN * 4 + 16, kPieces = BN / 4;
    float* out = reinterpret_cast<float*>(y);
#pragma unroll
    for (int ha = 0; ha < 2; ++ha) {  // (half the rows at a time)
      __syncthreads();
#pragma unroll
      for (int i = 0; i < QM; ++i)
#pragma unroll
        for (int hb = 0; hb < 2; ++hb)
#pragma unroll
          for (int t = 0; t < QN; ++t)
            *reinterpret_cast<f32x4_t*>(lds + row_of(0, i) * kStride + col_of(hb, t) * 4) =
                f32x4_t{value(ha, hb, i, t, 0), value(ha, hb, i, t, 1), value(ha, hb, i, t, 2), value(ha, hb, i, t, 3)};
      __syncthreads();
#pragma unroll
      for (int at = 0; at < BM / 2 * kPieces; at += kTurnsThreads) {
        const int piece = at + thread, row = piece / kPieces, n = n0 + piece % kPieces * 4, m = m0 + ha * (BM / 2) + row;
        const f32x4_t v = *reinterpret_cast<const f32x4_t*>(lds + row * kStride + piece % kPieces * 16);
        if (m < M && n < N) *reinterpret_cast<f32x4_t*>(out + (size_t)m * N + n) = v;
      }
    }
    return;
  }
  constexpr int kStride = tile_cols * 2 + 16, kPieces = tile_cols / 8;
  __syncthreads();
#pragma unroll
  for (int ha = 0; ha < 2; ++ha)
#pragma unroll
    for (int i = 0; i < QM; ++i)
#pragma unroll
      for (int hb = 0; hb < (kGate ? 1 : 2); ++hb)
#pragma unroll
        for (int t = 0; t < QN; ++t) {
          float v[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float a = value(ha, hb, i, t, e);
            v[e] = kGate ? a * (1.0f / (1.0f + expf(-a))) * value(ha, 1, i, t, e) : a;
          }
          *reinterpret_cast<u32x2_t*>(lds + row_of(ha, i) * kStride + col_of(hb, t) * 2) = u32x2_t{pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3])};
        }
  __syncthreads();
#pragma unroll
  for (int at = 0; at < BM * kPieces; at += kTurnsThreads) {
    const int piece = at + thread, row = piece / kPieces, n = n0 + piece % kPieces * 8;
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(lds + row * kStride + piece % kPieces * 16);
    if (m0 + row < M && n < cols) *reinterpret_cast<u32x4_t*>(reinterpret_cast<uint16_t*>(y) + (size_t)(m0 + row) * cols + n) = v;
  }
}

}  // namespace ajq
