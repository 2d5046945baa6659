// Causal self-attention for a block of T new positions (prefill), head_dim HD = 128, 64 or 32, on bf16 MFMA
// with an online softmax: the T x (start + T) score matrix is never materialised.
//
//   out[b, t, h, :] = softmax_j( q[b, h, t, :] . k[b, hk, j, :] / sqrt(HD) ) v[b, hk, j, :],
//   j <= start + t,   hk = h / (H / Hkv)
//
// q is fp32 [B, H, T, HD] (already rotated); keys and values are read where the model keeps
// them, in the caches [B, Hkv, max_len, HD] (fp32 or bf16), rows 0 .. start + T - 1; out is
// fp32 or bf16 [B, T, H * HD], the layout the output projection takes.  (The layouts below are
// written out for HD = 128; with 64 a row is 128 B = 8 chunks = 4 segments and there are two k-steps, with 32 a row is
// 64 B = 4 chunks = 2 segments and there is one.)
//
// A workgroup of 4 waves owns 128 query rows of one (b, h), a wave two groups of 16 of them
// (every key and value fragment read from LDS meets both), and walks the keys in blocks of 64.
// Both products run transposed so that no operand changes layout between them:
//   S^T = K Q^T :  A = 16 keys x 32 dims from the row-major key tile in LDS, B = the wave's Q
//                  fragments (registers, bf16, pre-scaled by log2(e) / sqrt(HD)); lane
//                  (g = l / 16, r = l % 16) receives keys 4g..4g+3 of query row r.  The
//                  accumulator starts at minus the row's reference point, so the MFMA result is
//                  the exponent itself.
//   O^T += V^T P^T: the lane's 8 probabilities of a 32-key half ARE its B fragment (contraction
//                  slot 8g + e <-> key 4g + e of the first 16-key tile for e < 4, of the second
//                  for e >= 4), and the A fragment takes the same keys of V^T with two
//                  transposing LDS reads (ds_read_b64_tr_b16) from the ROW-MAJOR value tile:
//                  nothing is transposed on the way into LDS.
// Both tiles are unpadded (a row is 256 B); the 16-byte chunks of a row sit in slots permuted by
// the row index so that the fragment reads spread over all banks.
//
// Softmax bookkeeping is kept off the common path.  A row's reference point only moves when an
// exponent would exceed 2^kPfSlack (always on the first keys): the test is one compare of the
// lane's sum of new probabilities (a sum of positives bounds each of them; inf passes it too),
// and only then are the maxima taken (across the four lanes of a row with two lane swaps), the
// probabilities recomputed and the accumulators rescaled.  Row sums stay per lane and meet once,
// at the end.  bf16 inputs, fp32 scores, probabilities rounded to bf16 for the second product,
// fp32 accumulators: the usual flash-attention arithmetic, not the eager fp32 one.
//
// Two kernels: attn_prefill_steps_kernel on bf16 caches interleaves both products and the softmax of three neighbouring half blocks;
// attn_prefill_kernel goes block by block, where that is the faster (prefill_in_steps) and for fp32 caches, which pass through
// registers that are converted on the way and leave none for the other, unless there is work enough to make a bf16 copy of the rows first
// (caches_to_bf16_kernel).
#pragma once
#include <type_traits>

#include "ajq_common.h"
#include "gemm_kernels.h"  // dma16: global -> LDS without registers

namespace ajq {

constexpr float kPfSlack = 8.0f;          // log2 of how far a row's exponents may exceed its reference point
// A lane's sum of new probabilities above which the reference point is revisited.  Up to there none of them passes 2^12; above, the largest of
// a block's 16 passes 2^8, of a step's 8 (attn_prefill_steps_kernel) 2^9, so that the revisit always finds one past the slack.
constexpr float kPfTrigger = 4096.0f;
constexpr int kPfBQ = 128, kPfBK = 64;

__device__ __forceinline__ u32x4_t pack8_bf16(const float* v) {
  return u32x4_t{pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]), pack2_bf16(v[4], v[5]), pack2_bf16(v[6], v[7])};
}
// 8 consecutive cache elements as loaded, and their bf16 form (made when they are needed, so
// that the loads can stay in flight meanwhile)
struct Raw8F32 {
  float4 a, b;
};
__device__ __forceinline__ Raw8F32 load8_raw(const float* p) {
  return Raw8F32{reinterpret_cast<const float4*>(p)[0], reinterpret_cast<const float4*>(p)[1]};
}
__device__ __forceinline__ u32x4_t load8_raw(const uint16_t* p) { return *reinterpret_cast<const u32x4_t*>(p); }
__device__ __forceinline__ u32x4_t to_bf16x8(const Raw8F32& r) {
  const float v[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
  return pack8_bf16(v);
}
__device__ __forceinline__ u32x4_t to_bf16x8(const u32x4_t& r) { return r; }

typedef short pf_i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) pf_i16x4_t pf_lds_i16x4_t;
typedef __attribute__((address_space(3))) const u32x4_t pf_lds_u32x4_t;
typedef __attribute__((address_space(3))) unsigned char pf_lds_char_t;
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Wint-to-pointer-cast"  // the host pass sees 64-bit pointers
// Transposing LDS read: within each block of 16 lanes, lane 4 a + j receives element j of the
// 8-byte rows addressed by lanes a, 4 + a, 8 + a and 12 + a of the block.
__device__ __forceinline__ u32x2_t pf_read_tr(uint32_t address) {
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((pf_lds_i16x4_t*)address));
}
__device__ __forceinline__ u32x4_t pf_read128(uint32_t address) { return *(pf_lds_u32x4_t*)address; }
#pragma clang diagnostic pop

// prefill_waits: fp32 caches that no two heads share, read by more heads than the L2s hold, gain from every request of a block being waited for at its
// barrier (kWait): the workgroups of a head then stay together and find each other's rows there.  Without, 64 columns and as many key heads: 256
// heads of 1024 keys 78.4 -> 92.0 us, of 2000 320 -> 340, 512 of 791 150 -> 153; where it does not matter the wait costs 1 .. 2 %
// (192 heads 0.997, 128 0.96 .. 1.04; two heads a key head 0.995 over 40 shapes; 128 columns 0.995, 32 0.995).
__host__ __device__ inline bool prefill_waits(int batch, int heads, int key_heads, int head_dim) {
  return head_dim == 64 && heads == key_heads && (long long)batch * heads > 192;
}
template <typename CacheT, int HD, bool kWait = false>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(const float* __restrict__ q, const CacheT* __restrict__ kcache,
                                                           const CacheT* __restrict__ vcache, int H, int Hkv, int T,
                                                           int start, int max_len, void* __restrict__ out, int out_bf16) {
  static_assert(HD == 128 || HD == 64 || HD == 32, "head_dim 128, 64 or 32");
  constexpr int kPfHD = HD;
  constexpr int RB = 2 * HD;          // bytes of a key (value) row as bf16
  constexpr int C = HD / 8;           // 16-byte chunks per row
  constexpr int KS = HD / 32;         // k-steps of the first product; also the parts a block's DMA is issued in
  constexpr int TT = HD / 16;         // 32-byte segments per row = 16-dim output tiles
  constexpr int kPfTileBytes = kPfBK * RB;  // one block of keys (or values) as bf16: 16 KiB at HD = 128
  // LDS map (byte addresses relative to lds0, the array's LDS address, which is 0 because the kernel
  // declares no other LDS; naming it also keeps the array allocated when nothing else refers to
  // it): two stages of a key tile and a value tile, 16 KiB each.
  //   stage s: keys at s * 32 Ki, values at s * 32 Ki + 16 Ki
  // Key tile: 16-byte chunk c of key row k sits at k * 256 + 16 * (c ^ (k & 15)).
  // Value tile: chunk c of row k sits at k * 256 + 16 * ((((c >> 1) ^ (k & 7)) << 1) | (c & 1))
  // (32-byte segments permuted: a transposing read takes 8 bytes of each of 16 keys).
  __shared__ __attribute__((aligned(1024))) unsigned char lds[4 * kPfTileBytes];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(pf_lds_char_t*)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  // Work order.  The hardware deals workgroups to the 8 XCDs round-robin by linear index and,
  // inside an XCD, hands the next one to whichever CU has room.  A query block's cost grows with
  // its position (causal), so the linear order is: XCD k takes a contiguous eighth of the (b, h)
  // pairs (the heads that share a cache head stay on one XCD and its L2) and walks its query
  // blocks from the longest to the shortest.  (With B * H not a multiple of 8: plain longest first.)
  const int qblocks = (T + kPfBQ - 1) / kPfBQ;
  const int BH = (int)(gridDim.x / (unsigned)qblocks);
  int qb, bh;
  if ((BH & 7) == 0) {
    const int per_xcd = BH >> 3, m = (int)(blockIdx.x >> 3);
    qb = qblocks - 1 - m / per_xcd;
    bh = (int)(blockIdx.x & 7) * per_xcd + m % per_xcd;
  } else {
    qb = qblocks - 1 - (int)blockIdx.x / BH;
    bh = (int)blockIdx.x % BH;
  }
  const int b = bh / H, h = bh % H, hk = h / (H / Hkv);
  const int q0 = qb * kPfBQ;
  const float qscale =  // log2(e) / sqrt(HD)
      1.4426950408889634f * (HD == 128 ? 0.08838834764831845f : HD == 64 ? 0.125f : 0.17677669529663687f);

  const CacheT* kbase = kcache + ((size_t)b * Hkv + hk) * max_len * kPfHD;
  const CacheT* vbase = vcache + ((size_t)b * Hkv + hk) * max_len * kPfHD;
  const int kv_len = start + T;                               // rows the caches hold for this call
  const int kv_end = min(kv_len, start + q0 + kPfBQ);         // keys any row of this workgroup may see
  const int nblk = (kv_end + kPfBK - 1) / kPfBK;
  const int wave_last_pos = start + q0 + 32 * wave + 31;      // last query position of this wave

  float m_run[2], l_run[2];
  f32x4_t negm[2];
  f32x4_t o[2][TT];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    m_run[u] = 0.f;
    l_run[u] = 0.f;
    negm[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < TT; ++t) o[u][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // ---- Keys and values on their way into LDS.
  // bf16 caches: global -> LDS directly, one block ahead.  A wave-wide request fills 1 KiB = 4 key
  // rows (8 rows at HD = 64); wave w takes rows 4 w .. 4 w + 3 of every group of 16, so (row & 15) = 4 w + lane / 16 is
  // fixed per lane and the chunk it must fetch for its slot is too.
  // fp32 caches: through registers (converted on the way), one block in registers while the
  // previous one is being read: chunk ci = tid + 256 i (i < 4) is (key ci / 16, dims 8 (ci % 16) ..).
  // Rows past the filled part of the cache repeat its last row (finite values; those keys are masked).
  constexpr bool kDma = sizeof(CacheT) == 2;
  constexpr int kReqRows = 1024 / RB;  // key rows of one wave-wide request: 4 (HD = 128) or 8
  const int krow = kReqRows * wave + lane / C, slot = lane % C;
  const uint32_t k_chunk = (uint32_t)(slot ^ (krow & (C - 1)));
  const uint32_t v_chunk = (uint32_t)((((slot >> 1) ^ (krow & (TT - 1))) << 1) | (slot & 1));
  // part i (0 .. KS - 1) of block jblk: this wave's kReqRows key rows and value rows of the i-th group of 4 * kReqRows
  auto issue_dma = [&](int jblk, int i) {
    const int kb0 = jblk * kPfBK;
    const uint32_t stage = lds0 + (uint32_t)((jblk & 1) * 2 * kPfTileBytes);
    const uint32_t k_to = stage + (uint32_t)((wave + 4 * i) * 1024), v_to = k_to + (uint32_t)kPfTileBytes;
    if (kb0 + kPfBK <= kv_len) {
      const size_t row0 = (size_t)(kb0 + 4 * kReqRows * i) * RB;
      dma16(reinterpret_cast<const char*>(kbase) + row0, (uint32_t)(krow * RB) + k_chunk * 16u, k_to);
      dma16(reinterpret_cast<const char*>(vbase) + row0, (uint32_t)(krow * RB) + v_chunk * 16u, v_to);
    } else {
      const uint32_t row = (uint32_t)min(kb0 + 4 * kReqRows * i + krow, kv_len - 1) * (uint32_t)RB;
      dma16(kbase, row + k_chunk * 16u, k_to);
      dma16(vbase, row + v_chunk * 16u, v_to);
    }
  };
  typedef decltype(load8_raw(kbase)) raw8_t;
  constexpr int kRegParts = kDma ? 0 : kPfBK * C / 256;  // 16-byte chunks of a block per thread: 4 (HD = 128) or 2
  raw8_t kraw[kDma ? 1 : kRegParts], vraw[kDma ? 1 : kRegParts];
  uint32_t k_st[kDma ? 1 : kRegParts], v_st[kDma ? 1 : kRegParts];
  auto fetch = [&](int kb0) {
#pragma unroll
    for (int i = 0; i < kRegParts; ++i) {
      const int ci = threadIdx.x + 256 * i;
      const size_t at = (size_t)min(kb0 + ci / C, kv_len - 1) * kPfHD + 8 * (ci % C);
      kraw[i] = load8_raw(kbase + at);
      vraw[i] = load8_raw(vbase + at);
    }
  };
#pragma unroll
  for (int i = 0; i < kRegParts; ++i) {
    const int ci = threadIdx.x + 256 * i, k = ci / C, c = ci % C;
    k_st[i] = (uint32_t)(k * RB + 16 * (c ^ (k & (C - 1))));
    v_st[i] = (uint32_t)(kPfTileBytes + k * RB + 16 * ((((c >> 1) ^ (k & (TT - 1))) << 1) | (c & 1)));
  }
  auto lay_down = [&](int stage) {
#pragma unroll
    for (int i = 0; i < kRegParts; ++i) {
      *reinterpret_cast<u32x4_t*>(lds + stage * 2 * kPfTileBytes + k_st[i]) = to_bf16x8(kraw[i]);
      *reinterpret_cast<u32x4_t*>(lds + stage * 2 * kPfTileBytes + v_st[i]) = to_bf16x8(vraw[i]);
    }
  };
  // ---- LDS read addresses (of the stage being read; flipped to the other stage after every block).
  // key fragment (tile jb, k-step s): row 16 jb + r, chunk 4 s + g  ->  (16 jb + r) * 256 + 16 * ((4 s + g) ^ r)
  uint32_t k_rd[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) k_rd[s] = lds0 + (uint32_t)(r * RB + 16 * ((4 * s + g) ^ (r & (C - 1))));
  // value fragment (half hf, slots 4 w2 .. 4 w2 + 3, dims 16 t ..): this lane addresses 8 bytes of key
  // 32 hf + 16 w2 + 4 g + (r >> 2): piece (r & 3) of the 32-byte segment t, which sits in slot t ^ (key & 7)
  const int vkey = 4 * g + (r >> 2);  // (16 w2 and 32 hf do not change key & 7)
  uint32_t v_rd[TT];
#pragma unroll
  for (int t = 0; t < TT; ++t)
    v_rd[t] = lds0 + (uint32_t)(kPfTileBytes + vkey * RB + 32 * (t ^ (vkey & (TT - 1))) + 8 * (r & 3));

  if (kDma) {
#pragma unroll
    for (int i = 0; i < KS; ++i) issue_dma(0, i);
  } else {
    fetch(0);
    lay_down(0);
    if (nblk > 1) fetch(kPfBK);
  }
  // ---- (after the first block's requests, so that both round trips to memory overlap)
  // Q fragments of the wave's two groups of 16 rows: Q[qrow][32 s + 8 g .. + 8), scaled, bf16.
  // Group u of wave w holds rows q0 + 32 w + 16 u .. + 15; this lane's row of it is qrow[u].
  int qrow[2], q_pos[2];
  u32x4_t qf[2][KS];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    qrow[u] = q0 + 32 * wave + 16 * u + r;
    q_pos[u] = start + qrow[u];
    const float* qp = q + ((size_t)bh * T + min(qrow[u], T - 1)) * kPfHD + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float4 a = reinterpret_cast<const float4*>(qp + 32 * s)[0], c = reinterpret_cast<const float4*>(qp + 32 * s)[1];
      const float v[8] = {a.x * qscale, a.y * qscale, a.z * qscale, a.w * qscale,
                          c.x * qscale, c.y * qscale, c.z * qscale, c.w * qscale};
      qf[u][s] = pack8_bf16(v);
    }
  }
  if (kDma || kWait) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int j = 0; j < nblk; ++j) {
    // One barrier per block: block j is complete in stage j & 1 (it landed before the previous
    // barrier); block j + 1 goes into the other stage, which was last read before that barrier
    // too (fp32 caches: from registers, while block j + 2 starts its flight from memory).
    const int kb0 = j * kPfBK;
    // bf16 caches: the requests for block j + 1 are issued between the products below (one part
    // per k-step), or here by a wave that has no products to form
    const bool more = j + 1 < nblk;
    if (more) {
      if (kDma) {
        if (kb0 > wave_last_pos) {
#pragma unroll
          for (int i = 0; i < KS; ++i) issue_dma(j + 1, i);
        }
      } else {
        lay_down((j + 1) & 1);
        if (j + 2 < nblk) fetch(kb0 + 2 * kPfBK);
      }
    }
    // a wave whose last query lies before the block has nothing to add
    if (kb0 <= wave_last_pos) {
      // ---- exponents of the four 16-key tiles: sc[u][jb][i] = S[qrow[u]][key kb0 + 16 jb + 4 g + i] - m_run[u]
      // (log2 units).  k-step outermost: the eight products of a step are independent, and a key
      // fragment is read once for both query groups.
      f32x4_t sc[2][4];
      u32x4_t ka[4];
#pragma unroll
      for (int jb = 0; jb < 4; ++jb) ka[jb] = pf_read128(k_rd[0] + (uint32_t)(jb * 16 * RB));
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        u32x4_t kn[4];
        if (kDma && s < KS - 1) {  // (the fp32 path has no registers to spare for a second set)
#pragma unroll
          for (int jb = 0; jb < 4; ++jb) kn[jb] = pf_read128(k_rd[s + 1] + (uint32_t)(jb * 16 * RB));
        }
#pragma unroll
        for (int jb = 0; jb < 4; ++jb)
#pragma unroll
          for (int u = 0; u < 2; ++u) sc[u][jb] = mfma16(ka[jb], qf[u][s], s == 0 ? negm[u] : sc[u][jb]);
        if (kDma && more) issue_dma(j + 1, s);
        if (s < KS - 1) {
#pragma unroll
          for (int jb = 0; jb < 4; ++jb) ka[jb] = kDma ? kn[jb] : pf_read128(k_rd[s + 1] + (uint32_t)(jb * 16 * RB));
        }
      }
      // only blocks that reach past the wave's first query position need the causal mask
      if (kb0 + kPfBK - 1 > wave_last_pos - 31) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int jb = 0; jb < 4; ++jb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (kb0 + 16 * jb + 4 * g + i > q_pos[u]) sc[u][jb][i] = -INFINITY;  // (also hides rows past kv_len)
      }
      // The reference point of a row moves only when an exponent has outgrown it by more than
      // kPfSlack (and on the first block, where it is still arbitrary).  One query group at a
      // time, so that only one group's exponents and probabilities are live together.
      u32x4_t pf[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float p[16], psum = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          p[e] = __builtin_amdgcn_exp2f(sc[u][e >> 2][e & 3]);  // v_exp_f32: underflow to 0 is what is wanted
          psum += p[e];
        }
        const bool revisit = j == 0 || psum > kPfTrigger;
        if (__builtin_amdgcn_ballot_w64(revisit) != 0) {
          float mx = -INFINITY;
#pragma unroll
          for (int e = 0; e < 16; ++e) mx = fmaxf(mx, sc[u][e >> 2][e & 3]);
          mx = quad_max(mx);
          const bool move = j == 0 || mx > kPfSlack;
          const float shift = move ? mx : 0.f;
          const float corr = (move && j != 0) ? __builtin_amdgcn_exp2f(-shift) : 1.0f;
          psum = 0.f;
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            p[e] = __builtin_amdgcn_exp2f(sc[u][e >> 2][e & 3] - shift);
            psum += p[e];
          }
          m_run[u] += shift;
          negm[u] = f32x4_t{-m_run[u], -m_run[u], -m_run[u], -m_run[u]};
          l_run[u] *= corr;
#pragma unroll
          for (int t = 0; t < TT; ++t) o[u][t] *= corr;
        }
        l_run[u] += psum;
        pf[u][0] = pack8_bf16(&p[0]);
        pf[u][1] = pack8_bf16(&p[8]);
      }
      // ---- O^T[hd 16 t + 4 g + i][qrow] += sum over the keys of each 32-key half; a value fragment
      // (two transposing reads: the half's first and second 16-key tile) meets both query groups.
      // The second half's fragments are requested as the first half's are consumed.
      constexpr int kRing = kDma ? (TT < 8 ? TT : 8) : 4;  // fragments in flight (the fp32 path has fewer registers to spare)
      auto v_lo = [&](int i) { return pf_read_tr(v_rd[i % TT] + (uint32_t)((i / TT) * 32 * RB)); };
      auto v_hi = [&](int i) { return pf_read_tr(v_rd[i % TT] + (uint32_t)((i / TT) * 32 * RB + 16 * RB)); };
      u32x2_t vlo[kRing], vhi[kRing];
#pragma unroll
      for (int i = 0; i < kRing; ++i) {
        vlo[i] = v_lo(i);
        vhi[i] = v_hi(i);
      }
#pragma unroll
      for (int i = 0; i < 2 * TT; ++i) {  // i = TT hf + t
        const u32x4_t vf = {vlo[i % kRing].x, vlo[i % kRing].y, vhi[i % kRing].x, vhi[i % kRing].y};
#pragma unroll
        for (int u = 0; u < 2; ++u) o[u][i % TT] = mfma16(vf, pf[u][i / TT], o[u][i % TT]);
        if (i + kRing < 2 * TT) {
          vlo[i % kRing] = v_lo(i + kRing);
          vhi[i % kRing] = v_hi(i + kRing);
        }
      }
    }
    // flip every read address to the other stage
#pragma unroll
    for (int s = 0; s < KS; ++s) k_rd[s] ^= (uint32_t)(2 * kPfTileBytes);
#pragma unroll
    for (int t = 0; t < TT; ++t) v_rd[t] ^= (uint32_t)(2 * kPfTileBytes);
    // the next block must have landed and every wave must be done with this one (fp32 caches: the block in registers may still be on its way, prefill_waits)
    if (kDma || kWait) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const float inv = 1.0f / quad_sum(l_run[u]);
    if (qrow[u] >= T) continue;
    const size_t at = ((size_t)b * T + qrow[u]) * ((size_t)H * kPfHD) + (size_t)h * kPfHD + 4 * g;
    if (out_bf16) {
      uint16_t* dst = reinterpret_cast<uint16_t*>(out) + at;
#pragma unroll
      for (int t = 0; t < TT; ++t)
        *reinterpret_cast<u32x2_t*>(dst + 16 * t) =
            u32x2_t{pack2_bf16(o[u][t][0] * inv, o[u][t][1] * inv), pack2_bf16(o[u][t][2] * inv, o[u][t][3] * inv)};
    } else {
      float* dst = reinterpret_cast<float*>(out) + at;
#pragma unroll
      for (int t = 0; t < TT; ++t)
        *reinterpret_cast<float4*>(dst + 16 * t) =
            float4{o[u][t][0] * inv, o[u][t][1] * inv, o[u][t][2] * inv, o[u][t][3] * inv};
    }
  }
}

// The first `rows8` groups of eight elements of every (b, hk) of both fp32 caches (pitch `stride` elements), rounded to bf16 as the kernel
// above does it and packed.  A thread eight elements, the caches in blockIdx.y; bounded by HBM (4 x 8 heads x 2048 rows of 128: 101 MB).
__global__ __launch_bounds__(256) void caches_to_bf16_kernel(const float* __restrict__ k, const float* __restrict__ v, uint16_t* __restrict__ kb,
                                                             uint16_t* __restrict__ vb, long long rows8, long long stride, long long groups8) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= groups8) return;
  const float* from = (blockIdx.y ? v : k) + i / rows8 * stride + i % rows8 * 8;
  *reinterpret_cast<u32x4_t*>((blockIdx.y ? vb : kb) + 8 * i) = to_bf16x8(load8_raw(from));
}

// bf16 caches.  The keys are walked in steps of 32.  Step t holds three things that need nothing of each other: the exponents of step t + 1, the
// softmax of step t, and the values of step t - 1 times their probabilities; they are laid out in HD / 16 pieces of two MFMAs of either product, their
// share of the exponentials and sums, and the fragments three pieces ahead, in that order for good (sched_barrier): a wave has MFMAs and
// vector work to issue side by side instead of one after the other, and two waves per SIMD fill what is left.  Before, each wave went through
// product, softmax and product in turn and a CU's two workgroups overlapped by chance: 3440 cycles per 64 keys and two waves, 2730 now (64 MFMAs a
// wave are 2048).  What bounds it is the clock (2.19 -> 1.95 GHz as the matrix pipes fill).  B = 4, 32 / 8 heads, T = 2048: 164 -> 152 us alone, 171 -> 155
// in a row; a few short grids, where a wave's own length counts: 0.79 .. 0.9 of the time.
//
// Keys run a step ahead of the values, so key block j + 2 and value block j + 1 are asked for in the second step of block j, behind the one
// barrier per block: every wave has consumed what lay there (keys of block j, values of block j - 1), and what it
// reads next (keys j + 1, values j) was asked for a block before and waited for in front of that barrier.
// Four steps at places known to the compiler make the body; a wave's last ones (masked, or with blocks cut short) go one by one.
//
// prefill_in_steps: which bf16 calls it takes (figures: its time over attn_prefill_kernel's).  Heads of 128 but for a few of up to 256 keys: a last block
// that is more than half full is two masked steps there, which counts while a few rows behind others are all there is to do (1.04 .. 1.08; less than
// half full 0.98) and while a CU's two workgroups finish together (257 .. 512 of 33 .. 128 keys: 1.03 .. 1.10); 9300 other shapes 0.975, the most 1.07.  Narrower ones have
// few MFMAs in a step beside its latency, so short prompts are faster in whole blocks: 64 columns 1.03 .. 1.09 at 40 .. 64 keys, 0.99 / 1.09 at 100, 1.03 at
// 192, 1.00 at 256, 0.93 at 512, 0.79 at 4096 with few workgroups; with more than a round of them from 128 on (200 keys: 0.98), over 194 shapes 0.93 (left: 1.05 where rounds come
// out even, 1024 workgroups of 4096 queries).  32 columns: 1.04 ..
// 1.10 up to 256, 0.985 at 333, 0.96 at 512 and 0.83 at 4096 while two workgroups a CU hold the launch; beyond, the exponentials bound both and the
// steps' share of vector work is the larger (768 workgroups and more: 1.01 .. 1.05; 384 of 312 queries 1.04, 512 of 900 0.91).
__host__ __device__ inline bool prefill_in_steps(long long heads, int T, int start, int head_dim) {
  const long long workgroups = heads * ((T + kPfBQ - 1) / kPfBQ), keys = (long long)start + T;
  if (head_dim == 128) {
    if (keys <= 32 || keys > 256) return true;
    if (workgroups <= 256) return T > 64 || start == 0 || ((keys - 1) & 32) == 0;
    return workgroups > 512 || T <= 32 || keys > 128;
  }
  if (head_dim == 64) return keys >= 256 || (keys > 128 && workgroups > 256);
  return keys > 320 && (workgroups <= 256 || (workgroups <= 512 && T >= 600));
}
template <int HD>
__global__ __launch_bounds__(256, 2) void attn_prefill_steps_kernel(const float* __restrict__ q, const uint16_t* __restrict__ kcache,
                                                                 const uint16_t* __restrict__ vcache, int H, int Hkv, int T,
                                                                 int start, int max_len, void* __restrict__ out, int out_bf16) {
  static_assert(HD == 128 || HD == 64 || HD == 32, "head_dim 128, 64 or 32");
  // bytes of a row, 16-byte chunks of it, k-steps of the first product (and a wave's requests per tile), 16-dim output tiles
  constexpr int RB = 2 * HD, C = HD / 8, KS = HD / 32, TT = HD / 16, U = 2, kAhead = 3;
  constexpr int kTile = kPfBK * RB;  // LDS: two stages of a key tile and a value tile, laid out as below
  __shared__ __attribute__((aligned(1024))) unsigned char lds[4 * kTile];
  const uint32_t lds0 = (uint32_t)(uintptr_t)(pf_lds_char_t*)lds;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  // (work order: see attn_prefill_kernel)
  const int qblocks = (T + kPfBQ - 1) / kPfBQ;
  const int BH = (int)(gridDim.x / (unsigned)qblocks);
  int qb, bh;
  if ((BH & 7) == 0) {
    const int per_xcd = BH >> 3, m = (int)(blockIdx.x >> 3);
    qb = qblocks - 1 - m / per_xcd;
    bh = (int)(blockIdx.x & 7) * per_xcd + m % per_xcd;
  } else {
    qb = qblocks - 1 - (int)blockIdx.x / BH;
    bh = (int)blockIdx.x % BH;
  }
  const int b = bh / H, h = bh % H, hk = h / (H / Hkv);
  const int q0 = qb * kPfBQ;
  const float qscale = 1.4426950408889634f * (HD == 128 ? 0.08838834764831845f : HD == 64 ? 0.125f : 0.17677669529663687f);
  const uint16_t* kbase = kcache + ((size_t)b * Hkv + hk) * max_len * HD;
  const uint16_t* vbase = vcache + ((size_t)b * Hkv + hk) * max_len * HD;
  const int kv_len = start + T;
  const int kv_end = min(kv_len, start + q0 + kPfBQ);
  const int nblk = (kv_end + kPfBK - 1) / kPfBK;
  const int wave_first = q0 + 16 * U * wave;
  const int first_pos = start + wave_first;                                   // of this wave's queries
  const int steps = wave_first < T ? (min(first_pos + 16 * U - 1, kv_len - 1) >> 5) + 1 : 0;  // of 32 keys each
  float m_run[U] = {}, l_run[U] = {};
  f32x4_t negm[U] = {};
  f32x4_t o[U][TT];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int t = 0; t < TT; ++t) o[u][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // ---- requests: 1 KiB of rows each, global -> LDS; wave w takes rows kReqRows w .. of every group of 4 kReqRows, so the chunk that belongs in a lane's
  // slot is the same for all of them.  Rows past the filled part of the cache repeat its last row (finite values; those keys are masked).
  constexpr int kReqRows = 1024 / RB;
  const int krow = kReqRows * wave + lane / C, slot = lane % C;
  const uint32_t k_chunk = (uint32_t)(slot ^ (krow & (C - 1))) * 16u;
  const uint32_t v_chunk = (uint32_t)((((slot >> 1) ^ (krow & (TT - 1))) << 1) | (slot & 1)) * 16u;
  const uint32_t k_lane = (uint32_t)(krow * RB) + k_chunk, v_lane = (uint32_t)(krow * RB) + v_chunk;
  auto place = [&](bool values, int i, int stage) __attribute__((always_inline)) {
    return lds0 + (uint32_t)(stage * 2 * kTile + (values ? kTile : 0) + (wave + 4 * i) * 1024);
  };
  auto request = [&](int j, bool values) __attribute__((always_inline)) {  // of block j < nblk
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const uint32_t row = (uint32_t)min(4 * kReqRows * i + krow, kv_len - 1 - j * kPfBK) * (uint32_t)RB;
      dma16(reinterpret_cast<const char*>(values ? vbase : kbase) + (size_t)j * kPfBK * RB, row + (values ? v_chunk : k_chunk), place(values, i, j & 1));
    }
  };
  // ---- LDS read addresses within stage 0 (fragments and their places: see attn_prefill_kernel)
  uint32_t k_rd[KS], v_rd[TT];
#pragma unroll
  for (int s = 0; s < KS; ++s) k_rd[s] = lds0 + (uint32_t)(r * RB + 16 * ((4 * s + g) ^ (r & (C - 1))));
  const int vkey = 4 * g + (r >> 2);
#pragma unroll
  for (int t = 0; t < TT; ++t) v_rd[t] = lds0 + (uint32_t)(kTile + vkey * RB + 32 * (t ^ (vkey & (TT - 1))) + 8 * (r & 3));

  request(0, false);
  request(0, true);
  int q_pos[U];
  u32x4_t qf[U][KS];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int row = wave_first + 16 * u + r;
    q_pos[u] = start + row;
    const float* qp = q + ((size_t)bh * T + min(row, T - 1)) * HD + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const float4 a = reinterpret_cast<const float4*>(qp + 32 * s)[0], c = reinterpret_cast<const float4*>(qp + 32 * s)[1];
      const float v[8] = {a.x * qscale, a.y * qscale, a.z * qscale, a.w * qscale, c.x * qscale, c.y * qscale, c.z * qscale, c.w * qscale};
      qf[u][s] = pack8_bf16(v);
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" : "+v"(qf[u][s]));
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (nblk > 1) request(1, false);
  turn_barrier();
  f32x4_t sn[U][2];  // exponents of the step ahead
  u32x4_t pf[U];     // probabilities of the step behind
  auto key_frag = [&](int at, int i) __attribute__((always_inline)) { return pf_read128(k_rd[i >> 1] + (uint32_t)(at + (i & 1) * 16 * RB)); };
  auto score = [&](const u32x4_t& kf, int i) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u) sn[u][i & 1] = mfma16(kf, qf[u][i >> 1], i < 2 ? negm[u] : sn[u][i & 1]);
  };
  // Step t: exponents from the keys at k_at, values at v_at (kV: not in the very first, which takes its reference points instead), and req(piece)
  auto step = [&](int t, auto values, auto masked, int k_at, int v_at, auto req) __attribute__((always_inline)) {
    constexpr bool kV = decltype(values)::value;
    f32x4_t sc[U][2];
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) sc[u][jb] = sn[u][jb];
    u32x4_t kf[TT];
    u32x2_t vl[TT], vh[TT];
    auto fetch = [&](int i) __attribute__((always_inline)) {
      kf[i] = key_frag(k_at, i);
      if (kV) {
        vl[i] = pf_read_tr(v_rd[i] + (uint32_t)v_at);
        vh[i] = pf_read_tr(v_rd[i] + (uint32_t)(v_at + 16 * RB));
      }
    };
#pragma unroll
    for (int i = 0; i < (kAhead < TT ? kAhead : TT); ++i) fetch(i);
    if (decltype(masked)::value && 32 * t + 31 > first_pos) {
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int jb = 0; jb < 2; ++jb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (32 * t + 16 * jb + 4 * g + i > q_pos[u]) sc[u][jb][i] = -INFINITY;
    }
    u32x4_t pn[U];
    float p[U][8], psum[U] = {};
    constexpr int kPer = 8 * U / TT;  // exponentials of a piece
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      if (i + kAhead < TT) fetch(i + kAhead);
      req(i);
      score(kf[i], i);
#pragma unroll
      for (int x = 0; x < kPer; ++x) {
        const int u = (i * kPer + x) >> 3, e = (i * kPer + x) & 7;
        p[u][e] = __builtin_amdgcn_exp2f(sc[u][e >> 2][e & 3]);
        psum[u] += p[u][e];
      }
      if (U * (i + 1) % TT == 0) {  // a group of rows is through (pinned: the compiler would sink it behind the branches below)
        const int u = U * i / TT;
        pn[u] = pack8_bf16(p[u]);
        asm volatile("" : "+v"(pn[u]), "+v"(psum[u]));
      }
      if (kV) {
        const u32x4_t vf = {vl[i].x, vl[i].y, vh[i].x, vh[i].y};
#pragma unroll
        for (int u = 0; u < U; ++u) o[u][i] = mfma16(vf, pf[u], o[u][i]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool revisit = !kV || psum[u] > kPfTrigger;
      if (!kV || __builtin_amdgcn_ballot_w64(revisit) != 0) {
        float mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < 8; ++e) mx = fmaxf(mx, sc[u][e >> 2][e & 3]);
        if (!kV)  // the first reference point is that of the whole first block
#pragma unroll
          for (int e = 0; e < 8; ++e) mx = fmaxf(mx, 32 + 16 * (e >> 2) + 4 * g + (e & 3) > q_pos[u] ? -INFINITY : sn[u][e >> 2][e & 3]);
        mx = quad_max(mx);
        const bool move = !kV || mx > kPfSlack;
        const float shift = move ? mx : 0.f;
        const float corr = (move && kV) ? __builtin_amdgcn_exp2f(-shift) : 1.0f;
        psum[u] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p[u][e] = __builtin_amdgcn_exp2f(sc[u][e >> 2][e & 3] - shift);
          psum[u] += p[u][e];
        }
        pn[u] = pack8_bf16(p[u]);
        m_run[u] += shift;
        negm[u] = f32x4_t{-m_run[u], -m_run[u], -m_run[u], -m_run[u]};
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) sn[u][jb] -= shift;  // (began at the old reference point)
        if (kV) {
          l_run[u] *= corr;
#pragma unroll
          for (int tt = 0; tt < TT; ++tt) o[u][tt] *= corr;
        }
      }
      l_run[u] += psum[u];
      pf[u] = pn[u];
    }
  };
  auto last_values = [&](int v_at) __attribute__((always_inline)) {
    u32x2_t vl[TT], vh[TT];
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      vl[i] = pf_read_tr(v_rd[i] + (uint32_t)v_at);
      vh[i] = pf_read_tr(v_rd[i] + (uint32_t)(v_at + 16 * RB));
    }
#pragma unroll
    for (int i = 0; i < TT; ++i) {
      const u32x4_t vf = {vl[i].x, vl[i].y, vh[i].x, vh[i].y};
#pragma unroll
      for (int u = 0; u < U; ++u) o[u][i] = mfma16(vf, pf[u], o[u][i]);
    }
  };
  constexpr std::integral_constant<bool, true> yes{};
  constexpr std::integral_constant<bool, false> no{};
  auto none = [](int) {};
  if (steps > 0) {
    u32x4_t kf[TT];
#pragma unroll
    for (int i = 0; i < TT; ++i) kf[i] = key_frag(0, i);
#pragma unroll
    for (int i = 0; i < TT; ++i) score(kf[i], i);
    step(0, no, yes, 32 * RB, 0, none);
  }
  // blocks j (even) and j + 1: the second step of j, both of j + 1, the first of j + 2
  int j = 0;
  const char* k_from = reinterpret_cast<const char*>(kbase) + 2 * kPfBK * RB;
  const char* v_from = reinterpret_cast<const char*>(vbase) + kPfBK * RB;
  for (; 2 * j + 5 < steps && 64 * j + 159 <= first_pos && (j + 4) * kPfBK <= kv_end; j += 2) {
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      turn_barrier();
      step(2 * j + 2 * x + 1, yes, no, (x ^ 1) * 2 * kTile, x * 2 * kTile, [&](int i) __attribute__((always_inline)) {
        if (i < KS) dma16(k_from + i * 4096, k_lane, place(false, i, x));
        else dma16(v_from + (i - KS) * 4096, v_lane, place(true, i - KS, x ^ 1));
      });
      k_from += kPfBK * RB;
      v_from += kPfBK * RB;
      step(2 * j + 2 * x + 2, yes, no, (x ^ 1) * 2 * kTile + 32 * RB, x * 2 * kTile + 32 * RB, none);
    }
  }
  for (int t = 2 * j + 1; t < 2 * nblk; ++t) {
    const int block = t >> 1;
    if (t & 1) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      turn_barrier();
      if (block + 2 < nblk) request(block + 2, false);
      if (block + 1 < nblk) request(block + 1, true);
    }
    auto half = [&](int n) { return ((n >> 1) & 1) * 2 * kTile + (n & 1) * 32 * RB; };  // where step n's keys (values) lie
    // (the last step's exponents of the one behind it are of no use, whatever lies there)
    if (t < steps) step(t, yes, yes, half(t + 1), half(t - 1), none);
    else if (t == steps) last_values(half(t - 1));
  }
  if (steps == 2 * nblk) last_values(((nblk - 1) & 1) * 2 * kTile + 32 * RB);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const float inv = 1.0f / quad_sum(l_run[u]);
    const int row = wave_first + 16 * u + r;
    if (row >= T) continue;
    const size_t at = ((size_t)b * T + row) * ((size_t)H * HD) + (size_t)h * HD + 4 * g;
    if (out_bf16) {
      uint16_t* dst = reinterpret_cast<uint16_t*>(out) + at;
#pragma unroll
      for (int t = 0; t < TT; ++t)
        *reinterpret_cast<u32x2_t*>(dst + 16 * t) =
            u32x2_t{pack2_bf16(o[u][t][0] * inv, o[u][t][1] * inv), pack2_bf16(o[u][t][2] * inv, o[u][t][3] * inv)};
    } else {
      float* dst = reinterpret_cast<float*>(out) + at;
#pragma unroll
      for (int t = 0; t < TT; ++t)
        *reinterpret_cast<float4*>(dst + 16 * t) = float4{o[u][t][0] * inv, o[u][t][1] * inv, o[u][t][2] * inv, o[u][t][3] * inv};
    }
  }
}

}  // namespace ajq
