// Grouped-query attention whose values are the projected keys: the row operators around it.  (The attention itself is
// latent_attention.h's: windowed_prefill_kernel / windowed_attention_kernel for prompts and any width, latent_decode_kernel
// for one token, to which a key/value head is a "sequence" and its query heads are the heads.)
//
// A cache row of one key/value head is (value | key), dimp columns each: the key as projected, and the same key normed and
// rotated.
#pragma once
#include "dense_gemv_kernels.h"

namespace ajq {

// cos and sin of position * half_turns[i] * pi for i < pairs, by the threads of a workgroup.  The product and its reduction
// to (-1, 1] half turns are double, so that any position has an angle that is exact to fp32.
__device__ __forceinline__ void angles(const double* __restrict__ half_turns, int pairs, int position, float* cosine, float* sine) {
  for (int i = threadIdx.x; i < pairs; i += blockDim.x) {
    const double a = (double)position * half_turns[i];
    sincospif((float)(a - 2.0 * rint(0.5 * a)), sine + i, cosine + i);
  }
}

struct KeyValueShape {
  int heads, groups, dim, dimp, rot;  // rot <= dim, the first dimensions of a head; component i pairs with i + rot / 2
  float eps;
};

// One head of a projection row, normed over dim and rotated, of any width and with any pairs, by a team of LPH lanes: four columns
// per lane and turn, through put(column, values); columns dim .. dimp are zero and stay so (the gain is zero there).
template <int LPH, typename Y, typename Put>
__device__ __forceinline__ void norm_rotate(const Y* __restrict__ src, const KeyValueShape& s, const float* __restrict__ gain,
                                            const float* cosine, const float* sine, int lane, Put&& put) {
  float ss = 0.f;
  for (int i = 4 * lane; i < s.dimp; i += 4 * LPH) {
    const float4 v = load4(src + i);
    ss += (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
  }
#pragma unroll
  for (int off = LPH / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
  const Divisor by(sqrtf(ss / (float)s.dim + s.eps));
  const int half = s.rot >> 1;
  auto one = [&](int i) { return by.divide(to_f32(src[i])) * gain[i]; };
  auto turned = [&](int i) {
    if (i >= s.rot) return one(i);
    if (i < half) return one(i) * cosine[i] - one(i + half) * sine[i];
    return one(i) * cosine[i - half] + one(i - half) * sine[i - half];
  };
  for (int i = 4 * lane; i < s.dimp; i += 4 * LPH) put(i, float4{turned(i), turned(i + 1), turned(i + 2), turned(i + 3)});
}

// four normed columns, turned against those half the rotated width away: v, w over the norm, times gains and (cos, -+ sin)
__device__ __forceinline__ float4 turned_quad(const float4& v, const float4& w, const Divisor& by, const float4& g, const float4& h, const float4& c,
                                              const float4& d) {
  return float4{by.divide(v.x) * g.x * c.x + by.divide(w.x) * h.x * d.x, by.divide(v.y) * g.y * c.y + by.divide(w.y) * h.y * d.y,
                by.divide(v.z) * g.z * c.z + by.divide(w.z) * h.z * d.z, by.divide(v.w) * g.w * c.w + by.divide(w.w) * h.w * d.w};
}

struct KeyValueSplit {
  const void* y;            // [M, ldy]: queries (heads x dimp), keys (groups x dimp), then whatever else
  int ldy;
  KeyValueShape s;
  const float *q_gain, *k_gain;  // [dimp]
  const double* half_turns; // [rot / 2]
  int start;                // position of the first token, or
  const long long* pos;     // device-side position (seq = 1): the row goes to its slot of a ring
  int seq, prior, cap, kept;
  void* q;                  // [M, heads, q_ld], the query from column q_at on, zeros ahead of it
  int q_ld, q_at;
  void* rows;               // row slot of (b, group) at b * rows_batch + group * rows_head + slot * 2 dimp
  long long rows_batch, rows_head;
};
// Grid (tokens, slices): the heads of a token are dealt to the teams of LPH lanes of its workgroups.  QUADS: four columns per lane
// hold a head, and its pairs too (dimp <= 4 LPH, half the rotated width a multiple of 4): a head is read once, the first one
// before the angles are known, every other one ahead of the arithmetic of the one before; gains and angles stay in registers.
template <typename Y, typename T, int LPH, bool QUADS>
__global__ __launch_bounds__(256) void key_value_split_kernel(KeyValueSplit a) {
  extern __shared__ __attribute__((aligned(16))) float trig[];
  constexpr int kTeams = 256 / LPH;
  const KeyValueShape s = a.s;
  const int m = blockIdx.x, b = m / a.seq, t = m % a.seq;
  const int half = s.rot >> 1, pitch = (half + 3) & ~3, all = s.heads + s.groups, stride = kTeams * gridDim.y;
  const int p = clamped_position(a.pos, a.start + t, 0x7FFFFFFF);
  const int slot = a.pos ? ring_slot(p, a.cap, a.kept) : a.prior + t;
  const int lane = threadIdx.x % LPH, first = kTeams * blockIdx.y + threadIdx.x / LPH;
  const Y* row = reinterpret_cast<const Y*>(a.y) + (size_t)m * a.ldy;
  auto query = [&](int n) { return reinterpret_cast<T*>(a.q) + ((size_t)m * s.heads + n) * a.q_ld; };
  auto key = [&](int n) {
    return reinterpret_cast<T*>(a.rows) + (size_t)b * a.rows_batch + (size_t)(n - s.heads) * a.rows_head + (size_t)slot * (2 * s.dimp);
  };
  if constexpr (QUADS) {
    const float4 zero = float4{0.f, 0.f, 0.f, 0.f};
    const int i = 4 * lane, o = i < half ? i + half : i - half, e = i < half ? i : o;
    const bool mine = i < s.dimp, pairs = mine && i < s.rot;
    auto read = [&](int n, float4& v, float4& w) {
      v = w = zero;
      if (n < all && mine) v = load4(row + n * s.dimp + i);
      if (n < all && pairs) w = load4(row + n * s.dimp + o);
    };
    float4 v, w, gq = zero, hq = zero, gk = zero, hk = zero, c = float4{1.f, 1.f, 1.f, 1.f}, d = zero;
    read(first, v, w);
    if (mine) { gq = load4(a.q_gain + i); gk = load4(a.k_gain + i); }
    if (pairs) { hq = load4(a.q_gain + o); hk = load4(a.k_gain + o); }
    angles(a.half_turns, half, p, trig, trig + pitch);
    __syncthreads();
    if (pairs) {
      c = load4(trig + e);
      d = load4(trig + pitch + e);
      if (i < half) d = float4{-d.x, -d.y, -d.z, -d.w};
    }
    for (int n = first; n < all; n += stride) {
      float4 nv, nw;
      read(n + stride, nv, nw);
      float ss = (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w);
#pragma unroll
      for (int off = LPH / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
      const Divisor by(sqrtf(ss / (float)s.dim + s.eps));
      const bool is_query = n < s.heads;
      const float4 out = turned_quad(v, w, by, is_query ? gq : gk, is_query ? hq : hk, c, d);
      if (is_query) {
        T* dst = query(n);
        for (int k = i; k < a.q_at; k += 4 * LPH) store4(dst + k, zero);
        if (mine) store4(dst + a.q_at + i, out);
      } else if (mine) {
        T* dst = key(n);
        store4(dst + i, v);
        store4(dst + s.dimp + i, out);
      }
      v = nv;
      w = nw;
    }
  } else {
    angles(a.half_turns, half, p, trig, trig + pitch);
    __syncthreads();
    for (int n = first; n < all; n += stride) {
      const Y* src = row + n * s.dimp;
      if (n < s.heads) {
        T* dst = query(n);
        for (int i = 4 * lane; i < a.q_at; i += 4 * LPH) store4(dst + i, float4{0.f, 0.f, 0.f, 0.f});
        norm_rotate<LPH>(src, s, a.q_gain, trig, trig + pitch, lane, [&](int i, float4 v) { store4(dst + a.q_at + i, v); });
      } else {
        T* dst = key(n);
        for (int i = 4 * lane; i < s.dimp; i += 4 * LPH) store4(dst + i, load4(src + i));
        norm_rotate<LPH>(src, s, a.k_gain, trig, trig + pitch, lane, [&](int i, float4 v) { store4(dst + s.dimp + i, v); });
      }
    }
  }
}

// key_value_split_kernel's one token per sequence at the front of the decode attention: every chunk's workgroup makes its key/value
// head's queries from the projection row (as four columns per lane, so half the rotated width is a multiple of 4), and the one whose
// rows hold the token's slot makes the new row too, writes it to the ring and lays it over what its block brought from there.
// The rows and gains are requested ahead of the position, waited for, then the block's requests go out and the norms, the angles
// and the turns run beside them.  A workgroup holds the 16 heads of one key/value head at most.  Launch and latency bound: what
// it replaces is a launch of 20 rows of arithmetic.  16 heads of 128 on 4 rings of 1028 rows, both launches -> this one: 1
// sequence 7.0 -> 5.2 us, 4: 9.0 -> 6.6, 16: 13.9 -> 10.8, 64: 28.2 -> 25.5; 98 shapes: 0.78, the most 0.93.
__device__ __forceinline__ void pin(float4& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }
struct GroupRow {
  const float* y;           // [B, ldy]: queries (groups x share x dimp), keys (groups x dimp), ..
  const float *q_gain, *k_gain;
  const double* half_turns;
  int ldy, groups, dim, rot, kept;
  float eps;
};
constexpr int kGroupShare = 16;
template <int KS>
struct GroupFront {
  static constexpr bool kMakesRow = true;
  static constexpr int kDim = 16 * KS, kLanes = kDim <= 64 ? 16 : kDim <= 128 ? 32 : 64, kTeams = 256 / kLanes;  // lanes a head, heads at once
  static constexpr int kTurns = (kGroupShare + kTeams) / kTeams, kLd = kDim + 8;
  struct Lds {
    float trig[2][kDim / 2];
    __attribute__((aligned(16))) uint16_t q[kGroupShare][kLd], row[2 * kDim];
  };
  const GroupRow k;
  Lds& lds;
  float4 v[kTurns], w[kTurns], gq, hq, gk, hk;
  double half_turn;
  int slot, unit;
  __device__ __forceinline__ GroupFront(const GroupRow& k, Lds& lds) : k(k), lds(lds) {}
  __device__ __forceinline__ void request(const LatentDecode& a, int of, int, u32x4_t (&)[KS]) {
    unit = of;
    const int dimp = a.rankp, half = k.rot >> 1, i = 4 * (threadIdx.x % kLanes), team = threadIdx.x / kLanes;
    const int at = min(i, dimp - 4), other = i >= k.rot ? at : i < half ? i + half : i - half;
    const float* row = k.y + (size_t)(unit / k.groups) * k.ldy;
    const int group = unit % k.groups;
#pragma unroll
    for (int t = 0; t < kTurns; ++t)
      if (kTeams * t <= a.heads) {
        const int n = min(team + kTeams * t, a.heads);
        const float* src = row + (n < a.heads ? group * a.heads + n : k.groups * a.heads + group) * dimp;
        v[t] = load4(src + at);
        w[t] = load4(src + other);
      }
    gq = load4(k.q_gain + at); hq = load4(k.q_gain + other);
    gk = load4(k.k_gain + at); hk = load4(k.k_gain + other);
    half_turn = k.rot ? k.half_turns[min((int)threadIdx.x, half - 1)] : 0.0;
  }
  template <typename Fetch>
  __device__ __forceinline__ void ready(const LatentDecode& a, int position, int begin, int end, u32x4_t (&qf)[KS], Fetch&& fetch) {
    const int dimp = a.rankp, half = k.rot >> 1, lane = threadIdx.x % kLanes, i = 4 * lane, team = threadIdx.x / kLanes;
    const bool mine = i < dimp, pairs = i < k.rot;
    slot = ring_slot(position, a.cap, k.kept);
#pragma unroll
    for (int t = 0; t < kTurns; ++t) {
      pin(v[t]);
      pin(w[t]);
    }
    pin(gq); pin(hq); pin(gk); pin(hk);
    asm volatile("" : "+v"(half_turn));
    fetch();
    if ((int)threadIdx.x < half) {  // as `angles`
      const double x = (double)position * half_turn;
      sincospif((float)(x - 2.0 * rint(0.5 * x)), &lds.trig[1][threadIdx.x], &lds.trig[0][threadIdx.x]);
    }
    __syncthreads();
    const float4 zero = float4{0.f, 0.f, 0.f, 0.f};
    float4 c = float4{1.f, 1.f, 1.f, 1.f}, d = zero;
    if (pairs) {
      const int e = i < half ? i : i - half;
      c = load4(&lds.trig[0][e]);
      d = load4(&lds.trig[1][e]);
      if (i < half) d = float4{-d.x, -d.y, -d.z, -d.w};
    }
#pragma unroll
    for (int t = 0; t < kTurns; ++t) {
      const int n = team + kTeams * t;
      if (kTeams * t > a.heads) continue;
      const float4 own = mine ? v[t] : zero, far = pairs ? w[t] : zero;
      float ss = (own.x * own.x + own.y * own.y) + (own.z * own.z + own.w * own.w);
#pragma unroll
      for (int off = kLanes / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
      const Divisor by(sqrtf(ss / (float)k.dim + k.eps));
      const bool is_query = n < a.heads;
      const float4 out = turned_quad(own, far, by, is_query ? gq : gk, is_query ? hq : hk, c, d);
      if (mine && is_query) store4(&lds.q[n][i], out);
      if (mine && n == a.heads) {
        store4(lds.row + i, own);
        store4(lds.row + dimp + i, out);
      }
    }
    __syncthreads();
    const int r = threadIdx.x & 15, g = (threadIdx.x & 63) >> 4, first = dimp >> 3;  // (zeros ahead of the key's columns and past them)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int at = 4 * s + g;
      qf[s] = u32x4_t{0u, 0u, 0u, 0u};
      if (at >= first && at < 2 * first) qf[s] = *reinterpret_cast<const u32x4_t*>(&lds.q[min(r, a.heads - 1)][8 * (at - first)]);
    }
  }
  // the new row, in the block that brought its slot: over what lay there, and into the ring
  __device__ __forceinline__ void place(const LatentDecode& a, unsigned char* stages, int stage, int j0, int end) {
    if (slot < j0 || slot >= min(j0 + kLatentRows, end)) return;
    const int at = slot - j0, c = threadIdx.x;
    auto put = [&](int row, int c, const u32x4_t& piece) {
      *reinterpret_cast<u32x4_t*>(stages + stage + (c >> 3) * (kLatentRows * 128) + row * 128 + 16 * ((c & 7) ^ ((row & 6) | ((row >> 3) & 1)))) = piece;
    };
    // What lay in the slot may be no number, which a weight of zero does not silence: neither in the chunks past the width, which repeat
    // the row's last one, nor in the values of the rows past the end, which repeat the last row.
    if (c < 4 * KS) {
      const bool live = c < (a.width >> 3);
      const u32x4_t piece = live ? *reinterpret_cast<const u32x4_t*>(lds.row + 8 * c) : u32x4_t{0u, 0u, 0u, 0u};
      put(at, c, piece);
      if (live) *reinterpret_cast<u32x4_t*>(const_cast<uint16_t*>(a.ring) + ((size_t)unit * a.cap + slot) * a.width + 8 * c) = piece;
    }
    if (slot == end - 1 && (c & 63) < (a.rankp >> 3))
      for (int row = at + 1 + (c >> 6); row < kLatentRows; row += 4) put(row, c & 63, u32x4_t{0u, 0u, 0u, 0u});
    __syncthreads();
  }
};
template <int KS>
__global__ __launch_bounds__(256) void group_decode_kernel(LatentDecode a, GroupRow k) {
  __shared__ typename GroupFront<KS>::Lds lds;
  GroupFront<KS> front(k, lds);
  latent_decode<KS, (KS + 3) / 4, 1>(a, front);
}

// Merge of latent_decode_kernel's row chunks (a sequence there is a (b, key/value head) here) and the output gate:
// out[b, head, c] = sigmoid(gate) * sum over chunks.  One workgroup per (b, head).
struct GroupMerge {
  const float* sums;        // as latent_decode_kernel leaves them, for batch * groups sequences of `share` heads
  const float2* heads_in;   // [B * groups, share, chunks]
  const float* gate;        // [b * gate_ld + head * dimp + c] before the sigmoid, or null
  uint16_t* out;            // [B, out_ld], head h at column h * dimp
  int groups, share, chunks, dimp, gate_ld, out_ld;
};
__global__ __launch_bounds__(256) void group_merge_kernel(GroupMerge a) {
  __shared__ float weight[kLatentMaxChunks];
  __shared__ float4 part[256];
  const int tid = threadIdx.x, lane = tid & 63, heads = a.groups * a.share;
  const int b = blockIdx.x / heads, head = blockIdx.x % heads, h = head % a.share;
  const int unit = b * a.groups + head / a.share;
  const int quads = a.dimp >> 2, split = max(1, min(256 / quads, a.chunks)), which = tid / quads;
  // what the sums need from memory, before the chunks' weights are known: a launch is one round trip, not three
  const int c = 4 * (tid % quads);
  const float* src = a.sums + latent_sums_at(unit, h >> 4, 0, a.share, a.chunks, a.dimp) + 256 * (c >> 4) + 16 * (h & 15) + (c & 15);
  constexpr int kAhead = 4;
  float4 ahead[kAhead], z = float4{0.f, 0.f, 0.f, 0.f};
  auto request = [&](int s0) {
#pragma unroll
    for (int k = 0; k < kAhead; ++k) ahead[k] = load4(src + (size_t)min(s0 + k * split, a.chunks - 1) * (16 * a.dimp));
  };
  request(which);
  if (a.gate) z = load4(a.gate + (size_t)b * a.gate_ld + (size_t)head * a.dimp + c);
  if (tid < 64) {  // a lane per chunk
    const bool mine = lane < a.chunks;
    const float2 ml = mine ? a.heads_in[((size_t)unit * a.share + h) * a.chunks + lane] : float2{-INFINITY, 0.f};
    const float top = wave_max64(ml.x);
    const float e = ml.x == -INFINITY ? 0.f : exp2f(ml.x - top);
    const float total = wave_sum(ml.y * e);
    if (mine) weight[lane] = e / total;
  }
  __syncthreads();
  float4 sum = float4{0.f, 0.f, 0.f, 0.f};
  if (which < split) {
    for (int s0 = which; s0 < a.chunks; s0 += kAhead * split) {
      if (s0 > which) request(s0);
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        if (s0 + k * split >= a.chunks) break;
        const float4 v = ahead[k];
        const float f = weight[s0 + k * split];
        sum.x = fmaf(v.x, f, sum.x); sum.y = fmaf(v.y, f, sum.y); sum.z = fmaf(v.z, f, sum.z); sum.w = fmaf(v.w, f, sum.w);
      }
    }
  }
  part[tid] = sum;
  __syncthreads();
  if (which > 0) return;
  for (int o = 1; o < split; ++o) {
    const float4 v = part[tid + o * quads];
    sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
  }
  if (a.gate) {
    sum.x *= sigmoid_f32(z.x); sum.y *= sigmoid_f32(z.y); sum.z *= sigmoid_f32(z.z); sum.w *= sigmoid_f32(z.w);
  }
  store4(a.out + (size_t)b * a.out_ld + (size_t)head * a.dimp + c, sum);
}

}  // namespace ajq
