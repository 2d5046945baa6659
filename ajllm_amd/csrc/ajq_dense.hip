// C ABI of libajq_dense.so (include/ajq_dense.h): argument validation, launch geometry, error reporting.
#include <algorithm>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>

#include "../../include/ajq_dense.h"
#include "ajq_common.h"
#include "dense_gemm_kernels.h"
#include "dense_kernels.h"
#include "latent_attention.h"
#include "dense_gemv_kernels.h"
#include "grouped_attention.h"
#include "scan_kernels.h"
#include "stream_kernels.h"

using namespace ajq;

namespace {

thread_local char g_error[512] = "";

int fail(int status, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
  return status;
}
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
bool known(int dtype) { return dtype == AJQD_BF16 || dtype == AJQD_F32; }
int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(AJQ_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
  return AJQ_OK;
}
const long long* positions64(const int64_t* p) { return reinterpret_cast<const long long*>(p); }

// Calls fn(T{}, U{}) for the element types of two dtype flags.
template <typename F>
void with_types(int a, int b, F&& fn) {
  if (a == AJQD_BF16 && b == AJQD_BF16) fn(uint16_t{}, uint16_t{});
  else if (a == AJQD_BF16) fn(uint16_t{}, float{});
  else if (b == AJQD_BF16) fn(float{}, uint16_t{});
  else fn(float{}, float{});
}

constexpr int kLdsLimit = 160 * 1024;
template <typename K>
int allow_lds(K kernel, int bytes, const char* what) {
  if (bytes > kLdsLimit) return fail(AJQ_ERR_UNSUPPORTED, "%s: %d bytes of LDS needed", what, bytes);
  if (bytes > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(AJQ_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
  }
  return AJQ_OK;
}

int check_shape(const ajqd_latent_shape* s, const char* what) {
  if (!s) return fail(AJQ_ERR_NULL, "%s: null shape", what);
  if (s->heads < 1 || s->dimp < 8 || s->dimp % 8 || s->rot < 2 || s->rot % 2 || s->rotp < s->rot || s->rotp % 8 || s->rank < 1 ||
      s->rankp < s->rank || s->rankp % 16)
    return fail(AJQ_ERR_SHAPE, "%s: unsupported latent shape (heads=%d dimp=%d rot=%d/%d rank=%d/%d)", what, s->heads, s->dimp,
                s->rot, s->rotp, s->rank, s->rankp);
  return AJQ_OK;
}
LatentShape device_shape(const ajqd_latent_shape* s) {
  return LatentShape{s->heads, s->dimp, s->rot, s->rotp, s->rank, s->rankp, s->eps};
}

int check_attention(const ajqd_windowed_attention_args* a, const char* what) {
  if (!a || !a->q || !a->k1 || (a->d2 && !a->k2) || !a->v || !a->out) return fail(AJQ_ERR_NULL, "%s: null pointer argument", what);
  if (a->batch < 1 || a->heads < 1 || a->seq < 1 || a->rows < 1 || a->prior < 0 || a->d1 < 8 || a->d2 < 0 || a->dv < 16 ||
      a->d1 % 8 || a->d2 % 8 || a->dv % 16 || a->out_ld < a->heads * a->dv || a->out_ld % 4 || a->keep < 0 || a->share < 0 ||
      (a->share > 1 && a->heads % a->share) || (a->column_gates && (a->gate_ld < a->heads * a->dv || a->gate_ld % 4)))
    return fail(AJQ_ERR_SHAPE, "%s: unsupported shape (B=%d H=%d T=%d rows=%d prior=%d d=%d+%d dv=%d)", what, a->batch, a->heads,
                a->seq, a->rows, a->prior, a->d1, a->d2, a->dv);
  if (a->pos ? a->seq != 1 : (long long)a->prior + a->seq > a->rows)
    return fail(AJQ_ERR_SHAPE, "%s: %d + %d queries do not fit %d rows", what, a->prior, a->seq, a->rows);
  if (!(a->scale > 0.f)) return fail(AJQ_ERR_SHAPE, "%s: the score scale must be positive", what);
  if (a->k1_row % 8 || a->k1_head % 8 || a->k2_row % 8 || a->v_row % 8 || a->v_head % 8 || a->k1_batch % 8 || a->k2_batch % 8 ||
      a->v_batch % 8 || !aligned16(a->q) || !aligned16(a->k1) || !aligned16(a->k2) || !aligned16(a->v) || !aligned16(a->out) || !aligned16(a->column_gates))
    return fail(AJQ_ERR_ALIGN, "%s: rows must start on 16-byte boundaries", what);
  return AJQ_OK;
}
WindowedAttention device_attention(const ajqd_windowed_attention_args* a) {
  WindowedAttention w;
  w.q = a->q; w.k1 = a->k1; w.k2 = a->k2; w.v = a->v; w.sink = a->sink; w.gates = a->gates;
  w.pos = positions64(a->pos); w.out = a->out;
  w.k1_batch = a->k1_batch; w.k2_batch = a->k2_batch; w.v_batch = a->v_batch;
  w.k1_row = a->k1_row; w.k1_head = a->k1_head; w.k2_row = a->k2_row; w.v_row = a->v_row; w.v_head = a->v_head;
  w.d1 = a->d1; w.d2 = a->d2; w.dv = a->dv;
  w.batch = a->batch; w.heads = a->heads; w.seq = a->seq;
  w.keep = a->keep; w.share = a->share > 1 ? a->share : 1; w.gate_ld = a->gate_ld; w.column_gates = a->column_gates;
  w.rows = a->rows; w.prior = a->prior; w.window = a->window; w.out_ld = a->out_ld; w.scale = a->scale;
  return w;
}

// ---- prompt attention: the smallest built (key steps, value tiles) that hold the widths
int prefill_ks(int d) { const int s = (d + 31) / 32; return s <= 4 ? s : s <= 6 ? 6 : s <= 8 ? 8 : 0; }
int prefill_vt(int dv) { const int t = (dv + 15) / 16; return t <= 2 ? 2 : t <= 4 ? 4 : t <= 6 ? 6 : t <= 8 ? 8 : t <= 16 ? 16 : 0; }
template <int KS, int VT>
int launch_prefill(const WindowedAttention& w, hipStream_t stream) {
  constexpr int U = KS + VT > 16 ? 1 : 2;
  constexpr int bytes = 2 * kPfBK * 128 * prefill_panels(KS, VT);
  auto kernel = windowed_prefill_kernel<KS, VT, U>;
  if (int e = allow_lds(kernel, bytes, "ajqd_windowed_prefill")) return e;
  const long long blocks = (long long)((w.seq + 64 * U - 1) / (64 * U)) * w.batch * w.heads;
  if (blocks > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_windowed_prefill: too many workgroups");
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), bytes, stream, w);
  return check_launch("ajqd_windowed_prefill");
}
template <int KS>
int launch_prefill_vt(int vt, const WindowedAttention& w, hipStream_t stream) {
  switch (vt) {
    case 2: return launch_prefill<KS, 2>(w, stream);
    case 4: return launch_prefill<KS, 4>(w, stream);
    case 6: return launch_prefill<KS, 6>(w, stream);
    case 8: return launch_prefill<KS, 8>(w, stream);
    default: return launch_prefill<KS, 16>(w, stream);
  }
}

// ---- products of many rows: tiles of 64 QM x 128 QN.  Microseconds of a tile that has a CU to itself, of its 64 k, and of its output's
// bytes per element; and of the launch.  They settle the choice and are not the kernels' times: fitted to 345 random products (1 .. 9000
// rows, 64 .. 22000 columns, k up to 18000; every tile, k in one piece and in up to 24 parts) in a row of milliseconds with weights that are
// in no cache, as a model's are, each by how near the best of its size it is.  (Fitted to short runs on weights that stay cached, 1500
// rows, 16384 -> 4096 came out as one piece: 162 us against 155 in two parts there, but 188 against 168 in a model.)
// On 690 others (2 .. 9000 rows, 16 .. 116000 columns, k 64 .. 18432) they are 25 % off (rms), as a rule 17 % low and at large sizes, where
// the clock falls, up to 40 % (8192 x 8192 x 8192: 551 us, measured 679).  What they choose takes 1.1 % longer than the best of the size
// on average and more than 10 % at 26 of them (118 rows, 8192 -> 13936: 66.4 us, 55.9 in three parts).  Times with a power and a
// memory limit, fitted without that weighting to 10 %, chose worse (3 %).
struct ProductTile {
  int qm, qn;
  float launch, tile, step, out;
};
constexpr ProductTile kProductTiles[] = {{4, 2, 0.0f, 3.606f, 1.038f, 0.603f}, {3, 2, 0.0f, 2.748f, 0.883f, 0.58f}, {2, 2, 0.0f, 1.862f, 0.709f, 0.522f},
                                         {3, 1, 0.925f, 1.376f, 0.573f, 0.299f}, {2, 1, 0.941f, 0.78f, 0.473f, 0.323f}, {1, 1, 1.982f, 0.0f, 0.381f, 0.209f}};
constexpr float kSharedTile = 1.224f;                        // of two tiles on one CU, against half of each alone
constexpr float kSumLaunch = 2.392f, kSumMegabyte = 0.299f;   // adding the parts: the launch, and what it reads and writes
constexpr int kProductParts[] = {1, 2, 3, 4, 6, 8, 12, 16, 24};
constexpr int kCus = 256;
constexpr int kProductMaxK = 1 << 22;   // of a row's elements too: a tile's offsets are 32 bits
bool product_made(int rows, int n, int k) { return rows >= 1 && n >= 16 && n % 16 == 0 && k >= 64 && k % 64 == 0 && k <= kProductMaxK; }
long long product_tiles(int qm, int qn, int rows, int n) { return (long long)((rows + 64 * qm - 1) / (64 * qm)) * ((n + 128 * qn - 1) / (128 * qn)); }
// steps of 64 k in a part, and the parts that come of it
int part_steps(int k, int parts) { return (k / 64 + parts - 1) / parts; }
int whole_parts(int k, int parts) { const int steps = part_steps(k, parts); return (k / 64 + steps - 1) / steps; }
float product_us(const ProductTile& t, int rows, int n, int k, int out_bytes, int parts) {
  const float turns = (float)product_tiles(t.qm, t.qn, rows, n) * whole_parts(k, parts) / kCus;
  // two tiles of one column quadrant share a CU, and a round that they fill half takes half as long
  const float rounds = t.qn == 2 || turns <= 1.f ? ceilf(turns) : 0.5f * kSharedTile * ceilf(2.f * turns);
  const float us = t.launch + rounds * (t.tile + t.step * (float)part_steps(k, parts) + t.out * (float)(parts > 1 ? 4 : out_bytes));
  return parts == 1 ? us : us + kSumLaunch + kSumMegabyte * 1e-6f * (float)rows * (float)n * (float)(4 * parts + out_bytes);
}
int pick_product_tile(int rows, int n, int k, int out_bytes, int parts, float* us = nullptr) {
  int best = 0;
  float least = 0.f;
  for (int i = 0; i < (int)(sizeof(kProductTiles) / sizeof(kProductTiles[0])); ++i) {
    const float now = product_us(kProductTiles[i], rows, n, k, out_bytes, parts);
    if (i == 0 || now < least) { best = i; least = now; }
  }
  if (us) *us = least;
  return best;
}
int product_out_bytes(int out_dtype, int pairs) { return out_dtype == AJQD_F32 ? 4 : pairs ? 1 : 2; }
template <int QM, int QN, int EPI>
int launch_product(const DenseGemm& a, hipStream_t stream) {
  constexpr int bytes = tile_lds_bytes(64 * QM, 128 * QN, EPI);
  auto kernel = dense_gemm_kernel<QM, QN, EPI>;
  if (int e = allow_lds(kernel, bytes, "ajqd_product")) return e;
  const long long blocks = product_tiles(QM, QN, a.m, a.n);
  if (blocks > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_product: too many workgroups");
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks, (a.k + a.part - 1) / a.part), dim3(kTileThreads), bytes, stream, a);
  return check_launch("ajqd_product");
}
template <int EPI>
int launch_product_tile(int tile, const DenseGemm& a, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_product<4, 2, EPI>(a, stream);
    case 1: return launch_product<3, 2, EPI>(a, stream);
    case 2: return launch_product<2, 2, EPI>(a, stream);
    case 3: return launch_product<3, 1, EPI>(a, stream);
    case 4: return launch_product<2, 1, EPI>(a, stream);
    default: return launch_product<1, 1, EPI>(a, stream);
  }
}

// ---- products of one decode step
constexpr int kTwoWaveColumns = 256;  // products of one or two blocks of columns run on two waves (stream_rows)
constexpr int kLongRow = 8192;
// Batch rows go through LDS (stream_rows) where K is whole blocks and the trip gains something (figures: the time over that from memory).  From 1024
// columns on with more than 16 sequences, 2048 with fewer (half of that would still gain, 512 columns 0.92 .. 0.98 at 32 sequences and 0.95 .. 0.98 at
// 16, but not at eight and fewer: 0.98 .. 1.03).  With five to eight a wave whose share is a block short waits for the others, until K hides that (5
// sequences, 96 tiles of dense_in: K = 2048 1.00, 2176 1.03, 2560 1.00, 3200 1.025, 4096 0.995; 7: 1.02 at 2176, 0.98 from 2560 on) or there is more
// than a round of workgroups (0.95 .. 0.98).  Up to four, an instruction brings few bytes either way: eight waves gain with even shares or 3072
// columns (width 1024, one sequence: K = 2048 0.955, 2176 1.01, 3584 0.95, 8192 0.89; width 2048 at 2176 and 2560: 1.04), four waves in the first
// half of a second round (320 tiles: 0.96 .. 1.00) and with long rows (K = 9216: 0.93 at 129 tiles, 0.96 at 320).  A round that is nearly full keeps the
// memory busy by itself, but where rows lie 16 KiB apart (256 tiles: K = 4096 1.01, 8192 0.94, 9216 1.02, 11136 1.02).
bool staged_rows(int batch, int k, int waves, long long tiles) {
  if (k % kStreamBlock != 0 || k < (batch > kGemvBatch ? 1024 : 2048)) return false;
  if (batch > 8) return true;
  const bool even = k % (kStreamBlock * waves) == 0;
  if (batch > 4) return waves == 8 || even || tiles > kCus || k >= (batch <= 6 ? 3584 : 2560);
  if (waves == 8) return even || k >= 3072;
  return (tiles > kCus && tiles <= 384) || (k >= kLongRow && (tiles <= 192 || tiles > kCus || k % kLongRow == 0));
}
// How dense_out and dense_out_streams cut [width, k]: up to 128 tiles of 16 rows leave half the CUs idle, tiles of 8 rows on eight
// waves use them all (2048 x 8192: 9.7 -> 7.5 us at 4 sequences, 15.4 -> 12.8 at 32), where K gives each of them a block (1024 x 512: 3.0 us
// with them, 2.5 without).  More than 16 sequences: two row tiles per workgroup share the activations from 512 tiles on (35424 x 4096: 84 -> 65 us),
// staged rows wherever one each would be more than a round of the CUs (5856 x 2048: 9.5 us, 7.9 with two; 4096 x 16384: 29.5, 38.0 with two); below
// that, rows that are not staged have two blocks in flight instead (4096 x 18440: 44.2 -> 42.6) where K gives each wave several (5120 x 256,
// 64 sequences: 9.1 us with two, 5.1 with one).  Up to 16, long staged rows that come out even: two blocks at a time (4096 x 16384: 26.6 -> 24.4;
// 4096 x 8448, 5 sequences: 12.7, 12.3 with one), with more than eight sequences, whose rows are half of what is asked for, only where rows lie whole
// multiples of 16 KiB apart (0.977 of the time with one) or, past twelve, of 4 KiB (9 sequences: 4032 x 11264 17.45 us, 16.2 with one).  K of one or two
// blocks: two waves (32000 x 128, one sequence: 5.2 us on four, 4.4 on two).
// More than four streams leave a wave of 16-row tiles and two batch tiles no registers for more than the plainest form: rows from memory, one row
// tile, one block at a time takes 240, every other form 280 and more, and then a CU holds one workgroup instead of two (12 streams of 2064
// columns, 33 sequences, K = 1152: 17.0 us, 34.1 with staged rows; 16 of 2560, 48 sequences, K = 2048: 28.7, 39.5).  Rows of 8192 columns make up
// for that (8 of 4096, 64 sequences: 44.4 us staged, 50.4 from memory) but where the last batch block is nearly empty (5 of 2560, 33: 34.5, 33.6).  Rows off the 128-column
// grid that are long beside what the streams take have two blocks in flight where there is a workgroup per CU anyway (6 of 2976, 31 sequences, K =
// 16024: 49.3 -> 44.6; 15 of 2336, K = 13576: 1.085).  Up to 16 sequences two blocks of more than eight's staged rows take 273 registers
// (13 of 11168, 12 sequences, K = 10240: 80.9 us, 55.1 with one; 140 shapes: 1.087 of the time from memory, 0.922 with one).
struct OutCut {
  int rows, rt, bt, uq, xq;  // row tile, row tiles, batch tiles, blocks at a time, batch rows' instructions
  dim3 grid;
  int threads;
};
OutCut out_cut(int batch, int width, int k, bool sums, int streams) {
  OutCut c;
  c.bt = batch > kGemvBatch ? 2 : 1;
  const int blocks = (batch + kGemvBatch * c.bt - 1) / (kGemvBatch * c.bt);
  const long long tiles = (long long)(width / 16) * blocks;
  c.rows = tiles <= 128 && (sums || k >= 1024) ? 8 : 16;
  const bool few = c.rows == 16 && c.bt == 1 && k <= kTwoWaveColumns, plain = c.rows == 16 && c.bt == 2 && streams > 4;
  const bool staged = staged_rows(batch, k, c.rows == 8 ? 8 : 4, tiles) && (!plain || k >= kLongRow);
  c.xq = few || !staged ? kStreamDirect : batch <= 4 ? 1 : batch <= 8 ? 2 : 4;
  c.rt = c.bt == 2 && width % 32 == 0 && (staged ? c.rows == 16 && tiles > kCus : !plain && width >= 8192) ? 2 : 1;
  const bool pays = c.xq < 4 ? k % 1024 == 0 : streams <= 4 && (k % 8192 == 0 || (batch > 12 && k % 2048 == 0));
  const bool room = plain ? tiles <= kCus && k >= kLongRow && k >= 1100 * streams : k >= 2048;
  c.uq = c.rows == 16 && c.rt == 1 && !few && (c.bt == 1 ? staged && k >= kLongRow && pays : !staged && room) ? 2 : 1;
  c.grid = dim3(width / (c.rows * c.rt), blocks);
  c.threads = c.rows == 8 ? 512 : few ? 128 : 256;
  return c;
}
// How dense_in cuts [16 (tiles1 + tiles2), k] without the norm.  More than 16 sequences: two batch tiles and two row tiles per workgroup, or, where one each is
// no more than a round of the CUs, one on eight waves (2560 x 2048, 32 sequences: 8.7 -> 6.8 us; 4608 x 2048, 288 tiles: 9.2 with two, 11.6 so).  Up to
// four: two blocks at a time where they come out even and the last round of workgroups is up to three quarters full, and not beyond 384, from where
// the rows' trip is for nothing (one sequence, K = 4096: 96 tiles 0.93 of the time, 192 0.99, 256 1.03, 288 0.96, 384 0.97, 480 1.03, 1024 1.03; K =
// 2048: 0.97, 0.97, 1.03, 0.96, 0.98, 1.00, 1.02).
struct InCut {
  int waves, rt, bt, uq, xq;
};
InCut in_cut(int batch, int k, int tiles1, int tiles2) {
  InCut c{4, 1, batch > kGemvBatch ? 2 : 1, 1, kStreamDirect};
  const int blocks = (batch + kGemvBatch * c.bt - 1) / (kGemvBatch * c.bt);
  const long long tiles = ((long long)tiles1 + tiles2) * blocks;
  if (k <= kTwoWaveColumns) {
    c.waves = 2;
    return c;
  }
  const bool staged = staged_rows(batch, k, 4, tiles);
  if (c.bt == 2) {
    if (staged && tiles <= kCus) c.waves = 8, c.xq = 4;
    else if (tiles1 != 1 && tiles2 != 1) c.rt = 2, c.xq = staged ? 4 : kStreamDirect;
  } else if (batch > 4) {
    if (staged) c.xq = batch > 8 ? 4 : 2;
  } else if (k % 1024 == 0 && k >= 2048 && (tiles <= 192 || (tiles > kCus && tiles <= 384))) {
    c.uq = 2, c.xq = 1;
  }
  return c;
}
template <int N> using Int = std::integral_constant<int, N>;
// go(waves, row tile, row tiles, batch tiles, blocks at a time, batch rows' instructions) of a cut; kMany: more than four streams
template <bool kMany, typename Go>
int with_out_cut(const OutCut& c, Go&& go) {
  if (c.threads == 128) return go(Int<2>{}, Int<16>{}, Int<1>{}, Int<1>{}, Int<1>{}, Int<kStreamDirect>{});
  if (c.bt == 2) {
    if (c.rows == 8) return c.xq == 4 ? go(Int<8>{}, Int<8>{}, Int<1>{}, Int<2>{}, Int<1>{}, Int<4>{})
                                      : go(Int<8>{}, Int<8>{}, Int<1>{}, Int<2>{}, Int<1>{}, Int<kStreamDirect>{});
    if (c.xq == 4) return c.rt == 2 ? go(Int<4>{}, Int<16>{}, Int<2>{}, Int<2>{}, Int<1>{}, Int<4>{}) : go(Int<4>{}, Int<16>{}, Int<1>{}, Int<2>{}, Int<1>{}, Int<4>{});
    if (c.uq == 2) return go(Int<4>{}, Int<16>{}, Int<1>{}, Int<2>{}, Int<2>{}, Int<kStreamDirect>{});
    if constexpr (!kMany) {
      if (c.rt == 2) return go(Int<4>{}, Int<16>{}, Int<2>{}, Int<2>{}, Int<1>{}, Int<kStreamDirect>{});
    }
    return go(Int<4>{}, Int<16>{}, Int<1>{}, Int<2>{}, Int<1>{}, Int<kStreamDirect>{});
  }
  auto with = [&](auto xq) {
    if (c.rows == 8) return go(Int<8>{}, Int<8>{}, Int<1>{}, Int<1>{}, Int<1>{}, xq);
    if constexpr (xq() != kStreamDirect && !(kMany && xq() == 4)) {
      if (c.uq == 2) return go(Int<4>{}, Int<16>{}, Int<1>{}, Int<1>{}, Int<2>{}, xq);
    }
    return go(Int<4>{}, Int<16>{}, Int<1>{}, Int<1>{}, Int<1>{}, xq);
  };
  return c.xq == 1 ? with(Int<1>{}) : c.xq == 2 ? with(Int<2>{}) : c.xq == 4 ? with(Int<4>{}) : with(Int<kStreamDirect>{});
}

// ---- decode attention: (column steps, latent tiles per wave) that hold the widths
int latent_tiles(int rankp) { const int t = (rankp + 63) / 64; return t <= 2 ? 2 : t <= 4 ? 4 : t <= 8 ? 8 : 0; }
int latent_steps(int width) { const int s = (width + 31) / 32; return s <= 4 ? 4 : s <= 6 ? 6 : s <= 8 ? 8 : s <= 10 ? 10 : s <= 18 ? 18 : 0; }
// the chunks' sums, then (maximum, denominator) per head and chunk
float2* heads_at(const float* partial, int batch, int heads, int chunks, int rankp) {
  return reinterpret_cast<float2*>(const_cast<float*>(partial) + latent_sums_at(batch, 0, 0, heads, chunks, rankp));
}
constexpr int kDecodeWorkgroups = 256;  // one per CU (its LDS holds two blocks of rows)
int latent_head_groups(int heads) { return heads <= 16 ? 1 : (heads + 31) / 32; }  // one or two head tiles per workgroup
// ---- several residual streams
int stream_room(int s) { return s <= 2 ? 2 : s <= 4 ? 4 : kMaxStreams; }
int check_streams(int streams, const char* what) {
  if (streams < 1 || streams > kMaxStreams) return fail(AJQ_ERR_UNSUPPORTED, "%s: %d streams (1 .. %d are built)", what, streams, kMaxStreams);
  return AJQ_OK;
}

// ---- selective scan: lanes per channel and states per lane.  More lanes than the states ask for where there are few channels:
// the time loop is sequential, so what counts then is its length per step and not the work.
template <typename T>
int launch_scan(const Scan& a, int batch, hipStream_t stream) {
  const long long lanes = (long long)batch * a.inner;
  auto go = [&](auto kernel, int per_channel) {
    const int channels = 256 / per_channel;
    hipLaunchKernelGGL(kernel, dim3((a.inner + channels - 1) / channels, batch), dim3(256), 0, stream, a, ScanParts{});
    return check_launch("ajqd_scan");
  };
  const bool few = lanes * 4 < 2 * 65536, fewer = lanes * 8 < 2 * 65536;  // (65536 lanes: a wave on every SIMD)
  const int n = a.states;
  if (n <= 16 && fewer) return go(scan_kernel<T, 16, 1, kScanWhole>, 16);
  if (n <= 16 && few) return go(scan_kernel<T, 8, 2, kScanWhole>, 8);
  if (n <= 16) return go(scan_kernel<T, 4, 4, kScanWhole>, 4);
  if (n <= 32 && fewer) return go(scan_kernel<T, 16, 2, kScanWhole>, 16);
  if (n <= 32 && few) return go(scan_kernel<T, 8, 4, kScanWhole>, 8);
  if (n <= 24) return go(scan_kernel<T, 4, 6, kScanWhole>, 4);
  if (n <= 32) return go(scan_kernel<T, 4, 8, kScanWhole>, 4);
  if (n <= 64) return few ? go(scan_kernel<T, 16, 4, kScanWhole>, 16) : go(scan_kernel<T, 8, 8, kScanWhole>, 8);
  if (n <= 128) return go(scan_kernel<T, 16, 8, kScanWhole>, 16);
  if (n <= 256) return go(scan_kernel<T, 32, 8, kScanWhole>, 32);
  return fail(AJQ_ERR_UNSUPPORTED, "ajqd_scan: %d states per channel (up to 256 are built)", n);
}
// In parts: four lanes per channel, the fewest there are (the part's own work counts now, not the length of its loop).
constexpr int kScanPartLanes = 4, kScanPartTokens = 32;  // a part is a multiple of the kernel's tile
template <typename T, int NS>
int launch_scan_parts(const Scan& a, int batch, int count, const ScanParts& parts, hipStream_t stream) {
  const int channels = 256 / kScanPartLanes, blocks = (a.inner + channels - 1) / channels;
  hipLaunchKernelGGL((scan_kernel<T, kScanPartLanes, NS, kScanEnds>), dim3(blocks, batch, count - 1), dim3(256), 0, stream, a, parts);
  hipLaunchKernelGGL((scan_kernel<T, kScanPartLanes, NS, kScanPart>), dim3(blocks, batch, count), dim3(256), 0, stream, a, parts);
  return check_launch("ajqd_scan_in_parts");
}


}  // namespace

extern "C" {

const char* ajqd_last_error(void) { return g_error; }

int ajqd_embed(const int64_t* tokens, int rows, int seq, const void* table, int vocab, const void* positions,
               int table_rows, int start, const int64_t* pos, const float* extra, float* x, float* embedded, int width,
               int dtype, void* stream) {
  if (!tokens || !table || !x) return fail(AJQ_ERR_NULL, "ajqd_embed: null pointer argument");
  if (rows < 1 || seq < 1 || rows % seq || vocab < 1 || width < 8 || width % 8 || (pos && seq != 1) ||
      (positions && (table_rows < 1 || start < 0 || (!pos && (long long)start + seq > table_rows))))
    return fail(AJQ_ERR_SHAPE, "ajqd_embed: unsupported shape (rows=%d seq=%d vocab=%d positions=%d start=%d width=%d)", rows, seq,
                vocab, table_rows, start, width);
  if (!known(dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_embed: unknown dtype %d", dtype);
  with_types(dtype, dtype, [&](auto t, auto) {
    using T = decltype(t);
    hipLaunchKernelGGL(embed_kernel<T>, dim3(rows), dim3(256), 0, (hipStream_t)stream, (const long long*)tokens, (const T*)table,
                       vocab, (const T*)positions, table_rows, start, positions64(pos), seq, extra, x, embedded, width);
  });
  return check_launch("ajqd_embed");
}

int ajqd_add_norms(float* x, const void* delta, int delta_dtype, const float* again, const float* step,
                   const float* gain1, const float* gain2, float eps, int center, void* out1, void* out2, int rows,
                   int true_width, int width, int dtype, void* stream) {
  if (!x || (out1 && !gain1) || (out2 && !gain2)) return fail(AJQ_ERR_NULL, "ajqd_add_norms: null pointer argument");
  if (rows < 1 || true_width < 1 || width < true_width || width % 8)
    return fail(AJQ_ERR_SHAPE, "ajqd_add_norms: unsupported shape (rows=%d width=%d of %d)", rows, true_width, width);
  if (!known(dtype) || !known(delta_dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_add_norms: unknown dtype");
  with_types(dtype, delta_dtype, [&](auto t, auto d) {
    using T = decltype(t);
    using DT = decltype(d);
    hipLaunchKernelGGL((add_norms_kernel<T, DT>), dim3(rows), dim3(256), 0, (hipStream_t)stream, x, (const DT*)delta, again, step,
                       gain1, gain2, eps, center, (T*)out1, (T*)out2, true_width, width);
  });
  return check_launch("ajqd_add_norms");
}

int ajqd_latent_split(const void* y, int y_dtype, int ldy, const ajqd_latent_shape* shape, const float* latent_gain,
                      const float* cosine, const float* sine, int table_rows, int rows, int seq, int start, const int64_t* pos,
                      int prior, int cap, void* qu, int qu_ld, void* qr, int qr_ld, void* cache_rows, int64_t rows_batch,
                      float* gates, int dtype, void* stream) {
  if (int e = check_shape(shape, "ajqd_latent_split")) return e;
  if (!y || !latent_gain || !cosine || !sine || !qu || !qr || !cache_rows || !gates)
    return fail(AJQ_ERR_NULL, "ajqd_latent_split: null pointer argument");
  const int width = shape->rankp + shape->rotp;
  if (rows < 1 || seq < 1 || rows % seq || start < 0 || prior < 0 || table_rows < 1 || qu_ld < shape->dimp || qr_ld < shape->rotp ||
      ldy < shape->heads * (shape->dimp + shape->rotp) + width + shape->heads || (pos ? (seq != 1 || cap < 1) : (long long)start + seq > table_rows) ||
      rows_batch < (int64_t)(pos ? cap : prior + seq) * width)
    return fail(AJQ_ERR_SHAPE, "ajqd_latent_split: unsupported shape (rows=%d seq=%d start=%d prior=%d cap=%d ldy=%d)", rows, seq,
                start, prior, cap, ldy);
  if (!known(dtype) || !known(y_dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_latent_split: unknown dtype");
  const LatentShape s = device_shape(shape);
  with_types(y_dtype, dtype, [&](auto yt, auto t) {
    using Y = decltype(yt);
    using T = decltype(t);
    hipLaunchKernelGGL((latent_split_kernel<Y, T>), dim3(rows), dim3(256), 0, (hipStream_t)stream, (const Y*)y, ldy, s, latent_gain,
                       cosine, sine, table_rows, start, positions64(pos), seq, prior, cap, (T*)qu, qu_ld, (T*)qr, qr_ld,
                       (T*)cache_rows, (long long)rows_batch, gates);
  });
  return check_launch("ajqd_latent_split");
}

int ajqd_ring_copy(void* ring, int cap, int kept, void* linear, int lines, int line_bytes, int first_row, int position, int count,
                   int row_bytes, int batch, int to_ring, void* stream) {
  if (!ring || !linear) return fail(AJQ_ERR_NULL, "ajqd_ring_copy: null pointer argument");
  if (cap < 1 || kept < 0 || kept > cap || count < 1 || first_row < 0 || (long long)first_row + count > lines || position < 0 ||
      batch < 1 || row_bytes < 16 || row_bytes % 16 || line_bytes < row_bytes || line_bytes % 16 ||
      (long long)position + count - (position > kept ? position : kept) > cap - kept)
    return fail(AJQ_ERR_SHAPE, "ajqd_ring_copy: unsupported shape (cap=%d lines=%d first=%d position=%d count=%d)", cap, lines,
                first_row, position, count);
  if (!aligned16(ring) || !aligned16(linear)) return fail(AJQ_ERR_ALIGN, "ajqd_ring_copy: buffers must be 16-byte aligned");
  const long long blocks = ((long long)batch * count * (row_bytes / 16) + 255) / 256;
  if (blocks > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_ring_copy: too many elements");
  hipLaunchKernelGGL(ring_copy_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (u32x4_t*)ring, cap, kept,
                     (u32x4_t*)linear, lines, line_bytes / 16, first_row, position, count, row_bytes / 16, batch, to_ring);
  return check_launch("ajqd_ring_copy");
}

int ajqd_gated_activation(const void* y, int y_dtype, void* out, int out_ld, int rows, int width, int act, int dtype,
                          void* stream) {
  if (!y || !out) return fail(AJQ_ERR_NULL, "ajqd_gated_activation: null pointer argument");
  if (rows < 1 || width < 8 || width % 8 || out_ld < width || out_ld % 4)
    return fail(AJQ_ERR_SHAPE, "ajqd_gated_activation: unsupported shape (rows=%d width=%d out_ld=%d)", rows, width, out_ld);
  if (!known(dtype) || !known(y_dtype) || act < 0 || act > AJQD_ACT_SQUARED_RELU)
    return fail(AJQ_ERR_UNSUPPORTED, "ajqd_gated_activation: unknown dtype or activation");
  const long long blocks = ((long long)rows * (width / 4) + 255) / 256;
  if (blocks > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_gated_activation: too many elements");
  with_types(y_dtype, dtype, [&](auto yt, auto t) {
    using Y = decltype(yt);
    using T = decltype(t);
    hipLaunchKernelGGL((gated_activation_kernel<Y, T>), dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (const Y*)y, (T*)out,
                       out_ld, rows, width, act);
  });
  return check_launch("ajqd_gated_activation");
}

int ajqd_product_better(int rows, int n, int k) {
  if (!product_made(rows, n, k)) return 0;
  // A workgroup goes through all of k here: few tiles and a long k are made faster in parts with the activation behind them (61 rows,
  // 8576 -> 528: 37 us against 20; 919 rows, 15488 -> 640: 78 against 53).  Up to k = 2048 (13 us in one wave of workgroups) or from a tile
  // per CU on one piece is the faster as a rule: over 433 such products 0.75 of the time of the other way.  24 of them are slower by more
  // than 5 % (16 rows, 2048 -> 2048: 19.7 us against 10.6; 582 rows, 11264 -> 8656: 147 against 135) and stay, as their activation is taken
  // of the fp32 sum here and of its bf16 rounding there.
  return k <= 2048 || product_tiles(1, 1, rows, n) >= kCus;
}

}  // extern "C"
namespace {
int check_product(const char* name, const ajqd_product_args* a) {
  if (!a || !a->x || !a->w || !a->y) return fail(AJQ_ERR_NULL, "%s: null pointer argument", name);
  const int columns = a->pairs ? a->n / 2 : a->n, multiple = a->out_dtype == AJQD_F32 ? 4 : 8;
  if (!product_made(a->rows, a->n, a->k) || a->ldx < a->k || a->ldx > kProductMaxK || a->ldy < columns)
    return fail(AJQ_ERR_SHAPE, "%s: unsupported shape (rows=%d n=%d k=%d ldx=%d ldy=%d)", name, a->rows, a->n, a->k, a->ldx, a->ldy);
  if (!known(a->out_dtype) || a->act < -1 || a->act > AJQD_ACT_SQUARED_RELU || (a->out_dtype == AJQD_F32 && a->act >= 0) || (a->pairs && a->act < 0))
    return fail(AJQ_ERR_UNSUPPORTED, "%s: unsupported output (dtype=%d act=%d pairs=%d)", name, a->out_dtype, a->act, a->pairs);
  if (a->ldx % 8 || a->ldy % multiple || !aligned16(a->x) || !aligned16(a->w) || !aligned16(a->y))
    return fail(AJQ_ERR_ALIGN, "%s: rows must start on 16-byte boundaries", name);
  return AJQ_OK;
}
}  // namespace
extern "C" {

int ajqd_product(const ajqd_product_args* a, void* stream) {
  if (int e = check_product("ajqd_product", a)) return e;
  DenseGemm d{(const uint16_t*)a->x, (const uint16_t*)a->w, a->y, a->rows, a->n, a->k, a->ldx, a->ldy, a->act, a->k};
  const int tile = pick_product_tile(a->rows, a->n, a->k, product_out_bytes(a->out_dtype, a->pairs), 1);
  if (a->out_dtype == AJQD_F32) return launch_product_tile<kTileF32>(tile, d, (hipStream_t)stream);
  if (a->act < 0) return launch_product_tile<kTileBf16>(tile, d, (hipStream_t)stream);
  return a->pairs ? launch_product_tile<kTilePairs>(tile, d, (hipStream_t)stream) : launch_product_tile<kTileAct>(tile, d, (hipStream_t)stream);
}

int ajqd_product_parts(int rows, int n, int k, int out_dtype) {
  if (!product_made(rows, n, k) || !known(out_dtype)) return 0;
  // Few tiles leave the chip idle for all of k: then its parts are made side by side, as many as the estimates say.  Against the vendor's
  // products over the 345: 0.45 of their time (110 rows, 16960 -> 4544: 33 us, theirs 101, in one piece 83; 463 rows, 11392 -> 384: 15,
  // 27, 56; 1500 rows, 8192 -> 288: 20, 22, 42); over 690 others 0.80 of it where a product takes 40 us or more, and nine are slower by 3 to
  // 10 %, most of them heads of 17 to 250 rows (63 rows, 3008 -> 43408: 59.7 us, 54.5).  Large outputs stay in one piece (4096 rows,
  // 18432 -> 4096: 413 us, in two parts 447).
  int best = 1;
  float least = 0.f, us;
  for (int parts : kProductParts) {
    // (what the estimates were fitted to; 128 MiB of sums at most)
    if (parts > 1 && (k / parts < 256 || (long long)rows * n * parts > (1LL << 25))) continue;
    pick_product_tile(rows, n, k, product_out_bytes(out_dtype, 0), parts, &us);
    if (parts == 1 || us < least) { best = parts; least = us; }
  }
  return whole_parts(k, best);
}
int ajqd_product_tile(int rows, int n, int k, int out_dtype, int pairs, int parts) {
  if (!product_made(rows, n, k) || !known(out_dtype)) return 0;
  parts = whole_parts(k, std::max(1, std::min(parts, k / 64)));
  const ProductTile& t = kProductTiles[pick_product_tile(rows, n, k, product_out_bytes(out_dtype, pairs), parts)];
  return 64 * t.qm << 16 | 128 * t.qn;
}
size_t ajqd_product_workspace(int rows, int n, int parts) { return parts > 1 ? (size_t)parts * rows * n * sizeof(float) : 0; }
int ajqd_product_in_parts(const ajqd_product_args* a, int parts, float* workspace, void* stream) {
  if (int e = check_product("ajqd_product_in_parts", a)) return e;
  if (a->act >= 0) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_product_in_parts: an activation takes the product in one piece");
  if (parts > 1) parts = whole_parts(a->k, std::min(parts, a->k / 64));
  if (parts < 2) return ajqd_product(a, stream);
  if (!workspace) return fail(AJQ_ERR_NULL, "ajqd_product_in_parts: null workspace");
  if (!aligned16(workspace)) return fail(AJQ_ERR_ALIGN, "ajqd_product_in_parts: the workspace must start on a 16-byte boundary");
  const long long blocks = ((long long)a->rows * (a->n / 8) + 255) / 256;
  if (parts > 65535 || blocks > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_product_in_parts: too many workgroups");
  const int out_bytes = product_out_bytes(a->out_dtype, 0), tile = pick_product_tile(a->rows, a->n, a->k, out_bytes, parts);
  const DenseGemm d{(const uint16_t*)a->x, (const uint16_t*)a->w, workspace, a->rows, a->n, a->k, a->ldx, a->n, -1, 64 * part_steps(a->k, parts)};
  if (int e = launch_product_tile<kTileF32>(tile, d, (hipStream_t)stream)) return e;
  if (out_bytes == 4)
    hipLaunchKernelGGL(sum_parts_kernel<float>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, workspace, parts, a->rows, a->n, (float*)a->y, a->ldy);
  else
    hipLaunchKernelGGL(sum_parts_kernel<uint16_t>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, workspace, parts, a->rows, a->n, (uint16_t*)a->y, a->ldy);
  return check_launch("ajqd_product_in_parts");
}

int ajqd_matvec(const void* w, const void* x, int x_batch, int x_group, void* y, int y_batch, int y_group, int groups,
                int n, int k, int batch, int dtype, int out_dtype, void* stream) {
  if (!w || !x || !y) return fail(AJQ_ERR_NULL, "ajqd_matvec: null pointer argument");
  if (n < 1 || k < 8 || k % 8 || groups < 1 || groups > 65535 || batch < 1 || batch > 65535 || x_batch % 4 || x_group % 4)
    return fail(AJQ_ERR_SHAPE, "ajqd_matvec: unsupported shape (groups=%d n=%d k=%d batch=%d)", groups, n, k, batch);
  if (!known(dtype) || !known(out_dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_matvec: unknown dtype");
  with_types(dtype, out_dtype, [&](auto t, auto o) {
    using T = decltype(t);
    using O = decltype(o);
    hipLaunchKernelGGL((matvec_kernel<T, O>), dim3((n + 3) / 4, groups, batch), dim3(256), 0, (hipStream_t)stream, (const T*)w,
                       (const T*)x, x_batch, x_group, (O*)y, y_batch, y_group, n, k);
  });
  return check_launch("ajqd_matvec");
}

int ajqd_windowed_attention(const ajqd_windowed_attention_args* args, int dtype, int out_dtype, void* stream) {
  if (int e = check_attention(args, "ajqd_windowed_attention")) return e;
  if (!known(dtype) || !known(out_dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_windowed_attention: unknown dtype");
  if (args->heads > 65535) return fail(AJQ_ERR_SHAPE, "ajqd_windowed_attention: too many heads");
  const int bytes = 4 * (args->d1 + args->d2 + args->dv + 64);
  const WindowedAttention w = device_attention(args);
  int status = AJQ_OK;
  with_types(dtype, out_dtype, [&](auto t, auto o) {
    auto kernel = windowed_attention_kernel<decltype(t), decltype(o)>;
    status = allow_lds(kernel, bytes, "ajqd_windowed_attention");
    if (status == AJQ_OK)
      hipLaunchKernelGGL(kernel, dim3(w.batch * w.seq, w.heads), dim3(64), bytes, (hipStream_t)stream, w);
  });
  return status != AJQ_OK ? status : check_launch("ajqd_windowed_attention");
}

int ajqd_windowed_prefill_supported(int d1, int d2, int dv) {
  return d1 >= 8 && d2 >= 0 && d1 % 8 == 0 && d2 % 8 == 0 && dv >= 16 && dv % 16 == 0 && prefill_ks(d1 + d2) && prefill_vt(dv);
}

int ajqd_windowed_prefill(const ajqd_windowed_attention_args* args, void* stream) {
  if (int e = check_attention(args, "ajqd_windowed_prefill")) return e;
  if (args->pos) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_windowed_prefill: takes no device-side position");
  if (!ajqd_windowed_prefill_supported(args->d1, args->d2, args->dv))
    return fail(AJQ_ERR_UNSUPPORTED, "ajqd_windowed_prefill: widths %d + %d / %d are not built", args->d1, args->d2, args->dv);
  const WindowedAttention w = device_attention(args);
  const int vt = prefill_vt(args->dv);
  switch (prefill_ks(args->d1 + args->d2)) {
    case 1: return launch_prefill_vt<1>(vt, w, (hipStream_t)stream);
    case 2: return launch_prefill_vt<2>(vt, w, (hipStream_t)stream);
    case 3: return launch_prefill_vt<3>(vt, w, (hipStream_t)stream);
    case 4: return launch_prefill_vt<4>(vt, w, (hipStream_t)stream);
    case 6: return launch_prefill_vt<6>(vt, w, (hipStream_t)stream);
    default: return launch_prefill_vt<8>(vt, w, (hipStream_t)stream);
  }
}

static int dense_in(const char* name, const ajqd_dense_in_args* a, const float* sums, int parts, void* stream) {
  if (!a || (a->x ? (a->tiles1 && !a->gain1) || (a->tiles2 && !a->gain2) : (a->tiles1 && !a->n1) || (a->tiles2 && !a->n2)) ||
      (a->tiles1 && (!a->w1 || !a->y1)) || (a->tiles2 && (!a->w2 || !a->gated)))
    return fail(AJQ_ERR_NULL, "%s: null pointer argument", name);
  if (a->batch < 1 || a->true_width < 1 || a->width < a->true_width || a->width % 8 || a->tiles1 < 0 || a->tiles2 < 0 ||
      a->tiles1 + a->tiles2 < 1 || (a->tiles2 && (a->gated_ld < (a->pairs ? 8 : 16) * a->tiles2 || a->gated_ld % 4)))
    return fail(AJQ_ERR_SHAPE, "%s: unsupported shape (batch=%d width=%d/%d tiles=%d+%d)", name, a->batch, a->true_width, a->width,
                a->tiles1, a->tiles2);
  if (a->act < 0 || a->act > AJQD_ACT_SQUARED_RELU) return fail(AJQ_ERR_UNSUPPORTED, "%s: unknown activation", name);
  if (a->x && a->batch > 4) return fail(AJQ_ERR_UNSUPPORTED, "%s: the norm prologue takes at most 4 rows", name);
  DenseIn d;
  d.x = a->x; d.n1 = (const uint16_t*)a->n1; d.n2 = (const uint16_t*)a->n2; d.gain1 = a->gain1; d.gain2 = a->gain2;
  d.w1 = (const uint16_t*)a->w1; d.w2 = (const uint16_t*)a->w2; d.y1 = a->y1; d.gated = (uint16_t*)a->gated;
  d.batch = a->batch; d.D = a->true_width; d.Dp = a->width; d.tiles1 = a->tiles1; d.tiles2 = a->tiles2;
  d.gated_ld = a->gated_ld; d.act = a->act; d.center = a->center; d.pairs = a->pairs; d.eps = a->eps;
  d.sums = sums; d.parts = parts;
  const InCut c = in_cut(a->batch, a->width, a->tiles1, a->tiles2);
  const int block = kGemvBatch * c.bt;
  const dim3 grid((a->tiles1 + c.rt - 1) / c.rt + (a->tiles2 + c.rt - 1) / c.rt, (a->batch + block - 1) / block);
  const int bytes = a->x ? 2 * a->batch * (a->width + 8) : 0;
  auto go = [&](auto kernel, int threads) {
    if (int e = allow_lds(kernel, bytes, name)) return e;
    hipLaunchKernelGGL(kernel, grid, dim3(threads), bytes, (hipStream_t)stream, d);
    return check_launch(name);
  };
  if (a->x) {
    // (rows so long that a workgroup's staging would not fit beside them run on two waves)
    // (and rows of more than 4096 columns on eight, whose registers hold them between the norm's passes: 8192 columns, 4 rows, 0 + 13648: 59.9
    // us on eight waves of the half-line form before, 96.7 on four of this one; 2016 + 6912: 43.7, 70.9, and 46.6 on eight)
    if (bytes > 140 * 1024 || c.waves == 2) return go(dense_in_kernel<2, true, 1, 1, kStreamFrom, 1>, 128);
    if (a->width > 4096 && bytes <= 120 * 1024) return go(dense_in_kernel<8, true, 1, 1, kStreamFrom, 1>, 512);
    return go(dense_in_kernel<4, true, 1, 1, kStreamFrom, 1>, 256);
  }
  if (c.waves == 2) return c.bt == 2 ? go(dense_in_kernel<2, false, 1, 2, kStreamDirect, 1>, 128) : go(dense_in_kernel<2, false, 1, 1, kStreamDirect, 1>, 128);
  if (c.waves == 8) return go(dense_in_kernel<8, false, 1, 2, 4, 1>, 512);
  if (c.rt == 2) return c.xq == 4 ? go(dense_in_kernel<4, false, 2, 2, 4, 1>, 256) : go(dense_in_kernel<4, false, 2, 2, kStreamDirect, 1>, 256);
  if (c.bt == 2) return go(dense_in_kernel<4, false, 1, 2, kStreamDirect, 1>, 256);
  switch (c.xq) {
    case 1: return go(dense_in_kernel<4, false, 1, 1, 1, 2>, 256);
    case 2: return go(dense_in_kernel<4, false, 1, 1, 2, 1>, 256);
    case 4: return go(dense_in_kernel<4, false, 1, 1, 4, 1>, 256);
    default: return go(dense_in_kernel<4, false, 1, 1, kStreamDirect, 1>, 256);
  }
}

int ajqd_dense_in_form(int batch, int k, int tiles1, int tiles2) {
  if (batch < 1 || k < 8 || k % 8 || tiles1 < 0 || tiles2 < 0 || tiles1 + tiles2 < 1) return 0;
  const InCut c = in_cut(batch, k, tiles1, tiles2);
  return 100000 * c.waves + 20000 + 1000 * c.rt + 100 * c.bt + 10 * c.uq + (c.xq > 0 ? c.xq : 0);
}

int ajqd_dense_in(const ajqd_dense_in_args* a, void* stream) { return dense_in("ajqd_dense_in", a, nullptr, 0, stream); }

int ajqd_dense_in_scaled(const ajqd_dense_in_args* a, const float* sums, int parts, void* stream) {
  if (!a || !sums) return fail(AJQ_ERR_NULL, "ajqd_dense_in_scaled: null pointer argument");
  if (a->x || a->center || parts < 1) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_dense_in_scaled: sums of squares go with scaled rows of an RMS norm");
  return dense_in("ajqd_dense_in_scaled", a, sums, parts, stream);
}

int ajqd_dense_out(const void* in, const void* w, float* x, const float* again, const float* step, int batch, int k,
                   int width, void* stream) {
  if (!in || !w || !x) return fail(AJQ_ERR_NULL, "ajqd_dense_out: null pointer argument");
  if (batch < 1 || k < 8 || k % 8 || width < 16 || width % 16)
    return fail(AJQ_ERR_SHAPE, "ajqd_dense_out: unsupported shape (batch=%d k=%d width=%d)", batch, k, width);
  DenseOut d{(const uint16_t*)in, (const uint16_t*)w, x, again, step, batch, k, width};
  const OutCut c = out_cut(batch, width, k, false, 1);
  return with_out_cut<false>(c, [&](auto waves, auto rows, auto rt, auto bt, auto uq, auto xq) {
    hipLaunchKernelGGL((dense_out_kernel<waves(), rows(), rt(), bt(), uq(), xq()>), c.grid, dim3(c.threads), 0, (hipStream_t)stream, d);
    return check_launch("ajqd_dense_out");
  });
}
int ajqd_latent_absorb(const float* y, int ldy, const ajqd_latent_shape* shape, const void* ukt, const float* latent_gain,
                       const float* cosine, const float* sine, int table_rows, const int64_t* pos, void* q, void* ring, int cap,
                       int batch, void* stream) {
  if (int e = check_shape(shape, "ajqd_latent_absorb")) return e;
  if (!y || !ukt || !latent_gain || !cosine || !sine || !pos || !q || !ring)
    return fail(AJQ_ERR_NULL, "ajqd_latent_absorb: null pointer argument");
  if (batch < 1 || cap < 1 || table_rows < 1 || ldy % 4 ||
      ldy < shape->heads * (shape->dimp + shape->rotp) + shape->rankp + shape->rotp + shape->heads)
    return fail(AJQ_ERR_SHAPE, "ajqd_latent_absorb: unsupported shape (batch=%d cap=%d ldy=%d)", batch, cap, ldy);
  const int groups = (shape->rankp / 16 + 3) / 4;
  LatentAbsorb d{y, (const uint16_t*)ukt, latent_gain, cosine, sine, positions64(pos), (uint16_t*)q, (uint16_t*)ring,
                 batch, ldy, table_rows, cap, groups, device_shape(shape)};
  hipLaunchKernelGGL(latent_absorb_kernel, dim3(shape->heads * groups + 4 + shape->heads, (batch + kGemvBatch - 1) / kGemvBatch), dim3(256), 0,
                     (hipStream_t)stream, d);
  return check_launch("ajqd_latent_absorb");
}

int ajqd_latent_decode_chunks(int batch, int heads, int rankp, int rotp, int cap) {
  if (batch < 1 || heads < 1 || cap < 1 || rankp < 16 || rankp % 16 || rotp < 8 || rotp % 8 || !latent_tiles(rankp) ||
      !latent_steps(rankp + rotp))
    return 0;
  const int groups = batch * latent_head_groups(heads);
  int s = (kDecodeWorkgroups + groups - 1) / groups;
  const int by_rows = (cap + kLatentRows - 1) / kLatentRows;
  if (s > by_rows) s = by_rows;
  return s < 1 ? 1 : s > kLatentMaxChunks ? kLatentMaxChunks : s;
}

size_t ajqd_latent_decode_workspace(int batch, int heads, int rankp, int chunks) {
  if (batch < 1 || heads < 1 || rankp < 1 || chunks < 1) return 0;
  return 4 * (size_t)latent_sums_at(batch, 0, 0, heads, chunks, rankp) + 8 * (size_t)batch * heads * chunks;
}

int ajqd_latent_decode(const void* q, const void* ring, const int64_t* pos, float* partial, int batch, int heads, int rankp,
                       int rotp, int cap, int chunks, int first_column, float scale, void* stream) {
  if (!q || !ring || !pos || !partial) return fail(AJQ_ERR_NULL, "ajqd_latent_decode: null pointer argument");
  if (ajqd_latent_decode_chunks(batch, heads, rankp, rotp, cap) == 0)
    return fail(AJQ_ERR_UNSUPPORTED, "ajqd_latent_decode: widths %d + %d are not built", rankp, rotp);
  if (chunks < 1 || chunks > kLatentMaxChunks || first_column < 0 || first_column >= rankp + rotp || !(scale > 0.f))
    return fail(AJQ_ERR_SHAPE, "ajqd_latent_decode: unsupported shape (batch=%d chunks=%d)", batch, chunks);
  LatentDecode d{(const uint16_t*)q, (const uint16_t*)ring, positions64(pos), partial,
                 heads_at(partial, batch, heads, chunks, rankp), batch, heads, rankp, rankp + rotp, cap, chunks, first_column / 32, scale * kLog2eF};
  // Two head tiles share a workgroup and its rows where there is more than one workgroup per CU; below that one each, on twice
  // the CUs: 32 heads, rows of 576, a chunk per 64 of 560 rows, 1 / 8 / 16 sequences (two tiles make 10 / 80 / 160 workgroups):
  // 8.8 / 9.8 / 10.6 us with two, 6.1 / 7.3 / 13.0 with one.
  const long long singles = (long long)((heads + 15) / 16) * chunks * batch;
  const bool two = heads > 16 && singles > kDecodeWorkgroups;
  const long long blocks = two ? (long long)((heads + 31) / 32) * chunks * batch : singles;
  if (blocks > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_latent_decode: too many workgroups");
  auto go = [&](auto kernel, int ks) {
    const int bytes = latent_decode_lds(ks, two ? 2 : 1);
    if (int e = allow_lds(kernel, bytes, "ajqd_latent_decode")) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(two ? 512 : 256), bytes, (hipStream_t)stream, d);
    return check_launch("ajqd_latent_decode");
  };
  auto pick = [&](auto one, auto both, int ks) { return two ? go(both, ks) : go(one, ks); };
  const int tiles = latent_tiles(rankp);
#define AJQD_DECODE(KS, RT) pick(latent_decode_kernel<KS, RT, 1>, latent_decode_kernel<KS, RT, 2>, KS)
  switch (latent_steps(rankp + rotp)) {
    case 4: return AJQD_DECODE(4, 2);  // (at most 128 columns: two tiles per wave)
    case 6: return tiles == 2 ? AJQD_DECODE(6, 2) : AJQD_DECODE(6, 3);
    case 8: return tiles == 2 ? AJQD_DECODE(8, 2) : AJQD_DECODE(8, 4);
    case 10: return tiles == 2 ? AJQD_DECODE(10, 2) : tiles == 4 ? AJQD_DECODE(10, 4) : AJQD_DECODE(10, 5);
    default: return tiles == 2 ? AJQD_DECODE(18, 2) : tiles == 4 ? AJQD_DECODE(18, 4) : AJQD_DECODE(18, 8);
  }
#undef AJQD_DECODE
}

int ajqd_latent_expand(const float* partial, const float* sink, const float* gate, int gate_ld, const void* uv, void* out,
                       int out_ld, int batch, int heads, int chunks, int rankp, int vdimp, void* stream) {
  if (!partial || !uv || !out) return fail(AJQ_ERR_NULL, "ajqd_latent_expand: null pointer argument");
  if (batch < 1 || heads < 1 || chunks < 1 || chunks > kLatentMaxChunks || rankp < 16 || rankp % 16 || vdimp < 16 || vdimp % 16 ||
      out_ld < heads * vdimp || out_ld % 4)
    return fail(AJQ_ERR_SHAPE, "ajqd_latent_expand: unsupported shape (batch=%d heads=%d chunks=%d rankp=%d vdimp=%d)", batch,
                heads, chunks, rankp, vdimp);
  if (rankp > kExpandRank) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_latent_expand: latents of %d are not built", rankp);
  // A workgroup reads a part of a head's weights and the chunks' sums of a few sequences, at what one CU takes in: the cut that
  // makes both small and still leaves no more than one workgroup per CU.  (512 x 128 weights, 10 chunks: 16 heads, 8 sequences: 5.6 us
  // with 2 tiles x 2 sequences, 7.9 with 8 x 4; 32 heads, 8 sequences: 7.5 with 8 x 1, 8.1 with 8 x 4, 11.5 with 2 x 2, and with
  // 32 chunks 8.8 with 8 x 1, 13.8 with 8 x 4; 16 sequences: 7.9 with 8 x 2, 8.4 with 8 x 4, 13.7 with 8 x 1.)
  auto go = [&](auto kernel, int tw, int eb) {
    const int groups = (vdimp / 16 + tw - 1) / tw, bytes = 2 * eb * (rankp + 8);
    LatentExpand d{partial, heads_at(partial, batch, heads, chunks, rankp), sink, gate, (const uint16_t*)uv, (uint16_t*)out, batch, heads, chunks, rankp, vdimp, gate_ld, out_ld, groups};
    hipLaunchKernelGGL(kernel, dim3(heads * groups, (batch + eb - 1) / eb), dim3(512), bytes, (hipStream_t)stream, d);
    return check_launch("ajqd_latent_expand");
  };
  auto fits = [&](int tw, int eb) { return (long long)heads * ((vdimp / 16 + tw - 1) / tw) * ((batch + eb - 1) / eb) <= kDecodeWorkgroups; };
  // (many chunks of more than four sequences: every workgroup of a head repeats their sums; 8 sequences, 16 heads, 32 chunks: 13.8 us with 2
  // tiles x 2 sequences, 7.9 with 8 x 1)
  if (fits(2, 2) && (batch <= 4 || chunks <= 16)) return go(latent_expand_kernel<2, 2>, 2, 2);
  if (batch <= 4) return go(latent_expand_kernel<2, 4>, 2, 4);
  if (fits(8, 1)) return go(latent_expand_kernel<8, 1>, 8, 1);
  if (fits(8, 2)) return go(latent_expand_kernel<8, 2>, 8, 2);
  return go(latent_expand_kernel<8, 4>, 8, 4);
}

// ---- several residual streams
int ajqd_embed_streams(const int64_t* tokens, int rows, const void* table, int vocab, const float* in, float* x, float* u, int streams,
                       int width, int dtype, void* stream) {
  if (!tokens || !table || !x || (u && !in)) return fail(AJQ_ERR_NULL, "ajqd_embed_streams: null pointer argument");
  if (int e = check_streams(streams, "ajqd_embed_streams")) return e;
  if (rows < 1 || vocab < 1 || width < 8 || width % 8)
    return fail(AJQ_ERR_SHAPE, "ajqd_embed_streams: unsupported shape (rows=%d vocab=%d width=%d)", rows, vocab, width);
  if (!known(dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_embed_streams: unknown dtype %d", dtype);
  with_types(dtype, dtype, [&](auto t, auto) {
    using T = decltype(t);
    hipLaunchKernelGGL(embed_streams_kernel<T>, dim3(rows), dim3(256), 0, (hipStream_t)stream, (const long long*)tokens, (const T*)table,
                       vocab, in, x, u, streams, width);
  });
  return check_launch("ajqd_embed_streams");
}

int ajqd_streams_norm(float* x, const float* delta, const float* scale, const float* out, const float* mix, const float* in,
                      const float* gain, float eps, void* normed, float* u, int streams, int rows, int true_width, int width, int dtype,
                      void* stream) {
  if (!x || (delta && (!scale || !out || !mix)) || (normed && !gain)) return fail(AJQ_ERR_NULL, "ajqd_streams_norm: null pointer argument");
  if (int e = check_streams(streams, "ajqd_streams_norm")) return e;
  if (rows < 1 || true_width < 1 || width < true_width || width % 8)
    return fail(AJQ_ERR_SHAPE, "ajqd_streams_norm: unsupported shape (rows=%d width=%d of %d)", rows, true_width, width);
  if (!known(dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_streams_norm: unknown dtype %d", dtype);
  with_types(dtype, dtype, [&](auto t, auto) {
    using T = decltype(t);
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(rows), dim3(256), 0, (hipStream_t)stream, x, delta, scale, out, mix, in, gain, eps, (T*)normed, u,
                         streams, true_width, width);
    };
    switch (stream_room(streams)) {
      case 2: go(streams_norm_kernel<T, 2>); break;
      case 4: go(streams_norm_kernel<T, 4>); break;
      default: go(streams_norm_kernel<T, kMaxStreams>); break;
    }
  });
  return check_launch("ajqd_streams_norm");
}

static int dense_out_streams(const char* name, DenseOutStreams d, void* stream) {
  const int batch = d.batch, k = d.K, width = d.Dp, streams = d.streams;
  if (!d.in || !d.w || !d.x || !d.scale || !d.out || !d.mix) return fail(AJQ_ERR_NULL, "%s: null pointer argument", name);
  if (int e = check_streams(streams, name)) return e;
  if (batch < 1 || k < 8 || k % 8 || width < 16 || width % 16)
    return fail(AJQ_ERR_SHAPE, "%s: unsupported shape (batch=%d k=%d width=%d)", name, batch, k, width);
  const OutCut c = out_cut(batch, width, k, !d.u, streams);
  auto pick = [&](auto room) {
    return with_out_cut<(room() > 4)>(c, [&](auto waves, auto rows, auto rt, auto bt, auto uq, auto xq) {
      hipLaunchKernelGGL((dense_out_streams_kernel<waves(), rows(), rt(), bt(), uq(), xq(), decltype(room)::value>), c.grid, dim3(c.threads), 0,
                         (hipStream_t)stream, d);
      return check_launch(name);
    });
  };
  switch (stream_room(streams)) {
    case 2: return pick(std::integral_constant<int, 2>{});
    case 4: return pick(std::integral_constant<int, 4>{});
    default: return pick(std::integral_constant<int, kMaxStreams>{});
  }
}

int ajqd_dense_out_streams(const void* in, const void* w, float* x, const float* scale, const float* out, const float* mix,
                           const float* next, float* u, int streams, int batch, int k, int width, void* stream) {
  if (!u) return fail(AJQ_ERR_NULL, "ajqd_dense_out_streams: null pointer argument");
  return dense_out_streams("ajqd_dense_out_streams", DenseOutStreams{(const uint16_t*)in, (const uint16_t*)w, x, scale, out, mix, next, u, nullptr,
                                                                     nullptr, nullptr, batch, k, width, streams}, stream);
}

int ajqd_dense_out_parts(int batch, int width) { return batch < 1 || width < 16 || width % 16 ? 0 : width / out_cut(batch, width, kTwoWaveColumns, true, 1).rows; }

int ajqd_dense_out_form(int batch, int k, int width, int streams, int scaled) {
  if (batch < 1 || k < 8 || k % 8 || width < 16 || width % 16 || streams < 0 || streams > kMaxStreams) return 0;
  const OutCut c = out_cut(batch, width, k, scaled != 0, streams < 1 ? 1 : streams);
  return 100000 * (c.threads / 64) + 10000 * (c.rows / 8) + 1000 * c.rt + 100 * c.bt + 10 * c.uq + (c.xq > 0 ? c.xq : 0);
}

int ajqd_dense_out_streams_scaled(const void* in, const void* w, float* x, const float* scale, const float* out, const float* mix,
                                  const float* next, const float* gain, void* scaled, float* sums, int streams, int batch, int k, int width,
                                  void* stream) {
  if (!gain || !scaled || !sums) return fail(AJQ_ERR_NULL, "ajqd_dense_out_streams_scaled: null pointer argument");
  return dense_out_streams("ajqd_dense_out_streams_scaled", DenseOutStreams{(const uint16_t*)in, (const uint16_t*)w, x, scale, out, mix, next, nullptr,
                                                                            gain, (uint16_t*)scaled, sums, batch, k, width, streams}, stream);
}

int ajqd_activation(const void* y, void* out, int64_t count, int act, int dtype, void* stream) {
  if (!y || !out) return fail(AJQ_ERR_NULL, "ajqd_activation: null pointer argument");
  if (count < 8 || count % 8 || count / 8 / 256 > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_activation: unsupported count %lld", (long long)count);
  if (!aligned16(y) || !aligned16(out)) return fail(AJQ_ERR_ALIGN, "ajqd_activation: buffers must be 16-byte aligned");
  if (!known(dtype) || act < 0 || act > AJQD_ACT_SQUARED_RELU) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_activation: unknown dtype or activation");
  with_types(dtype, dtype, [&](auto t, auto) {
    using T = decltype(t);
    hipLaunchKernelGGL(activation_kernel<T>, dim3((unsigned)((count / 8 + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (const T*)y, (T*)out,
                       (long long)count / 8, act);
  });
  return check_launch("ajqd_activation");
}

// ---- grouped-query attention
int ajqd_key_value_split(const ajqd_key_value_split_args* a, int y_dtype, int dtype, void* stream) {
  if (!a || !a->y || !a->q_gain || !a->k_gain || (a->rot && !a->half_turns) || !a->q || !a->rows)
    return fail(AJQ_ERR_NULL, "ajqd_key_value_split: null pointer argument");
  if (a->tokens < 1 || a->seq < 1 || a->tokens % a->seq || a->heads < 1 || a->groups < 1 || a->dim < 1 || a->dimp < a->dim || a->dimp % 16 ||
      a->rot < 0 || a->rot % 2 || a->rot > a->dim || a->start < 0 || a->ldy < (a->heads + a->groups) * a->dimp || a->ldy % 4 || a->q_at < 0 ||
      a->q_at % 4 || a->q_ld < a->q_at + a->dimp || a->q_ld % 4 || a->prior < 0 || a->rows_batch < 0 || a->rows_head < 0 || a->rows_batch % 8 ||
      a->rows_head % 8 || (a->pos ? (a->seq != 1 || a->cap < 1 || a->kept < 0 || a->kept >= a->cap) : (int64_t)a->start + a->seq > 0x7FFFFFFF))
    return fail(AJQ_ERR_SHAPE, "ajqd_key_value_split: unsupported shape (tokens=%d seq=%d heads=%d groups=%d dim=%d/%d rot=%d cap=%d kept=%d)",
                a->tokens, a->seq, a->heads, a->groups, a->dim, a->dimp, a->rot, a->cap, a->kept);
  const int64_t need = (int64_t)(a->pos ? a->cap : a->prior + a->seq) * 2 * a->dimp;
  if ((a->groups > 1 && a->rows_head < need) || (a->tokens > a->seq && a->rows_batch < need))
    return fail(AJQ_ERR_SHAPE, "ajqd_key_value_split: rows of neighbouring heads or sequences overlap");
  if (!known(dtype) || !known(y_dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_key_value_split: unknown dtype");
  if (!aligned16(a->y) || !aligned16(a->q) || !aligned16(a->rows)) return fail(AJQ_ERR_ALIGN, "ajqd_key_value_split: rows must be 16-byte aligned");
  KeyValueSplit k;
  k.y = a->y; k.ldy = a->ldy; k.s = KeyValueShape{a->heads, a->groups, a->dim, a->dimp, a->rot, a->eps};
  k.q_gain = a->q_gain; k.k_gain = a->k_gain; k.half_turns = a->half_turns; k.start = a->start; k.pos = positions64(a->pos);
  k.seq = a->seq; k.prior = a->prior; k.cap = a->cap; k.kept = a->kept; k.q = a->q; k.q_ld = a->q_ld; k.q_at = a->q_at;
  k.rows = a->rows; k.rows_batch = a->rows_batch; k.rows_head = a->rows_head;
  const int bytes = 4 * 2 * ((a->rot / 2 + 3) & ~3);
  int status = AJQ_OK;
  with_types(y_dtype, dtype, [&](auto yt, auto t) {
    using Y = decltype(yt);
    using T = decltype(t);
    const bool quads = (a->rot / 2) % 4 == 0 && a->dimp <= 256;
    auto go = [&](auto lanes, auto whole) {
      constexpr int L = decltype(lanes)::value;
      auto kernel = key_value_split_kernel<Y, T, L, decltype(whole)::value>;
      // few tokens: a head per team, so that the heads of a token go side by side
      const int teams = 256 / L, slices = a->tokens < 256 ? (a->heads + a->groups + teams - 1) / teams : 1;
      status = allow_lds(kernel, bytes, "ajqd_key_value_split");
      if (status == AJQ_OK) hipLaunchKernelGGL(kernel, dim3(a->tokens, slices), dim3(256), bytes, (hipStream_t)stream, k);
    };
    auto pick = [&](auto whole) {
      if (a->dimp <= 64) go(std::integral_constant<int, 16>{}, whole);
      else if (a->dimp <= 128) go(std::integral_constant<int, 32>{}, whole);
      else go(std::integral_constant<int, 64>{}, whole);
    };
    if (quads) pick(std::true_type{});
    else pick(std::false_type{});
  });
  return status != AJQ_OK ? status : check_launch("ajqd_key_value_split");
}

int ajqd_group_decode_built(int share, int dimp, int rot) {
  return share >= 1 && share <= kGroupShare && dimp >= 16 && dimp % 16 == 0 && latent_steps(2 * dimp) > 0 && latent_steps(2 * dimp) <= 10 && rot >= 0 && rot % 8 == 0;
}

// Heads of up to 128 columns: two workgroups share a CU and one's front runs beside the other's rows (160 shapes: 0.84 of the time of two launches, the
// most 1.02).  Wider ones have a CU each, so the front is paid once a round and only one round may be; it takes a turn per four heads (up to 7 heads: 160
// shapes 0.70 .. 1.02), and with a third turn pays where the rings are long enough to fill the chip (8 heads, 256 workgroups: 0.82 .. 0.96, 1.07 at the
// first positions; 2 to 128: 0.88 .. 1.10; 16 heads: 0.93 .. 1.25; 26 x 10 workgroups, two rounds: 1.08 .. 1.39).
int ajqd_group_decode_better(int units, int share, int dimp, int rot, int chunks) {
  if (!ajqd_group_decode_built(share, dimp, rot) || units < 1 || chunks < 1) return 0;
  const long long workgroups = (long long)units * chunks;
  return dimp <= 128 || (workgroups <= kCus && (share <= 7 || (share <= 11 && workgroups > 128)));
}

int ajqd_group_decode(const ajqd_key_value_split_args* a, float* partial, int chunks, float scale, void* stream) {
  if (!a || !partial || !a->y || !a->q_gain || !a->k_gain || (a->rot && !a->half_turns) || !a->rows || !a->pos)
    return fail(AJQ_ERR_NULL, "ajqd_group_decode: null pointer argument");
  if (a->tokens < 1 || a->seq != 1 || a->groups < 1 || a->heads < 1 || a->heads % a->groups || a->dim < 1 || a->dimp < a->dim || a->rot > a->dim ||
      a->ldy < (a->heads + a->groups) * a->dimp || a->ldy % 4 || a->cap < 1 || a->kept < 0 || a->kept >= a->cap || a->prior != 0 ||
      a->rows_head != (int64_t)a->cap * 2 * a->dimp || a->rows_batch != a->groups * a->rows_head || chunks < 1 || chunks > kLatentMaxChunks || !(scale > 0.f))
    return fail(AJQ_ERR_SHAPE, "ajqd_group_decode: unsupported shape (tokens=%d heads=%d groups=%d dim=%d/%d rot=%d cap=%d kept=%d chunks=%d)", a->tokens,
                a->heads, a->groups, a->dim, a->dimp, a->rot, a->cap, a->kept, chunks);
  const int share = a->heads / a->groups;
  if (!ajqd_group_decode_built(share, a->dimp, a->rot))
    return fail(AJQ_ERR_UNSUPPORTED, "ajqd_group_decode: %d heads of %d columns, %d of them turned, are not built", share, a->dimp, a->rot);
  if (!aligned16(a->y) || !aligned16(a->rows) || !aligned16(a->q_gain) || !aligned16(a->k_gain))
    return fail(AJQ_ERR_ALIGN, "ajqd_group_decode: rows must be 16-byte aligned");
  const long long units = (long long)a->tokens * a->groups;
  if (units * chunks > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_group_decode: too many workgroups");
  LatentDecode d{nullptr, (const uint16_t*)a->rows, positions64(a->pos), partial, heads_at(partial, (int)units, share, chunks, a->dimp), (int)units, share,
                 a->dimp, 2 * a->dimp, a->cap, chunks, a->dimp / 32, scale * kLog2eF};
  GroupRow k{(const float*)a->y, a->q_gain, a->k_gain, a->half_turns, a->ldy, a->groups, a->dim, a->rot, a->kept, a->eps};
  auto go = [&](auto kernel, int ks) {
    const int bytes = latent_decode_lds(ks, 1);
    if (int e = allow_lds(kernel, bytes, "ajqd_group_decode")) return e;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(units * chunks)), dim3(256), bytes, (hipStream_t)stream, d, k);
    return check_launch("ajqd_group_decode");
  };
  switch (latent_steps(2 * a->dimp)) {
    case 4: return go(group_decode_kernel<4>, 4);
    case 6: return go(group_decode_kernel<6>, 6);
    case 8: return go(group_decode_kernel<8>, 8);
    default: return go(group_decode_kernel<10>, 10);
  }
}

int ajqd_group_merge(const float* partial, const float* gate, int gate_ld, void* out, int out_ld, int batch, int groups, int share,
                     int chunks, int dimp, void* stream) {
  if (!partial || !out) return fail(AJQ_ERR_NULL, "ajqd_group_merge: null pointer argument");
  if (batch < 1 || groups < 1 || share < 1 || chunks < 1 || chunks > kLatentMaxChunks || dimp < 16 || dimp % 16 || dimp > 1024 ||
      out_ld < groups * share * dimp || out_ld % 4 || (gate && (gate_ld < groups * share * dimp || gate_ld % 4)) ||
      (long long)batch * groups * share > 0x7FFFFFFFll)
    return fail(AJQ_ERR_SHAPE, "ajqd_group_merge: unsupported shape (batch=%d groups=%d share=%d chunks=%d dimp=%d)", batch, groups, share,
                chunks, dimp);
  GroupMerge m{partial, heads_at(partial, batch * groups, share, chunks, dimp), gate, (uint16_t*)out, groups, share, chunks, dimp, gate_ld, out_ld};
  hipLaunchKernelGGL(group_merge_kernel, dim3(batch * groups * share), dim3(256), 0, (hipStream_t)stream, m);
  return check_launch("ajqd_group_merge");
}

// ---- selective scan
int ajqd_conv_silu(const void* y, int ldy, void* ring, const float* weight, const float* bias, int start, const int64_t* pos, int rows,
                   int seq, int inner, int taps, void* out, int dtype, void* stream) {
  if (!y || !weight || !bias || !out || (!ring && taps > 1 && (start > 0 || pos))) return fail(AJQ_ERR_NULL, "ajqd_conv_silu: null pointer argument");
  if (rows < 1 || seq < 1 || rows % seq || inner < 8 || inner % 8 || taps < 1 || ldy < inner || ldy % 8 || start < 0 || (pos && seq != 1))
    return fail(AJQ_ERR_SHAPE, "ajqd_conv_silu: unsupported shape (rows=%d seq=%d inner=%d taps=%d ldy=%d)", rows, seq, inner, taps, ldy);
  if (!known(dtype)) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_conv_silu: unknown dtype %d", dtype);
  if (!aligned16(y) || !aligned16(ring) || !aligned16(out)) return fail(AJQ_ERR_ALIGN, "ajqd_conv_silu: rows must be 16-byte aligned");
  const long long blocks = ((long long)rows * (inner / 8) + 255) / 256;
  if (blocks > 0x7FFFFFFFll) return fail(AJQ_ERR_SHAPE, "ajqd_conv_silu: too many elements");
  ConvSilu c{y, ldy, ring, weight, bias, start, positions64(pos), rows, seq, inner, taps, out};
  const long long run_blocks = ((long long)(rows / seq) * ((seq + kConvTokens - 1) / kConvTokens) * (inner / 8) + 255) / 256;
  with_types(dtype, dtype, [&](auto t, auto) {
    using T = decltype(t);
    auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)run_blocks), dim3(256), 0, (hipStream_t)stream, c); };
    if (!pos && taps == 2) return run(conv_silu_run_kernel<T, 2>);
    if (!pos && taps == 3) return run(conv_silu_run_kernel<T, 3>);
    if (!pos && taps == 4) return run(conv_silu_run_kernel<T, 4>);
    hipLaunchKernelGGL(conv_silu_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, c);
  });
  return check_launch("ajqd_conv_silu");
}

}  // extern "C"
namespace {
int check_scan(const char* name, const ajqd_scan_args* a, int dtype) {
  if (!a || !a->x || !a->dt || !a->low || !a->z || !a->a2 || !a->d || !a->dt_bias || !a->out || (!a->state && (a->start > 0 || a->pos)))
    return fail(AJQ_ERR_NULL, "%s: null pointer argument", name);
  if (a->batch < 1 || a->batch > 65535 || a->seq < 1 || a->inner < 8 || a->inner % 8 || a->states < 4 || a->states % 4 || a->start < 0 ||
      a->dt_ld < a->inner || a->dt_ld % 8 || a->z_ld < a->inner || a->z_ld % 8 || a->out_ld < a->inner || a->out_ld % 8 || a->b_col < 0 ||
      a->c_col < 0 || a->low_ld < a->b_col + a->states || a->low_ld < a->c_col + a->states || (a->pos && a->seq != 1))
    return fail(AJQ_ERR_SHAPE, "%s: unsupported shape (batch=%d seq=%d inner=%d states=%d)", name, a->batch, a->seq, a->inner, a->states);
  if (!known(dtype)) return fail(AJQ_ERR_UNSUPPORTED, "%s: unknown dtype %d", name, dtype);
  if (!aligned16(a->x) || !aligned16(a->dt) || !aligned16(a->z) || !aligned16(a->out) || !aligned16(a->d) || !aligned16(a->dt_bias))
    return fail(AJQ_ERR_ALIGN, "%s: rows must be 16-byte aligned", name);
  return AJQ_OK;
}
Scan device_scan(const ajqd_scan_args* a) {
  return Scan{a->x, a->dt, a->low, a->z, a->a2, a->d, a->dt_bias, a->state, a->start, positions64(a->pos), a->seq, a->inner, a->states,
              a->dt_ld, a->low_ld, a->b_col, a->c_col, a->z_ld, a->out_ld, a->out};
}
}  // namespace
extern "C" {

int ajqd_scan(const ajqd_scan_args* a, int dtype, void* stream) {
  if (int e = check_scan("ajqd_scan", a, dtype)) return e;
  const Scan s = device_scan(a);
  return dtype == AJQD_BF16 ? launch_scan<uint16_t>(s, a->batch, (hipStream_t)stream) : launch_scan<float>(s, a->batch, (hipStream_t)stream);
}

int ajqd_scan_parts(int batch, int seq, int inner, int states) {
  if (batch < 1 || seq < 1 || inner < 8 || states < 1 || states > 16) return 1;
  // The states are gone through twice then, so it pays where one piece leaves a SIMD with fewer than four waves (us, one piece against
  // parts: 8192 channels, 1500 tokens 168 / 120, 192 tokens 30 / 23; 2048 channels, 2048 tokens 160 / 53, 192 tokens 16.5 / 13.9; 12288
  // channels, 700 tokens 97 / 85; but 16384, 700 tokens 106 / 106, and 128 tokens of 8192 channels 15.2 / 16.9).  About four waves on
  // every SIMD, parts of one tile of tokens at least: few parts of a short prompt are slower than one piece (300 tokens of 2048
  // channels: 23 in one, 37 in two, 19 in six).
  const long long channels = (long long)batch * inner;
  if (channels >= 16384 || seq < 192) return 1;
  const long long tiles = (seq + kScanPartTokens - 1) / kScanPartTokens;
  return (int)std::min({tiles, std::max(6LL, 4 * 65536 / (channels * kScanPartLanes)), 128LL});  // (a part goes through all ends before it)
}
size_t ajqd_scan_workspace(int batch, int inner, int states, int parts) {
  return parts > 1 ? ((size_t)parts * states + parts - 1) * batch * inner * sizeof(float) : 0;
}
int ajqd_scan_in_parts(const ajqd_scan_args* a, int parts, float* workspace, int dtype, void* stream) {
  if (int e = check_scan("ajqd_scan_in_parts", a, dtype)) return e;
  if (parts < 2) return ajqd_scan(a, dtype, stream);
  if (a->states > 16 || a->pos) return fail(AJQ_ERR_UNSUPPORTED, "ajqd_scan_in_parts: up to 16 states of a prompt are built (%d)", a->states);
  if (!workspace) return fail(AJQ_ERR_NULL, "ajqd_scan_in_parts: null workspace");
  const int tiles = (a->seq + kScanPartTokens - 1) / kScanPartTokens;
  parts = std::min(parts, tiles);
  const int length = (tiles + parts - 1) / parts * kScanPartTokens;
  const int count = (a->seq + length - 1) / length;
  if (count < 2) return ajqd_scan(a, dtype, stream);
  if (count > 65535) return fail(AJQ_ERR_SHAPE, "ajqd_scan_in_parts: %d parts", count);
  const ScanParts cut{workspace, workspace + (size_t)count * a->batch * a->inner * a->states, length};
  const Scan s = device_scan(a);
  return dtype == AJQD_BF16 ? launch_scan_parts<uint16_t, 4>(s, a->batch, count, cut, (hipStream_t)stream)
                            : launch_scan_parts<float, 4>(s, a->batch, count, cut, (hipStream_t)stream);
}

// scan_project: the smallest block that holds a part; two row tiles, which share the convolution, where single ones are more than one a CU
struct ScanCut {
  int kb, rt;
};
static ScanCut scan_cut(int batch, int inner, int rows, int splits) {
  const int part = 32 * (((inner + 31) / 32 + splits - 1) / splits);
  const long long tiles = (long long)(rows / 16) * splits * ((batch + kGemvBatch - 1) / kGemvBatch);
  return ScanCut{part <= scan_block(2) ? 2 : part <= scan_block(4) ? 4 : 8, tiles > kCus && rows >= 32 ? 2 : 1};
}
// scan_step: sequences a workgroup of the wide kernel, 0 for the narrow one (a workgroup per CU).  Eight read the weights and decays less often, four
// carry half a lane's chain.  Three workgroups of four find room on a CU, two of eight: eight where they take one round instead of two (us with four /
// eight: 24 of 8192 channels 12.7 / 13.8; 13 of 13440 13.3 / 11.6, 33 of 6672 with 64 states 28.3 / 25.4; 16 of 17360 18.2 / 20.5, 13 of
// 18576 with 64 states 48.4 / 61.9) and past two rounds of four (31 of 13440 33.6 / 30.3, 33 of 13744 33.6 / 30.1), unless there are many states, which lie
// in a lane's chain (64 states, 64 of 9664: 89 / 100; 48 of 6992: 48 / 63).
static int scan_step_batch(int batch, int inner, int rank, int states) {
  if (rank <= kNarrowRank && (long long)(inner / 16) * ((batch + kNarrowBatch - 1) / kNarrowBatch) <= kCus) return 0;
  const long long fours = (long long)((inner + 63) / 64) * ((batch + 3) / 4);
  return (fours > 3 * kCus && fours <= 4 * kCus) || (fours > 6 * kCus && states <= 32) ? 8 : 4;
}

int ajqd_scan_form(int batch, int inner, int rows, int splits, int rank, int states) {
  if (batch < 1 || inner < 16 || inner % 16 || rows < 16 || rows % 16 || splits < 1 || rank < 8 || states < 4) return 0;
  const ScanCut c = scan_cut(batch, inner, rows, splits);
  return 1000 * c.kb + 100 * c.rt + 10 * (rows / 16 % 2) + scan_step_batch(batch, inner, rank, states);
}

// Parts of the projection: what smaller blocks save in scan_project_kernel, the step's kernel pays in parts (0.04 us a part at
// 4 sequences, 0.15 at 16 of 8192 channels, 0.13 at 64 of 4096).  Both launches with blocks of 1024 / 512 / 256: 4 sequences
// of 4096 channels 9.6 / 8.5 / 8.3 us, 16: 15.2 / 12.2 / 11.2, 64: 22.5 / 20.1 / 21.0; 5120, 12: 14.1 / 12.0 / 11.6; 8192, 1: 10.6 / 10.9 / 11.5,
// 8: 14.3 / 14.3 / 15.7, 16: 19.1 / 18.2 / 19.5, 24: 22.4 / 21.9 / 24.5, 32: 24.5 / 24.8 (512), 64: 40.0 / 42.6 / 48.6.  Few sequences of more than 4096
// channels pay the parts and have little to convolve: 2 of 4640, rank 288, 9.4 / 9.4 / 9.8; 3 of 4960, 128 states, 22.0 / 22.1 / 23.2.
int ajqd_scan_splits(int batch, int inner) {
  const int block = inner <= 5120 ? scan_block(batch > 32 || (batch <= 4 && inner > 4096) ? 4 : 2) : scan_block(batch > 8 && batch <= 24 && inner <= 10240 ? 4 : 8);
  const int s = (inner + block - 1) / block, most = inner <= 10240 ? 20 : 8;  // (not timed past 10240 channels: as it was)
  return s < 1 ? 1 : s > most ? most : s;
}

int ajqd_scan_project(const float* y, int ldy, const void* ring, const float* weight, const float* bias, const int64_t* pos, const void* w,
                      float* partial, int batch, int inner, int taps, int rows, int splits, void* stream) {
  if (!y || !weight || !bias || !pos || !w || !partial || (!ring && taps > 1)) return fail(AJQ_ERR_NULL, "ajqd_scan_project: null pointer argument");
  if (batch < 1 || inner < 8 || inner % 8 || taps < 1 || rows < 16 || rows % 16 || splits < 1 || splits > 65535 || ldy < 2 * inner || ldy % 4)
    return fail(AJQ_ERR_SHAPE, "ajqd_scan_project: unsupported shape (batch=%d inner=%d taps=%d rows=%d splits=%d)", batch, inner, taps, rows, splits);
  ScanProject p{y, (const uint16_t*)ring, weight, bias, positions64(pos), (const uint16_t*)w, partial, batch, ldy, inner, taps, rows, splits};
  const ScanCut c = scan_cut(batch, inner, rows, splits);
  const int kb = c.kb, rt = c.rt;
  const dim3 grid((rows / 16 + rt - 1) / rt, splits, (batch + kGemvBatch - 1) / kGemvBatch);
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, (hipStream_t)stream, p); };
  auto with = [&](auto steps) {
    constexpr int S = decltype(steps)::value;
    if (taps == 4) rt == 2 ? go(scan_project_kernel<2, 4, S>) : go(scan_project_kernel<1, 4, S>);
    else rt == 2 ? go(scan_project_kernel<2, 0, S>) : go(scan_project_kernel<1, 0, S>);
  };
  kb == 2 ? with(Int<2>{}) : kb == 4 ? with(Int<4>{}) : with(Int<8>{});
  return check_launch("ajqd_scan_project");
}

int ajqd_scan_step(const ajqd_scan_step_args* a, void* stream) {
  if (!a || !a->y || !a->weight || !a->bias || !a->pos || !a->partial || !a->w_dt || !a->dt_bias || !a->a2 || !a->d || !a->state || !a->out ||
      (!a->ring && a->taps > 1))
    return fail(AJQ_ERR_NULL, "ajqd_scan_step: null pointer argument");
  if (a->batch < 1 || a->inner < 16 || a->inner % 16 || a->taps < 1 || a->rank < 8 || a->rank % 8 || a->states < 4 || a->states % 4 ||
      a->rows < a->rank + 2 * a->states || a->splits < 1 || a->ldy < 2 * a->inner || a->out_ld < a->inner)
    return fail(AJQ_ERR_SHAPE, "ajqd_scan_step: unsupported shape (batch=%d inner=%d rank=%d states=%d rows=%d)", a->batch, a->inner, a->rank,
                a->states, a->rows);
  ScanStep s{a->y, (uint16_t*)a->ring, a->weight, a->bias, positions64(a->pos), a->partial, (const uint16_t*)a->w_dt, a->dt_bias, a->a2, a->d,
             a->state, (uint16_t*)a->out, a->batch, a->ldy, a->inner, a->taps, a->rows, a->splits, a->rank, a->states, a->out_ld};
  auto go = [&](auto kernel, int channels, int bb) {
    const int bytes = scan_step_lds(a->rank, a->states, bb);
    if (int e = allow_lds(kernel, bytes, "ajqd_scan_step")) return e;
    hipLaunchKernelGGL(kernel, dim3((a->inner + channels - 1) / channels, (a->batch + bb - 1) / bb), dim3(256), bytes, (hipStream_t)stream, s);
    return check_launch("ajqd_scan_step");
  };
  switch (scan_step_batch(a->batch, a->inner, a->rank, a->states)) {
    case 0: return go(scan_step_narrow_kernel, 16, kNarrowBatch);
    case 4: return go(scan_step_kernel<4>, 64, 4);
    default: return go(scan_step_kernel<8>, 64, 8);
  }
}

}  // extern "C"
