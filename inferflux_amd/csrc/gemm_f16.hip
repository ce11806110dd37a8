// gemm_f16.hip -- launch planning of the prefill GEMM (gemm_f16.h) and the
// kernels around it: the activation pre-pass and the ordered K-split sum.
#include "gemm_f16.h"

#include <algorithm>
#include <cmath>
#include <mutex>

namespace ifx {

hipError_t launch_gemm_f16_q4(int tile, bool ah, const F16Args &g, int grid, hipStream_t s);
hipError_t launch_gemm_f16_q6(int tile, bool ah, const F16Args &g, int grid, hipStream_t s);
hipError_t launch_gemm_f16_q8(int tile, bool ah, const F16Args &g, int grid, hipStream_t s);

// Q8_1 activations -> fp16 in the GEMM's staging order (64 bytes per block),
// once per GEMM instead of once per weight tile, with the conversion the
// GEMM applies itself (i8x4_to_h on the block's fp16 d), so both give the
// same bits.  Thread t writes 16 bytes, words 4q..4q+3 of block t/4
// (q = t%4), i.e. codes 8q..8q+7: consecutive threads store consecutive
// 16-byte chunks.
__global__ __launch_bounds__(256) void k_q8_1_to_f16(const uint8_t *__restrict__ A,
                                                     u32x4 *__restrict__ out, int64_t nchunks) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (t >= nchunks) return;
  const uint8_t *src = A + (t >> 2) * kQ8_1Bytes;
  const int q = static_cast<int>(t & 3);
  const h2 d = splat(h2f(ldg<uint32_t>(src) & 0xFFFFu));
  const u32x2 c = ldg<u32x2>(src + 4 + 8 * q);
  uint32_t o[4];
  i8x4_to_h(c.x, d, o[0], o[1]);
  i8x4_to_h(c.y, d, o[2], o[3]);
  out[t] = u32x4{o[0], o[1], o[2], o[3]};
}

// The ordered reduction of a launch with slots: y = ((s_0 + s_1) + ...) over
// the splits' slots in split order, then the epilogue (mode 1: + Y, 2:
// + bias[n]).  Four consecutive outputs per thread (16-byte accesses when
// M * N % 4 == 0 and Y is 16-byte aligned).
__global__ __launch_bounds__(256) void k_split_sum(const float *__restrict__ slots,
                                                   float *__restrict__ Y,
                                                   const float *__restrict__ bias, int64_t mn,
                                                   int N, int splits, int mode) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i >= mn) return;
  if ((mn & 3) == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0) {
    f32x4 t = *reinterpret_cast<const f32x4 *>(slots + i);
    for (int sp = 1; sp < splits; ++sp) t += *reinterpret_cast<const f32x4 *>(slots + sp * mn + i);
    if (mode == 1) t += *reinterpret_cast<const f32x4 *>(Y + i);
    if (mode == 2) {
      const int n = static_cast<int>(i % N);
      t += f32x4{bias[n], bias[(n + 1) % N], bias[(n + 2) % N], bias[(n + 3) % N]};
    }
    *reinterpret_cast<f32x4 *>(Y + i) = t;
    return;
  }
  for (int64_t k = i; k < mn && k < i + 4; ++k) {
    float t = slots[k];
    for (int sp = 1; sp < splits; ++sp) t += slots[sp * mn + k];
    if (mode == 1) t += Y[k];
    if (mode == 2) t += bias[k % N];
    Y[k] = t;
  }
}

namespace {

// The tiles of launch_by_tile (rows, columns, K waves), and what a launch of
// each costs by quant type (Q4_K, Q6_K, Q8_0): R rounds of 256 workgroups, one
// a CU, and K values a workgroup take R (a + b K / 1024) + c w K / 1024 us, w
// the rounds the workgroups fill.  Fitted to launches with HBM-cold weights.  What
// counts is the choice: over 3069 graph-replayed launches, all tiles at M = 33 to
// 1999, N = 256 to 49152, K = 256 to 27648, the tile with the least cost took 1.007 of
// the best one's time on average, 1.13 at most.  As times the figures are low, by 8 %
// in the median (25 % for nine in ten: mostly K below 1024 and the small tiles).
// One 256 x 256 tile with fp16 weights in LDS for all of them took 65 us at
// 173 x 11008 x 2048 (Q4_K; 27 now) and 147 at 512 x 5120 x 5120 (50): a grid of
// few workgroups leaves CUs idle, and a short batch pads the tile.
struct TileInfo {
  int bm, bn, kw;
  struct {
    float a, b, c;
  } cost[3];
};
constexpr TileInfo kF16Tiles[] = {
    {128, 512, 1, {{17.0f, 19.4f, 7.0f}, {}, {}}},
    {128, 256, 2, {{9.6f, 11.9f, 4.6f}, {}, {9.9f, 17.0f, 3.9f}}},
    {96, 256, 2, {{9.6f, 9.0f, 3.6f}, {8.2f, 14.7f, 3.2f}, {11.1f, 11.2f, 3.7f}}},
    {64, 256, 2, {{7.1f, 7.4f, 2.1f}, {7.5f, 11.9f, 1.7f}, {8.1f, 11.8f, 1.3f}}},
    {64, 128, 4, {{4.9f, 4.8f, 1.1f}, {4.7f, 6.8f, 1.2f}, {5.8f, 6.0f, 0.8f}}},
    {32, 128, 4, {{3.2f, 3.9f, 0.5f}, {3.8f, 5.6f, 0.4f}, {3.8f, 5.3f, 0.7f}}},
    {32, 64, 8, {{3.3f, 2.1f, 0.4f}, {4.3f, 3.1f, 0.5f}, {4.2f, 2.7f, 0.3f}}},
    {128, 256, 1, {{}, {10.4f, 14.1f, 4.2f}, {}}},
    {256, 256, 1, {{}, {14.0f, 26.8f, 5.5f}, {14.9f, 24.0f, 6.9f}}},
    {64, 128, 1, {{3.0f, 7.2f, 0.0f}, {3.4f, 8.1f, 0.0f}, {}}},
};
constexpr int kNTiles = sizeof(kF16Tiles) / sizeof(kF16Tiles[0]);

// Long prompts' narrow projections in order: a launch of kOrderedM rows or more
// whose sums no split along K divides (K-quants, less than kOrderedN columns in
// all) can take the last tile, 64 x 128 without K waves, and takes a tile
// with K waves only where that is slower by more than kOrderedCost.  K and V of
// a 14B layer at M = 1999 (Q4_K 1999 x 1024 x 5120) take 46 us so and 38 with K
// waves, under 1 % of the layer, and all its outputs have the bits of a sum
// over K in steps of 16 (Q, O, gate and up take 128 x 512, down 256 x 256).  K and V of a
// 3B model (256 columns, 20 us against 11), wider projections where the plan takes a
// tile with K waves (1024 x 5120 x 5120, 91 against 74), Q8_0 (59 against 45 at
// 1999 x 1024 x 5120) and shorter prompts (512 x 1024 x 5120, 40 against 19) keep
// the K waves.
constexpr int kOrderedTile = kNTiles - 1;
constexpr int kOrderedM = 1024, kOrderedN = 2048;
constexpr float kOrderedCost = 1.25f;

struct Plan {
  int tile, m_tiles, n_tiles, splits, spw;
};

// Most K splits that a shape may take: as many as fill the chip once over a
// grid of 256 x 256 tiles, keeping 512 values of K each.  This line is part
// of the interface and does not move with the tiles: it says which shapes
// need the ordered reduction's workspace and how much, and which give the
// same bits on every run without it.
int max_splits(int count, const int *N, int M, int K) {
  const int nch = K / 64;
  int most = 256;
  for (int i = 0; i < count; ++i) {
    const int64_t tiles = int64_t{1} * ((M + 255) / 256) * ((N[i] + 255) / 256);
    int sp = tiles < 192 ? std::max(1, std::min(static_cast<int>(256 / tiles), nch / 8)) : 1;
    const int each = (nch + sp - 1) / sp;
    sp = (nch + each - 1) / each;
    most = std::min(most, sp);
  }
  return most;
}

// Tile and K splits of a launch: the cheapest by the table.  Only fp32 outputs
// split (their partial sums meet in Y by atomics, or in slots), when the tiles
// alone do not fill the CUs, up to max_splits; the reduction adds about 4 us and,
// a megabyte of partial sums, 0.5 us with atomics and 0.25 in slots (planned alike,
// the ordered 200 x 5120 x 5120 Q8_0 did not split, 44 us; in slots 37.)  What the
// ordered plan does not split the other does not either, its splits cost more.
// A launch that would leave three quarters of the CUs idle always splits.
// splits_req > 0 forces the count (tests; at most one split per group of stages).
Plan f16_plan(int qt, bool f16, bool ordered, int count, const int *N, int M, int K, int splits_req) {
  const int ty = qt == kTypeQ4_K ? 0 : qt == kTypeQ6_K ? 1 : 2;
  const int nch = K / kBK;
  const int forced = [] {  // IFX_F16_TILE (tuning)
    const char *e = tuning_env("IFX_F16_TILE");
    return e ? atoi(e) : -1;
  }();
  const int cap = f16 ? 1 : max_splits(count, N, M, K);
  int64_t n_sum = 0;
  for (int i = 0; i < count; ++i) n_sum += N[i];
  const bool in_order = qt != kTypeQ8_0 && M >= kOrderedM && n_sum < kOrderedN && cap == 1;
  Plan best{};
  float best_cost = 0.0f;
  for (int ti = 0; ti < kNTiles; ++ti) {
    if (forced >= 0 ? ti != forced : ti == kOrderedTile && !in_order) continue;
    const TileInfo &t = kF16Tiles[ti];
    if (t.cost[ty].b == 0.0f) continue;  // not a tile of this type
    Plan p{};
    p.tile = ti;
    p.m_tiles = (M + t.bm - 1) / t.bm;
    int64_t wg = 0;
    for (int i = 0; i < count; ++i) wg += (N[i] + t.bn - 1) / t.bn;
    p.n_tiles = static_cast<int>(wg);
    wg *= p.m_tiles;
    const int kc = t.kw * (qt == kTypeQ8_0 ? 1 : 2);  // chunks of a group
    const int groups = (nch + kc - 1) / kc;
    int most = 1;
    if (!f16 && wg < 192) most = std::max(1, std::min(static_cast<int>(256 / wg), cap));
    int least = most > 1 && wg <= 64 ? 2 : 1;
    if (splits_req > 0 && !f16) least = most = splits_req;
    for (int sp = least; sp <= most; ++sp) {
      p.spw = (groups + sp - 1) / sp;
      p.splits = (groups + p.spw - 1) / p.spw;
      const float w = static_cast<float>(wg * p.splits) / 256.0f, rounds = std::ceil(w);
      const float k = static_cast<float>(std::min(p.spw * kc, nch) * kBK) / 1024.0f;
      float cost = rounds * (t.cost[ty].a + t.cost[ty].b * k) + t.cost[ty].c * w * k;
      if (in_order && t.kw > 1) cost *= kOrderedCost;
      if (p.splits > 1) cost += 4.0f + (ordered ? 1e-6f : 2e-6f) * p.splits * static_cast<float>(n_sum) * M;
      if (best_cost == 0.0f || cost < best_cost) best_cost = cost, best = p;
    }
  }
  return best;
}

// slots: NULL, or the ordered reduction's slots (splits x M x N fp32) for a
// launch that splits K (one projection).
hipError_t launch_qt(int qtype, int count, const void *const *W, const uint8_t *A, void *A16, void *const *Y,
                     const int *N, const void *bias, bool f16, int M, int K, int mode,
                     int splits_req, float *slots, hipStream_t s) {
  const Plan p = f16_plan(qtype, f16, slots != nullptr, count, N, M, K, splits_req);
  const TileInfo &t = kF16Tiles[p.tile];
  F16Args g{};
  for (int i = 0, end = 0; i < kMaxSeg; ++i) {
    const int k = i < count ? i : count - 1;
    if (i < count) end += (N[i] + t.bn - 1) / t.bn;
    g.seg[i] = {static_cast<const uint8_t *>(W[k]), Y[k], N[k], end};
  }
  g.A = A;
  g.bias = bias;
  g.M = M;
  g.K = K;
  g.mode = mode;
  g.m_tiles = p.m_tiles;
  g.splits = p.splits;
  g.spw = p.spw;
  const bool ordered = p.splits > 1 && slots;
  g.epi = ordered ? kEpiSlot : p.splits > 1 ? kEpiAtomic : f16 ? kEpiF16 : kEpiF32;
  if (ordered) g.seg[0].Y = slots;
  g.vec = 1;
  for (int i = 0; i < count; ++i)
    if (N[i] % (f16 ? 8 : 4) || reinterpret_cast<uintptr_t>(g.seg[i].Y) % 16) g.vec = 0;
  if (g.epi == kEpiAtomic && mode != 1) {  // store / bias: the workgroups add into a zeroed Y
    FillArgs f{};
    for (int i = 0; i < count; ++i) {
      f.y[i] = static_cast<float *>(Y[i]);
      f.n[i] = static_cast<int64_t>(M) * N[i];
    }
    if (launch_fill_zero(f, count, s) != hipSuccess) return last_error();
  }
  const int grid = p.m_tiles * p.n_tiles * p.splits;
  if (A16) {
    const int64_t nchunks = static_cast<int64_t>(M) * (K >> 5) * 4;
    IFX_LAUNCH0(k_q8_1_to_f16, dim3(static_cast<unsigned>((nchunks + 255) / 256)), dim3(256), 0, s,
                A, static_cast<u32x4 *>(A16), nchunks);
    const hipError_t e = last_error();
    if (e != hipSuccess) return e;
    g.A = static_cast<const uint8_t *>(A16);
  }
  const hipError_t e = qtype == kTypeQ4_K   ? launch_gemm_f16_q4(p.tile, A16 != nullptr, g, grid, s)
                       : qtype == kTypeQ6_K ? launch_gemm_f16_q6(p.tile, A16 != nullptr, g, grid, s)
                                            : launch_gemm_f16_q8(p.tile, A16 != nullptr, g, grid, s);
  if (e != hipSuccess || !ordered) return e;
  const int64_t mn = static_cast<int64_t>(M) * N[0];
  IFX_LAUNCH0(k_split_sum, dim3(static_cast<unsigned>((mn + 1023) / 1024)), dim3(256), 0, s, slots,
              static_cast<float *>(Y[0]), static_cast<const float *>(bias), mn, N[0], p.splits,
              mode);
  return last_error();
}

}  // namespace

bool gemm_f16_fits(int qtype, int K) {
  if (qtype == kTypeQ4_K || qtype == kTypeQ6_K) return K % 256 == 0;
  if (qtype == kTypeQ8_0) return K % kBK == 0;
  return false;
}

// Bytes of the fp16 activation copy (M x K halves), or 0 when they would not fit
// 32 bits.  Part of the interface; launches use a copy below kMaxBufferBytes only.
int64_t gemm_f16_workspace_bytes(int M, int K) {
  const int64_t b = static_cast<int64_t>(M) * K * 2;
  return b < (int64_t{1} << 32) ? b : 0;
}

// Bytes of the ordered reduction's slots (splits x M x N fp32), or 0 when
// the launch does not split K.
int64_t gemm_f16_slot_bytes(int qtype, bool f16, int M, int N, int K) {
  const int splits = f16_plan(qtype, f16, true, 1, &N, M, K, 0).splits;
  return splits > 1 ? static_cast<int64_t>(splits) * M * N * 4 : 0;
}

// splits_req: 0 = chosen from the tile grid, else forced (tests).  A16:
// caller-owned workspace of gemm_f16_workspace_bytes(M, K) bytes (16-byte
// aligned) for the fp16 activations, converted once before the GEMM; NULL:
// each workgroup converts its Q8_1 activation tiles itself.  Same results.
// slots: NULL (K splits add with fp32 atomics into a zeroed Y), or
// gemm_f16_slot_bytes of 16-byte aligned memory for the ordered reduction.
hipError_t launch_gemm_f16_grouped(int qtype, int count, const void *const *W, const void *A,
                                   void *A16, void *const *Y, const int *N, const void *bias,
                                   bool f16, int M, int K, int mode, int splits_req,
                                   hipStream_t stream, float *slots) {
  const uint8_t *a = static_cast<const uint8_t *>(A);
  if (!gemm_f16_fits(qtype, K)) return hipErrorInvalidValue;
  // chunks past K read zeros at kOobOffset, which has to lie past the copy
  const uint64_t copy = gemm_f16_workspace_bytes(M, K);
  if (copy == 0 || copy >= kMaxBufferBytes) A16 = nullptr;
  return launch_qt(qtype, count, W, a, A16, Y, N, bias, f16, M, K, mode, splits_req, slots, stream);
}

hipError_t launch_gemm_f16(int qtype, const void *W, const void *A, void *A16, void *Y,
                           const void *bias, bool f16, int M, int N, int K, int mode,
                           int splits_req, hipStream_t stream, float *slots) {
  return launch_gemm_f16_grouped(qtype, 1, &W, A, A16, &Y, &N, bias, f16, M, K, mode, splits_req,
                                 stream, slots);
}

// ---------------------------------------------------------------------------
// Static workspace of the no-alloc prefill entry (ifx_qgemm_prefill_noalloc):
// the fp16 activation copy lives in this array instead of caller memory.
// Each GPU holds its own copy, at its own address, until the process ends.
// On the host `scratch` names a host-side stand-in, never a device address:
// host code uses only the address hipGetSymbolAddress returns for the
// current device.
static __device__ __align__(256) uint8_t scratch[IFX_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void *g_scratch_ptr[kMaxDevices];  // per device, resolved on first use
}  // namespace

// Device address of `scratch` on the current device, resolved once per
// device with that device current.
hipError_t scratch_address(void **out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (!p) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}

}  // namespace ifx
