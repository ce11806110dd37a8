// gemm_mfma.hip -- int8-MFMA GEMM for prefill and large decode batches
// (M > 32) on gfx950: y[m][n] = sum_k W[n][k] * a[m][k], W raw GGUF Q4_K /
// Q6_K / Q8_0 blocks, a Q8_1 blocks of 32, fp32 accumulate.
//
// The reference has no quantized GEMM above M = 64: it dequantizes W to
// FP16 and calls cuBLAS (runtime/backends/cuda/native/
// quantized_weight_map.cpp:176-233, cublas_gemm.h:47; caller
// transformer_forward.cu:1479), and its MMQ kernels for 9 <= M <= 64
// (kernels/mmq.cuh:41-835) use dp4a.  This kernel keeps the MMQ arithmetic
// of the GEMV path -- an exact integer dot per 32-value block (16-value
// group for Q6_K), then fp32 scaling by the weight and activation block
// scales -- with the integer dot on the matrix cores.
//
// Tiling: a workgroup of one to four 256-thread groups owns a 128 (m) x 128 (n) output tile (64 x
// 64 when that gives fewer than two workgroups per CU); a group's four waves
// are 2 x 2, each owning 2 x 2 (or one) MFMA tiles of 32 x 32.
// A group's K loop steps one 256-value super-block at a time:
//   1. the next super-block's A items (Q8_1 blocks of 128 rows) and raw W
//      bytes (16-byte chunks of 128 rows) are loaded into registers while
//      the current one is computed; at the top of a step they are written
//      to LDS (about 61 KB for Q4_K: two workgroups per CU);
//   2. each wave unpacks W codes to int8 MFMA operands from LDS (Q4_K
//      nibbles; Q6_K 4+2 bits minus 32; Q8_0 as is) and runs
//      v_mfma_i32_32x32x32_i8 per 32-value block (two
//      v_mfma_i32_32x32x16_i8 for Q6_K, whose scales are per 16 values);
//   3. the int32 block results are scaled into fp32 accumulators with
//      three VALU operations per output (scale product, convert, FMA):
//      Q4_K  acc += C * (da * d*sc) - sa * (dmin*m)          (mmvq.cuh:115-125)
//      Q6_K  acc += (sc0*C0 + sc1*C1) * (da * d)             (mmvq.cuh:467-471)
//      Q8_0  acc += C * (da * dw)                            (mmvq.cuh:886-889)
//      The Q4_K min term is an fp32 GEMM over the 8 sub-blocks of a
//      super-block, run on the matrix cores (v_mfma_f32_32x32x2f32) into
//      the same accumulators, so it costs no VALU time.
// This per-block rescaling (the activation d varies per row and per 32
// values, the weight scale per column and per 32 values) is VALU work: at
// three operations per output per block it bounds the kernel near 15 % of the
// int8 MFMA peak.  Not the fewest possible at this exactness: fp16 operands sc q
// (at most 945) and activation codes are whole numbers whose 32-value sums fp32
// holds exactly, which leaves Q4_K one FMA per output and block at half the
// matrix rate (not built).
// MFMA lane layouts (32x32 output): lane l supplies row (l % 32) of A and
// column (l % 32) of B for the K half (l / 32); it receives column l % 32
// and rows 8*(i/4) + 4*(l/32) + (i%4), i = 0..15, of the result.
#include "ifx_common.h"

namespace ifx {

namespace {

constexpr int kApitch = 256 + 16;  // int8 codes per staged A row (+pad vs bank conflicts)

template <int QT>
struct GFmt;
template <>
struct GFmt<kTypeQ4_K> {  // raw super-block per row: 9 chunks of 16 bytes
  static constexpr int kSb = 144, kPitch = 144 + 16, kChunks = 9;
};
template <>
struct GFmt<kTypeQ6_K> {  // 210 bytes; the 14th chunk carries only d
  static constexpr int kSb = 210, kPitch = 224 + 16, kChunks = 14;
};
template <>
struct GFmt<kTypeQ8_0> {  // codes of 8 blocks [row][b*32], d separately
  static constexpr int kSb = 272, kPitch = 256 + 16, kChunks = 0;
};

// Workgroup tile: 64*S x 64*S (m x n); each of the 2 x 2 waves owns S x S
// MFMA tiles of 32 x 32.
template <int QT, int S>
struct Smem {
  static constexpr int kBM = 64 * S, kBN = 64 * S;
  int8_t a[kBM * kApitch];             // activation codes [m][k within super-block]
  float da[8][kBM];                    // Q8_1 d per block, [block][m]
  float sa[8][kBM];                    // Q8_1 s per block, [block][m]
  uint8_t w[kBN * GFmt<QT>::kPitch];   // raw W super-block per row (Q8_0: codes)
  float dw[QT == kTypeQ8_0 ? 8 : 1][kBN];  // Q8_0 per-block weight d
};

// One super-block of the workgroup's tile in a thread's registers.
template <int QT, int S>
struct Prefetch {
  static constexpr int kBM = 64 * S, kBN = 64 * S;
  static constexpr int kAItems = kBM * 8 / 256;  // (row, block) items per thread
  static constexpr int kWItems =
      QT == kTypeQ8_0 ? kBN * 8 / 256 : (kBN * GFmt<QT>::kChunks + 255) / 256;
  uint32_t ads[kAItems];
  i32x4 a0[kAItems], a1[kAItems];
  u32x4 w0[kWItems];
  u32x4 w1[QT == kTypeQ8_0 ? kWItems : 1];  // Q8_0: codes 16-31
  uint32_t wd[QT == kTypeQ8_0 ? kWItems : 1];
};

__device__ __forceinline__ i32x16 mfma32(i32x4 a, i32x4 b) {
  const i32x16 z = {0};
  return __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, z, 0, 0, 0);
}

__device__ __forceinline__ i32x16 mfma16(int64_t a, int64_t b) {
  const i32x16 z = {0};
  return __builtin_amdgcn_mfma_i32_32x32x16_i8(a, b, z, 0, 0, 0);
}

// Q6_K code bytes v in [0, 63] -> int8 (v - 32), four per dword, no carries:
// flip bit 5, then sign-extend the new bit 5 into bits 6 and 7.
__device__ __forceinline__ uint32_t q6_minus32(uint32_t v) {
  uint32_t x = v ^ 0x20202020u;
  const uint32_t t = x & 0x20202020u;
  return x | (t << 1) | (t << 2);
}

template <int QT, int S>
__device__ __forceinline__ void fetch(Prefetch<QT, S> &pf, rsrc_t Wr, rsrc_t Ar, uint32_t w_row,
                                      uint32_t a_row, int m0, int n0, int M, int N, int sblk,
                                      int tid) {
  constexpr int kBN = Prefetch<QT, S>::kBN;
#pragma unroll
  for (int i = 0; i < Prefetch<QT, S>::kAItems; ++i) {
    const int it = tid + 256 * i;
    const int r = it >> 3, b = it & 7;
    pf.ads[i] = 0;
    pf.a0[i] = pf.a1[i] = i32x4{0, 0, 0, 0};
    if (m0 + r < M) {
      const uint32_t o = (m0 + r) * a_row + (sblk * 8 + b) * kQ8_1Bytes;
      pf.ads[i] = bload<uint32_t>(Ar, o, 0);
      pf.a0[i] = bload<i32x4>(Ar, o + 4, 0);
      pf.a1[i] = bload<i32x4>(Ar, o + 20, 0);
    }
  }
  using F = GFmt<QT>;
  if constexpr (QT == kTypeQ8_0) {
#pragma unroll
    for (int i = 0; i < Prefetch<QT, S>::kWItems; ++i) {
      const int it = tid + 256 * i;
      const int r = it >> 3, b = it & 7;
      const uint32_t o = min(n0 + r, N - 1) * w_row + (sblk * 8 + b) * kQ8_0Bytes;
      pf.wd[i] = wload<uint16_t>(Wr, o, 0);
      pf.w0[i] = wload<u32x4>(Wr, o + 2, 0);
      pf.w1[i] = wload<u32x4>(Wr, o + 18, 0);
    }
  } else {
#pragma unroll
    for (int i = 0; i < Prefetch<QT, S>::kWItems; ++i) {
      const int c = tid + 256 * i;
      pf.w0[i] = u32x4{0, 0, 0, 0};
      if (c < kBN * F::kChunks) {
        const int r = c / F::kChunks, part = c - r * F::kChunks;
        const uint32_t o = min(n0 + r, N - 1) * w_row + sblk * F::kSb + 16 * part;
        // the last Q6_K chunk holds only d: a 16-byte load could cross the
        // end of the tensor on its last super-block (and then read zeros)
        if (QT == kTypeQ6_K && part == 13) pf.w0[i].x = wload<uint16_t>(Wr, o, 0);
        else pf.w0[i] = wload<u32x4>(Wr, o, 0);
      }
    }
  }
}

template <int QT, int S>
__device__ __forceinline__ void commit(Smem<QT, S> &sm, const Prefetch<QT, S> &pf,
                                       int tid) {
  constexpr int kBN = Prefetch<QT, S>::kBN;
#pragma unroll
  for (int i = 0; i < Prefetch<QT, S>::kAItems; ++i) {
    const int it = tid + 256 * i;
    const int r = it >> 3, b = it & 7;
    *reinterpret_cast<i32x4 *>(&sm.a[r * kApitch + b * 32]) = pf.a0[i];
    *reinterpret_cast<i32x4 *>(&sm.a[r * kApitch + b * 32 + 16]) = pf.a1[i];
    sm.da[b][r] = h2f(pf.ads[i] & 0xFFFFu);
    sm.sa[b][r] = h2f(pf.ads[i] >> 16);
  }
  using F = GFmt<QT>;
  if constexpr (QT == kTypeQ8_0) {
#pragma unroll
    for (int i = 0; i < Prefetch<QT, S>::kWItems; ++i) {
      const int it = tid + 256 * i;
      const int r = it >> 3, b = it & 7;
      *reinterpret_cast<u32x4 *>(&sm.w[r * F::kPitch + b * 32]) = pf.w0[i];
      *reinterpret_cast<u32x4 *>(&sm.w[r * F::kPitch + b * 32 + 16]) = pf.w1[i];
      sm.dw[b][r] = h2f(pf.wd[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < Prefetch<QT, S>::kWItems; ++i) {
      const int c = tid + 256 * i;
      if (c < kBN * F::kChunks) {
        const int r = c / F::kChunks, part = c - r * F::kChunks;
        *reinterpret_cast<u32x4 *>(&sm.w[r * F::kPitch + 16 * part]) = pf.w0[i];
      }
    }
  }
}

constexpr int kMaxSeg = 3;

// A projection of the launch: its weights, output, rows, and the n tile that
// ends it.
struct MfmaSeg {
  const uint8_t *W;
  void *Y;
  int N, end;
};
struct MfmaArgs {
  MfmaSeg seg[kMaxSeg];
  const uint8_t *A;
  const void *bias;
  int M, K, mode;
};

}  // namespace

// KW groups of four waves share an output tile: group g walks super-blocks
// g, g + KW, ... with an LDS stage of its own, and the groups' sums meet in
// LDS in group order (no atomics; the same bits on every run).  Bound by the
// VALU (three operations per output and block: 9 us of a CU for one 64 x 64
// tile over K = 2048) and, with one group, by each step's load that a single
// wave per SIMD cannot hide.  A launch takes up to three projections of the
// same activations: 3B gate and up (11008 x 2048 Q4_K) at M = 60, two
// launches 42 us, one 26.
template <int QT, int S, bool F16OUT, int KW>
__global__ __launch_bounds__(256 * KW, KW == 1 ? 2 : 4) void k_gemm_mfma(MfmaArgs g) {
  using F = GFmt<QT>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_raw[];
  constexpr int kBM = 64 * S, kBN = 64 * S;
  const int kg = KW == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  Smem<QT, S> &sm = reinterpret_cast<Smem<QT, S> *>(smem_raw)[kg];
  // One group needs no mask, but the compiler allots registers and orders the loop
  // by whether there is one.  us with / without: Q6_K 5120 x 27648 at M = 48
  // 539 / 515, Q4_K 27648 x 5120 at M = 512 327 / 313, Q8_0 5120 x 5120 at
  // M = 512 82.8 / 81.3; Q6_K on large tiles (fewer spills) 151936 x 2048 at
  // M = 70 344 / 390, Q4_K on small ones 49152 x 512 at M = 60 14.6 / 14.8.
  constexpr bool kMask = KW > 1 || (QT == kTypeQ6_K && S == 2) || (QT == kTypeQ4_K && S == 1);
  const int tid = kMask ? threadIdx.x & 255 : threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int bx = blockIdx.x;
  const int sg = (bx >= g.seg[0].end) + (bx >= g.seg[1].end);
  const uint8_t *W = g.seg[sg].W, *A = g.A;
  void *Y = g.seg[sg].Y;
  const void *bias = g.bias;
  const int M = g.M, N = g.seg[sg].N, K = g.K, mode = g.mode;
  const int nt = bx - (sg ? g.seg[sg - 1].end : 0);
  const int wm = wave & 1, wn = wave >> 1;  // wave position in the 2 x 2 grid
  const int m0 = blockIdx.y * kBM, n0 = nt * kBN;
  const int l32 = lane & 31, h = lane >> 5;
  const int nblk32 = K >> 5;
  const uint32_t a_row = static_cast<uint32_t>(nblk32) * kQ8_1Bytes;
  const uint32_t w_row = static_cast<uint32_t>(QT == kTypeQ8_0 ? nblk32 * kQ8_0Bytes
                                                               : (K >> 8) * F::kSb);
  const rsrc_t Wr = make_rsrc(W, w_row * static_cast<uint32_t>(N));
  const rsrc_t Ar = make_rsrc(A, a_row * static_cast<uint32_t>(M));

  f32x16 acc[S][S];
#pragma unroll
  for (int a = 0; a < S; ++a)
#pragma unroll
    for (int b = 0; b < S; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.0f;

  // Rows of this wave's A tiles and columns of its B tiles; first of the 4
  // consecutive result rows this lane holds per group of 4.
  int ar[S], bn[S], rbase[S];
#pragma unroll
  for (int j = 0; j < S; ++j) {
    ar[j] = wm * 32 * S + 32 * j + l32;
    bn[j] = wn * 32 * S + 32 * j + l32;
    rbase[j] = wm * 32 * S + 32 * j + 4 * h;
  }

  const int nsteps = K >> 8;
  Prefetch<QT, S> pf;
  // a group past the last super-block loads the last one again and adds
  // nothing (every wave meets every barrier)
  fetch<QT, S>(pf, Wr, Ar, w_row, a_row, m0, n0, M, N, min(kg, nsteps - 1), tid);
  for (int s0 = 0; s0 < nsteps; s0 += KW) {
    const int sblk = s0 + kg;
    __syncthreads();  // previous step's LDS reads are done
    commit<QT, S>(sm, pf, tid);
    __syncthreads();
    if (s0 + KW < nsteps)
      fetch<QT, S>(pf, Wr, Ar, w_row, a_row, m0, n0, M, N, min(sblk + KW, nsteps - 1), tid);
    if (KW > 1 && sblk >= nsteps) continue;

    if constexpr (QT == kTypeQ4_K) {
      float dsc[S][8];
#pragma unroll
      for (int t = 0; t < S; ++t) {
        const u32x4 hdr = *reinterpret_cast<const u32x4 *>(&sm.w[bn[t] * F::kPitch]);
        const float d = h2f(hdr.x & 0xFFFFu), dmin = h2f(hdr.x >> 16);
        const uint32_t S0 = hdr.y, S1 = hdr.z, S2 = hdr.w;
        const uint32_t sc_lo = S0 & 0x3F3F3F3Fu, m_lo = S1 & 0x3F3F3F3Fu;
        const uint32_t sc_hi = (S2 & 0x0F0F0F0Fu) | ((S0 >> 2) & 0x30303030u);
        const uint32_t m_hi = ((S2 >> 4) & 0x0F0F0F0Fu) | ((S1 >> 2) & 0x30303030u);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          dsc[t][j] = d * static_cast<float>((sc_lo >> (8 * j)) & 0xFFu);
          dsc[t][j + 4] = d * static_cast<float>((sc_hi >> (8 * j)) & 0xFFu);
        }
        // min term on the matrix cores, subtracted straight from the
        // accumulators: K = sub-blocks 2j + h, j = 0..3
        const uint64_t mm = static_cast<uint64_t>(m_lo) | (static_cast<uint64_t>(m_hi) << 32);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int blk = 2 * j + h;
          const float fm = -(dmin * static_cast<float>((mm >> (8 * blk)) & 0xFFu));
#pragma unroll
          for (int s = 0; s < S; ++s)
            acc[s][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(sm.sa[blk][ar[s]], fm, acc[s][t],
                                                             0, 0, 0);
        }
      }
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        // Sub-blocks 2p (low nibbles) and 2p+1 (high nibbles) share qs bytes.
        u32x4 q[S];
#pragma unroll
        for (int t = 0; t < S; ++t)
          q[t] = *reinterpret_cast<const u32x4 *>(&sm.w[bn[t] * F::kPitch + 16 + p * 32 + 16 * h]);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const int sb = 2 * p + half;
          const int sh = 4 * half;
          i32x4 bw[S], av[S];
#pragma unroll
          for (int t = 0; t < S; ++t)
            bw[t] = i32x4{static_cast<int>((q[t].x >> sh) & 0x0F0F0F0Fu),
                          static_cast<int>((q[t].y >> sh) & 0x0F0F0F0Fu),
                          static_cast<int>((q[t].z >> sh) & 0x0F0F0F0Fu),
                          static_cast<int>((q[t].w >> sh) & 0x0F0F0F0Fu)};
#pragma unroll
          for (int s = 0; s < S; ++s)
            av[s] = *reinterpret_cast<const i32x4 *>(&sm.a[ar[s] * kApitch + sb * 32 + 16 * h]);
#pragma unroll
          for (int s = 0; s < S; ++s) {
            f32x4 fa[4];
#pragma unroll
            for (int g = 0; g < 4; ++g)
              fa[g] = *reinterpret_cast<const f32x4 *>(&sm.da[sb][rbase[s] + 8 * g]);
#pragma unroll
            for (int t = 0; t < S; ++t) {
              const i32x16 c = mfma32(av[s], bw[t]);
              const float w = dsc[t][sb];
#pragma unroll
              for (int i = 0; i < 16; ++i)
                acc[s][t][i] += static_cast<float>(c[i]) * (fa[i >> 2][i & 3] * w);
            }
          }
        }
      }
    } else if constexpr (QT == kTypeQ6_K) {
      float dq[S];
      uint32_t scw[S][4];
#pragma unroll
      for (int t = 0; t < S; ++t) {
        const uint8_t *row = &sm.w[bn[t] * F::kPitch];
        dq[t] = h2f(*reinterpret_cast<const uint16_t *>(row + 208));
        const u32x4 s4 = *reinterpret_cast<const u32x4 *>(row + 192);
        scw[t][0] = s4.x; scw[t][1] = s4.y; scw[t][2] = s4.z; scw[t][3] = s4.w;
      }
#pragma unroll
      for (int g = 0; g < 2; ++g) {
#pragma unroll
        for (int sub = 0; sub < 4; ++sub) {
          const int sb = g * 4 + sub;  // Q8_1 block within the super-block
          // 16-value group u (0/1): values 16u..16u+15 of this 32-run; this
          // lane supplies values 16u + 8h .. 16u + 8h + 7.
          int64_t bq[S][2];
          int sc0[S], sc1[S];
#pragma unroll
          for (int t = 0; t < S; ++t) {
            const uint8_t *row = &sm.w[bn[t] * F::kPitch];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              const int e = 16 * u + 8 * h;
              const u32x2 ql = *reinterpret_cast<const u32x2 *>(row + g * 64 + (sub & 1) * 32 + e);
              const u32x2 qh = *reinterpret_cast<const u32x2 *>(row + 128 + g * 32 + e);
              const int lsh = (sub >= 2) ? 4 : 0, hsh = 2 * sub;
              const uint32_t v0 = ((ql.x >> lsh) & 0x0F0F0F0Fu) | (((qh.x >> hsh) & 0x03030303u) << 4);
              const uint32_t v1 = ((ql.y >> lsh) & 0x0F0F0F0Fu) | (((qh.y >> hsh) & 0x03030303u) << 4);
              bq[t][u] = static_cast<int64_t>(q6_minus32(v0)) |
                         (static_cast<int64_t>(q6_minus32(v1)) << 32);
            }
            // scales[g*8 + 2*sub + u]
            const uint32_t sw = scw[t][2 * g + (sub >> 1)] >> (16 * (sub & 1));
            sc0[t] = static_cast<int8_t>(sw & 0xFFu);
            sc1[t] = static_cast<int8_t>((sw >> 8) & 0xFFu);
          }
#pragma unroll
          for (int s = 0; s < S; ++s) {
            int64_t aq[2];
#pragma unroll
            for (int u = 0; u < 2; ++u)
              aq[u] = *reinterpret_cast<const int64_t *>(&sm.a[ar[s] * kApitch + sb * 32 + 16 * u + 8 * h]);
            f32x4 fa[4];
#pragma unroll
            for (int gg = 0; gg < 4; ++gg)
              fa[gg] = *reinterpret_cast<const f32x4 *>(&sm.da[sb][rbase[s] + 8 * gg]);
#pragma unroll
            for (int t = 0; t < S; ++t) {
              const i32x16 c0 = mfma16(aq[0], bq[t][0]);
              const i32x16 c1 = mfma16(aq[1], bq[t][1]);
              const float dd = dq[t];
#pragma unroll
              for (int i = 0; i < 16; ++i) {
                const int ci = __mul24(c0[i], sc0[t]) + __mul24(c1[i], sc1[t]);
                acc[s][t][i] += static_cast<float>(ci) * (fa[i >> 2][i & 3] * dd);
              }
            }
          }
        }
      }
    } else {
#pragma unroll
      for (int b = 0; b < 8; ++b) {
        i32x4 bw[S];
        float dwv[S];
#pragma unroll
        for (int t = 0; t < S; ++t) {
          bw[t] = *reinterpret_cast<const i32x4 *>(&sm.w[bn[t] * F::kPitch + b * 32 + 16 * h]);
          dwv[t] = sm.dw[b][bn[t]];
        }
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const i32x4 av = *reinterpret_cast<const i32x4 *>(&sm.a[ar[s] * kApitch + b * 32 + 16 * h]);
          f32x4 fa[4];
#pragma unroll
          for (int gg = 0; gg < 4; ++gg)
            fa[gg] = *reinterpret_cast<const f32x4 *>(&sm.da[b][rbase[s] + 8 * gg]);
#pragma unroll
          for (int t = 0; t < S; ++t) {
            const i32x16 c = mfma32(av, bw[t]);
#pragma unroll
            for (int i = 0; i < 16; ++i)
              acc[s][t][i] += static_cast<float>(c[i]) * (fa[i >> 2][i & 3] * dwv[t]);
          }
        }
      }
    }
  }

  // The groups' sums meet in LDS; group g then owns 16 / KW of each tile's
  // values.
  constexpr int kOwn = 16 / KW;
  if constexpr (KW > 1) {
    float *part = reinterpret_cast<float *>(smem_raw);  // [group][t, s, i][thread]
    constexpr int kVals = S * S * 16;
    static_assert(kVals * 256 * 4 <= sizeof(Smem<QT, S>), "the sums reuse the stages");
    __syncthreads();
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < S; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          part[(kg * kVals + (s * S + t) * 16 + i) * 256 + tid] = acc[s][t][i];
    __syncthreads();
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < S; ++t)
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
          const int v = (s * S + t) * 16 + kg * kOwn + i;
          float sum = part[v * 256 + tid];
#pragma unroll
          for (int k = 1; k < KW; ++k) sum += part[(k * kVals + v) * 256 + tid];
          acc[s][t][i] = sum;
        }
  }

  // Epilogue: lane holds column n and rows rbase + 8g + j.
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int t = 0; t < S; ++t) {
      const int n = n0 + wn * 32 * S + 32 * t + l32;
      if (n >= N) continue;
#pragma unroll
      for (int i = 0; i < kOwn; ++i) {
        const int v = kg * kOwn + i;
        const int m = m0 + wm * 32 * S + 32 * s + 8 * (v >> 2) + 4 * h + (v & 3);
        if (m >= M) continue;
        const int64_t o = static_cast<int64_t>(m) * N + n;
        float y = acc[s][t][i];
        if constexpr (F16OUT) {
          uint16_t *Yh = static_cast<uint16_t *>(Y);
          if (mode == 1) y += h2f(Yh[o]);
          else if (mode == 2) y += h2f(static_cast<const uint16_t *>(bias)[n]);
          Yh[o] = static_cast<uint16_t>(f2h_bits(y));
        } else {
          float *Yf = static_cast<float *>(Y);
          if (mode == 1) y += Yf[o];
          else if (mode == 2) y += static_cast<const float *>(bias)[n];
          Yf[o] = y;
        }
      }
    }
}

template <int QT, int S, bool F16OUT, int KW>
static hipError_t launch_k(const MfmaArgs &g, dim3 grid, hipStream_t s) {
  const size_t shm = KW * sizeof(Smem<QT, S>);
  if (!note_launch("k_gemm_mfma", {QT, S, F16OUT}, {KW})) return hipSuccess;
  // The staged tiles can exceed the 64 KiB default; gfx950 has 160 KiB of LDS.
  // set once per kernel (function-local static: thread-safe)
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void *>(&k_gemm_mfma<QT, S, F16OUT, KW>),
      hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(shm));
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL((k_gemm_mfma<QT, S, F16OUT, KW>), grid, dim3(256 * KW), shm, s, g);
  return last_error();
}

template <int QT, int S, int KW>
static hipError_t launch_s(MfmaArgs &g, int count, bool f16, hipStream_t s) {
  constexpr int kB = 64 * S;
  int end = 0;
  for (int i = 0; i < kMaxSeg; ++i) {
    if (i < count) end += (g.seg[i].N + kB - 1) / kB;
    g.seg[i].end = end;
  }
  const dim3 grid(end, (g.M + kB - 1) / kB);
  return f16 ? launch_k<QT, S, true, KW>(g, grid, s) : launch_k<QT, S, false, KW>(g, grid, s);
}

// 128 x 128 workgroup tiles when they give at least two workgroups per CU
// and the batch fills more than half of their rows (LM head 151936 x 2048 at
// M = 60, large / small tiles: Q4_K 167 / 99 us, Q8_0 177 / 115), else 64 x 64
// (e.g. N = 5120 at M = 512: 160 large tiles, 640 small).  With no more small
// tiles than CUs, four groups of waves share each; up to two tiles a CU, two
// groups.  us for 1 / 2 / 4 groups:
//   Q4_K 11008 x 2048 at M = 60 (172 tiles)      20.9 / 17.0 / 16.1
//   Q4_K 13824 x 5120 at M = 64 (216)            45.3 / 35.5 / 32.6
//   Q4_K 22016 x 2048 at M = 60 (344)            27.3 / 26.3 / 30.4
//   Q4_K 27648 x 5120 at M = 64 (432)            60.3 / 54.1 / 60.2
//   Q8_0 2048 x 11008 at M = 60 (32)             93.5 / 81.4 / 74.9
//   Q8_0 11008 x 2048 at M = 60 (172)            20.5 /      / 18.8
//   Q8_0 22016 x 2048 at M = 64 (344)            27.6 / 29.6 / 33.7
//   Q8_0 27648 x 5120 at M = 64 (432)            63.9 / 69.5
//   Q8_0 20480 x 8192 at M = 60 (320)            88.7 / 100
//   Q8_0 13824 x 5120 at M = 127 (432)           61.2 / 57.3 / 65.9
// so Q8_0 (less unpacking to hide the loads behind) takes two groups only
// from K = 4096 on and where two tiles share their weights (M > 64).  Groups
// need super-blocks enough: at K = 256 four took Q4_K 2048 x 256 from 5.0 to 6.5
// and Q8_0 from 4.7 to 7.9, at K = 512 Q8_0 16384 x 512 from 8.1 to 9.5 (Q4_K 8.3, 8.5;
// 2048 x 512 7.0, 6.9), at K = 1024 Q8_0 2048 x 1024 11.1 to 9.5; two at K = 768
// Q4_K 24576 x 768 from 13.0 to 14.7.  Q6_K runs here on request only and keeps one
// group.
template <int QT>
static hipError_t launch_qt(MfmaArgs &g, int count, bool f16, hipStream_t s) {
  int64_t big = 0, small = 0;
  for (int i = 0; i < count; ++i) {
    big += static_cast<int64_t>((g.seg[i].N + 127) / 128) * ((g.M + 127) / 128);
    small += static_cast<int64_t>((g.seg[i].N + 63) / 64) * ((g.M + 63) / 64);
  }
  if (big >= 512 && g.M > 64) return launch_s<QT, 2, 1>(g, count, f16, s);
  if constexpr (QT != kTypeQ6_K) {
    constexpr bool q8 = QT == kTypeQ8_0;
    if (small <= 256 && g.K >= (q8 ? 1024 : 512)) return launch_s<QT, 1, 4>(g, count, f16, s);
    if (small > 256 && small <= 512 && g.K >= (q8 ? 4096 : 1024) && (!q8 || g.M > 64))
      return launch_s<QT, 1, 2>(g, count, f16, s);
  }
  return launch_s<QT, 1, 1>(g, count, f16, s);
}

hipError_t launch_gemv(int qtype, const void *W, const void *A, void *Y, const void *bias,
                       bool f16, int M, int N, int K, int mode, hipStream_t stream);

// K % 256 == 0 is required for the super-block K loop; Q8_0 weights with
// K % 256 != 0 run on the GEMV kernel in groups of 8 columns instead.
hipError_t launch_gemm_mfma_grouped(int qtype, int count, const void *const *W, const void *A,
                                    void *const *Y, const int *N, const void *bias, bool f16,
                                    int M, int K, int mode, hipStream_t stream) {
  if (K % 256 != 0) {
    for (int i = 0; i < count; ++i) {
      const hipError_t e = launch_gemv(qtype, W[i], A, Y[i], bias, f16, M, N[i], K, mode, stream);
      if (e != hipSuccess) return e;
    }
    return hipSuccess;
  }
  MfmaArgs g{};
  for (int i = 0; i < kMaxSeg; ++i) {
    const int k = i < count ? i : count - 1;
    g.seg[i] = {static_cast<const uint8_t *>(W[k]), Y[k], N[k], 0};
  }
  g.A = static_cast<const uint8_t *>(A);
  g.bias = bias;
  g.M = M;
  g.K = K;
  g.mode = mode;
  switch (qtype) {
  case kTypeQ4_K: return launch_qt<kTypeQ4_K>(g, count, f16, stream);
  case kTypeQ6_K: return launch_qt<kTypeQ6_K>(g, count, f16, stream);
  case kTypeQ8_0: return launch_qt<kTypeQ8_0>(g, count, f16, stream);
  default: return hipErrorInvalidValue;
  }
}

hipError_t launch_gemm_mfma(int qtype, const void *W, const void *A, void *Y, const void *bias,
                            bool f16, int M, int N, int K, int mode, hipStream_t stream) {
  return launch_gemm_mfma_grouped(qtype, 1, &W, A, &Y, &N, bias, f16, M, K, mode, stream);
}

}  // namespace ifx
