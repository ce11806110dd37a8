// gemm_f16.h -- the prefill GEMM kernel on the fp16 matrix cores of gfx950,
// with the weights dequantized inside the kernel: y[m][n] = sum_k W[n][k] *
// x[m][k], W raw GGUF Q4_K / Q6_K / Q8_0 blocks, x given as Q8_1 blocks of 32,
// fp32 accumulate.  One translation unit per quant type instantiates it
// (gemm_f16_q4.hip, _q6.hip, _q8.hip); gemm_f16.hip plans the launches.
//
// This is the arithmetic of the reference's prefill path, fused: above its
// MMQ limit the reference dequantizes W to an FP16 scratch copy
// (runtime/backends/cuda/native/quantized_weight_map.cpp:176-233, element
// formulas kernels/quant_common.cuh:100-188) and multiplies it with cuBLAS
// in FP16 with fp32 accumulation (cublas_gemm.h:47, called at
// transformer_forward.cu:1479).  Here the FP16 copy never exists.  Per
// element, w = fp16(d*sc) * q - fp16(dmin*m) (Q4_K), fp16(d*sc) * (q - 32)
// (Q6_K), fp16(d) * q (Q8_0), each one fp16 fused multiply-add or multiply;
// x = fp16(d_a) * q_a.  The rounding of w and x to fp16 (relative 2^-11) is
// the reference's own FP16 prefill rounding; the integer-exact int8 kernel
// (gemm_mfma.hip) remains for mid-size batches.
//
// Why not int8: the per-32-value rescale of int8 MFMA results costs three
// VALU operations per output per block and bounds that kernel near 15 % of
// the int8 peak.  Dequantizing to fp16 costs about two VALU operations per
// weight element instead, once for all the batch rows of a tile (128 or 256 at most).
//
// How a workgroup works.  Its waves tile the output along n (each owns NT x 32
// weight rows and all 32 MT batch rows of the tile) and, for small tiles, K:
//   * Activations are converted to fp16 once per workgroup into a
//     double-buffered LDS stage that all its waves read.
//   * Weights go through LDS raw, into an area of the wave that owns the rows,
//     and each lane dequantizes just what it feeds to its MFMAs: no fp16
//     weights in LDS, no weight is converted twice in a workgroup, and no
//     barrier guards them.  With the 256 x 256 tile this replaces (weights
//     stored to LDS as fp16 and read back by four waves each) a K step of 64
//     values moved 256 KB through LDS a workgroup; 128 x 512 moves 180.
//   * Packed fp16 dequant: four code bytes become two fp16 pairs with a mask
//     or byte permute each, (0x6400 | b) = 1024 + b, then v_pk_add / v_pk_fma.
//     The pairs hold values (0, 2) and (1, 3) of each group of four; both
//     operands are stored in that order, so the K permutation cancels in the
//     dot product.
//   * The operands of the next MFMA slot are made while one runs, so that the
//     conversion's VALU work (about 170 instructions a wave and 64 values,
//     against 32 MFMAs) issues between MFMAs.
// MFMA lane layouts (32x32x16 f16): lane l supplies row (l % 32) of A and
// column (l % 32) of B, with 8 K values for K half l / 32; it receives
// column l % 32 and rows 8*(i/4) + 4*(l/32) + (i%4), i = 0..15.
#pragma once

#include "../../include/ifx_qgemm.h"
#include "ifx_common.h"

#include <type_traits>

namespace ifx {

// A launch of 1..3 projections that read the same activations.
constexpr int kMaxSeg = 3;
struct F16Seg {
  const uint8_t *W;
  void *Y;
  int N;
  int tile_end;  // weight tiles of this and the segments before it
};
enum F16Epi { kEpiF32 = 0, kEpiF16 = 1, kEpiAtomic = 2, kEpiSlot = 3 };
struct F16Args {
  F16Seg seg[kMaxSeg];
  const uint8_t *A;
  const void *bias;
  int M, K, mode, epi, m_tiles, splits, spw;  // spw: groups per split
  int vec;  // every output row starts on 16 bytes
};

namespace {

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));

constexpr int kBK = 64;      // K values per chunk
constexpr int kPitch = kBK;  // halves per staged activation row
// A staged row is its 64 K values as eight 16-byte groups, unpadded; group
// g of row r sits at position g ^ swz(r).  The swizzle makes both access
// patterns conflict-free on 64 banks (16 lanes per b128 phase) and on 32
// banks (8 lanes): the MFMA operand reads (lanes 0-31 and 32-63 read one
// group each of rows l % 32) and the stage writes (threads 2r, 2r + 1: the
// groups 4 p + j of row r).
__device__ __forceinline__ int swz(int r) {
  // (r & 1) ^ g[(r >> 1) & 7] with g = {0, 6, 3, 5, 1, 7, 2, 4}
  return (r & 1) ^ ((0x8B9AF0 >> (3 * ((r >> 1) & 7))) & 7);
}
// Halves offset of group g of row r in a staged chunk.
__device__ __forceinline__ int slot(int r, int g) { return r * kPitch + 8 * (g ^ swz(r)); }

constexpr uint32_t kMagic = 0x64006400u;  // fp16 1024.0 in both halves

__device__ __forceinline__ h2 as_h2(uint32_t u) { return __builtin_bit_cast(h2, u); }
__device__ __forceinline__ uint32_t as_u32(h2 h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ h2 splat(float f) {
  const _Float16 h = static_cast<_Float16>(f);
  return h2{h, h};
}

// Signed byte codes (four per word) times scale d -> two fp16 pairs holding
// values (0, 2) and (1, 3).  q ^ 0x80 = q + 128 as an unsigned byte, so
// (0x6400 | byte) - 1152 = q exactly; the product is rounded once.
__device__ __forceinline__ void i8x4_to_h(uint32_t x, h2 d, uint32_t &p02, uint32_t &p13) {
  const uint32_t mg = vreg(kMagic);
  x ^= 0x80808080u;
  const h2 off = {static_cast<_Float16>(-1152.0f), static_cast<_Float16>(-1152.0f)};
  // byte permutes place two code bytes under the magic's high bytes
  const h2 a = as_h2(__builtin_amdgcn_perm(mg, x, 0x05020500u)) + off;
  const h2 b = as_h2(__builtin_amdgcn_perm(mg, x, 0x05030501u)) + off;
  p02 = as_u32(a * d);
  p13 = as_u32(b * d);
}

// Unsigned byte codes v (< 1024) -> fp16 pairs of (v + bias) * d.
__device__ __forceinline__ void u8x4_to_h(uint32_t x, h2 bias, h2 d, uint32_t &p02,
                                          uint32_t &p13) {
  const uint32_t mg = vreg(kMagic);
  const h2 a = as_h2(__builtin_amdgcn_perm(mg, x, 0x05020500u)) + bias;
  const h2 b = as_h2(__builtin_amdgcn_perm(mg, x, 0x05030501u)) + bias;
  p02 = as_u32(a * d);
  p13 = as_u32(b * d);
}

// Nibble codes of a word of packed 4-bit codes (HI = 0: low, 1: high
// nibbles) -> fp16 pairs q * d - mn of bytes (0, 2) and (1, 3).  Low
// nibbles sit in mantissa bits 0..3 under the magic 1024 (ulp 1): 1024 + q;
// high nibbles stay in bits 4..7, under the magic 64 (0x5400, ulp 1/16)
// also exactly 64 + q, so neither needs more than the one shift by 8.
template <int HI>
__device__ __forceinline__ void q4x4_to_h(uint32_t x, h2 d, h2 mn, uint32_t &p02, uint32_t &p13) {
  constexpr uint32_t msk = HI ? 0x00F000F0u : 0x000F000Fu;
  const uint32_t mg = vreg(HI ? 0x54005400u : kMagic);
  const h2 bias = splat(HI ? -64.0f : -1024.0f);
  const h2 a = as_h2((x & msk) | mg) + bias;
  const h2 b = as_h2(((x >> 8) & msk) | mg) + bias;
  p02 = as_u32(__builtin_elementwise_fma(a, d, -mn));
  p13 = as_u32(__builtin_elementwise_fma(b, d, -mn));
}

// The 32 activation values of one Q8_1 block as fp16, in the order the GEMM
// stores them: word 2j / 2j+1 holds values (4j, 4j+2) / (4j+1, 4j+3).
__device__ __forceinline__ void q8_1_block_to_h(uint32_t ads, u32x4 a0, u32x4 a1, uint32_t (&o)[16]) {
  const h2 d = splat(h2f(ads & 0xFFFFu));
  const uint32_t in[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
  for (int j = 0; j < 8; ++j) i8x4_to_h(in[j], d, o[2 * j], o[2 * j + 1]);
}

// Q8_1 blocks of chunk c (64 values): first and second 32-value half.
// Q4_K: sub-blocks 2p, 2p+1 of super-block c/4 (they share qs bytes).
// Q6_K: sub-blocks hf and hf + 2 of 128-value half g (they share ql/qh
// bytes), c = 4*sb + 2*g + hf.  Q8_0: blocks 2c, 2c+1.
template <int QT>
__device__ __forceinline__ int chunk_block(int c, int half) {
  if constexpr (QT == kTypeQ6_K) {
    const int sb = c >> 2, g = (c >> 1) & 1, hf = c & 1;
    return sb * 8 + g * 4 + hf + 2 * half;
  } else {
    return 2 * c + half;
  }
}

// Raw activation bytes of one staged item: (row, block half) of a chunk.
template <bool AH>
struct RawA {
  u32x4 a[AH ? 4 : 2];  // Q8_1 codes; AH: the block's 64 fp16 bytes
  uint32_t ds;          // Q8_1 {d, s}
};

template <int QT, bool AH>
__device__ __forceinline__ void fetch_a(RawA<AH> &r, rsrc_t Ar, uint32_t a_off, int c, int part) {
  if constexpr (AH) {  // already converted: 32 fp16 values in commit_a's order
    const uint32_t o = a_off + chunk_block<QT>(c, part) * 64;
#pragma unroll
    for (int j = 0; j < 4; ++j) r.a[j] = bload<u32x4>(Ar, o + 16 * j, 0);
  } else {
    const uint32_t o = a_off + chunk_block<QT>(c, part) * kQ8_1Bytes;
    r.ds = bload<uint32_t>(Ar, o, 0);
    r.a[0] = bload<u32x4>(Ar, o + 4, 0);
    r.a[1] = bload<u32x4>(Ar, o + 20, 0);
  }
}

// Converts one item and stores its four 16-byte groups.
template <bool AH>
__device__ __forceinline__ void commit_a(_Float16 *chunk, const RawA<AH> &r, int row, int part) {
  if constexpr (AH) {
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<u32x4 *>(chunk + slot(row, 4 * part + j)) = r.a[j];
  } else {
    uint32_t o[16];
    q8_1_block_to_h(r.ds, r.a[0], r.a[1], o);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<u32x4 *>(chunk + slot(row, 4 * part + j)) =
          u32x4{o[4 * j], o[4 * j + 1], o[4 * j + 2], o[4 * j + 3]};
  }
}

// Weights pass through LDS as they are (raw), so that global loads run along
// the rows: one lane's 16 bytes come from a row of its own, and gathering 64
// rows that way costs the vector cache an access a lane and the L2 a request
// for every 32 bytes of a line.  Each wave stages the rows of its own MFMA
// tiles, one or two chunks (a unit) at a time; no other wave reads them, so no barrier
// guards them.  A staged row holds its codes in 16-byte pieces, one or two for
// each K half h, then its fp16 scales.  A piece is 8 bytes from 8 h on and 8
// from 16 + 8 h on, so that slot sl of a chunk multiplies its values 16 sl ..
// + 15: the sum of an output runs over K in order, 16 values at a time, on
// every tile whose waves do not split K.
//   Q4_K  piece 2 ch + h: qs of chunk ch (both nibbles); 8 bytes a chunk:
//         (d sc0, d sc1), (dmin m0, dmin m1)
//   Q6_K  pieces 2 ch + h: ql; 4 + h: qh; 8 bytes a chunk: (d sc0, d sc1) of
//         its values 0 .. 15 of each sub-block, then of 16 .. 31
//   Q8_0  (one chunk) pieces 2 h + b: the codes of block 2 c + b; 4 bytes a
//         block: (d, d)
template <int QT>
struct WRow {
  static constexpr int kUnit = QT == kTypeQ8_0 ? 1 : 2;  // chunks
  static constexpr int kPieces = QT == kTypeQ6_K ? 6 : 4;
  static constexpr int kScale = 16 * kPieces;  // byte offset of the scales
  static constexpr int kUsed = kScale + 8 * kUnit;
  // an odd number of 16-byte units: lanes of consecutive rows read distinct banks
  static constexpr int kPitch = ((kUsed + 15) / 16 | 1) * 16;
};

// A lane's share of one unit of its wave's R = 32 NT rows.
template <int QT, int NT>
struct RawW {
  static constexpr int kR = 32 * NT;
  static constexpr int kCodes = kR * WRow<QT>::kPieces / 64;  // 16-byte pieces a lane
  static constexpr int kHeads = (kR + 63) / 64;               // rows a lane (scales)
  u32x4 q[kCodes];
  // Q4_K: header of row lane; Q6_K: scales (8 bytes) and d of row lane; Q8_0:
  // the dword after q
  u32x4 hd[QT == kTypeQ8_0 ? 1 : kHeads];
  uint32_t d[QT == kTypeQ8_0 ? kCodes / 2 : kHeads];
};

// Unit `un` of row n0 + r for rows r < 32 NT (rows past N repeat the last).
template <int QT, int NT>
__device__ __forceinline__ void fetch_w(RawW<QT, NT> &w, rsrc_t Wr, int n0, int N, uint32_t w_row,
                                        int un, int lane) {
  using R = RawW<QT, NT>;
  if constexpr (QT == kTypeQ4_K) {
    const uint32_t o = (un >> 1) * kQ4KBytes;
#pragma unroll
    for (int i = 0; i < R::kCodes; ++i) {  // 4 lanes a row: the half's 64 qs bytes
      const int r = 16 * i + (lane >> 2);
      w.q[i] = wload<u32x4>(Wr, min(n0 + r, N - 1) * w_row + 16 * (lane & 3), o + 16 + 64 * (un & 1));
    }
#pragma unroll
    for (int i = 0; i < R::kHeads; ++i)
      w.hd[i] = wload<u32x4>(Wr, min(n0 + 64 * i + lane % R::kR, N - 1) * w_row, o);
  } else if constexpr (QT == kTypeQ6_K) {
    const int g = un & 1;
    const uint32_t o = (un >> 1) * kQ6KBytes;
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) {  // 4 lanes a row: the half's 64 ql bytes
      const int r = 16 * i + (lane >> 2);
      w.q[i] = wload<u32x4>(Wr, min(n0 + r, N - 1) * w_row + 16 * (lane & 3), o + 64 * g);
    }
#pragma unroll
    for (int i = 0; i < NT; ++i) {  // 2 lanes a row: its 32 qh bytes
      const int r = 32 * i + (lane >> 1);
      w.q[2 * NT + i] = wload<u32x4>(Wr, min(n0 + r, N - 1) * w_row + 16 * (lane & 1), o + 128 + 32 * g);
    }
#pragma unroll
    for (int i = 0; i < R::kHeads; ++i) {
      const uint32_t ro = min(n0 + 64 * i + lane % R::kR, N - 1) * w_row;
      const u32x2 sc = wload<u32x2>(Wr, ro, o + 192 + 8 * g);
      w.hd[i] = u32x4{sc.x, sc.y, 0, 0};
      w.d[i] = wload<uint16_t>(Wr, ro, o + 208);
    }
  } else {
#pragma unroll
    for (int i = 0; i < R::kCodes / 2; ++i) {  // 2 lanes a row: its two blocks
      const int r = 32 * i + (lane >> 1);
      const uint32_t ro = min(n0 + r, N - 1) * w_row + (lane & 1) * kQ8_0Bytes;
      // the codes start 2 bytes into the block: read whole dwords from there
      // down (a 2-byte aligned 16-byte load costs about twice)
      const uint32_t co = (ro + 2) & ~3u;
      w.q[2 * i] = wload<u32x4>(Wr, co, un * 2 * kQ8_0Bytes);
      w.q[2 * i + 1] = wload<u32x4>(Wr, co + 16, un * 2 * kQ8_0Bytes);
      w.d[i] = wload<uint32_t>(Wr, co + 32, un * 2 * kQ8_0Bytes);
    }
  }
}

// 16 bytes from a piece-aligned place p: the two K halves' 8 bytes of a piece
// each (8-byte stores: one instruction, no more bank cycles than a 16-byte one).
__device__ __forceinline__ void put_halves(uint8_t *p, u32x4 q) {
  *reinterpret_cast<u32x2 *>(p) = u32x2{q.x, q.y};
  *reinterpret_cast<u32x2 *>(p + 16) = u32x2{q.z, q.w};
}

// Scales: small integers become fp16 exactly under the magic 1024 (sc ^ 0x80
// for Q6_K's signed ones), so each product is rounded once, as d * sc in
// fp32 rounded to fp16 would be.
template <int QT, int NT>
__device__ __forceinline__ void commit_w(uint8_t *rows, const RawW<QT, NT> &w, int un, int lane) {
  using R = RawW<QT, NT>;
  using L = WRow<QT>;
  const uint32_t mg = vreg(kMagic);
  if constexpr (QT == kTypeQ4_K) {
#pragma unroll
    for (int i = 0; i < R::kCodes; ++i)
      put_halves(rows + (16 * i + (lane >> 2)) * L::kPitch + 32 * ((lane >> 1) & 1) + 8 * (lane & 1), w.q[i]);
#pragma unroll
    for (int i = 0; i < R::kHeads; ++i) {
      // get_scale_min_k4 (quant_common.cuh:83-94): sub-blocks 0..3 (un even)
      // or 4..7 of the super-block
      const h2 dd = as_h2(w.hd[i].x);
      const h2 d = __builtin_shufflevector(dd, dd, 0, 0), n = __builtin_shufflevector(dd, dd, 1, 1);
      const h2 off = splat(-1024.0f);
      const uint32_t S0 = w.hd[i].y, S1 = w.hd[i].z, S2 = w.hd[i].w;
      // branch-free on the wave-uniform half: mask m all ones for the upper one
      const uint32_t m = 0u - static_cast<uint32_t>(un & 1);
      const uint32_t sc = (S0 & 0x3F3F3F3Fu & ~m) | (((S2 & 0x0F0F0F0Fu) | ((S0 >> 2) & 0x30303030u)) & m);
      const uint32_t mn = (S1 & 0x3F3F3F3Fu & ~m) | ((((S2 >> 4) & 0x0F0F0F0Fu) | ((S1 >> 2) & 0x30303030u)) & m);
      u32x4 o;
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const uint32_t sel = p ? 0x05030502u : 0x05010500u;
        o[2 * p] = as_u32((as_h2(__builtin_amdgcn_perm(mg, sc, sel)) + off) * d);
        o[2 * p + 1] = as_u32((as_h2(__builtin_amdgcn_perm(mg, mn, sel)) + off) * n);
      }
      if (R::kR % 64 == 0 || lane < R::kR)
        *reinterpret_cast<u32x4 *>(rows + (64 * i + lane) * L::kPitch + L::kScale) = o;
    }
  } else if constexpr (QT == kTypeQ6_K) {
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i)
      put_halves(rows + (16 * i + (lane >> 2)) * L::kPitch + 32 * ((lane >> 1) & 1) + 8 * (lane & 1), w.q[i]);
#pragma unroll
    for (int i = 0; i < NT; ++i)
      put_halves(rows + (32 * i + (lane >> 1)) * L::kPitch + 64 + 8 * (lane & 1), w.q[2 * NT + i]);
#pragma unroll
    for (int i = 0; i < R::kHeads; ++i) {
      const h2 d = splat(h2f(w.d[i]));
      u32x4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) {  // chunk hf = k >> 1, values 16 p .. with p = k & 1: bytes 2 hf + p of both words
        const uint32_t b = ((w.hd[i].x >> (8 * k)) & 0xFFu) | (((w.hd[i].y >> (8 * k)) & 0xFFu) << 16);
        o[k] = as_u32((as_h2((b ^ 0x00800080u) | mg) + splat(-1152.0f)) * d);
      }
      if (R::kR % 64 == 0 || lane < R::kR)
        *reinterpret_cast<u32x4 *>(rows + (64 * i + lane) * L::kPitch + L::kScale) = o;
    }
  } else {
#pragma unroll
    for (int i = 0; i < R::kCodes / 2; ++i) {
      uint8_t *t = rows + (32 * i + (lane >> 1)) * L::kPitch;
      // even blocks of a row begin on a dword: their codes are 2 bytes in
      const uint32_t sh = lane & 1 ? 0 : 16;
      const u32x4 a = w.q[2 * i], b = w.q[2 * i + 1];
      auto cat = [&](uint32_t hi, uint32_t lo) { return __builtin_amdgcn_alignbit(hi, lo, sh); };
      *reinterpret_cast<u32x4 *>(t + 16 * (lane & 1)) =
          u32x4{cat(a.y, a.x), cat(a.z, a.y), cat(b.y, b.x), cat(b.z, b.y)};
      *reinterpret_cast<u32x4 *>(t + 32 + 16 * (lane & 1)) =
          u32x4{cat(a.w, a.z), cat(b.x, a.w), cat(b.w, b.z), cat(w.d[i], b.w)};
      // d: the low half of the even block's first dword; the odd block's
      // follows the even one's codes (the high half of the lane before's last)
      const uint32_t before = dpp<0xA0>(0u, w.d[i]);  // quad_perm [0,0,2,2], in all lanes
      const uint32_t d = lane & 1 ? before >> 16 : a.x & 0xFFFFu;
      *reinterpret_cast<uint32_t *>(t + L::kScale + 4 * (lane & 1)) = d | (d << 16);
    }
  }
}

// One lane's staged weights of a chunk: the 32 values that its K half h =
// lane / 32 supplies to the chunk's four MFMAs, and their scales (d; n: Q4_K's
// minima, Q6_K's scales of values 16 .. 31, Q8_0's second block).
template <int QT>
struct LaneW {
  u32x4 q, x;
  h2 d, n;
};
template <int QT>
__device__ __forceinline__ LaneW<QT> read_w(const uint8_t *row, int ch, int h) {
  using L = WRow<QT>;
  LaneW<QT> w;
  if constexpr (QT == kTypeQ4_K) {
    w.q = *reinterpret_cast<const u32x4 *>(row + 16 * (2 * ch + h));
    const u32x2 s = *reinterpret_cast<const u32x2 *>(row + L::kScale + 8 * ch);
    w.d = as_h2(s.x);
    w.n = as_h2(s.y);
  } else if constexpr (QT == kTypeQ6_K) {
    w.q = *reinterpret_cast<const u32x4 *>(row + 16 * (2 * ch + h));
    const u32x4 x = *reinterpret_cast<const u32x4 *>(row + 64 + 16 * h);
    w.x = u32x4{x.x >> (2 * ch), x.y >> (2 * ch), x.z >> (2 * ch), x.w >> (2 * ch)};
    const u32x2 s = *reinterpret_cast<const u32x2 *>(row + L::kScale + 8 * ch);
    w.d = as_h2(s.x);
    w.n = as_h2(s.y);
  } else {
    w.q = *reinterpret_cast<const u32x4 *>(row + 32 * h);
    w.x = *reinterpret_cast<const u32x4 *>(row + 32 * h + 16);
    const u32x2 s = *reinterpret_cast<const u32x2 *>(row + L::kScale);
    w.d = as_h2(s.x);
    w.n = as_h2(s.y);
  }
  return w;
}

// The lane's eight fp16 weights of MFMA slot sl (0..3) of the chunk.
template <int QT>
__device__ __forceinline__ h8 w_slot(const LaneW<QT> &w, int sl) {
  uint32_t o[4];
  const h2 ds = (QT == kTypeQ6_K && (sl & 1)) || (QT == kTypeQ8_0 && sl >= 2) ? w.n : w.d;
  const h2 d = sl < 2 || QT == kTypeQ8_0 ? __builtin_shufflevector(ds, ds, 0, 0)
                                         : __builtin_shufflevector(ds, ds, 1, 1);
  if constexpr (QT == kTypeQ4_K) {
    const h2 n = sl < 2 ? __builtin_shufflevector(w.n, w.n, 0, 0)
                        : __builtin_shufflevector(w.n, w.n, 1, 1);
    const uint32_t x0 = (sl & 1) ? w.q.z : w.q.x, x1 = (sl & 1) ? w.q.w : w.q.y;
    if (sl < 2) {
      q4x4_to_h<0>(x0, d, n, o[0], o[1]);
      q4x4_to_h<0>(x1, d, n, o[2], o[3]);
    } else {
      q4x4_to_h<1>(x0, d, n, o[0], o[1]);
      q4x4_to_h<1>(x1, d, n, o[2], o[3]);
    }
  } else if constexpr (QT == kTypeQ6_K) {
    // low nibbles of ql with qh bits 0, 1 (slots 0, 1), high nibbles with
    // bits 4, 5; dequant_q6k_element (quant_common.cuh:161-177)
    const h2 b = splat(-1056.0f);
    const uint32_t l[2] = {(sl & 1) ? w.q.z : w.q.x, (sl & 1) ? w.q.w : w.q.y};
    const uint32_t y[2] = {(sl & 1) ? w.x.z : w.x.x, (sl & 1) ? w.x.w : w.x.y};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t v = sl < 2 ? (l[i] & 0x0F0F0F0Fu) | ((y[i] << 4) & 0x30303030u)
                                : ((l[i] >> 4) & 0x0F0F0F0Fu) | (y[i] & 0x30303030u);
      u8x4_to_h(v, b, d, o[2 * i], o[2 * i + 1]);
    }
  } else {
    const u32x4 v = sl < 2 ? w.q : w.x;
    i8x4_to_h((sl & 1) ? v.z : v.x, d, o[0], o[1]);
    i8x4_to_h((sl & 1) ? v.w : v.y, d, o[2], o[3]);
  }
  return __builtin_bit_cast(h8, u32x4{o[0], o[1], o[2], o[3]});
}

// Activation group (8 values) that K half h supplies to slot sl: the
// values the weights of that half and slot belong to.
__device__ __forceinline__ int a_group(int sl, int h) { return 2 * sl + h; }

// C consecutive outputs (m, n ..) = v by the launch's epilogue, in 16-byte
// accesses: of launches whose row pitch allows them (g.vec; C divides N).
template <int C>
__device__ __forceinline__ void put(const F16Args &g, void *Y, int N, int split, int m, int n,
                                    f32x4 (&v)[C / 4]) {
  if (m >= g.M || n >= N) return;
  const int64_t o = static_cast<int64_t>(m) * N + n;
  if (g.epi == kEpiF16) {
    if constexpr (C == 8) {
      uint16_t *p = static_cast<uint16_t *>(Y) + o;
      const uint16_t *bias = static_cast<const uint16_t *>(g.bias);
      u32x4 t = {0, 0, 0, 0};
      if (g.mode == 1) t = *reinterpret_cast<const u32x4 *>(p);
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const uint32_t h = (t[k >> 1] >> (16 * (k & 1))) & 0xFFFFu;
        if (g.mode == 1) v[k >> 2][k & 3] += h2f(h);
        else if (g.mode == 2) v[k >> 2][k & 3] += h2f(bias[n + k]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        t[k] = f2h_bits(v[k >> 1][2 * (k & 1)]) | f2h_bits(v[k >> 1][2 * (k & 1) + 1]) << 16;
      *reinterpret_cast<u32x4 *>(p) = t;
    }
    return;
  }
  if constexpr (C == 4) {
    const bool slot = g.epi == kEpiSlot;
    float *p = static_cast<float *>(Y) + (slot ? static_cast<int64_t>(split) * g.M * N : 0) + o;
    const float *bias = static_cast<const float *>(g.bias);
    const int mode = slot ? 0 : g.mode;
    if (mode == 1) v[0] += *reinterpret_cast<const f32x4 *>(p);
    else if (mode == 2) v[0] += f32x4{bias[n], bias[n + 1], bias[n + 2], bias[n + 3]};
    *reinterpret_cast<f32x4 *>(p) = v[0];
  }
}

// Tile shapes.  MT x NT MFMA tiles of 32 x 32 per wave (m x n), WN x KW waves
// (n x units of a group); AU chunks per wave and activation stage.
template <int QT, int MT_, int NT_, int WN_, int KW_, int AU_>
struct Tile {
  static constexpr int MT = MT_, NT = NT_, WN = WN_, KW = KW_, AU = AU_;
  // a group: what every wave does between two returns to the loop's head
  static constexpr int US = WRow<QT>::kUnit, G = US > AU ? US : AU;  // chunks of a unit, of a group
  static constexpr int kSteps = G / AU, kUnits = G / US;             // stages, units of a group
  static constexpr int BM = 32 * MT, BN = 32 * NT * WN, KC = KW * AU;
  static constexpr int kThreads = 64 * WN * KW;
  // activation items of a stage: (row, chunk, half), a row's in consecutive threads
  static constexpr int kAItems = BM * 2 * KC;
  static constexpr int kAPt = (kAItems + kThreads - 1) / kThreads;
  static constexpr int kABytes = KC * BM * kPitch * 2;
  static constexpr int kWWave = 32 * NT * WRow<QT>::kPitch;
  static constexpr int kStages = 2 * kABytes + WN * KW * kWWave;
  // results pass through LDS, PI x NT MFMA tiles of every wave at a time
  static constexpr int PI = MT % 2 == 0 ? 2 : 1;
  static constexpr int kTileF = 1024 + 32;  // floats of a tile: a skew of half the banks
  static constexpr int kPartF = PI * NT * kTileF;  // floats of a wave
  static constexpr int kSumBytes = WN * KW * kPartF * 4;
  static constexpr int kLds = kStages > kSumBytes ? kStages : kSumBytes;
  static_assert(kLds <= 160 * 1024 && G % AU == 0 && G % US == 0, "LDS");
};

}  // namespace

template <int QT, bool AH, int MT, int NT, int WN, int KW, int AU>
__global__ __launch_bounds__(64 * WN * KW, 2) void k_gemm_f16(const F16Args g) {
  using T = Tile<QT, MT, NT, WN, KW, AU>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem_raw[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave % WN, kw = wave / WN;
  const int l32 = lane & 31, h = lane >> 5;

  // XCD-aware tile order: workgroup b runs on XCD b % 8; give each XCD a
  // contiguous run of the (n, split, m) tile sequence.
  const int total = gridDim.x;
  int b = blockIdx.x;
  if ((total & 7) == 0) b = (b & 7) * (total >> 3) + (b >> 3);
  // scalar: a descriptor chosen by a value in a vector register would put
  // every weight load in a readfirstlane loop
  const int rest = __builtin_amdgcn_readfirstlane(b / g.m_tiles);
  const int mt = b - rest * g.m_tiles;
  int nt = __builtin_amdgcn_readfirstlane(rest / g.splits);
  const int split = rest - nt * g.splits;
  const uint8_t *W = g.seg[0].W;
  void *Y = g.seg[0].Y;
  int N = g.seg[0].N;
  if (nt >= g.seg[0].tile_end) {
    const bool third = nt >= g.seg[1].tile_end;
    W = third ? g.seg[2].W : g.seg[1].W;
    Y = third ? g.seg[2].Y : g.seg[1].Y;
    N = third ? g.seg[2].N : g.seg[1].N;
    nt -= third ? g.seg[1].tile_end : g.seg[0].tile_end;
  }
  const int m0 = mt * T::BM, n0 = nt * T::BN;
  const int M = g.M, K = g.K;
  const int nch = K / kBK;
  constexpr int kGroup = KW * T::G;  // chunks of all waves' group
  const int g_begin = split * g.spw;
  const int g_end = min((nch + kGroup - 1) / kGroup, g_begin + g.spw);

  const int nblk32 = K >> 5;
  // AH: A holds fp16 activations (64 bytes per 32-value block)
  const uint32_t a_row = static_cast<uint32_t>(nblk32) * (AH ? 64 : kQ8_1Bytes);
  const uint32_t w_row = static_cast<uint32_t>(row_bytes(QT, K));
  const uint64_t wp = reinterpret_cast<uint64_t>(W);
  const uint64_t wu = static_cast<uint64_t>(static_cast<uint32_t>(
                          __builtin_amdgcn_readfirstlane(static_cast<int>(wp >> 32))))
                          << 32 |
                      static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(wp)));
  const uint32_t w_bytes = __builtin_amdgcn_readfirstlane(w_row * static_cast<uint32_t>(N));
  const rsrc_t Ar = make_rsrc(g.A, a_row * static_cast<uint32_t>(M));
  const void *const wq = reinterpret_cast<const void *>(wu);

  f32x16 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // Stage x = (group, step): waves kw compute chunks step * AU .. of the G chunks
  // from (group * KW + kw) * G on.  Items: it = ((row * KW + kw) * AU + chunk) * 2 + half.
  // Rows past M or N repeat the last row (their outputs are never stored); a
  // chunk past K reads zeros through an empty range, so it adds nothing.
  RawA<AH> ra[T::kAPt];
  RawW<QT, NT> rw;
  const int x_begin = g_begin * T::kSteps, x_last = max(x_begin, g_end * T::kSteps - 1);
  auto item_chunk = [&](int x, int it) {
    const int k = (it >> 1) % T::KC;
    return (x / T::kSteps * KW + k / AU) * T::G + x % T::kSteps * AU + k % AU;
  };
  auto fetch_stage = [&](int x) {
    x = min(x, x_last);
#pragma unroll
    for (int u = 0; u < T::kAPt; ++u) {
      const int it = tid + T::kThreads * u;
      const int row = it / (2 * T::KC), c = item_chunk(x, it);
      // (a chunk past K reads zeros, past every tensor)
      if (T::kAItems % T::kThreads == 0 || it < T::kAItems)
        fetch_a<QT, AH>(ra[u], Ar, c < nch ? min(m0 + row, M - 1) * a_row : kOobOffset, c < nch ? c : 0,
                        it & 1);
    }
  };
  auto commit_stage = [&](int buf) {
    _Float16 *base = reinterpret_cast<_Float16 *>(smem_raw + buf * T::kABytes);
#pragma unroll
    for (int u = 0; u < T::kAPt; ++u) {
      const int it = tid + T::kThreads * u;
      const int row = it / (2 * T::KC), k = (it >> 1) % T::KC;
      if (T::kAItems % T::kThreads == 0 || it < T::kAItems)
        commit_a<AH>(base + k * T::BM * kPitch, ra[u], row, it & 1);
    }
  };
  const int n_wave = n0 + 32 * NT * wn;
  uint8_t *wrows = smem_raw + 2 * T::kABytes + wave * T::kWWave;
  // The wave's q-th unit (q counts kUnits a group) by its place along K.
  auto unit_of = [&](int q) {
    q = min(q, g_end * T::kUnits - 1);
    return __builtin_amdgcn_readfirstlane((q / T::kUnits * KW + kw) * T::kUnits + q % T::kUnits);
  };
  auto fetch_unit = [&](int q) {
    const int un = unit_of(q);
    // a unit past K reads zeros through an empty range
    const bool in = un * T::US < nch;
    fetch_w<QT, NT>(rw, make_rsrc(wq, __builtin_amdgcn_readfirstlane(in ? w_bytes : 0)), n_wave, N,
                    w_row, un, lane);
  };

  auto lane_weights = [&](LaneW<QT> (&lw)[NT], int ch) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
      lw[j] = read_w<QT>(wrows + (32 * j + l32) * WRow<QT>::kPitch, ch, h);
  };
  auto read_a = [&](h8 (&f)[MT], const _Float16 *sa, int sl) {
    // rows l32 + 32 i share swz(l32): period 16
    const int ga = 8 * (a_group(sl, h) ^ swz(l32));
#pragma unroll
    for (int i = 0; i < MT; ++i)
      f[i] = *reinterpret_cast<const h8 *>(sa + (l32 + 32 * i) * kPitch + ga);
  };

  // Stage x is computed from one buffer while stage x + 1's activations are
  // converted into the other and stage x + 2's are fetched; a unit's weights are
  // fetched a unit ahead and staged as the last chunk of the unit before begins
  // its last slot.  Within a stage the operands of the next slot (A
  // from LDS, W dequantized) are made while the MFMAs of one run.  Past the
  // end the last stage is fetched again, into a buffer nobody reads, so the
  // loop body holds no branches.
  // Loads complete in issue order; the prologue issues them in the loop's
  // order (activations, then weights), or the loop's waits would count for it
  // and wait for the weights just issued.
  fetch_stage(x_begin);
  fetch_unit(g_begin * T::kUnits);
  commit_stage(0);
  fetch_stage(x_begin + 1);
  commit_w<QT, NT>(wrows, rw, unit_of(g_begin * T::kUnits), lane);
  wave_sync();  // lanes read rows that others staged
  fetch_unit(g_begin * T::kUnits + 1);
  LaneW<QT> lw[NT];
  h8 fa[2][MT], fb[2][NT];
  lane_weights(lw, 0);
#pragma unroll
  for (int j = 0; j < NT; ++j) fb[0][j] = w_slot<QT>(lw[j], 0);
  __syncthreads();

  int x = x_begin;
  for (int gr = g_begin; gr < g_end; ++gr) {
#pragma unroll
    for (int st = 0; st < T::kSteps; ++st, ++x) {
      const int buf = T::kSteps % 2 == 0 ? st & 1 : (x - x_begin) & 1;
      const _Float16 *abuf =
          reinterpret_cast<const _Float16 *>(smem_raw + buf * T::kABytes) + kw * AU * T::BM * kPitch;
      read_a(fa[0], abuf, 0);
      commit_stage(buf ^ 1);
      fetch_stage(x + 2);
#pragma unroll
      for (int ph = 0; ph < 4 * AU; ++ph) {
        const int cur = ph & 1, nxt = cur ^ 1, sl = ph & 3, ch = st * AU + ph / 4;
        if (ph + 1 < 4 * AU) read_a(fa[nxt], abuf + (ph + 1) / 4 * T::BM * kPitch, (ph + 1) & 3);
        if (sl == 3) {
          if ((ch + 1) % T::US == 0) {
            const int q = gr * T::kUnits + ch / T::US;
            // the rows staged before have been read (with these two fences the
            // compiler's schedule is the better one: Q8_0 512 x 13824 x 5120 on
            // 128 x 256 123 -> 102 us, geomean over 384 launches 0.98, all in 1.04)
            wave_sync();
            commit_w<QT, NT>(wrows, rw, unit_of(q + 1), lane);
            wave_sync();
            fetch_unit(q + 2);
          }
          lane_weights(lw, (ch + 1) % T::US);
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) fb[nxt][j] = w_slot<QT>(lw[j], (sl + 1) & 3);
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int i = 0; i < MT; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[cur][i], fb[cur][j], acc[i][j], 0, 0, 0);
      }
      __syncthreads();
    }
  }

  // Results pass through LDS: the K groups' sums meet there in group order,
  // and the stores run along the rows.  Tile (i, j) of a wave is kept as its
  // accumulators lie, element e of lane l at 64 e + l (row 8 (e / 4) + 4 (l / 32)
  // + e % 4, column l % 32), so a row's 32 columns are contiguous.
  float *sum = reinterpret_cast<float *>(smem_raw);
  constexpr int kRows = 32 * T::PI / KW;  // rows of a pass that one wave stores
  auto store = [&](auto cols, int i0) __attribute__((always_inline)) {
    constexpr int C = decltype(cols)::value, kLanes = 32 * NT / C, kRpi = 64 / kLanes;
    const int col = lane % kLanes * C;
#pragma unroll
    for (int r0 = 0; r0 < kRows; r0 += kRpi) {
      const int rw = r0 + lane / kLanes, r = kw * kRows + rw, rr = r & 31;
      const float *p = sum + wn * T::kPartF + ((r >> 5) * NT + (col >> 5)) * T::kTileF +
                       64 * (4 * (rr >> 3) + (rr & 3)) + 32 * ((rr >> 2) & 1) + (col & 31);
      f32x4 v[C / 4];
      if (kRows % kRpi == 0 || rw < kRows) {
#pragma unroll
        for (int k = 0; k < C / 4; ++k) {
          v[k] = *reinterpret_cast<const f32x4 *>(p + 4 * k);
#pragma unroll
          for (int c = 1; c < KW; ++c)
            v[k] += *reinterpret_cast<const f32x4 *>(p + c * WN * T::kPartF + 4 * k);
        }
        put<C>(g, Y, N, split, m0 + 32 * i0 + r, n_wave + col, v);
      }
    }
  };
  // Atomic adds, and stores to rows that do not start on 16 bytes: a column a
  // lane, so that a wave's accesses fall on whole lines, and the sums of several
  // rows read before the first is stored.  us with 4 or 8 single stores a lane / so:
  // Q4_K 1905 x 30662 x 512 167 / 126 (a multiple of 8, 16-byte stores: 116),
  // 743 x 16385 x 512 44 / 31, Q6_K 464 x 17874 x 1024 to fp16 59 / 47.
  auto put_columns = [&](auto epi, int i0) __attribute__((always_inline)) {
    constexpr int E = decltype(epi)::value, B = kRows / 2 < 8 ? kRows / 2 : 8;
    using O = std::conditional_t<E == kEpiF16, uint16_t, float>;
    const int row = m0 + 32 * i0 + kw * kRows + h, n = n_wave + l32;
    O *y = static_cast<O *>(Y) + (E == kEpiSlot ? static_cast<int64_t>(split) * M * N : 0) +
           static_cast<int64_t>(row) * N + n;
    const bool with_y = (E == kEpiF32 || E == kEpiF16) && g.mode == 1;
    const bool with_bias = E != kEpiSlot && g.mode == 2 && (E != kEpiAtomic || split == 0);
    const auto f32 = [](O v) __attribute__((always_inline)) {
      if constexpr (E == kEpiF16) return h2f(v);
      else return v;
    };
#pragma unroll
    for (int r0 = 0; r0 < kRows; r0 += 2 * B) {
      float v[B][NT];
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const int r = kw * kRows + r0 + 2 * b + h, rr = r & 31;
          const float *p = sum + wn * T::kPartF + ((r >> 5) * NT + j) * T::kTileF +
                           64 * (4 * (rr >> 3) + (rr & 3)) + 32 * ((rr >> 2) & 1) + l32;
          v[b][j] = p[0];
#pragma unroll
          for (int c = 1; c < KW; ++c) v[b][j] += p[c * WN * T::kPartF];
        }
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          if (row + r0 + 2 * b < M && n + 32 * j < N) {
            O *o = y + static_cast<int64_t>(r0 + 2 * b) * N + 32 * j;
            float t = v[b][j];
            if (with_y) t += f32(*o);
            if (with_bias) t += f32(static_cast<const O *>(g.bias)[n + 32 * j]);
            if constexpr (E == kEpiAtomic) atomicAdd(o, t);
            else if constexpr (E == kEpiF16) *o = static_cast<uint16_t>(f2h_bits(t));
            else *o = t;
          }
    }
  };
  auto pass = [&](auto first) __attribute__((always_inline)) {
    constexpr int i0 = decltype(first)::value;
    if constexpr (i0 < MT) {
      if constexpr (i0 > 0) {  // the pass before has been read
        if constexpr (KW > 1) __syncthreads();
        else wave_sync();
      }
      float *d = sum + (kw * WN + wn) * T::kPartF + lane;
#pragma unroll
      for (int i = 0; i < T::PI; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) d[(i * NT + j) * T::kTileF + 64 * e] = acc[i0 + i][j][e];
      if constexpr (KW > 1) __syncthreads();
      else wave_sync();
      if (g.epi == kEpiAtomic) put_columns(std::integral_constant<int, kEpiAtomic>{}, i0);
      else if (!g.vec && g.epi == kEpiF16) put_columns(std::integral_constant<int, kEpiF16>{}, i0);
      else if (!g.vec && g.epi == kEpiSlot) put_columns(std::integral_constant<int, kEpiSlot>{}, i0);
      else if (!g.vec) put_columns(std::integral_constant<int, kEpiF32>{}, i0);
      else if (g.epi == kEpiF16) store(std::integral_constant<int, 8>{}, i0);
      else store(std::integral_constant<int, 4>{}, i0);
    }
  };
  pass(std::integral_constant<int, 0>{});
  pass(std::integral_constant<int, T::PI>{});
  pass(std::integral_constant<int, 2 * T::PI>{});
  pass(std::integral_constant<int, 3 * T::PI>{});
}

// Tile of a launch by index (f16_plan).
template <int QT, bool AH, int MT, int NT, int WN, int KW, int AU>
hipError_t launch_tile(const F16Args &g, int grid, hipStream_t s) {
  using T = Tile<QT, MT, NT, WN, KW, AU>;
  const auto fn = k_gemm_f16<QT, AH, MT, NT, WN, KW, AU>;
  if (!dry_run()) {  // set once per instantiation (a function-local static: thread-safe)
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void *>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, T::kLds);
    if (attr != hipSuccess) return attr;
  }
  // type, waves, epilogue (fp16; 1 atomic, 2 slots) and AH, then the tile
  if (note_launch("k_gemm_f16", {QT, T::kThreads / 64, g.epi == kEpiF16,
                                 g.epi == kEpiAtomic ? 1 : g.epi == kEpiSlot ? 2 : 0, AH},
                  {MT, NT, WN, KW, AU}))
    hipLaunchKernelGGL(fn, dim3(static_cast<unsigned>(grid)), dim3(T::kThreads), T::kLds, s, g);
  return last_error();
}

// The tiles a launch can take (kF16Tiles in gemm_f16.hip).  All but the last have
// eight waves; those with fewer along n split the stage's K range.  The last, on
// four waves, sums K in order (kOrderedTile).  The largest is 128 x 512 for Q4_K
// and 256 x 256 for Q6_K and Q8_0, where a weight is then converted once for 256
// rows, not 128.  us on 128 x 512 / on 256 x 256, x 27648 x 5120 with the fp16 copy at
// M = 384, 512, 1999, and 1999 x 13824 x 5120 without:
//   Q8_0  185 / 150   184 / 155   720 / 628   355 / 335
//   Q6_K  196 / 170   197 / 182   768 / 732   384 / 351
//   Q4_K  135 / 146   153 / 153   598 / 624   297 / 316
// Q6_K's 128 x 256 has its waves along n, too: with two K waves it needed more
// registers than there are (four spilled with the fp16 copy) and took, with
// the copy, 126 us at 256 x 27648 x 5120 (110 now), without 53 at 512 x 11008 x 2048 (48).
template <int QT, bool AH>
hipError_t launch_by_tile(int tile, const F16Args &g, int grid, hipStream_t s) {
  switch (tile) {
  case 0:
    if constexpr (QT != kTypeQ4_K) return hipErrorInvalidValue;  // not planned
    else return launch_tile<QT, AH, 4, 2, 8, 1, 2>(g, grid, s);
  case 1:
    if constexpr (QT == kTypeQ6_K) return hipErrorInvalidValue;
    else return launch_tile<QT, AH, 4, 2, 4, 2, 1>(g, grid, s);
  case 2: return launch_tile<QT, AH, 3, 2, 4, 2, 1>(g, grid, s);
  case 3: return launch_tile<QT, AH, 2, 2, 4, 2, QT == kTypeQ8_0 || AH ? 1 : 2>(g, grid, s);
  case 4: return launch_tile<QT, AH, 2, 2, 2, 4, 1>(g, grid, s);
  case 5: return launch_tile<QT, AH, 1, 2, 2, 4, 1>(g, grid, s);
  case 6: return launch_tile<QT, AH, 1, 2, 1, 8, 1>(g, grid, s);
  case 7:
    if constexpr (QT != kTypeQ6_K) return hipErrorInvalidValue;
    else return launch_tile<QT, AH, 4, 1, 8, 1, 2>(g, grid, s);
  case 8:
    if constexpr (QT == kTypeQ4_K) return hipErrorInvalidValue;
    else return launch_tile<QT, AH, 8, 1, 8, 1, 1>(g, grid, s);
  default:
    if constexpr (QT == kTypeQ8_0 || AH) return hipErrorInvalidValue;
    else return launch_tile<QT, AH, 2, 1, 4, 1, 2>(g, grid, s);
  }
}

}  // namespace ifx
