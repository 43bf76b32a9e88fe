// Device-side helpers shared by the gfx950 kernels: bit casts, fp16 scale decoding, wave64 reductions.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

namespace htpops {

constexpr int kWave = 64;
constexpr int kQK   = 32;  // values per quant block (reference: include/dsp/quants.h:7)

// 4-byte aligned 16-byte vector: quant rows are only dword aligned (18- and 34-byte blocks).
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

__device__ __forceinline__ float half_bits_to_float(uint32_t bits16) {
  return __half2float(__ushort_as_half((unsigned short) (bits16 & 0xffffu)));
}

__device__ __forceinline__ int dot4_i8(uint32_t a, uint32_t b, int acc) {
  return __builtin_amdgcn_sdot4((int) a, (int) b, acc, false);
}

// Sum over the `width` (power of two, <= 64) consecutive lanes that share lane / width.
template <int width>
__device__ __forceinline__ float group_sum(float v) {
#pragma unroll
  for (int off = width / 2; off > 0; off >>= 1) {
    v += __shfl_xor(v, off, kWave);
  }
  return v;
}

template <int width>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
  for (int off = width / 2; off > 0; off >>= 1) {
    v = fmaxf(v, __shfl_xor(v, off, kWave));
  }
  return v;
}

// The same over the 64 lanes of a wave and over quads with DPP row operations: no trip through the LDS crossbar, which
// is what a kernel that is one chain of dependent latencies wants. Every lane gets the result. (The additions of
// wave_sum come in another order than group_sum's; kernels that must agree bit for bit use the same one.)
#define HTPOPS_DPP_STEP(op, ctrl, rows) \
  v = op(v, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(ident), __float_as_int(v), ctrl, rows, 0xf, false)))
__device__ __forceinline__ float dpp_add(float a, float b) {
  return a + b;
}
__device__ __forceinline__ float wave_max(float v) {
  const float ident = -INFINITY;
  HTPOPS_DPP_STEP(fmaxf, 0xB1, 0xf);   // quad_perm [1,0,3,2]
  HTPOPS_DPP_STEP(fmaxf, 0x4E, 0xf);   // quad_perm [2,3,0,1]
  HTPOPS_DPP_STEP(fmaxf, 0x141, 0xf);  // row_half_mirror
  HTPOPS_DPP_STEP(fmaxf, 0x140, 0xf);  // row_mirror: every lane of a 16-lane row holds the row's
  HTPOPS_DPP_STEP(fmaxf, 0x142, 0xa);  // row_bcast15 into rows 1 and 3
  HTPOPS_DPP_STEP(fmaxf, 0x143, 0xc);  // row_bcast31 into rows 2 and 3: lane 63 holds the wave's
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ float wave_sum(float v) {
  const float ident = 0.0f;
  HTPOPS_DPP_STEP(dpp_add, 0xB1, 0xf);
  HTPOPS_DPP_STEP(dpp_add, 0x4E, 0xf);
  HTPOPS_DPP_STEP(dpp_add, 0x141, 0xf);
  HTPOPS_DPP_STEP(dpp_add, 0x140, 0xf);
  HTPOPS_DPP_STEP(dpp_add, 0x142, 0xa);
  HTPOPS_DPP_STEP(dpp_add, 0x143, 0xc);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
// maximum over the four lanes of a quad (the same pairs in the same order as group_max<4>)
__device__ __forceinline__ float quad_max(float v) {
  const float ident = -INFINITY;
  HTPOPS_DPP_STEP(fmaxf, 0x4E, 0xf);  // quad_perm [2,3,0,1]
  HTPOPS_DPP_STEP(fmaxf, 0xB1, 0xf);  // quad_perm [1,0,3,2]
  return v;
}
#undef HTPOPS_DPP_STEP

// Workgroups are handed to the 8 XCDs round robin: the index of workgroup b of n when each XCD is to have neighbouring indices.
// RMSNorm + Q8_0 that writes operand order goes by it, a workgroup to a row: the 16-byte pieces of eight rows are one cache line,
// which would otherwise lie partly written in eight L2 caches (layers of 128 / 256 / 400 rows of Q8_0, hidden 1536 / 1536 /
// 2048, 85.5 -> 84.3, 113.5 -> 110.7, 162.7 -> 160.3 us, with the plain quantizer, whose waves held one row then, doing so
// too; a single row tile, whose few rows all go everywhere, 12.7 -> 13.2, stays as it comes).
__device__ __forceinline__ unsigned xcd_neighbours(unsigned b, unsigned n) {
  const unsigned xcd = b & 7u;
  return xcd * (n >> 3) + min(xcd, n & 7u) + (b >> 3);
}

// The eight values of a lane and its quad's block: quants (two dwords) and fp16 scale
__device__ __forceinline__ uint2 quantize_eight(const float x[8], uint16_t *scale) {
  float amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    amax = fmaxf(amax, fabsf(x[i]));
  }
  amax = quad_max(amax);

  const float d  = amax / 127.0f;
  const float id = (d != 0.0f) ? 1.0f / d : 0.0f;

  int q[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    q[i] = (int) roundf(x[i] * id);
  }
  *scale = __half_as_ushort(__float2half_rn(d));
  return { (uint32_t) ((q[0] & 0xff) | ((q[1] & 0xff) << 8) | ((q[2] & 0xff) << 16) | ((uint32_t) q[3] << 24)),
           (uint32_t) ((q[4] & 0xff) | ((q[5] & 0xff) << 8) | ((q[6] & 0xff) << 16) | ((uint32_t) q[7] << 24)) };
}

// A block's 34 bytes from the four lanes that hold it, to 2-byte aligned memory or LDS
__device__ __forceinline__ void store_q8_0_block(uint16_t *block, int part, uint2 quants, uint16_t scale) {
  uint16_t *to = block + 1 + part * 4;
  to[0]        = (uint16_t) quants.x;
  to[1]        = (uint16_t) (quants.x >> 16);
  to[2]        = (uint16_t) quants.y;
  to[3]        = (uint16_t) (quants.y >> 16);
  if (part == 0) {
    block[0] = scale;
  }
}

// Rows that a launch of other work quantizes to Q8_0 beside it (see QuantizeJob): its workgroups `first` and on do that, THREADS
// / 4 blocks each, with the arithmetic of quantize_q8_0_kernel (four lanes a block). No other launch has to be paid for a few
// KB of rows, nor waited for.
struct QuantizeBeside {
  const float *src   = nullptr;
  uint8_t     *dst   = nullptr;
  unsigned     blocks = 0;
  int          first  = 0x7fffffff;
};
__device__ __forceinline__ void quantize_beside(const QuantizeBeside &job, int workgroup, int threads) {
  const unsigned block = (unsigned) workgroup * (unsigned) (threads / 4) + threadIdx.x / 4, part = threadIdx.x & 3u;
  const bool     live  = block < job.blocks;
  float          x[8];
  const float4  *p  = reinterpret_cast<const float4 *>(job.src + (size_t) (live ? block : 0u) * kQK + part * 8);
  const float4   v0 = p[0], v1 = p[1];
  x[0] = v0.x, x[1] = v0.y, x[2] = v0.z, x[3] = v0.w, x[4] = v1.x, x[5] = v1.y, x[6] = v1.z, x[7] = v1.w;
  uint16_t    scale;
  const uint2 quants = quantize_eight(x, &scale);
  if (live) {
    store_q8_0_block(reinterpret_cast<uint16_t *>(job.dst + (size_t) block * 34), (int) part, quants, scale);
  }
}

// Activations in the operand order of the int8 matmul, [32-row tile][block][64 lanes] of 16 bytes: lane (c = row % 32, h)
// holds elements 16 h .. 16 h + 15 of its row's block. The scale array behind them holds a dword (fp16 scale, 0) per row and
// block, [tile][block][64] with zeros in the upper 32, and ends in one row of 64 zeros.
// In the operand order of the FP6 matmul (k % 64 == 0): [32-row tile][step of two blocks] of kFp6ActTile bytes, each quant split
// as 16 hi + lo into two E2M3 planes (see the head of gemm_fp6_lds.hip, and its converter of stored rows, whose bytes these are);
// the scales behind, [kFp6RowBlock rows][step][row] of (fp16, fp16, 0).
constexpr int kFp6ActTile = 3 * 1024, kFp6RowBlock = 128;
struct ActFragments {
  uint2    *frag   = nullptr;
  uint32_t *scales = nullptr;
  int       m_tiles = 0, nblk = 0;
};
inline ActFragments act_fragments_at(void *base, int m, int k, ActOrder order) {
  ActFragments f;
  if (base) {
    f.m_tiles = (m + 31) / 32, f.nblk = k / kQK;
    f.frag   = static_cast<uint2 *>(base);
    const size_t operand = order == kActFp6 ? (size_t) f.m_tiles * (f.nblk / 2) * kFp6ActTile :
                                              ((size_t) f.m_tiles * f.nblk * 1024 + 255) & ~(size_t) 255;
    f.scales = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(base) + operand);
  }
  return f;
}
// eight quants of a block (those of lane `part` of the quad that holds it) and, from lanes 0 and 1, its scale
__device__ __forceinline__ void store_act_fragment(const ActFragments &f, int row, int kb, int part, uint2 quants, uint16_t scale) {
  const size_t at = ((size_t) (row >> 5) * f.nblk + kb) * 64 + (row & 31);
  f.frag[(at + 32 * (part >> 1)) * 2 + (part & 1)] = quants;
  if (part < 2) {
    f.scales[at + 32 * part] = part == 0 ? scale : 0u;
  }
}
// The codes of four quants as E2M3, 24 bits: low nibbles (0..15) and high ones (two's complement) as sign and magnitude, times 1/8.
__device__ __forceinline__ uint32_t fp6_pack(uint32_t c) {
  return (c & 0x3fu) | ((c >> 2) & 0xfc0u) | ((c >> 4) & 0x3f000u) | ((c >> 6) & 0xfc0000u);
}
__device__ __forceinline__ uint32_t fp6_low_codes(uint32_t q) {
  return fp6_pack(q & 0x0f0f0f0fu);
}
__device__ __forceinline__ uint32_t fp6_high_codes(uint32_t q) {
  const uint32_t h = (q >> 4) & 0x0f0f0f0fu, neg = (h >> 3) & 0x01010101u;
  return fp6_pack(((h ^ (neg * 15u)) + neg) | (neg << 5));  // |hi| <= 8 per byte, no carry between bytes
}
template <int PERM>
__device__ __forceinline__ uint32_t quad_move(uint32_t v) {
  return (uint32_t) __builtin_amdgcn_mov_dpp((int) v, PERM, 0xf, 0xf, true);
}
// The same for the FP6 order, by the whole quad that holds the block. A lane's eight quants are six bytes of either plane; lanes
// 0 and 2 gather the first 16 of the 24 bytes of the high and of the low plane, lanes 1 and 3 the other 8, and store them whole.
__device__ __forceinline__ void store_act_fp6(const ActFragments &f, int row, int kb, int part, uint2 quants, uint16_t scale) {
  const uint32_t h0 = fp6_high_codes(quants.x), h1 = fp6_high_codes(quants.y);
  const uint32_t l0 = fp6_low_codes(quants.x), l1 = fp6_low_codes(quants.y);
  const uint32_t hx = h0 | (h1 << 24), hy = h1 >> 8, lx = l0 | (l1 << 24), ly = l1 >> 8;
  const bool     low = part >= 2;
  const uint32_t x03h = quad_move<0xcc>(hx), x03l = quad_move<0xcc>(lx);  // of lane 0 for the heads, of lane 3 for the tails
  const uint32_t y03h = quad_move<0xcc>(hy), y03l = quad_move<0xcc>(ly);
  const uint32_t x1h = quad_move<0x55>(hx), x1l = quad_move<0x55>(lx);
  const uint32_t y12h = quad_move<0x99>(hy), y12l = quad_move<0x99>(ly);  // of lane 1 for the heads, of lane 2 for the tails
  const uint32_t x2h = quad_move<0xaa>(hx), x2l = quad_move<0xaa>(lx);
  const uint32_t x03 = low ? x03l : x03h, y03 = low ? y03l : y03h, x1 = low ? x1l : x1h, y12 = low ? y12l : y12h,
                 x2 = low ? x2l : x2h;
  const size_t step = (size_t) (row / 32) * (f.nblk / 2) + kb / 2;
  const int    b = kb & 1, lane = (row & 31) + (low ? 32 : 0);
  uint8_t     *tile = reinterpret_cast<uint8_t *>(f.frag) + step * kFp6ActTile;
  uint32_t    *sc   = f.scales + (((size_t) (row / kFp6RowBlock) * (f.nblk / 2) + kb / 2) * kFp6RowBlock + row % kFp6RowBlock) * 2;
  if ((part & 1) == 0) {
    reinterpret_cast<uint4 *>(tile + 2048 * b)[lane] = make_uint4(x03, y03 | (x1 << 16), (x1 >> 16) | (y12 << 16), x2);
  } else {
    reinterpret_cast<uint2 *>(tile + 1024 + 512 * b)[lane] = make_uint2(y12 | (x03 << 16), (x03 >> 16) | (y03 << 16));
  }
  if (part == 0) {
    reinterpret_cast<uint16_t *>(sc)[b] = scale;
  } else if (part == 1 && b == 0) {
    sc[1] = 0u;
  }
}
// the row of zeros, from 64 threads of the grid
__device__ __forceinline__ void end_act_fragments(const ActFragments &f, int thread) {
  if (thread < 64) {
    f.scales[(size_t) f.m_tiles * f.nblk * 64 + thread] = 0u;
  }
}

}  // namespace htpops
