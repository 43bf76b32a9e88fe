// Device-side helpers shared by the gfx950 kernels: bit casts, fp16 scale decoding, wave64 reductions.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

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
// The quantizers that write operand order go by it: the 16-byte pieces of eight rows are one cache line, which would
// otherwise lie partly written in eight L2 caches (layers of 128 / 256 / 400 rows of Q8_0, hidden 1536 / 1536 / 2048, 85.5 -> 84.3,
// 113.5 -> 110.7, 162.7 -> 160.3 us; 100 fp32 rows of 8960 against 1537 22.4 -> 21.6; a single row tile, whose few rows all go
// everywhere, 12.7 -> 13.2, stays as it comes).
__device__ __forceinline__ unsigned xcd_neighbours(unsigned b, unsigned n) {
  const unsigned xcd = b & 7u;
  return xcd * (n >> 3) + min(xcd, n & 7u) + (b >> 3);
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
  float          x[8], amax = 0.0f;
  const float4  *p  = reinterpret_cast<const float4 *>(job.src + (size_t) (live ? block : 0u) * kQK + part * 8);
  const float4   v0 = p[0], v1 = p[1];
  x[0] = v0.x, x[1] = v0.y, x[2] = v0.z, x[3] = v0.w, x[4] = v1.x, x[5] = v1.y, x[6] = v1.z, x[7] = v1.w;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    amax = fmaxf(amax, fabsf(x[i]));
  }
  amax = quad_max(amax);
  const float d  = amax / 127.0f;
  const float id = (d != 0.0f) ? 1.0f / d : 0.0f;
  if (!live) {
    return;
  }
  uint16_t *to = reinterpret_cast<uint16_t *>(job.dst + (size_t) block * 34);
  if (part == 0) {
    to[0] = __half_as_ushort(__float2half_rn(d));
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q0 = (int) roundf(x[2 * i] * id), q1 = (int) roundf(x[2 * i + 1] * id);
    to[1 + part * 4 + i] = (uint16_t) ((q0 & 0xff) | ((q1 & 0xff) << 8));
  }
}

// Activations in the operand order of the int8 matmul, [32-row tile][block][64 lanes] of 16 bytes: lane (c = row % 32, h)
// holds elements 16 h .. 16 h + 15 of its row's block. The scale array behind them holds a dword (fp16 scale, 0) per row and
// block, [tile][block][64] with zeros in the upper 32, and ends in one row of 64 zeros.
struct ActFragments {
  uint2    *frag   = nullptr;
  uint32_t *scales = nullptr;
  int       m_tiles = 0, nblk = 0;
};
inline ActFragments act_fragments_at(void *base, int m, int k) {
  ActFragments f;
  if (base) {
    f.m_tiles = (m + 31) / 32, f.nblk = k / kQK;
    f.frag   = static_cast<uint2 *>(base);
    f.scales = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(base) + (((size_t) f.m_tiles * f.nblk * 1024 + 255) & ~(size_t) 255));
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
// the row of zeros, from 64 threads of the grid
__device__ __forceinline__ void end_act_fragments(const ActFragments &f, int thread) {
  if (thread < 64) {
    f.scales[(size_t) f.m_tiles * f.nblk * 64 + thread] = 0u;
  }
}

}  // namespace htpops
