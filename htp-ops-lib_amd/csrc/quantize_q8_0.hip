// Q8_0 activation quantizer for gfx950.
//
// Replaces the fp32 -> fp16 activation staging of the reference (src/dsp/ops/mat_mul.c:89-128) with ggml's
// Q8_0 arithmetic: per 32-value block d = amax / 127, id = d ? 1/d : 0, q = roundf(x * id), scale = fp16(d).
// Bandwidth bound: 128 B read and 34 B written per block.
//
// Mapping: four lanes share a block (8 floats = two 16-byte loads each). amax is exchanged inside the quad,
// each lane rounds its eight values, and a wave's sixteen blocks (544 contiguous bytes) are assembled in LDS so
// that the 34-byte blocks leave as aligned dword stores.
#include "device_utils.h"
#include "kernels.h"

namespace htpops {

namespace {

constexpr int kThreads        = 256;
constexpr int kBlocksPerWave  = 16;                        // 64 lanes / 4 lanes per block
constexpr int kBlocksPerGroup = kBlocksPerWave * (kThreads / kWave);
constexpr int kWaveOutBytes   = kBlocksPerWave * 34;       // 544
constexpr int kWaveOutDwords  = kWaveOutBytes / 4;         // 136

__device__ __forceinline__ void load_eight(float x[8], const float *src, bool live) {
  if (live) {
    const float4 *p  = reinterpret_cast<const float4 *>(src);
    const float4  v0 = p[0];
    const float4  v1 = p[1];
    x[0] = v0.x, x[1] = v0.y, x[2] = v0.z, x[3] = v0.w;
    x[4] = v1.x, x[5] = v1.y, x[6] = v1.z, x[7] = v1.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = 0.0f;
    }
  }
}

// the image is private to its wave: a wavefront-scope release/acquire pair orders the LDS traffic
__device__ __forceinline__ void image_complete() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// total_blocks = m * k / 32; blocks are contiguous in both src (128 B each) and dst (34 B each).
__global__ __launch_bounds__(kThreads) void quantize_q8_0_kernel(uint8_t *__restrict__ dst, const float *__restrict__ src,
                                                                  long long total_blocks) {
  __shared__ __attribute__((aligned(16))) uint16_t stage[kThreads / kWave][kWaveOutBytes / 2];

  const int       lane       = threadIdx.x & (kWave - 1);
  const int       wave       = threadIdx.x / kWave;
  const long long wave_block = ((long long) blockIdx.x * (kThreads / kWave) + wave) * kBlocksPerWave;
  if (wave_block >= total_blocks) {
    return;
  }
  const long long block = wave_block + (lane >> 2);
  const int       part  = lane & 3;  // which 8 of the block's 32 values
  float           x[8];
  uint16_t        scale;
  load_eight(x, src + block * kQK + part * 8, block < total_blocks);
  const uint2 quants = quantize_eight(x, &scale);

  uint16_t *img = stage[wave];
  store_q8_0_block(img + (lane >> 2) * 17, part, quants, scale);
  image_complete();

  // 16 blocks start at a multiple of 16 blocks = 544 bytes, so the image is dword aligned in dst.
  long long remaining = total_blocks - wave_block;
  const int n_dwords  = remaining >= kBlocksPerWave ? kWaveOutDwords : (int) (remaining * 34 / 4);
  const int n_bytes   = remaining >= kBlocksPerWave ? kWaveOutBytes : (int) (remaining * 34);
  uint32_t       *out32 = reinterpret_cast<uint32_t *>(dst + wave_block * 34);
  const uint32_t *img32 = reinterpret_cast<const uint32_t *>(img);
  for (int i = lane; i < n_dwords; i += kWave) {
    out32[i] = img32[i];
  }
  // an odd number of trailing blocks leaves two bytes
  if (lane == 0 && (n_bytes & 3)) {
    reinterpret_cast<uint16_t *>(dst + wave_block * 34)[n_bytes / 2 - 1] = img[n_bytes / 2 - 1];
  }
}

// The same rows, also in the operand order ORDER of the matmul behind (see ActFragments); dst may be nullptr. There the 16 bytes
// of neighbouring rows lie side by side, so a wave's sixteen blocks are two blocks of eight rows: its stores of the operand
// are whole lines of 128 bytes, and its pieces of the rows in block_q8_0 form 68 bytes, continued by its neighbours. (With
// sixteen blocks of one row a store instruction went to 32 lines, an eighth of each: int8 order of 128 rows of 1536 / 8960
// 4.0 -> 3.1 / 5.6 -> 4.4 us, of 27 rows of 8960 5.1 -> 3.0, FP6 order of 512 rows of 4096 / 11008 6.0 -> 5.9 / 13.8 -> 12.1; the
// rows alone 5.4 / 8.2 and the launch that put them into FP6 order 5.5 / 6.3. Neighbouring groups on one XCD: the same,
// but 64 rows of 1056 12.7 -> 13.1 with their matmul.)
constexpr int kRowsPerWave = 8;
template <int ORDER>
__global__ __launch_bounds__(kThreads) void quantize_operand_kernel(uint8_t *__restrict__ dst, const float *__restrict__ src, int m,
                                                                     unsigned groups_per_row, ActFragments fragments) {
  __shared__ __attribute__((aligned(16))) uint16_t stage[kThreads / kWave][kWaveOutBytes / 2];

  const int lane = threadIdx.x & (kWave - 1);
  const int wave = threadIdx.x / kWave;
  if (ORDER == kActI8 && blockIdx.x == 0 && threadIdx.x < kWave) {
    end_act_fragments(fragments, threadIdx.x);
  }
  const unsigned group = blockIdx.x;
  const int      row0 = (int) (group / groups_per_row) * kRowsPerWave, nblk = fragments.nblk;
  const int      kb0 = ((int) (group % groups_per_row) * (kThreads / kWave) + wave) * 2;
  if (kb0 >= nblk) {
    return;
  }
  const int  part = lane & 3, r = (lane >> 2) & 7, b = lane >> 5;
  const int  row = row0 + r, kb = kb0 + b;
  const bool live = row < m && kb < nblk;
  float      x[8];
  uint16_t   scale;
  load_eight(x, src + ((size_t) row * nblk + kb) * kQK + part * 8, live);
  const uint2 quants = quantize_eight(x, &scale);
  if (live) {
    if constexpr (ORDER == kActFp6) {
      store_act_fp6(fragments, row, kb, part, quants, scale);
    } else {
      store_act_fragment(fragments, row, kb, part, quants, scale);
    }
  }
  if (dst == nullptr) {
    return;
  }

  // LDS image of this wave's pieces of eight rows, 68 bytes each
  uint16_t *img = stage[wave];
  store_q8_0_block(img + r * 34 + b * 17, part, quants, scale);
  image_complete();
  uint8_t *out = dst + ((size_t) row0 * nblk + kb0) * 34;
  if (nblk % 2 == 0) {  // pieces of whole dwords
    for (int i = lane; i < kRowsPerWave * 17; i += kWave) {
      const int to = i / 17;
      if (row0 + to < m) {
        reinterpret_cast<uint32_t *>(out + (size_t) to * nblk * 34)[i % 17] = reinterpret_cast<const uint32_t *>(img)[i];
      }
    }
  } else {
    for (int i = lane; i < kRowsPerWave * 34; i += kWave) {
      const int to = i / 34, at = i % 34;
      if (row0 + to < m && (at < 17 || kb0 + 1 < nblk)) {
        reinterpret_cast<uint16_t *>(out + (size_t) to * nblk * 34)[at] = img[i];
      }
    }
  }
}

}  // namespace

hipError_t launch_quantize_q8_0(hipStream_t stream, void *dst, const float *src, int k, int m, void *act_fragments,
                                ActOrder order) {
  const long long total_blocks = (long long) m * (k / kQK);
  const long long groups       = (total_blocks + kBlocksPerGroup - 1) / kBlocksPerGroup;
  if (act_fragments) {
    if (total_blocks > 0x7fffffffLL) {
      return hipErrorInvalidValue;
    }
    const unsigned per_row = (unsigned) ((k / kQK + 2 * (kThreads / kWave) - 1) / (2 * (kThreads / kWave)));
    const unsigned rows    = (unsigned) ((m + kRowsPerWave - 1) / kRowsPerWave);
    if ((unsigned long long) per_row * rows > 0x7fffffffULL) {
      return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(order == kActFp6 ? quantize_operand_kernel<kActFp6> : quantize_operand_kernel<kActI8>, dim3(per_row * rows),
                       dim3(kThreads), 0, stream, (uint8_t *) dst, src, m, per_row, act_fragments_at(act_fragments, m, k, order));
  } else {
    hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned) groups), dim3(kThreads), 0, stream, (uint8_t *) dst, src,
                       total_blocks);
  }
  return hipGetLastError();
}

}  // namespace htpops
