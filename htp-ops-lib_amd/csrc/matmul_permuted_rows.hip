// Activation rows against the reference's own weight formats (its ops 1-4), read as they lie in memory.
//
// Replaces hmx_mat_mul_permuted_w16a32 and hmx_mat_mul_permuted_qk_0_d16a32 (reference: src/dsp/ops/mat_mul.c:758-855,
// :875-1153; fp16 tiles of src/host/test.c:300-312, super-blocks of 8 K rows x 32 columns with one fp16 scale per 2 x 16
// patch, dequantizers mat_mul.c:308-508): fp16 activations times weights that are fp16(quant * scale), sums in fp32,
// results rounded to fp16. With few rows the bound is the stream over the weight bytes (144 B per 256 Q4_0 or IQ4_NL
// weights, 272 B of Q8_0, 512 B of fp16): a converted fp16 copy would be 3.6 times the bytes of the 4-bit formats, so
// nothing is converted and the weights are turned to fp16 in registers, on their way into the matrix cores. The first
// kernel below takes up to 32 rows, the second more.
//
// The formats suit that: the 8 K rows of one column of a super-block are ONE dword of nibbles (two bytes per row pair
// for Q8_0, a dword per row pair for fp16 tiles), and those are exactly the 8 values that a lane feeds to
// v_mfma_f32_16x16x32_f16. A wave takes a 32 x 32 tile per step: lane (g = lane / 16, i = lane % 16) holds K rows
// 8 g .. 8 g + 7 (super-block g of the tile) of columns 2 i and 2 i + 1, two matrix instructions per step and 16 rows.
// A workgroup owns 32 columns over all of K, its waves take every eighth tile (the tiles of a column group are
// contiguous, so a workgroup reads one stream), and their sums meet in LDS in wave order: a result does not depend on
// the launch it is part of. Several steps of every wave are in flight before the first use.
// Measured on MI355X, a message with the seven projections of a Llama-7B layer over Q4_0 super-blocks, one token
// (114 MB): 24.0 us = 4.75 TB/s; 29.0 with all 16 bytes of a super-block's scales loaded by every lane (the path into the
// CU then carried 24 bytes a lane and step instead of 12, and registers kept a CU to fewer waves), 374 us for a launch
// per matrix over fp16 copies in operand order (7 x 41 us on 64 to 172 workgroups, each behind a 5 us conversion of the
// row). Vector-ALU work is about 30 instructions per step and wave, 10 us of it; 8 steps in flight instead of 4 for the 4-bit
// formats 24.5 us, 4 or 16 waves per workgroup (before) 30.3 and 31.0 against 28.1.
// The activations, rounded to fp16, are read from LDS where they fit (one or a few rows: every workgroup converts them
// for itself), else from a copy in operand order that one small launch makes.
#include "device_utils.h"
#include "kernels.h"

#include <algorithm>

namespace htpops {

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float    v4f __attribute__((ext_vector_type(4)));

constexpr int kRowsWaves   = 8;
constexpr int kRowsThreads = kRowsWaves * kWave;
// Activations up to this many bytes are kept in LDS (two workgroups per compute unit at least; with 80 KiB allowed,
// 8 rows of 4096 against IQ4_NL ran at 26.4 us per layer of seven 4096 x 4096 matrices, against 21.7 us in operand order).
constexpr int kRowsActLds    = 64 * 1024;
constexpr int kRowsWideTiles = 512;  // column groups of a launch from which a workgroup takes two (see the launcher)

struct RowsMember {
  float         *out;
  const float   *act;   // fp32 rows
  const uint4   *frag;  // the same in operand order (kernels that do not keep them in LDS)
  const uint8_t *weight;
  int            k, n, first;  // first: this member's first workgroup
};
struct RowsArgs {
  RowsMember member[kPermutedGroupMax];
  int        count, m;
};

template <int KIND>
struct RawStep;  // what a lane loads of one 32 x 32 tile
template <>
struct RawStep<1> {
  static constexpr int kTileBytes = 2048;
  uint2                q[4];  // K row pair 4 g + v, columns 2 i and 2 i + 1
};
template <>
struct RawStep<2> {
  static constexpr int kTileBytes = 4 * 144;
  uint32_t             s;  // two of the 8 scales of super-block g: those of place i % 4; the quad holds all
  uint2                q;  // 8 nibbles of column 2 i, 8 of column 2 i + 1
};
template <>
struct RawStep<4> : RawStep<2> {};
template <>
struct RawStep<3> {
  static constexpr int kTileBytes = 4 * 272;
  uint32_t             s;
  uint32_t             q[4];  // row pair v: two bytes of column 2 i, two of column 2 i + 1
};

template <int KIND>
__device__ __forceinline__ void load_step(RawStep<KIND> &r, const uint8_t *__restrict__ tile, int g, int i) {
  if constexpr (KIND == 1) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      r.q[v] = *reinterpret_cast<const uint2 *>(tile + (uint32_t) (4 * g * 128 + 8 * i) + 128 * v);
    }
  } else if constexpr (KIND == 3) {
    r.s = *reinterpret_cast<const uint32_t *>(tile + (uint32_t) (g * 272 + 4 * (i & 3)));
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      r.q[v] = *reinterpret_cast<const uint32_t *>(tile + (uint32_t) (g * 272 + 4 * i) + 16 + 64 * v);
    }
  } else {
    r.s = *reinterpret_cast<const uint32_t *>(tile + (uint32_t) (g * 144 + 4 * (i & 3)));
    r.q = *reinterpret_cast<const uint2 *>(tile + (uint32_t) (g * 144 + 8 * i) + 16);
  }
}

__device__ __forceinline__ v2h as_v2h(uint32_t x) {
  return __builtin_bit_cast(v2h, x);
}
// The four scales of a lane's columns, each in both halves of a dword, out of the dwords that the lanes of its quad loaded (one
// load of 16 bytes per lane would ask for the same bytes sixteen times: 16 turns of the path into the CU instead of 4)
__device__ __forceinline__ void scales_of_quad(uint32_t own, uint32_t half_sel, v2h (&sc)[4]) {
  // (half_sel is the same throughout a quad)
  const int x = (int) __builtin_amdgcn_perm(own, own, half_sel);
  sc[0] = as_v2h((uint32_t) __builtin_amdgcn_mov_dpp(x, 0x00, 0xf, 0xf, true));
  sc[1] = as_v2h((uint32_t) __builtin_amdgcn_mov_dpp(x, 0x55, 0xf, 0xf, true));
  sc[2] = as_v2h((uint32_t) __builtin_amdgcn_mov_dpp(x, 0xaa, 0xf, 0xf, true));
  sc[3] = as_v2h((uint32_t) __builtin_amdgcn_mov_dpp(x, 0xff, 0xf, 0xf, true));
}
// (a | b) of the masks below turns bytes into fp16 numbers 1024 + byte: 0x64xx
__device__ __forceinline__ v2h biased_to_half(uint32_t x, _Float16 bias) {
  return as_v2h(x) - (v2h){ bias, bias };  // exact: integers below 2048
}

// IQ4_NL code book (reference: src/dsp/ops/mat_mul.c:29-32), every value + 128: the four nibbles in the low halves of
// x's bytes -> four bytes. (The usual way to look 16 bytes up with byte permutes: one for either half of the book by the low three
// bits, one that picks by the fourth.)
__device__ __forceinline__ uint32_t iq4_nl_bytes(uint32_t x) {
  const uint32_t low3 = x & 0x07070707u;
  const uint32_t a    = __builtin_amdgcn_perm(0x766a5d4fu, 0x3f2d1801u, low3);  // values 0 .. 7
  const uint32_t b    = __builtin_amdgcn_perm(0xf1d9c5b5u, 0xa6998d81u, low3);  // values 8 .. 15
  return __builtin_amdgcn_perm(b, a, 0x03020100u + ((x & 0x08080808u) >> 1));
}

// The B operand of column 2 i + J: K rows 8 g + 2 v, + 1 in dword v. Each weight is fp16(quant) * fp16(scale) rounded
// once, as the reference's dequantizers make it (mat_mul.c:308-508). `sc` holds the four scales of the lane's columns,
// each in both halves of a dword.
struct VectorConstants {
  uint32_t exponents = 0x64006400u;  // (in a vector register, so that masking and merging are one instruction)
};
template <int KIND, int J>
__device__ __forceinline__ v8h dequant(const RawStep<KIND> &r, const v2h (&sc)[4], const VectorConstants &c) {
  v2h h[4];
  if constexpr (KIND == 1) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      h[v] = as_v2h(J ? r.q[v].y : r.q[v].x);
    }
  } else if constexpr (KIND == 2) {
    // byte b holds row pair b & 1 (low nibble) and 2 + (b & 1) (high nibble), row b / 2 of the pair
    const uint32_t q = J ? r.q.y : r.q.x;
    const uint32_t q8 = q >> 8;
    // low nibbles give 1024 + n, high ones 1024 + 16 n, which a fused multiply-add turns into n - 8 exactly as well
    const v2h lo_bias = { (_Float16) 1032.0f, (_Float16) 1032.0f }, sixteenth = { (_Float16) 0.0625f, (_Float16) 0.0625f },
              hi_bias = { (_Float16) -72.0f, (_Float16) -72.0f };
    h[0] = (as_v2h((q & 0x000f000fu) | c.exponents) - lo_bias) * sc[0];
    h[1] = (as_v2h((q8 & 0x000f000fu) | c.exponents) - lo_bias) * sc[1];
    h[2] = __builtin_elementwise_fma(as_v2h((q & 0x00f000f0u) | c.exponents), sixteenth, hi_bias) * sc[2];
    h[3] = __builtin_elementwise_fma(as_v2h((q8 & 0x00f000f0u) | c.exponents), sixteenth, hi_bias) * sc[3];
  } else if constexpr (KIND == 4) {
    const uint32_t q  = J ? r.q.y : r.q.x;
    const uint32_t lo = iq4_nl_bytes(q), hi = iq4_nl_bytes(q >> 4);  // (the masks inside drop the other nibbles)
    h[0] = biased_to_half(__builtin_amdgcn_perm(0x64646464u, lo, 0x04020400u), (_Float16) 1152.0f) * sc[0];
    h[1] = biased_to_half(__builtin_amdgcn_perm(0x64646464u, lo, 0x04030401u), (_Float16) 1152.0f) * sc[1];
    h[2] = biased_to_half(__builtin_amdgcn_perm(0x64646464u, hi, 0x04020400u), (_Float16) 1152.0f) * sc[2];
    h[3] = biased_to_half(__builtin_amdgcn_perm(0x64646464u, hi, 0x04030401u), (_Float16) 1152.0f) * sc[3];
  } else {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const uint32_t u = r.q[v] ^ 0x80808080u;
      h[v] = biased_to_half(__builtin_amdgcn_perm(0x64646464u, u, J ? 0x04030402u : 0x04010400u), (_Float16) 1152.0f) * sc[v];
    }
  }
  return __builtin_shufflevector(__builtin_shufflevector(h[0], h[1], 0, 1, 2, 3), __builtin_shufflevector(h[2], h[3], 0, 1, 2, 3),
                                 0, 1, 2, 3, 4, 5, 6, 7);
}

// MT row tiles of 16; NT column groups of 32 per workgroup (sharing the activations); ACT_LDS: the activations are
// converted into LDS by every workgroup
template <int KIND, int MT, int NT, bool ACT_LDS>
__global__ __launch_bounds__(kRowsThreads) void permuted_rows_kernel(const RowsArgs args) {
  extern __shared__ __align__(16) uint8_t rows_lds[];  // activations [m][k + 8] halfs, then the waves' sums
  int idx = 0;
  while (idx + 1 < args.count && (int) blockIdx.x >= args.member[idx + 1].first) {
    ++idx;
  }
  const RowsMember &mb  = args.member[idx];
  const int   m = args.m, k = mb.k, n = mb.n;
  const int   lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int   g = lane >> 4, i = lane & 15;
  const int   nt0 = ((int) blockIdx.x - mb.first) * NT, n_tiles = n / 32, k_tiles = k / 32;
  // Steps of a wave in flight. Eight of Q8_0 cost a workgroup per CU (hidden 2048, ffn 5632: one row 13.1 against 12.0 us, 20
  // rows 20.0 / 16.3); 16 rows in operand order, which travel with the weights, gain (IQ4_NL, 2048, 8960: 17.8 against 20.5).
  constexpr int DEPTH = KIND == 1 || ((KIND == 2 || KIND == 4) && MT == 1 && !ACT_LDS) ? 8 : 4;
  const uint8_t *w[NT];
#pragma unroll
  for (int c = 0; c < NT; ++c) {
    w[c] = mb.weight + (size_t) min(nt0 + c, n_tiles - 1) * k_tiles * RawStep<KIND>::kTileBytes;
  }

  // the first rows' values are requested before the weights, so that waiting for them leaves the weights in flight
  constexpr int kAhead = 6;
  float4        pre[kAhead];
  const int     quads = m * (k / 4);
  if constexpr (ACT_LDS) {
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      pre[u] = reinterpret_cast<const float4 *>(mb.act)[min((int) threadIdx.x + u * kRowsThreads, quads - 1)];
    }
    asm volatile("" ::: "memory");
  }
  RawStep<KIND> raw[DEPTH][NT];
  uint4         af[DEPTH][MT];
  auto          load = [&](int d, int step) {
    const int kt = min(wave + step * kRowsWaves, k_tiles - 1);  // (branch-free: steps past the end repeat the last tile)
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      load_step(raw[d][c], w[c] + (size_t) kt * RawStep<KIND>::kTileBytes, g, i);
    }
    if constexpr (!ACT_LDS) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        af[d][t] = mb.frag[((size_t) t * k_tiles + kt) * kWave + lane];
      }
    }
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    load(d, d);
  }
  const int pitch = k + 8;  // halfs
  if constexpr (ACT_LDS) {
    _Float16 *act = reinterpret_cast<_Float16 *>(rows_lds);
    auto      put = [&](int q, const float4 &x) {
      const int row = q / (k / 4), c = q - row * (k / 4);
      *reinterpret_cast<v4h *>(act + (size_t) row * pitch + 4 * c) =
        (v4h){ (_Float16) x.x, (_Float16) x.y, (_Float16) x.z, (_Float16) x.w };
    };
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      const int q = (int) threadIdx.x + u * kRowsThreads;
      if (q < quads) {
        put(q, pre[u]);
      }
    }
    for (int q = (int) threadIdx.x + kAhead * kRowsThreads; q < quads; q += kRowsThreads) {
      put(q, reinterpret_cast<const float4 *>(mb.act)[q]);
    }
    // (not __syncthreads: its fence would wait for the weights as well)
    asm volatile("s_waitcnt lgkmcnt(0)\n s_barrier" ::: "memory");
  }

  v4f acc[MT][NT][2];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int c = 0; c < NT; ++c) {
      acc[t][c][0] = acc[t][c][1] = (v4f){ 0.0f, 0.0f, 0.0f, 0.0f };
    }
  }
  const uint32_t half_sel = (i >> 3) ? 0x03020302u : 0x01000100u;  // columns 16 .. 31 take the odd scales
  const uint8_t *a_lds[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    // (rows past the last one repeat it: a result row depends on its own row only, and theirs are not stored)
    a_lds[t] = rows_lds + ((size_t) min(16 * t + i, m - 1) * pitch + 8 * g) * 2;
  }
  VectorConstants vc;
  asm("" : "+v"(vc.exponents));
  auto use = [&](int d, int step) {
    const int kt = wave + step * kRowsWaves;
    if (kt < k_tiles) {
      v8h a[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        if constexpr (ACT_LDS) {
          a[t] = *reinterpret_cast<const v8h *>(a_lds[t] + (size_t) kt * 64);
        } else {
          a[t] = __builtin_bit_cast(v8h, af[d][t]);
        }
      }
#pragma unroll
      for (int c = 0; c < NT; ++c) {
        v2h sc[4];
        if constexpr (KIND != 1) {
          scales_of_quad(raw[d][c].s, half_sel, sc);
        }
        const v8h b0 = dequant<KIND, 0>(raw[d][c], sc, vc), b1 = dequant<KIND, 1>(raw[d][c], sc, vc);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          acc[t][c][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], b0, acc[t][c][0], 0, 0, 0);
          acc[t][c][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], b1, acc[t][c][1], 0, 0, 0);
        }
      }
    }
  };
  const int steps = (k_tiles + kRowsWaves - 1) / kRowsWaves;
  int       s0    = 0;
  for (; s0 + DEPTH < steps; s0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      use(d, s0 + d);
      load(d, s0 + d + DEPTH);
    }
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    use(d, s0 + d);
  }

  // the waves' sums: D[4 g + r][i] of tile (t, c, j) is row 16 t + 4 g + r, column 2 i + j of column group c
  __syncthreads();  // (everybody is done with the activations)
  float    *red  = reinterpret_cast<float *>(rows_lds);  // [wave][row][32 NT]
  const int rows = min(m, 16 * MT);
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * t + 4 * g + r;
      if (row < rows) {
#pragma unroll
        for (int c = 0; c < NT; ++c) {
          *reinterpret_cast<float2 *>(red + ((size_t) wave * rows + row) * (32 * NT) + 32 * c + 2 * i) =
            make_float2(acc[t][c][0][r], acc[t][c][1][r]);
        }
      }
    }
  }
  __syncthreads();
  for (int o = threadIdx.x; o < rows * 32 * NT; o += kRowsThreads) {
    float sum = 0.0f;
#pragma unroll
    for (int u = 0; u < kRowsWaves; ++u) {
      sum += red[(size_t) u * rows * (32 * NT) + o];
    }
    const int col = nt0 * 32 + o % (32 * NT);
    if (NT == 1 || col < n) {
      mb.out[(size_t) (o / (32 * NT)) * n + col] = (float) (_Float16) sum;  // the reference stores fp16 results
    }
  }
}

// fp32 rows -> fp16 in A operand order: [row tile of 16][K step of 32][lane], lane (g, i) = row i, K 8 g .. 8 g + 7;
// rows past the last one are zeros
struct RowsActArgs {
  const float *src[kPermutedGroupMax];
  uint4       *dst[kPermutedGroupMax];
  int          k[kPermutedGroupMax], first[kPermutedGroupMax];
  int          count, m, tiles;
};
__global__ __launch_bounds__(256) void permuted_rows_act_kernel(const RowsActArgs args) {
  int idx = 0;
  while (idx + 1 < args.count && (int) blockIdx.x >= args.first[idx + 1]) {
    ++idx;
  }
  const int k = args.k[idx], k_tiles = k / 32;
  const unsigned t = (blockIdx.x - (unsigned) args.first[idx]) * 256u + threadIdx.x, f = t >> 6;  // (a grid is less than 2^32 threads)
  const int lane = t & 63, step = (int) (f % (unsigned) k_tiles), tile = (int) (f / (unsigned) k_tiles);
  if (tile >= args.tiles) {
    return;
  }
  const int row = 16 * tile + (lane & 15);
  uint4     o   = make_uint4(0, 0, 0, 0);
  if (row < args.m) {
    const float4 *s = reinterpret_cast<const float4 *>(args.src[idx] + (size_t) row * k + 32 * step + 8 * (lane >> 4));
    const float4  a = s[0], b = s[1];
    const v8h     h = { (_Float16) a.x, (_Float16) a.y, (_Float16) a.z, (_Float16) a.w,
                        (_Float16) b.x, (_Float16) b.y, (_Float16) b.z, (_Float16) b.w };
    o = __builtin_bit_cast(uint4, h);
  }
  args.dst[idx][t] = o;
}

// ---- more than 32 rows ----------------------------------------------------------------------------------------------
// The same weights, turned to fp16 in registers by every wave that multiplies with them; what has to be saved here is the path
// from L2 into a CU (with both operands as fp16 in memory it was the limit: 16 KiB per K step of 16 and workgroup of
// 128 x 128 outputs at 30 bytes a nanosecond). A workgroup owns R row tiles of 16 x 4 column groups of 32; its four waves
// are two column halves times two halves of K, added through LDS at the end. A wave holds R x 64 outputs: the two column
// groups' weights come straight into registers, kDepth K steps of 32 ahead (4-bit formats: 1.1 KiB a step), each turned to
// fp16 once for R matrix instructions per operand; the rows, fp16 in operand order, come into LDS by DMA in a ring of four
// slots, three steps ahead, and are read as they are used. One barrier a step; two workgroups on a CU fill each
// other's gaps. The matmuls of a message that nothing orders share a launch, longest walk first; a long K is dealt to
// several workgroups (gemm_parts).
// Seven projections, 300 rows (hidden 2048, ffn 5632, IQ4_NL), weights not in a cache: 50.8 us (605 TFLOP/s), 76.2 before long
// K was split and row tiles were chosen by the walks, 94.7 with fp16 copies of the weights staged through LDS like the rows
// and 264.8 with a launch per matrix over such copies. Of it, 25 are the rows' conversion, the launches and the ends
// of the walks, 15 the matrix instructions (timing-only builds; they add up, two waves a SIMD cover little of each
// other). Workgroups of eight waves over twice the columns, which halve the rows' traffic: 55.2.
struct GemmMember {
  float         *out;
  const uint8_t *frag, *weight;
  int            n_tiles, k_tiles, col_begin;  // col_begin: in units of 4 column groups and one part of K
  int            parts;                        // workgroups that share a tile's K; their sums meet in `exchange`:
  uint64_t      *exchange;                     // [row tile][column group][part][4][lane] pairs of neighbouring columns
  unsigned      *tickets;                      // zeroed counters, one per wave of a tile, left zeroed
};
struct GemmArgs {
  GemmMember member[kPermutedGroupMax];
  int        count, cols, m, row_tiles, row_blocks;
};

template <int KIND>
struct RawLoads {  // load instructions of a step and column group
  static constexpr int kCount = KIND == 1 ? 4 : KIND == 3 ? 5 : 2;
};

// load_step through a buffer resource: one instruction per field, whatever surrounds it (they are counted below)
template <int KIND>
__device__ __forceinline__ void load_step_counted(RawStep<KIND> &r, __amdgpu_buffer_rsrc_t tiles, int at, int g, int i) {
  if constexpr (KIND == 1) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      r.q[v] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(tiles, 4 * g * 128 + 8 * i + 128 * v, at, 0));
    }
  } else if constexpr (KIND == 3) {
    r.s = __builtin_amdgcn_raw_buffer_load_b32(tiles, g * 272 + 4 * (i & 3), at, 0);
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      r.q[v] = __builtin_amdgcn_raw_buffer_load_b32(tiles, g * 272 + 4 * i + 16 + 64 * v, at, 0);
    }
  } else {
    r.s = __builtin_amdgcn_raw_buffer_load_b32(tiles, g * 144 + 4 * (i & 3), at, 0);
    r.q = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(tiles, g * 144 + 8 * i + 16, at, 0));
  }
}

__device__ __forceinline__ int part_begin(int part, int k_tiles, int parts) {
  return (int) ((unsigned) part * (unsigned) k_tiles / (unsigned) parts);
}

template <int KIND, int R>
__global__ __launch_bounds__(256, 2) void permuted_gemm_kernel(const GemmArgs args) {
  constexpr int RING = 4, kDepth = 4;
  constexpr int APART = (R + 1) / 2;                      // row pieces of 1 KiB that a wave brings per step (an odd one is brought twice)
  constexpr int BLOADS = 2 * RawLoads<KIND>::kCount;      // weight loads of a wave per step
  __shared__ __align__(1024) uint8_t lds[RING][2 * R * 1024];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kh = wave >> 1, wn = wave & 1;
  const int g = lane >> 4, i = lane & 15;
  // Workgroup ids go round the 8 XCDs: the row blocks of a column block follow each other on one XCD, so its weights come
  // from that L2 for all but the first, and the column blocks (longest K first) are dealt out evenly.
  const int turn = (int) blockIdx.x >> 3;
  const int col  = turn / args.row_blocks * 8 + ((int) blockIdx.x & 7), rb = turn % args.row_blocks;
  if (col >= args.cols) {
    return;
  }
  int id = 0;
  while (id + 1 < args.count && col >= args.member[id + 1].col_begin) {
    ++id;
  }
  const GemmMember &mb = args.member[id];
  const int n_tiles = mb.n_tiles, k_tiles = mb.k_tiles, parts = mb.parts;
  const int col_blocks = (n_tiles + 3) / 4, part = (col - mb.col_begin) / col_blocks, cb = (col - mb.col_begin) % col_blocks;
  const int mt0 = rb * R, nt0 = cb * 4 + 2 * wn;
  // this wave's half of the workgroup's part of K: steps kt0 .. kt0 + mine - 1 (both halves run `steps` turns)
  const int kt_begin = part_begin(part, k_tiles, parts), whole = part_begin(part + 1, k_tiles, parts) - kt_begin;
  const int steps = (whole + 1) / 2;
  const int kt0 = kt_begin + kh * steps, mine = kh == 0 ? steps : whole - steps;
  auto      step_at = [&](int s) { return min(kt0 + s, k_tiles - 1); };  // (past the end: the last step again)

  __amdgpu_buffer_rsrc_t tiles[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint8_t *base = mb.weight + (size_t) min(nt0 + c, n_tiles - 1) * k_tiles * RawStep<KIND>::kTileBytes;
    tiles[c] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0, (int) 0xffffffffu, 0x00020000);
  }
  RawStep<KIND> raw[kDepth][2];
  auto load = [&](int d, int s) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      load_step_counted<KIND>(raw[d][c], tiles[c], step_at(s) * RawStep<KIND>::kTileBytes, g, i);
    }
  };
  const uint8_t *src[APART];
  uint32_t       to[APART];
#pragma unroll
  for (int p = 0; p < APART; ++p) {
    const int t = min(2 * p + wn, R - 1);
    src[p] = mb.frag + (size_t) min(mt0 + t, args.row_tiles - 1) * k_tiles * 1024;
    to[p]  = (uint32_t) (uintptr_t) &lds[0][0] + (uint32_t) (kh * R + t) * 1024;
  }
  auto fetch = [&](int s) {
    const size_t   off  = (size_t) step_at(s) * 1024;
    const uint32_t slot = (uint32_t) (s & (RING - 1)) * (2 * R * 1024);
#pragma unroll
    for (int p = 0; p < APART; ++p) {
      asm volatile("s_mov_b32 m0, %2\n s_nop 0\n global_load_lds_dwordx4 %0, %1" ::"v"(lane * 16), "s"(src[p] + off), "s"(slot + to[p]) : "memory");
    }
  };

  v4f acc[R][2][2];
#pragma unroll
  for (int t = 0; t < R; ++t) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      acc[t][c][0] = acc[t][c][1] = (v4f){ 0.0f, 0.0f, 0.0f, 0.0f };
    }
  }
  const uint32_t  half_sel = (i >> 3) ? 0x03020302u : 0x01000100u;  // columns 16 .. 31 take the odd scales
  VectorConstants vc;
  asm("" : "+v"(vc.exponents));

  // Requests in order: weights of step 0, then rows of step s and weights of step s + 1 in turn; from turn s on, rows of step
  // s + 3 and weights of step s + kDepth.
#pragma unroll
  for (int s = 0; s < kDepth; ++s) {
    load(s, s);
    asm volatile("" ::: "memory");
    if (s < RING - 1) {
      fetch(s);
    }
  }
  for (int s0 = 0; s0 < steps; s0 += kDepth) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      const int s = s0 + d;
      if (s >= steps) {
        break;
      }
      // This wave's rows of step s have landed: behind them it has asked for the rows of two steps and the weights of three.
      // Behind the barrier everybody's have, and nobody reads the slot of step s - 1 any more.
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * APART + 3 * BLOADS) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      fetch(s + RING - 1);
      v8h b[2][2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        v2h sc[4];
        if constexpr (KIND != 1) {
          scales_of_quad(raw[d][c].s, half_sel, sc);
        }
        b[c][0] = dequant<KIND, 0>(raw[d][c], sc, vc), b[c][1] = dequant<KIND, 1>(raw[d][c], sc, vc);
      }
      load(d, s + kDepth);
      asm volatile("" ::: "memory");
      if (s < mine) {
        const uint8_t *rows = &lds[s & (RING - 1)][kh * R * 1024] + lane * 16;
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const v8h a = *reinterpret_cast<const v8h *>(rows + t * 1024);
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            acc[t][c][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[c][0], acc[t][c][0], 0, 0, 0);
            acc[t][c][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[c][1], acc[t][c][1], 0, 0, 0);
          }
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (rows past the end have landed before the ring is used again)

  // The halves of K hand each other the sums of every second row tile and finish the others;
  // D[4 g + r][i] of tile (t, c, j) is row 16 t + 4 g + r, column 2 i + j of group c
  // (one column group after the other: what the ring has room for)
  static_assert(2 * R * 2 * kWave * sizeof(v4f) <= sizeof(lds), "the sums of a column group fit");
  constexpr int OWN = (R + 1) / 2;
  v4f *xch = reinterpret_cast<v4f *>(&lds[0][0]) + (size_t) wn * R * 2 * kWave + lane;  // [row tile][2]
  v4f  sum[OWN][2][2];                                                                // of row tiles kh, kh + 2, ..
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    __syncthreads();
#pragma unroll
    for (int t = 0; t < R; ++t) {
      if ((t & 1) != kh) {
        xch[2 * t * kWave] = acc[t][c][0], xch[(2 * t + 1) * kWave] = acc[t][c][1];
      }
    }
    __syncthreads();
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const v4f own = kh == 0 ? acc[2 * o][c][j] : acc[min(2 * o + 1, R - 1)][c][j];  // (past the last one: never stored)
        sum[o][c][j]  = own + xch[(2 * min(2 * o + kh, R - 1) + j) * kWave];
      }
    }
  }
  auto exists = [&](int o, int c) { return 2 * o + kh < R && mt0 + 2 * o + kh < args.row_tiles && nt0 + c < n_tiles; };
  if (parts > 1) {
    // The parts of K meet in memory: every wave leaves its sums there and takes a ticket, and the wave that comes last adds all
    // parts in part order, its own included. (Device-scope stores, acknowledged before the ticket is taken, and device-scope
    // loads behind it: see shared_operand_workgroup in gemm_i8_fragments.hip.)
    auto place = [&](int o, int c, int p) {
      return mb.exchange + (((size_t) (mt0 + 2 * o + kh) * n_tiles + nt0 + c) * parts + p) * (4 * kWave) + lane;
    };
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if (exists(o, c)) {
          uint64_t *to_ = place(o, c, part);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            __hip_atomic_store(to_ + r * kWave, __builtin_bit_cast(uint64_t, make_float2(sum[o][c][0][r], sum[o][c][1][r])),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          }
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    unsigned *counter = mb.tickets + ((size_t) cb * args.row_blocks + rb) * 4 + wave, ticket = 0;
    if (lane == 0) {
      ticket = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    ticket = __builtin_amdgcn_readfirstlane(ticket);
    if (ticket != (unsigned) (parts - 1)) {
      return;
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (lane == 0) {
      __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
    }
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      sum[o][0][0] = sum[o][0][1] = sum[o][1][0] = sum[o][1][1] = (v4f){ 0.0f, 0.0f, 0.0f, 0.0f };
    }
    for (int p = 0; p < parts; p += 2) {  // two parts per trip to memory
      uint64_t x[2][OWN][2][4];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
#pragma unroll
          for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              x[u][o][c][r] = exists(o, c) && p + u < parts ? __hip_atomic_load(place(o, c, p + u) + r * kWave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
            }
          }
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
#pragma unroll
        for (int o = 0; o < OWN; ++o) {
#pragma unroll
          for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float2 f = __builtin_bit_cast(float2, x[u][o][c][r]);
              sum[o][c][0][r] += f.x, sum[o][c][1][r] += f.y;
            }
          }
        }
      }
    }
  }
  const int n = n_tiles * 32;
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (exists(o, c)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * (mt0 + 2 * o + kh) + 4 * g + r;
          if (row < args.m) {  // (the reference stores fp16 results)
            *reinterpret_cast<float2 *>(mb.out + (size_t) row * n + 32 * (nt0 + c) + 2 * i) =
              make_float2((float) (_Float16) sum[o][c][0][r], (float) (_Float16) sum[o][c][1][r]);
          }
        }
      }
    }
  }
}

__global__ __launch_bounds__(256) void copy_results_kernel(uint4 *__restrict__ dst, const uint4 *__restrict__ src, size_t count) {
  for (size_t i = (size_t) blockIdx.x * 256 + threadIdx.x; i < count; i += (size_t) gridDim.x * 256) {
    dst[i] = src[i];
  }
}

template <int KIND>
hipError_t launch_gemm_kind(hipStream_t stream, const GemmArgs &args, unsigned grid, int r) {
  void (*kernel)(GemmArgs) = nullptr;
  switch (r) {
    case 2: kernel = permuted_gemm_kernel<KIND, 2>; break;
    case 3: kernel = permuted_gemm_kernel<KIND, 3>; break;
    case 4: kernel = permuted_gemm_kernel<KIND, 4>; break;
    case 5: kernel = permuted_gemm_kernel<KIND, 5>; break;
    case 6: kernel = permuted_gemm_kernel<KIND, 6>; break;
    case 7: kernel = permuted_gemm_kernel<KIND, 7>; break;
    case 8: kernel = permuted_gemm_kernel<KIND, 8>; break;
    case 9: kernel = permuted_gemm_kernel<KIND, 9>; break;
    case 10:
      if constexpr (KIND != 1) {  // (ten row tiles and four steps of fp16 weights do not fit the registers)
        kernel = permuted_gemm_kernel<KIND, 10>;
      }
      break;
  }
  if (!kernel) {
    return hipErrorInvalidValue;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, stream, args);
  return hipGetLastError();
}

bool act_in_lds(int m, int k) {
  return (size_t) m * (k + 8) * 2 <= kRowsActLds;
}

template <int KIND>
hipError_t launch_kind(hipStream_t stream, const RowsArgs &args, unsigned grid, size_t lds, bool act_lds, bool wide) {
  void (*kernel)(RowsArgs) = nullptr;
  if (args.m <= 16) {
    kernel = act_lds ? permuted_rows_kernel<KIND, 1, 1, true> : permuted_rows_kernel<KIND, 1, 1, false>;
  } else {
    kernel = act_lds ? permuted_rows_kernel<KIND, 2, 1, true> : permuted_rows_kernel<KIND, 2, 1, false>;
    if constexpr (KIND == 2 || KIND == 4) {
      kernel = wide ? permuted_rows_kernel<KIND, 2, 2, false> : kernel;
    }
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(kRowsThreads), lds, stream, args);
  return hipGetLastError();
}

size_t act_bytes(int m, int k) {
  return (size_t) ((m + 15) / 16) * 16 * (size_t) k * 2;
}

// Workgroups that share a tile's K, from the matmul's own sizes: its sums do not depend on what else is in the launch. A long
// K beside short ones, as a down projection has it, would walk on alone when the others are done: pieces of about 22 steps
// (1408 of K). K up to 4096 stays whole where rows and columns give workgroups enough, and so does what fills the device
// anyway: the pieces' sums go through memory. Seven projections, whole / in pieces: 300 rows, hidden 2048, ffn 5632, IQ4_NL
// 70.9 / 52.8 us (pieces of 30 steps 61.6, of 16 53.4); 81 rows, 736, 6720, Q4_0 44.8 / 21.7; 128 rows, 4096, 8960, Q4_0 88.1
// / 74.5 (69.9 of 40 steps); 300 rows of those 138.1 / 138.5, and 147 with up to 512 workgroups instead of 192.
int gemm_parts(int m, int n, int k) {
  const int  steps = k / 64, row_tiles = (m + 15) / 16;
  const long alone = (long) ((n / 32 + 3) / 4) * ((row_tiles + 7) / 8);
  if (steps <= 64 && row_tiles > 4 && alone > 16) {
    return 1;
  }
  return (int) std::max<long>(1, std::min<long>({ 8, 192 / alone, steps / 22 }));
}

size_t exchange_bytes(int m, int n, int k) {
  const int parts = gemm_parts(m, n, k);
  return parts > 1 ? (size_t) ((m + 15) / 16) * 16 * (size_t) n * 4 * parts : 0;
}

}  // namespace

namespace {

// copies of the activations in operand order, one for the members that read the same rows
size_t operand_order_bytes(const PermutedMatMul *members, int count, int m) {
  size_t bytes = 0;
  for (int j = 0; j < count; ++j) {
    bool first = true;
    for (int i = 0; i < j; ++i) {
      first = first && !(members[i].act == members[j].act && members[i].k == members[j].k);
    }
    bytes += first ? act_bytes(m, members[j].k) : 0;
  }
  return bytes;
}

}  // namespace

size_t permuted_gemm_workspace_bytes(const PermutedMatMul *members, int count, int m) {
  size_t bytes = operand_order_bytes(members, count, m);
  for (int j = 0; j < count; ++j) {
    bytes += exchange_bytes(m, members[j].n, members[j].k);
  }
  return bytes;
}

size_t permuted_rows_workspace_bytes(const PermutedMatMul *members, int count, int m) {
  bool act_lds = true;
  for (int j = 0; j < count; ++j) {
    act_lds = act_lds && act_in_lds(m, members[j].k);
  }
  return act_lds ? 0 : operand_order_bytes(members, count, m);
}

hipError_t launch_permuted_rows_group(hipStream_t stream, const PermutedMatMul *members, int count, int m, int weight_kind,
                                      void *workspace) {
  if (count < 1 || count > kPermutedGroupMax || m < 1 || m > kPermutedRowsMax || weight_kind < 1 || weight_kind > 4) {
    return hipErrorInvalidValue;
  }
  // the members with the longest columns first (a workgroup walks a column group's whole K), so that the launch does
  // not end with them
  int order[kPermutedGroupMax];
  for (int j = 0; j < count; ++j) {
    order[j] = j;
  }
  std::stable_sort(order, order + count, [&](int a, int b) { return members[a].k > members[b].k; });
  bool act_lds = true;
  int  k_max   = 0;
  for (int j = 0; j < count; ++j) {
    if (members[j].k % 32 != 0 || members[j].n % 32 != 0 || members[j].k <= 0 || members[j].n <= 0) {
      return hipErrorInvalidValue;
    }
    act_lds = act_lds && act_in_lds(m, members[j].k);
    k_max   = std::max(k_max, members[j].k);
  }
  // Activations in operand order come from L2, once per workgroup: with 17 .. 32 rows (2 KiB per step, against 576 B of
  // 4-bit weights) and column groups enough, a workgroup takes two and halves that traffic (Llama-7B shapes, 32 rows of
  // Q4_0: 48 -> 45 us). With up to 16 rows it changes nothing (39.0 against 38.4 us), and the wider formats lose
  // (16 rows of fp16 tiles: 34.8 against 24.7 us).
  int groups = 0;
  for (int j = 0; j < count; ++j) {
    groups += members[j].n / 32;
  }
  const bool wide = !act_lds && m > 16 && (weight_kind == 2 || weight_kind == 4) && groups >= kRowsWideTiles;
  RowsArgs   args;
  args.count = count, args.m = m;
  unsigned     grid = 0;
  RowsActArgs  conv;
  unsigned     conv_grid = 0;
  conv.count = 0, conv.m = m, conv.tiles = (m + 15) / 16;
  uint8_t *ws = static_cast<uint8_t *>(workspace);
  for (int j = 0; j < count; ++j) {
    const PermutedMatMul &p = members[order[j]];
    RowsMember           &a = args.member[j];
    a.out = p.out, a.act = p.act, a.frag = nullptr, a.weight = static_cast<const uint8_t *>(p.weight), a.k = p.k, a.n = p.n;
    a.first = (int) grid;
    grid += (unsigned) (wide ? (p.n / 32 + 1) / 2 : p.n / 32);
    if (!act_lds) {
      int c = 0;
      while (c < conv.count && !(conv.src[c] == p.act && conv.k[c] == p.k)) {
        ++c;
      }
      if (c == conv.count) {
        conv.src[c] = p.act, conv.k[c] = p.k, conv.dst[c] = reinterpret_cast<uint4 *>(ws), conv.first[c] = (int) conv_grid;
        ws += act_bytes(m, p.k);
        conv_grid += (unsigned) ((act_bytes(m, p.k) / 16 + 255) / 256);
        ++conv.count;
      }
      a.frag = conv.dst[c];
    }
  }
  if (!act_lds) {
    hipLaunchKernelGGL(permuted_rows_act_kernel, dim3(conv_grid), dim3(256), 0, stream, conv);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) {
      return e;
    }
  }
  const size_t red = (size_t) kRowsWaves * m * 32 * (wide ? 2 : 1) * sizeof(float);
  const size_t lds = std::max(red, act_lds ? (size_t) m * (k_max + 8) * 2 : 0);
  switch (weight_kind) {
    case 1:
      return launch_kind<1>(stream, args, grid, lds, act_lds, wide);
    case 2:
      return launch_kind<2>(stream, args, grid, lds, act_lds, wide);
    case 3:
      return launch_kind<3>(stream, args, grid, lds, act_lds, wide);
    default:
      return launch_kind<4>(stream, args, grid, lds, act_lds, wide);
  }
}

hipError_t launch_permuted_gemm_group(hipStream_t stream, const PermutedMatMul *members, int count, int m, int weight_kind,
                                      void *workspace, unsigned *tickets) {
  if (count < 1 || count > kPermutedGroupMax || m < 1 || weight_kind < 1 || weight_kind > 4) {
    return hipErrorInvalidValue;
  }
  int order[kPermutedGroupMax], parts[kPermutedGroupMax];
  const size_t tile_bytes = weight_kind == 1 ? 2048 : weight_kind == 3 ? 4 * 272 : 4 * 144;
  for (int j = 0; j < count; ++j) {
    if (members[j].k % 32 != 0 || members[j].n % 32 != 0 || members[j].k <= 0 || members[j].n <= 0) {
      return hipErrorInvalidValue;
    }
    if ((size_t) (members[j].k / 32) * tile_bytes > 0x7fffffffu) {
      return hipErrorNotSupported;  // (the kernel's offsets within a column group are 32 bits)
    }
    order[j] = j, parts[j] = gemm_parts(m, members[j].n, members[j].k);
  }
  // the longest walks first
  std::stable_sort(order, order + count, [&](int a, int b) { return members[a].k / parts[a] > members[b].k / parts[b]; });
  GemmArgs    args = {};
  RowsActArgs conv = {};
  unsigned    conv_grid = 0;
  uint8_t    *ws = static_cast<uint8_t *>(workspace);
  args.count = count, args.m = m, args.row_tiles = conv.tiles = (m + 15) / 16, conv.m = m;
  for (int j = 0; j < count; ++j) {
    const PermutedMatMul &p = members[order[j]];
    int                   c = 0;
    while (c < conv.count && !(conv.src[c] == p.act && conv.k[c] == p.k)) {
      ++c;
    }
    if (c == conv.count) {
      conv.src[c] = p.act, conv.k[c] = p.k, conv.dst[c] = reinterpret_cast<uint4 *>(ws), conv.first[c] = (int) conv_grid;
      ws += act_bytes(m, p.k);
      conv_grid += (unsigned) ((act_bytes(m, p.k) / 16 + 255) / 256);
      ++conv.count;
    }
    args.member[j] = { p.out, reinterpret_cast<const uint8_t *>(conv.dst[c]), static_cast<const uint8_t *>(p.weight), p.n / 32,
                       p.k / 32, 0, parts[order[j]], nullptr, nullptr };
  }
  hipLaunchKernelGGL(permuted_rows_act_kernel, dim3(conv_grid), dim3(256), 0, stream, conv);
  if (hipError_t e = hipGetLastError(); e != hipSuccess) {
    return e;
  }
  for (int j = 0; j < count; ++j) {
    args.member[j].col_begin = args.cols;
    args.cols += (args.member[j].n_tiles + 3) / 4 * args.member[j].parts;
  }
  // Row tiles per workgroup: many save the path into the CU, few give work for all CUs. A walk takes about steps x (2 + row
  // tiles) whatever shares the CU with it (0.9 of that alone on it); the launch takes as long as the longest, or 1.8 times an
  // even share for each of 512 workgroups (512 is what the device holds). Among about equals the larger tile. Over 32 mixes of
  // seven projections (33 to 300 rows, hidden 512 to 4096) the choice is 1.3 % from the best tile in the mean, 14 % at worst.
  // 300 rows, hidden 2048, ffn 5632, IQ4_NL: ten tiles 52.1 us, seven 67.2, five 64.2; 150 rows, 768, 2048: two 20.7, ten 35.5.
  const int most = weight_kind == 1 ? 9 : 10;
  int       r    = most;
  double    best = 0.0;
  for (int t = most; t >= 2; --t) {
    const int blocks = (args.row_tiles + t - 1) / t, each = std::max(2, (args.row_tiles + blocks - 1) / blocks);
    double    share = 0.0, longest = 0.0;
    for (int j = 0; j < count; ++j) {
      const GemmMember &mb   = args.member[j];
      const double      walk = ((mb.k_tiles + mb.parts - 1) / mb.parts) * (2 + each);
      share += walk * ((mb.n_tiles + 3) / 4) * mb.parts * blocks / 512, longest = std::max(longest, walk);
    }
    const double time = std::max(1.8 * share, (long) args.cols * blocks <= 256 ? 0.9 * longest : longest);
    if (t == most || time < 0.95 * best) {
      r = t, best = time;
    }
  }
  args.row_blocks = (args.row_tiles + r - 1) / r;
  r = std::max(2, (args.row_tiles + args.row_blocks - 1) / args.row_blocks);
  for (int j = 0; j < count; ++j) {
    GemmMember &mb = args.member[j];
    if (mb.parts > 1) {
      mb.exchange = reinterpret_cast<uint64_t *>(ws), mb.tickets = tickets;
      ws += exchange_bytes(m, mb.n_tiles * 32, mb.k_tiles * 32);
      tickets += (size_t) ((mb.n_tiles + 3) / 4) * args.row_blocks * 4;  // (at most 96 x 4 x 4 a member: a split one has few tiles)
    }
  }
  const long long grid = (long long) ((args.cols + 7) / 8) * 8 * args.row_blocks;
  if (grid > 0x7fffffffLL) {
    return hipErrorInvalidValue;
  }
  switch (weight_kind) {
    case 1:
      return launch_gemm_kind<1>(stream, args, (unsigned) grid, r);
    case 2:
      return launch_gemm_kind<2>(stream, args, (unsigned) grid, r);
    case 3:
      return launch_gemm_kind<3>(stream, args, (unsigned) grid, r);
    default:
      return launch_gemm_kind<4>(stream, args, (unsigned) grid, r);
  }
}

hipError_t launch_copy_results(hipStream_t stream, float *dst, const float *src, size_t bytes) {
  const size_t count = bytes / 16;
  hipLaunchKernelGGL(copy_results_kernel, dim3((unsigned) std::min<size_t>((count + 255) / 256, 4096)), dim3(256), 0, stream,
                     reinterpret_cast<uint4 *>(dst), reinterpret_cast<const uint4 *>(src), count);
  return hipGetLastError();
}

}  // namespace htpops
