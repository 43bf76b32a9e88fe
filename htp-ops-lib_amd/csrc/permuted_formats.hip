// The reference's native weight formats (its ops 1-4) on gfx950.
//
// The Hexagon backend keeps weights in the order its matrix unit consumes: fp16 in 32x32 tiles
// (hmx_mat_mul_permuted_w16a32, reference: src/dsp/ops/mat_mul.c:758-855, layout src/host/test.c:300-312) or
// quantized "super-blocks" of 8 K rows x 32 N columns with one fp16 scale per 2 x 16 patch
// (hmx_mat_mul_permuted_qk_0_d16a32, mat_mul.c:875-1153; dequantizers :308-508). Both paths multiply fp16
// activations by fp16 weights and round the result to fp16.
//
// Here a weight buffer is converted ONCE (weights are immutable for the reference too, op_executor.cc:130) into the
// order the gfx950 matrix core consumes, and cached by the caller: for every 32-column tile and every 16-wide K step
// the 64 lanes' 16-byte B operands of v_mfma_f32_32x32x16_f16 lie in one contiguous KiB ("fragment order"), so the
// matmul kernel needs neither LDS nor any shuffling: both operands are loaded straight into MFMA registers.
//   lane (c = lane % 32, h = lane / 32) of fragment (tile, step) holds W[16 step + 8 h .. + 7][32 tile + c].
// Activations are converted per call (fp32 -> fp16, round to nearest even) into the same order with rows on lanes.
#include "device_utils.h"
#include "kernels.h"

namespace htpops {

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float    v16f __attribute__((ext_vector_type(16)));

// IQ4_NL code book (reference: src/dsp/ops/mat_mul.c:29-32)
__constant__ int8_t kIq4nlDev[16] = { -127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113 };

// one thread = one 16-byte fragment piece: 8 consecutive K of one column
struct PieceCoord {
  int  tile_n, step, c, h;  // fragment coordinates
  int  k_tile, kb;          // 32x32 source tile along K, first K row inside it (0, 8, 16, 24)
  bool ok;
};

__device__ __forceinline__ PieceCoord piece_coord(size_t t, int k_steps, int n_tiles) {
  PieceCoord p;
  const int lane = (int) (t & 63);
  const size_t f = t >> 6;
  p.step   = (int) (f % (size_t) k_steps);
  p.tile_n = (int) (f / (size_t) k_steps);
  p.c = lane & 31, p.h = lane >> 5;
  const int k0 = 16 * p.step + 8 * p.h;
  p.k_tile = k0 >> 5, p.kb = k0 & 31;
  p.ok = p.tile_n < n_tiles;
  return p;
}

// fp16 tiles: element (k1, n1) of a tile sits at (k1 & ~1) * 32 + n1 * 2 + (k1 & 1)
__global__ __launch_bounds__(256) void repack_w16_tiles_kernel(uint4 *__restrict__ dst, const uint32_t *__restrict__ src,
                                                               int k_steps, int n_tiles) {
  const size_t     t = (size_t) blockIdx.x * 256 + threadIdx.x;
  const PieceCoord p = piece_coord(t, k_steps, n_tiles);
  if (!p.ok) {
    return;
  }
  const size_t tile = (size_t) p.tile_n * (k_steps / 2) + p.k_tile;
  const uint32_t *s = src + tile * 512 + (size_t) (p.kb * 32 + p.c * 2) / 2;  // dword = one K pair of column c
  dst[t] = make_uint4(s[0], s[32], s[64], s[96]);                             // row pairs are 64 halfs apart
}

__device__ __forceinline__ uint32_t pack_halfs(float a, float b) {
  // fp16(q) * fp16(scale) is exact in fp32 (|q| <= 127, 11-bit significand); one rounding to fp16
  const _Float16 x = (_Float16) a, y = (_Float16) b;
  return (uint32_t) __builtin_bit_cast(uint16_t, x) | ((uint32_t) __builtin_bit_cast(uint16_t, y) << 16);
}

// Q4_0 / IQ4_NL super-blocks (144 B: 8 scales, 128 quant bytes). The 8 K rows of a piece are the four vectors of
// ONE super-block at elements 2c and 2c + 1: vector v takes the low (v < 2) or high nibble of bytes 4c + (v & 1)
// and 4c + 2 + (v & 1), scale 2v + c / 16 (reference: mat_mul.c:319-325, :383-405).
template <bool IQ4_NL>
__global__ __launch_bounds__(256) void dequant_permuted_q4_kernel(uint4 *__restrict__ dst, const uint8_t *__restrict__ src,
                                                                  int k_steps, int n_tiles) {
  const size_t     t = (size_t) blockIdx.x * 256 + threadIdx.x;
  const PieceCoord p = piece_coord(t, k_steps, n_tiles);
  if (!p.ok) {
    return;
  }
  const size_t    tile = (size_t) p.tile_n * (k_steps / 2) + p.k_tile;
  const uint8_t  *sb   = src + (tile * 4 + (size_t) (p.kb >> 3)) * 144;
  const uint16_t *sc   = reinterpret_cast<const uint16_t *>(sb);
  const uint8_t  *qs   = sb + 16 + 4 * p.c;
  uint32_t        out[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float d  = half_bits_to_float(sc[2 * v + (p.c >> 4)]);
    const int   b0 = qs[v & 1], b1 = qs[2 + (v & 1)];
    const int   n0 = (v & 2) ? (b0 >> 4) : (b0 & 15), n1 = (v & 2) ? (b1 >> 4) : (b1 & 15);
    const int   q0 = IQ4_NL ? (int) kIq4nlDev[n0] : n0 - 8, q1 = IQ4_NL ? (int) kIq4nlDev[n1] : n1 - 8;
    out[v]         = pack_halfs((float) q0 * d, (float) q1 * d);
  }
  dst[t] = make_uint4(out[0], out[1], out[2], out[3]);
}

// Q8_0 super-blocks (272 B: 8 scales, 256 int8): vector v = quants[64 v .. 64 v + 63] (mat_mul.c:483-505)
__global__ __launch_bounds__(256) void dequant_permuted_q8_kernel(uint4 *__restrict__ dst, const uint8_t *__restrict__ src,
                                                                  int k_steps, int n_tiles) {
  const size_t     t = (size_t) blockIdx.x * 256 + threadIdx.x;
  const PieceCoord p = piece_coord(t, k_steps, n_tiles);
  if (!p.ok) {
    return;
  }
  const size_t    tile = (size_t) p.tile_n * (k_steps / 2) + p.k_tile;
  const uint8_t  *sb   = src + (tile * 4 + (size_t) (p.kb >> 3)) * 272;
  const uint16_t *sc   = reinterpret_cast<const uint16_t *>(sb);
  const int8_t   *qs   = reinterpret_cast<const int8_t *>(sb + 16) + 2 * p.c;
  uint32_t        out[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float d = half_bits_to_float(sc[2 * v + (p.c >> 4)]);
    out[v]        = pack_halfs((float) qs[64 * v] * d, (float) qs[64 * v + 1] * d);
  }
  dst[t] = make_uint4(out[0], out[1], out[2], out[3]);
}

// activations fp32 [m][k] -> fragment order with rows on lanes; rows >= m are zero. One grid row per activation matrix.
struct ActMembers {
  const float *src[kPermutedGroupMax];
  uint4       *dst[kPermutedGroupMax];
  int          k[kPermutedGroupMax];
};

__global__ __launch_bounds__(256) void act_to_fragments_kernel(ActMembers members, int m, int m_tiles) {
  const size_t t = (size_t) blockIdx.x * 256 + threadIdx.x;
  const int    k = members.k[blockIdx.y], k_steps = k / 16;
  const int    lane = (int) (t & 63);
  const size_t f    = t >> 6;
  const int    step = (int) (f % (size_t) k_steps), tile = (int) (f / (size_t) k_steps);
  if (tile >= m_tiles) {
    return;
  }
  const int row = tile * 32 + (lane & 31);
  uint4     o   = make_uint4(0, 0, 0, 0);
  if (row < m) {
    const float4 *s = reinterpret_cast<const float4 *>(members.src[blockIdx.y] + (size_t) row * k + 16 * step + 8 * (lane >> 5));
    const float4  a = s[0], b = s[1];
    o = make_uint4(pack_halfs(a.x, a.y), pack_halfs(a.z, a.w), pack_halfs(b.x, b.y), pack_halfs(b.z, b.w));
  }
  members.dst[blockIdx.y][t] = o;
}

// out[m][n] = fp16(sum_k A[m][k] * W[k][n]) widened to fp32; both operands in fragment order; the matmuls of a message
// that nothing orders in one launch.
// A workgroup owns MT row tiles x 4 column tiles of 32 x 32. Its four waves are two column halves times two halves of K;
// a wave holds MT x 2 tiles, and the halves of K are added through LDS at the end. The operand pieces of a step (16 of K: MT KiB of rows that two
// waves share, 2 KiB of columns per wave) come into LDS by DMA as they lie in memory, in a ring of four slots, requested
// three steps ahead; the fragments of step s + 1 are read while the products of step s run, so a step costs one barrier.
// A wave reads (MT + 2) KiB of LDS for 2 MT matrix instructions: from MT = 3 on less than the LDS delivers while
// they run. Straight into registers (each wave its own 4 KiB of a step for four instructions, a launch per matrix)
// the path from L2 into a CU was the limit: 300 rows, seven
// projections of hidden 2048 / ffn 5632 took 264.8 us, now 94.6 (72 of them here = 430 TFLOP/s; the copies are 59 MB).
// A sum's order depends on k alone (never on MT or on the other members of a launch).
struct GemmMembers {
  float       *out[kPermutedGroupMax];
  const uint8_t *a[kPermutedGroupMax], *w[kPermutedGroupMax];
  int          n_tiles[kPermutedGroupMax], k_steps[kPermutedGroupMax];
  int          col_begin[kPermutedGroupMax + 1];  // in units of 4 column tiles
  int          count;
};

template <int MT>
__global__ __launch_bounds__(256, 2) void gemm_f16_fragments_kernel(GemmMembers members, int m, int m_tiles, int row_blocks) {
  constexpr int RING  = 4;
  constexpr int STEP  = 2 * MT + 8;            // KiB of a step: the rows of both K halves, the columns of four waves
  constexpr int APART = (MT + 1) / 2;          // row pieces that a wave brings (a shared odd one is brought twice)
  constexpr int PIECES = APART + 2;            // DMA instructions of a wave and step
  __shared__ __align__(1024) uint8_t lds[RING][STEP * 1024];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kh = wave >> 1, wn = wave & 1;
  // Workgroup ids go round the 8 XCDs: the row blocks of a column block follow each other on one XCD, so its weights come
  // from that L2 for all but the first, and the column blocks (longest K first) are dealt out evenly.
  const int turn = (int) blockIdx.x >> 3;
  const int col  = turn / row_blocks * 8 + ((int) blockIdx.x & 7), rb = turn % row_blocks;
  if (col >= members.col_begin[members.count]) {
    return;
  }
  int id = 0;
  while (id + 1 < members.count && col >= members.col_begin[id + 1]) {
    ++id;
  }
  const int n_tiles = members.n_tiles[id], k_steps = members.k_steps[id], steps = k_steps / 2;
  const int mt0 = rb * MT, nt0 = (col - members.col_begin[id]) * 4 + 2 * wn;

  // what this wave brings of every step: pieces of 1 KiB, the steps of a tile behind each other
  const uint8_t *src[PIECES];
  uint32_t       to[PIECES];
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    if (p < APART) {
      const int i = min(p * 2 + wn, MT - 1);
      src[p] = members.a[id] + (size_t) min(mt0 + i, m_tiles - 1) * k_steps * 1024;
      to[p]  = (uint32_t) (kh * MT + i) * 1024;
    } else {
      const int j = p - APART;
      src[p] = members.w[id] + (size_t) min(nt0 + j, n_tiles - 1) * k_steps * 1024;
      to[p]  = (uint32_t) (2 * MT + 2 * wave + j) * 1024;
    }
    src[p] += (size_t) kh * steps * 1024;
  }
  const uint32_t lds0 = (uint32_t) (uintptr_t) &lds[0][0];
  auto fetch = [&](int step) {  // (past the end: the last step again, so that the count of requests in flight stays)
    const size_t   off  = (size_t) min(step, steps - 1) * 1024;
    const uint32_t slot = lds0 + (uint32_t) (step & (RING - 1)) * (STEP * 1024);
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      asm volatile("s_mov_b32 m0, %2\n s_nop 0\n global_load_lds_dwordx4 %0, %1" ::"v"(lane * 16), "s"(src[p] + off), "s"(slot + to[p]) : "memory");
    }
  };
  struct Frags {
    uint4 a[MT], b[2];
  };
  auto read = [&](Frags &f, int step) {
    const uint8_t *slot = lds[step & (RING - 1)];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      f.a[i] = *reinterpret_cast<const uint4 *>(slot + (kh * MT + i) * 1024 + lane * 16);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f.b[j] = *reinterpret_cast<const uint4 *>(slot + (2 * MT + 2 * wave + j) * 1024 + lane * 16);
    }
  };
  v16f acc[MT][2];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] = 0.0f;
      }
    }
  }
  // Behind the barrier of step s everybody's pieces of step s + 1 have landed (all but the youngest two steps' requests
  // have returned) and the fragments of step s are in everybody's registers, so its slot takes step s + 4.
  auto turn_over = [&](int s, Frags &now, Frags &next) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(2 * PIECES) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch(s + RING);
    read(next, s + 1);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, now.a[i]), __builtin_bit_cast(v8h, now.b[j]),
                                                           acc[i][j], 0, 0, 0);
      }
    }
  };
#pragma unroll
  for (int s = 0; s < RING; ++s) {
    fetch(s);
  }
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * PIECES) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  Frags f0, f1;
  read(f0, 0);
  int s = 0;
  for (; s + 1 < steps; s += 2) {
    turn_over(s, f0, f1);
    turn_over(s + 1, f1, f0);
  }
  if (s < steps) {
    turn_over(s, f0, f1);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");

  // D[i][j]: j = lane % 32 (column), i = 8 (r / 4) + 4 (lane / 32) + r % 4 (row)
  float *xch = reinterpret_cast<float *>(&lds[0][0]) + (size_t) wn * 2 * 16 * 64 + lane;
  static_assert(2 * 2 * 16 * 64 * sizeof(float) <= sizeof(lds), "a row tile of both column halves fits");
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    __syncthreads();  // nobody reads the ring, or the row tile before, any more
    if (kh == 1) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          xch[(16 * j + r) * 64] = acc[i][j][r];
        }
      }
    }
    __syncthreads();
    if (kh == 0 && mt0 + i < m_tiles) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if (nt0 + j < n_tiles) {
          const int c = (nt0 + j) * 32 + (lane & 31);
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int row = (mt0 + i) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
            const float sum = acc[i][j][r] + xch[(16 * j + r) * 64];
            if (row < m) {
              members.out[id][(size_t) row * (n_tiles * 32) + c] = (float) (_Float16) sum;  // the reference stores fp16 results
            }
          }
        }
      }
    }
  }
}

}  // namespace

size_t permuted_weight_fragment_bytes(int k, int n) {
  return (size_t) k * (size_t) n * 2;
}

size_t permuted_act_fragment_bytes(int m, int k) {
  return (size_t) ((m + 31) / 32) * 32 * (size_t) k * 2;
}

hipError_t launch_permuted_weight_to_fragments(hipStream_t stream, void *dst, const void *src, int k, int n,
                                               int weight_kind) {
  if (k % 32 != 0 || n % 32 != 0 || weight_kind < 1 || weight_kind > 4) {
    return hipErrorInvalidValue;
  }
  const int    k_steps = k / 16, n_tiles = n / 32;
  const size_t pieces  = (size_t) k_steps * n_tiles * 64;
  const dim3   grid((unsigned) ((pieces + 255) / 256));
  uint4       *d = static_cast<uint4 *>(dst);
  switch (weight_kind) {
    case 1:
      hipLaunchKernelGGL(repack_w16_tiles_kernel, grid, dim3(256), 0, stream, d, static_cast<const uint32_t *>(src),
                         k_steps, n_tiles);
      break;
    case 2:
      hipLaunchKernelGGL(dequant_permuted_q4_kernel<false>, grid, dim3(256), 0, stream, d,
                         static_cast<const uint8_t *>(src), k_steps, n_tiles);
      break;
    case 3:
      hipLaunchKernelGGL(dequant_permuted_q8_kernel, grid, dim3(256), 0, stream, d, static_cast<const uint8_t *>(src),
                         k_steps, n_tiles);
      break;
    default:
      hipLaunchKernelGGL(dequant_permuted_q4_kernel<true>, grid, dim3(256), 0, stream, d,
                         static_cast<const uint8_t *>(src), k_steps, n_tiles);
      break;
  }
  return hipGetLastError();
}

size_t permuted_gemm_workspace_bytes(const PermutedMatMul *members, int count, int m) {
  size_t total = 0;
  for (int i = 0; i < count; ++i) {
    bool seen = false;
    for (int j = 0; j < i; ++j) {
      seen = seen || (members[j].act == members[i].act && members[j].k == members[i].k);
    }
    total += seen ? 0 : permuted_act_fragment_bytes(m, members[i].k);
  }
  return total;
}

hipError_t launch_permuted_gemm_group(hipStream_t stream, const PermutedMatMul *members, const void *const *weight_fragments,
                                      int count, int m, void *workspace) {
  if (count <= 0 || count > kPermutedGroupMax || m <= 0) {
    return hipErrorInvalidValue;
  }
  const int   m_tiles = (m + 31) / 32;
  ActMembers  acts    = {};
  GemmMembers g       = {};
  int         n_acts = 0, order[kPermutedGroupMax], act_of[kPermutedGroupMax], k_max = 0;
  uint8_t    *ws     = static_cast<uint8_t *>(workspace);
  for (int i = 0; i < count; ++i) {
    const PermutedMatMul &p = members[i];
    if (p.k % 32 != 0 || p.n % 32 != 0) {
      return hipErrorInvalidValue;
    }
    int j = 0;
    while (j < n_acts && !(acts.src[j] == p.act && acts.k[j] == p.k)) {
      ++j;
    }
    if (j == n_acts) {
      acts.src[j] = p.act, acts.k[j] = p.k, acts.dst[j] = reinterpret_cast<uint4 *>(ws);
      ws += permuted_act_fragment_bytes(m, p.k);
      ++n_acts;
      k_max = p.k > k_max ? p.k : k_max;
    }
    act_of[i] = j;
    int at = i;  // longest K first: the launch ends with short workgroups
    while (at > 0 && members[order[at - 1]].k < p.k) {
      order[at] = order[at - 1];
      --at;
    }
    order[at] = i;
  }
  const size_t a_pieces = (size_t) m_tiles * (k_max / 16) * 64;
  hipLaunchKernelGGL(act_to_fragments_kernel, dim3((unsigned) ((a_pieces + 255) / 256), (unsigned) n_acts), dim3(256), 0, stream,
                     acts, m, m_tiles);
  if (hipError_t e = hipGetLastError(); e != hipSuccess) {
    return e;
  }
  int cols = 0;
  g.count  = count;
  for (int i = 0; i < count; ++i) {
    const PermutedMatMul &p = members[order[i]];
    g.out[i] = p.out, g.a[i] = reinterpret_cast<const uint8_t *>(acts.dst[act_of[order[i]]]);
    g.w[i]       = static_cast<const uint8_t *>(weight_fragments[order[i]]);
    g.n_tiles[i] = p.n / 32, g.k_steps[i] = p.k / 16;
    g.col_begin[i] = cols;
    cols += (p.n / 32 + 3) / 4;
  }
  g.col_begin[count] = cols;
  // The most row tiles per workgroup that still give every CU one workgroup (two fit), spread evenly over the row blocks.
  int mt = m_tiles < 5 ? m_tiles : 5;
  while (mt > 1 && (long) cols * ((m_tiles + mt - 1) / mt) < 256) {
    --mt;
  }
  const int row_blocks = (m_tiles + mt - 1) / mt;
  mt = (m_tiles + row_blocks - 1) / row_blocks;
  const long long grid = (long long) ((cols + 7) / 8) * 8 * row_blocks;
  if (grid > 0x7fffffffLL) {
    return hipErrorInvalidValue;
  }
#define HTPOPS_GEMM(MT)                                                                                               \
  hipLaunchKernelGGL(gemm_f16_fragments_kernel<MT>, dim3((unsigned) grid), dim3(256), 0, stream, g, m, m_tiles, row_blocks)
  switch (mt) {
    case 1: HTPOPS_GEMM(1); break;
    case 2: HTPOPS_GEMM(2); break;
    case 3: HTPOPS_GEMM(3); break;
    case 4: HTPOPS_GEMM(4); break;
    default: HTPOPS_GEMM(5); break;
  }
#undef HTPOPS_GEMM
  return hipGetLastError();
}

}  // namespace htpops
