// Attention for gfx950: O = softmax(Q K^T / sqrt(D) + mask) V per head, GQA by h_kv = h / (n_heads / n_kv_heads).
//
// Replaces simple_flash_attn (reference: src/dsp/ops/flash_attn.c:1368-1420, core :139-825): the same blockwise
// online-softmax recurrence with exp2 and the scale 1/sqrt(D) * log2(e) (reference :210-215, :1440), laid out for
// 64-wide wavefronts and MFMA instead of HVX/HMX tiles in VTCM. Q/O are fp32 (the reference op) or fp16; K/V fp16
// [kv_len][n_kv_heads][D]; the optional fp16 mask [qo_len][align_up(kv_len, 64)] is ADDED to the scaled scores (the
// scalar routine's convention, reference :1505-1512); `causal` hides key j from query i when j > i + kv_len - qo_len.
//
// The kernels:
//  * prefill (several query rows, head_dim 64 or 128): one workgroup = 32 query rows x up to 4 query heads of one KV head (one
//    wave per head, so a K/V tile staged in LDS serves the whole GQA group). Scores are computed transposed,
//    S^T = K Q^T with v_mfma_f32_32x32x16_f16, which puts one query per lane: row max / row sum are register
//    reductions plus one exchange between the two lane halves. K and V blocks come into LDS as they lie in memory, by
//    DMA (global_load_lds) into two buffers that take turns: the next block is on its way while one is used. V^T for
//    O^T += V^T P^T is read out of the row-major tile with the transposing LDS read (ds_read_b64_tr_b16); P goes from
//    the score registers straight into the MFMA B operand. Scores are accumulated on top of minus the running
//    maximum, so most blocks need no rescaling. Under `causal`, KV blocks above the diagonal are skipped and the
//    longest query blocks start first. Timing-only builds on the 256-CU device (2048 x 2048 causal, 32 / 8 heads of
//    128, ten calls behind idle: 59 us; 48 to 50 us sustained) put the kernel without any matrix instruction and without the
//    exponentials at 39 us, without the DMA at 51 us. The matrix instructions alone take 16 us, the LDS reads (every wave reads
//    the whole K and V tile for its 32 queries, 1 KiB per matrix instruction) about 14: the bound is that scores, softmax and
//    P V of a block follow each other.
//  * decode (qo_len == 1, head_dim 64 or 128): bandwidth bound. The KV range is split across workgroups (n_kv_heads
//    alone would leave the GPU idle); both products run on the matrix cores with the heads of the GQA group as one
//    operand, and a second tiny kernel merges the per-split (max, sum, O) partials in one trip to memory.
//  * head dims that are other multiples of 16 up to 256 (the reference's flash_attn_sp_hdim.c domain): the prefill kernel
//    with rows padded to a multiple of 32, for one query row too (keys split over workgroups as in every grid that
//    would leave CUs idle, where it pays: see prefill_plan); the probabilities as fp16 pairs. 500 causal rows by mask, 16 / 4 heads of 96: 364 us in the
//    plain kernel, 18.7 us here.
//  * any other even head_dim up to 256: a plain kernel without MFMA.
#include "device_utils.h"
#include "kernels.h"

#include <algorithm>

namespace htpops {

namespace {

// What a mask value contributes to a score. Added as it is (the reference's scalar routine,
// src/dsp/ops/flash_attn.c:1505-1512), or, with `threshold`, selecting the key: kept (0) iff mask > -16, dropped
// (-inf) otherwise, NaN included (the kernel the reference dispatches, src/dsp/ops/flash_attn.c:448-460).
__device__ __forceinline__ float mask_term(_Float16 mv, bool threshold) {
  const float f = (float) mv;
  return threshold ? (f > -16.0f ? 0.0f : -INFINITY) : f;
}

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float    v16f __attribute__((ext_vector_type(16)));

constexpr float kLog2e = 1.44269504f;

__device__ __forceinline__ float fast_exp2(float x) {
  return __builtin_amdgcn_exp2f(x);  // v_exp_f32; exp2(-inf) = 0
}

// ------------------------------------------------------------------------------------------------ prefill

// Two states (max, sum, O) of one query become one: m takes the larger maximum; the factors of the state that m belonged to
// (`keep`) and of the other (returned). Written once, and with the fused operations spelled out, so that the same states
// give the same bits wherever they meet.
__device__ __forceinline__ float fold_factors(float &m, float other, float &keep) {
  const float m_new  = fmaxf(m, other);
  const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;  // nothing visible at all: keep the exponents finite
  keep = fast_exp2(m - m_safe);
  m    = m_new;
  return fast_exp2(other - m_safe);
}
__device__ __forceinline__ float fold(float fa, float a, float fb, float b) {
  return __builtin_fmaf(fa, a, fb * b);
}
template <int N>
struct Const {
  static constexpr int value = N;
};

constexpr int kPfThreads = 256;  // threads of one key group: 4 waves, one per query head
constexpr int kBQ        = 32;  // query rows per wave tile
constexpr int kBK        = 64;  // keys per KV block
constexpr int kPfMergeChunk = 8;  // shares whose parts the merge kernel has under way at a time

// One key group's share of LDS. K and V tiles of a block of keys, two buffers each: the next block arrives by DMA while
// one is used (the DMA chooses what each lane fetches, not where it lands: a lane lands 16 bytes behind its neighbour).
// Head dims up to DP are kept in rows of DP halfs; a row's 16-byte pieces are arranged so that the 16-byte fragment
// reads of 8 neighbouring K rows and the transposing reads of 4 neighbouring V rows fall into different banks: where
// DP % 64 == 0 the pieces are exclusive-or'ed with low bits of the row number (K: key % 8; V: 2 (key % 4), which keeps
// 32-byte pieces whole for the transposing reads), else K rows are one piece longer (an odd number of them) and V rows,
// an odd multiple of 64 bytes, lie right as they are.
template <int DP, bool MASK>
struct PrefillSmem {
  static constexpr bool kXor     = DP % 64 == 0;
  static constexpr int  kKPieces = kXor ? DP / 8 : DP / 8 + 1;  // 16-byte pieces of a K row, of a V row
  static constexpr int  kVPieces = DP / 8;
  uint8_t k[2][kBK * kKPieces * 16];
  uint8_t v[2][kBK * kVPieces * 16];
  // each wave's mask values of the next block ([query][64 keys] halfs, the pieces of a row exclusive-or'ed with query % 8)
  uint8_t mask[MASK ? kPfThreads / kWave : 1][MASK ? kBQ * kBK * 2 : 16];
};

// Floats of one 32-query tile of one head in the split-KV partials, for `units` = 4 * 32-column tiles of O^T: the
// (max, sum) pair of each lane, then unit for unit the lanes' four values.
__host__ __device__ constexpr size_t prefill_partial_floats(int units) {
  return (size_t) units * 4 * kWave + 2 * kWave;
}

// FULL: head_dim == DP (64 or 128); else head_dim is any multiple of 16 in (DP - 32, DP], and the probabilities are
// fp16 pairs (two matrix instructions per fragment of V): the plain kernel that these head dims took before held them in
// fp32. GROUPS = 1 or 2 key groups per workgroup (4 waves each); with 2 they take alternate KV blocks of the
// same queries. MASK: there is one (a kernel of its own: the tests for it cost 2048 x 2048 without one 1 to 2 %). With
// `shares` > 1 the blocks of a workgroup's queries are dealt to that many workgroups (gridDim.z), each of which leaves its
// (max, sum, O) in `part` for flash_attn_prefill_merge_kernel. ALL: one workgroup walks all shares itself and folds them in
// registers in the order and with the arithmetic of that kernel: the same bits without any memory between workgroups, for
// launches that must not hold an address of the context's (the mask may be absent then). It is bound by latency, like the
// unsplit walk, and pays for every share a handing-over through LDS: 5 rows over 1029 keys, 12 / 2 heads of 128, 8 shares 45 us
// against 20 us unsplit and 12 us on 32 workgroups; 500 rows over 500, 16 / 4 heads of 96, 22 us against 19.
template <int DP, bool FULL, bool QO_F32, int GROUPS, bool MASK, bool ALL>
__global__ __launch_bounds__(kPfThreads *GROUPS, DP <= 128 ? 2 : 1) void flash_attn_prefill_kernel(
  void *__restrict__ o_ptr, const void *__restrict__ q_ptr, const _Float16 *__restrict__ k_ptr,
  const _Float16 *__restrict__ v_ptr, const _Float16 *__restrict__ mask, int qo_len, int kv_len, int n_heads,
  int n_kv_heads, int head_dim, int flags, float *__restrict__ part, int shares) {
  using Smem = PrefillSmem<DP, MASK>;
  const bool causal = (flags & 1) != 0, mask_threshold = (flags & 2) != 0;
  __shared__ __align__(1024) Smem sm_all[GROUPS];
  constexpr int KSTEPS = DP / 16;  // MFMA k-steps over the head dimension
  constexpr int DT     = DP / 32;  // 32-row tiles of O^T
  constexpr float kPScale = FULL ? 1.0f : 32768.0f;  // of the probabilities: O and l are both too large by it
  const int     D      = FULL ? DP : head_dim;
  // With GROUPS = 2, two groups of 4 waves work on the same queries and heads: group g takes KV blocks g, g + 2, ...
  // with its own K/V tiles in LDS and its own running (max, sum, O); the two states are merged through LDS at the
  // end. The longest workgroup then walks half as many iterations, which pays when the grid is too small to keep two
  // independent workgroups on every CU busy to the end (few query blocks, or the uneven lengths under `causal`).
  const int grp = __builtin_amdgcn_readfirstlane((int) threadIdx.x / kPfThreads);  // (the same for a wave)
  Smem     &sm  = sm_all[grp];

  const int group = n_heads / n_kv_heads;
  const int gc    = group < 4 ? group : 4;  // heads handled by one workgroup
  const int qsub  = 4 / gc;                 // query sub-blocks per workgroup (waves left over when group < 4)
  const int sub_groups = (group + gc - 1) / gc;

  const int tid  = threadIdx.x % kPfThreads;  // within the key group
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5;
  const int col  = lane & 31;

  // grid: x = (KV head, head sub-group), y = query block, LAST query block first. Workgroups are dispatched in
  // linear order with x fastest, so under `causal` the long blocks (most visible keys) start first and the short ones
  // fill the tail; consecutive workgroups, which go to different XCDs, work on different KV heads, so one XCD's L2
  // keeps seeing the same K/V stream.
  const int q_block  = (int) (gridDim.y - 1 - blockIdx.y);
  const int h_kv     = blockIdx.x / sub_groups;
  const int h_in_grp = (blockIdx.x % sub_groups) * gc + wave % gc;
  const int  head    = h_kv * group + (h_in_grp < group ? h_in_grp : 0);
  const int  q_base  = (q_block * qsub + (wave / gc < qsub ? wave / gc : 0)) * kBQ;
  // waves without a head or without a query only help to bring the tiles
  const bool wave_on = h_in_grp < group && wave / gc < qsub && q_base < qo_len;
  const int  q_row   = q_base + col;                  // this lane's query
  const bool q_ok    = wave_on && q_row < qo_len;
  const int  q_clamp = q_row < qo_len ? q_row : qo_len - 1;

  const size_t qo_stride = (size_t) n_heads * D;
  const size_t kv_stride = (size_t) n_kv_heads * D;
  const size_t mask_ld   = ((size_t) kv_len + 63) / 64 * 64;
  const float  scale     = (1.0f / sqrtf((float) D)) * kLog2e;

  // Q fragments (B operand of S^T = K Q^T): lane (query, half) holds d = 16 s + 8 half .. + 7 for every k-step s
  v8h qf[KSTEPS];
  {
    const size_t base = (size_t) q_clamp * qo_stride + (size_t) head * D;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      const int d0 = 16 * s + 8 * half;
      if (!FULL && s == KSTEPS - 1 && 16 * s >= D) {  // (this step is left out below)
        qf[s] = (v8h){ 0, 0, 0, 0, 0, 0, 0, 0 };
        continue;
      }
      if (QO_F32) {
        const float4 *p  = reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(q_ptr) + base + d0);
        const float4  a  = p[0], b = p[1];
        qf[s][0] = (_Float16) (a.x * scale), qf[s][1] = (_Float16) (a.y * scale);
        qf[s][2] = (_Float16) (a.z * scale), qf[s][3] = (_Float16) (a.w * scale);
        qf[s][4] = (_Float16) (b.x * scale), qf[s][5] = (_Float16) (b.y * scale);
        qf[s][6] = (_Float16) (b.z * scale), qf[s][7] = (_Float16) (b.w * scale);
      } else {
        const v8h raw = *reinterpret_cast<const v8h *>(reinterpret_cast<const _Float16 *>(q_ptr) + base + d0);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          qf[s][e] = (_Float16) ((float) raw[e] * scale);
        }
      }
    }
  }

  v16f  oacc[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      oacc[t][r] = 0.0f;
    }
  }
  float m_run = -INFINITY;  // running max of this lane's query (same in both halves)
  float l_run = 0.0f;       // running sum over this half's keys only; halves are added at the end

  // keys visible to the LAST query row of the workgroup bound the KV loop under `causal`
  const int q_hi     = min(qo_len, (q_block + 1) * qsub * kBQ) - 1;
  const int kv_limit = causal ? max(0, min(kv_len, q_hi + (kv_len - qo_len) + 1)) : kv_len;
  const int q_shift  = kv_len - qo_len;
  // last key this lane's query may see, relative to the first key this lane holds in a block (key0 = 4 * half)
  const int vis_last = (causal ? min(kv_len - 1, q_row + q_shift) : kv_len - 1) - 4 * half;
  const int per = ((kv_limit + kBK - 1) / kBK + shares - 1) / shares * kBK;  // keys of a share

  // The next K/V block travels global memory -> LDS by DMA (global_load_lds, 1 KiB per instruction: no registers, no
  // stores) while the current one is being used. A tile of 64 rows is as many instructions as a row has pieces, the four
  // waves take every fourth; lane L of instruction i lands at piece 64 i + L of the tile and fetches what belongs there
  // (a row's last piece again where that lies behind the head dim). Per lane the source offsets inside a block never
  // change (kept in registers); what changes per block is a base address the same for all lanes.
  constexpr int KP = Smem::kKPieces, VP = Smem::kVPieces;
  constexpr int KROWB = KP * 16, VROWB = VP * 16;          // bytes of a row in LDS
  constexpr int KDMA = (KP + 3) / 4, VDMA = (VP + 3) / 4;  // instructions per wave and tile, at most
  auto k_piece = [&](int j, int &row) {
    const int p = (wave + 4 * j) * kWave + lane;
    row = p / KP;
    return min((p % KP) ^ (Smem::kXor ? row & 7 : 0), D / 8 - 1);
  };
  auto v_piece = [&](int j, int &row) {
    const int p = (wave + 4 * j) * kWave + lane;
    row = p / VP;
    return min((p % VP) ^ (Smem::kXor ? 2 * (row & 3) : 0), D / 8 - 1);
  };
  uint32_t k_src[KDMA], v_src[VDMA];  // byte offset of this lane's piece from the block's first row of this KV head
#pragma unroll
  for (int j = 0; j < KDMA; ++j) {
    int       row;
    const int piece = k_piece(j, row);
    k_src[j] = (uint32_t) row * (uint32_t) (kv_stride * 2) + 16u * (uint32_t) piece;
  }
#pragma unroll
  for (int j = 0; j < VDMA; ++j) {
    int       row;
    const int piece = v_piece(j, row);
    v_src[j] = (uint32_t) row * (uint32_t) (kv_stride * 2) + 16u * (uint32_t) piece;
  }
  auto fetch = [&](int k0, int buf) __attribute__((always_inline)) {  // (in registers: the DMA takes scalar bases)
    const uint32_t to_k = (uint32_t) (uintptr_t) sm.k[buf], to_v = (uint32_t) (uintptr_t) sm.v[buf];
    if (k0 + kBK <= kv_len) {
      const uint8_t *kb = reinterpret_cast<const uint8_t *>(k_ptr + (size_t) h_kv * D + (size_t) k0 * kv_stride);
      const uint8_t *vb = reinterpret_cast<const uint8_t *>(v_ptr + (size_t) h_kv * D + (size_t) k0 * kv_stride);
#pragma unroll
      for (int j = 0; j < KDMA; ++j) {
        if (KP % 4 == 0 || wave + 4 * j < KP) {
          asm volatile("s_mov_b32 m0, %2\n s_nop 0\n global_load_lds_dwordx4 %0, %1" ::"v"(k_src[j]), "s"(kb),
                       "s"(to_k + (uint32_t) ((wave + 4 * j) * 1024))
                       : "memory");
        }
      }
#pragma unroll
      for (int j = 0; j < VDMA; ++j) {
        if (VP % 4 == 0 || wave + 4 * j < VP) {
          asm volatile("s_mov_b32 m0, %2\n s_nop 0\n global_load_lds_dwordx4 %0, %1" ::"v"(v_src[j]), "s"(vb),
                       "s"(to_v + (uint32_t) ((wave + 4 * j) * 1024))
                       : "memory");
        }
      }
      return;
    }
    // last, partial block: rows past the end repeat the last key (their scores are hidden below)
#pragma unroll
    for (int j = 0; j < KDMA + VDMA; ++j) {
      const bool isv = j >= KDMA;
      const int  jj  = isv ? j - KDMA : j;
      if (wave + 4 * jj >= (isv ? VP : KP)) {
        continue;
      }
      int       row;
      const int piece = isv ? v_piece(jj, row) : k_piece(jj, row);
      const int key   = min(k0 + row, kv_len - 1);
      const _Float16 *src = (isv ? v_ptr : k_ptr) + (size_t) key * kv_stride + (size_t) h_kv * D + 8 * piece;
      asm volatile("s_mov_b32 m0, %1\n s_nop 0\n global_load_lds_dwordx4 %0, off" ::"v"(src),
                   "s"((isv ? to_v : to_k) + (uint32_t) ((wave + 4 * jj) * 1024))
                   : "memory");
    }
  };
  // The wave's mask values of a block travel the same way, each wave its own (no barrier needed): 32 rows of 128 bytes,
  // 16 bytes a lane, or 4 bytes a lane where the mask is not 16-byte aligned. (Loads into registers, 8 bytes a lane from
  // 32 rows at once, cost the address path 512 cycles per wave and block, as much as half the matrix instructions.)
  const bool mask_wide = (reinterpret_cast<uintptr_t>(mask) & 15) == 0 && mask_ld < ((size_t) 1 << 25);  // (32-bit offsets)
  const int  mask_rows = min(kBQ, qo_len - q_base);  // rows past the last query repeat it
  uint32_t   mask_src[4];  // byte offset of this lane's piece of rows 8 i .. 8 i + 7
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * i + (lane >> 3);
    mask_src[i]   = (uint32_t) min(row, mask_rows - 1) * (uint32_t) (mask_ld * 2) + 16u * (uint32_t) ((lane & 7) ^ (row & 7));
  }
  auto fetch_mask = [&](int k0) __attribute__((always_inline)) {
    const _Float16 *base = mask + (size_t) q_base * mask_ld + k0;
    const uint32_t  to   = (uint32_t) (uintptr_t) sm.mask[wave];
    if (mask_wide) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        asm volatile("s_mov_b32 m0, %2\n s_nop 0\n global_load_lds_dwordx4 %0, %1" ::"v"(mask_src[i]), "s"(base),
                     "s"(to + (uint32_t) (i * 1024))
                     : "memory");
      }
    } else {
#pragma unroll 1
      for (int i = 0; i < 16; ++i) {
        const int       row = 2 * i + (lane >> 5), d = lane & 31;
        const _Float16 *src = base + (size_t) min(row, mask_rows - 1) * mask_ld + 8 * ((d >> 2) ^ (row & 7)) + 2 * (d & 3);
        asm volatile("s_mov_b32 m0, %1\n s_nop 0\n global_load_lds_dword %0, off" ::"v"(src), "s"(to + (uint32_t) (i * 256)) : "memory");
      }
    }
  };
  // where this lane's fragments lie in a tile (bytes): K row `col` (+ 32 per tile), piece 2 s + half; V: the lane
  // (16-lane group g = lane / 16, i = lane % 16 = 4 j + q) points at row 4 half + j (+ 16 u + 8 per read), the 8-byte
  // piece q of columns 32 t + 16 (g & 1) .. + 15, and receives column 32 t + 16 (g & 1) + i of four rows (columns behind
  // the head dim repeat its last 16 and are not stored)
  uint32_t k_at[KSTEPS], v_at[DT];
  {
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      k_at[s] = (uint32_t) (col * KROWB + 16 * ((2 * s + half) ^ (Smem::kXor ? col & 7 : 0)));
    }
    const int g = lane >> 4, j = (lane >> 2) & 3, q = lane & 3;
#pragma unroll
    for (int t = 0; t < DT; ++t) {
      const int c0 = FULL ? 32 * t + 16 * (g & 1) : min(32 * t + 16 * (g & 1), D - 16);
      v_at[t] = (uint32_t) ((4 * half + j) * VROWB + 16 * ((c0 / 8 + (q >> 1)) ^ (Smem::kXor ? 2 * j : 0)) + 8 * (q & 1));
    }
  }
  typedef short v4s __attribute__((ext_vector_type(4)));

  const bool use_mask = MASK && wave_on && (!ALL || mask != nullptr);
  uint2      mreg[2][4];  // this lane's 2 x 16 mask values: keys 32 kt + 8 rg + 4 half + 0 .. 3

  // the keys of share `z`, from an empty state
  auto walk = [&](int z) __attribute__((always_inline)) {
    const int k_lo = z * per, k_hi = min(kv_limit, k_lo + per);
    if constexpr (ALL) {
      __syncthreads();  // (nobody uses LDS for the share before any more)
      m_run = -INFINITY, l_run = 0.0f;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          oacc[t][r] = 0.0f;
        }
      }
    }
    if (k_lo + grp * kBK < k_hi) {
      fetch(k_lo + grp * kBK, 0);
      if (use_mask) {
        fetch_mask(k_lo + grp * kBK);
      }
    }

    int it = 0;
    for (int kk = k_lo; kk < k_hi; kk += GROUPS * kBK, ++it) {
      const int  k0   = kk + grp * kBK;  // this key group's block of the iteration
      const int  buf  = it & 1;
      // this wave's share of the block has landed; behind the barrier everybody's has, and nobody reads the other
      // buffer (the previous block) any more
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      bool live = wave_on && k0 < k_hi;  // (the last iteration may have a block for the first group only)
      bool plain = true;                 // no mask value of the wave's block is anything but zero
      if (use_mask && k0 < k_hi) {
        uint32_t all = 0xffffffffu, any = 0;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
          for (int rg = 0; rg < 4; ++rg) {
            mreg[kt][rg] = *reinterpret_cast<const uint2 *>(sm.mask[wave] + col * 128 + 16 * ((4 * kt + rg) ^ (col & 7)) + 8 * half);
            all &= mreg[kt][rg].x & mreg[kt][rg].y;
            any |= mreg[kt][rg].x | mreg[kt][rg].y;
          }
        }
        // (the values are in registers before the next block's overwrite them)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        plain = __builtin_amdgcn_ballot_w64((any & 0x7fff7fffu) != 0) == 0;
        // A block that the mask hides from all 32 queries (-inf throughout; a causal mask hides half of a prompt's blocks)
        // is passed over, as under `causal`.
        if (__builtin_amdgcn_ballot_w64(!(all == 0xfc00fc00u && any == 0xfc00fc00u)) == 0) {
          live = false;
        }
      }
      if (k0 + GROUPS * kBK < k_hi) {
        fetch(k0 + GROUPS * kBK, buf ^ 1);
        if (use_mask) {
          fetch_mask(k0 + GROUPS * kBK);
        }
      }
      if (!live) {
        continue;
      }
      const uint8_t *k_tile = sm.k[buf], *v_tile = sm.v[buf];

      // ---- S^T - m = K Q^T - m: two 32-key tiles, accumulated on top of minus the running maximum ----
      // Scores come out of the MFMA already relative to the maximum seen so far, so a block that brings no new maximum
      // to any query of the wave (the usual case after the first few blocks) needs no subtraction and no rescaling.
      const bool  fresh = m_run == -INFINITY;  // nothing visible yet for this query
      const float m_ref = fresh ? 0.0f : m_run;
      v16f st[2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          st[kt][r] = -m_ref;
        }
      }
      // the two key tiles advance side by side (independent accumulators), and the fragments of step s + PF are
      // requested before the products of step s
      {
        constexpr int PF = 3;  // steps ahead (an LDS read takes longer to return than two steps' products to issue)
        v8h kf[PF + 1][2];
#pragma unroll
        for (int s = 0; s < PF && s < KSTEPS; ++s) {
#pragma unroll
          for (int kt = 0; kt < 2; ++kt) {
            kf[s][kt] = *reinterpret_cast<const v8h *>(k_tile + k_at[s] + 32 * kt * KROWB);
          }
        }
#pragma unroll
        for (int s = 0; s < KSTEPS; ++s) {
          if (s + PF < KSTEPS) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
              kf[(s + PF) % (PF + 1)][kt] = *reinterpret_cast<const v8h *>(k_tile + k_at[s + PF] + 32 * kt * KROWB);
            }
          }
          if (!FULL && s == KSTEPS - 1 && 16 * s >= D) {
            continue;  // (behind the head dim, the same for all waves)
          }
#pragma unroll
          for (int kt = 0; kt < 2; ++kt) {
            st[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[s % (PF + 1)][kt], qf[s], st[kt], 0, 0, 0);
          }
        }
      }

      // ---- mask (lane = query; register r of tile kt is key k0 + 32 kt + 8 (r / 4) + 4 half + r % 4) ----
      // Only blocks that mask values other than zero, the causal diagonal or the end of the keys touch pay for it (the same
      // for the whole wave).
      if (!plain || k0 + kBK > kv_len || (causal && k0 + kBK - 1 > q_base + q_shift)) {
        const int last = vis_last - k0;  // registers whose key offset 32 kt + 8 (r / 4) + r % 4 exceeds it are hidden
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
          for (int rg = 0; rg < 4; ++rg) {
            float add[4] = { 0.0f, 0.0f, 0.0f, 0.0f };
            if (!plain) {
              const v4h mv = __builtin_bit_cast(v4h, mreg[kt][rg]);
              add[0] = mask_term(mv[0], mask_threshold), add[1] = mask_term(mv[1], mask_threshold);
              add[2] = mask_term(mv[2], mask_threshold), add[3] = mask_term(mv[3], mask_threshold);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int r = 4 * rg + e;
              st[kt][r]   = (32 * kt + 8 * rg + e > last) ? -INFINITY : st[kt][r] + add[e];
            }
          }
        }
      }

      // ---- online softmax on scores relative to m_ref ----
      float mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          mx = fmaxf(mx, st[kt][r]);
        }
      }
      {
        // both 32-lane halves of the wave hold the same queries: v_permlane32_swap hands each the other's maximum
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
        mx            = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1]));
      }
      // the first visible block of a query sets its maximum (either sign), later blocks only raise it
      const bool move = fresh ? (mx != -INFINITY) : (mx > 0.0f);
      if (__builtin_amdgcn_ballot_w64(move) != 0) {
        // (a statement the compiler cannot run ahead of the test: without it the 97 instructions below are turned into
        // selects and run for every block)
        asm volatile("" ::: "memory");
        const float delta = move ? mx : 0.0f;
        const float alpha = fresh ? 0.0f : fast_exp2(-delta);  // O and l of a fresh query are still zero
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            st[kt][r] -= delta;
          }
        }
#pragma unroll
        for (int t = 0; t < DT; ++t) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            oacc[t][r] *= alpha;
          }
        }
        l_run *= alpha;
        m_run = move ? m_ref + mx : m_run;
      }
      // the probabilities, rounded to fp16 in pairs as the matrix instruction takes them. FULL: the row sum adds up the
      // rounded values (v_dot2_f32_f16 with ones: two per instruction, fp32 sums), so O and l see the same numbers; else
      // they are at most 2^15 and cut off, what is cut off goes into a second fp16 pair, and the row sum adds up the fp32
      // values. That holds 21 bits of each down to 2^-18 of the largest and 2^-39 of it below: behind a key that takes all but
      // 2^-16 of the weight and has a value of zero the result is off by 7e-7, as with fp32 probabilities. (Unscaled pairs end
      // at 2^-25 of the largest: 3e-5.) Where the first half is not zero neither is the second: times an infinite value it
      // must not become not-a-number.
      uint32_t pk[2][8], pk_lo[FULL ? 1 : 2][FULL ? 1 : 8];
      float    psum[4] = { 0.0f, 0.0f, 0.0f, 0.0f };  // (four chains: an addition waits for the one before it in its chain)
      {
        const v2h ones = { (_Float16) 1.0f, (_Float16) 1.0f }, least = __builtin_bit_cast(v2h, 0x00010001u);  // (2^-24)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            const float p0 = fast_exp2(st[kt][r]) * kPScale, p1 = fast_exp2(st[kt][r + 1]) * kPScale;
            if constexpr (FULL) {
              const v2h p2  = { (_Float16) p0, (_Float16) p1 };
              pk[kt][r / 2] = __builtin_bit_cast(uint32_t, p2);
              psum[(r / 2) & 3] = __builtin_amdgcn_fdot2(p2, ones, psum[(r / 2) & 3], false);
            } else {
              const v2h hi      = __builtin_bit_cast(v2h, __builtin_amdgcn_cvt_pkrtz(p0, p1));
              const v2h lo      = { (_Float16) (p0 - (float) hi[0]), (_Float16) (p1 - (float) hi[1]) };
              pk[kt][r / 2]     = __builtin_bit_cast(uint32_t, hi);
              pk_lo[kt][r / 2]  = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(lo, __builtin_elementwise_min(hi, least)));
              psum[(r / 2) & 3] += p0 + p1;
            }
          }
        }
      }
      l_run += (psum[0] + psum[1]) + (psum[2] + psum[3]);

      // ---- O^T += V^T P^T ----
      // MFMA (kt, u) covers keys 32 kt + 16 u + {4 half + 0..3, 8 + 4 half + 0..3}: exactly registers 8 u .. 8 u + 7
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const v8h pf = __builtin_bit_cast(v8h, make_uint4(pk[kt][4 * u], pk[kt][4 * u + 1], pk[kt][4 * u + 2], pk[kt][4 * u + 3]));
#pragma unroll
          for (int t = 0; t < DT; ++t) {
            // (V^T fragment: column 32 t + lane % 32 of keys 32 kt + 16 u + 4 half + 0 .. 3 and + 8 .. 11)
            const uint8_t *at = v_tile + v_at[t] + (32 * kt + 16 * u) * VROWB;
            const v4s a0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *) at);
            const v4s a1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *) (at + 8 * VROWB));
            const v8h vf = __builtin_bit_cast(v8h, (short __attribute__((ext_vector_type(8)))){ a0[0], a0[1], a0[2], a0[3],
                                                                                               a1[0], a1[1], a1[2], a1[3] });
            oacc[t]      = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf, oacc[t], 0, 0, 0);
            if constexpr (!FULL) {
              const v8h pl = __builtin_bit_cast(v8h, make_uint4(pk_lo[kt][4 * u], pk_lo[kt][4 * u + 1], pk_lo[kt][4 * u + 2],
                                                                pk_lo[kt][4 * u + 3]));
              oacc[t]      = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pl, oacc[t], 0, 0, 0);
            }
          }
        }
      }
    }

  };

  // O = O^T / l, one query per lane; register r of tile t is d = 32 t + 8 (r / 4) + 4 half + r % 4
  auto store = [&](int t, const v16f &o, float inv) {
    if (!q_ok) {
      return;
    }
    const size_t base = (size_t) q_row * qo_stride + (size_t) head * D;
#pragma unroll
    for (int rg = 0; rg < 4; ++rg) {
      const int d0 = 32 * t + 8 * rg + 4 * half;
      if (!FULL && d0 >= D) {
        continue;
      }
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = o[4 * rg + e] * inv;
      }
      if (QO_F32) {
        *reinterpret_cast<float4 *>(reinterpret_cast<float *>(o_ptr) + base + d0) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
        v4h hv = { (_Float16) v[0], (_Float16) v[1], (_Float16) v[2], (_Float16) v[3] };
        *reinterpret_cast<v4h *>(reinterpret_cast<_Float16 *>(o_ptr) + base + d0) = hv;
      }
    }
  };

  // ---- all shares in this workgroup. With two key groups, each folds its half of the columns (the first KEEP tiles of O,
  // and the others), so that the totals of a group are half the registers. ----
  if constexpr (ALL) {
    constexpr int KEEP  = GROUPS == 2 ? (DT + 1) / 2 : DT;
    constexpr int STATE = 16 * KEEP + 2;  // floats per lane that a group hands to the other
    static_assert(GROUPS == 1 || (size_t) 2 * (kPfThreads / kWave) * STATE * kWave * sizeof(float) <= sizeof(sm_all),
                  "the handed-over states fit the K/V tiles");
    float *to = reinterpret_cast<float *>(&sm_all[0]) + (size_t) ((1 - grp) * 4 + wave) * STATE * kWave + lane;
    const float *from = reinterpret_cast<const float *>(&sm_all[0]) + (size_t) (grp * 4 + wave) * STATE * kWave + lane;
    float m_tot = -INFINITY, l_tot = 0.0f;
    v16f  total[KEEP];
#pragma unroll
    for (int t = 0; t < KEEP; ++t) {
      total[t] = (v16f){ 0 };
    }
    // the runs of shares in the order in which the merge kernel's waves take them
    const int waves = shares > kPfMergeChunk ? 4 : 1;
    for (int w = 0; w < waves; ++w) {
      float m_wave = -INFINITY, l_wave = 0.0f;
      v16f  sum[KEEP];
#pragma unroll
      for (int t = 0; t < KEEP; ++t) {
        sum[t] = (v16f){ 0 };
      }
      for (int s0 = w * kPfMergeChunk; s0 < shares; s0 += waves * kPfMergeChunk) {
        for (int z = s0; z < min(s0 + kPfMergeChunk, shares); ++z) {
          walk(z);
          float m_own = m_run, l_own = l_run + __shfl_xor(l_run, 32, kWave);
          if constexpr (GROUPS == 2) {
            __syncthreads();  // everybody is done with the tiles
            to[0] = m_own, to[kWave] = l_own;
            auto give = [&](auto first, auto count) {
#pragma unroll
              for (int t = 0; t < decltype(count)::value; ++t) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                  to[(2 + 16 * t + r) * kWave] = oacc[decltype(first)::value + t][r];
                }
              }
            };
            if (grp == 0) {
              give(Const<KEEP>(), Const<DT - KEEP>());
            } else {
              give(Const<0>(), Const<KEEP>());
            }
            __syncthreads();
            const float m_other = from[0], l_other = from[kWave];
            float       own;
            const float other = fold_factors(m_own, m_other, own);
            l_own = grp == 0 ? fold(own, l_own, other, l_other) : fold(other, l_other, own, l_own);
            if (grp == 0) {
#pragma unroll
              for (int t = 0; t < KEEP; ++t) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                  oacc[t][r] = fold(own, oacc[t][r], other, from[(2 + 16 * t + r) * kWave]);
                }
              }
            } else {
#pragma unroll
              for (int t = 0; t < DT - KEEP; ++t) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                  oacc[t][r] = fold(other, from[(2 + 16 * t + r) * kWave], own, oacc[KEEP + t][r]);
                }
              }
            }
          }
          float       keep;
          const float add = fold_factors(m_wave, m_own, keep);
          l_wave          = fold(add, l_own, keep, l_wave);
#pragma unroll
          for (int t = 0; t < KEEP; ++t) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              sum[t][r] = fold(add, oacc[t][r], keep, sum[t][r]);
            }
          }
        }
      }
      float       keep;
      const float add = fold_factors(m_tot, m_wave, keep);
      l_tot           = fold(add, l_wave, keep, l_tot);
#pragma unroll
      for (int t = 0; t < KEEP; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          total[t][r] = fold(add, sum[t][r], keep, total[t][r]);
        }
      }
    }
    const float inv = 1.0f / l_tot;
#pragma unroll
    for (int t = 0; t < KEEP; ++t) {
      if (grp == 0) {
        store(t, total[t], inv);
      } else if (KEEP + t < DT) {
        store(KEEP + t, total[t], inv);
      }
    }
    return;
  }

  walk((int) blockIdx.z);

  // ---- the second key group hands its state over: m, l and O of the same query, lane for lane ----
  float l_tot = l_run + __shfl_xor(l_run, 32, kWave);
  if constexpr (GROUPS == 2) {
    constexpr int STATE = 16 * DT + 2;  // floats per lane
    static_assert((size_t) (kPfThreads / kWave) * STATE * kWave * sizeof(float) <= sizeof(sm_all),
                  "the handed-over state fits the K/V tiles");
    float *xch = reinterpret_cast<float *>(&sm_all[0]) + (size_t) wave * STATE * kWave + lane;
    __syncthreads();  // everybody is done with the tiles
    if (grp == 1) {
      xch[0] = m_run, xch[kWave] = l_tot;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          xch[(2 + 16 * t + r) * kWave] = oacc[t][r];
        }
      }
    }
    __syncthreads();
    if (grp == 1) {
      return;
    }
    const float m1 = xch[0], l1 = xch[kWave];
    float       a0;
    const float a1 = fold_factors(m_run, m1, a0);
    l_tot = fold(a0, l_tot, a1, l1);
#pragma unroll
    for (int t = 0; t < DT; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        oacc[t][r] = fold(a0, oacc[t][r], a1, xch[(2 + 16 * t + r) * kWave]);
      }
    }
  }

  // ---- a share of the keys only: leave (max, sum, O) as they are, lane for lane ----
  if (shares > 1) {
    if (wave_on) {
      const size_t n_tiles = (size_t) ((qo_len + kBQ - 1) / kBQ) * n_heads;
      const size_t tile    = (size_t) (q_base / kBQ) * n_heads + head;
      float *rec = part + ((size_t) blockIdx.z * n_tiles + tile) * prefill_partial_floats(4 * DT);
      reinterpret_cast<float2 *>(rec)[lane] = make_float2(m_run, l_tot);
      float4 *out = reinterpret_cast<float4 *>(rec + 2 * kWave) + lane;
#pragma unroll
      for (int t = 0; t < DT; ++t) {
#pragma unroll
        for (int rg = 0; rg < 4; ++rg) {
          out[(4 * t + rg) * kWave] = make_float4(oacc[t][4 * rg], oacc[t][4 * rg + 1], oacc[t][4 * rg + 2], oacc[t][4 * rg + 3]);
        }
      }
    }
    return;
  }

  const float inv = 1.0f / l_tot;
#pragma unroll
  for (int t = 0; t < DT; ++t) {
    store(t, oacc[t], inv);
  }
}

// Puts the shares of a split prefill together: G waves per 32-query tile, head and unit of four output columns per half
// (`units` of them), lane for lane as the prefill kernel left them. Each takes every G-th run of kPfMergeChunk shares, all
// loads of a run requested before the first use, folded one by one into a running (max, sum, O); with G = 4 (more
// shares than a run holds) the four states meet in LDS (one row, 16384 keys, 16 / 4 heads of 96, 64 shares: 23.0 -> 19.2 us).
// Q8 (QO_F32, G = 1, D = 8 units, a multiple of 32): the four waves of a workgroup hold one block of 32 output columns of 32 rows,
// which are also stored as Q8_0 in `q8_out` and (1 + ActOrder) in that operand order, whose lines they fill (12 heads of 128,
// 128 rows into int8 order: 3.9 -> 4.3 us for the launch of 3.1 behind it; 32 heads, 512 rows into FP6 order 8.1 -> 12.2 for one
// of 5.9).
template <bool QO_F32, int G, int Q8>
__global__ __launch_bounds__(256) void flash_attn_prefill_merge_kernel(void *__restrict__ o_ptr,
                                                                       const float *__restrict__ part, int n_splits,
                                                                       int n_tiles, int units, int qo_len, int n_heads,
                                                                       int D, uint8_t *__restrict__ q8_out, ActFragments fragments) {
  static_assert(Q8 < 0 || (QO_F32 && G == 1), "quantized rows come from one trip over fp32 rows");
  __shared__ float states[G == 1 ? 1 : G][6][G == 1 ? 1 : kWave];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
  const int id   = G == 1 ? (int) blockIdx.x * 4 + wave : (int) blockIdx.x;
  const int tile = id / units, unit = id % units;
  if (tile >= n_tiles) {  // (G = 4: the whole workgroup or none of it)
    return;
  }
  const size_t stride = (size_t) n_tiles * prefill_partial_floats(units);
  const float *rec    = part + (size_t) tile * prefill_partial_floats(units);
  float        m_run = -INFINITY, l_run = 0.0f;
  float        v[4]  = { 0.0f, 0.0f, 0.0f, 0.0f };
  for (int s0 = G == 1 ? 0 : wave * kPfMergeChunk; s0 < n_splits; s0 += G * kPfMergeChunk) {
    float2 ml[kPfMergeChunk];
    float4 x[kPfMergeChunk];
#pragma unroll
    for (int u = 0; u < kPfMergeChunk; ++u) {
      ml[u] = make_float2(-INFINITY, 0.0f);
      x[u]  = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (s0 + u < n_splits) {
        const float *at = rec + (size_t) (s0 + u) * stride;
        ml[u] = reinterpret_cast<const float2 *>(at)[lane];
        x[u]  = reinterpret_cast<const float4 *>(at + 2 * kWave)[(size_t) unit * kWave + lane];
      }
    }
#pragma unroll
    for (int u = 0; u < kPfMergeChunk; ++u) {
      float       keep;
      const float f = fold_factors(m_run, ml[u].x, keep);
      l_run = fold(f, ml[u].y, keep, l_run);
      v[0] = fold(f, x[u].x, keep, v[0]), v[1] = fold(f, x[u].y, keep, v[1]);
      v[2] = fold(f, x[u].z, keep, v[2]), v[3] = fold(f, x[u].w, keep, v[3]);
    }
  }
  if constexpr (G > 1) {
    states[wave][0][lane] = m_run, states[wave][1][lane] = l_run;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      states[wave][2 + e][lane] = v[e];
    }
    __syncthreads();
    if (wave != 0) {
      return;
    }
#pragma unroll
    for (int w = 1; w < G; ++w) {  // (a wave without shares has m = -inf, l = v = 0)
      float       keep;
      const float f = fold_factors(m_run, states[w][0][lane], keep);
      l_run = fold(f, states[w][1][lane], keep, l_run);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = fold(f, states[w][2 + e][lane], keep, v[e]);
      }
    }
  }
  const int   head = tile % n_heads, q_row = tile / n_heads * kBQ + (lane & 31);
  const int   d0   = 8 * unit + 4 * (lane >> 5);
  const float inv  = 1.0f / l_run;
  if (q_row < qo_len && d0 < D) {
    const size_t at = ((size_t) q_row * n_heads + head) * D + d0;
    if (QO_F32) {
      *reinterpret_cast<float4 *>(reinterpret_cast<float *>(o_ptr) + at) = make_float4(v[0] * inv, v[1] * inv, v[2] * inv, v[3] * inv);
    } else {
      v4h hv = { (_Float16) (v[0] * inv), (_Float16) (v[1] * inv), (_Float16) (v[2] * inv), (_Float16) (v[3] * inv) };
      *reinterpret_cast<v4h *>(reinterpret_cast<_Float16 *>(o_ptr) + at) = hv;
    }
  }
  if constexpr (Q8 >= 0) {
    __shared__ float rows[kBQ][kQK + 1];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      rows[lane & 31][8 * wave + 4 * (lane >> 5) + e] = v[e] * inv;
    }
    if (Q8 == 1 + kActI8 && blockIdx.x == 0) {
      end_act_fragments(fragments, threadIdx.x);
    }
    __syncthreads();
    const int row = tile / n_heads * kBQ + ((int) threadIdx.x >> 2), qpart = (int) threadIdx.x & 3;
    if (threadIdx.x >= 4 * kBQ || row >= qo_len) {  // (a quad of lanes has one row)
      return;
    }
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      x[i] = rows[threadIdx.x >> 2][8 * qpart + i];
    }
    uint16_t     scale;
    const uint2  quants = quantize_eight(x, &scale);
    const int    kb     = (head * units + unit) / 4;
    const size_t nblk   = (size_t) n_heads * units / 4;
    store_q8_0_block(reinterpret_cast<uint16_t *>(q8_out + ((size_t) row * nblk + kb) * 34), qpart, quants, scale);
    if constexpr (Q8 == 1 + kActFp6) {
      store_act_fp6(fragments, row, kb, qpart, quants, scale);
    } else if constexpr (Q8 == 1 + kActI8) {
      store_act_fragment(fragments, row, kb, qpart, quants, scale);
    }
  }
}

// ------------------------------------------------------------------------------------------------ decode

constexpr int kDecWaveKeys = 32;  // keys of one wave: two 16-key score tiles = one k step of P V
constexpr int kDecMaxGroup = 8;   // query heads scored per pass against one K/V stream
constexpr int kDecSplit    = 128; // keys per workgroup (four waves) ...
constexpr int kDecSplitShort = 64;  // ... and for short contexts (two waves), where 128 would leave most CUs without a workgroup

// partial record per (head, split): m, l, then D floats of un-normalised O.
// A workgroup owns SPLIT consecutive keys of one KV head; each of its SPLIT / 32 waves owns 32 of them and works
// without the others until the end. Both products run on the matrix cores (v_mfma_f32_16x16x32_f16), with up to 16
// query heads of the GQA group as the 16 rows (columns) of a tile:
//  * scores S = K Q^T: K in the A operand as it lies in memory (a lane loads 16 bytes of a key row per k step, all of
//    a wave's K loads issued before the first use); the queries in the B operand, fp32 queries scaled and split into an
//    fp16 pair (two instructions per k step: the scores are those of the fp32 queries to about 2^-22), fp16 queries as
//    they are with the scale applied to the score. A lane then holds, for one head, the scores of 4 keys per tile.
//  * softmax against the wave's own maximum, in those registers; rounded to fp16 they ARE the A operand of
//  * O = P V: the contraction runs over the wave's 32 keys, key 16 t + 4 g + i (tile t, lane group g, register i)
//    in k slot 8 g + 4 t + i. V is the B operand: a lane needs 8 keys at one column. The V rows come into LDS as they
//    are by DMA (global_load_lds, no registers), and ds_read_b64_tr_b16 hands each lane of a 16-lane group one column
//    of the 4 rows x 16 columns that the group's lanes point at (lanes 4 j .. 4 j + 3 at the four 8-byte pieces of
//    row j). Within a row the 32-byte pieces are stored exclusive-or'ed with the row number's low bits (the DMA
//    chooses what each lane fetches, not where it lands), so the four rows of a read lie in different banks.
// The waves' (max, sum, O) are put together through LDS with the factor exp2(m_wave - m_all) per wave and head.
// Measured on MI355X (32 query / 8 KV heads of 128, cold K/V; the split-KV launch alone, kv_len 4096 / 16384): all on
// the vector ALU (8 multiply-adds, 4 lane exchanges and an exponential per key, head and lane) 7.5 / 17.0 us; scores on
// the matrix cores and P V with v_dot2_f32_f16 6.3 / 15.3 us; this version: see the launcher. A variant in which a
// workgroup walks several chunks of keys with the next chunk on its way, about one workgroup per compute unit, was
// slower (17.0 us at 16384), and so was merging inside this launch behind a ticket per KV head (18-19 us at 4096).
template <int D, int GH, bool QO_F32, int SPLIT>
__global__ __launch_bounds__(SPLIT / kDecWaveKeys * kWave) void flash_attn_decode_kernel(
  float *__restrict__ part, const void *__restrict__ q_ptr, const _Float16 *__restrict__ k_ptr,
  const _Float16 *__restrict__ v_ptr, const _Float16 *__restrict__ mask, int kv_len, int n_heads, int n_kv_heads,
  int head0_in_group, int n_splits, int mask_threshold) {
  constexpr int WAVES   = SPLIT / kDecWaveKeys;
  constexpr int THREADS = WAVES * kWave;
  constexpr int KSTEPS  = D / 32;  // k steps of a score tile
  constexpr int CT      = D / 16;  // 16-column tiles of O
  constexpr int ROWB    = D * 2;   // bytes of a K or V row
  constexpr int CHUNKS  = ROWB / 16;            // 16-byte pieces of a row
  constexpr int DMA_ROWS = 1024 / ROWB;         // rows per DMA instruction (1 KiB)
  constexpr int DMAS    = kDecWaveKeys / DMA_ROWS;
  static_assert(GH <= 16 && (D == 64 || D == 128), "heads are the 16 rows of a tile");
  typedef float v4f __attribute__((ext_vector_type(4)));
  typedef short v4s __attribute__((ext_vector_type(4)));
  // LDS: V rows [SPLIT][D] halfs (wave w: rows 32 w ..), then o_w[WAVES][GH][D], red_l[WAVES][GH], red_m[WAVES][GH]
  extern __shared__ __align__(1024) uint8_t dec_lds[];
  float *o_sh  = reinterpret_cast<float *>(dec_lds + SPLIT * ROWB);
  float *red_l = o_sh + WAVES * GH * D, *red_m = red_l + WAVES * GH;

  const int group = n_heads / n_kv_heads;
  const int h_kv  = blockIdx.y;
  const int split = blockIdx.x;
  const int lane  = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col   = lane & 15;   // head of the pass (scores, P), column of the tile (V, O)
  const int kg    = lane >> 4;   // lane group: which 8 of a k step's 32 slots; rows 4 kg .. 4 kg + 3 of a result
  const float scale = (1.0f / sqrtf((float) D)) * kLog2e;
  const size_t kv_stride = (size_t) n_kv_heads * D;

  const int k_end  = min(kv_len, (split + 1) * SPLIT);
  const int k_wave = split * SPLIT + wave * kDecWaveKeys;  // this wave's keys: k_wave + 0 .. 31; keys from k_end on are
                                                           // read as key k_end - 1 and score -inf

  // V first (loads return in order: the K loads the compiler counts are then the youngest, and its waits for them
  // also cover these). DMA instruction i brings rows DMA_ROWS i .. of the wave's 32; lane L lands at byte 16 L of
  // that KiB = row L / CHUNKS, piece L % CHUNKS, and fetches the piece that belongs there.
  uint8_t *v_wave = dec_lds + wave * kDecWaveKeys * ROWB;
  {
    const uint32_t to = (uint32_t) (uintptr_t) v_wave;
#pragma unroll
    for (int i = 0; i < DMAS; ++i) {
      const int row   = i * DMA_ROWS + lane / CHUNKS;
      const int piece = (lane % CHUNKS) ^ (2 * (row & 3));  // (32-byte pieces exclusive-or'ed with the row's low bits)
      const int key   = min(k_wave + row, k_end - 1);
      const _Float16 *src = v_ptr + (size_t) key * kv_stride + (size_t) h_kv * D + 8 * piece;
      asm volatile("s_mov_b32 m0, %1\n s_nop 0\n global_load_lds_dwordx4 %0, off" ::"v"(src), "s"(to + (uint32_t) (i * 1024)) : "memory");
    }
  }
  // the queries: head `col` of the pass, dims 32 s + 8 kg .. + 7
  v8h qf[KSTEPS], qf_lo[KSTEPS];
  {
    const bool   q_on = col < GH && head0_in_group + col < group;
    const size_t base = (size_t) (h_kv * group + min(head0_in_group + col, group - 1)) * D + 8 * kg;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      if (QO_F32) {
        const float4 *qp = reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(q_ptr) + base + 32 * s);
        const float4  q0 = qp[0], q1 = qp[1];
        const float   on   = q_on ? scale : 0.0f;
        const float   x[8] = { q0.x * on, q0.y * on, q0.z * on, q0.w * on, q1.x * on, q1.y * on, q1.z * on, q1.w * on };
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          qf[s][e]    = (_Float16) x[e];
          qf_lo[s][e] = (_Float16) (x[e] - (float) qf[s][e]);
        }
      } else {
        const v8h qv = *reinterpret_cast<const v8h *>(reinterpret_cast<const _Float16 *>(q_ptr) + base + 32 * s);
        qf[s]        = q_on ? qv : (v8h){ 0, 0, 0, 0, 0, 0, 0, 0 };
        qf_lo[s]     = (v8h){ 0, 0, 0, 0, 0, 0, 0, 0 };  // (not used)
      }
    }
  }
  // K: row `col` of tile t is key 16 t + col of the wave
  v8h kf[2][KSTEPS];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int    key = min(k_wave + 16 * t + col, k_end - 1);
    const size_t off = (size_t) key * kv_stride + (size_t) h_kv * D + 8 * kg;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      kf[t][s] = *reinterpret_cast<const v8h *>(k_ptr + off + 32 * s);
    }
  }
  // row 0 of the mask (qo_len == 1) for the 8 keys of this lane, requested with the rest
  float mk[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = k_wave + 16 * t + 4 * kg + i;
      mk[t][i] = (mask && key < k_end) ? mask_term(mask[key], mask_threshold != 0) : 0.0f;
    }
  }

  // scores of head `col` for keys 16 t + 4 kg + i
  float sc[2][4];
  float m_w = -INFINITY;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    v4f acc = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[t][s], qf[s], acc, 0, 0, 0);
      if (QO_F32) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[t][s], qf_lo[s], acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool  live = k_wave + 16 * t + 4 * kg + i < k_end;
      const float v    = (QO_F32 ? acc[i] : acc[i] * scale) + mk[t][i];
      sc[t][i]         = live ? v : -INFINITY;
      m_w              = fmaxf(m_w, sc[t][i]);
    }
  }
  // the wave's maximum of head `col`: over the four lane groups
  m_w = fmaxf(m_w, __shfl_xor(m_w, 16, kWave));
  m_w = fmaxf(m_w, __shfl_xor(m_w, 32, kWave));
  const float m_safe = (m_w == -INFINITY) ? 0.0f : m_w;
  float       l_w    = 0.0f;
  v8h         pf;  // A operand of P V: k slot 8 kg + 4 t + i
#pragma unroll
  for (int t = 0; t < 2; ++t) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float pr = fast_exp2(sc[t][i] - m_safe);
      l_w += pr;
      pf[4 * t + i] = (_Float16) pr;
    }
  }
  l_w += __shfl_xor(l_w, 16, kWave);
  l_w += __shfl_xor(l_w, 32, kWave);
  if (kg == 0 && col < GH) {
    red_m[wave * GH + col] = m_w;
    red_l[wave * GH + col] = l_w;
  }

  // O = P V. (Every load of this wave has returned by now: the K loads were the youngest. The wait is written out
  // because the compiler knows nothing of the DMA.) Read h of tile c: lane (group kg, col = 4 j + q) points at row
  // 16 h + 4 kg + j, halfs 16 c + 4 q .. + 3, and receives column 16 c + col of rows 16 h + 4 kg + 0 .. 3.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  v4f oacc[CT];
  {
    const int j = col >> 2, q = col & 3;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      v4s b[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row   = 16 * h + 4 * kg + j;
        const int piece = (2 * c + (q >> 1)) ^ (2 * (row & 3));
        const uint8_t *at = v_wave + row * ROWB + piece * 16 + 8 * (q & 1);
        b[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *) at);
      }
      const v8h bf = __builtin_bit_cast(v8h, (short __attribute__((ext_vector_type(8)))){ b[0][0], b[0][1], b[0][2], b[0][3],
                                                                                           b[1][0], b[1][1], b[1][2], b[1][3] });
      const v4f zero = { 0.0f, 0.0f, 0.0f, 0.0f };
      oacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pf, bf, zero, 0, 0, 0);
    }
  }
  // rows 4 kg + i of the result are heads: this lane's column 16 c + col of each
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int g = 4 * kg + i;
    if (g < GH) {
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        o_sh[((size_t) wave * GH + g) * D + 16 * c + col] = oacc[c][i];
      }
    }
  }
  __syncthreads();
  // put the waves together, each with its factor: two neighbouring columns per thread
  for (int i = threadIdx.x * 2; i < GH * D; i += THREADS * 2) {
    const int g = i / D, d = i % D;
    if (head0_in_group + g >= group) {
      continue;
    }
    float m_all = red_m[g];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      m_all = fmaxf(m_all, red_m[w * GH + g]);
    }
    const float m_ref = (m_all == -INFINITY) ? 0.0f : m_all;
    float       v0 = 0.0f, v1 = 0.0f, l = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float  f = fast_exp2(red_m[w * GH + g] - m_ref);
      const float2 x = *reinterpret_cast<const float2 *>(o_sh + ((size_t) w * GH + g) * D + d);
      l += red_l[w * GH + g] * f;
      v0 += x.x * f, v1 += x.y * f;
    }
    const int head = h_kv * group + head0_in_group + g;
    float    *rec  = part + ((size_t) head * n_splits + split) * (D + 2);
    *reinterpret_cast<float2 *>(rec + 2 + d) = make_float2(v0, v1);
    if (d == 0) {
      *reinterpret_cast<float2 *>(rec) = make_float2(m_all, l);
    }
  }
}

// One workgroup per head: MG groups of D threads, one thread per output column in each; group j merges the j-th part
// of the splits, then the groups' (max, sum, column) are put together through LDS (MG = 1: nothing to put together;
// measured at 32 heads of 128: 32 splits 3.2 us with one group, 4.2 with four; 128 splits 5.7 and 4.0). A group takes its splits
// 64 at a time with every load of a chunk -- the (max, sum) pair of split `lane` and this thread's column of all 64
// records -- requested before the first use, so a chunk costs one trip to memory (kv_len up to 32768 at 128 keys per
// split: the whole merge is one trip). Each wave works the rescale factors out for itself (lane s holds that of split
// s, read back with v_readlane); chunks are folded into a running (max, sum, column) like KV blocks are.
constexpr int kMergeChunk  = 64;
constexpr int kMergeGroups = 4;  // for more than kMergeChunk splits

template <int D, bool QO_F32, int MG>
__global__ __launch_bounds__(D *MG) void flash_attn_decode_merge_kernel(void *__restrict__ o_ptr,
                                                                        const float *__restrict__ part, int n_splits,
                                                                        uint8_t *__restrict__ q8_out) {
  // (q8_out, fp32 output only: the output row is also written as Q8_0 blocks, the bytes the Q8_0 quantizer makes of
  // it; a block is 32 neighbouring columns, one half of a wave)
  extern __shared__ float merge_lds[];  // MG > 1 only: the groups' columns [MG][D], then their (max, sum) [MG][2]
  static_assert(D % kWave == 0, "a wave lies in one group");
  const int    head = blockIdx.x, d = threadIdx.x % D, lane = threadIdx.x & (kWave - 1);
  // (the same for the whole wave, and known to be: the bounds below then stay in scalar registers and the 64 loads of a
  // chunk are switched by scalar branches instead of one lane mask each)
  const int    grp  = __builtin_amdgcn_readfirstlane((int) threadIdx.x / D);
  const float *rec0 = part + (size_t) head * n_splits * (D + 2);
  const int    per  = (n_splits + MG - 1) / MG;  // splits of a group
  const int    s_begin = grp * per, s_end = min(n_splits, s_begin + per);
  float        m_run = -INFINITY, l_run = 0.0f, v_run = 0.0f;
  for (int s0 = s_begin; s0 < s_end; s0 += kMergeChunk) {
    const int  left = s_end - s0;  // >= 1
    const bool mine = lane < kMergeChunk && lane < left;
    float      m_s = -INFINITY, l_s = 0.0f;
    if (mine) {
      const float2 ml = *reinterpret_cast<const float2 *>(rec0 + (size_t) (s0 + lane) * (D + 2));
      m_s = ml.x, l_s = ml.y;
    }
    float x[kMergeChunk];
#pragma unroll
    for (int u = 0; u < kMergeChunk; ++u) {
      x[u] = u < left ? rec0[(size_t) (s0 + u) * (D + 2) + 2 + d] : 0.0f;
    }
    const float m_new  = fmaxf(m_run, wave_max(m_s));
    const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;
    const float keep   = fast_exp2(m_run - m_safe);  // 0 for the first chunk
    const float f      = fast_exp2(m_s - m_safe);    // 0 in lanes without a split
    float       lf     = l_s * f;
    asm("" : "+v"(lf));  // (a product of its own: not fused into the sum's first addition)
    l_run              = __builtin_fmaf(l_run, keep, wave_sum(lf));
    float v            = 0.0f;
#pragma unroll
    for (int u = 0; u < kMergeChunk; ++u) {
      v = __builtin_fmaf(x[u], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f), u)), v);
    }
    v_run = __builtin_fmaf(v_run, keep, v);
    m_run = m_new;
  }
  if (MG > 1) {
    float *grp_v = merge_lds, *grp_ml = merge_lds + MG * D;
    grp_v[grp * D + d] = v_run;
    if (d == 0) {
      grp_ml[2 * grp] = m_run, grp_ml[2 * grp + 1] = l_run;
    }
    __syncthreads();
    if (grp != 0) {
      return;
    }
    float m_all = grp_ml[0];
#pragma unroll
    for (int j = 1; j < MG; ++j) {
      m_all = fmaxf(m_all, grp_ml[2 * j]);
    }
    const float m_safe = (m_all == -INFINITY) ? 0.0f : m_all;
    l_run = 0.0f, v_run = 0.0f;
#pragma unroll
    for (int j = 0; j < MG; ++j) {  // (a group without splits has m = -inf, l = v = 0)
      const float f = fast_exp2(grp_ml[2 * j] - m_safe);
      l_run += grp_ml[2 * j + 1] * f;
      v_run += grp_v[j * D + d] * f;
    }
  }
  float out = v_run * (1.0f / l_run);
  asm("" : "+v"(out));  // (rounded here, not fused into the conversion)
  if (QO_F32) {
    reinterpret_cast<float *>(o_ptr)[(size_t) head * D + d] = out;
    if (q8_out != nullptr) {
      float amax = fabsf(out);
#define HTPOPS_DPP_MAX(ctrl) \
  amax = fmaxf(amax, __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(amax), __float_as_int(amax), ctrl, 0xf, 0xf, false)))
      HTPOPS_DPP_MAX(0xB1);   // quad_perm [1,0,3,2]
      HTPOPS_DPP_MAX(0x4E);   // quad_perm [2,3,0,1]
      HTPOPS_DPP_MAX(0x141);  // row_half_mirror
      HTPOPS_DPP_MAX(0x140);  // row_mirror: the 16 lanes of a row
#undef HTPOPS_DPP_MAX
      amax            = fmaxf(amax, __shfl_xor(amax, 16, kWave));  // the two rows of the block
      const float dq  = amax / 127.0f;
      const float id  = (dq != 0.0f) ? 1.0f / dq : 0.0f;
      const int   col = head * D + d;
      uint8_t    *blk = q8_out + (size_t) (col >> 5) * 34;
      blk[2 + (col & 31)] = (uint8_t) (int) roundf(out * id);
      if ((col & 31) == 0) {
        *reinterpret_cast<uint16_t *>(blk) = __half_as_ushort(__float2half_rn(dq));
      }
    }
  } else {
    reinterpret_cast<_Float16 *>(o_ptr)[(size_t) head * D + d] = (_Float16) out;
  }
}

// ------------------------------------------------------------------------------------------------ a few rows

// The same for a few query rows (several sequences' tokens, drafted tokens that are verified): the rows of a score tile are
// the (query, head) pairs of a GQA group, query by query, 16 to a workgroup (blockIdx.z). Bound by latency: two short launches,
// a wave has 32 keys and one trip to memory. The prefill kernel gives every head a tile of 32 queries of its own and walks
// 64 keys at a time, a microsecond a turn: 5 rows over 1029 keys, 12 / 2 heads of 128, fp32 with a mask 12.5 us there, 8.5 here;
// 4 rows over 3000, 32 / 8 heads 17.8 and 10.0 (see few_plan).
// Keys that a row may not see score -inf whatever K holds, and a wave none of whose keys is seen by any row leaves its V alone,
// as the prefill kernel passes over such blocks. fp32 queries count with 22 bits here, with 11 there.
// ALL: one workgroup walks all splits of its rows, once for the maxima and sums and once more for O, with the arithmetic of
// this kernel and of flash_attn_decode_merge_kernel (at most kMergeChunk splits): the same bits without memory between
// workgroups, for launches that must not hold an address of the context's.
constexpr int kFewRows = 16;

template <int D, bool QO_F32, int SPLIT, bool ALL>
__global__ __launch_bounds__(SPLIT / kDecWaveKeys * kWave) void flash_attn_few_rows_kernel(
  void *__restrict__ out, const void *__restrict__ q_ptr, const _Float16 *__restrict__ k_ptr, const _Float16 *__restrict__ v_ptr,
  const _Float16 *__restrict__ mask, int qo_len, int kv_len, int n_heads, int n_kv_heads, int n_splits, int flags) {
  constexpr int WAVES   = SPLIT / kDecWaveKeys;
  constexpr int THREADS = WAVES * kWave;
  constexpr int KSTEPS  = D / 32;  // k steps of a score tile
  constexpr int CT      = D / 16;  // 16-column tiles of O
  constexpr int ROWB    = D * 2;   // bytes of a K or V row
  constexpr int CHUNKS  = ROWB / 16;
  constexpr int DMA_ROWS = 1024 / ROWB;
  constexpr int DMAS    = kDecWaveKeys / DMA_ROWS;
  constexpr int PAIRS   = kFewRows * D / 2 / THREADS;  // pairs of neighbouring columns that a thread puts together
  typedef float v4f __attribute__((ext_vector_type(4)));
  typedef short v4s __attribute__((ext_vector_type(4)));
  // a wave's V rows and, when it is done with them, its O [16][D]: the same bytes
  static_assert(kDecWaveKeys * ROWB == kFewRows * D * (int) sizeof(float), "O takes the place of V");
  __shared__ __align__(1024) uint8_t v_sh[SPLIT * ROWB];
  __shared__ float red_m[WAVES][kFewRows], red_l[WAVES][kFewRows];
  __shared__ float tab_m[ALL ? kFewRows : 1][kMergeChunk], tab_l[ALL ? kFewRows : 1][kMergeChunk];

  const bool causal = (flags & 1) != 0, mask_threshold = (flags & 2) != 0;
  const int  group = n_heads / n_kv_heads, rows = qo_len * group;
  const int  h_kv  = blockIdx.y, row0 = (int) blockIdx.z * kFewRows;
  const int  lane  = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int  col   = lane & 15, kg = lane >> 4;
  const float  scale     = (1.0f / sqrtf((float) D)) * kLog2e;
  const size_t kv_stride = (size_t) n_kv_heads * D;
  const size_t mask_ld   = ((size_t) kv_len + 63) / 64 * 64;
  // this lane's row of the score tile (rows past the last one repeat it with queries of zero; nobody reads their results)
  const int row = min(row0 + col, rows - 1), q_row = row / group, head = h_kv * group + row % group;
  const int vis_last = causal ? q_row + kv_len - qo_len : kv_len - 1;

  v8h qf[KSTEPS], qf_lo[KSTEPS];
  {
    const size_t base = ((size_t) q_row * n_heads + head) * D + 8 * kg;
    const bool   q_on = row0 + col < rows;
#pragma unroll
    for (int s = 0; s < KSTEPS; ++s) {
      if (QO_F32) {
        const float4 *qp = reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(q_ptr) + base + 32 * s);
        const float4  q0 = qp[0], q1 = qp[1];
        const float   x[8] = { q0.x * scale, q0.y * scale, q0.z * scale, q0.w * scale, q1.x * scale, q1.y * scale, q1.z * scale, q1.w * scale };
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          qf[s][e]    = q_on ? (_Float16) x[e] : (_Float16) 0.0f;
          qf_lo[s][e] = q_on ? (_Float16) (x[e] - (float) qf[s][e]) : (_Float16) 0.0f;
        }
      } else {
        const v8h qv = *reinterpret_cast<const v8h *>(reinterpret_cast<const _Float16 *>(q_ptr) + base + 32 * s);
        qf[s]        = q_on ? qv : (v8h){ 0, 0, 0, 0, 0, 0, 0, 0 };
        qf_lo[s]     = (v8h){ 0, 0, 0, 0, 0, 0, 0, 0 };  // (not used)
      }
    }
  }

  uint8_t *v_wave = v_sh + wave * kDecWaveKeys * ROWB;
  float   *o_wave = reinterpret_cast<float *>(v_wave);
  // one split: maxima and sums, and O (`with_o`), of every wave in LDS, behind a barrier
  auto walk = [&](int split, bool with_o) __attribute__((always_inline)) {
    const int k_end  = min(kv_len, (split + 1) * SPLIT);
    const int k_wave = split * SPLIT + wave * kDecWaveKeys;  // (keys from k_end on are read as key k_end - 1 and score -inf)
    if (with_o) {
      const uint32_t to = (uint32_t) (uintptr_t) v_wave;
#pragma unroll
      for (int i = 0; i < DMAS; ++i) {
        const int r     = i * DMA_ROWS + lane / CHUNKS;
        const int piece = (lane % CHUNKS) ^ (2 * (r & 3));
        const int key   = min(k_wave + r, k_end - 1);
        const _Float16 *src = v_ptr + (size_t) key * kv_stride + (size_t) h_kv * D + 8 * piece;
        asm volatile("s_mov_b32 m0, %1\n s_nop 0\n global_load_lds_dwordx4 %0, off" ::"v"(src), "s"(to + (uint32_t) (i * 1024)) : "memory");
      }
    }
    v8h kf[2][KSTEPS];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int    key = min(k_wave + 16 * t + col, k_end - 1);
      const size_t off = (size_t) key * kv_stride + (size_t) h_kv * D + 8 * kg;
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) {
        kf[t][s] = *reinterpret_cast<const v8h *>(k_ptr + off + 32 * s);
      }
    }
    // this row's mask for keys 16 t + 4 kg .. + 3 (a wave behind the last key reads the last one's: a mask row is whole
    // groups of 64)
    v4h mv[2];
    if (mask) {
      const _Float16 *at = mask + (size_t) q_row * mask_ld + min(k_wave, (kv_len - 1) / kDecWaveKeys * kDecWaveKeys) + 4 * kg;
      mv[0] = *reinterpret_cast<const v4h *>(at), mv[1] = *reinterpret_cast<const v4h *>(at + 16);
    }
    float sc[2][4], m_w = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      v4f acc = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
      for (int s = 0; s < KSTEPS; ++s) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[t][s], qf[s], acc, 0, 0, 0);
        if (QO_F32) {
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[t][s], qf_lo[s], acc, 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int   key = k_wave + 16 * t + 4 * kg + i;
        const float mk  = mask ? mask_term(mv[t][i], mask_threshold) : 0.0f;
        const bool  see = key < k_end && key <= vis_last && mk != -INFINITY;
        sc[t][i]        = see ? (QO_F32 ? acc[i] + mk : __builtin_fmaf(acc[i], scale, mk)) : -INFINITY;
        m_w             = fmaxf(m_w, sc[t][i]);
      }
    }
    m_w = fmaxf(m_w, __shfl_xor(m_w, 16, kWave));
    m_w = fmaxf(m_w, __shfl_xor(m_w, 32, kWave));
    const float m_safe = (m_w == -INFINITY) ? 0.0f : m_w;
    float       l_w    = 0.0f;
    v8h         pf;  // A operand of P V: k slot 8 kg + 4 t + i
    bool        seen = false;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        seen          = seen || sc[t][i] != -INFINITY;
        pf[4 * t + i] = (_Float16) fast_exp2(sc[t][i] - m_safe);
        l_w += (float) pf[4 * t + i];  // (as the prefill kernel: O and l see the same numbers)
      }
    }
    l_w += __shfl_xor(l_w, 16, kWave);
    l_w += __shfl_xor(l_w, 32, kWave);
    if (kg == 0) {
      red_m[wave][col] = m_w, red_l[wave][col] = l_w;
    }
    if (with_o) {
      const bool any = __builtin_amdgcn_ballot_w64(seen) != 0;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      v4f       oacc[CT];
      const int j = col >> 2, q = col & 3;
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        oacc[c] = (v4f){ 0.0f, 0.0f, 0.0f, 0.0f };
        if (any) {
          v4s b[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const int r     = 16 * h + 4 * kg + j;
            const int piece = (2 * c + (q >> 1)) ^ (2 * (r & 3));
            const uint8_t *at = v_wave + r * ROWB + piece * 16 + 8 * (q & 1);
            b[h] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((v4s __attribute__((address_space(3))) *) at);
          }
          const v8h bf = __builtin_bit_cast(v8h, (short __attribute__((ext_vector_type(8)))){ b[0][0], b[0][1], b[0][2], b[0][3],
                                                                                               b[1][0], b[1][1], b[1][2], b[1][3] });
          oacc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pf, bf, oacc[c], 0, 0, 0);
        }
      }
      // (every read of the wave's V rows has returned before the first of these stores)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          o_wave[(4 * kg + i) * D + 16 * c + col] = oacc[c][i];
        }
      }
    }
    __syncthreads();
  };
  // the waves of a split put together: row g, columns d and d + 1
  auto together = [&](int g, int d, float &m_all, float &l, float &v0, float &v1) {
    m_all = red_m[0][g];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      m_all = fmaxf(m_all, red_m[w][g]);
    }
    const float m_ref = (m_all == -INFINITY) ? 0.0f : m_all;
    v0 = 0.0f, v1 = 0.0f, l = 0.0f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      const float  f = fast_exp2(red_m[w][g] - m_ref);
      const float2 x = *reinterpret_cast<const float2 *>(v_sh + w * kDecWaveKeys * ROWB + (g * D + d) * 4);
      l  = __builtin_fmaf(red_l[w][g], f, l);
      v0 = __builtin_fmaf(x.x, f, v0), v1 = __builtin_fmaf(x.y, f, v1);
    }
  };
  if constexpr (!ALL) {
    const int split = blockIdx.x;
    walk(split, true);
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      const int i = 2 * ((int) threadIdx.x + p * THREADS), g = i / D, d = i % D, r = row0 + g;
      if (r >= rows) {
        continue;
      }
      float m_all, l, v0, v1;
      together(g, d, m_all, l, v0, v1);
      float *rec = static_cast<float *>(out) + (((size_t) (r / group) * n_heads + h_kv * group + r % group) * n_splits + split) * (D + 2);
      *reinterpret_cast<float2 *>(rec + 2 + d) = make_float2(v0, v1);
      if (d == 0) {
        *reinterpret_cast<float2 *>(rec) = make_float2(m_all, l);
      }
    }
    return;
  }
  if constexpr (ALL) {
    for (int split = 0; split < n_splits; ++split) {
      walk(split, false);
      if (threadIdx.x < kFewRows) {
        const int g = threadIdx.x;
        float     m_all = red_m[0][g], l = 0.0f;
        for (int w = 1; w < WAVES; ++w) {
          m_all = fmaxf(m_all, red_m[w][g]);
        }
        const float m_ref = (m_all == -INFINITY) ? 0.0f : m_all;
        for (int w = 0; w < WAVES; ++w) {
          l = __builtin_fmaf(red_l[w][g], fast_exp2(red_m[w][g] - m_ref), l);
        }
        tab_m[g][split] = m_all, tab_l[g][split] = l;
      }
      __syncthreads();
    }
    // every split's factor takes its maximum's place, the row's sum that of split 0
    for (int g = wave; g < kFewRows; g += WAVES) {
      const float m_s = lane < n_splits ? tab_m[g][lane] : -INFINITY, l_s = lane < n_splits ? tab_l[g][lane] : 0.0f;
      const float m_new = wave_max(m_s), m_safe = (m_new == -INFINITY) ? 0.0f : m_new, f = fast_exp2(m_s - m_safe);
      float       lf = l_s * f;
      asm("" : "+v"(lf));
      const float l_all = wave_sum(lf);
      tab_m[g][lane] = f;
      if (lane == 0) {
        tab_l[g][0] = l_all;
      }
    }
    float t0[PAIRS], t1[PAIRS];
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      t0[p] = t1[p] = 0.0f;
    }
    for (int split = 0; split < n_splits; ++split) {
      __syncthreads();  // (the factors are there; nobody reads the split before any more)
      walk(split, true);
#pragma unroll
      for (int p = 0; p < PAIRS; ++p) {
        const int i = 2 * ((int) threadIdx.x + p * THREADS), g = i / D;
        float     m_all, l, v0, v1;
        together(g, i % D, m_all, l, v0, v1);
        t0[p] = __builtin_fmaf(v0, tab_m[g][split], t0[p]), t1[p] = __builtin_fmaf(v1, tab_m[g][split], t1[p]);
      }
    }
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      const int i = 2 * ((int) threadIdx.x + p * THREADS), g = i / D, d = i % D, r = row0 + g;
      if (r >= rows) {
        continue;
      }
      const size_t at  = ((size_t) (r / group) * n_heads + h_kv * group + r % group) * D + d;
      const float  inv = 1.0f / tab_l[g][0];
      float        y0 = t0[p] * inv, y1 = t1[p] * inv;
      asm("" : "+v"(y0), "+v"(y1));
      if (QO_F32) {
        *reinterpret_cast<float2 *>(static_cast<float *>(out) + at) = make_float2(y0, y1);
      } else {
        *reinterpret_cast<v2h *>(static_cast<_Float16 *>(out) + at) = (v2h){ (_Float16) y0, (_Float16) y1 };
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------ any even head_dim

// Head dims the MFMA kernels above are not built for (even, but no multiple of 16; the reference routes head_dim % 64 != 0
// to its own variant, src/dsp/ops/flash_attn_sp_hdim.c:782-832, which only asks for an even head_dim). One workgroup
// per (query row, head); its four waves take every fourth 64-key block, with one key per lane for the scores (dot
// products of fp16 pairs, v_dot2_f32_f16) and one output column per lane (d = lane + 64 i) for O += p V, then merge their
// (max, sum, O) through LDS. Built for coverage, not speed: K rows are read straight from global memory.
constexpr int kGenThreads = 256;
constexpr int kGenMaxD    = 256;

template <bool QO_F32>
__global__ __launch_bounds__(kGenThreads) void flash_attn_any_dim_kernel(void *__restrict__ o_ptr,
                                                                         const void *__restrict__ q_ptr,
                                                                         const _Float16 *__restrict__ k_ptr,
                                                                         const _Float16 *__restrict__ v_ptr,
                                                                         const _Float16 *__restrict__ mask, int qo_len,
                                                                         int kv_len, int n_heads, int n_kv_heads,
                                                                         int head_dim, int flags) {
  const bool causal = (flags & 1) != 0, mask_threshold = (flags & 2) != 0;
  __shared__ v2h   q_sh[kGenMaxD / 2];
  __shared__ float part_o[4][kGenMaxD];
  __shared__ float part_ml[4][2];

  const int D     = head_dim;
  const int tid   = threadIdx.x;
  const int lane  = tid & 63;
  const int wave  = tid >> 6;
  const int row   = blockIdx.x;
  const int head  = blockIdx.y;
  const int h_kv  = head / (n_heads / n_kv_heads);
  const float scale = (1.0f / sqrtf((float) D)) * kLog2e;
  const size_t qo_base   = ((size_t) row * n_heads + head) * D;
  const size_t kv_stride = (size_t) n_kv_heads * D;
  const size_t mask_ld   = ((size_t) kv_len + 63) / 64 * 64;

  // the scaled query, rounded to fp16 like the MFMA kernels' B operand
  for (int i = tid; i < D / 2; i += kGenThreads) {
    float a, b;
    if (QO_F32) {
      a = reinterpret_cast<const float *>(q_ptr)[qo_base + 2 * i];
      b = reinterpret_cast<const float *>(q_ptr)[qo_base + 2 * i + 1];
    } else {
      a = (float) reinterpret_cast<const _Float16 *>(q_ptr)[qo_base + 2 * i];
      b = (float) reinterpret_cast<const _Float16 *>(q_ptr)[qo_base + 2 * i + 1];
    }
    q_sh[i] = v2h{ (_Float16) (a * scale), (_Float16) (b * scale) };
  }
  __syncthreads();

  const int kv_vis = causal ? min(kv_len, row + (kv_len - qo_len) + 1) : kv_len;  // keys 0 .. kv_vis - 1 are visible
  float m_run = -INFINITY, l_run = 0.0f;
  float acc[kGenMaxD / 64] = { 0.0f, 0.0f, 0.0f, 0.0f };
  for (int k0 = wave * 64; k0 < kv_vis; k0 += 4 * 64) {
    const int  key = k0 + lane;
    const bool on  = key < kv_vis;
    float      s   = -INFINITY;
    if (on) {
      const v2h *kr = reinterpret_cast<const v2h *>(k_ptr + (size_t) key * kv_stride + (size_t) h_kv * D);
      float      d0 = 0.0f, d1 = 0.0f;
      int        i  = 0;
      for (; i + 1 < D / 2; i += 2) {
        d0 = __builtin_amdgcn_fdot2(q_sh[i], kr[i], d0, false);
        d1 = __builtin_amdgcn_fdot2(q_sh[i + 1], kr[i + 1], d1, false);
      }
      if (i < D / 2) {
        d0 = __builtin_amdgcn_fdot2(q_sh[i], kr[i], d0, false);
      }
      s = d0 + d1;
      if (mask) {
        s += mask_term(mask[(size_t) row * mask_ld + key], mask_threshold);
      }
    }
    float mx = s;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      mx = fmaxf(mx, __shfl_xor(mx, off, kWave));
    }
    const float m_new  = fmaxf(m_run, mx);
    const float m_safe = (m_new == -INFINITY) ? 0.0f : m_new;  // everything masked so far: keep exp2 arguments finite
    const float alpha  = fast_exp2(m_run - m_safe);
    const float p      = fast_exp2(s - m_safe);  // 0 for hidden keys
    float       psum   = p;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      psum += __shfl_xor(psum, off, kWave);
    }
    l_run = l_run * alpha + psum;
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < kGenMaxD / 64; ++i) {
      acc[i] *= alpha;
    }
    const int n_keys = min(64, kv_vis - k0);
    for (int j = 0; j < n_keys; ++j) {
      const float     pj = __shfl(p, j, kWave);
      const _Float16 *vr = v_ptr + (size_t) (k0 + j) * kv_stride + (size_t) h_kv * D;
#pragma unroll
      for (int i = 0; i < kGenMaxD / 64; ++i) {
        const int d = lane + 64 * i;
        if (d < D) {
          acc[i] += pj * (float) vr[d];
        }
      }
    }
  }

  // merge the four waves
  if (lane == 0) {
    part_ml[wave][0] = m_run;
    part_ml[wave][1] = l_run;
  }
#pragma unroll
  for (int i = 0; i < kGenMaxD / 64; ++i) {
    part_o[wave][lane + 64 * i] = acc[i];
  }
  __syncthreads();
  float m_all = -INFINITY;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    m_all = fmaxf(m_all, part_ml[w][0]);
  }
  const float m_safe = (m_all == -INFINITY) ? 0.0f : m_all;
  float       l_all  = 0.0f;
  float       wgt[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    wgt[w] = fast_exp2(part_ml[w][0] - m_safe);
    l_all += wgt[w] * part_ml[w][1];
  }
  for (int d = tid; d < D; d += kGenThreads) {
    float o = 0.0f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      o += wgt[w] * part_o[w][d];
    }
    o /= l_all;
    if (QO_F32) {
      reinterpret_cast<float *>(o_ptr)[qo_base + d] = o;
    } else {
      reinterpret_cast<_Float16 *>(o_ptr)[qo_base + d] = (_Float16) o;
    }
  }
}

// The launch of a prefill: grid (x, q_blocks, splits). It follows the sizes alone, so that every entry point splits the keys
// of a request alike.
constexpr unsigned kCus = 256;
constexpr int prefill_key_groups(int dp) {  // the most that LDS and registers of a CU hold
  return dp <= 128 ? 2 : 1;
}
struct PrefillPlan {
  unsigned x, q_blocks, splits;
  size_t   tiles;  // of 32 queries of one head
};
PrefillPlan prefill_plan(int dp, int qo_len, int kv_len, int n_heads, int n_kv_heads, bool mask, int forced) {
  const int group      = n_heads / n_kv_heads;
  const int gc         = group < 4 ? group : 4;
  const int qsub       = 4 / gc;
  const int sub_groups = (group + gc - 1) / gc;
  PrefillPlan p;
  p.x        = (unsigned) (n_kv_heads * sub_groups);
  p.q_blocks = (unsigned) ((qo_len + qsub * kBQ - 1) / (qsub * kBQ));
  p.tiles    = (size_t) ((qo_len + kBQ - 1) / kBQ) * n_heads;
  p.splits   = 1;
  // Split the keys while that gives CUs without a workgroup one, down to two blocks per key group and workgroup, where the
  // blocks that the longest workgroup is spared take longer than the parts and their merge: a turn of the key groups
  // some 0.2 us and 0.96 us per 128 of the padded head dim, 0.35 us more with a mask; the merge 1 us and 0.3 us for every MB
  // of parts. (526 shapes of
  // 2 to 1000 rows over 100 to 6000 keys, 8 head layouts: within 4 % of the better one everywhere. 512 rows over 512 keys,
  // causal, 32 / 8 heads of 128, unsplit / split 14.8 / 22.3 us, over 2012 keys 36.7 / 34.6, with a mask
  // 46.1 / 36.6; 2 rows over 1502 keys 25.7 / 12.8.)
  const unsigned wgs = p.x * p.q_blocks;
  if (!forced && wgs <= kCus / 2) {
    const size_t share  = p.tiles * prefill_partial_floats(dp / 8) * sizeof(float);
    const size_t blocks = ((size_t) kv_len + kBK - 1) / kBK, groups = (size_t) prefill_key_groups(dp);
    const size_t most   = std::min({ (size_t) (kCus / wgs), blocks / (2 * groups), kAttnSharesBytes / share });
    // (for few tiles down to one block, while one trip of the merge takes all shares: 5 rows over 1029 keys, 12 tiles, of a head
    // dim of 128, which few_plan takes now, 14.4 -> 12.6 us; but 128 rows over 1152, 48 tiles, 17.5 -> 17.8, and 500 rows over 500, 256 tiles, 18.7 -> 20.2)
    const size_t finer  = std::min({ (size_t) (kCus / wgs), blocks / groups, kAttnSharesBytes / share, (size_t) kPfMergeChunk });
    const size_t splits = most < 2 ? 1 : p.tiles <= 32 ? std::max(most, finer) : most;
    const auto   turns  = [&](size_t n) { return (n + groups - 1) / groups; };
    const size_t spared = turns(blocks) - turns((blocks + splits - 1) / splits);
    if (spared * (200 + 15 * (size_t) dp / 2 + (mask ? 350 : 0)) > 1000 + splits * share * 3 / 10000) {  // (ns)
      p.splits = (unsigned) splits;
    }
  }
  return p;
}

// A few rows: (query, head) pairs of a GQA group in tiles of 16
struct FewPlan {
  int split = 0, n_splits = 0;  // split = 0: not this way
};
FewPlan few_plan(int qo_len, int kv_len, int n_heads, int n_kv_heads, int head_dim, bool mask, int forced) {
  FewPlan    p;
  // Two short launches against the one or two of the prefill kernel, 12 / 2, 32 / 8, 28 / 4 and 8 / 8 heads of 128 and 16 / 8 of
  // 64, prefill / here: 2 to 16 rows over 1029 keys with a mask 9.8 - 14.8 / 6.9 - 11.9 us, over 200 7.2 - 12.1 / 6.9 - 8.7; 3 rows
  // of 32 / 8 heads over 600 keys without one 10.6 / 8.1, but over 120 6.7 / 7.9: one prefill launch of few turns. Every row
  // tile reads the keys again, so that many of them over many keys lose: 16 rows of 32 / 8 heads over 3000 keys (768
  // workgroups) 18.7 / 16.0, over 6000 (1504) 19.8 / 23.1; and with more rows the prefill kernel's tiles of 32 are fuller: 48 rows of
  // 28 / 4 over 600 (420) 14.3 / 12.2, 64 of 12 / 2 over 1500 (576) 13.1 / 13.8.
  const long rows  = (long) qo_len * (n_heads / n_kv_heads);
  const int  least = head_dim == 64 ? (mask ? 200 : 512) : (mask ? 128 : 384);
  if (forced || qo_len < 2 || (head_dim != 64 && head_dim != 128) || kv_len < least || rows > 512 || n_kv_heads > 65535) {
    return p;
  }
  const long tiles = (rows + kFewRows - 1) / kFewRows;
  const bool small = (long) ((kv_len + kDecSplit - 1) / kDecSplit) * n_kv_heads * tiles < 128 && (kv_len + kDecSplitShort - 1) / kDecSplitShort <= kMergeChunk;
  const int  split = small ? kDecSplitShort : kDecSplit;
  const int  n     = (kv_len + split - 1) / split;
  if (n <= kMergeChunk && n * n_kv_heads * tiles <= (qo_len > 16 ? 512 : 768) &&
      (size_t) qo_len * n_heads * n * (head_dim + 2) * sizeof(float) <= kAttnSharesBytes) {
    p.split = split, p.n_splits = n;
  }
  return p;
}

template <int D, bool QO_F32>
hipError_t launch_few_rows(hipStream_t stream, FewPlan plan, void *o, const void *q, const void *k, const void *v, const void *mask,
                           int qo_len, int kv_len, int n_heads, int n_kv_heads, bool causal, bool mask_threshold, float *scratch,
                           void *q8_out) {
  const unsigned tiles = (unsigned) ((qo_len * (n_heads / n_kv_heads) + kFewRows - 1) / kFewRows);
  const dim3     grid(scratch ? (unsigned) plan.n_splits : 1u, (unsigned) n_kv_heads, tiles);
  const int      flags = (causal ? 1 : 0) | (mask_threshold ? 2 : 0);
  void          *out   = scratch ? scratch : o;
#define HTPOPS_FEW(SPLIT, ALL)                                                                                        \
  hipLaunchKernelGGL((flash_attn_few_rows_kernel<D, QO_F32, SPLIT, ALL>), grid, dim3(SPLIT / kDecWaveKeys * kWave), 0, stream, out, q, \
                     (const _Float16 *) k, (const _Float16 *) v, (const _Float16 *) mask, qo_len, kv_len, n_heads, n_kv_heads,     \
                     plan.n_splits, flags)
  if (plan.split == kDecSplit) {
    if (scratch) {
      HTPOPS_FEW(kDecSplit, false);
    } else {
      HTPOPS_FEW(kDecSplit, true);
    }
  } else if (scratch) {
    HTPOPS_FEW(kDecSplitShort, false);
  } else {
    HTPOPS_FEW(kDecSplitShort, true);
  }
#undef HTPOPS_FEW
  if (hipError_t e = hipGetLastError(); e != hipSuccess || !scratch) {
    return e;
  }
  hipLaunchKernelGGL((flash_attn_decode_merge_kernel<D, QO_F32, 1>), dim3((unsigned) (qo_len * n_heads)), dim3(D), 0, stream, o, scratch,
                     plan.n_splits, QO_F32 ? static_cast<uint8_t *>(q8_out) : nullptr);
  return hipGetLastError();
}

template <int DP, bool FULL, bool QO_F32>
hipError_t launch_prefill(hipStream_t stream, void *o, const void *q, const void *k, const void *v, const void *mask,
                          int qo_len, int kv_len, int n_heads, int n_kv_heads, int head_dim, bool causal, int forced,
                          bool mask_threshold, float *scratch, void *q8_out, void *act_fragments, ActOrder order) {
  const PrefillPlan plan = prefill_plan(DP, qo_len, kv_len, n_heads, n_kv_heads, mask != nullptr, forced);
  if (plan.q_blocks > 65535u) {
    return hipErrorInvalidValue;
  }
  constexpr int  kMaxGroups = prefill_key_groups(DP);
  const unsigned splits = plan.splits;
  const size_t   tiles  = plan.tiles;
  const bool     alone  = splits > 1 && scratch == nullptr;  // (a workgroup walks all shares)
  const dim3     grid(plan.x, plan.q_blocks, alone ? 1 : splits);
  // Two key groups per workgroup when the grid leaves CUs without a second workgroup, or (causal) when the workgroups
  // all fit at once and their uneven lengths would leave the long ones running alone. Measured on the 256-CU device,
  // 32 query / 8 KV heads of 128, ten calls behind idle: 2048 x 2048 causal 59 us against 65 us, 1024 x 1024 without `causal` 30
  // against 33 us; but 2048 x 2048 without `causal` 101 against 92 us. (A split grid never has more workgroups than CUs.)
  const unsigned all = plan.x * plan.q_blocks * splits;
  const bool     two = kMaxGroups == 2 && (forced ? forced == 2 : (all <= kCus || (causal && all <= 2 * kCus)));
  const int      flags = (causal ? 1 : 0) | (mask_threshold ? 2 : 0);
#define HTPOPS_LAUNCH(GROUPS, MASK, ALL)                                                                              \
  hipLaunchKernelGGL((flash_attn_prefill_kernel<DP, FULL, QO_F32, GROUPS, MASK, ALL>), grid, dim3(kPfThreads * GROUPS), 0, stream, \
                     o, q, (const _Float16 *) k, (const _Float16 *) v, (const _Float16 *) mask, qo_len, kv_len, n_heads, \
                     n_kv_heads, head_dim, flags, scratch, (int) splits)
  if (alone) {
    HTPOPS_LAUNCH(kMaxGroups, true, true);
  } else if (two && mask) {
    HTPOPS_LAUNCH(kMaxGroups, true, false);
  } else if (two) {
    HTPOPS_LAUNCH(kMaxGroups, false, false);
  } else if (mask) {
    HTPOPS_LAUNCH(1, true, false);
  } else {
    HTPOPS_LAUNCH(1, false, false);
  }
#undef HTPOPS_LAUNCH
  if (hipError_t e = hipGetLastError(); e != hipSuccess || splits == 1 || alone) {
    return e;
  }
  constexpr int kUnits = DP / 8;
  const ActFragments fragments = act_fragments_at(act_fragments, qo_len, n_heads * head_dim, order);
#define HTPOPS_MERGE(G, Q8, WORKGROUPS)                                                                               \
  hipLaunchKernelGGL((flash_attn_prefill_merge_kernel<QO_F32, G, Q8>), dim3((unsigned) (WORKGROUPS)), dim3(256), 0, stream, o, \
                     scratch, (int) splits, (int) tiles, kUnits, qo_len, n_heads, head_dim, static_cast<uint8_t *>(q8_out), \
                     fragments)
  if (splits > (unsigned) kPfMergeChunk) {
    HTPOPS_MERGE(4, -1, tiles * kUnits);
    return hipGetLastError();
  }
  if constexpr (QO_F32) {
    if (q8_out) {
      if (!act_fragments) {
        HTPOPS_MERGE(1, 0, tiles * kUnits / 4);
      } else if (order == kActFp6) {
        HTPOPS_MERGE(1, 1 + kActFp6, tiles * kUnits / 4);
      } else {
        HTPOPS_MERGE(1, 1 + kActI8, tiles * kUnits / 4);
      }
      return hipGetLastError();
    }
  }
  HTPOPS_MERGE(1, -1, (tiles * kUnits + 3) / 4);
#undef HTPOPS_MERGE
  return hipGetLastError();
}

template <int D, int GH, bool QO_F32, int SPLIT>
hipError_t launch_decode_pass(hipStream_t stream, dim3 grid, float *workspace, const void *q, const void *k, const void *v,
                              const void *mask, int kv_len, int n_heads, int n_kv_heads, int h0, int n_splits,
                              bool mask_threshold) {
  constexpr int    kWaves = SPLIT / kDecWaveKeys;
  // (the V rows; the waves' O, their sums and maxima)
  constexpr size_t kLds = (size_t) SPLIT * D * 2 + ((size_t) kWaves * GH * D + 2 * (size_t) kWaves * GH) * sizeof(float);
  static_assert(kLds <= 64 * 1024, "dynamic LDS without raising the limit");
  hipLaunchKernelGGL((flash_attn_decode_kernel<D, GH, QO_F32, SPLIT>), grid, dim3(kWaves * kWave), kLds, stream, workspace,
                     q, (const _Float16 *) k, (const _Float16 *) v, (const _Float16 *) mask, kv_len, n_heads, n_kv_heads,
                     h0, n_splits, mask_threshold ? 1 : 0);
  return hipGetLastError();
}

template <int D, bool QO_F32>
hipError_t launch_decode(hipStream_t stream, void *o, const void *q, const void *k, const void *v, const void *mask,
                         int kv_len, int n_heads, int n_kv_heads, float *workspace, void *q8_out, bool mask_threshold,
                         int parts = 3) {  // (bit 0: the split-KV launch, bit 1: the merge launch)
  const int  group    = n_heads / n_kv_heads;
  // 64-key chunks while 128-key ones would give fewer than 128 workgroups (measured at 8 KV heads: kv = 512 8.8 -> 7.1 us;
  // kv = 4096 and 16384 are 1 and 6 us slower with 64)
  const bool short_kv = (long) ((kv_len + kDecSplit - 1) / kDecSplit) * n_kv_heads < 128;
  const int  split    = short_kv ? kDecSplitShort : kDecSplit;
  const int  n_splits = (kv_len + split - 1) / split;
  const dim3 grid((unsigned) n_splits, (unsigned) n_kv_heads);
  for (int h0 = 0; h0 < group && (parts & 1); h0 += kDecMaxGroup) {
    const int  gh = group - h0;
    hipError_t e;
#define HTPOPS_DECODE(GH)                                                                                           \
  e = short_kv ? launch_decode_pass<D, GH, QO_F32, kDecSplitShort>(stream, grid, workspace, q, k, v, mask, kv_len, n_heads, \
                                                                  n_kv_heads, h0, n_splits, mask_threshold) :      \
                 launch_decode_pass<D, GH, QO_F32, kDecSplit>(stream, grid, workspace, q, k, v, mask, kv_len, n_heads,  \
                                                              n_kv_heads, h0, n_splits, mask_threshold)
    if (gh > 4) {
      HTPOPS_DECODE(8);
    } else if (gh > 2) {
      HTPOPS_DECODE(4);
    } else if (gh == 2) {
      HTPOPS_DECODE(2);
    } else {
      HTPOPS_DECODE(1);
    }
#undef HTPOPS_DECODE
    if (e != hipSuccess) {
      return e;
    }
  }
  if (!(parts & 2)) {
    return hipGetLastError();
  }
  uint8_t *q8 = QO_F32 ? static_cast<uint8_t *>(q8_out) : nullptr;
  if (n_splits > kMergeChunk) {
    hipLaunchKernelGGL((flash_attn_decode_merge_kernel<D, QO_F32, kMergeGroups>), dim3((unsigned) n_heads),
                       dim3(D * kMergeGroups), (size_t) kMergeGroups * (D + 2) * sizeof(float), stream, o, workspace,
                       n_splits, q8);
  } else {
    hipLaunchKernelGGL((flash_attn_decode_merge_kernel<D, QO_F32, 1>), dim3((unsigned) n_heads), dim3(D), 0, stream, o,
                       workspace, n_splits, q8);
  }
  return hipGetLastError();
}

}  // namespace

// (more rows than a few meet a matmul that wants them in operand order, which the quantizer leaves as well)
constexpr int kFewQ8Rows = 16;

namespace {

// Multiples of 16 fill the matrix instructions' k steps, and their rows (multiples of 32 bytes behind 16-byte aligned
// buffers) can be fetched 16 bytes at a time; every other even head dim, and more query blocks than a grid has rows, take
// the plain kernel. Head dims 64 and 128 have prefill (several rows) and decode (one row) kernels of their own.
bool takes_prefill(int qo_len, int head_dim) {
  return head_dim == 64 || head_dim == 128 ? qo_len > 1 : head_dim % 16 == 0 && qo_len <= 65535 * kBQ;
}

}  // namespace

bool flash_attn_writes_q8_0(int qo_len, int kv_len, int n_heads, int n_kv_heads, int head_dim, bool qo_is_f32, bool mask,
                            int forced_key_groups) {
  if (!qo_is_f32 || (qo_len == 1 && (head_dim == 64 || head_dim == 128))) {
    return qo_is_f32;
  }
  if (few_plan(qo_len, kv_len, n_heads, n_kv_heads, head_dim, mask, forced_key_groups).split != 0) {
    return qo_len <= kFewQ8Rows;
  }
  // a prefill whose shares are put together in one trip, whole blocks of a head to a workgroup
  if (!takes_prefill(qo_len, head_dim) || head_dim % 32 != 0) {
    return false;
  }
  const unsigned splits = prefill_plan(head_dim, qo_len, kv_len, n_heads, n_kv_heads, mask, forced_key_groups).splits;
  return splits > 1 && splits <= (unsigned) kPfMergeChunk;
}

size_t flash_attn_workspace_bytes(int qo_len, int kv_len, int n_heads, int head_dim) {
  if (qo_len != 1 || (head_dim != 64 && head_dim != 128)) {
    return 0;
  }
  const size_t n_splits = ((size_t) kv_len + kDecSplitShort - 1) / kDecSplitShort;  // the most there can be
  return (size_t) n_heads * n_splits * ((size_t) head_dim + 2) * sizeof(float);
}

bool flash_attn_splits_keys(int qo_len, int kv_len, int n_heads, int n_kv_heads, int head_dim, bool mask,
                            int forced_key_groups) {
  return few_plan(qo_len, kv_len, n_heads, n_kv_heads, head_dim, mask, forced_key_groups).split != 0 ||
         (takes_prefill(qo_len, head_dim) &&
          prefill_plan((head_dim + 31) / 32 * 32, qo_len, kv_len, n_heads, n_kv_heads, mask, forced_key_groups).splits > 1);
}

hipError_t launch_flash_attn_decode_part(hipStream_t stream, int part, void *o, const void *q, const void *k,
                                         const void *v, int kv_len, int n_heads, int n_kv_heads, int head_dim,
                                         bool qo_is_f32, void *workspace) {
  if ((head_dim != 64 && head_dim != 128) || (part != 1 && part != 2) || !workspace) {
    return hipErrorNotSupported;
  }
  float *ws = static_cast<float *>(workspace);
  if (head_dim == 128) {
    return qo_is_f32 ? launch_decode<128, true>(stream, o, q, k, v, nullptr, kv_len, n_heads, n_kv_heads, ws, nullptr, false, part) :
                       launch_decode<128, false>(stream, o, q, k, v, nullptr, kv_len, n_heads, n_kv_heads, ws, nullptr, false, part);
  }
  return qo_is_f32 ? launch_decode<64, true>(stream, o, q, k, v, nullptr, kv_len, n_heads, n_kv_heads, ws, nullptr, false, part) :
                     launch_decode<64, false>(stream, o, q, k, v, nullptr, kv_len, n_heads, n_kv_heads, ws, nullptr, false, part);
}

hipError_t launch_flash_attn(hipStream_t stream, void *o, const void *q, const void *k, const void *v,
                             const void *mask, int qo_len, int kv_len, int n_heads, int n_kv_heads, int head_dim,
                             bool qo_is_f32, bool causal, void *workspace, void *q8_out, int forced_key_groups,
                             bool mask_threshold, void *shares, void *act_fragments, ActOrder order) {
  // with a single query row the causal rule (key j visible iff j <= kv_len - 1) hides nothing
  if (qo_len == 1 && (head_dim == 64 || head_dim == 128)) {
    float *ws = static_cast<float *>(workspace);
    if (head_dim == 128) {
      return qo_is_f32 ? launch_decode<128, true>(stream, o, q, k, v, mask, kv_len, n_heads, n_kv_heads, ws, q8_out, mask_threshold) :
                         launch_decode<128, false>(stream, o, q, k, v, mask, kv_len, n_heads, n_kv_heads, ws, q8_out, mask_threshold);
    }
    return qo_is_f32 ? launch_decode<64, true>(stream, o, q, k, v, mask, kv_len, n_heads, n_kv_heads, ws, q8_out, mask_threshold) :
                       launch_decode<64, false>(stream, o, q, k, v, mask, kv_len, n_heads, n_kv_heads, ws, q8_out, mask_threshold);
  }
  const FewPlan few = few_plan(qo_len, kv_len, n_heads, n_kv_heads, head_dim, mask != nullptr, forced_key_groups);
  if (few.split != 0) {
    float *sh = static_cast<float *>(shares);
#define HTPOPS_FEW_ROWS(D, F32) \
  launch_few_rows<D, F32>(stream, few, o, q, k, v, mask, qo_len, kv_len, n_heads, n_kv_heads, causal, mask_threshold, sh, q8_out)
    return head_dim == 128 ? (qo_is_f32 ? HTPOPS_FEW_ROWS(128, true) : HTPOPS_FEW_ROWS(128, false)) :
                             (qo_is_f32 ? HTPOPS_FEW_ROWS(64, true) : HTPOPS_FEW_ROWS(64, false));
#undef HTPOPS_FEW_ROWS
  }
#define HTPOPS_PREFILL(DP, FULL)                                                                                     \
  qo_is_f32 ? launch_prefill<DP, FULL, true>(stream, o, q, k, v, mask, qo_len, kv_len, n_heads, n_kv_heads, head_dim, \
                                             causal, forced_key_groups, mask_threshold, static_cast<float *>(shares), q8_out, \
                                             act_fragments, order) :                                                  \
              launch_prefill<DP, FULL, false>(stream, o, q, k, v, mask, qo_len, kv_len, n_heads, n_kv_heads, head_dim, \
                                              causal, forced_key_groups, mask_threshold, static_cast<float *>(shares), q8_out, \
                                              act_fragments, order)
  if (head_dim == 128) {
    return HTPOPS_PREFILL(128, true);
  }
  if (head_dim == 64) {
    return HTPOPS_PREFILL(64, true);
  }
  if (head_dim <= 0 || head_dim % 2 != 0 || head_dim > kGenMaxD || n_heads > 65535) {
    return hipErrorNotSupported;
  }
  if (takes_prefill(qo_len, head_dim)) {
    switch ((head_dim + 31) / 32) {
      case 1: return HTPOPS_PREFILL(32, false);
      case 2: return HTPOPS_PREFILL(64, false);
      case 3: return HTPOPS_PREFILL(96, false);
      case 4: return HTPOPS_PREFILL(128, false);
      case 5: return HTPOPS_PREFILL(160, false);
      case 6: return HTPOPS_PREFILL(192, false);
      case 7: return HTPOPS_PREFILL(224, false);
      default: return HTPOPS_PREFILL(256, false);
    }
  }
#undef HTPOPS_PREFILL
  const dim3 grid((unsigned) qo_len, (unsigned) n_heads);
  if (qo_is_f32) {
    hipLaunchKernelGGL(flash_attn_any_dim_kernel<true>, grid, dim3(kGenThreads), 0, stream, o, q,
                       (const _Float16 *) k, (const _Float16 *) v, (const _Float16 *) mask, qo_len, kv_len, n_heads,
                       n_kv_heads, head_dim, (causal ? 1 : 0) | (mask_threshold ? 2 : 0));
  } else {
    hipLaunchKernelGGL(flash_attn_any_dim_kernel<false>, grid, dim3(kGenThreads), 0, stream, o, q,
                       (const _Float16 *) k, (const _Float16 *) v, (const _Float16 *) mask, qo_len, kv_len, n_heads,
                       n_kv_heads, head_dim, (causal ? 1 : 0) | (mask_threshold ? 2 : 0));
  }
  return hipGetLastError();
}

}  // namespace htpops
