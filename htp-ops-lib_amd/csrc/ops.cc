// The ops of the MI355X backend: request validation, kernel selection, launches.
//
// This is the replacement for execute_op_simple (reference: src/dsp/op_executor.cc:52-204): a request is validated on
// the host exactly where the reference rejects it (mat_mul.c:878-892, rms_norm.c:69-74, flash_attn.c:1373-1376) plus
// range checks the reference lacks, then its kernels are enqueued on the context's stream.
#include "context.h"

#include <algorithm>

namespace htpops {
namespace host {

// ---- op bodies on raw device pointers (validation that both the handle and the pointer entries share) ----

int op_rms_norm(htpops_context *ctx, float *dst, const float *src, const float *weight, float eps, int ne0, int ne1) {
  // reference: rms_norm.c:69-74 rejects null pointers, zero sizes and misaligned rows
  if (!dst || !src || ne0 <= 0 || ne1 <= 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm: null buffer or non-positive size (ne0=%d ne1=%d)", ne0, ne1);
  }
  if (!aligned(dst, 4) || !aligned(src, 4) || (weight && !aligned(weight, 4))) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm: buffers must be 4-byte aligned");
  }
  if (int r = need_device(ctx)) {
    return r;
  }
  note_device_write(ctx, dst, (size_t) ne0 * ne1 * 4);
  HTPOPS_HIP(ctx, launch_rms_norm_f32(ctx->stream, dst, src, weight, eps, ne0, ne1));
  return HTPOPS_OK;
}

namespace {

// where a quantizer of m rows of k leaves them in operand order as well (nullptr: nobody asked)
void wanted_fragments(htpops_context *ctx, int m, int k, void **where) {
  *where = nullptr;
  if (ctx->next_fragments_ws == 0 || (long long) m * (k / 32) > 0x7fffffffLL) {
    return;
  }
  // (no memory for what would only spare the matmul a launch: the rows are quantized without it)
  if (ensure_workspace(ctx, ctx->next_fragments_ws) == HTPOPS_OK) {
    *where = ctx->workspace;
  }
}

ActOrder next_order(const htpops_context *ctx) {
  return ctx->next_fragments_kind == (int) kPlanLdsFp6 ? kActFp6 : kActI8;
}

void note_fragments(htpops_context *ctx, const void *where, const void *rows, int m, int k) {
  if (where) {
    auto &af = ctx->act_fragments;
    af.src = rows, af.src_bytes = q8_0_bytes((size_t) m, (size_t) k), af.m = m, af.k = k, af.kind = ctx->next_fragments_kind;
  }
}

}  // namespace

int op_quantize(htpops_context *ctx, void *dst, const float *src, int k, int m) {
  if (!dst || !src || k <= 0 || m <= 0 || k % 32 != 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "quantize_q8_0: null buffer or bad size (k=%d m=%d, k %% 32 must be 0)", k, m);
  }
  if (!aligned(dst, 4) || !aligned(src, 16)) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "quantize_q8_0: src must be 16-byte and dst 4-byte aligned");
  }
  if (int r = need_device(ctx)) {
    return r;
  }
  void *frags = nullptr;
  wanted_fragments(ctx, m, k, &frags);
  note_device_write(ctx, dst, q8_0_bytes((size_t) m, (size_t) k));
  HTPOPS_HIP(ctx, launch_quantize_q8_0(ctx->stream, dst, src, k, m, frags, next_order(ctx)));
  note_fragments(ctx, frags, dst, m, k);
  return HTPOPS_OK;
}

int op_rms_norm_quantize(htpops_context *ctx, void *dst, const float *src, const float *weight, float eps, int ne0,
                         int ne1) {
  if (!dst || !src || ne0 <= 0 || ne1 <= 0 || ne0 % 32 != 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm_quantize: null buffer or bad size (ne0=%d ne1=%d)", ne0, ne1);
  }
  if (!aligned(dst, 4) || !aligned(src, 16) || (weight && !aligned(weight, 16))) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm_quantize: src/weight must be 16-byte and dst 4-byte aligned");
  }
  if (int r = need_device(ctx)) {
    return r;
  }
  if (ne0 <= 16384) {
    void *frags = nullptr;
    wanted_fragments(ctx, ne1, ne0, &frags);
    note_device_write(ctx, dst, q8_0_bytes((size_t) ne1, (size_t) ne0));
    HTPOPS_HIP(ctx, launch_rms_norm_quantize_q8_0(ctx->stream, dst, src, weight, eps, ne0, ne1, frags, next_order(ctx)));
    note_fragments(ctx, frags, dst, ne1, ne0);
    return HTPOPS_OK;
  }
  // very long rows: normalize into the workspace, then quantize
  size_t bytes;
  if (!mul3((size_t) ne0, (size_t) ne1, 4, &bytes)) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm_quantize: size overflow");
  }
  if (int r = ensure_workspace(ctx, bytes)) {
    return r;
  }
  note_device_write(ctx, dst, q8_0_bytes((size_t) ne1, (size_t) ne0));
  HTPOPS_HIP(ctx, launch_rms_norm_f32(ctx->stream, (float *) ctx->workspace, src, weight, eps, ne0, ne1));
  HTPOPS_HIP(ctx, launch_quantize_q8_0(ctx->stream, dst, (const float *) ctx->workspace, ne0, ne1));
  return HTPOPS_OK;
}

namespace {

int check_mat_mul(htpops_context *ctx, const void *dst, const void *act, const void *weight, int m, int k, int n,
                  int weight_type) {
  // reference: mat_mul.c:878-892
  if (!dst || !act || !weight || m <= 0 || k <= 0 || n <= 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul: null buffer or non-positive size (m=%d k=%d n=%d)", m, k, n);
  }
  if (k % 32 != 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul: k=%d is not a multiple of 32", k);
  }
  if (weight_type != kQ4_0 && weight_type != kQ8_0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul: unsupported weight type %d", weight_type);
  }
  if (!aligned(dst, 4) || !aligned(act, 2) || !aligned(weight, 2)) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul: misaligned buffer");
  }
  return HTPOPS_OK;
}

}  // namespace

// (*out stays nullptr when this matmul does not take the repacked-weight kernel: shape, weight type, activations not
// 16-byte aligned for the DMA into LDS, weights in memory whose copies may not be kept; the caller then uses the
// kernels that read the weights as they are. A failed allocation or conversion launch is an error, not a reason to
// switch kernels.)
bool prefers_block_pairs(const htpops_context *ctx, int m, int k, int n, int wt) {
  return (m == 2 || m == 3) && wt == kQ4_0 && ctx->opt.lane_order == 1 && matmul_block_pairs_fits(n, m, k, (WeightType) wt);
}

int lane_order_weights(htpops_context *ctx, const void *weight, const void *act, int m, int k, int n, int wt,
                       const void **out, bool *block_pairs) {
  *out         = nullptr;
  *block_pairs = ctx->opt.lane_order == 1 && matmul_block_pairs_fits(n, m, k, (WeightType) wt);
  if (ctx->opt.lane_order == 0 || !aligned(act, 16) ||
      !(*block_pairs || matmul_lane_order_fits(n, m, k, (WeightType) wt))) {
    return HTPOPS_OK;
  }
  const int kind = (*block_pairs ? kFragKindBlockPairs : kFragKindLaneOrder) + wt;
  if ((*out = find_copy(ctx, weight, kind, k, n)) != nullptr) {
    return HTPOPS_OK;
  }
  const size_t w_bytes = weight_bytes((size_t) n, (size_t) k, wt);
  if (!may_keep_copies(ctx, weight, w_bytes)) {
    return HTPOPS_OK;
  }
  void *fresh = nullptr;
  if (int r = new_copy(ctx, weight, w_bytes, kind, k, n, matmul_lane_order_weight_bytes(k, n, (WeightType) wt), &fresh)) {
    return r;
  }
  const hipError_t e = *block_pairs ? launch_weights_to_block_pairs(ctx->stream, fresh, weight, k, n, (WeightType) wt) :
                                      launch_weights_to_lane_order(ctx->stream, fresh, weight, k, n, (WeightType) wt);
  if (e != hipSuccess) {
    forget_copy(ctx, fresh);
    return hip_fail(ctx, e, "weight repack launch");
  }
  *out = fresh;
  return HTPOPS_OK;
}

// `act_aligned`: the Q8_0 activations start on a 4-byte boundary (the re-tiling pass of the FP6 kernel reads dwords)
// `overwrites`: the output lies over the weights (or, up to 32 rows, over the rows), so no copy of them is used or kept (one is
// made in the workspace, in order)
MatMulPlan plan_mat_mul(htpops_context *ctx, const void *weight, bool act_aligned, int m, int k, int n, int wt, bool overwrites) {
  MatMulPlan p;
  if (m < kManyRowsMinM || k % 32 != 0) {
    p.ws_bytes = mat_mul_workspace_bytes(m, k, n);
    return p;
  }
  auto lookup_copy = [&](int frag_kind) {
    p.frag_kind = frag_kind;
    p.cached    = overwrites ? nullptr : find_copy(ctx, weight, frag_kind, k, n);
    p.cacheable = !overwrites && !p.cached && may_keep_copies(ctx, weight, weight_bytes((size_t) n, (size_t) k, wt));
  };
  // Q4_0 weights whose converted copy may be kept, on a shape whose output tiles fill the device: the FP6 kernel over
  // that copy (half the vector-ALU work per block sum of the int8 path). Registered memory that was never prepared
  // (htpops_buffer_prepare_weights) may change behind the context's back, so nothing converted from it is kept, and
  // the FP6 conversion is too slow to redo per call.
  const int use_fp6 = ctx->opt.gemm_fp6;
  if (m >= kFp6MinM && wt == kQ4_0 && use_fp6 != 0 && gemm_fp6_lds_fits(m, k, n) && aligned(weight, 4) && act_aligned &&
      (use_fp6 > 0 || gemm_fp6_lds_fills_device(m, n))) {
    lookup_copy(kFragKindFp6Tiles + wt);
    if (p.cached || p.cacheable) {
      p.kind         = kPlanLdsFp6;
      p.act_bytes    = (gemm_fp6_lds_act_tile_bytes(m, k) + 255) & ~(size_t) 255;
      p.weight_bytes = gemm_fp6_lds_weight_tile_bytes(k, n);
      p.ws_bytes     = p.act_bytes;
      return p;
    }
  }
  // Up to 32 rows only over a copy that is kept: the kernels that read the weights as they are beat a conversion per call. And
  // only over one that needs no room another copy has (a cap on all of them): those kernels need none. And only large matrices
  // or long K (gemm_tile_units set: any). 17 rows of Q8_0 behind their quantizer, K-sliced kernel / here: k = 512 to 2048 and n
  // up to 2048 6.8 - 10.1 / 8.8 - 11.0 us; k = 4096 and n up to 2048 10.0 - 10.9 / 10.2 - 10.7, and the rows of one layer's q, k
  // and v should meet one kernel; k = 2048, n = 4096 10.5 / 11.2, k = 1536, n = 8960 14.8 / 12.4, k = n = 4096 13.6 / 11.2, k =
  // 8960, n = 1536 13.7 / 11.6, k = n = 8960 39 / 31. Layers of hidden 512 / 1024 / 1536 / 2048 with the line there, against
  // all matrices here, 41 / 46 / 57 / 56 and 48 / 51 / 59 / 59 us. What it costs: a message whose matrices are all ready and
  // fall on both sides takes two launches (seven projections of hidden 1536 24.8 against 17.6 us; seven K-sliced ones 65).
  if (m < kFp6MinM && !overwrites) {
    const bool large = k >= 4096 || (size_t) n * k > (size_t) 4 << 20 || ctx->opt.gemm_tile_units != 0;
    if (large) {
      lookup_copy(kFragKindRowLayout + wt);
    }
    if (!p.cached && !(p.cacheable && copy_fits_cap(ctx, (gemm_i8_weight_fragment_bytes(k, n) + 255) & ~(size_t) 255))) {
      p.cacheable = false;
      p.ws_bytes = mat_mul_workspace_bytes(m, k, n);
      return p;
    }
  }
  p.kind         = kPlanFragments;
  p.act_bytes    = (gemm_i8_act_fragment_bytes(m, k) + 255) & ~(size_t) 255;
  p.weight_bytes = (gemm_i8_weight_fragment_bytes(k, n) + 255) & ~(size_t) 255;
  lookup_copy(kFragKindRowLayout + wt);
  p.ws_bytes = p.act_bytes + ((p.cached || p.cacheable) ? 0 : p.weight_bytes) +
               ((gemm_i8_fragments_exchange_bytes(m, n, k, ctx->opt.gemm_tile_units) + 255) & ~(size_t) 255);
  return p;
}

int plan_weight_copy(htpops_context *ctx, MatMulPlan &plan, const void *weight, int k, int n, int wt, const void **out) {
  *out = plan.cached;
  if (plan.cached || !plan.cacheable || plan.kind == kPlanFewRows) {
    return HTPOPS_OK;
  }
  void *fresh = nullptr;
  if (int r = new_copy(ctx, weight, weight_bytes((size_t) n, (size_t) k, wt), plan.frag_kind, k, n, plan.weight_bytes, &fresh)) {
    return r;
  }
  const hipError_t e = plan.kind == kPlanLdsFp6 ? launch_q4_0_to_fp6_tiles(ctx->stream, fresh, weight, k, n) :
                                                  launch_weights_to_i8_fragments(ctx->stream, fresh, weight, k, n, (WeightType) wt);
  if (e != hipSuccess) {
    forget_copy(ctx, fresh);
    return fail(ctx, HTPOPS_ERR_HIP, "weight conversion: %s", hipGetErrorString(e));
  }
  plan.cached = fresh, plan.cacheable = false;
  *out = fresh;
  return HTPOPS_OK;
}

namespace {

// Up to 32 rows a copy only buys speed: where there is no memory for it, the matmul takes the kernels that read the weights
// as they are.
void settle_copy(htpops_context *ctx, MatMulPlan &plan, const void *weight, int m, int k, int n, int wt) {
  const void *copy = nullptr;
  if (plan.kind == kPlanFragments && m < kFp6MinM && plan.cacheable &&
      plan_weight_copy(ctx, plan, weight, k, n, wt, &copy) != HTPOPS_OK) {
    plan          = MatMulPlan();
    plan.ws_bytes = mat_mul_workspace_bytes(m, k, n);
  }
}

int run_few_rows(htpops_context *ctx, float *dst, const void *act, const void *weight, int m, int k, int n, int wt,
                 uint8_t *ws) {
  // hipErrorNotSupported from a launcher means "this kernel does not take the shape": try the next one. Any other
  // failure is reported.
  const void *lw    = nullptr;
  bool        pairs = false;
  if (prefers_block_pairs(ctx, m, k, n, wt)) {
    if (int r = lane_order_weights(ctx, weight, act, m, k, n, wt, &lw, &pairs)) {
      return r;
    }
  }
  if (!lw && ctx->opt.gemv_rows_kernel != 0 && gemv_rows_fits(m, k, (WeightType) wt) && aligned(act, 4) && aligned(weight, 4)) {
    const hipError_t e = launch_gemv_rows_group_q8_0_act(ctx->stream, 1, &dst, &act, &weight, &n, m, &k,
                                                                 (WeightType) wt);
    if (e == hipSuccess) {
      return HTPOPS_OK;
    }
    if (e != hipErrorNotSupported) {
      return hip_fail(ctx, e, "few-row mat_mul launch");
    }
    (void) hipGetLastError();
  }
  if (!lw) {
    if (int r = lane_order_weights(ctx, weight, act, m, k, n, wt, &lw, &pairs)) {
      return r;
    }
  }
  if (lw) {
    const hipError_t e = pairs ? launch_matmul_block_pairs_group(ctx->stream, 1, &dst, &act, &lw, &n, m, &k, (WeightType) wt) :
                                 launch_matmul_lane_order_group(ctx->stream, 1, &dst, &act, &lw, &n, m, k, (WeightType) wt,
                                                                ctx->opt.lane_order);
    if (e == hipSuccess) {
      return HTPOPS_OK;
    }
    if (e != hipErrorNotSupported) {
      return hip_fail(ctx, e, "repacked-weight mat_mul launch");
    }
    (void) hipGetLastError();
  }
  HTPOPS_HIP(ctx, launch_mat_mul_q8_0_act(ctx->stream, dst, act, weight, m, k, n, (WeightType) wt, ws,
                                                  ctx->tickets, kTicketSlots));
  return HTPOPS_OK;
}

bool writes_weights(const void *dst, const void *weight, int m, int k, int n, int wt) {
  return ranges_overlap(dst, (size_t) m * n * 4, weight, weight_bytes((size_t) n, (size_t) k, wt));
}

// `ws` is this matmul's share of the workspace (plan.ws_bytes, already ensured by the caller, who has noted the write to `dst`
// before planning: it drops copies). act = nullptr (int8 fragments only): the activations lie at its start in operand order
// already.
int run_mat_mul(htpops_context *ctx, MatMulPlan &plan, float *dst, const void *act, const void *weight, int m, int k,
                int n, int wt, uint8_t *ws) {
  if (plan.kind == kPlanFewRows) {
    ctx->act_fragments.src = nullptr;  // these kernels put something else at the start of the workspace
    const int r = run_few_rows(ctx, dst, act, weight, m, k, n, wt, ws);
    if (writes_weights(dst, weight, m, k, n, wt)) {  // a copy made just now is of weights that are gone
      note_device_write(ctx, dst, (size_t) m * n * 4);
    }
    return r;
  }
  // the converted copy of the weights, for the kernels that want one: kept with the buffer, or (weights whose copies
  // may not be kept; int8 fragments only) made in the workspace for this call
  const void *frags = nullptr;
  if (int r = plan_weight_copy(ctx, plan, weight, k, n, wt, &frags)) {
    return r;
  }
  if (!frags) {
    void            *fresh = ws + plan.act_bytes;
    const hipError_t e     = launch_weights_to_i8_fragments(ctx->stream, fresh, weight, k, n, (WeightType) wt);
    if (e != hipSuccess) {
      return fail(ctx, HTPOPS_ERR_HIP, "weight conversion: %s", hipGetErrorString(e));
    }
    frags = fresh;
  }
  // The converted activations at the start of the workspace are shared by the requests of a message that read the same
  // rows with the same kernel family (note_device_write has already cleared the record if this matmul writes into its own
  // activations).
  auto      &af    = ctx->act_fragments;
  const bool ready = !act || (af.src == act && af.m == m && af.k == k && af.kind == (int) plan.kind && ws == ctx->workspace);
  const bool keep  = act && (ready || (ctx->in_message && ws == ctx->workspace &&
                               !ranges_overlap(dst, (size_t) m * n * 4, act, q8_0_bytes((size_t) m, (size_t) k))));
  af.src = nullptr;
  if (plan.kind == kPlanLdsFp6) {
    HTPOPS_HIP(ctx, launch_gemm_fp6_lds(ctx->stream, dst, act, frags, m, k, n, ws, ready));
  } else {
    // (scratch for partial tiles at the end of this matmul's share of the workspace)
    const size_t xbytes = gemm_i8_fragments_exchange_bytes(m, n, k, ctx->opt.gemm_tile_units);
    HTPOPS_HIP(ctx, launch_gemm_i8_fragments(ctx->stream, dst, act, frags, m, k, n, ws, ready,
                                             ws + plan.ws_bytes - ((xbytes + 255) & ~(size_t) 255), xbytes, ctx->tickets,
                                             kTicketSlots, ctx->opt.gemm_tile_units));
  }
  if (keep) {
    af.src = act, af.src_bytes = q8_0_bytes((size_t) m, (size_t) k), af.m = m, af.k = k, af.kind = (int) plan.kind;
  }
  return HTPOPS_OK;
}

}  // namespace

int op_mat_mul_q8(htpops_context *ctx, float *dst, const void *act, const void *weight, int m, int k, int n,
                  int weight_type) {
  if (int r = check_mat_mul(ctx, dst, act, weight, m, k, n, weight_type)) {
    return r;
  }
  if (int r = need_device(ctx)) {
    return r;
  }
  note_device_write(ctx, dst, (size_t) m * n * 4);
  // (17 to 32 rows under the output are put into operand order first, like their weights: the K-sliced kernel reads rows while
  // other workgroups store. More rows always are.)
  const bool overwrites = writes_weights(dst, weight, m, k, n, weight_type) ||
                          (m < kFp6MinM && ranges_overlap(dst, (size_t) m * n * 4, act, q8_0_bytes((size_t) m, (size_t) k)));
  MatMulPlan plan = plan_mat_mul(ctx, weight, aligned(act, 4), m, k, n, weight_type, overwrites);
  settle_copy(ctx, plan, weight, m, k, n, weight_type);
  if (int r = ensure_workspace(ctx, plan.ws_bytes, /*keep_act_fragments=*/true)) {
    return r;
  }
  return run_mat_mul(ctx, plan, dst, act, weight, m, k, n, weight_type, static_cast<uint8_t *>(ctx->workspace));
}

int op_mat_mul_f32(htpops_context *ctx, float *dst, const float *act, const void *weight, int m, int k, int n,
                   int weight_type) {
  if (int r = check_mat_mul(ctx, dst, act, weight, m, k, n, weight_type)) {
    return r;
  }
  if (!aligned(act, 16)) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul: fp32 activations must be 16-byte aligned");
  }
  if (int r = need_device(ctx)) {
    return r;
  }
  note_device_write(ctx, dst, (size_t) m * n * 4);
  MatMulPlan plan = plan_mat_mul(ctx, weight, true, m, k, n, weight_type, writes_weights(dst, weight, m, k, n, weight_type));
  settle_copy(ctx, plan, weight, m, k, n, weight_type);
  if ((plan.kind == kPlanFragments || plan.kind == kPlanLdsFp6) && (long long) m * (k / 32) <= 0x7fffffffLL) {
    // the quantizer writes the operand order the matmul wants: the rows in block_q8_0 form would have one reader, another
    // launch that puts them into that order (33 rows, k = 8960, n = 1537: 3 of 18 us; 512 rows,
    // Q4_0, 4096 x 4096: 31.4 -> 29.1 us)
    if (int r = ensure_workspace(ctx, plan.ws_bytes)) {
      return r;
    }
    HTPOPS_HIP(ctx, launch_quantize_q8_0(ctx->stream, nullptr, act, k, m, ctx->workspace,
                                         plan.kind == kPlanLdsFp6 ? kActFp6 : kActI8));
    return run_mat_mul(ctx, plan, dst, nullptr, weight, m, k, n, weight_type, static_cast<uint8_t *>(ctx->workspace));
  }
  // workspace: [quantized activations][what the matmul itself needs]
  const size_t q_bytes = (q8_0_bytes((size_t) m, (size_t) k) + 255) & ~(size_t) 255;
  if (int r = ensure_workspace(ctx, q_bytes + plan.ws_bytes)) {
    return r;
  }
  uint8_t *ws = static_cast<uint8_t *>(ctx->workspace);
  HTPOPS_HIP(ctx, launch_quantize_q8_0(ctx->stream, ws, act, k, m));
  return run_mat_mul(ctx, plan, dst, ws, weight, m, k, n, weight_type, ws + q_bytes);
}

// The weights are read in their own formats at every row count: a converted copy would be up to 3.6 times the bytes.
int op_mat_mul_permuted_group(htpops_context *ctx, const PermutedMatMul *members, int count, int m, int kind) {
  for (int i = 0; i < count; ++i) {
    note_device_write(ctx, members[i].out, (size_t) m * members[i].n * 4);
  }
  const bool   few   = m <= kPermutedRowsMax;
  const size_t bytes = few ? permuted_rows_workspace_bytes(members, count, m) : permuted_gemm_workspace_bytes(members, count, m);
  // The kernels read rows and weights while other workgroups of the launch store results. A result that lies over either (only
  // a request by itself: the members of a batch leave each other's buffers alone) is made behind the workspace and copied.
  PermutedMatMul aside     = members[0];
  float *const   where     = aside.out;
  const size_t   out_bytes = (size_t) m * aside.n * 4, w_bytes = permuted_weight_bytes((size_t) aside.n, (size_t) aside.k, kind);
  const bool     overlaps  = count == 1 && (ranges_overlap(where, out_bytes, aside.act, (size_t) m * aside.k * 4) ||
                                        ranges_overlap(where, out_bytes, aside.weight, w_bytes));
  if (bytes > 0 || overlaps) {  // (rows that fit LDS need none, and leave what lies there alone)
    if (int r = ensure_workspace(ctx, bytes + (overlaps ? out_bytes : 0))) {
      return r;
    }
  }
  if (overlaps) {
    aside.out = reinterpret_cast<float *>(static_cast<uint8_t *>(ctx->workspace) + bytes);
    members   = &aside;
  }
  hipError_t e = few ? hipErrorNotSupported : launch_permuted_gemm_group(ctx->stream, members, count, m, kind, ctx->workspace, ctx->tickets);
  if (e == hipErrorNotSupported) {
    e = hipSuccess;
    for (int m0 = 0; m0 < m && e == hipSuccess; m0 += kPermutedRowsMax) {  // (once, but for a K that the other cannot address)
      PermutedMatMul part[kPermutedGroupMax];
      for (int i = 0; i < count; ++i) {
        part[i] = members[i];
        part[i].out += (size_t) m0 * part[i].n, part[i].act += (size_t) m0 * part[i].k;
      }
      e = launch_permuted_rows_group(ctx->stream, part, count, std::min(m - m0, kPermutedRowsMax), kind, ctx->workspace);
    }
  }
  HTPOPS_HIP(ctx, e);
  if (overlaps) {
    HTPOPS_HIP(ctx, launch_copy_results(ctx->stream, where, aside.out, out_bytes));
  }
  return HTPOPS_OK;
}

// hmx_mat_mul_permuted_w16a32 / hmx_mat_mul_permuted_qk_0_d16a32 (reference: src/dsp/ops/mat_mul.c:758-855, :875-1153)
int op_mat_mul_permuted(htpops_context *ctx, float *dst, const float *act, const void *weight, int m, int k, int n,
                        int kind) {
  // reference: mat_mul.c:760-769, :878-892
  if (!dst || !act || !weight || m <= 0 || k <= 0 || n <= 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul_permuted: null buffer or non-positive size (m=%d k=%d n=%d)", m, k, n);
  }
  if (k % 32 != 0 || n % 32 != 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul_permuted: k=%d and n=%d must be multiples of 32", k, n);
  }
  if (!aligned(dst, 128) || !aligned(act, 128) || !aligned(weight, 128)) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul_permuted: buffers must be 128-byte aligned");
  }
  if (int r = need_device(ctx)) {
    return r;
  }
  const PermutedMatMul one = { dst, act, weight, k, n };
  return op_mat_mul_permuted_group(ctx, &one, 1, m, kind);
}

namespace {

// Where shared keys meet, or nullptr: a caller is capturing the stream (or there was no memory). A graph of theirs may be
// launched beside the context's own work, or after the context is closed, so it must not hold an address of the context's.
// A recording of the context's own is launched on its stream only.
void *attention_shares(htpops_context *ctx) {
  const bool             recording = ctx->collect_ranges != nullptr;
  hipStreamCaptureStatus status    = hipStreamCaptureStatusNone;
  if (!recording && hipStreamIsCapturing(ctx->stream, &status) != hipSuccess) {
    (void) hipGetLastError();
    return nullptr;
  }
  return recording || status == hipStreamCaptureStatusNone ? ctx->attn_shares : nullptr;
}

}  // namespace

int op_flash_attn(htpops_context *ctx, void *o, const void *q, const void *k, const void *v, const void *mask,
                  int qo_len, int kv_len, int n_heads, int n_kv_heads, int head_dim, int qo_is_f32, int causal,
                  bool no_alloc) {
  if (!o || !q || !k || !v || qo_len <= 0 || kv_len <= 0 || n_heads <= 0 || n_kv_heads <= 0 || head_dim <= 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "flash_attn: null buffer or non-positive size");
  }
  // reference: flash_attn.c:1373-1376
  if (n_heads % n_kv_heads != 0) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "flash_attn: n_heads=%d is not a multiple of n_kv_heads=%d", n_heads,
                n_kv_heads);
  }
  // reference: flash_attn_sp_hdim.c:785-788 (an odd head_dim is refused)
  if (head_dim % 2 != 0 || head_dim > 256) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "flash_attn: head_dim=%d (even values up to 256 are built)", head_dim);
  }
  if (!aligned(o, 16) || !aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) || (mask && !aligned(mask, 8))) {
    return fail(ctx, HTPOPS_ERR_REJECTED, "flash_attn: q/k/v/o must be 16-byte aligned, the mask 8-byte aligned");
  }
  if (int r = need_device(ctx)) {
    return r;
  }
  const size_t ws_bytes = flash_attn_workspace_bytes(qo_len, kv_len, n_heads, head_dim);
  const size_t o_bytes  = (size_t) qo_len * n_heads * head_dim * (qo_is_f32 ? 4 : 2);
  void        *ws       = nullptr;
  if (no_alloc) {
    // nothing may be allocated or freed here: the partials go to this device's static scratch array, and an output
    // that would overwrite weights with a converted copy (whose release is a hipFree) is refused instead
    if (ws_bytes > kNoAllocScratchBytes) {
      return fail(ctx, HTPOPS_ERR_REJECTED,
                  "flash_attn (no allocation): %zu bytes of split-KV partials exceed the %zu-byte static scratch "
                  "(n_heads * ceil(kv_len / 64) * (head_dim + 2) * 4 must fit)", ws_bytes, kNoAllocScratchBytes);
    }
    for (const auto &e : ctx->frag_cache) {
      if (ranges_overlap(o, o_bytes, e.src, e.src_bytes)) {
        return fail(ctx, HTPOPS_ERR_REJECTED, "flash_attn (no allocation): the output overlaps cached weights");
      }
    }
    if (ctx->act_fragments.src && ranges_overlap(o, o_bytes, ctx->act_fragments.src, ctx->act_fragments.src_bytes)) {
      ctx->act_fragments.src = nullptr;
    }
    if (ws_bytes > 0 && !claim_static_scratch(ctx)) {
      return fail(ctx, HTPOPS_ERR_BUSY,
                  "flash_attn (no allocation): another context on this GPU is using the static scratch and has not "
                  "synchronized since");
    }
    ws = ctx->scratch_ptr;
  } else {
    if (int r = ensure_workspace(ctx, ws_bytes)) {
      return r;
    }
    note_device_write(ctx, o, o_bytes);
    ws = ctx->workspace;
  }
  void *shares = nullptr;
  if (flash_attn_splits_keys(qo_len, kv_len, n_heads, n_kv_heads, head_dim, mask != nullptr, ctx->opt.attn_key_groups)) {
    shares = attention_shares(ctx);
  }
  void *q8_out = nullptr;
  if (ctx->attn_q8_out && (qo_len == 1 || shares) &&
      flash_attn_writes_q8_0(qo_len, kv_len, n_heads, n_kv_heads, head_dim, qo_is_f32 != 0, mask != nullptr,
                             ctx->opt.attn_key_groups)) {
    q8_out = ctx->attn_q8_out;
    note_device_write(ctx, q8_out, q8_0_bytes((size_t) qo_len, (size_t) n_heads * head_dim));
  }
  // (17 rows and more, whose kernel needs no workspace of its own)
  void *frags = nullptr;
  if (q8_out && !ws_bytes) {
    wanted_fragments(ctx, qo_len, n_heads * head_dim, &frags);
  }
  HTPOPS_HIP(ctx, launch_flash_attn(ctx->stream, o, q, k, v, mask, qo_len, kv_len, n_heads, n_kv_heads, head_dim,
                                    qo_is_f32 != 0, causal != 0, ws, q8_out, ctx->opt.attn_key_groups,
                                    ctx->opt.attn_mask_threshold != 0, shares, frags, next_order(ctx)));
  note_fragments(ctx, frags, q8_out, qo_len, n_heads * head_dim);
  ctx->attn_q8_done = q8_out != nullptr;
  return HTPOPS_OK;
}


}  // namespace host
}  // namespace htpops

using namespace htpops;
using namespace htpops::host;

// ------------------------------------------------------------------------------------------------ ops

extern "C" int htpops_execute_op(htpops_context *ctx, const struct OpComputeRequest *req) {
  if (!ctx || !req) {
    return HTPOPS_ERR_REJECTED;
  }
  Lock lock(ctx->mu);
  if (!ctx->in_message) {
    ++ctx->use_serial;
  }
  switch (req->op) {
    case HTP_OPS_RMS_NORM_F32:
      {
        // reference: op_executor.cc:82-94
        const auto *p = reinterpret_cast<const RmsNormF32Params *>(req->payload);
        size_t      bytes;
        if (p->ne0 <= 0 || p->ne1 <= 0 || !mul3((size_t) p->ne0, (size_t) p->ne1, 4, &bytes)) {
          return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm: bad size (ne0=%d ne1=%d)", p->ne0, p->ne1);
        }
        return op_rms_norm(ctx, (float *) resolve(ctx, p->dst, bytes), (const float *) resolve(ctx, p->src, bytes),
                           nullptr, 1e-5f, p->ne0, p->ne1);
      }
    case HTP_OPS_RMS_NORM_F32_EX:
    case HTP_OPS_RMS_NORM_QUANTIZE_Q8_0:
      {
        const auto *p = reinterpret_cast<const RmsNormExParams *>(req->payload);
        size_t      bytes;
        if (p->ne0 <= 0 || p->ne1 <= 0 || !mul3((size_t) p->ne0, (size_t) p->ne1, 4, &bytes)) {
          return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm: bad size (ne0=%d ne1=%d)", p->ne0, p->ne1);
        }
        const float *w = nullptr;
        if (p->weight.fd >= 0) {
          w = (const float *) resolve(ctx, p->weight, (size_t) p->ne0 * 4);
          if (!w) {
            return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm: unknown weight buffer");
          }
        }
        const float *src = (const float *) resolve(ctx, p->src, bytes);
        if (req->op == HTP_OPS_RMS_NORM_F32_EX) {
          return op_rms_norm(ctx, (float *) resolve(ctx, p->dst, bytes), src, w, p->eps, p->ne0, p->ne1);
        }
        if (p->ne0 % 32 != 0) {
          return fail(ctx, HTPOPS_ERR_REJECTED, "rms_norm_quantize: ne0=%d is not a multiple of 32", p->ne0);
        }
        return op_rms_norm_quantize(ctx, resolve(ctx, p->dst, q8_0_bytes((size_t) p->ne1, (size_t) p->ne0)), src, w,
                                    p->eps, p->ne0, p->ne1);
      }
    case HTP_OPS_QUANTIZE_Q8_0:
      {
        const auto *p = reinterpret_cast<const RmsNormF32Params *>(req->payload);
        size_t      bytes;
        if (p->ne0 <= 0 || p->ne1 <= 0 || p->ne0 % 32 != 0 || !mul3((size_t) p->ne0, (size_t) p->ne1, 4, &bytes)) {
          return fail(ctx, HTPOPS_ERR_REJECTED, "quantize_q8_0: bad size (ne0=%d ne1=%d)", p->ne0, p->ne1);
        }
        return op_quantize(ctx, resolve(ctx, p->dst, q8_0_bytes((size_t) p->ne1, (size_t) p->ne0)),
                           (const float *) resolve(ctx, p->src, bytes), p->ne0, p->ne1);
      }
    case HTP_OPS_MAT_MUL_Q4_0_Q8_0:
    case HTP_OPS_MAT_MUL_Q8_0_Q8_0:
    case HTP_OPS_MAT_MUL_Q4_0_A32:
    case HTP_OPS_MAT_MUL_Q8_0_A32:
      {
        // reference: op_executor.cc:114-149 (sizes), with ggml row-layout weights
        const auto *p  = reinterpret_cast<const MatMulParams *>(req->payload);
        const int   wt = (req->op == HTP_OPS_MAT_MUL_Q4_0_Q8_0 || req->op == HTP_OPS_MAT_MUL_Q4_0_A32) ? kQ4_0 :
                                                                                                         kQ8_0;
        const bool  f32_act = req->op == HTP_OPS_MAT_MUL_Q4_0_A32 || req->op == HTP_OPS_MAT_MUL_Q8_0_A32;
        size_t      out_bytes, act_bytes;
        if (p->m <= 0 || p->k <= 0 || p->n <= 0 || p->k % 32 != 0 ||
            !mul3((size_t) p->m, (size_t) p->n, 4, &out_bytes) || !mul3((size_t) p->m, (size_t) p->k, 4, &act_bytes)) {
          return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul: bad size (m=%d k=%d n=%d)", p->m, p->k, p->n);
        }
        float      *out = (float *) resolve(ctx, p->output, out_bytes);
        const void *w   = resolve(ctx, p->weight, weight_bytes((size_t) p->n, (size_t) p->k, wt));
        if (f32_act) {
          return op_mat_mul_f32(ctx, out, (const float *) resolve(ctx, p->activation, act_bytes), w, p->m, p->k, p->n,
                                wt);
        }
        return op_mat_mul_q8(ctx, out, resolve(ctx, p->activation, q8_0_bytes((size_t) p->m, (size_t) p->k)), w, p->m,
                             p->k, p->n, wt);
      }
    case HTP_OPS_FLASH_ATTN_QO_F32_KV_F16:
    case HTP_OPS_FLASH_ATTN_F16:
      {
        // reference: op_executor.cc:151-196
        const bool  ext    = req->op == HTP_OPS_FLASH_ATTN_F16;
        const auto *p      = reinterpret_cast<const FlashAttnParams *>(req->payload);
        const int   causal = ext ? reinterpret_cast<const FlashAttnExParams *>(req->payload)->causal : 0;
        if (p->qo_len <= 0 || p->kv_len <= 0 || p->n_heads <= 0 || p->n_kv_heads <= 0 || p->head_dim <= 0) {
          return fail(ctx, HTPOPS_ERR_REJECTED, "flash_attn: non-positive size");
        }
        size_t qo_elems, kv_elems, qo_bytes, kv_bytes, mask_bytes;
        if (!mul3((size_t) p->qo_len, (size_t) p->n_heads, (size_t) p->head_dim, &qo_elems) ||
            !mul3((size_t) p->kv_len, (size_t) p->n_kv_heads, (size_t) p->head_dim, &kv_elems) ||
            !mul3(qo_elems, ext ? 2 : 4, 1, &qo_bytes) || !mul3(kv_elems, 2, 1, &kv_bytes) ||
            !mul3((size_t) p->qo_len, ((size_t) p->kv_len + 63) / 64 * 64, 2, &mask_bytes)) {
          return fail(ctx, HTPOPS_ERR_REJECTED, "flash_attn: size overflow");
        }
        const void *mask = nullptr;
        if (p->mask.fd >= 0 && lookup(ctx, p->mask.fd)) {
          // the kernel strides the mask by align_up(kv_len, 64) (reference: flash_attn.c:152)
          mask = resolve(ctx, p->mask, mask_bytes);
          if (!mask) {
            return fail(ctx, HTPOPS_ERR_REJECTED, "flash_attn: mask buffer smaller than qo_len * align_up(kv_len, 64) * 2");
          }
        }
        return op_flash_attn(ctx, resolve(ctx, p->o, qo_bytes), resolve(ctx, p->q, qo_bytes),
                             resolve(ctx, p->k, kv_bytes), resolve(ctx, p->v, kv_bytes), mask, p->qo_len, p->kv_len,
                             p->n_heads, p->n_kv_heads, p->head_dim, ext ? 0 : 1, causal);
      }
    case HTP_OPS_MAT_MUL_PERMUTED_W16A32:
    case HTP_OPS_MAT_MUL_PERMUTED_W4D16A32:
    case HTP_OPS_MAT_MUL_PERMUTED_W8D16A32:
    case HTP_OPS_MAT_MUL_PERMUTED_W4D16A32_IQ4_NL:
      {
        // reference: op_executor.cc:96-149; the op id doubles as the weight kind
        const auto *p    = reinterpret_cast<const MatMulParams *>(req->payload);
        const int   kind = (int) req->op;
        size_t      out_bytes, act_bytes;
        if (p->m <= 0 || p->k <= 0 || p->n <= 0 || p->k % 32 != 0 || p->n % 32 != 0 ||
            !mul3((size_t) p->m, (size_t) p->n, 4, &out_bytes) || !mul3((size_t) p->m, (size_t) p->k, 4, &act_bytes)) {
          return fail(ctx, HTPOPS_ERR_REJECTED, "mat_mul_permuted: bad size (m=%d k=%d n=%d)", p->m, p->k, p->n);
        }
        return op_mat_mul_permuted(ctx, (float *) resolve(ctx, p->output, out_bytes),
                                   (const float *) resolve(ctx, p->activation, act_bytes),
                                   resolve(ctx, p->weight, permuted_weight_bytes((size_t) p->n, (size_t) p->k, kind)),
                                   p->m, p->k, p->n, kind);
      }
    default:
      // the reference returns 0 without touching anything (op_executor.cc:200-203); a silent success on an
      // unknown op hides host bugs, so this backend reports it
      return fail(ctx, HTPOPS_ERR_REJECTED, "unknown op %u", req->op);
  }
}

// ------------------------------------------------------------------------------------------------ direct entries

extern "C" int htpops_rms_norm_f32(htpops_context *ctx, int dst_fd, int dst_offset, int src_fd, int src_offset,
                                   int ne0, int ne1) {
  struct {
    struct OpComputeRequest req;
    struct RmsNormF32Params params;
  } HTPOPS_PACKED r;
  r.req.op     = HTP_OPS_RMS_NORM_F32;
  r.params.dst = { dst_fd, dst_offset };
  r.params.src = { src_fd, src_offset };
  r.params.ne0 = ne0;
  r.params.ne1 = ne1;
  int ret      = htpops_execute_op(ctx, &r.req);
  if (ret != HTPOPS_OK) {
    return ret;
  }
  return htpops_synchronize(ctx);
}

extern "C" int htpops_mat_mul_permuted_w16a32(htpops_context *ctx, int output_fd, int output_offset,
                                              int activation_fd, int activation_offset, int weight_fd,
                                              int weight_offset, int m, int k, int n) {
  struct {
    struct OpComputeRequest req;
    struct MatMulParams     params;
  } HTPOPS_PACKED r;
  r.req.op            = HTP_OPS_MAT_MUL_PERMUTED_W16A32;
  r.params.output     = { output_fd, output_offset };
  r.params.activation = { activation_fd, activation_offset };
  r.params.weight     = { weight_fd, weight_offset };
  r.params.m          = m;
  r.params.k          = k;
  r.params.n          = n;
  int ret             = htpops_execute_op(ctx, &r.req);
  if (ret != HTPOPS_OK) {
    return ret;
  }
  return htpops_synchronize(ctx);
}

// ------------------------------------------------------------------------------------------------ pointer entries

extern "C" int htpops_rms_norm_f32_ex_ptr(htpops_context *ctx, float *dst, const float *src, const float *weight,
                                          float eps, int ne0, int ne1) {
  if (!ctx) {
    return HTPOPS_ERR_REJECTED;
  }
  Lock lock(ctx->mu);
  return op_rms_norm(ctx, dst, src, weight, eps, ne0, ne1);
}

extern "C" int htpops_quantize_q8_0_ptr(htpops_context *ctx, void *dst, const float *src, int k, int m) {
  if (!ctx) {
    return HTPOPS_ERR_REJECTED;
  }
  Lock lock(ctx->mu);
  return op_quantize(ctx, dst, src, k, m);
}

extern "C" int htpops_rms_norm_quantize_q8_0_ptr(htpops_context *ctx, void *dst, const float *src,
                                                 const float *weight, float eps, int ne0, int ne1) {
  if (!ctx) {
    return HTPOPS_ERR_REJECTED;
  }
  Lock lock(ctx->mu);
  return op_rms_norm_quantize(ctx, dst, src, weight, eps, ne0, ne1);
}

extern "C" int htpops_mat_mul_q8_0_act_ptr(htpops_context *ctx, float *dst, const void *act_q8_0, const void *weight,
                                           int m, int k, int n, int weight_type) {
  if (!ctx) {
    return HTPOPS_ERR_REJECTED;
  }
  Lock lock(ctx->mu);
  return op_mat_mul_q8(ctx, dst, act_q8_0, weight, m, k, n, weight_type);
}

extern "C" int htpops_mat_mul_f32_act_ptr(htpops_context *ctx, float *dst, const float *act, const void *weight, int m,
                                          int k, int n, int weight_type) {
  if (!ctx) {
    return HTPOPS_ERR_REJECTED;
  }
  Lock lock(ctx->mu);
  return op_mat_mul_f32(ctx, dst, act, weight, m, k, n, weight_type);
}

extern "C" int htpops_flash_attn_ptr(htpops_context *ctx, void *o, const void *q, const void *k, const void *v,
                                     const void *mask, int qo_len, int kv_len, int n_heads, int n_kv_heads,
                                     int head_dim, int qo_is_f32, int causal) {
  if (!ctx) {
    return HTPOPS_ERR_REJECTED;
  }
  Lock lock(ctx->mu);
  return op_flash_attn(ctx, o, q, k, v, mask, qo_len, kv_len, n_heads, n_kv_heads, head_dim, qo_is_f32, causal);
}

extern "C" int htpops_flash_attn_noalloc_ptr(htpops_context *ctx, void *o, const void *q, const void *k, const void *v,
                                             const void *mask, int qo_len, int kv_len, int n_heads, int n_kv_heads,
                                             int head_dim, int qo_is_f32, int causal) {
  if (!ctx) {
    return HTPOPS_ERR_REJECTED;
  }
  Lock lock(ctx->mu);
  return op_flash_attn(ctx, o, q, k, v, mask, qo_len, kv_len, n_heads, n_kv_heads, head_dim, qo_is_f32, causal,
                       /*no_alloc=*/true);
}
