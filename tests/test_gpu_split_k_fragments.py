"""GPU parity of the int8 fragment matmuls whose K is dealt to several waves and workgroups (17 rows and more, matrices too
small to fill the chip): against the oracle at the edges of the split, and grouped in a message against one request each."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl
from test_gpu_parity_core import check_mat_mul

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    yield c
    c.close()


@pytest.mark.parametrize("wt", [wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0])
@pytest.mark.parametrize("m,k,n", [
    (17, 64, 32), (20, 224, 40), (32, 256, 33),        # below, just below and at eight blocks; one pair of blocks
    (18, 1536, 100), (33, 1568, 70), (31, 3104, 17),   # 12 blocks a wave and one more; an odd number of blocks
    (65, 8960, 65), (40, 12320, 32),                   # five and eight workgroups per tile
    (128, 768, 64), (128, 1600, 96), (256, 8960, 33)]) # whole groups of four row tiles: one, two and five parts
def test_split_k_at_the_edges(ctx, oracle, wt, m, k, n):
    # the tolerance is `check_mat_mul`'s: exact block sums, fp32 over the blocks in another order
    rng = wl.rng_for(59, m * 131 + k + n + wt)
    first, x, w = check_mat_mul(ctx, oracle, rng, m, k, n, wt)
    again = ctx.run_mat_mul(oracle.quantize_q8_0(x), w, m, k, n, wt)
    assert np.array_equal(first, again)
    if m <= 32:  # (small matrices of so few rows take another kernel on their own)
        with ctx.option("gemm_tile_units", 1):
            check_mat_mul(ctx, oracle, rng, m, k, n, wt)


@pytest.mark.parametrize("wt", [wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0])
@pytest.mark.parametrize("m,k,n", [
    (97, 32, 16384), (128, 96, 16383), (110, 320, 16400),  # one, three and ten blocks; ragged columns
    (225, 64, 8161), (256, 1120, 8192)])                   # two row blocks, the last row tile ragged or whole
def test_staged_operands_at_the_edges(ctx, oracle, wt, m, k, n):
    ctx.set_option("gemm_fp6", 0)
    rng = wl.rng_for(59, m * 131 + k + n + wt)
    first, x, w = check_mat_mul(ctx, oracle, rng, m, k, n, wt)
    assert np.array_equal(first, ctx.run_mat_mul(oracle.quantize_q8_0(x), w, m, k, n, wt))
    ctx.set_option("gemm_fp6", api.DEFAULT_OPTIONS["gemm_fp6"])


@pytest.mark.parametrize("wt", [wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0])
@pytest.mark.parametrize("m,k,n", [
    (97, 32, 17920), (110, 96, 17921), (225, 320, 8961), (256, 1120, 8960),      # 280 to 511 workgroups of 128 rows: tiles of 64
    (128, 64, 32768), (200, 96, 16384), (512, 1056, 8161), (110, 2080, 32770)])  # 512 and more: tiles of 128
def test_staged_tiles_of_both_sizes(ctx, oracle, wt, m, k, n):
    with ctx.option("gemm_fp6", 0):
        check_mat_mul(ctx, oracle, wl.rng_for(59, m * 131 + k + n + wt), m, k, n, wt)


def test_staged_tiles_of_both_sizes_give_the_same_bits(ctx, oracle):
    # alone a matrix takes tiles of 64 rows, two of them in a message tiles of 128
    m, n, k, wt = 256, 8960, 608, wl.GGML_TYPE_Q8_0
    rng = wl.rng_for(61, 0)
    ha = ctx.upload(oracle.quantize_q8_0(wl.make_activations(rng, m, k)))
    ws = [ctx.upload(wl.make_weights(rng, n, k, wt)) for _ in range(2)]
    outs = [ctx.alloc(m * n * 4) for _ in range(4)]
    reqs = [(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(api.HTP_OPS_MAT_MUL_Q8_0_Q8_0, api.mat_mul_params(
        (outs[j], 0), (ha, 0), (ws[j % 2], 0), m, k, n))) for j in range(4)]
    for msg in (api.build_message(reqs[:2]), api.build_message(reqs[2:3]), api.build_message(reqs[3:])):
        assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
    both = [ctx.read(h, np.uint32, m * n) for h in outs]
    assert np.array_equal(both[0], both[2]) and np.array_equal(both[1], both[3]) and both[0].any()
    for h in [ha] + ws + outs:
        ctx.release(h)


@pytest.mark.parametrize("wt", [wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0])
@pytest.mark.parametrize("m", [17, 32])
def test_members_over_weights_as_they_are_and_over_copies_equal_single_requests(ctx, oracle, m, wt):
    # small matrices (K-sliced kernel, one to three slices) and large ones (fragments) in one message behind their quantizers,
    # in both orders; small ones over caller-owned memory; each output byte for byte what its own message gives
    rng = wl.rng_for(62, m + wt)
    op = api.HTP_OPS_MAT_MUL_Q4_0_Q8_0 if wt == wl.GGML_TYPE_Q4_0 else api.HTP_OPS_MAT_MUL_Q8_0_Q8_0
    shapes = [(300, 256), (1000, 1536), (4096, 4096), (64, 4096), (40, 2560), (33, 256)]
    xs = {k: ctx.upload(wl.make_activations(rng, m, k)) for k in (256, 1536, 2560, 4096)}
    acts = {k: ctx.alloc(m * (k // 32) * 34) for k in xs}
    quantize = {k: (api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params(
        (acts[k], 0), (xs[k], 0), k, m))) for k in xs}
    ws = [ctx.upload(wl.make_weights(rng, n, k, wt)) for n, k in shapes]
    alias = ctx.register(ctx.device_ptr(ws[1]), ctx.size(ws[1]))
    seen = [ws[0], alias] + ws[2:]
    results = []
    for order in ([0, 1, 2, 3, 4, 5], [2, 0, 5, 4, 3, 1], None):
        outs = [ctx.upload(np.zeros(m * n, np.float32)) for n, _ in shapes]
        req = lambda j: (api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(op, api.mat_mul_params(
            (outs[j], 0), (acts[shapes[j][1]], 0), (seen[j], 0), m, shapes[j][1], shapes[j][0])))
        msgs = [[quantize[k] for k in (256, 1536, 2560, 4096)] + [req(j) for j in order]] if order else \
            [[quantize[shapes[j][1]], req(j)] for j in range(len(shapes))]
        for msg in msgs:
            msg = api.build_message(msg)
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        if order:
            assert ctx.last_message_submissions() == 4 + 1
        results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in outs])
        for h in outs:
            ctx.release(h)
    for a, b, c in zip(*results):
        assert np.array_equal(a, b) and np.array_equal(a, c) and a.any()
    for h in list(xs.values()) + list(acts.values()) + ws + [alias]:
        ctx.release(h)


@pytest.mark.parametrize("m", [17, 50, 128])
def test_grouped_split_k_equals_single_requests(ctx, oracle, m):
    rng = wl.rng_for(60, m)
    wt, op = wl.GGML_TYPE_Q8_0, api.HTP_OPS_MAT_MUL_Q8_0_Q8_0
    shapes = [(96, 1536), (256, 1536), (64, 8960), (40, 256), (1000, 1536)] + ([(17920, 256)] if m == 128 else [])  # (the last: staged)
    acts = {k: ctx.upload(oracle.quantize_q8_0(wl.make_activations(rng, m, k))) for k in (1536, 8960, 256)}
    ws = [ctx.upload(wl.make_weights(rng, n, k, wt)) for n, k in shapes]
    results = []
    for grouped in (True, False):
        outs = [ctx.upload(np.zeros(m * n, np.float32)) for n, _ in shapes]
        reqs = [(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(op, api.mat_mul_params((outs[j], 0), (acts[k], 0), (ws[j], 0), m, k, n)))
                for j, (n, k) in enumerate(shapes)]
        for msg in ([api.build_message(reqs)] if grouped else [api.build_message([r]) for r in reqs]):
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        if grouped:
            assert ctx.last_message_submissions() == 1
        results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in outs])
        for h in outs:
            ctx.release(h)
    for a, b in zip(*results):
        assert np.array_equal(a, b) and a.any()
    for h in list(acts.values()) + ws:
        ctx.release(h)
