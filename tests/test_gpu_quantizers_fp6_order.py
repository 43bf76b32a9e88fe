"""GPU: the quantizers that also leave their rows in the operand order of the FP6-tile matmul behind them (op 13, RMSNorm and Q8_0 in
one, and op 14; the fp32-activation matmul, which quantizes into that order alone), against the same requests sent one message
each, where that order is made from the stored rows by a launch of its own: every output byte for byte, and against the oracle."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl

pytestmark = pytest.mark.gpu

Q4 = wl.GGML_TYPE_Q4_0


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    c.set_option("gemm_fp6", 1)  # (FP6 tiles at any size that fits)
    yield c
    c.close()


# rows that end a tile of 32, a row block of 128 or neither; k at the ends of what a thread of op 13 holds, odd step counts
@pytest.mark.parametrize("m", [33, 96, 128, 161])
@pytest.mark.parametrize("k", [64, 2048, 2112, 4096, 4160, 8256, 16384])
def test_quantized_rows_in_fp6_order(ctx, oracle, m, k):
    rng = wl.rng_for(99, m + k)
    n = 40
    x, g = wl.make_activations(rng, m, k), (1 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    x[0, :32] = 0.0
    w = wl.make_weights(rng, n, k, Q4)
    hx, hg, hw = ctx.upload(x), ctx.upload(g), ctx.upload(w)
    q_bytes, o_bytes = m * (k // 32) * 34, m * n * 4
    print("fp6 order", m, k, flush=True)
    # something else lies in the workspace first: the rows and scales that nobody writes must not matter
    ctx.run_mat_mul(oracle.quantize_q8_0(wl.make_activations(rng, 256, k) * 1e4), w, 256, k, n, Q4)
    rows_of = {}
    for quantizer in (api.HTP_OPS_RMS_NORM_QUANTIZE_Q8_0, api.HTP_OPS_QUANTIZE_Q8_0):
        results = []
        for together in (True, False):
            hq, ho = ctx.upload(np.zeros(q_bytes, np.uint8)), ctx.upload(np.zeros(o_bytes, np.uint8))
            body = api.rms_norm_ex_params((hq, 0), (hx, 0), (hg, 0), k, m, 1e-6) if quantizer == api.HTP_OPS_RMS_NORM_QUANTIZE_Q8_0 else \
                api.rms_norm_params((hq, 0), (hx, 0), k, m)
            reqs = [(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(quantizer, body)),
                    (api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(api.HTP_OPS_MAT_MUL_Q4_0_Q8_0,
                                                                         api.mat_mul_params((ho, 0), (hq, 0), (hw, 0), m, k, n)))]
            for msg in ([api.build_message(reqs)] if together else [api.build_message([r]) for r in reqs]):
                assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
            results.append((ctx.read(hq, np.uint8, q_bytes), ctx.read(ho, np.uint8, o_bytes)))
            ctx.release(hq), ctx.release(ho)
        for a, b in zip(*results):
            assert np.array_equal(a, b) and a.any()
        rows, out = results[0][0].reshape(m, -1), results[0][1].view(np.float32).reshape(m, n)
        want, mag = oracle.mat_mul_q8_0_act_f64(rows, w, m, k, n, Q4)
        assert np.all(np.abs(out - want) <= 1e-5 * mag)
        rows_of[quantizer] = (rows, out)
    # fp32 activations: the same rows, quantized into that order without being stored
    ho = ctx.upload(np.zeros(o_bytes, np.uint8))
    msg = api.build_message([(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(
        api.HTP_OPS_MAT_MUL_Q4_0_A32, api.mat_mul_params((ho, 0), (hx, 0), (hw, 0), m, k, n)))])
    assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
    assert np.array_equal(ctx.read(ho, np.float32, m * n).reshape(m, n), rows_of[api.HTP_OPS_QUANTIZE_Q8_0][1])
    for h in (hx, hg, hw, ho):
        ctx.release(h)
