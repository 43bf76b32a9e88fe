"""GPU: a prefill whose keys are split, the Q8_0 quantization of its fp32 output and the matmul over those rows in one message: the launch
that puts the shares together also quantizes, in the operand order of the matmul. Against one message per request, every
buffer byte for byte, and the stored rows against the oracle's quantizer."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl

pytestmark = pytest.mark.gpu

Q4, Q8 = wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    c.set_option("gemm_fp6", 1)          # (FP6 tiles at any size that fits)
    c.set_option("gemm_tile_units", 1)   # (as the int8 fragments of up to 32 rows)
    yield c
    c.close()


# rows that end a tile of 32 or not, a head of one to four blocks, odd block counts; two rows (no operand behind them)
@pytest.mark.parametrize("qo,kv,nh,nkv,d,masked", [
    (33, 1152, 16, 1, 128, False), (128, 1152, 12, 2, 128, True), (161, 1500, 8, 2, 64, True), (96, 2000, 6, 3, 96, False),
    (40, 1111, 7, 1, 32, True), (17, 700, 2, 1, 160, True), (2, 900, 6, 3, 96, True), (300, 1024, 4, 2, 128, False)])
@pytest.mark.parametrize("wt", [Q4, Q8, None])
def test_equals_one_message_per_request(ctx, oracle, qo, kv, nh, nkv, d, masked, wt):
    if wt is not None and qo < 17:
        wt = Q8
    rng = wl.rng_for(101, qo * 7 + kv + d)
    q, k, v = wl.make_attention_inputs(rng, qo, kv, nh, nkv, d)
    ne0, n = nh * d, 72
    mask = np.zeros((qo, (kv + 63) // 64 * 64), np.float16)
    mask[:, kv:] = -np.inf
    for i in range(qo):
        mask[i, kv - qo + i + 1:] = -np.inf
    hs = {"q": ctx.upload(q.astype(np.float32)), "k": ctx.upload(k), "v": ctx.upload(v), "mask": ctx.upload(mask)}
    if wt is not None:
        hs["w"] = ctx.upload(wl.make_weights(rng, n, ne0, wt))
    results = []

    def op(code, payload):
        return (api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(code, payload))

    print("attention, rows, matmul", qo, kv, nh, nkv, d, wt, flush=True)
    for together in (True, False):
        ho = ctx.upload(np.full(qo * ne0, np.nan, np.float32))
        hq8 = ctx.upload(np.full(qo * ne0 // 32 * 34, 0xA5, np.uint8))
        hout = ctx.upload(np.zeros(qo * n, np.float32))
        reqs = [op(api.HTP_OPS_FLASH_ATTN_QO_F32_KV_F16,
                   api.flash_attn_params((ho, 0), (hs["q"], 0), (hs["k"], 0), (hs["v"], 0), (hs["mask"] if masked else -1, 0), qo, kv, nh, nkv, d)),
                op(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params((hq8, 0), (ho, 0), ne0, qo))]
        if wt is not None:
            reqs.append(op(api.HTP_OPS_MAT_MUL_Q4_0_Q8_0 if wt == Q4 else api.HTP_OPS_MAT_MUL_Q8_0_Q8_0,
                           api.mat_mul_params((hout, 0), (hq8, 0), (hs["w"], 0), qo, ne0, n)))
        for msg in ([api.build_message(reqs)] if together else [api.build_message([r]) for r in reqs]):
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        if together:
            assert ctx.last_message_submissions() == len(reqs) - 1
        results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in (ho, hq8, hout)])
        for h in (ho, hq8, hout):
            ctx.release(h)
    for a, b in zip(*results):
        assert np.array_equal(a, b)
    rows = results[0][0].view(np.float32).reshape(qo, ne0)
    assert np.isfinite(rows).all()
    assert np.array_equal(results[0][1].reshape(qo, -1), oracle.quantize_q8_0(rows).reshape(qo, -1))
    for h in hs.values():
        ctx.release(h)
