"""GPU: attention of a few query rows over many keys (the (query, head) pairs of a GQA group as the rows of a score tile): against
the oracle at the edges of its tiles and splits, the same bits from every entry point, and the Q8_0 rows that its last
launch leaves for the request behind it."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl
from test_gpu_attention_shares import ATOL, test_entry_points_and_captured_calls_give_the_same_bits as same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    yield c
    c.close()


@pytest.mark.parametrize("qo,kv,nh,nkv,d", [
    (2, 200, 2, 1, 64), (2, 128, 4, 2, 128),        # the shortest keys, with a mask; a tile of four pairs
    (16, 513, 1, 1, 64), (17, 512, 3, 3, 64),       # a whole tile and one row more; a last split of one key
    (3, 4096, 7, 1, 128), (5, 4097, 11, 1, 64),     # 64 splits of 64 keys, one key more (128 each); pairs over tile edges
    (2, 8192, 6, 2, 64), (2, 8193, 2, 1, 64),       # 64 splits of 128; one key more is the prefill kernel's
    (40, 385, 4, 1, 128), (512, 600, 1, 1, 128)])   # more than 16 rows; as many pairs as there may be
@pytest.mark.parametrize("f32", [False, True])
def test_few_rows_at_the_edges(ctx, oracle, qo, kv, nh, nkv, d, f32):
    rng = wl.rng_for(90, qo * 1000 + kv + d)
    q, k, v = wl.make_attention_inputs(rng, qo, kv, nh, nkv, d)
    q = q.astype(np.float32) if f32 else q
    for mask, causal in ((None, not f32), (wl.make_causal_mask(qo, kv), False)):  # (the fp32 op has no causal flag)
        print("few rows", qo, kv, nh, nkv, d, f32, mask is not None, flush=True)
        got = ctx.run_flash_attn(q, k, v, mask, nh, nkv, d, causal=causal)
        want = oracle.flash_attn(q, k, v, mask, nh, nkv, d, causal)
        assert np.abs(got.astype(np.float32) - want.astype(np.float32)).max() <= ATOL


@pytest.mark.parametrize("qo,kv,nh,nkv,d", [(2, 300, 4, 1, 64), (3, 4096, 7, 1, 128), (17, 1500, 6, 2, 64), (2, 8192, 8, 4, 128)])
@pytest.mark.parametrize("f32", [False, True])
def test_captured_calls_give_the_same_bits(ctx, oracle, qo, kv, nh, nkv, d, f32):
    same_bits(ctx, oracle, qo, kv, nh, nkv, d, f32)


def test_keys_that_no_row_sees_may_hold_anything(ctx):
    # 32 keys and more behind the mask: nothing of them reaches the results, whatever they are
    qo, kv, nh, nkv, d, seen = 4, 700, 8, 2, 128, 576
    rng = wl.rng_for(91, 0)
    q, k, v = wl.make_attention_inputs(rng, qo, kv, nh, nkv, d)
    mask = np.zeros((qo, (kv + 63) // 64 * 64), np.float16)
    mask[:, seen:] = -np.inf
    got = []
    for value in (0.0, np.nan, np.inf):
        k[seen:], v[seen:] = value, value
        got.append(ctx.run_flash_attn(q.astype(np.float32), k, v, mask, nh, nkv, d, causal=False))
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.parametrize("qo,masked", [(2, False), (5, True), (16, True)])
def test_the_rows_a_quantizer_behind_it_wants(ctx, oracle, qo, masked):
    kv, nh, nkv, d = 1029, 12, 2, 128
    rng = wl.rng_for(92, qo)
    q, k, v = wl.make_attention_inputs(rng, qo, kv, nh, nkv, d)
    width = nh * d
    hq, hk, hv = ctx.upload(q.astype(np.float32)), ctx.upload(k), ctx.upload(v)
    hm = ctx.upload(wl.make_causal_mask(qo, kv)) if masked else None
    ho, hd = ctx.alloc(qo * width * 4), ctx.alloc(qo * width // 32 * 34)
    reqs = [(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(api.HTP_OPS_FLASH_ATTN_QO_F32_KV_F16, api.flash_attn_params(
                (ho, 0), (hq, 0), (hk, 0), (hv, 0), (hm if masked else -1, 0), qo, kv, nh, nkv, d))),
            (api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params((hd, 0), (ho, 0), width, qo)))]
    results = []
    for messages in ([reqs], [reqs[:1], reqs[1:]]):
        ctx.write(hd, np.zeros(ctx.size(hd), np.uint8))
        for m in messages:
            msg = api.build_message(m)
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        assert ctx.last_message_submissions() == 1
        results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in (ho, hd)])
    assert np.array_equal(results[0][0], results[1][0]) and np.array_equal(results[0][1], results[1][1])
    rows = results[0][0].view(np.float32).reshape(qo, width)
    assert np.array_equal(results[0][1].reshape(qo, -1), oracle.quantize_q8_0(rows).reshape(qo, -1).view(np.uint8))
    for h in (hq, hk, hv, ho, hd) + ((hm,) if masked else ()):
        ctx.release(h)
