"""GPU parity of attention where the keys of a query block are dealt to several workgroups, over the head dims that are
padded to a multiple of 32, and over masks that hide or leave alone whole blocks: against the oracle, at the edges."""
import ctypes

import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl

pytestmark = pytest.mark.gpu

ATOL = 2e-3  # as for every attention case: fp16 queries (and, at 64 and 128, probabilities)


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    yield c
    c.close()


@pytest.mark.parametrize("qo,kv,nh,nkv,d", [
    (1, 511, 4, 2, 96), (1, 3000, 8, 8, 16), (1, 2100, 5, 1, 256),     # one row; group sizes 2, 1 and 5
    (2, 1025, 12, 2, 128), (5, 1029, 12, 2, 128), (33, 513, 7, 1, 64), # a second head sub-group, a second query tile
    (31, 640, 3, 1, 160), (32, 1000, 4, 4, 48), (65, 700, 4, 1, 208), (40, 1100, 8, 4, 240), (70, 900, 2, 2, 112),
    (130, 130, 2, 1, 32), (100, 90, 4, 2, 96),                         # (the last: more queries than keys)
])
@pytest.mark.parametrize("f32", [False, True])
def test_shared_keys_and_padded_head_dims(ctx, oracle, qo, kv, nh, nkv, d, f32):
    rng = wl.rng_for(64, qo * 1000 + kv + d)
    q, k, v = wl.make_attention_inputs(rng, qo, kv, nh, nkv, d)
    q = q.astype(np.float32) if f32 else q
    ld = (kv + 63) // 64 * 64
    biases = np.full((qo, ld), -np.inf, np.float16)  # finite biases, two blocks left alone, one hidden
    biases[:, :kv] = rng.standard_normal((qo, kv)) * 2
    biases[:, 64:192] = np.float16(-0.0)
    biases[:, 192:256] = -np.inf
    biases[:, kv:] = -np.inf
    print("attention", qo, kv, nh, nkv, d, f32, flush=True)
    for mask, causal in ((None, qo <= kv), (biases, False)):
        got = ctx.run_flash_attn(q, k, v, mask, nh, nkv, d, causal=causal) if not f32 or causal is False else \
            ctx.run_flash_attn(q, k, v, wl.make_causal_mask(qo, kv), nh, nkv, d)
        want = oracle.flash_attn(q, k, v, wl.make_causal_mask(qo, kv) if f32 and causal else mask, nh, nkv, d, causal and not f32)
        assert got.dtype == q.dtype and np.abs(got.astype(np.float32) - want.astype(np.float32)).max() <= ATOL


@pytest.mark.parametrize("qo,kv,nh,nkv,d", [(5, 1029, 12, 2, 128), (1, 1500, 4, 2, 80)])
def test_mask_at_eight_bytes_and_the_call_that_allocates_nothing(ctx, oracle, qo, kv, nh, nkv, d):
    # a mask that is only 8-byte aligned, through both entry points on raw pointers: the same bytes from both
    rng = wl.rng_for(65, qo + kv)
    q, k, v = wl.make_attention_inputs(rng, qo, kv, nh, nkv, d)
    mask = wl.make_causal_mask(qo, kv)
    mask[:, 70:75] = -np.inf
    hq, hk, hv, ho = ctx.upload(q), ctx.upload(k), ctx.upload(v), ctx.alloc(q.nbytes)
    hm = ctx.upload(np.concatenate([np.zeros(4, np.float16), mask.reshape(-1)]))
    want = oracle.flash_attn(q, k, v, mask, nh, nkv, d, False)
    outs = []
    for fn in (ctx.lib.htpops_flash_attn_ptr, ctx.lib.htpops_flash_attn_noalloc_ptr):
        p = [ctypes.c_void_p(ctx.device_ptr(h)) for h in (ho, hq, hk, hv)] + [ctypes.c_void_p(ctx.device_ptr(hm) + 8)]
        assert fn(ctx._ctx, *p, qo, kv, nh, nkv, d, 0, 0) == 0, ctx.last_error()
        ctx.synchronize()
        outs.append(ctx.read(ho, np.float16, q.size).reshape(q.shape))
    for h in (hq, hk, hv, ho, hm):
        ctx.release(h)
    assert np.array_equal(outs[0].view(np.uint16), outs[1].view(np.uint16))
    assert np.abs(outs[0].astype(np.float32) - want.astype(np.float32)).max() <= ATOL
