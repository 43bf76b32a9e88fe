"""GPU parity of the many-row matmuls over the reference's own weight formats (ops 1-4 with more than 32 rows): row counts
and column counts at the edges of a workgroup's tiles, one K step per half, and grouping inside a message."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl
from test_gpu_parity_permuted import OPS, check, make_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    yield c
    c.close()


@pytest.mark.parametrize("kind,m,k,n", [
    (1, 33, 32, 32), (2, 65, 64, 128), (3, 64, 96, 160), (4, 97, 160, 64),     # one step of K in all; one, two, three per half
    (1, 100, 512, 4096 + 32), (2, 130, 256, 8192), (4, 290, 2048, 96),         # two row tiles of 16 per workgroup
    (4, 33, 64, 32768), (2, 64, 96, 32768), (3, 160, 128, 32768 + 96),         # three, four, five of them
    (3, 96, 32, 32768), (4, 300, 64, 16384), (1, 128, 96, 32768), (2, 350, 64, 16384 + 32)])  # six, seven, eight, eight
def test_many_rows_at_the_edges(ctx, oracle, kind, m, k, n):
    check(ctx, oracle, kind, m, k, n, m * 3 + k + n)


def test_many_rows_grouped_with_caller_owned_weights(ctx):
    # one message: shared rows, different k (a long one last), and a member whose weights lie in registered memory: every
    # output byte for byte what one message per request gives
    rng = wl.rng_for(88, 0)
    m, kind = 70, 4
    shapes = [(128, 96), (64, 1056), (416, 96), (128, 2080)]  # (n, k)
    acts = {k: ctx.upload(wl.make_activations(rng, m, k)) for k in (96, 1056, 2080)}
    ws = [ctx.upload(np.ascontiguousarray(make_weights(rng, n, k, kind)[0]).view(np.uint8)) for n, k in shapes]
    for foreign in (False, True):
        seen = list(ws)
        if foreign:
            seen[1] = ctx.register(ctx.device_ptr(ws[1]), ctx.size(ws[1]))
        results = []
        for grouped in (True, False):
            outs = [ctx.upload(np.zeros(m * n, np.float32)) for n, _ in shapes]
            reqs = [(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(OPS[kind], api.mat_mul_params(
                (outs[j], 0), (acts[k], 0), (seen[j], 0), m, k, n))) for j, (n, k) in enumerate(shapes)]
            for msg in ([api.build_message(reqs)] if grouped else [api.build_message([r]) for r in reqs]):
                assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
            results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in outs])
            for h in outs:
                ctx.release(h)
        for a, b in zip(*results):
            assert np.array_equal(a, b) and a.any()
        if foreign:
            ctx.release(seen[1])
    for h in list(acts.values()) + ws:
        ctx.release(h)


@pytest.mark.parametrize("kind,m,k,n", [
    (2, 40, 1408, 32), (4, 40, 2816, 64), (1, 100, 4256, 96),        # whole; two parts; three uneven ones
    (3, 33, 11296, 32), (2, 129, 11296, 160), (4, 300, 5664, 256),   # eight, ragged tiles and columns
    (4, 160, 64, 65536), (3, 320, 96, 32768 + 32), (1, 144, 32, 65536)])  # ten row tiles per workgroup, nine
def test_split_k_and_large_row_blocks(ctx, oracle, kind, m, k, n):
    # twice: the counters that the parts meet at are left as they were found
    check(ctx, oracle, kind, m, k, n, m + 5 * k + n)
    check(ctx, oracle, kind, m, k, n, m + 5 * k + n)


@pytest.mark.parametrize("kind", [1, 4])
def test_split_members_equal_single_requests(ctx, kind):
    # members of two, three and eight parts beside whole ones: byte for byte what one message per request gives
    rng = wl.rng_for(89, kind)
    m, shapes = 70, [(128, 96), (96, 4160), (64, 2816), (32, 11296), (416, 96)]  # (n, k)
    acts = {k: ctx.upload(wl.make_activations(rng, m, k)) for k in (96, 2816, 4160, 11296)}
    ws = [ctx.upload(np.ascontiguousarray(make_weights(rng, n, k, kind)[0]).view(np.uint8)) for n, k in shapes]
    results = []
    for grouped in (True, False, True):
        outs = [ctx.upload(np.zeros(m * n, np.float32)) for n, _ in shapes]
        reqs = [(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(OPS[kind], api.mat_mul_params(
            (outs[j], 0), (acts[k], 0), (ws[j], 0), m, k, n))) for j, (n, k) in enumerate(shapes)]
        for msg in ([api.build_message(reqs)] if grouped else [api.build_message([r]) for r in reqs]):
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in outs])
        for h in outs:
            ctx.release(h)
    for a, b, c in zip(*results):
        assert np.array_equal(a, b) and np.array_equal(a, c) and a.any()
    for h in list(acts.values()) + ws:
        ctx.release(h)
