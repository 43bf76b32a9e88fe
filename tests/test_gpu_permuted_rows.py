"""GPU parity of the few-row matmuls over the reference's own weight formats (ops 1-4 with up to 32 rows, the weights read
as they lie): sizes at the edges of its tiles, and grouping inside a message."""
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


@pytest.mark.parametrize("kind", [1, 2, 3, 4])
@pytest.mark.parametrize("m,k,n", [
    (1, 32, 32), (2, 256, 32),       # one tile; one tile per wave
    (1, 32 * 33, 96), (3, 32 * 65, 64),  # a step of one wave only, behind 4 and 8 whole ones
    (16, 2016, 64), (17, 96, 32),    # the last single row tile, activations at the edge of LDS; the first double one
    (16, 2080, 64), (32, 1056, 160), # activations in operand order, one and two row tiles
    (1, 12320, 32), (5, 6560, 32),   # long rows: more activations than are requested ahead; just past LDS
])
def test_few_rows_at_the_edges(ctx, oracle, kind, m, k, n):
    # the tolerance is `check`'s: fp32 accumulation plus one fp16 spacing
    check(ctx, oracle, kind, m, k, n, m * 7 + k + n)


@pytest.mark.parametrize("kind", [2, 4])
def test_two_column_groups_per_workgroup(ctx, oracle, kind):
    # 17 .. 32 rows, activations past LDS, at least 512 column groups of 32 (an odd number: the last workgroup has one)
    check(ctx, oracle, kind, 19, 1760, 513 * 32, 3)


@pytest.mark.parametrize("kind,m", [(1, 1), (2, 1), (3, 7), (4, 32), (2, 40)])
def test_grouped_requests_equal_their_own_launches(ctx, kind, m):
    # Requests of a message that nothing orders share a launch; the last two depend on earlier ones (one reads an output,
    # one overwrites an output). Every output must hold, byte for byte, what one message per request gives.
    rng = wl.rng_for(87, kind * 100 + m)
    shapes = [(128, 96), (64, 256), (96, 96), (128, 1056)]  # (n, k)
    acts = {k: ctx.upload(wl.make_activations(rng, m, k)) for k in (96, 256, 1056)}
    ws = [ctx.upload(np.ascontiguousarray(make_weights(rng, n, k, kind)[0]).view(np.uint8)) for n, k in shapes]
    w_last = ctx.upload(np.ascontiguousarray(make_weights(rng, 64, 96, kind)[0]).view(np.uint8))
    results = []
    for grouped in (True, False):
        outs = [ctx.upload(np.zeros(m * n, np.float32)) for n, _ in shapes] + [ctx.upload(np.zeros(m * 64, np.float32))]
        reqs = [api.mat_mul_params((outs[j], 0), (acts[k], 0), (ws[j], 0), m, k, n) for j, (n, k) in enumerate(shapes)]
        reqs.append(api.mat_mul_params((outs[4], 0), (outs[2], 0), (w_last, 0), m, 96, 64))     # reads output 2
        reqs.append(api.mat_mul_params((outs[1], 0), (acts[96], 0), (w_last, 0), m, 96, 64))    # overwrites output 1
        reqs = [(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(OPS[kind], r)) for r in reqs]
        for msg in ([api.build_message(reqs)] if grouped else [api.build_message([r]) for r in reqs]):
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        if grouped:
            assert ctx.last_message_submissions() == 2
        results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in outs])
        for h in outs:
            ctx.release(h)
    for a, b in zip(*results):
        assert np.array_equal(a, b) and a.any()
    for h in list(acts.values()) + ws + [w_last]:
        ctx.release(h)


def test_rows_in_lds_take_no_workspace():
    # one row of a decode step: nothing is allocated for it, and what an earlier request left in the workspace stays
    rng = wl.rng_for(89, 0)
    k, n = 2048, 256
    with api.Context(device=0) as own:
        x, (raw, _) = own.upload(wl.make_activations(rng, 1, k)), make_weights(rng, n, k, 2)
        w, out = own.upload(np.ascontiguousarray(raw).view(np.uint8)), own.alloc(n * 4)
        assert own.execute(OPS[2], api.mat_mul_params((out, 0), (x, 0), (w, 0), 1, k, n)) == 0, own.last_error()
        own.synchronize()
        assert own.workspace_bytes() == 0
        # 32 rows in operand order: one copy for two members that read the same rows
        xs, outs = own.upload(wl.make_activations(rng, 32, k)), [own.alloc(32 * n * 4) for _ in range(2)]
        msg = api.build_message([(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(OPS[2], api.mat_mul_params(
            (o, 0), (xs, 0), (w, 0), 32, k, n))) for o in outs])
        assert own.process_message(msg) == 0 and not any(api.message_request_states(msg)), own.last_error()
        assert own.workspace_bytes() == 1 << 20  # (128 KiB, rounded up)
        assert np.array_equal(own.read(outs[0], np.uint8, 32 * n * 4), own.read(outs[1], np.uint8, 32 * n * 4))


@pytest.mark.parametrize("m,k", [(1, (1 << 26) + 64), (33, (1 << 25) + 32)])
def test_more_than_four_and_two_gib_of_weights_in_one_column_group(m, k):
    # 32 columns of fp16 tiles: offsets that 32 and 31 bits do not hold. All zeros but for one weight here and there.
    zeros = np.zeros(1 << 28, np.uint8)
    with api.Context(device=0) as own:
        def cleared(nbytes):
            h = own.alloc(nbytes)
            for at in range(0, nbytes, zeros.size):
                own.write(h, zeros[:min(zeros.size, nbytes - at)], at)
            return h
        print("permuted matmul over %.1f GiB of weights" % (k * 64 / 2**30), flush=True)
        act, weight, out = cleared(m * k * 4), cleared(k * 64), own.alloc(m * 32 * 4)
        want = np.zeros((m, 32), np.float32)
        places = [(0, 3), (k // 2 + 1, 5), (k - 1, 31), (k - 33, 0)]
        for i, (kk, col) in enumerate(places):
            own.write(weight, np.float16([1.5 + i]), (kk // 32 * 1024 + (kk % 32 & ~1) * 32 + col * 2 + (kk & 1)) * 2)
            for row in {0, m - 1}:
                own.write(act, np.float32([2.0 + row]), (row * k + kk) * 4)
                want[row, col] = (1.5 + i) * (2.0 + row)
        assert own.execute(OPS[1], api.mat_mul_params((out, 0), (act, 0), (weight, 0), m, k, 32)) == 0, own.last_error()
        own.synchronize()
        assert np.array_equal(own.read(out, np.float32, m * 32).reshape(m, 32), want)
