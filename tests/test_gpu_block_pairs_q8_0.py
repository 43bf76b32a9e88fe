"""GPU parity of 2 to 8 rows against Q8_0 weights of long K, two blocks per matrix instruction: against the oracle at the edges of
its tiles and steps, and members of different k in one launch against one request each."""
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


@pytest.mark.parametrize("m,k,n", [(4, 4096, 16), (5, 4352, 4112), (8, 4096 + 256, 33 * 16), (7, 13312, 48),  # one tile; odd quads; long rows
                                   (2, 12544, 32), (4, 3840, 48)])  # two rows past the kernel that keeps them in registers; short K
def test_two_blocks_per_instruction(ctx, oracle, m, k, n):
    rng = wl.rng_for(93, m * 17 + k + n)
    got, x, w = check_mat_mul(ctx, oracle, rng, m, k, n, wl.GGML_TYPE_Q8_0)
    assert np.array_equal(ctx.run_mat_mul(oracle.quantize_q8_0(x), w, m, k, n, wl.GGML_TYPE_Q8_0), got)


def test_members_of_different_k_equal_single_requests(ctx, oracle):
    rng = wl.rng_for(94, 0)
    m, wt, op = 6, wl.GGML_TYPE_Q8_0, api.HTP_OPS_MAT_MUL_Q8_0_Q8_0
    shapes = [(4096, 4096), (256, 8960), (48, 4352), (1536, 4096)]
    acts = {k: ctx.upload(oracle.quantize_q8_0(wl.make_activations(rng, m, k))) for k in (4096, 8960, 4352)}
    ws = [ctx.upload(wl.make_weights(rng, n, k, wt)) for n, k in shapes]
    results = []
    for grouped in (True, False):
        outs = [ctx.upload(np.zeros(m * n, np.float32)) for n, _ in shapes]
        reqs = [(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(op, api.mat_mul_params((outs[j], 0), (acts[k], 0), (ws[j], 0), m, k, n)))
                for j, (n, k) in enumerate(shapes)]
        for msg in ([api.build_message(reqs)] if grouped else [api.build_message([r]) for r in reqs]):
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        assert ctx.last_message_submissions() == 1
        results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in outs])
        for h in outs:
            ctx.release(h)
    for a, b in zip(*results):
        assert np.array_equal(a, b) and a.any()
    for h in list(acts.values()) + ws:
        ctx.release(h)
