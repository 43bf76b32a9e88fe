"""GPU: ops 1-4 with an output that lies over the activations or the weights of the same request. The result is what the
same request gives with an output of its own, byte for byte: reads come before writes, whatever the launch looks like."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl
from test_gpu_parity_permuted import OPS, make_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    yield c
    c.close()


# one row and a few (rows in LDS), 20 rows in operand order, more than 32; more column groups of 32 than are resident
@pytest.mark.parametrize("kind,m,k,n", [(1, 1, 64, 1600 * 32), (2, 1, 512, 800 * 32), (3, 5, 96, 900 * 32), (4, 20, 1760, 800 * 32),
                                        (2, 64, 96, 800 * 32), (1, 40, 4096, 4096), (4, 1, 4096, 4096), (3, 2, 64, 32)])
@pytest.mark.parametrize("over", ["rows", "end of the rows", "weights", "end of the weights"])
def test_output_over_an_operand(ctx, kind, m, k, n, over):
    message = over.startswith("end")  # (both ways to send a request)
    rng = wl.rng_for(94, kind * 1000 + m + k + n)
    x = np.ascontiguousarray(wl.make_activations(rng, m, k))
    raw = make_weights(rng, n, k, kind)[0] if kind == 1 else wl.make_permuted_weights(rng, n, k, kind)
    raw = np.ascontiguousarray(raw).view(np.uint8).reshape(-1)
    out_bytes, operand = m * n * 4, x.view(np.uint8).reshape(-1) if "rows" in over else raw
    # the operand lies in the middle of a buffer that has room for the output around it
    room = (out_bytes + 127) // 128 * 128
    image = np.zeros(room + (operand.size + 127) // 128 * 128 + room, np.uint8)
    image[room:room + operand.size] = operand
    at = (operand.size - 1) // 128 * 128 + 128 if message else room
    print("permuted over", over, kind, m, k, n, message, flush=True)

    def run(out, act, w):
        body = api.mat_mul_params(out, act, w, m, k, n)
        if message:
            msg = api.build_message([(api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(OPS[kind], body))])
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        else:
            assert ctx.execute(OPS[kind], body) == 0, ctx.last_error()
            ctx.synchronize()
        return ctx.read(out[0], np.uint8, out_bytes, out[1])

    ha, hw, ho, hb = ctx.upload(x), ctx.upload(raw), ctx.alloc(out_bytes), ctx.upload(image)
    try:
        alone = run((ho, 0), (ha, 0), (hw, 0))
        inside = run((hb, at), (hb, room) if "rows" in over else (ha, 0), (hw, 0) if "rows" in over else (hb, room))
        assert np.array_equal(alone, inside) and alone.any()
        # nothing beside the output was written
        image[at:at + out_bytes] = inside
        assert np.array_equal(ctx.read(hb, np.uint8, image.size), image)
    finally:
        for h in (ha, hw, ho, hb):
            ctx.release(h)
