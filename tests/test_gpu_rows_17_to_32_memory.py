"""GPU: 17 to 32 rows where the converted copy, which only buys speed there, has no room: under a cap that other copies fill,
the weights are read as they are and nothing is evicted."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grouped", [False, True])
def test_a_copy_that_does_not_fit_the_cap_is_not_made(oracle, grouped):
    wt, m, k, n = wl.GGML_TYPE_Q8_0, 24, 4096, 1024
    rng = wl.rng_for(97, 0)
    ws = [wl.make_weights(rng, n, k, wt) for _ in range(3)]
    x = wl.make_activations(rng, m, k)
    with api.Context(device=0) as other, api.Context(device=0) as ctx:
        ctx.set_option("converted_cap_mib", 8)  # a copy takes 4.5 MiB
        hx, hq, hws = ctx.upload(x), ctx.alloc(m * (k // 32) * 34), [ctx.upload(w) for w in ws]
        outs = [ctx.alloc(m * n * 4) for _ in ws]
        # the same weights in memory of another context: no copy may be kept of those
        foreign = [ctx.register(other.device_ptr(h), other.size(h)) for h in (other.upload(w) for w in ws)]
        op = lambda code, body: (api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(code, body))
        quantize = op(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params((hq, 0), (hx, 0), k, m))

        def run(handles):
            reqs = [op(api.HTP_OPS_MAT_MUL_Q8_0_Q8_0, api.mat_mul_params((o, 0), (hq, 0), (h, 0), m, k, n)) for o, h in zip(outs, handles)]
            for msg in ([[quantize] + reqs] if grouped else [[quantize, r] for r in reqs]):
                msg = api.build_message(msg)
                assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
            return [ctx.read(o, np.float32, m * n).reshape(m, n) for o in outs]

        plain = run(foreign)
        assert ctx.converted_bytes() == 0
        first = run(hws)
        made = ctx.converted_bytes()
        assert 4 << 20 < made <= 8 << 20  # one
        again = run(hws)
        assert ctx.converted_bytes() == made
        a = oracle.quantize_q8_0(x)
        for i in range(3):
            assert np.array_equal(first[i], again[i])
            assert i == 0 or np.array_equal(first[i], plain[i])
            want, mag = oracle.mat_mul_q8_0_act_f64(a, ws[i][:64], m, k, 64, wt)
            assert np.all(np.abs(first[i][:, :64] - want) <= 1e-5 * mag)
        # room for all: copies are made from then on
        ctx.set_option("converted_cap_mib", 0)
        run(hws)
        assert ctx.converted_bytes() > made
