# A Q8_0 quantization that nothing orders against the matmuls before it in its message runs in their launch, on workgroups of
# its own (one row and the kernels of 2..16 rows that take it), or behind them. Either way every buffer must hold, byte for
# byte, what one message per request gives; what reads or overwrites something of the matmuls keeps its place.
import numpy as np
import pytest

from pyhtpops import api, workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    yield c
    c.close()


OPS = {2: api.HTP_OPS_MAT_MUL_Q4_0_Q8_0, 8: api.HTP_OPS_MAT_MUL_Q8_0_Q8_0}


# (wt, rows of the matmuls, their k, their n, rows x values of the quantization)
CASES = [
    (2, 1, 4096, (4096, 1024), (1, 11008)),   # one row, the row made in its matmuls' launch or not
    (8, 1, 1536, (8960, 96), (3, 352)),
    (2, 1, 96, (32,), (16, 32)),              # one matmul; fewer blocks than a workgroup takes
    (8, 2, 1536, (1536, 256), (2, 8960)),
    (2, 3, 4096, (2048, 11008), (3, 11008)),
    (8, 5, 1536, (8960, 4096), (5, 8960)),
    (8, 8, 4096, (1024, 4096), (8, 11008)),
    (2, 8, 4096, (64,), (8, 11008)),          # too little beside it for a small launch
    (8, 16, 1536, (32, 64), (16, 1536)),
    (2, 16, 4096, (4096, 4096), (1, 11008)),
]


# (made: the matmuls' row is quantized in their launch, which only one row can be)
@pytest.mark.parametrize("wt,m,k,ns,quant,made", [c + (made,) for c in CASES for made in ((False, True) if c[1] == 1 else (False,))])
def test_equals_one_message_per_request(ctx, oracle, wt, m, k, ns, quant, made):
    rng = wl.rng_for(91, m * 7919 + k + quant[1])
    x, hidden = wl.make_activations(rng, m, k), wl.make_activations(rng, *quant)
    hidden[0, :32] = 0.0
    hx, hh = ctx.upload(x), ctx.upload(hidden)
    hw = [ctx.upload(wl.make_weights(rng, n, k, wt)) for n in ns]
    results = []

    def op(code, payload):
        return (api.REQUEST_TYPE_OP_COMPUTE, api.op_compute_request(code, payload))

    for together in (True, False):
        ha = ctx.upload(oracle.quantize_q8_0(x).reshape(-1)) if not made else ctx.upload(np.zeros(m * k // 32 * 34, np.uint8))
        hq = [ctx.upload(np.full(quant[0] * quant[1] // 32 * 34, 0xA5, np.uint8)) for _ in range(2)]
        ho = [ctx.upload(np.zeros(m * n, np.float32)) for n in ns]
        h2 = ctx.upload(np.zeros(m * ns[0], np.float32))
        hq2 = ctx.upload(np.zeros(m * ns[0] // 32 * 34, np.uint8))
        reqs = [op(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params((ha, 0), (hx, 0), k, m))] if made else []
        reqs += [op(OPS[wt], api.mat_mul_params((o, 0), (ha, 0), (w, 0), m, k, n)) for o, w, n in zip(ho, hw, ns)]
        reqs.append(op(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params((hq[0], 0), (hh, 0), quant[1], quant[0])))
        reqs.append(op(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params((hq[1], 0), (hh, 0), quant[1], quant[0])))  # behind it
        # ordered: a matmul behind, a quantization of what a matmul wrote, one over the rows that it read
        reqs.append(op(OPS[wt], api.mat_mul_params((h2, 0), (ha, 0), (hw[0], 0), m, k, ns[0])))
        reqs.append(op(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params((hq2, 0), (h2, 0), ns[0], m)))
        reqs.append(op(OPS[wt], api.mat_mul_params((h2, 0), (ha, 0), (hw[0], 0), m, k, ns[0])))
        if m * k <= quant[0] * quant[1]:
            reqs.append(op(api.HTP_OPS_QUANTIZE_Q8_0, api.rms_norm_params((ha, 0), (hh, 0), k, m)))
        for msg in ([api.build_message(reqs)] if together else [api.build_message([r]) for r in reqs]):
            assert ctx.process_message(msg) == 0 and not any(api.message_request_states(msg)), ctx.last_error()
        hs = [ha, h2, hq2] + hq + ho
        results.append([ctx.read(h, np.uint8, ctx.size(h)) for h in hs])
        for h in hs:
            ctx.release(h)
    try:
        for i, (a, b) in enumerate(zip(*results)):
            assert np.array_equal(a, b), "buffer %d" % i
        assert np.array_equal(results[0][3], oracle.quantize_q8_0(hidden).reshape(-1))
        assert np.array_equal(results[0][4], results[0][3])
    finally:
        for h in [hx, hh] + hw:
            ctx.release(h)
