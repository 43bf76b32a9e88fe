"""GPU: a many-row matmul whose output lies over its own weights, of which the context holds (or would keep) a converted
copy: the result is that of an output elsewhere, and no copy of the overwritten weights answers a later request."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl

pytestmark = pytest.mark.gpu

OPS = {(wl.GGML_TYPE_Q4_0, False): api.HTP_OPS_MAT_MUL_Q4_0_Q8_0, (wl.GGML_TYPE_Q8_0, False): api.HTP_OPS_MAT_MUL_Q8_0_Q8_0,
       (wl.GGML_TYPE_Q4_0, True): api.HTP_OPS_MAT_MUL_Q4_0_A32, (wl.GGML_TYPE_Q8_0, True): api.HTP_OPS_MAT_MUL_Q8_0_A32}


@pytest.mark.parametrize("wt", [wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0])
@pytest.mark.parametrize("m,k,n", [(20, 1024, 2048), (32, 8960, 64), (40, 512, 700), (512, 1024, 8192)])  # (the last: FP6 for Q4_0)
@pytest.mark.parametrize("fp32_rows", [False, True])
def test_output_over_the_weights(oracle, wt, m, k, n, fp32_rows):
    rng = wl.rng_for(95, m + k + n + wt)
    w, x = np.ascontiguousarray(wl.make_weights(rng, n, k, wt)).view(np.uint8).reshape(-1), wl.make_activations(rng, m, k)
    x = x if fp32_rows else oracle.quantize_q8_0(x)
    out_bytes = m * n * 4
    at = w.size // 2 // 256 * 256  # the output covers the weights' second half and what lies behind
    image = np.zeros(max(w.size, at + out_bytes), np.uint8)
    image[:w.size] = w
    print("matmul over its weights", wt, m, k, n, fp32_rows, flush=True)
    with api.Context(device=0) as ctx:
        op = OPS[wt, fp32_rows]
        hx, hw, hb, ho = ctx.upload(x), ctx.upload(w), ctx.upload(image), ctx.alloc(out_bytes)

        def run(out, weights, rows=m):
            assert ctx.execute(op, api.mat_mul_params(out, (hx, 0), (weights, 0), rows, k, n)) == 0, ctx.last_error()
            ctx.synchronize()
            return ctx.read(out[0], np.float32, rows * n, out[1]).reshape(rows, n)

        want = run((ho, 0), hw)
        assert np.array_equal(want, run((ho, 0), hb)) and want.any()  # (a copy of the second buffer's weights is there now)
        got = run((hb, at), hb)
        if m == 32 or m == 40:
            assert np.array_equal(want, got)
        else:  # (a converted copy in the workspace: not the kernels of few rows and small matrices or of FP6 tiles, but other fp32
               # sums over the same exact block sums)
            assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
        # what lies there now, read as weights: the columns whose blocks were left alone are what they were
        left = at // (w.size // n)
        assert np.array_equal(run((ho, 0), hb)[:, :left], want[:, :left])
        ctx.write(hb, image)
        assert np.array_equal(run((ho, 0), hb), want)


@pytest.mark.parametrize("wt", [wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0])
@pytest.mark.parametrize("m", [8, 12])  # (over copies in two operand orders, made by the request that overwrites the weights)
@pytest.mark.parametrize("fp32_rows", [False, True])
def test_few_rows_over_the_weights_leave_no_copy_of_them(oracle, wt, m, fp32_rows):
    k, n = 1024, 2048
    rng = wl.rng_for(96, m + wt)
    w, x = np.ascontiguousarray(wl.make_weights(rng, n, k, wt)).view(np.uint8).reshape(-1), wl.make_activations(rng, m, k)
    x = x if fp32_rows else oracle.quantize_q8_0(x)
    print("few rows over the weights", wt, m, fp32_rows, flush=True)
    with api.Context(device=0) as ctx:
        hx, hw, hb, ho = ctx.upload(x), ctx.upload(w), ctx.upload(w), ctx.alloc(m * n * 4)

        def run(out, weights):
            assert ctx.execute(OPS[wt, fp32_rows], api.mat_mul_params(out, (hx, 0), (weights, 0), m, k, n)) == 0, ctx.last_error()
            ctx.synchronize()
            return ctx.read(out[0], np.uint8, m * n * 4, out[1])

        want = run((ho, 0), hw)
        assert np.array_equal(run((hb, w.size // 2 // 256 * 256), hb), want)
        # what lies there now, against the same bytes in a buffer of their own
        other = ctx.upload(ctx.read(hb, np.uint8, w.size))
        assert np.array_equal(run((ho, 0), hb), run((ho, 0), other))


@pytest.mark.parametrize("wt", [wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0])
# (17 to 32 rows of small matrices take the K-sliced kernel otherwise; more column tiles than are resident; more rows)
@pytest.mark.parametrize("m,k,n", [(17, 64, 32 * 1600), (24, 1024, 2048), (32, 512, 700), (32, 4096, 1024), (40, 512, 700)])
@pytest.mark.parametrize("at_end", [False, True])
def test_output_over_the_rows(oracle, wt, m, k, n, at_end):
    rng = wl.rng_for(97, m + k + n + wt)
    w, q = wl.make_weights(rng, n, k, wt), np.ascontiguousarray(oracle.quantize_q8_0(wl.make_activations(rng, m, k)))
    q, out_bytes = q.view(np.uint8).reshape(-1), m * n * 4
    at = (q.size - 1) // 16 * 16 if at_end else 0
    image = np.zeros(max(q.size, at + out_bytes), np.uint8)
    image[:q.size] = q
    print("matmul over its rows", wt, m, k, n, at_end, flush=True)
    with api.Context(device=0) as ctx:
        op = OPS[wt, False]
        hx, hw, hb, ho = ctx.upload(q), ctx.upload(w), ctx.upload(image), ctx.alloc(out_bytes)

        def run(out, rows):
            assert ctx.execute(op, api.mat_mul_params(out, (rows, 0), (hw, 0), m, k, n)) == 0, ctx.last_error()
            ctx.synchronize()
            return ctx.read(out[0], np.float32, m * n, out[1]).reshape(m, n)

        want, got = run((ho, 0), hx), run((hb, at), hb)
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max() and want.any()  # (other fp32 sums of the same exact block sums)
