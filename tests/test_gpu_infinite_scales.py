"""GPU: weight blocks whose fp16 scale is infinite, 17 rows and more over int8 fragments. The columns that hold one get what
the oracle gives (an infinity, or not a number where the oracle has none either) and the others are left alone, however a
matmul's K is dealt out."""
import numpy as np
import pytest

from pyhtpops import api
from pyhtpops import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = api.Context(device=0)
    yield c
    c.close()


@pytest.mark.parametrize("wt", [wl.GGML_TYPE_Q4_0, wl.GGML_TYPE_Q8_0])
@pytest.mark.parametrize("m,k,n", [
    (20, 8960, 70), (40, 1536, 100), (33, 256, 40), (17, 1568, 70),                              # K over waves and workgroups
    (128, 1024, 96), (128, 8960, 64), (70, 1024, 8200), (600, 512, 1100),                        # operands shared, 64 x 64 tiles
    (128, 96, 17920), (128, 96, 32768)])                                                      # staged, tiles of 64 and of 128 rows
def test_infinite_weight_scales(ctx, oracle, wt, m, k, n):
    rng = wl.rng_for(96, m + k + n + wt)
    w = np.ascontiguousarray(wl.make_weights(rng, n, k, wt)).view(np.uint8).reshape(n, k // 32, -1).copy()
    inf = np.array([np.inf], np.float16).view(np.uint8)
    cols = np.unique(np.r_[rng.integers(0, n, 12), n - 1])
    for i, c in enumerate(cols):  # one block each, at the ends and at the seams of every way to deal out K
        w[c, [0, k // 32 - 1, k // 64, int(rng.integers(0, k // 32))][i % 4], :2] = inf
    a = oracle.quantize_q8_0(wl.make_activations(rng, m, k))
    print("infinite scales", wt, m, k, n, flush=True)
    with ctx.option("gemm_fp6", 0):  # (the FP6 tiles hold fp32 scales of their own; here: the kernels over fp16 scales)
        got = ctx.run_mat_mul(a, w, m, k, n, wt)
        if m <= 32:  # (small matrices of so few rows take another kernel on their own)
            with ctx.option("gemm_tile_units", 1):
                forced = ctx.run_mat_mul(a, w, m, k, n, wt)
            assert np.array_equal(np.isnan(got), np.isnan(forced)) and np.array_equal(np.isposinf(got), np.isposinf(forced))
    want = oracle.mat_mul_q8_0_act(a, w, m, k, n, wt, n_threads=8)
    others = np.setdiff1d(np.arange(n), cols)
    assert np.isfinite(got[:, others]).all() and np.abs(got[:, others] - want[:, others]).max() <= 1e-4 * np.abs(want[:, others]).max()
    assert np.isinf(got[:, cols]).any()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
