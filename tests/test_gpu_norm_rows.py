"""GPU: the norms over row lengths around what a workgroup keeps in registers (float4 per thread, 16384 floats), rows that
are no whole float4 or do not start on 16 bytes, and in place, against 64-bit sums: 24-bit inputs summed in up to
16384 / 1024 steps per thread and a tree, so a relative error of about 20 x 2^-24 in the factor; 4e-6 allowed, of
the value and of the largest one (LayerNorm subtracts a mean)."""
import numpy as np
import pytest

import wgml_amd as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 252, 256, 257, 1024, 1028, 2048, 4095, 4096, 4100, 8192, 16384, 16388, 20001])
@pytest.mark.parametrize("start", [0, 1])
def test_norms_of_rows(gpu, n, start):
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n + start) * 3 + 1).astype(np.float32)
    w = (1 + 0.1 * rng.standard_normal(n + start)).astype(np.float32)
    xd, wd = x[start:].astype(np.float64), w[start:].astype(np.float64)
    xs, ws = W.GpuVector.init(gpu, x).rows(start, n), W.GpuVector.init(gpu, w).rows(start, n)
    out = W.GpuVector.init(gpu, np.full(n, np.nan, np.float32))
    want = xd / np.sqrt((xd ** 2).mean() + 1e-5) * wd
    W.RmsNorm.from_device(gpu).dispatch(W.RmsNormConfig(1e-5), out, xs, ws)
    got = out.read()
    assert (np.abs(got - want) <= 4e-6 * (np.abs(want) + np.abs(want).max())).all()
    W.RmsNorm.from_device(gpu).dispatch(W.RmsNormConfig(1e-5), xs, xs, ws)  # onto its own input
    assert np.array_equal(xs.read(), got) if start == 0 else np.abs(xs.read() - got).max() <= 4e-6 * np.abs(got).max()
    xs = W.GpuVector.init(gpu, x).rows(start, n)
    W.LayerNorm.from_device(gpu).dispatch(out, xs)
    d = xd - xd.mean()
    want = d / np.sqrt((d ** 2).mean() + 1e-5)
    assert (np.abs(out.read() - want) <= 4e-6 * (np.abs(want) + np.abs(want).max() + 1e-3 * np.abs(xd).max())).all()
