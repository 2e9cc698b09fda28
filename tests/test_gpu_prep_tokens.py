"""GPU: tokens are shared out to the XCDs in eights in runs of more than 64 (prep_token): one token more and less than whole rounds of
64 and eights of them.  Every token against its own product of one row, to the bound of test_gpu_gemm_exact.py."""
import numpy as np
import pytest

import oracle as orc
import wgml_amd as W
from test_gpu_gemm_exact import random_blocks, split_bound

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [63, 64, 65, 71, 72, 73, 119, 121, 127, 128])
@pytest.mark.parametrize("qtype", [W.Q8_0, W.Q4_K])  # without and with the sums of activations
def test_every_token(gpu, qtype, T):
    nrows, ncols = 33, 768
    raw = random_blocks(qtype, nrows * ncols, T)
    w = orc.dequantize(qtype, raw, nrows * ncols).reshape(nrows, ncols).astype(np.float64)
    x = W.rng_normal(T, T * ncols).reshape(T, ncols) * np.exp2(np.arange(T) % 23 - 11)[:, None].astype(np.float32)
    out = W.GpuVector.init(gpu, np.full(T * nrows, np.nan, dtype=np.float32))
    W.GemmQuant.from_device(gpu).dispatch(out, W.GpuQuantMatrix(gpu, qtype, nrows, ncols, raw), W.GpuVector.init(gpu, x.reshape(-1)), T)
    err = np.abs(out.read().reshape(T, nrows) - x.astype(np.float64) @ w.T)
    assert (err <= 2 * split_bound(qtype, np.abs(x).astype(np.float64), w)).all()
