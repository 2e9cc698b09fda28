"""GPU parity: the batched product where its tiles, units and operand forms end, on random block bits.

Random bytes reach the largest integers of a format (Q6_K: (q - 32) * scale of 4064 and more, which one f16
number does not hold; Q5_K: 31 * 63) and every sign.  With split operands the weights are exact and an
activation keeps 22 bits, so a result is off by at most 2^-22 of sum |w x| (half a last place of the low part,
as rows scale to at most 1024), plus fp32 sums: K / 32 + 4 roundings of 2^-24 of sums no larger than
sum |q scale x| + sum |min x|, the two parts of a weight apart.  Twice that is allowed.
"""
import numpy as np
import pytest

import oracle as orc
import wgml_amd as W

pytestmark = pytest.mark.gpu
SIZES = {W.Q4_0: 18, W.Q4_1: 20, W.Q5_0: 22, W.Q5_1: 24, W.Q8_0: 34, W.Q4_K: 144, W.Q5_K: 176, W.Q6_K: 210, W.Q8_K: 292}
SCALES = {W.Q4_0: [0], W.Q4_1: [0, 2], W.Q5_0: [0], W.Q5_1: [0, 2], W.Q8_0: [0], W.Q4_K: [0, 2], W.Q5_K: [0, 2], W.Q6_K: [208]}


def random_blocks(qtype, n_elems, seed):
    rng = np.random.default_rng(seed)
    b = rng.integers(0, 256, (n_elems // (32 if SIZES[qtype] < 40 else 256), SIZES[qtype]), dtype=np.uint8)
    d = lambda: (rng.uniform(0.5, 1.5, len(b)) * 1e-3 * rng.choice([-1, 1], len(b)))  # noqa: E731
    for at in SCALES.get(qtype, []):
        b[:, at:at + 2] = d().astype(np.float16).view(np.uint8).reshape(-1, 2)
    if qtype == W.Q8_K:
        b[:, :4] = d().astype(np.float32).view(np.uint8).reshape(-1, 4)
    return b.reshape(-1)


@pytest.mark.parametrize("qtype", list(SIZES))
@pytest.mark.parametrize("T,nrows,units", [(1, 1, 1), (16, 63, 1), (33, 65, 2), (48, 64, 3), (49, 130, 2), (65, 16, 5),
                                           (96, 17, 1), (97, 129, 2), (128, 64, 9)])
def test_products_to_fp32_rounding(gpu, qtype, T, nrows, units):
    ncols = 256 * units - (0 if SIZES[qtype] > 40 else 32 * (units + T) % 224)
    raw = random_blocks(qtype, nrows * ncols, T)
    w = orc.dequantize(qtype, raw, nrows * ncols).reshape(nrows, ncols).astype(np.float64)
    x = W.rng_normal(T, T * ncols).reshape(T, ncols)
    out = W.GpuVector.init(gpu, np.full(T * nrows, np.nan, dtype=np.float32))
    m = W.GpuQuantMatrix(gpu, qtype, nrows, ncols, raw)
    W.GemmQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x.reshape(-1)), T)
    got = out.read().reshape(T, nrows)
    xa = np.abs(x).astype(np.float64)
    parts = xa @ np.abs(w).T + (xa.sum(1)[:, None] * 2 * np.abs(w).max() if qtype in (W.Q4_1, W.Q5_1, W.Q4_K, W.Q5_K) else 0)
    low = np.abs(x).max(1)[:, None] * 2.0 ** -34 * np.abs(w).sum(1)[None, :]  # low parts at the bottom of f16
    bound = 2 * (2.0 ** -22 * (xa @ np.abs(w).T) + (ncols / 32 + 4) * 2.0 ** -24 * parts + low)
    assert (np.abs(got - x.astype(np.float64) @ w.T) <= bound).all()


@pytest.mark.parametrize("qtype", list(SIZES))
def test_nothing_behind_the_last_row_is_multiplied(gpu, qtype):
    """A row that ends inside a unit of 256 columns: rows behind it, and the end of the matrix, hold other weights."""
    ncols = 256 if SIZES[qtype] > 40 else 32
    raw = random_blocks(qtype, 3 * ncols, 7)
    x = W.rng_normal(3, 5 * ncols).reshape(5, ncols)
    whole = []
    for rows in (3, 1):
        out = W.GpuVector.uninit(gpu, 5 * rows)
        m = W.GpuQuantMatrix(gpu, qtype, rows, ncols, raw[:rows * len(raw) // 3])
        W.GemmQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x.reshape(-1)), 5)
        whole.append(out.read().reshape(5, rows)[:, 0])
    assert np.array_equal(whole[0], whole[1]) and np.isfinite(whole[0]).all()
