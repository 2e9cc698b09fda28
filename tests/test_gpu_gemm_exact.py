"""GPU parity: the batched products, short and long runs, where tiles, units and operand forms end, on random block bits.

Random bytes reach the largest integers of a format (Q6_K: (q - 32) * scale of 4064 and more, which one f16
number does not hold; Q5_K: 31 * 63) and every sign.  With split operands the weights are exact and an
activation keeps 22 bits, so a result is off by at most 2^-22 of sum |w x| (half a last place of the low part,
as rows scale to at most 1024), plus fp32 sums: K / 32 + 4 roundings of 2^-24 of sums no larger than
sum |w x| or, where a weight is an integer's part and an offset, sum |x| times twice the largest weight.  Twice that is allowed.
"""
import ctypes

import numpy as np
import pytest

import npref
import oracle as orc
import wgml_amd as W
from wgml_amd import _lib
from wgml_amd.models import HostMatrix, Llama2, Llama2Config

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
    assert (np.abs(got - x.astype(np.float64) @ w.T) <= 2 * split_bound(qtype, xa, w)).all()


def split_bound(qtype, xa, w):
    parts = xa @ np.abs(w).T + (xa.sum(1)[:, None] * 2 * np.abs(w).max() if qtype in (W.Q4_1, W.Q5_1, W.Q4_K, W.Q5_K) else 0)
    low = xa.max(1)[:, None] * 2.0 ** -34 * np.abs(w).sum(1)[None, :]  # low parts at the bottom of f16
    return 2.0 ** -22 * (xa @ np.abs(w).T) + (xa.shape[1] / 32 + 4) * 2.0 ** -24 * parts + low


@pytest.mark.parametrize("qtype", list(SIZES))
@pytest.mark.parametrize("T,nrows,units", [(1, 17, 2), (16, 64, 1), (17, 65, 3), (33, 130, 2), (49, 63, 5), (65, 64, 2),
                                           (96, 130, 3), (97, 16, 1), (128, 65, 9)])
def test_products_in_plain_f16(gpu, qtype, T, nrows, units):
    """An activation keeps 11 bits (half a last place: 2^-11 of |w x|, low parts as above), integers of a weight
    are exact but for Q6_K's products, which keep 11 bits too; fp32 sums as in split precision."""
    ncols = 256 * units - (0 if SIZES[qtype] > 40 else 32 * (units + T) % 224)
    raw = random_blocks(qtype, nrows * ncols, T)
    w = orc.dequantize(qtype, raw, nrows * ncols).reshape(nrows, ncols).astype(np.float64)
    x = W.rng_normal(T, T * ncols).reshape(T, ncols)
    out = W.GpuVector.init(gpu, np.full(T * nrows, np.nan, dtype=np.float32))
    m = W.GpuQuantMatrix(gpu, qtype, nrows, ncols, raw)
    gpu.set_gemm_precision(0)
    try:
        W.GemmQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x.reshape(-1)), T)
    finally:
        gpu.set_gemm_precision(1)
    xa = np.abs(x).astype(np.float64)
    bound = 2.0 ** -11 * (2 if qtype == W.Q6_K else 1) * (xa @ np.abs(w).T) + 2 * split_bound(qtype, xa, w)
    assert (np.abs(out.read().reshape(T, nrows) - x.astype(np.float64) @ w.T) <= bound).all()


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


def test_rows_beyond_four_gigabytes(gpu):
    """Q8_K takes 292 bytes for 256 weights: a matrix of fewer than 2^32 weights whose last rows start behind 2^32 bytes."""
    nrows, ncols = 58000, 1 << 16
    row = ncols // 256 * 292
    raw, rows = np.zeros(nrows * row, np.uint8), [0, 1, 542, 543, (1 << 32) // row, (1 << 32) // row + 1, nrows - 1]
    some = random_blocks(W.Q8_K, len(rows) * ncols, 9)
    for i, r in enumerate(rows):
        raw[r * row:(r + 1) * row] = some[i * row:(i + 1) * row]
    x = W.rng_normal(4, 2 * ncols).reshape(2, ncols)
    out, few = W.GpuVector.uninit(gpu, 2 * nrows), W.GpuVector.uninit(gpu, 2 * len(rows))
    m = W.GpuQuantMatrix(gpu, W.Q8_K, nrows, ncols, raw)
    W.GemmQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x.reshape(-1)), 2)
    got = out.read().reshape(2, nrows)
    m = W.GpuQuantMatrix(gpu, W.Q8_K, len(rows), ncols, some)
    W.GemmQuant.from_device(gpu).dispatch(few, m, W.GpuVector.init(gpu, x.reshape(-1)), 2)
    # (the few rows are a product of their own with another split of K: 2048 fp32 sums in another order, sqrt(2048) 2^-24)
    want = few.read().reshape(2, len(rows))
    assert np.abs(got[:, rows] - want).max() <= 4e-6 * np.abs(want).max()
    assert not np.delete(got, rows, axis=1).any()


def v_rows(gpu, qtype, raw, nrows, ncols, x, precision=1):
    """The product of a matrix with the rows of x, RMS-normalised, as a run of len(x) prompt tokens multiplies it: V of
    the first layer, between matrices of the same format for Q and K (one launch), and what it multiplied."""
    heads = ncols // 32
    cfg = Llama2Config(dim=ncols, hidden_dim=256, n_layers=1, n_q_heads=heads, n_kv_heads=nrows // 32, vocab_size=len(x),
                       seq_len=len(x), rope_base_freq=10000.0, rms_norm_eps=1e-5)
    m = Llama2(gpu, cfg)
    other = {"attn_q": (ncols, ncols), "attn_k": (nrows, ncols), "attn_output": (ncols, ncols), "ffn_gate": (256, ncols),
             "ffn_up": (256, ncols), "ffn_down": (ncols, 256)}
    for i, (name, (r, c)) in enumerate(other.items()):
        m.set_matrix(name, 0, HostMatrix(qtype, r, c, random_blocks(qtype, r * c, 50 + i)))
    m.set_matrix("attn_v", 0, HostMatrix(qtype, nrows, ncols, raw))
    m.set_matrix("output", 0, HostMatrix(W.F32, len(x), ncols, np.zeros(4 * len(x) * ncols, np.uint8)))
    for name in ("attn_norm", "ffn_norm", "output_norm"):
        m.set_vector(name, 0, np.ones(ncols))
    te = np.ascontiguousarray(x, np.float32)
    _lib.call("wgml_llama2_set_token_embd", m._h, te.ctypes.data_as(ctypes.c_void_p))
    gpu.set_gemm_precision(precision)
    try:
        m.prefill(np.arange(len(x), dtype=np.uint32))
    finally:
        gpu.set_gemm_precision(1)
    xd = te.astype(np.float64)
    return np.asarray(m.kv_download(0, 1, 0, len(x))), xd / np.sqrt((xd ** 2).mean(1, keepdims=True) + 1e-5)


@pytest.mark.parametrize("precision", [1, 0], ids=["split_f16", "plain_f16"])
@pytest.mark.parametrize("qtype", list(SIZES))
@pytest.mark.parametrize("T,nrows,ncols", [(129, 32, 512), (200, 96, 288), (256, 160, 320), (257, 320, 1280), (300, 64, 256),
                                           (513, 256, 512)])
def test_long_runs(gpu, qtype, T, nrows, ncols, precision):
    """As above, in tiles of 128 rows x 256 tokens (K and V beside the Q matrix, which is ncols rows): two more roundings of
    2^-22 in the norm; plain f16 rounds the weights themselves as well, times 2^8, of which the smallest keep 2^-25."""
    if ncols % 256 and SIZES[qtype] > 40:
        nrows, ncols = 96, 768
    raw = random_blocks(qtype, nrows * ncols, T)
    w = orc.dequantize(qtype, raw, nrows * ncols).reshape(nrows, ncols).astype(np.float64)
    got, x = v_rows(gpu, qtype, raw, nrows, ncols, W.rng_normal(T, T * ncols).reshape(T, ncols), precision)
    xa = np.abs(x)
    bound = 2 * split_bound(qtype, xa, w) + 2.0 ** -21 * (xa @ np.abs(w).T)
    if precision == 0:
        bound += 2.0 ** -10 * (xa @ np.abs(w).T) + 2.0 ** -33 * xa.sum(1)[:, None]
    assert (np.abs(got - x @ w.T) <= bound).all()


@pytest.mark.parametrize("long_run", [False, True], ids=["product", "long_run"])
@pytest.mark.parametrize("qtype", list(SIZES))
def test_parts_of_a_weight_do_not_cancel(gpu, qtype, long_run):
    """Activations of one sign, weights around zero: d q and the minimum of a Q4_1 weight are each a hundred times the
    sum of their products, so fp32 sums of the one and of the other would be off by 1.7e-6 (Q4_1, Q5_1) to 4e-6 (Q4_K,
    Q5_K) of its rms.  Sums no larger than the result: N = 3 K / 32 + K / 256 roundings of 2^-24 / sqrt(3) at most, with
    random signs: sqrt(N) 3.4e-8 = 3.5e-7 of it at K = 1024, and 1.2e-7 for the second parts of activations and
    of sums of 32 (23 bits).  A factor common to a row of V is that row's norm, in fp32 on the device."""
    K, R, T = 1024, 256, 200 if long_run else 48
    values = W.rng_normal(1, R * K, 0.0, 0.02)
    raw = npref.encode_simple(qtype, values) if qtype in (W.Q4_0, W.Q4_1, W.Q5_0, W.Q5_1, W.Q5_K, W.Q8_K) \
        else np.asarray(W.quantize(qtype, values))
    w = orc.dequantize(qtype, raw, R * K).reshape(R, K).astype(np.float64)
    z = W.rng_normal(2, T * K).reshape(T, K)
    for x in (np.abs(z), z + np.float32(3), np.maximum(z, np.float32(-0.2))):
        if long_run:
            got, xd = v_rows(gpu, qtype, raw, R, K, x)
        else:
            out, xd = W.GpuVector.uninit(gpu, T * R), x.astype(np.float64)
            m = W.GpuQuantMatrix(gpu, qtype, R, K, raw)
            W.GemmQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x.reshape(-1)), T)
            got = out.read().reshape(T, R)
        want = xd @ w.T
        factor = (got * want).sum(1, keepdims=True) / (want ** 2).sum(1, keepdims=True)
        assert np.abs(factor - 1).max() <= 1e-6
        assert np.sqrt(((got - factor * want) ** 2).mean()) <= 5e-7 * np.sqrt((want ** 2).mean())
