"""GPU: the arg-max of a token loop taken from the maxima that the output product's waves leave, against the arg-max kernel over the
logits (decode_greedy_sync: a launch of its own, a read-back per token): every format and both activations, fewer rows than waves,
one row and several per wave, rows in pairs (Q8_0, 16384 rows and up to 1024 columns), as many waves as there is room for maxima and more;
then ties, infinities and NaN, where the first largest logit counts and only a NaN in row 0 does.  Tokens are equal."""
import numpy as np
import pytest

import npref
import wgml_amd as W
from wgml_amd.models import HostMatrix, Llama2, Llama2Config, synth_llama

pytestmark = pytest.mark.gpu
FORMATS = [W.Q8_0, W.Q4_K, W.Q6_K, W.Q5_K, W.Q8_K, W.Q4_0, W.Q4_1, W.Q5_0, W.Q5_1, W.F32, W.F16]


@pytest.fixture(scope="module")
def gpu():
    return W.GpuInstance(0)


def matrix(qtype, rows, cols, w):
    if qtype == W.F32:
        return HostMatrix(qtype, rows, cols, np.ascontiguousarray(w, np.float32).view(np.uint8).reshape(-1))
    if qtype == W.F16:
        return HostMatrix(qtype, rows, cols, w.astype(np.float16).view(np.uint8).reshape(-1))
    enc = W.quantize if qtype in (W.Q8_0, W.Q4_K, W.Q6_K) else npref.encode_simple
    return HostMatrix(qtype, rows, cols, enc(qtype, w.reshape(-1)))


def model(gpu, qtype, vocab, dim, weights=None):
    cfg = Llama2Config(dim=dim, hidden_dim=2 * dim, n_layers=1, n_q_heads=dim // 64, n_kv_heads=dim // 64, vocab_size=vocab, seq_len=64,
                       rope_base_freq=10000.0, rms_norm_eps=1e-5)
    w = synth_llama(cfg, seed=vocab + dim, scheme="q8_0")
    if weights is None:
        weights = np.random.default_rng(vocab).standard_normal((vocab, dim)).astype(np.float32)
    w.output = matrix(qtype, vocab, dim, weights)
    return Llama2(gpu, cfg).load(w)


def same_tokens(m, first, steps=12):
    want = m.decode_greedy_sync(first, 0, steps)
    got = m.decode_greedy(first, 0, steps)
    assert np.array_equal(got, want)
    logits = m.logits()
    assert got[-1] == np.argmax(logits)
    return got


@pytest.mark.parametrize("qtype", FORMATS)
@pytest.mark.parametrize("vocab", [3, 1003, 4097, 20011])
def test_tokens(gpu, qtype, vocab):
    for dim in (256, 768) if vocab > 1003 else (256, 768, 2304):
        same_tokens(model(gpu, qtype, vocab, dim), 1)


@pytest.mark.parametrize("qtype", [W.Q8_0, W.Q4_K, W.Q6_K])
def test_fp32_activations(gpu, qtype):
    gpu.set_tuning(gpu.TUNE_GEMV_F32_ACTIVATIONS, 1)
    try:
        same_tokens(model(gpu, qtype, 5003, 512), 2)
    finally:
        gpu.set_tuning(gpu.TUNE_GEMV_F32_ACTIVATIONS, 0)


def test_tall(gpu):
    """Many results per wave: 300001 rows, at most 8192 waves."""
    same_tokens(model(gpu, W.Q8_0, 300001, 256), 7)


@pytest.mark.parametrize("vocab", [1048576, 1048578])
def test_more_waves_than_room_for_maxima(gpu, vocab):
    """A wave parks 64 results: from 1048577 rows on there are more waves than kMaxRowMaxima, and the arg-max is that of the logits
    (test_host_routes.py sees the kernels)."""
    weights = np.resize(np.random.default_rng(1).standard_normal((50021, 64)).astype(np.float32), (vocab, 64))  # ties between waves
    weights[vocab - 3] = 1.5 * weights[17]
    same_tokens(model(gpu, W.Q8_0, vocab, 64, weights), 7, steps=4)


@pytest.mark.parametrize("qtype", [W.F32, W.F16])
def test_ties_and_values_without_order(gpu, qtype):
    dim, vocab = 768, 9001
    rng = np.random.default_rng(3)
    base = rng.standard_normal((vocab, dim)).astype(np.float32)
    zero = np.zeros_like(base)
    m = model(gpu, qtype, vocab, dim, zero)  # all equal: the first
    assert not m.decode_greedy(5, 0, 4).any()
    twice = base.copy()
    twice[4500:9000] = twice[:4500]  # every logit of the first half once more
    t = same_tokens(model(gpu, qtype, vocab, dim, twice), 5)
    assert (t < 4500).sum() + (t == 9000).sum() == len(t)
    nan = base.copy()
    nan[[1, 63, 64, 4096, 9000]] = np.nan  # passed over
    m = model(gpu, qtype, vocab, dim, nan)
    t = m.decode_greedy(5, 0, 1)
    assert t[0] == np.nanargmax(m.logits())
    nan[0] = np.nan  # stays the best of a scan for v > best that begins with it
    assert model(gpu, qtype, vocab, dim, nan).decode_greedy(5, 0, 1)[0] == 0
