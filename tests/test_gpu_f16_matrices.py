"""GPU: matrices of F16 tensors, which stay 16 bits wide from 528 columns on (rows of whole tiles of 16 up to 32768) and are expanded to
f32 otherwise.  Either way a product is that of the same values as an F32 tensor: the same multiply-adds in the same order, so equal
bits, with subnormal, largest and infinite halves among them."""
import numpy as np
import pytest

import wgml_amd as W
from wgml_amd.models import Gpt2, Gpt2Params, HostMatrix, Llama2, Llama2Config, synth_gpt2, synth_llama

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return W.GpuInstance(0)


def halves(rng, n):
    v = (rng.standard_normal(n) * 0.05).astype(np.float16)
    odd = rng.integers(0, n, 9)
    v[odd] = np.array([6e-8, -6e-8, 6.1e-5, 65504, -65504, 0, -0.0, 1e-6, -1], np.float16)
    return v


def product(gpu, qtype, data, rows, cols, x):
    m = W.GpuQuantMatrix(gpu, qtype, rows, cols, data.view(np.uint8).reshape(-1))
    kept = qtype == W.F16 and 512 < cols <= 32768 and cols % 16 == 0
    assert m.shape() == (W.F32, rows, cols) and m.gguf_bytes() == (2 if kept else 4) * rows * cols
    out = W.GpuVector.uninit(gpu, rows)
    W.GemvQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x))
    return out.read(), m


@pytest.mark.parametrize("cols", [512, 516, 528, 536, 768, 1008, 1024, 1040, 3072, 32752, 32768])
@pytest.mark.parametrize("rows", [1, 17, 515, 8193])
def test_same_bits_as_f32(gpu, rows, cols):
    if rows * cols > 1 << 25:
        rows = 1031
    rng = np.random.default_rng(cols + rows)
    h, x = halves(rng, rows * cols), rng.standard_normal(cols).astype(np.float32)
    (got, m), (want, _) = product(gpu, W.F16, h, rows, cols, x), product(gpu, W.F32, h.astype(np.float32), rows, cols, x)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    back = W.GpuVector.uninit(gpu, rows * cols)
    W.Quantization.from_device(gpu).dequantize(back, m)
    assert np.array_equal(back.read().view(np.uint32), h.astype(np.float32).view(np.uint32))


def test_infinities_and_nan(gpu):
    rows, cols = 40, 768
    h = halves(np.random.default_rng(1), rows * cols).reshape(rows, cols)
    h[3, 5], h[4, 767], h[5, 0] = np.inf, -np.inf, np.nan
    x = np.ones(cols, np.float32)
    got, want = product(gpu, W.F16, h, rows, cols, x)[0], product(gpu, W.F32, h.astype(np.float32), rows, cols, x)[0]
    assert np.array_equal(got, want, equal_nan=True) and got[3] == np.inf and got[4] == -np.inf and np.isnan(got[5])


def as_half(m, qtype):
    v = m.data.view(np.float32).astype(np.float16)
    return HostMatrix(qtype, m.nrows, m.ncols, (v if qtype == W.F16 else v.astype(np.float32)).view(np.uint8).reshape(-1))


def converted(w, names, qtype_of):
    for i, layer in enumerate(w.layers):
        for k, v in list(layer.items()):
            if isinstance(v, HostMatrix):
                layer[k] = as_half(v, qtype_of(k, i))
    for n in names:
        setattr(w, n, as_half(getattr(w, n), qtype_of(n, -1)))
    return w


@pytest.mark.parametrize("dim", [384, 576, 768])  # 384: attention and output matrices expanded, the down projection not
def test_gpt2(gpu, dim):
    p = Gpt2Params(n_vocab=1003, n_seq=64, n_embd=dim, n_head=6, n_layer=2, ff_len=4 * dim, attn_b=3 * dim)
    got = {}
    for q in (W.F16, W.F32):
        m = Gpt2(gpu, p).load(converted(synth_gpt2(p, 5, W.F32), ["lm_head"], lambda k, i: q))
        got[q] = (m.generate_greedy(W.prompt_tokens(5, 4, p.n_vocab), 24), m.logits())
    assert np.array_equal(got[W.F16][0], got[W.F32][0]) and np.array_equal(got[W.F16][1], got[W.F32][1])


@pytest.mark.parametrize("mixed", [False, True])
def test_llama(gpu, mixed):
    """Mixed: F16 beside F32 matrices of the same layer."""
    cfg = Llama2Config(dim=768, hidden_dim=1280, n_layers=2, n_q_heads=12, n_kv_heads=6, vocab_size=1009, seq_len=64,
                       rope_base_freq=10000.0, rms_norm_eps=1e-5)
    other = lambda k, i: W.F32 if k in ("attn_k", "ffn_up") else W.F16  # noqa: E731
    got = []
    for of in (other if mixed else lambda k, i: W.F16, lambda k, i: W.F32):
        m = Llama2(gpu, cfg).load(converted(synth_llama(cfg, 9, "f32"), ["output"], of))
        m.prefill(W.prompt_tokens(5, 9, cfg.vocab_size))
        got.append((m.decode_greedy(3, 9, 20), m.logits()))
    if mixed:
        assert np.abs(got[0][1] - got[1][1]).max() <= 2e-5 * np.abs(got[1][1]).max()
    else:
        assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("f32", [("attn_k", "ffn_up"), ("attn_q", "ffn_gate"), ("attn_k", "attn_v"), ("attn_v",), ("ffn_gate",)])
@pytest.mark.parametrize("dim,hidden,heads,kv", [(544, 1040, 17, 17), (768, 1280, 12, 6), (1040, 2064, 13, 13)])
def test_f16_beside_f32_in_one_launch(gpu, f32, dim, hidden, heads, kv):
    """The values and the order of the sums are those of a layer all in F32."""
    cfg = Llama2Config(dim=dim, hidden_dim=hidden, n_layers=2, n_q_heads=heads, n_kv_heads=kv, vocab_size=331, seq_len=64,
                       rope_base_freq=10000.0, rms_norm_eps=1e-5)
    got = []
    for of in (lambda k, i: W.F32 if k in f32 else W.F16, lambda k, i: W.F32):
        m = Llama2(gpu, cfg).load(converted(synth_llama(cfg, 9, "f32"), ["output"], of))
        got.append((m.decode_greedy(3, 0, 20), m.logits()))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
