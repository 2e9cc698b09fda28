"""Dense f32 matrices (F32 tensors, and F16 ones, expanded at creation up to 512 columns and of the same bits beyond): rows of a multiple of 16 columns
in the shared GEMV body, other widths and most narrow matrices on the general kernel
(test_host_routes.py has the line).  Against float64."""
import numpy as np
import pytest

import oracle as orc
import wgml_amd as W
from wgml_amd.models import Gpt2, Gpt2Params, HostMatrix, Llama2, Llama2Config, synth_gpt2, synth_llama

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    return W.GpuInstance(0)


def _bound(a, x):
    # a lane adds 16 products per step of 1024 columns one after the other, six more additions
    # join the lanes: each adds at most 2^-24 of the sum of magnitudes
    steps = (a.shape[1] + 1023) // 1024
    return (16 * steps + 8) * 2.0 ** -24 * (np.abs(a).astype(np.float64) @ np.abs(x).astype(np.float64))


# a tile is 16 columns, a step 1024, the largest row 32768; 20 and 1004 are no whole tiles
@pytest.mark.parametrize("ncols", [16, 768, 1008, 1024, 1040, 3072, 32752, 32768, 20, 1004])
@pytest.mark.parametrize("nrows", [1, 17, 515])
def test_gemv_f32_rows(gpu, nrows, ncols):
    rng = np.random.default_rng(ncols + nrows)
    a = rng.standard_normal((nrows, ncols)).astype(np.float32)
    x = rng.standard_normal(ncols).astype(np.float32)
    out = W.GpuVector.uninit(gpu, nrows)
    m = W.GpuQuantMatrix(gpu, W.F32, nrows, ncols, a.view(np.uint8).reshape(-1))
    W.GemvQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x))
    err = np.abs(out.read() - a.astype(np.float64) @ x.astype(np.float64))
    # (the general kernel adds 4 products per 256 columns: no more than the bound counts)
    assert (err <= _bound(a, x)).all(), err.max()


# rows below a step in the shared body; more rows than one result per lane and wave of the machine in
# the shared body and in the general kernel
@pytest.mark.parametrize("nrows,ncols", [(8193, 272), (8193, 1008), (32769, 144), (300001, 272), (300001, 32)])
def test_gemv_f32_tall(gpu, nrows, ncols):
    rng = np.random.default_rng(5)
    a = rng.standard_normal((nrows, ncols), dtype=np.float32)
    x = rng.standard_normal(ncols).astype(np.float32)
    out = W.GpuVector.uninit(gpu, len(a))
    m = W.GpuQuantMatrix(gpu, W.F32, len(a), ncols, a.view(np.uint8).reshape(-1))
    W.GemvQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x))
    assert (np.abs(out.read() - a.astype(np.float64) @ x) <= _bound(a, x)).all()


def _same(got, want):
    # sums of the same fp32 products in another order, through two layers
    assert np.abs(got - want).max() <= 2e-5 * np.abs(want).max()


@pytest.mark.parametrize("n_embd,as_f16", [(64, False), (96, True), (72, False)])  # 72: no whole tiles
def test_gpt2_dense(gpu, n_embd, as_f16):
    p = Gpt2Params(n_vocab=1003, n_seq=64, n_embd=n_embd, n_head=4 if n_embd != 72 else 2, n_layer=2,
                   ff_len=4 * n_embd, attn_b=3 * n_embd)
    w = synth_gpt2(p, 5, W.F32)
    ref = orc.Gpt2(w)
    if as_f16:
        def half(m):
            v = m.data.view(np.float32).astype(np.float16)
            return (HostMatrix(W.F16, m.nrows, m.ncols, v.view(np.uint8)),
                    HostMatrix(W.F32, m.nrows, m.ncols, v.astype(np.float32).view(np.uint8)))
        small, exact = synth_gpt2(p, 5, W.F32), synth_gpt2(p, 5, W.F32)
        for ls, le in zip(small.layers, exact.layers):
            for k, v in list(ls.items()):
                if isinstance(v, HostMatrix):
                    ls[k], le[k] = half(v)
        small.lm_head, exact.lm_head = half(w.lm_head)
        w, ref = small, orc.Gpt2(exact)
    prompt = W.prompt_tokens(5, 4, p.n_vocab)
    want, _ = ref.generate_greedy(prompt, 24)
    m = Gpt2(gpu, p).load(w)
    assert np.array_equal(m.generate_greedy(prompt, 24), want)
    folded = m.logits()
    m.set_fusion(0)
    assert np.array_equal(m.generate_greedy(prompt, 24), want)
    _same(folded, m.logits())


@pytest.mark.parametrize("model_type", [0, 1])
@pytest.mark.parametrize("f32_activations", [0, 1])
def test_llama_dense(gpu, model_type, f32_activations):
    cfg = Llama2Config(dim=128, hidden_dim=352, n_layers=2, n_q_heads=4, n_kv_heads=2, vocab_size=777, seq_len=64)
    w = synth_llama(cfg, 6, "f32")
    ref = orc.Llama2(w, rope_variant=model_type)
    prompt = W.prompt_tokens(6, 5, cfg.vocab_size)
    want, _ = ref.generate_greedy(prompt, 24)
    own = W.GpuInstance(0)
    own.set_tuning(own.TUNE_GEMV_F32_ACTIVATIONS, f32_activations)
    m = Llama2(own, cfg, model_type).load(w)
    assert np.array_equal(m.generate_greedy(prompt, 24), want)
    fused = m.logits()
    m.set_fusion(0)
    assert np.array_equal(m.generate_greedy(prompt, 24), want)
    _same(fused, m.logits())
    m.set_fusion(3)
    m.prefill(prompt)  # no batched product for dense matrices: steps through the prompt
    m2 = Llama2(own, cfg, model_type).load(w)
    for pos, t in enumerate(prompt):
        m2.forward(int(t), pos)
    assert np.array_equal(m.logits(), m2.logits())
