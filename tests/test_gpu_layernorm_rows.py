"""GPU: the LayerNorm folded into the products of GPT-2 on both sides of its lines: up to 1024 columns the staging waves find mean and
variance by themselves (one float4 per lane and wave: 64, 128, 192 and 256 of them), beyond that the workgroup does.  Against one
launch per operation of the reference, whose LayerNorm is a kernel of its own; with a row far from zero mean, whose variance is lost
if it is not taken about the mean.

Bound: both sides round the normalised row to 16 bits per block of 32 (2^-16 of its largest value); the rest is fp32 rounding."""
import numpy as np
import pytest

import npref
import wgml_amd as W
from wgml_amd.models import Gpt2, Gpt2HostWeights, Gpt2Params, HostMatrix

pytestmark = pytest.mark.gpu
FORMATS = [W.Q8_0, W.Q4_0, W.Q4_1, W.Q5_0, W.Q5_1, W.F16]


def model(gpu, qtype, heads, dim, shift, n_vocab=200):
    rng = np.random.default_rng(dim + qtype)
    p = Gpt2Params(n_vocab=n_vocab, n_seq=32, n_embd=dim, n_head=heads, n_layer=2, ff_len=2 * dim, attn_b=3 * dim)

    def mat(rows, cols):
        w = (rng.standard_normal(rows * cols) * 0.05).astype(np.float32)
        if qtype == W.F16:
            return HostMatrix(qtype, rows, cols, w.astype(np.float16).view(np.uint8))
        raw = W.quantize(qtype, w) if qtype in (W.Q8_0, W.Q4_K, W.Q6_K) else npref.encode_simple(qtype, w)
        return HostMatrix(qtype, rows, cols, raw)

    def vec(n, at=0.0):
        return (at + 0.1 * rng.standard_normal(n)).astype(np.float32)

    w = Gpt2HostWeights(params=p)
    for _ in range(p.n_layer):
        w.layers.append({"attn_w": mat(3 * dim, dim), "attn_proj_w": mat(dim, dim), "mlp_fc_w": mat(2 * dim, dim),
                         "mlp_proj_w": mat(dim, 2 * dim), "attn_b": vec(3 * dim), "attn_proj_b": vec(dim), "mlp_fc_b": vec(2 * dim),
                         "mlp_proj_b": vec(dim), "ln_1_g": vec(dim, 1.0), "ln_1_b": vec(dim), "ln_2_g": vec(dim, 1.0),
                         "ln_2_b": vec(dim)})
    w.wte = vec(n_vocab * dim, shift).reshape(n_vocab, dim)
    w.wpe = vec(p.n_seq * dim).reshape(p.n_seq, dim)
    w.lm_head = mat(n_vocab, dim)
    w.ln_f_g, w.ln_f_b = vec(dim, 1.0), vec(dim)
    return Gpt2(gpu, p).load(w)


def compare(gpu, qtype, heads, dim, shift, tol):
    m = model(gpu, qtype, heads, dim, shift)
    got = {}
    for level in (1, 0):
        m.set_fusion(level)
        for pos, tok in enumerate((3, 77, 150)):
            m.forward(tok, pos)
        got[level] = m.logits()
    assert np.abs(got[1] - got[0]).max() <= tol * np.abs(got[0]).max()


@pytest.mark.parametrize("qtype", FORMATS)
@pytest.mark.parametrize("heads,dim", [(1, 32), (3, 96), (4, 256), (9, 288), (8, 512), (12, 768), (31, 992), (16, 1024), (33, 1056),
                                       (20, 1280), (36, 2304)])
@pytest.mark.parametrize("shift", [0.0, 30.0])
def test_folded_layernorm(gpu, qtype, heads, dim, shift):
    # shift: the variance of 0.1 about a mean of 30 leaves fp32 three digits fewer on either side (2^-24 * 30 / 0.1 = 1.8e-5
    # per value; both sides subtract a mean rounded differently)
    tol = (2e-4 if qtype != W.F16 else 2e-5) if shift == 0 else 1e-3
    compare(gpu, qtype, heads, dim, shift, tol)


@pytest.mark.parametrize("qtype", [W.Q4_K, W.Q6_K, W.Q5_K, W.Q8_K, W.Q8_0])
@pytest.mark.parametrize("f32", [False, True])
def test_folded_layernorm_other_kernels(gpu, qtype, f32):
    if f32 and qtype in (W.Q5_K, W.Q8_K):
        return  # fp32 activations do not exist for them
    gpu.set_tuning(gpu.TUNE_GEMV_F32_ACTIVATIONS, int(f32))
    try:
        for dim in (768, 1280):
            compare(gpu, qtype, dim // 64, dim, 0.0, 2e-5 if f32 else 2e-4)
    finally:
        gpu.set_tuning(gpu.TUNE_GEMV_F32_ACTIVATIONS, 0)


def test_tall_output_matrix_takes_two_rows_per_wave(gpu):
    m = model(gpu, W.Q8_0, 12, 768, 0.0, n_vocab=16391)
    got = {}
    for level in (1, 0):
        m.set_fusion(level)
        m.forward(5, 0)
        got[level] = m.logits()
    assert np.abs(got[1] - got[0]).max() <= 2e-4 * np.abs(got[0]).max()
