"""GPU parity: GPT-2's prompt as products over all its tokens against the token loop's steps.

A context with plain-f16 products leaves the prompt to the steps, so the same model runs both ways.
The step's products take their input as 16-bit block fixed point (up to 1e-3 of the largest logit
over a whole model, the bound of test_gpu_models.py), the batched ones are exact to fp32 rounding:
about 1e-6 of a row's magnitude each, so that the logits after a prompt are within PROMPT of the
oracle's (three layers of four products and the output matrix; 1.2e-6 measured).  LayerNorm or GELU
rows without their low halves would put them off by 7e-5 to 4e-4 here.
"""
import numpy as np
import pytest

import oracle as orc
import wgml_amd as W
from wgml_amd.models import Gpt2, Gpt2Params, synth_gpt2

pytestmark = pytest.mark.gpu
PROMPT = 1.3e-5  # 13 products


def model_weights(p, qtype):
    w = synth_gpt2(p, seed=9, qtype=qtype)
    rng = np.random.default_rng(2)
    for layer in w.layers:
        for g in ("ln_1_g", "ln_2_g"):
            layer[g] = (1 + 0.2 * rng.standard_normal(p.n_embd)).astype(np.float32)
        for b in ("ln_1_b", "ln_2_b"):
            layer[b] = (0.2 * rng.standard_normal(p.n_embd)).astype(np.float32)
    w.ln_f_b = (0.2 * rng.standard_normal(p.n_embd)).astype(np.float32)
    return w


def stepped(gpu, m, prompt, n_total):
    gpu.set_gemm_precision(0)
    try:
        return m.generate_greedy(prompt, n_total)
    finally:
        gpu.set_gemm_precision(1)


# below the limit, at it, odd, a whole run, a run and one token; nothing or something to generate
@pytest.mark.parametrize("n_prompt", [7, 8, 33, 128, 129])
@pytest.mark.parametrize("n_new", [0, 9])
@pytest.mark.parametrize("n_embd,n_head,qtype", [(128, 4, W.Q8_0), (96, 4, W.Q8_0), (256, 1, W.Q4_K),
                                                 (320, 5, W.Q8_0)])
def test_batched_prompt_matches_the_steps(gpu, n_prompt, n_new, n_embd, n_head, qtype):
    p = Gpt2Params(n_vocab=331, n_seq=150, n_embd=n_embd, n_head=n_head, n_layer=3, ff_len=4 * n_embd,
                   attn_b=3 * n_embd)
    w = model_weights(p, qtype)
    prompt = W.prompt_tokens(9, n_prompt, p.n_vocab)
    n_total = n_prompt + n_new
    m = Gpt2(gpu, p).load(w)
    m.generate_greedy(prompt[:1], 1)
    step_launches = m.launches_per_token()
    got = m.generate_greedy(prompt, n_total)
    logits = m.logits().copy()
    if n_new == 0:  # (with tokens to generate the last step's launches and logits are there)
        assert (m.launches_per_token() < step_launches) == (n_prompt >= 8)
        ref = orc.Gpt2(w)
        for pos, token in enumerate(prompt):
            exact = ref.forward(int(token), pos)
        error = np.abs(logits - exact).max() / np.abs(exact).max()
        print(f"logit error {error:.1e}")
        assert error <= (PROMPT if n_prompt >= 8 else 1e-3)
    want = stepped(gpu, m, prompt, n_total)
    _, margins = orc.Gpt2(w).generate_greedy(prompt, n_total)
    scale = float(np.abs(m.logits()).max())
    decided = np.asarray(margins) > 4e-3 * scale
    upto = n_total
    for i in range(n_prompt - 1, n_total):  # a near-tie changes what follows it
        if not decided[i]:
            upto = i
            break
    keep = decided.copy()
    keep[upto:] = False
    assert keep.sum() >= min(n_prompt, 4)
    assert np.array_equal(got[keep], want[keep])
    if np.array_equal(got[n_prompt - 1:], want[n_prompt - 1:]):
        assert np.abs(logits - m.logits()).max() <= 2e-3 * scale
    assert np.array_equal(m.generate_greedy(prompt, n_total), got)
