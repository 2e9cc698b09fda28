"""GPU parity: sampled generation whose prompt goes through the layers in one pass.

The oracle's forward and sampler give the token for every coin.  Two forwards differ by up to 1e-3
of the largest logit, so a coin that lies close to a boundary between tokens may fall on either
side: a position counts where the oracle samples the same token for the coin moved by 0.02 either
way (the tokens' probabilities move by less: exp of 1e-3 x largest logit (below 8) / temperature).
"""
import numpy as np
import pytest

import oracle as orc
import wgml_amd as W
from wgml_amd.models import Llama2, Llama2Config, LlamaModelType, synth_llama

pytestmark = pytest.mark.gpu


# below the limit, at it, odd, a whole run, more than a run (steps)
@pytest.mark.parametrize("n_prompt", [1, 5, 6, 33, 128, 131])
@pytest.mark.parametrize("model_type", [LlamaModelType.Llama, LlamaModelType.Qwen2])
@pytest.mark.parametrize("n_new,temperature,topp", [(0, 0.7, 0.95), (8, 0.7, 0.9), (8, 0.0, 0.9), (3, 1.0, 1.0)])
def test_sampled_generation_from_a_prompt(gpu, n_prompt, model_type, n_new, temperature, topp):
    cfg = Llama2Config(dim=256, hidden_dim=512, n_layers=2, n_q_heads=4, n_kv_heads=2, vocab_size=331,
                       seq_len=160, rope_base_freq=10000.0, rms_norm_eps=1e-5)
    w = synth_llama(cfg, seed=51, scheme="q4_k_m")
    if model_type == LlamaModelType.Qwen2:
        rng = np.random.default_rng(1)
        for layer in w.layers:
            for name, n in (("attn_q_bias", cfg.dim), ("attn_k_bias", cfg.kv_dim), ("attn_v_bias", cfg.kv_dim)):
                layer[name] = (0.1 * rng.standard_normal(n)).astype(np.float32)
    prompt = W.prompt_tokens(51, n_prompt, cfg.vocab_size)
    n_total = n_prompt + n_new
    coins = W.rng_uniform(1234, n_total)
    m = Llama2(gpu, cfg, model_type).load(w)
    got = m.generate_sampled(prompt, n_total, temperature, topp, 1234)
    logits = m.logits().copy()
    assert np.array_equal(m.generate_sampled(prompt, n_total, temperature, topp, 1234), got)
    ref = orc.Llama2(w, rope_variant=model_type)
    checked = 0
    for pos in range(n_total):  # the oracle follows the tokens that were generated
        want = ref.forward(int(prompt[pos] if pos < n_prompt else got[pos - 1]), pos).astype(np.float32)
        assert np.abs(want).max() < 8
        if temperature == 0.0:
            top = np.sort(want)[-2:]
            if top[1] - top[0] > 2e-3 * np.abs(want).max():
                assert int(got[pos]) == int(np.argmax(want)), pos
                checked += 1
            continue
        near = {orc.sample(want.copy(), temperature, topp, float(np.clip(coins[pos] + d, 0, 0.99999)))
                for d in (-0.02, -0.01, 0.0, 0.01, 0.02)}
        if len(near) == 1:
            assert int(got[pos]) in near, pos
            checked += 1
        else:  # a boundary is close: one of the tokens around it
            lo, hi = (np.exp((want - want.max()) / temperature) >= 1e-6).nonzero()[0][[0, -1]]
            assert lo <= int(got[pos]) <= hi
    assert np.abs(logits - want).max() <= 1e-3 * np.abs(want).max()
    if temperature == 0.0 and n_total > 8:
        assert checked > n_total // 2
