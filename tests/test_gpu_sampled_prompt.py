"""GPU parity: sampled generation whose prompt goes through the layers in one pass.

The oracle's forward and sampler give the token for every coin.  Two forwards differ by up to E =
1e-3 of the largest logit (the bound of test_gpu_models.py), which changes a probability by a factor
within exp(+-E / temperature) before they are normalised and so moves a boundary F between tokens by
at most F (1 - F) (exp(2 E / temperature) - 1), no more than a quarter of that bracket; and it may
change the order of tokens inside the nucleus.  A position is decided where the oracle samples the
same token for the coin moved that far either way and for logits changed by up to E; elsewhere the
token has to be one of those that this gives.  The output matrix is scaled so that, as with a trained
model, few tokens hold most of the probability: about two positions in three are decided.
"""
import numpy as np
import pytest

import oracle as orc
import wgml_amd as W
from wgml_amd.models import HostMatrix, Llama2, Llama2Config, LlamaModelType, synth_llama

pytestmark = pytest.mark.gpu


def likely_tokens(logits, temperature, topp, coin):
    """Tokens that a forward within E of these logits may sample."""
    e = 1e-3 * np.abs(logits).max()
    shift = (np.exp(2 * e / temperature) - 1) / 4
    rng = np.random.default_rng(3)
    forms = [logits] + [(logits + rng.uniform(-e, e, logits.size)).astype(np.float32) for _ in range(6)]
    coins = np.clip([coin, coin - shift, coin + shift, coin - shift / 2, coin + shift / 2], 0, 0.999999)
    return {orc.sample(l, temperature, topp, float(np.float32(c))) for l in forms for c in coins}


# below the limit, at it, odd, groups of rows read back that end with the prompt or not, a whole run,
# more than a run (steps)
@pytest.mark.parametrize("n_prompt", [1, 5, 6, 9, 10, 33, 128, 131])
@pytest.mark.parametrize("model_type", [LlamaModelType.Llama, LlamaModelType.Qwen2])
@pytest.mark.parametrize("n_new,temperature,topp", [(0, 0.7, 0.95), (8, 0.7, 0.9), (8, 0.0, 0.9), (3, 1.0, 1.0)])
def test_sampled_generation_from_a_prompt(gpu, n_prompt, model_type, n_new, temperature, topp):
    cfg = Llama2Config(dim=256, hidden_dim=512, n_layers=2, n_q_heads=4, n_kv_heads=2, vocab_size=331,
                       seq_len=160, rope_base_freq=10000.0, rms_norm_eps=1e-5)
    w = synth_llama(cfg, seed=51, scheme="q4_k_m")
    w.output = HostMatrix(W.Q6_K, cfg.vocab_size, cfg.dim,
                          W.quantize(W.Q6_K, W.rng_normal(77, cfg.vocab_size * cfg.dim, 0.0, 0.2)))
    if model_type == LlamaModelType.Qwen2:
        rng = np.random.default_rng(1)
        for layer in w.layers:
            for name, n in (("attn_q_bias", cfg.dim), ("attn_k_bias", cfg.kv_dim), ("attn_v_bias", cfg.kv_dim)):
                layer[name] = (0.1 * rng.standard_normal(n)).astype(np.float32)
    prompt = W.prompt_tokens(51, n_prompt, cfg.vocab_size)
    n_total = n_prompt + n_new
    coins = W.rng_uniform(1234, n_total)
    m = Llama2(gpu, cfg, model_type).load(w)
    m.forward(0, 0)
    step_launches = m.launches_per_token()
    got = m.generate_sampled(prompt, n_total, temperature, topp, 1234)
    if n_new == 0:  # (with tokens to generate the last step's launches are there)
        assert (m.launches_per_token() < step_launches) == (6 <= n_prompt <= 128)
    logits = m.logits().copy()
    assert np.array_equal(m.generate_sampled(prompt, n_total, temperature, topp, 1234), got)
    ref = orc.Llama2(w, rope_variant=model_type)
    checked = other_coin = 0
    for pos in range(n_total):  # the oracle follows the tokens that were generated
        want = ref.forward(int(prompt[pos] if pos < n_prompt else got[pos - 1]), pos).astype(np.float32)
        if temperature == 0.0:
            top = np.sort(want)[-2:]
            if top[1] - top[0] > 2e-3 * np.abs(want).max():
                assert int(got[pos]) == int(np.argmax(want)), pos
                checked += 1
            continue
        tokens = likely_tokens(want, temperature, topp, coins[pos])
        assert int(got[pos]) in tokens, pos
        checked += len(tokens) == 1
        # would the position before's coin have given itself away here?
        other_coin += int(got[pos]) not in likely_tokens(want, temperature, topp, coins[pos - 1])
    assert np.abs(logits - want).max() <= 1e-3 * np.abs(want).max()
    assert checked >= n_total // 3
    if temperature > 0.0 and n_total > 8:
        assert other_coin >= n_total // 3
