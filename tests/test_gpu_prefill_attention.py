"""GPU: attention of 16 tokens per workgroup turns blocks of 16 cache rows in LDS: fewer blocks than waves, last blocks of 1, 15 and 16
rows, heads that are not shared out over the XCDs in eights, groups of one and three.  Against a workgroup per token, whose
fp32 sums have another order: the bound of test_gpu_prefill_long.py."""
import numpy as np
import pytest

import wgml_amd as W
from test_gpu_prefill_long import config, state, weights
from wgml_amd.models import Llama2, LlamaModelType

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,start", [(2, 0), (15, 0), (16, 0), (17, 16), (33, 47), (49, 79), (400, 33)])
@pytest.mark.parametrize("heads,kv_heads,head_size", [(3, 1, 32), (12, 4, 48), (5, 5, 64), (24, 8, 96), (6, 2, 112), (3, 3, 128)])
def test_blocks_and_heads(gpu, heads, kv_heads, head_size, n, start):
    cfg = config(heads * head_size, 256, heads, kv_heads, 440)
    w = weights(cfg, "q8_0", False)
    toks = W.prompt_tokens(9, start + n, cfg.vocab_size)
    got = []
    for per_token in (0, 1):
        m = Llama2(gpu, cfg, LlamaModelType.Llama).load(w)
        gpu.set_tuning(gpu.TUNE_PREFILL_ATTENTION_PER_TOKEN, per_token)
        try:
            if start:
                m.prefill(toks[:start])
            m.prefill(toks[start:], start_pos=start)
        finally:
            gpu.set_tuning(gpu.TUNE_PREFILL_ATTENTION_PER_TOKEN, 0)
        got.append(state(m, cfg, start + n))
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.abs(a - b).max() <= 2e-4 * np.abs(b).max()
