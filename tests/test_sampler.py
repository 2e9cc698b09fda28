"""The CPU sampler (models/sampler.rs:14-130): the oracle's restatement is pinned by what the
algorithm fixes (closed forms on small distributions, an independent numpy construction of the
nucleus, the empirical distribution over many coins); the library's sampler must then return
the oracle's token for every coin.  No GPU needed."""
import ctypes as C
import subprocess
from pathlib import Path

import numpy as np
import pytest

import oracle as orc
import wgml_amd as W


def np_topp(p, topp, coin):
    """Independent construction: nucleus = shortest prefix of the descending order whose mass
    exceeds topp; draw proportionally inside it."""
    n = p.size
    cand = np.flatnonzero(p >= np.float32((1.0 - topp) / (n - 1)))
    order = cand[np.argsort(-p[cand], kind="stable")]
    cum = np.cumsum(p[order], dtype=np.float32)
    over = np.flatnonzero(cum > np.float32(topp))
    last = over[0] if over.size else order.size - 1
    r = np.float32(coin) * cum[last]
    inside = np.flatnonzero(np.float32(r) < cum[:last + 1])
    return int(order[inside[0]] if inside.size else order[last])


def test_mult_closed_form():
    p = np.float32([0.1, 0.2, 0.3, 0.4])
    for coin, want in ((0.0, 0), (0.0999, 0), (0.1, 1), (0.29, 1), (0.31, 2), (0.61, 3), (0.999, 3)):
        assert orc.sample_mult(p, coin) == want
    assert orc.sample_mult(np.float32([0.5, 0.25]), 0.9) == 1  # rounding guard: last index


def test_topp_closed_form():
    p = np.float32([0.05, 0.5, 0.15, 0.3])
    # descending: 1 (0.5), 3 (0.3), 2 (0.15), 0 (0.05); topp 0.7 -> nucleus {1, 3} (0.8 > 0.7)
    for coin in np.linspace(0, 0.999, 50):
        t = orc.sample_topp(p, 0.7, float(coin))
        assert t == (1 if coin * 0.8 < 0.5 else 3)
    # topp 0.4 -> nucleus {1} only
    assert {orc.sample_topp(p, 0.4, c) for c in (0.0, 0.5, 0.99)} == {1}
    # ties keep index order (stable sort): 0.4, 0.4 -> index 0 comes first and is the nucleus
    assert {orc.sample_topp(np.float32([0.4, 0.4, 0.2]), 0.3, c) for c in (0.0, 0.5, 0.99)} == {0}


def test_oracle_matches_independent_nucleus_and_distribution():
    rng = np.random.default_rng(0)
    logits = (rng.standard_normal(500) * 3).astype(np.float32)
    p = np.exp(logits - logits.max()).astype(np.float32)
    p /= p.sum(dtype=np.float32)
    for topp in (0.3, 0.9, 0.95):
        for coin in rng.random(200):
            assert orc.sample_topp(p, topp, float(coin)) == np_topp(p, topp, float(coin))
    # multinomial branch: empirical frequencies follow p
    coins = (np.arange(20000) + 0.5) / 20000
    counts = np.bincount([orc.sample_mult(p, float(c)) for c in coins], minlength=p.size)
    np.testing.assert_allclose(counts / coins.size, p, atol=2e-4)


@pytest.mark.parametrize("temperature,topp", [(0.0, 0.9), (0.7, 0.95), (1.3, 0.0), (1.0, 1.0),
                                              (0.2, 0.5)])
def test_library_sampler_equals_oracle(temperature, topp):
    rng = np.random.default_rng(5)
    s = W.Sampler(None, temperature, topp)
    for trial in range(40):
        logits = (rng.standard_normal(1000) * 2).astype(np.float32)
        if trial % 5 == 0:
            logits[17] = logits[400] = logits.max() + 1  # a tie at the top
        coin = float(W.rng_uniform(trial, 1)[0])
        assert s.sample(logits.copy(), coin) == orc.sample(logits, temperature, topp, coin)


def test_temperature_zero_is_argmax_and_probabilities_are_written_back():
    logits = np.float32([0.5, 2.0, 2.0, -1.0])
    assert W.Sampler(None, 0.0, 0.9).sample(logits.copy(), 0.3) == 1
    v = logits.copy()
    W.Sampler(None, 0.5, 0.0).sample(v, 0.3)
    e = np.exp((logits / np.float32(0.5)) - np.float32(4.0))
    np.testing.assert_allclose(v, e / e.sum(), rtol=1e-6)


def test_argument_checks_and_coins():
    with pytest.raises(W.WgmlError):
        W.Sampler(None, 1.0, 0.5).sample(np.zeros(4, np.float32), 1.0)  # coin must be < 1
    with pytest.raises(W.WgmlError):
        W.Sampler(None, -1.0, 0.5).sample(np.zeros(4, np.float32), 0.5)
    c = W.rng_uniform(9, 10000)
    assert c.min() >= 0.0 and c.max() < 1.0 and abs(c.mean() - 0.5) < 0.02
    assert np.array_equal(c[:100], W.rng_uniform(9, 100))


def _exp_arguments():
    """Every 1009th float of [-104, -0], those around -87 (where the sampler hands over to std::exp)
    and around the smallest results, both zeros and -inf."""
    bits = np.arange(0x80000000, np.float32(-104).view(np.uint32), 1009, dtype=np.uint64).astype(np.uint32)
    near = [np.float32(v).view(np.uint32) + np.arange(-40, 41) for v in (-87.0, -87.33655, -103.27893, -0.6931472)]
    return np.concatenate([bits.view(np.float32), np.concatenate(near).astype(np.uint32).view(np.float32),
                           np.float32([0.0, -0.0, -np.inf, np.finfo(np.float32).min])])


@pytest.fixture(scope="module")
def exp_block(tmp_path_factory):
    here = Path(__file__).parent
    out = tmp_path_factory.mktemp("exp_block") / "exp_block.so"
    subprocess.run(["g++", "-shared", "-fPIC", "-O2", "-std=c++17", "-ffp-contract=off", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-o", str(out), str(here / "exp_block.cpp")], check=True,
                   capture_output=True)
    return C.CDLL(str(out))


@pytest.mark.parametrize("avx2", [0, 1])
def test_blocks_of_exp_are_std_exp_bit_for_bit(exp_block, avx2):
    if avx2 and not exp_block.cpu_has_avx2():
        pytest.skip("no AVX2 on this machine")
    x = _exp_arguments()
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    got, want, asked = np.empty_like(x), np.empty_like(x), C.c_uint32()
    exp_block.std_exp(p(x), x.size, p(want))
    exp_block.take_exp(p(x), x.size, avx2, p(got), C.byref(asked))
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    ordinary = x >= -87  # std::exp answers for about 4 % of these and for all of the others
    assert asked.value - (~ordinary).sum() < 0.06 * ordinary.sum()


# one element, a block short of one, a whole one, one into the next, many
@pytest.mark.parametrize("n", [1, 255, 256, 257, 4000])
def test_probabilities_are_those_of_the_oracle_bit_for_bit(n):
    x = _exp_arguments()
    rng = np.random.default_rng(n)
    for trial in range(60):
        logits = rng.choice(x[x > -30] if trial % 3 else x, n)
        logits[rng.integers(n)] = 0.0  # the maximum
        if trial % 4 == 0:
            logits = logits + np.float32(3.7)
        got, want = logits.copy(), logits.copy()
        coin, t = float(W.rng_uniform(trial, 1)[0]), (1.0, 0.7)[trial % 2]
        a = W.Sampler(None, t, (0.9, 0.0)[trial % 2]).sample(got, coin)
        b = orc.lib.orc_sample(want.ctypes.data_as(C.c_void_p), n, t, (0.9, 0.0)[trial % 2], coin)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        assert a == b
