"""GPU: launches of several matrices on both sides of the 64 MB that decide between one workgroup per compute unit and as many as fit:
gate/up pairs and row pairs (rotated at position 0, which changes nothing, and plain), more rows than one round of workgroups parks,
and a gated job beside a plain one.

Bound: the quantized formats take activations as 16-bit block fixed point, in steps of 2^-15 of a block's largest value, which is 2 to 3
standard deviations: an error of 2e-5 of a result's, at random.  Gating multiplies two such results.  2e-4 of the largest result is
ten times that (the dense formats' fp32 sums are far below)."""
import numpy as np
import pytest

import npref
import oracle as orc
import wgml_amd as W
from test_gpu_gemv import _fused

pytestmark = pytest.mark.gpu


def matrix(gpu, qtype, nrows, ncols, seed, x):
    """The matrix and its product with x: 61 different rows in turn."""
    n = 61 * ncols
    if qtype in (W.F32, W.F16):
        w = (0.05 * np.random.default_rng(seed).standard_normal((61, ncols))).astype(np.float16)
        raw = (w if qtype == W.F16 else w.astype(np.float32)).view(np.uint8).reshape(61, -1)
        some = w.astype(np.float64) @ x.astype(np.float64)
    else:
        raw = npref.random_blocks(qtype, n // npref.BLOCK_ELEMS[qtype], seed=seed).view(np.uint8).reshape(61, -1)
        some = orc.dequantize(qtype, raw.reshape(-1), n).reshape(61, ncols).astype(np.float64) @ x.astype(np.float64)
    turn = np.arange(nrows) % 61
    return W.GpuQuantMatrix(gpu, qtype, nrows, ncols, raw[turn].reshape(-1)), some[turn]


def gated(g, u):
    with np.errstate(over="ignore"):
        return u * (g / (1.0 + np.exp(-g)))


def check(got, want):
    assert np.abs(got - want).max() <= 2e-4 * np.abs(want).max()


@pytest.fixture(scope="module")
def gpu():
    return W.GpuInstance(0)


# MB of both matrices: 96, 48, 74, 107, 71, 32, 71, 67
@pytest.mark.parametrize("qtype,nrows,ncols", [(W.Q8_0, 11008, 4096), (W.Q8_0, 5504, 4096), (W.Q6_K, 11008, 4096), (W.Q4_K, 46400, 2048),
                                               (W.Q4_0, 15403, 4096), (W.F16, 4001, 2000), (W.F16, 8700, 2048), (W.F32, 4097, 2064)])
def test_gate_and_up(gpu, qtype, nrows, ncols):
    x = 0.1 * W.rng_normal(5, ncols)
    (g, want_g), (u, want_u) = matrix(gpu, qtype, nrows, ncols, 1, x), matrix(gpu, qtype, nrows, ncols, 2, x)
    check(_fused(gpu, [g], [u], [2], nrows, x)[0], gated(want_g, want_u))


# MB of the three: 78, 39, 90, 68, 80, 74
@pytest.mark.parametrize("qtype,nrows,ncols", [(W.Q8_0, 6002, 4096), (W.Q8_0, 3002, 4096), (W.Q6_K, 17900, 2048), (W.Q5_1, 7402, 4096),
                                               (W.F16, 6500, 2064), (W.F32, 8002, 768)])
def test_row_pairs(gpu, qtype, nrows, ncols):
    x = 0.1 * W.rng_normal(6, ncols)
    mats, want = zip(*[matrix(gpu, qtype, nrows, ncols, 3 + i, x) for i in range(3)])
    got = _fused(gpu, list(mats), [None] * 3, [1, 1, 0], nrows, x)
    for i in range(3):
        check(got[i], want[i])


def test_a_gated_job_beside_a_plain_one(gpu):
    x = 0.1 * W.rng_normal(7, 4096)
    (g, wg), (u, wu), (p, wp) = (matrix(gpu, W.Q8_0, 515, 4096, 8 + i, x) for i in range(3))
    for mats, partner, modes, want in (([g, p], [u, None], [2, 0], [gated(wg, wu), wp]), ([p, g], [None, u], [0, 2], [wp, gated(wg, wu)])):
        got = _fused(gpu, mats, partner, modes, 515, x)
        check(got[0], want[0])
        check(got[1], want[1])
